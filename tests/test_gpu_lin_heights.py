"""The JVP, the VJP and the adjoint residual with the tile height chosen by level size
against the per-point form, bit for bit, on both sides of each line of the choice (256 CUs):
the VJP's tiles with a CU each and not, resident at once and not, the JVP's likewise."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import random_state

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from glide_amd import _lib  # noqa: E402


@pytest.mark.parametrize("gl", [False, True])
@pytest.mark.parametrize("shape", [(128, 512), (129, 512), (384, 512), (385, 512), (70, 1)])
def test_choice_by_level_size_same_bits(shape, gl):
    ny, nx = shape
    s = random_state(ny=ny, nx=nx, seed=ny + 3 * nx)
    s["mask"][ny // 3:: 7, nx // 2:: 5] = 1.0
    prm = O.params(gl_derivatives=gl)
    g = _lib.GlideGeom(ny, nx, s["dx"], s["dt"])
    p = _lib.GlideParams(prm.n, prm.eps_reg, prm.water_drag, prm.calving_rate, prm.gl_sigmoid_c, prm.gl_derivatives)
    rng = np.random.default_rng(ny)
    d = {k: torch.as_tensor(np.ascontiguousarray(v, dtype=np.float64), device="cuda")
         for k, v in dict({k: s[k] for k in ("U", "bed", "B", "beta", "mask", "gamma")}, Lambda=rng.normal(size=s["U"].size),
                          f_adj=rng.normal(size=s["U"].size)).items()}
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    out = []
    for ty in (0, -1):
        _lib.call("glide_set_tile_height", 1, ty)
        res = [torch.full_like(d["U"], float("nan")) for _ in range(3)]
        for name, r in zip(("glide_jvp", "glide_vjp"), res):
            _lib.call(name, ctypes.byref(g), ctypes.byref(p), r.data_ptr(), d["U"].data_ptr(), d["Lambda"].data_ptr(),
                      *(d[k].data_ptr() for k in ("bed", "B", "beta", "mask", "gamma")), st)
        lev = _lib.GlideLevel()
        lev.g, lev.p, lev.r_adj = g, p, res[2].data_ptr()
        for k, t in d.items():
            setattr(lev, k, t.data_ptr())
        _lib.call("glide_adjoint_residual", ctypes.byref(lev), st)
        torch.cuda.synchronize()
        out.append(res)
    for a, b in zip(*out):
        assert torch.isfinite(a).all() and torch.equal(a, b)
