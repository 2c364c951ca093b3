"""The adjoint smoother's one-pass colours against the separate adjoint
residual and Vanka pass, bit for bit: the tiles read their neighbours' lambda
from one array and write another, so sizes end at, before and after a tile."""
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

DEV = torch.device("cuda")


@pytest.mark.parametrize("gl", [False, True])
@pytest.mark.parametrize("shape", [(2, 2), (3, 63), (4, 64), (5, 65), (33, 130), (130, 66), (512, 70), (260, 258), (520, 380)])
def test_colour_in_one_pass_same_bits(gl, shape):
    ny, nx = shape
    s = random_state(ny=ny, nx=nx, seed=ny + 7 * nx)
    prm = O.params(gl_derivatives=gl)
    rng = np.random.default_rng(ny * nx)
    nt, nc = s["U"].size, ny * nx
    H, gamma = s["U"][nt - nc:], np.asarray(s["gamma"]).ravel()
    gamma[::5] = H[::5] + 1.0   # held cells
    lam0, f_adj = rng.normal(size=nt), rng.normal(size=nt)
    d = {k: torch.as_tensor(np.ascontiguousarray(v, dtype=np.float64).ravel(), device=DEV)
         for k, v in dict(U=s["U"], bed=s["bed"], B=s["B"], beta=s["beta"], gamma=gamma, f_adj=f_adj).items()}
    lev = (_lib.GlideLevel * 1)()
    lev[0].g = _lib.GlideGeom(ny, nx, s["dx"], s["dt"])
    lev[0].p = _lib.GlideParams(prm.n, prm.eps_reg, prm.water_drag, prm.calving_rate, prm.gl_sigmoid_c, prm.gl_derivatives)
    for k in ("f", "r", "w", "z", "Lambda", "r_adj"):
        d[k] = torch.zeros(nt, dtype=torch.float64, device=DEV)
    for k in ("chi", "mask"):
        d[k] = torch.zeros(nc, dtype=torch.float64, device=DEV)
    d["scratch"] = torch.zeros(5 * nc, dtype=torch.float64, device=DEV)
    d["active"] = torch.zeros(nc, dtype=torch.uint8, device=DEV)
    for k, t in d.items():
        setattr(lev[0], k, t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ref, r_ref = None, None
    mask = torch.as_tensor((H <= gamma + 0.1).astype(np.float64), device=DEV)
    for one_pass in (False, True):
        d["Lambda"].copy_(torch.as_tensor(lam0))
        d["mask"].copy_(mask)
        if one_pass:
            _lib.call("glide_adjoint_vcycle", lev, 1, ctypes.byref(_lib.schedule(adj_coarse=3)), st)
        else:
            p = lambda k: ctypes.c_void_p(d[k].data_ptr())  # noqa: E731
            for color in (0, 1) * 3:
                _lib.call("glide_adjoint_residual", ctypes.byref(lev[0]), st)
                _lib.call("glide_vanka_adjoint_pass", ctypes.byref(lev[0].g), ctypes.byref(lev[0].p), p("Lambda"),
                          p("Lambda"), p("mask"), p("r_adj"), p("U"), p("bed"), p("B"), p("beta"), p("gamma"), color, 1.0,
                          st)
            ref, r_ref = d["Lambda"].cpu().numpy(), d["r_adj"].cpu().numpy()
        torch.cuda.synchronize()
    assert np.isfinite(ref).all() and not np.array_equal(ref, lam0)
    assert np.array_equal(d["Lambda"].cpu().numpy(), ref)
    assert np.array_equal(d["r_adj"].cpu().numpy(), r_ref)
