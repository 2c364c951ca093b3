"""The residual with one tile a workgroup and with workgroups that loop over tiles
(glide_set_persistence) against the CPU oracle: the same bits.  More tiles than 256
workgroups, whole chunks of them and not, edge faces from the last tiles."""
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


@pytest.mark.parametrize("shape", [(2072, 64), (1031, 130), (515, 321), (3, 5)])
def test_residual_loop_bitwise(shape):
    ny, nx = shape
    s = random_state(ny=ny, nx=nx, seed=ny + nx)
    prm = O.params()
    ref = O.residual(ny, nx, s["dx"], s["dt"], prm, s["U"], s["f"], s["bed"], s["B"], s["beta"], s["mask"], s["gamma"])
    g = _lib.GlideGeom(ny, nx, s["dx"], s["dt"])
    p = _lib.GlideParams(prm.n, prm.eps_reg, prm.water_drag, prm.calving_rate, prm.gl_sigmoid_c, prm.gl_derivatives)
    d = {k: torch.as_tensor(np.ascontiguousarray(s[k], dtype=np.float64), device="cuda")
         for k in ("U", "f", "bed", "B", "beta", "mask", "gamma")}
    try:
        for per_cu in (64, 1):
            _lib.call("glide_set_persistence", 1, per_cu)
            r = torch.full_like(d["U"], float("nan"))
            _lib.call("glide_residual", ctypes.byref(g), ctypes.byref(p), r.data_ptr(), d["U"].data_ptr(), d["f"].data_ptr(),
                      None, d["bed"].data_ptr(), d["B"].data_ptr(), d["beta"].data_ptr(), d["mask"].data_ptr(),
                      d["gamma"].data_ptr(), torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            assert np.array_equal(r.cpu().numpy(), ref)
    finally:
        _lib.call("glide_set_persistence", 1, 64)
