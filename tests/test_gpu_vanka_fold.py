"""Large-level Vanka sweeps without an apply pass (k_vanka_fold): several sweeps of one call
against as many calls of one sweep, which run the smoother and its apply pass, and, for two
sweeps, the CPU oracle: the same bits.  Levels: less than a 64 x 4 tile, whole tiles, one row
or column more, interior tiles, one tile wide or high; idle blocks that leave whole tiles
idle; even and odd counts.  The scratch starts as NaN: no value of it may be read unwritten."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import random_state

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover - collected only where a GPU is present
    pytest.skip("no GPU", allow_module_level=True)

from glide_amd import _lib  # noqa: E402


@pytest.mark.parametrize("local", [False, True])
@pytest.mark.parametrize("n", [2, 3, 4, 5])
@pytest.mark.parametrize("shape", [(9, 12), (4, 64), (5, 300), (40, 123), (64, 128), (65, 129), (67, 191), (131, 193),
                                   (260, 266), (600, 40)])
def test_sweeps_without_apply_bitwise(shape, n, local):
    ny, nx = shape
    s = random_state(ny=ny, nx=nx, seed=11 * ny + nx, vel=100.0)
    dev = {k: torch.as_tensor(np.ascontiguousarray(s[k]), device="cuda") for k in ("U", "f", "bed", "B", "beta", "gamma")}
    prm = O.params()
    g = _lib.GlideGeom(ny, nx, s["dx"], s["dt"])
    p = _lib.GlideParams(prm.n, prm.eps_reg, prm.water_drag, prm.calving_rate, prm.gl_sigmoid_c, prm.gl_derivatives)
    nby, nbx = ny // 14 + 1, nx // 14 + 1
    blk = None
    if local:
        b = np.random.default_rng(n).random((nby, nbx)) < 0.15
        blk = torch.as_tensor(b.astype(np.uint8).reshape(-1), device="cuda")

    def sweeps(calls, each):
        U = dev["U"].clone()
        scratch = torch.full((5 * ny * nx,), float("nan"), dtype=torch.float64, device="cuda")
        for _ in range(calls):
            _lib.call("glide_vanka_sweep", ctypes.byref(g), ctypes.byref(p), U.data_ptr(), dev["f"].data_ptr(),
                      dev["bed"].data_ptr(), dev["B"].data_ptr(), dev["beta"].data_ptr(), dev["gamma"].data_ptr(),
                      blk.data_ptr() if local else None, each, 10, scratch.data_ptr(),
                      torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return U.cpu().numpy()

    try:
        _lib.call("glide_set_small_levels", 0, 0)
        ref, out = sweeps(n, 1), sweeps(1, n)
    finally:
        _lib.call("glide_set_small_levels", 208 * 208, 2)
    assert np.isfinite(ref).all()
    assert np.array_equal(ref, out)
    if n == 2 and ny * nx <= 13000:
        cells = np.array([[b[i // 14, j // 14] for j in range(nx)] for i in range(ny)]).astype(np.uint8) if local else None
        o = s["U"]
        for _ in range(n):
            o = O.vanka_sweep(ny, nx, s["dx"], s["dt"], prm, o, s["f"], s["bed"], s["B"], s["beta"], s["gamma"],
                              active=cells)
        assert np.array_equal(out, o)
