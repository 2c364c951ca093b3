"""Small-level Vanka sweeps that run several to a launch (k_vanka_multi) against the
one-sweep-a-launch path with its apply pass and, for a few sweeps, the CPU oracle: the
same bits.  Levels: of one tile (16 cells a side or fewer), one cell more, one side of
either kind, tiles of 3, 2 and 1 sweeps that end at, before and past a level's edge; with
and without idle blocks; counts that divide evenly into launches and not."""
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
@pytest.mark.parametrize("n", [1, 2, 3, 7, 10])
@pytest.mark.parametrize("shape", [(1, 1), (1, 40), (9, 12), (16, 16), (17, 16), (16, 77), (33, 17), (64, 64), (70, 75),
                                   (128, 128), (135, 100), (150, 170), (20, 1200)])
def test_sweeps_of_one_launch_bitwise(shape, n, local):
    ny, nx = shape
    s = random_state(ny=ny, nx=nx, seed=7 * ny + nx, vel=100.0)
    dev = {k: torch.as_tensor(np.ascontiguousarray(s[k]), device="cuda") for k in ("U", "f", "bed", "B", "beta", "gamma")}
    prm = O.params()
    g = _lib.GlideGeom(ny, nx, s["dx"], s["dt"])
    p = _lib.GlideParams(prm.n, prm.eps_reg, prm.water_drag, prm.calving_rate, prm.gl_sigmoid_c, prm.gl_derivatives)
    nby, nbx = ny // 14 + 1, nx // 14 + 1
    blk = None
    if local:
        b = np.random.default_rng(n).random((nby, nbx)) < 0.4
        blk = torch.as_tensor(b.astype(np.uint8).reshape(-1), device="cuda")
    out = []
    try:
        for cells in (0, 1 << 20):
            _lib.call("glide_set_small_levels", cells, 2)
            U = dev["U"].clone()
            scratch = torch.full((5 * ny * nx,), float("nan"), dtype=torch.float64, device="cuda")
            _lib.call("glide_vanka_sweep", ctypes.byref(g), ctypes.byref(p), U.data_ptr(), dev["f"].data_ptr(),
                      dev["bed"].data_ptr(), dev["B"].data_ptr(), dev["beta"].data_ptr(), dev["gamma"].data_ptr(),
                      blk.data_ptr() if local else None, n, 10, scratch.data_ptr(),
                      torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            out.append(U.cpu().numpy())
    finally:
        _lib.call("glide_set_small_levels", 208 * 208, 2)
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1])
    if n <= 2 and ny * nx <= 5000:
        cells = np.array([[b[i // 14, j // 14] for j in range(nx)] for i in range(ny)]).astype(np.uint8) if local else None
        ref = s["U"]
        for _ in range(n):
            ref = O.vanka_sweep(ny, nx, s["dx"], s["dt"], prm, ref, s["f"], s["bed"], s["B"], s["beta"], s["gamma"],
                                active=cells)
        assert np.array_equal(out[1], ref)
