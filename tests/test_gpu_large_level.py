"""Levels of more tiles than 64 workgroups a CU, the most that glide_set_persistence
counts: one tile a workgroup as on every smaller level.  Sweeps of one call against as many
calls of one sweep, and against the kernels that loop over tiles; the residual likewise.
The same bits."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover - collected only where a GPU is present
    pytest.skip("no GPU", allow_module_level=True)

from glide_amd import _lib  # noqa: E402


@pytest.mark.parametrize("local", [False, True])
@pytest.mark.parametrize("ny,nx", [(2056, 2050), (16500, 250)])   # 16962 and 16500 tiles of 64 x 4
def test_one_tile_a_workgroup_same_bits(ny, nx, local):
    gen = torch.Generator(device="cuda").manual_seed(ny)
    nu, nv, nc = ny * (nx + 1), (ny + 1) * nx, ny * nx

    def uniform(lo, hi, n=nc):
        return lo + (hi - lo) * torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)

    U0 = torch.cat([uniform(-100.0, 100.0, nu + nv), uniform(0.1, 1500.0)])
    bed, B, beta = uniform(-1500.0, 800.0), uniform(19.0, 29.0), uniform(0.01, 1.0)
    f = uniform(-1.0, 1.0, nu + nv + nc)
    gamma, mask = torch.full((nc,), 0.1, dtype=torch.float64, device="cuda"), (uniform(0.0, 1.0) < 0.1).double()
    blk = (uniform(0.0, 1.0, (ny // 14 + 1) * (nx // 14 + 1)) < 0.1).to(torch.uint8) if local else None
    g, p = _lib.GlideGeom(ny, nx, 2000.0, 10.0), _lib.GlideParams(3.0, 1e-6, 1e-3, 1.0, 0.1, 0)
    st = torch.cuda.current_stream().cuda_stream

    def sweeps(calls, each):
        U = U0.clone()
        scratch = torch.full((5 * nc,), float("nan"), dtype=torch.float64, device="cuda")
        for _ in range(calls):
            _lib.call("glide_vanka_sweep", ctypes.byref(g), ctypes.byref(p), U.data_ptr(), f.data_ptr(), bed.data_ptr(),
                      B.data_ptr(), beta.data_ptr(), gamma.data_ptr(), blk.data_ptr() if local else None, each, 3,
                      scratch.data_ptr(), st)
        torch.cuda.synchronize()
        return U

    def residual():
        r = torch.full_like(U0, float("nan"))
        _lib.call("glide_residual", ctypes.byref(g), ctypes.byref(p), r.data_ptr(), U0.data_ptr(), f.data_ptr(), None,
                  bed.data_ptr(), B.data_ptr(), beta.data_ptr(), mask.data_ptr(), gamma.data_ptr(), st)
        torch.cuda.synchronize()
        return r

    single, folded, r = sweeps(3, 1), sweeps(1, 3), residual()
    try:
        _lib.call("glide_set_persistence", 0, 8)
        _lib.call("glide_set_persistence", 1, 8)
        looped, r_looped = sweeps(1, 3), residual()
    finally:
        _lib.call("glide_set_persistence", 0, 64)
        _lib.call("glide_set_persistence", 1, 64)
    assert torch.isfinite(single).all() and not torch.equal(single, U0)
    assert torch.equal(single, folded) and torch.equal(single, looped)
    assert torch.isfinite(r).all() and torch.equal(r, r_looped)
