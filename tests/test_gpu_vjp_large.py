"""The VJP and the adjoint residual of levels that the last-level cache doesn't hold (tiles
row by row, stores past the caches) and just below them against the per-point form: the
same bits."""
import ctypes

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from glide_amd import _lib  # noqa: E402


@pytest.mark.parametrize("gl", [0, 1])
@pytest.mark.parametrize("ny,nx", [(1600, 1613), (1600, 1614), (1601, 1728), (65, 40000)])   # the line: 2581110 cells
def test_large_levels_same_bits(ny, nx, gl):
    gen = torch.Generator(device="cuda").manual_seed(ny + nx)
    nu, nv, nc = ny * (nx + 1), (ny + 1) * nx, ny * nx

    def uniform(lo, hi, n=nc):
        return lo + (hi - lo) * torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)

    d = dict(U=torch.cat([uniform(-100.0, 100.0, nu + nv), uniform(0.1, 1500.0)]), bed=uniform(-1500.0, 800.0),
             B=uniform(19.0, 29.0), beta=uniform(0.01, 1.0), mask=(uniform(0.0, 1.0) < 0.1).double(),
             gamma=uniform(0.1, 0.2), Lambda=uniform(-1.0, 1.0, nu + nv + nc), f_adj=uniform(-1.0, 1.0, nu + nv + nc))
    lev = _lib.GlideLevel()
    lev.g, lev.p = _lib.GlideGeom(ny, nx, 2000.0, 10.0), _lib.GlideParams(3.0, 1e-6, 1e-3, 1.0, 0.1, gl)
    for k, t in d.items():
        setattr(lev, k, t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    out = []
    for ty in (0, -1):
        _lib.call("glide_set_tile_height", 1, ty)
        l, r = (torch.full_like(d["U"], float("nan")) for _ in range(2))
        _lib.call("glide_vjp", ctypes.byref(lev.g), ctypes.byref(lev.p), l.data_ptr(), d["U"].data_ptr(),
                  d["Lambda"].data_ptr(), *(d[k].data_ptr() for k in ("bed", "B", "beta", "mask", "gamma")), st)
        lev.r_adj = r.data_ptr()
        _lib.call("glide_adjoint_residual", ctypes.byref(lev), st)
        torch.cuda.synchronize()
        out.append((l, r))
    for a, b in zip(*out):
        assert torch.isfinite(a).all() and torch.equal(a, b)
