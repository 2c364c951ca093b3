"""Combinations of the sweep kernels that the other tests leave out, bit for bit.
Grounding-line derivatives on: folded sweeps and several sweeps a launch against the CPU
oracle, batched members (several sweeps a launch, folded, and the smoother with its apply
pass in a phase with a level too narrow to fold) against the members alone.  Full folded
sweeps over more than 600 rows against single ones.  The adjoint's colours with a scratch
of NaN against a scratch of zeros."""
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
from glide_amd import synthetic as S  # noqa: E402
from glide_amd.ensemble import Ensemble  # noqa: E402
from glide_amd.physics import IcePhysics  # noqa: E402

NAN = float("nan")


def _params(prm):
    return _lib.GlideParams(prm.n, prm.eps_reg, prm.water_drag, prm.calving_rate, prm.gl_sigmoid_c, prm.gl_derivatives)


def _sweeps(s, prm, blk, calls, each):
    ny, nx = s["ny"], s["nx"]
    g, p = _lib.GlideGeom(ny, nx, s["dx"], s["dt"]), _params(prm)
    d = {k: torch.as_tensor(np.ascontiguousarray(s[k]), device="cuda") for k in ("U", "f", "bed", "B", "beta", "gamma")}
    b = torch.as_tensor(blk.astype(np.uint8).reshape(-1), device="cuda") if blk is not None else None
    scratch = torch.full((5 * ny * nx,), NAN, dtype=torch.float64, device="cuda")
    for _ in range(calls):
        _lib.call("glide_vanka_sweep", ctypes.byref(g), ctypes.byref(p), d["U"].data_ptr(), d["f"].data_ptr(),
                  d["bed"].data_ptr(), d["B"].data_ptr(), d["beta"].data_ptr(), d["gamma"].data_ptr(),
                  b.data_ptr() if b is not None else None, each, 10, scratch.data_ptr(),
                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return d["U"].cpu().numpy()


@pytest.mark.parametrize("local", [False, True])
@pytest.mark.parametrize("cells", [0, 208 * 208])   # folded, and several sweeps a launch
@pytest.mark.parametrize("shape,n", [((9, 12), 2), ((65, 129), 3), ((40, 123), 4)])
def test_grounding_line_derivatives(shape, n, cells, local):
    ny, nx = shape
    s = random_state(ny=ny, nx=nx, seed=5 * ny + nx, vel=100.0)
    prm = O.params(gl_derivatives=True)
    blk = np.random.default_rng(n).random((ny // 14 + 1, nx // 14 + 1)) < 0.4 if local else None
    _lib.call("glide_set_small_levels", cells, 2)
    out = _sweeps(s, prm, blk, 1, n)
    active = np.array([[blk[i // 14, j // 14] for j in range(nx)] for i in range(ny)]).astype(np.uint8) if local else None
    ref = s["U"]
    for _ in range(n):
        ref = O.vanka_sweep(ny, nx, s["dx"], s["dt"], prm, ref, s["f"], s["bed"], s["B"], s["beta"], s["gamma"],
                            active=active)
    assert np.isfinite(ref).all() and np.array_equal(out, ref)


@pytest.mark.parametrize("gl", [False, True])
@pytest.mark.parametrize("shape", [(1031, 130), (700, 517)])
def test_full_folds_of_many_rows(shape, gl):
    s = random_state(ny=shape[0], nx=shape[1], seed=sum(shape), vel=100.0)
    prm = O.params(gl_derivatives=gl)
    ref, out = _sweeps(s, prm, None, 4, 1), _sweeps(s, prm, None, 1, 4)
    assert np.isfinite(ref).all() and np.array_equal(ref, out)


@pytest.mark.parametrize("gl", [False, True])
@pytest.mark.parametrize("sizes,levels,form", [([(32, 48), (16, 16)], 1, 3), ([(256, 272), (64, 128), (130, 66)], 2, -1),
                                               ([(264, 256), (256, 4)], 1, 0)])
def test_batched_members(sizes, levels, form, gl):
    sched = dict(pre=4, post=3, coarse=6, local_passes=2, local_sweeps=2, n_newton=5)
    data = S.ensemble_members(sizes, seed0=910, dx=2000.0)

    def make(d):
        ph = IcePhysics(d["ny"], d["nx"], d["dx"], n_levels=levels, gl_derivatives=gl)
        ph.set_geometry(d["bed"], d["H"])
        ph.set_parameters(B=d["B"], beta=d["beta"], smb=d["smb"])
        ph.set_schedule(**sched)
        return ph

    solo, batch = [make(d) for d in data], [make(d) for d in data]
    for ph in solo:
        ph.forward(10.0, n_vcycles=1)
    ens = Ensemble(batch)
    assert ens.sweep_form(0) == form
    ens.set_schedule(**sched)
    ens.forward(10.0, n_vcycles=1)
    torch.cuda.synchronize()
    for a, b in zip(solo, batch):
        ua, ub = a.grid.U.cpu().numpy(), b.grid.U.cpu().numpy()
        assert np.isfinite(ua).all() and np.array_equal(ua, ub)
    ens.close()


@pytest.mark.parametrize("shape", [(1, 7), (5, 65), (130, 66), (260, 258), (520, 380)])
def test_adjoint_leaves_nothing_unwritten(shape):
    ny, nx = shape
    s = random_state(ny=ny, nx=nx, seed=ny + nx)
    prm = O.params(gl_derivatives=True)
    rng = np.random.default_rng(ny)
    nt, nc = s["U"].size, ny * nx
    lam0, f_adj = rng.normal(size=nt), rng.normal(size=nt)
    out = []
    for fill in (0.0, NAN):
        d = {k: torch.as_tensor(np.ascontiguousarray(v, dtype=np.float64).ravel().copy(), device="cuda") for k, v in dict(
            U=s["U"], bed=s["bed"], B=s["B"], beta=s["beta"], gamma=s["gamma"], f_adj=f_adj, Lambda=lam0).items()}
        d.update({k: torch.zeros(nt, dtype=torch.float64, device="cuda") for k in ("f", "r", "w", "z", "r_adj")})
        d.update({k: torch.zeros(nc, dtype=torch.float64, device="cuda") for k in ("chi", "mask")})
        d["scratch"] = torch.full((5 * nc,), fill, dtype=torch.float64, device="cuda")
        d["active"] = torch.zeros(nc, dtype=torch.uint8, device="cuda")
        lev = (_lib.GlideLevel * 1)()
        lev[0].g, lev[0].p = _lib.GlideGeom(ny, nx, s["dx"], s["dt"]), _params(prm)
        for k, t in d.items():
            setattr(lev[0], k, t.data_ptr())
        _lib.call("glide_adjoint_vcycle", lev, 1, ctypes.byref(_lib.schedule(adj_coarse=3)),
                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        out.append((d["Lambda"].cpu().numpy(), d["r_adj"].cpu().numpy()))
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)
