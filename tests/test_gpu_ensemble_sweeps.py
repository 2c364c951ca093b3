"""Batched sweeps whose launches take several sweeps each, or fold the apply pass into the
next one, against the members solved alone (the single-level sweeps, which the oracle pins):
the same bits.  Ensembles whose finest phase takes 3, 2 and 1 sweeps a launch and, too large
for that, none; counts that divide evenly into launches and not; a level too narrow to fold."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from glide_amd import synthetic as S  # noqa: E402
from glide_amd.ensemble import Ensemble  # noqa: E402
from glide_amd.physics import IcePhysics  # noqa: E402


@pytest.mark.parametrize("counts", [(1, 2), (3, 5), (10, 7)])
@pytest.mark.parametrize("sizes", [[(32, 48), (16, 16)], [(96, 96), (64, 80)], [(128, 144), (96, 64), (16, 40)],
                                   [(256, 272), (64, 128), (130, 66)], [(264, 256), (256, 4)]])
def test_batched_sweeps_bitwise(sizes, counts):
    pre, post = counts
    sched = dict(pre=pre, post=post, coarse=7, local_passes=2, local_sweeps=post, n_newton=4)
    data = S.ensemble_members(sizes, seed0=900, dx=2000.0)

    def make(d):
        ph = IcePhysics(d["ny"], d["nx"], d["dx"], n_levels=min(2, d["n_levels"]))
        ph.set_geometry(d["bed"], d["H"])
        ph.set_parameters(B=d["B"], beta=d["beta"], smb=d["smb"])
        ph.set_schedule(**sched)
        return ph

    solo = [make(d) for d in data]
    for ph in solo:
        ph.forward(10.0, n_vcycles=1)
    batch = [make(d) for d in data]
    ens = Ensemble(batch)
    ens.set_schedule(**sched)
    ens.forward(10.0, n_vcycles=1)
    torch.cuda.synchronize()
    for k, (a, b) in enumerate(zip(solo, batch)):
        ua, ub = a.grid.U.cpu().numpy(), b.grid.U.cpu().numpy()
        assert np.isfinite(ua).all() and np.array_equal(ua, ub), f"member {k}"
    ens.close()
