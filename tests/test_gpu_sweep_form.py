"""The autotuner times the smoother's tile heights only on phases whose sweeps run it
(several sweeps a launch and folded sweeps have one shape), and the timing of a sweep
in its phase's form leaves the members' state alone: ensembles whose phases take several
sweeps a launch, no apply pass, and the smoother with one (a level too narrow to fold)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():  # pragma: no cover
    pytest.skip("no GPU", allow_module_level=True)

from glide_amd import _lib  # noqa: E402
from glide_amd import synthetic as S  # noqa: E402
from glide_amd.autotune import tune  # noqa: E402
from glide_amd.ensemble import Ensemble  # noqa: E402
from glide_amd.physics import IcePhysics  # noqa: E402


# sizes, levels, and the form of each phase (finest first)
@pytest.mark.parametrize("sizes,levels,forms", [([(32, 48), (16, 16)], 1, [3]), ([(256, 272), (264, 256)], 2, [-1, 1]),
                                                ([(264, 256), (256, 4)], 1, [0])])
def test_heights_are_timed_where_they_are_run(sizes, levels, forms):
    members = []
    for d in S.ensemble_members(sizes, seed0=900, dx=2000.0):
        ph = IcePhysics(d["ny"], d["nx"], d["dx"], n_levels=levels)
        ph.set_geometry(d["bed"], d["H"])
        ph.set_parameters(B=d["B"], beta=d["beta"], smb=d["smb"])
        members.append(ph)
    ens = Ensemble(members)
    ens.forward(10.0, n_vcycles=1)
    got = [ens.sweep_form(p) for p in range(ens.n_phases)]
    assert got == forms, got
    torch.cuda.synchronize()
    before = [m.grid.U.cpu().numpy() for m in members]
    for p in range(ens.n_phases + 1):
        for local in (False, True):
            assert ens.time_sweep(p, local, reps=2) > 0.0
    rec = tune(ens, reps=1, use_cache=False)
    torch.cuda.synchronize()
    assert set(rec["times_ms"]["vanka"]) == {str(p) for p, f in enumerate(got) if f == 0}
    assert all(rec["choice"]["vanka"][str(p)] == 4 for p, f in enumerate(got) if f)
    for m, u in zip(members, before):
        assert np.array_equal(m.grid.U.cpu().numpy(), u)
    with pytest.raises(_lib.GlideError):
        ens.sweep_form(ens.n_phases + 1)
    ens.close()
