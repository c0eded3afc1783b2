"""Calls of two barotropic substeps: one launch per substep below 160 000 points
(all members' together in an ensemble), two blocked launches from there on.  Grids
on both sides against the oracle, bit-exact, and ensembles against single runs."""
import numpy as np
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, BC_WALL, Config, make_case

pytestmark = pytest.mark.gpu
FIELDS = ("eta", "ubt", "vbt", "ubt_av", "vbt_av", "eta_av")


def _run(cls, *args):
    r = cls(*args)
    r.step(3)
    r.synchronize()
    return r


@pytest.mark.parametrize("bc_y", [BC_WALL, BC_PERIODIC])
@pytest.mark.parametrize("ni,nj", [(16, 11), (398, 397), (398, 398)])   # 159 600 and 160 000 points
def test_two_substeps(ni, nj, bc_y):
    from hackathon_mom6_miniapp_amd.model import Ensemble, Model
    from oracle.pyoracle import Oracle

    print(f"[gpu bt two] {ni}x{nj} bc_y={bc_y}", flush=True)
    cfg = Config(ni=ni, nj=nj, nk=1, bt_nsteps=2, dt=20.0, bc_x=BC_PERIODIC, bc_y=bc_y, coriolis="betaplane", f0=1e-4,
                 beta=2e-11 if bc_y == BC_WALL else 0.0, Kh=1e3)
    case = make_case(cfg, seed=ni, bump=(0.5, 40.0e3))
    ora = Oracle(cfg, case)
    ora.step(3)
    gpu, ens = _run(Model, cfg, case), _run(Ensemble, [cfg, cfg], [case, case])
    for f in FIELDS:
        want = ora.field(f).squeeze()
        assert np.array_equal(gpu.get(f).squeeze(), want), f
        for m in ens.members:
            assert np.array_equal(m.get(f).squeeze(), want), f
    gpu.close()
    ens.close()
