"""The blocked barotropic kernel: several substeps per launch on 64 x 64 staged
regions whose valid part shrinks by 3 per substep.  Against one launch per
substep and the oracle, bit-exact, at grids one point around one and two output
tiles, grids so small that a region holds a periodic domain several times, a
domain of several tiles, every boundary type, and 1 to 35 substeps per call
(one launch, the uneven split of the last ones, either velocity first)."""
from dataclasses import replace

import numpy as np
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, BC_STATIC, BC_WALL, Config, make_case

pytestmark = pytest.mark.gpu

BCS = {"static": (BC_STATIC, BC_STATIC), "walls": (BC_PERIODIC, BC_WALL), "periodic": (BC_PERIODIC, BC_PERIODIC),
       "periodic_y": (BC_STATIC, BC_PERIODIC)}
FIELDS = ("eta", "ubt", "vbt", "ubt_av", "vbt_av", "eta_av")


@pytest.mark.parametrize("bc", sorted(BCS))
@pytest.mark.parametrize("ni,nj,nstep", [(10, 10, 5), (16, 11, 2), (17, 30, 1), (47, 48, 6), (48, 47, 7), (96, 50, 11),
                                         (97, 20, 3), (150, 131, 35)])
def test_blocked_substeps(ni, nj, nstep, bc):
    from hackathon_mom6_miniapp_amd.model import Model
    from oracle.pyoracle import Oracle

    cfg = Config(ni=ni, nj=nj, nk=1, bt_nsteps=nstep, dt=10.0 * nstep, bc_x=BCS[bc][0], bc_y=BCS[bc][1],
                 coriolis="betaplane", f0=1e-4, beta=2e-11, Kh=1e3)
    case = make_case(cfg, seed=ni + nstep, bump=(0.5, 40.0e3))
    rng = np.random.default_rng(ni * nj)
    for f, m in (("ubt", "mask2dCu"), ("vbt", "mask2dCv")):   # also in the halos, as stored (not yet images)
        case[f] = np.asfortranarray(0.05 * rng.standard_normal(case[f].shape) * case[m])
    ora = Oracle(cfg, case)
    ora.step(2)
    for opts in ({}, {"bt_substeps": 1}, {"bt_substeps": 3}, {"bt_substeps": 5, "bt_rows": 0}):
        print(f"[gpu bt blocks] {ni}x{nj} {bc} nstep={nstep} {opts}", flush=True)
        gpu = Model(cfg, case)
        for k, v in opts.items():
            gpu.set_option(k, v)
        gpu.step(2)
        gpu.synchronize()
        for f in FIELDS:
            # (at nk = 1 a field of the model reads as 2D)
            assert np.array_equal(gpu.get(f).squeeze(), ora.field(f).squeeze()), (opts, f)
        gpu.close()
