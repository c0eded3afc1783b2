"""Launch-shape options return to the rule and reach the lengths it uses.

* momentum_tile and momentum_splits: marches of up to 4, 5, 8, 32, 64 and 128 rows
  on a grid of 33, against the automatic march, and back to it with 0;
* bt_substeps: 6 to 16 substeps per launch (output tiles down to 16 x 16) against
  one launch per substep, and back to the automatic number with 0.

Bit for bit, in a model and an ensemble."""
import numpy as np
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, BC_STATIC, BC_WALL, Config, make_case

pytestmark = pytest.mark.gpu

FIELDS = ("u", "v", "h", "up", "vp", "eta", "ubt", "vbt", "ubt_av", "vbt_av", "eta_av")


def _cfg(ni, nj, nk, nstep, bc=(BC_PERIODIC, BC_WALL), bih=False):
    return Config(ni=ni, nj=nj, nk=nk, bt_nsteps=nstep, dt=10.0 * nstep, bc_x=bc[0], bc_y=bc[1],
                  coriolis="betaplane", f0=1e-4, beta=2e-11, Kh=1e3, biharmonic=bih, Ah=1e11)


def _same(a, b, what):
    for f in FIELDS:
        assert np.array_equal(a.get(f), b.get(f)), (what, f)


@pytest.mark.parametrize("bih", [False, True])
@pytest.mark.parametrize("nk", [1, 3])
def test_march_lengths(nk, bih):
    from hackathon_mom6_miniapp_amd.model import Ensemble, Model

    cfg = _cfg(66, 37, nk, 4, bih=bih)   # 33 rows
    case = make_case(cfg, init="seeded", seed=nk)
    want = Model(cfg, case)
    want.step(3)
    want.synchronize()
    # (tile, splits): 8*tile/splits rows, at least 4
    for tile, splits in ((4, 8), (4, 6), (8, 8), (16, 4), (8, 2), (4, 1), (16, 1), (0, 0), (0, 16), (8, 0), (0, 0)):
        print(f"[gpu options] nk={nk} biharmonic={bih} tile={tile} splits={splits}", flush=True)
        one, ens = Model(cfg, case), Ensemble([cfg, cfg], [case, case])
        for m in (one, ens):
            m.step(1)
            m.set_option("momentum_tile", 16)
            m.set_option("momentum_splits", 2)
            m.step(1)
            m.set_option("momentum_tile", tile)
            m.set_option("momentum_splits", splits)
            m.step(1)
            m.synchronize()
        _same(want, one, (tile, splits))
        _same(want, ens.members[1], (tile, splits))
        one.close()
        ens.close()
    want.close()


@pytest.mark.parametrize("bc", [(BC_STATIC, BC_STATIC), (BC_PERIODIC, BC_WALL), (BC_PERIODIC, BC_PERIODIC)])
@pytest.mark.parametrize("ni,nj,nstep", [(20, 19, 17), (53, 21, 33), (38, 70, 16)])
def test_substeps_per_launch(ni, nj, nstep, bc):
    from hackathon_mom6_miniapp_amd.model import Ensemble, Model

    cfg = _cfg(ni, nj, 1, nstep, bc)
    case = make_case(cfg, seed=ni, bump=(0.5, 40.0e3))
    want = Model(cfg, case)
    want.set_option("bt_substeps", 1)
    want.step(2)
    want.synchronize()
    for n in (6, 8, 14, 15, 16, 0):
        print(f"[gpu options] {ni}x{nj} {bc} nstep={nstep} bt_substeps={n}", flush=True)
        one, ens = Model(cfg, case), Ensemble([cfg, cfg], [case, case])
        for m in (one, ens):
            m.set_option("bt_substeps", 3)
            m.step(1)
            m.set_option("bt_substeps", n)
            m.step(1)
            m.synchronize()
        _same(want, one, n)
        _same(want, ens.members[1], n)
        one.close()
        ens.close()
    want.close()


def test_refused_values():
    from hackathon_mom6_miniapp_amd._lib import Mom6hError
    from hackathon_mom6_miniapp_amd.model import Ensemble, Model

    cfg = _cfg(20, 16, 2, 4)
    case = make_case(cfg, init="seeded", seed=1)
    one, ens = Model(cfg, case), Ensemble([cfg], [case])
    for m in (one, ens):
        for key, values in (("momentum_tile", (-1, -0.5, 3, 32)), ("momentum_splits", (-1, -0.5)),
                            ("bt_substeps", (-1, 0.5, 2.5, 17))):
            for v in values:
                with pytest.raises(Mom6hError):
                    m.set_option(key, v)
        m.close()
