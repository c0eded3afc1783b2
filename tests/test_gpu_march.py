"""The fused momentum stencil's march: one wave covers 62 columns (60 with the
biharmonic term) and a chunk of rows of one layer.  Widths one column around
one and two strips, the smallest grid, and marches from 4 rows to more than
the grid has, against the oracle (bit-exact in FP64) and, for the FP32 form,
against the FP64 path."""
from dataclasses import replace

import numpy as np
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, BC_WALL, Config, make_case

pytestmark = pytest.mark.gpu

# (ni, nj): the compute domain is (ni - 4) x (nj - 4)
SIZES = [(10, 10), (64, 13), (65, 22), (66, 14), (67, 37), (124, 12), (125, 16), (128, 12), (129, 41)]


def _cfg(ni, nj, bih, **kw):
    return Config(ni=ni, nj=nj, nk=3, bt_nsteps=6, bc_x=BC_PERIODIC, bc_y=BC_WALL, coriolis="betaplane", f0=1e-4,
                  beta=2e-11, Kh=1e3, biharmonic=bih, Ah=1e11 if bih else 1e10, **kw)


@pytest.mark.parametrize("bih", [False, True])
@pytest.mark.parametrize("ni,nj", SIZES)
def test_march_edges(ni, nj, bih):
    from hackathon_mom6_miniapp_amd.model import Model
    from oracle.pyoracle import Oracle

    cfg = _cfg(ni, nj, bih, no_slip=ni % 2 == 1)
    case = make_case(cfg, seed=ni + nj)
    ora = Oracle(cfg, case)
    ora.step(2)
    mixed = None
    for tile, splits in ((None, None), (4, 8), (4, 3), (16, 1)):
        print(f"[gpu march] {ni}x{nj} biharmonic={bih} tile={tile} splits={splits}", flush=True)
        gpu, mix = Model(cfg, case), Model(replace(cfg, precision="mixed"), case)
        for m in (gpu, mix):
            if tile is not None:
                m.set_option("momentum_tile", tile)
                m.set_option("momentum_splits", min(splits, cfg.nk))
            m.step(2)
            m.synchronize()
        for f in ("u", "v", "up", "vp", "h"):
            assert np.array_equal(gpu.get(f), ora.field(f)), (tile, splits, f)
            # FP32 storage (2**-24 relative) through two steps of a few hundred
            # operations on values no larger than the field's maximum
            assert np.abs(mix.get(f) - ora.field(f)).max() <= 1e-5 * np.abs(ora.field(f)).max(), (tile, splits, f)
        got = [mix.get(f) for f in ("u", "v", "h")]
        assert mixed is None or all(np.array_equal(a, b) for a, b in zip(mixed, got))
        mixed = got
        gpu.close()
        mix.close()
