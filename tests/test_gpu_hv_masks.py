"""hor_visc's march with constant coefficients reads 0/1 masks as bytes and other
masks as they are: land inside the domain and fractional masks, Laplacian and
biharmonic, chunks of 8 rows and of 40, against the oracle bit for bit."""
import numpy as np
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, BC_WALL, Config, make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bih", [False, True])
@pytest.mark.parametrize("no_slip", [False, True])
@pytest.mark.parametrize("masks", ["land", "fractional T", "fractional Bu"])
@pytest.mark.parametrize("ni,nj,nk", [(10, 10, 2), (61, 31, 3), (130, 419, 70)])   # 70 levels: 40 rows per wave
def test_masks(ni, nj, nk, masks, no_slip, bih):
    from hackathon_mom6_miniapp_amd.model import Model
    from oracle.pyoracle import Oracle

    print(f"[gpu hv masks] {ni}x{nj}x{nk} {masks} no_slip={no_slip} biharmonic={bih}", flush=True)
    cfg = Config(ni=ni, nj=nj, nk=nk, bt_nsteps=1, bc_x=BC_PERIODIC, bc_y=BC_WALL, coriolis="betaplane", f0=1e-4,
                 beta=2e-11, Kh=20.0, Ah=1e9, biharmonic=bih, no_slip=no_slip)
    case = make_case(cfg, seed=ni)
    rng = np.random.default_rng(ni)
    for name in ("mask2dT", "mask2dBu"):
        m = np.array(case[name], order="F")
        m[rng.random(m.shape) < 0.1] = 0.0
        if masks.endswith(name[6:]):
            m[rng.random(m.shape) < 0.1] *= 0.625
        case[name] = m
    gpu, ora = Model(cfg, case), Oracle(cfg, case)
    gpu.set_option("fused", 0.0)
    gpu.step(1)
    gpu.synchronize()
    ora.step(1)
    for f in ("diffu", "diffv", "u", "v"):
        assert np.array_equal(gpu.get(f), ora.field(f)), f
    gpu.close()
