"""The fields del2u and del2v of a biharmonic model: Del2 of the velocities that
the last corrector started from (up, vp), asked for before the first step (zero),
after steps, and followed through later steps by their device address; zero
outside their ranges.  Against the formula in numpy in the model's type and
order of operations, bit for bit; in a model (also replayed as a graph) and an
ensemble.  A model without the term has no such fields."""
from dataclasses import replace

import numpy as np
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, BC_WALL, Config, make_case

pytestmark = pytest.mark.gpu

CFG = Config(ni=70, nj=22, nk=3, bt_nsteps=4, bc_x=BC_PERIODIC, bc_y=BC_WALL, coriolis="betaplane", f0=1e-4,
             beta=2e-11, Kh=1e3, biharmonic=True, Ah=1e11, no_slip=True)


def _del2(cfg, case, up, vp):
    T = np.float32 if cfg.precision == "mixed" else np.float64
    dx = cfg.dx_km * 1000.0
    idx = 1.0 / dx
    r, i1, i3, a2 = T(dx * idx), T(idx), T(idx * idx * idx), T(dx * dx)
    u, v, m = up.astype(T), vp.astype(T), case["mask2dBu"].astype(T)[:, :, None]
    xx, xy = np.zeros_like(u), np.zeros_like(u)
    dudx = r * ((i1 * u[1:, 1:]) - (i1 * u[:-1, 1:]))
    dvdy = r * ((i1 * v[1:, 1:]) - (i1 * v[1:, :-1]))
    xx[1:, 1:] = dudx - dvdy
    dvdx = r * ((v[1:, :-1] * i1) - (v[:-1, :-1] * i1))
    dudy = r * ((u[:-1, 1:] * i1) - (u[:-1, :-1] * i1))
    slip = T(2.0) - m if cfg.no_slip else m
    xy[:-1, :-1] = slip[:-1, :-1] * (dvdx + dudy)
    isd, _, jsd, _, isc, iec, jsc, jec = cfg.bounds
    i0, i1_, j0, j1 = isc - isd, iec - isd, jsc - jsd, jec - jsd
    du, dv = np.zeros_like(u), np.zeros_like(v)
    I, J = slice(i0 - 1, i1_ + 1), slice(j0, j1 + 1)
    du[I, J] = i3 * ((a2 * xy[I, J]) - (a2 * xy[I, j0 - 1:j1])) + i3 * ((a2 * xx[i0:i1_ + 2, J]) - (a2 * xx[I, J]))
    I, J = slice(i0, i1_ + 1), slice(j0 - 1, j1 + 1)
    dv[I, J] = i3 * ((a2 * xy[I, J]) - (a2 * xy[i0 - 1:i1_, J])) - i3 * ((a2 * xx[I, j0:j1 + 2]) - (a2 * xx[I, J]))
    return du, dv


def _check(cfg, case, model, ptr=None):
    want = _del2(cfg, case, model.get("up"), model.get("vp"))
    for f, w in zip(("del2u", "del2v"), want):
        assert w.any() and np.array_equal(model.get(f), w), f
        if ptr:
            assert model.device_ptr(f) == ptr[f]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_del2_fields(precision):
    from hackathon_mom6_miniapp_amd.model import Ensemble, Model

    print(f"[gpu del2] {precision}", flush=True)
    cfg = replace(CFG, precision=precision)
    case = make_case(cfg, init="seeded", seed=4)
    ens, late = Ensemble([cfg, cfg], [case, case]), Model(cfg, case)
    single, graph = Model(cfg, case), Model(cfg, case, graph=True)
    early = (single, graph, ens.members[0])
    assert not single.get("del2u").any() and not graph.get("del2v").any() and not ens.members[0].get("del2u").any()
    assert single.field_bytes("del2u") == (4 if precision == "mixed" else 8)
    ptrs = [{f: m.device_ptr(f) for f in ("del2u", "del2v")} for m in early]
    for n in (1, 2):
        for m in (ens, late, single, graph):
            m.step(n)
            m.synchronize()
        for m, p in zip(early, ptrs):
            _check(cfg, case, m, p)
    _check(cfg, case, late)
    _check(cfg, case, ens.members[1])
    for m in (ens, late, single, graph):
        m.close()


def test_no_del2_without_the_term():
    from hackathon_mom6_miniapp_amd._lib import Mom6hError
    from hackathon_mom6_miniapp_amd.model import Model

    cfg = replace(CFG, biharmonic=False)
    m = Model(cfg, make_case(cfg, init="seeded", seed=4))
    with pytest.raises(Mom6hError):
        m.get("del2u")
    m.close()
