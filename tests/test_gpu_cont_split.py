"""The zonal continuity pass with a column's levels split over four waves:
depths on both sides of every slot class, rows that end one face around a
block's 62, called through the module API on states that take each of its
branches, against the oracle bit for bit.

* seeded: random velocities, limited and unlimited cells, with and without a
  transport target (the zero-target iteration of BT_cont), both limiters;
* rest: zero velocities (the u = 0 branch of the layer flux) in half the columns;
* close: velocities of a column that differ by units in the last place, where
  BT_cont's test velocities must be folded in k order;
* land: faces whose mask is not 1, where the CFL bracket must be folded in k order."""
import ctypes as C

import numpy as np
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, BC_WALL, Config, make_case

pytestmark = pytest.mark.gpu

BT = ("FA_u_EE", "FA_u_E0", "FA_u_W0", "FA_u_WW", "uBT_WW", "uBT_EE", "BT_h_u")


def _state(kind, cfg, case):
    rng = np.random.default_rng(cfg.nk + cfg.ni)
    u, h = np.array(case["u"], order="F"), np.array(case["h0"], order="F")
    h[rng.random(h.shape) < 0.05] = 1.0e-10          # cells at the limiter's minimum
    mask = np.array(case["mask2dCu"], order="F")
    if kind == "rest":
        u[::2] = 0.0
    elif kind == "close":
        ulp = rng.integers(-2, 3, size=u.shape)
        u = np.asfortranarray(u[:, :, :1] * (1.0 + ulp * 2.0 ** -52))
    elif kind == "land":
        mask[rng.random(mask.shape) < 0.1] = 0.0
        mask[3, :] = 0.5
    return u, h, mask


@pytest.mark.parametrize("kind,ni,target,monotonic", [
    ("seeded", 65, False, False), ("seeded", 66, True, False), ("seeded", 128, False, True),
    ("rest", 66, False, False), ("close", 64, False, False), ("close", 65, True, False), ("land", 66, True, False)])
@pytest.mark.parametrize("nk", [1, 3, 4, 16, 17, 29, 41, 53, 64, 65, 75, 76, 77, 80])
def test_split_pass(nk, kind, ni, target, monotonic):
    from hackathon_mom6_miniapp_amd._lib import check, lib
    from oracle.pyoracle import Oracle

    print(f"[gpu continuity split] nk={nk} {kind} ni={ni} target={target} monotonic={monotonic}", flush=True)
    cfg = Config(ni=ni, nj=10, nk=nk, bt_nsteps=6, bc_x=BC_PERIODIC, bc_y=BC_WALL, coriolis="betaplane", f0=1e-4,
                 beta=2e-11, Kh=1e3, monotonic=monotonic)
    case = make_case(cfg, init="seeded", seed=nk)
    u, h, mask = _state(kind, cfg, case)
    case["mask2dCu"] = mask
    ora = Oracle(cfg, case)
    shape = (cfg.n1, cfg.n2, nk)
    uhbt = np.zeros(shape[:2], order="F")
    if target:
        uhbt[:] = np.random.default_rng(5).normal(0.0, 2.0e5, uhbt.shape)
    ora.field("uhbt")[...] = uhbt
    oh, ouh = np.zeros(shape, order="F"), np.zeros(shape, order="F")
    ora.call("om_continuity_ppm", u.reshape(shape, order="F"), h.reshape(shape, order="F"), oh, ouh, scalar=cfg.dt)

    L, cs, dx = lib(), C.c_void_p(), cfg.dx_km * 1000.0
    keep = [np.full(shape[:2], x, order="F") for x in (1.0 / (dx * dx), 1.0 / dx, dx)]
    keep += [np.asfortranarray(case["mask2dT"]), mask]
    iarea, idx, dxs, mT, mCu = [a.ctypes.data_as(C.POINTER(C.c_double)) for a in keep]
    check(L.mom6h_continuity_init(C.byref(cs), *cfg.bounds, nk, iarea, idx, dxs, mT, int(monotonic), dxs, dxs, mCu))
    dev, ptrs = [], {}

    def up(a):
        p = C.c_void_p()
        check(L.mom6h_malloc(C.byref(p), a.nbytes))
        check(L.mom6h_memcpy_h2d(p, a.ctypes.data_as(C.c_void_p), a.nbytes))
        dev.append(p)
        return p

    for n in ("h", "uh", "u_cor", "BT_h_u"):
        ptrs[n] = up(np.zeros(shape, order="F"))
    for n in BT[:6] + ("du_cor",):
        ptrs[n] = up(np.zeros(shape[:2], order="F"))
    bt = (C.c_void_p * 7)(*[ptrs[n] for n in BT])
    check(L.mom6h_continuity_ppm(cs, up(u), up(h), ptrs["h"], ptrs["uh"], C.c_double(cfg.dt),
                                 up(uhbt) if target else C.c_void_p(), C.byref(bt), ptrs["u_cor"],
                                 ptrs["du_cor"], 0, C.c_void_p()))
    check(L.mom6h_device_synchronize())
    isd, ied, jsd, jed, isc, iec, jsc, jec = cfg.bounds
    cells, faces = (slice(isc - 1, iec), slice(jsc - 1, jec)), (slice(isc - 2, iec), slice(jsc - 1, jec))
    want = dict(h=oh, uh=ouh, **{n: ora.field(n) for n in BT + ("u_cor", "du_cor")})
    for n, p in ptrs.items():
        got = np.zeros(want[n].shape, order="F")
        check(L.mom6h_memcpy_d2h(got.ctypes.data_as(C.c_void_p), p, got.nbytes))
        at = cells if n == "h" else faces
        assert np.array_equal(got[at], want[n][at]), n
    check(L.mom6h_continuity_end(cs))
    for p in dev:
        check(L.mom6h_free(p))
