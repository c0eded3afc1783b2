"""Planes whose byte offsets over several levels pass 4 GiB take kernels of their
own: the zonal continuity with one buffer base per level (and an ensemble's member
by member), the vertical viscosity with one wave per column.  Shallow wide grids
that repeat a small pattern, against a small grid holding the pattern once, bit
for bit: each column or row sees the same values there.  The small grids are held
against the oracle by the other tests."""
import ctypes as C
from dataclasses import replace

import numpy as np
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, Config, make_case

pytestmark = pytest.mark.gpu

DX = 1.0e4


def _bounds(n1, n2):
    return 1, n1, 1, n2, 4, n1 - 3, 4, n2 - 3


def _at(n, period):
    """Position in the pattern of each index of an axis (3 halo cells on either side)."""
    return (np.arange(n) - 3) % period


def _D(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


class _Device:
    """Device copies of host arrays, freed together."""

    def __init__(self):
        from hackathon_mom6_miniapp_amd._lib import check, lib
        self.L, self.check, self.held = lib(), check, []

    def up(self, a):
        p = C.c_void_p()
        self.check(self.L.mom6h_malloc(C.byref(p), a.nbytes))
        self.held.append(p)
        self.check(self.L.mom6h_memcpy_h2d(p, np.ascontiguousarray(a).ctypes.data_as(C.c_void_p), a.nbytes))
        return p

    def zeros(self, *shape):
        p = C.c_void_p()
        n = 8 * int(np.prod(shape))
        self.check(self.L.mom6h_malloc(C.byref(p), n))
        self.held.append(p)
        self.check(self.L.mom6h_memset(p, 0, n))
        return p

    def down(self, p, *shape):
        a = np.empty(shape)
        self.check(self.L.mom6h_memcpy_d2h(a.ctypes.data_as(C.c_void_p), p, a.nbytes))
        return a

    def free(self):
        for p in self.held:
            self.check(self.L.mom6h_free(p))


# ------------------------------------------------------------- continuity --
def _continuity(n1, n2, nk, base, target):
    """Zonal pass on n2 rows that repeat the 8 rows of base; yields every output, one at a time."""
    d = _Device()
    L, check, cs = d.L, d.check, C.c_void_p()
    rows = _at(n2, 8)
    keep = [np.full((n2, n1), x) for x in (1.0 / (DX * DX), 1.0 / DX, DX, 1.0)]
    iarea, idx, dx, one = [_D(a) for a in keep]
    check(L.mom6h_continuity_init(C.byref(cs), *_bounds(n1, n2), nk, iarea, idx, dx, one, 0, dx, dx, one))
    del keep
    u, h = d.up(base["u"][:, rows]), d.up(base["h"][:, rows])
    uhbt = d.up(base["uhbt"][rows]) if target else C.c_void_p()
    out = {f: (d.zeros(nk, n2, n1), nk) for f in ("h", "uh", "u_cor", "h_u")}
    out.update({f: (d.zeros(n2, n1), 1) for f in ("EE", "E0", "W0", "WW", "uWW", "uEE", "du_cor")})
    bt = (C.c_void_p * 7)(*[out[f][0] for f in ("EE", "E0", "W0", "WW", "uWW", "uEE", "h_u")])
    check(L.mom6h_continuity_ppm(cs, u, h, out["h"][0], out["uh"][0], C.c_double(300.0), uhbt, C.byref(bt),
                                 out["u_cor"][0], out["du_cor"][0], 0, C.c_void_p()))
    check(L.mom6h_device_synchronize())
    for f, (q, k) in out.items():
        yield f, d.down(q, k, n2, n1)
    check(L.mom6h_continuity_end(cs))
    d.free()


@pytest.mark.parametrize("target", [False, True])
def test_zonal_continuity(target):
    n1, n2, nk = 8200, 8192, 3
    assert 8 * n1 * n2 * 8 >= 2 ** 32 > 8 * n1 * 14 * 8
    rng = np.random.default_rng(7)
    base = dict(u=0.05 * rng.standard_normal((nk, 8, n1)), h=4000.0 / nk + 0.5 * rng.standard_normal((nk, 8, n1)),
                uhbt=2.0e5 * rng.standard_normal((8, n1)))
    small = dict(_continuity(n1, 14, nk, base, target))
    reps = (n2 - 6) // 8
    for f, w in _continuity(n1, n2, nk, base, target):
        print(f"[gpu wide] continuity {n1}x{n2}x{nk} target={target}: {f}", flush=True)
        i = slice(3, n1 - 3) if f == "h" else slice(2, n1 - 3)
        s = small[f][:, 3:11, i]
        assert np.abs(s).max() > 0.0, f
        for k in range(w.shape[0]):
            got = w[k, 3:3 + 8 * reps].reshape(reps, 8, n1)[:, :, i]
            assert (got == s[k]).all(), (f, k)


def test_planes_of_4_gib():
    """Zonal and meridional pass of one layer whose plane alone passes 32-bit offsets."""
    n1, n2 = 23176, 23176
    assert n1 * n2 * 8 >= 2 ** 32
    rng = np.random.default_rng(7)
    base = dict(u=0.05 * rng.standard_normal((8, n1)), h=4000.0 + 0.5 * rng.standard_normal((8, n1)))

    def run(n2):
        d = _Device()
        L, check, cs = d.L, d.check, C.c_void_p()
        rows = _at(n2, 8)
        one = np.ones((n2, n1))   # every metric 1
        check(L.mom6h_continuity_init(C.byref(cs), *_bounds(n1, n2), 1, *[_D(one)] * 4, 0, *[_D(one)] * 3))
        check(L.mom6h_continuity_set_meridional(cs, *[_D(one)] * 5))
        del one
        print(f"[gpu wide] continuity {n1}x{n2}x1: set up", flush=True)
        u, h = d.up(base["u"][rows]), d.up(base["h"][rows])
        for axis, fn in (("x", L.mom6h_continuity_ppm), ("y", L.mom6h_continuity_ppm_y)):
            out = {axis + "h": d.zeros(n2, n1), axis + "flux": d.zeros(n2, n1)}
            check(fn(cs, u, h, *out.values(), C.c_double(0.5), C.c_void_p(), C.c_void_p(), C.c_void_p(), C.c_void_p(),
                     0, C.c_void_p()))
            check(L.mom6h_device_synchronize())
            for f, q in out.items():
                yield f, d.down(q, n2, n1)
        check(L.mom6h_continuity_end(cs))
        d.free()

    small = dict(run(14))
    reps = (n2 - 6) // 8
    for f, w in run(n2):
        print(f"[gpu wide] continuity {n1}x{n2}x1: {f}", flush=True)
        s = small[f][3:11, 3:n1 - 3]
        assert np.abs(s).max() > 0.0, f
        for q in range(reps):
            assert np.array_equal(w[3 + 8 * q:11 + 8 * q, 3:n1 - 3], s), (f, q)


# --------------------------------------------------------------- vert_visc --
def _vert_visc(n, nk, base, ray3d, keep):
    """Yields u, v, the kept coefficients and bottom stresses of a call on an n x n grid that repeats base's 8 x 8."""
    d = _Device()
    L, check, cs = d.L, d.check, C.c_void_p()
    at = _at(n, 8)
    wide = lambda f: base[f][..., at, :][..., at]  # noqa: E731
    mask = np.ascontiguousarray(wide("mask"))
    check(L.mom6h_vert_visc_init(C.byref(cs), *_bounds(n, n), nk, _D(mask), _D(mask),
                                 *[C.c_double(v) for v in (1e-4, 1e-2, 1e-2, 40.0, 10.0)]))
    check(L.mom6h_vert_visc_keep_coefficients(cs, int(keep)))
    p = [C.c_void_p() for _ in range(6)]
    check(L.mom6h_vert_visc_arrays(cs, *[C.byref(q) for q in p]))
    u, v, h, tau = d.up(wide("u")), d.up(wide("v")), d.up(wide("h")), d.up(wide("taux"))
    args = [cs, u, v, h, C.c_double(300.0), tau, tau]
    if ray3d:
        ray = d.up(wide("ray"))
        check(L.mom6h_vert_visc_ray3d(*args, ray, ray, C.c_void_p()))
    else:
        check(L.mom6h_vert_visc(*args, tau, tau, C.c_void_p()))
    check(L.mom6h_device_synchronize())
    out = [("u", u, nk), ("v", v, nk), ("taux_bot", p[4], 1), ("tauy_bot", p[5], 1)]
    if keep:
        out += [("a_u", p[0], nk + 1), ("a_v", p[1], nk + 1), ("h_u", p[2], nk), ("h_v", p[3], nk)]
    for f, q, k in out:
        yield f, d.down(q, k, n, n)
    check(L.mom6h_vert_visc_end(cs))
    d.free()


@pytest.mark.parametrize("ray3d,keep", [(False, False), (True, True)])
def test_vert_visc(ray3d, keep):
    n, nk = 5190, 5
    assert 20 * n * n * 8 >= 2 ** 32
    rng = np.random.default_rng(7)
    rnd = rng.standard_normal
    base = dict(u=0.05 * rnd((nk, 8, 8)), v=0.05 * rnd((nk, 8, 8)), h=20.0 + rnd((nk, 8, 8)), taux=0.1 * rnd((8, 8)),
                ray=1e-4 * np.abs(rnd((nk, 8, 8))), mask=(rnd((8, 8)) > -1.0).astype(float))
    small = dict(_vert_visc(14, nk, base, ray3d, keep))
    reps = (n - 6) // 8
    for f, w in _vert_visc(n, nk, base, ray3d, keep):
        print(f"[gpu wide] vert_visc {n}x{n}x{nk} ray3d={ray3d} keep={keep}: {f}", flush=True)
        s = small[f][:, 3:11, 3:11]
        assert np.abs(s).max() > 0.0, f
        for k in range(w.shape[0]):
            got = w[k, 3:3 + 8 * reps, 3:3 + 8 * reps].reshape(reps, 8, reps, 8)
            assert (got == s[k][:, None, :]).all(), (f, k)


# ---------------------------------------------------- models and ensembles --
class _Repeated(dict):
    """The 12 x 12 interior of a small case repeated over a grid, array by array as asked for."""

    def __init__(self, cfg, case):
        super().__init__(case)
        self.at = [3 + _at(n, 12) for n in (cfg.n1, cfg.n2)]

    def __getitem__(self, name):
        return np.asfortranarray(super().__getitem__(name)[self.at[0]][:, self.at[1]])


@pytest.mark.parametrize("form,ni,nk", [("mixed model", 5188, 4), ("mixed ensemble", 5188, 4), ("fp64 ensemble", 8200, 1)])
def test_steps(form, ni, nk):
    """One step; points at least 30 from the domain's edges (farther than a step of
    4 barotropic substeps reaches), where the reference's ranges break the pattern."""
    from hackathon_mom6_miniapp_amd.model import Ensemble, Model

    precision = form.split()[0]
    base_cfg = Config(ni=16, nj=16, nk=nk, bt_nsteps=4, dt=100.0, bc_x=BC_PERIODIC, bc_y=BC_PERIODIC,
                      coriolis="fplane", f0=1e-4, Kh=1e3, precision=precision)
    base = make_case(base_cfg, init="seeded", seed=5, bump=(0.5, 40.0e3))
    small_cfg, cfg = replace(base_cfg, ni=76, nj=76), replace(base_cfg, ni=ni, nj=ni)
    assert (ni - 4) % 12 == 0 and cfg.n1 ** 2 * 8 * (8 if precision == "fp64" else 20) >= 2 ** 32
    small_case, wide_case = _Repeated(small_cfg, base), _Repeated(cfg, base)
    small = Model(small_cfg, small_case)
    small.step(1)
    small.synchronize()
    print(f"[gpu wide] {form} {ni}x{ni}x{nk}: set up", flush=True)
    if form.endswith("model"):
        run = Model(cfg, wide_case)
        members = [run]
    else:
        run = Ensemble([small_cfg, cfg], [small_case, wide_case])
        members = run.members
    print(f"[gpu wide] {form} {ni}x{ni}x{nk}: step", flush=True)
    run.step(1)
    run.synchronize()
    for f in ("u", "v", "h", "up", "vp", "eta"):
        s = small.get(f)[39 - 6:39 + 6, 39 - 6:39 + 6]   # 30 .. 42 of 72
        s = np.roll(s, (6, 6), (0, 1)).reshape(12, 12, -1)
        assert np.abs(s).max() > 0.0, f
        for m in members:
            w = m.get(f)
            w = w.reshape(w.shape[0], w.shape[1], -1)
            reps = (w.shape[0] - 6) // 12 - 6
            for k in range(w.shape[2]):
                got = w[39:-39, 39:-39, k].T.reshape(reps, 12, reps, 12)
                assert (got == s[:, :, k].T[:, None, :]).all(), (f, k)
        print(f"[gpu wide] {form}: {f} agrees", flush=True)
    run.close()
    small.close()
