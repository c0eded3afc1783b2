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


def _host(n1, n2, value):
    a = np.full((n2, n1), value)
    return a, a.ctypes.data_as(C.POINTER(C.c_double))


def _ptr(t):
    return C.c_void_p(t.data_ptr()) if t is not None else C.c_void_p()


# ------------------------------------------------------------- continuity --
def _continuity(n1, n2, nk, base, target):
    """Zonal pass on n2 rows that repeat the 8 rows of base; every output."""
    import torch

    from hackathon_mom6_miniapp_amd._lib import check, lib

    rows = torch.as_tensor(_at(n2, 8), device="cuda")
    u, h = (base[f][:, rows, :].contiguous() for f in ("u", "h"))
    uhbt = base["uhbt"][rows].contiguous() if target else None
    L, cs = lib(), C.c_void_p()
    keep = [_host(n1, n2, x) for x in (1.0 / (DX * DX), 1.0 / DX, DX, 1.0)]
    iarea, idx, dx, one = [p for _, p in keep]
    check(L.mom6h_continuity_init(C.byref(cs), *_bounds(n1, n2), nk, iarea, idx, dx, one, 0, dx, dx, one))
    del keep
    out = {f: torch.zeros(nk, n2, n1, dtype=torch.float64, device="cuda") for f in ("h", "uh", "u_cor", "h_u")}
    for f in ("EE", "E0", "W0", "WW", "uWW", "uEE", "du_cor"):
        out[f] = torch.zeros(1, n2, n1, dtype=torch.float64, device="cuda")
    bt = (C.c_void_p * 7)(*[out[f].data_ptr() for f in ("EE", "E0", "W0", "WW", "uWW", "uEE", "h_u")])
    torch.cuda.synchronize()
    check(L.mom6h_continuity_ppm(cs, _ptr(u), _ptr(h), _ptr(out["h"]), _ptr(out["uh"]), C.c_double(300.0), _ptr(uhbt),
                                 C.byref(bt), _ptr(out["u_cor"]), _ptr(out["du_cor"]), 0, C.c_void_p()))
    check(L.mom6h_device_synchronize())
    check(L.mom6h_continuity_end(cs))
    return out


@pytest.mark.parametrize("target", [False, True])
def test_zonal_continuity(target):
    import torch

    n1, n2, nk = 8200, 8192, 5
    assert 8 * n1 * n2 * 8 >= 2 ** 32 > 8 * n1 * 14 * 8
    g = torch.Generator(device="cuda").manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64, device="cuda")  # noqa: E731
    base = dict(u=0.05 * rnd(nk, 8, n1), h=4000.0 / nk + 0.5 * rnd(nk, 8, n1), uhbt=2.0e5 * rnd(8, n1))
    small = _continuity(n1, 14, nk, base, target)
    print(f"[gpu wide] continuity {n1}x{n2}x{nk} target={target}", flush=True)
    wide = _continuity(n1, n2, nk, base, target)
    reps = (n2 - 6) // 8
    for f, w in wide.items():
        i = slice(3, n1 - 3) if f == "h" else slice(2, n1 - 3)
        s = small[f][:, 3:11, i]
        assert s.abs().max() > 0.0, f
        for k in range(w.shape[0]):
            got = w[k, 3:3 + 8 * reps, i].reshape(reps, 8, -1)
            assert bool((got == s[k]).all()), (f, k)


def test_planes_of_4_gib():
    """Zonal and meridional pass of one layer whose plane alone passes 32-bit offsets."""
    import torch

    from hackathon_mom6_miniapp_amd._lib import check, lib

    n1, n2 = 23176, 23176
    assert n1 * n2 * 8 >= 2 ** 32
    g = torch.Generator(device="cuda").manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64, device="cuda")  # noqa: E731
    base = dict(u=0.05 * rnd(8, n1), h=4000.0 + 0.5 * rnd(8, n1))

    def run(n2):
        rows = torch.as_tensor(_at(n2, 8), device="cuda")
        u, h = (base[f][rows].contiguous() for f in ("u", "h"))
        L, cs = lib(), C.c_void_p()
        keep, one = _host(n1, n2, 1.0)   # every metric 1
        check(L.mom6h_continuity_init(C.byref(cs), *_bounds(n1, n2), 1, *[one] * 4, 0, *[one] * 3))
        check(L.mom6h_continuity_set_meridional(cs, *[one] * 5))
        out = {f: torch.zeros(n2, n1, dtype=torch.float64, device="cuda") for f in ("hx", "uh", "hy", "vh")}
        torch.cuda.synchronize()
        for fn, x, t in ((L.mom6h_continuity_ppm, "hx", "uh"), (L.mom6h_continuity_ppm_y, "hy", "vh")):
            check(fn(cs, _ptr(u), _ptr(h), _ptr(out[x]), _ptr(out[t]), C.c_double(0.5), C.c_void_p(), C.c_void_p(),
                     C.c_void_p(), C.c_void_p(), 0, C.c_void_p()))
        check(L.mom6h_device_synchronize())
        check(L.mom6h_continuity_end(cs))
        return out

    small = run(14)
    print(f"[gpu wide] continuity {n1}x{n2}x1", flush=True)
    wide = run(n2)
    reps = (n2 - 6) // 8
    for f, w in wide.items():
        s = small[f][3:11, 3:n1 - 3]
        assert s.abs().max() > 0.0, f
        got = w[3:3 + 8 * reps, 3:n1 - 3]
        for q in range(0, reps, 64):
            part = got[8 * q:8 * (q + 64)]
            assert bool((part.reshape(part.shape[0] // 8, 8, -1) == s).all()), (f, q)


# --------------------------------------------------------------- vert_visc --
def _vert_visc(n, nk, base, ray3d, keep):
    """u, v and the kept coefficients of a call on an n x n grid that repeats the 8 x 8 pattern of base."""
    import torch

    from hackathon_mom6_miniapp_amd._lib import check, lib

    at = torch.as_tensor(_at(n, 8), device="cuda")
    x = {f: a[..., at, :][..., at].contiguous() for f, a in base.items()}
    L, cs = lib(), C.c_void_p()
    mask = x["mask"].cpu().numpy()
    m = mask.ctypes.data_as(C.POINTER(C.c_double))
    check(L.mom6h_vert_visc_init(C.byref(cs), *_bounds(n, n), nk, m, m, *[C.c_double(v) for v in
                                                                          (1e-4, 1e-2, 1e-2, 40.0, 10.0)]))
    check(L.mom6h_vert_visc_keep_coefficients(cs, int(keep)))
    p = [C.c_void_p() for _ in range(6)]
    check(L.mom6h_vert_visc_arrays(cs, *[C.byref(q) for q in p]))
    torch.cuda.synchronize()
    args = [cs, _ptr(x["u"]), _ptr(x["v"]), _ptr(x["h"]), C.c_double(300.0), _ptr(x["taux"]), _ptr(x["taux"])]
    if ray3d:
        check(L.mom6h_vert_visc_ray3d(*args, _ptr(x["ray"]), _ptr(x["ray"]), C.c_void_p()))
    else:
        check(L.mom6h_vert_visc(*args, _ptr(x["taux"]), _ptr(x["taux"]), C.c_void_p()))
    check(L.mom6h_device_synchronize())
    out = dict(u=x["u"], v=x["v"])
    for f, q, k in zip(("a_u", "a_v", "h_u", "h_v", "taux_bot", "tauy_bot"), p, (nk + 1, nk + 1, nk, nk, 1, 1)):
        if keep or k == 1:
            out[f] = torch.empty(k, n, n, dtype=torch.float64, device="cuda")
            check(L.mom6h_memcpy_d2d(_ptr(out[f]), q, out[f].numel() * 8))
    check(L.mom6h_device_synchronize())
    check(L.mom6h_vert_visc_end(cs))
    return out


@pytest.mark.parametrize("ray3d,keep", [(False, False), (False, True), (True, True)])
def test_vert_visc(ray3d, keep):
    import torch

    n, nk = 5190, 9
    assert 20 * n * n * 8 >= 2 ** 32
    g = torch.Generator(device="cuda").manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64, device="cuda")  # noqa: E731
    base = dict(u=0.05 * rnd(nk, 8, 8), v=0.05 * rnd(nk, 8, 8), h=20.0 + rnd(nk, 8, 8), taux=0.1 * rnd(8, 8),
                ray=1e-4 * rnd(nk, 8, 8).abs(), mask=(rnd(8, 8) > -1.0).double())
    small = _vert_visc(14, nk, base, ray3d, keep)
    print(f"[gpu wide] vert_visc {n}x{n}x{nk} ray3d={ray3d} keep={keep}", flush=True)
    wide = _vert_visc(n, nk, base, ray3d, keep)
    reps = (n - 6) // 8
    for f, w in wide.items():
        s = small[f][:, 3:11, 3:11]
        assert s.abs().max() > 0.0, f
        for k in range(w.shape[0]):
            got = w[k, 3:3 + 8 * reps, 3:3 + 8 * reps].reshape(reps, 8, reps, 8)
            assert bool((got == s[k][:, None, :]).all()), (f, k)


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
