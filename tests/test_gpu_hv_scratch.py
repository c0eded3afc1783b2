"""The biharmonic operator holds its two 3D work fields only where the general
kernels run: a constant-metric grid allocates neither (the march keeps Del2 in
registers) until the option "general" asks for those kernels, which then give the
same tendencies, also in a step captured as a graph; a grid whose biharmonic or
closure metrics vary allocates them with the metrics."""
import ctypes as C

import numpy as np
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, BC_WALL, Config, make_case

pytestmark = pytest.mark.gpu


def _free():
    hip = C.CDLL("libamdhip64.so")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("vary", ["nothing", "biharmonic", "closure"])
def test_work_fields_where_needed(vary):
    from hackathon_mom6_miniapp_amd._lib import check, lib

    cfg = Config(ni=318, nj=254, nk=100, bt_nsteps=4, bc_x=BC_PERIODIC, bc_y=BC_WALL)
    L, cs, dx = lib(), C.c_void_p(), cfg.dx_km * 1000.0
    shape, field = (cfg.n1, cfg.n2), 8 * cfg.n1 * cfg.n2 * cfg.nk   # 65.5 MB per 3D field
    D = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
    full = lambda x: np.full(shape, x, order="F")  # noqa: E731
    wave = 1.0 + 0.1 * np.sin(np.arange(cfg.n1))[:, None]
    unit, idx, iarea, area = full(1.0), full(1.0 / dx), full(1.0 / dx ** 2), full(dx ** 2)
    i3 = np.asfortranarray(full(dx ** -3) * (wave if vary == "biharmonic" else 1.0))
    aT = np.asfortranarray(area * (wave if vary == "closure" else 1.0))
    check(L.mom6h_hor_visc_init(C.byref(cs), *cfg.bounds, cfg.nk, C.c_double(20.0), C.c_double(1e-3),
                                *[D(a) for a in [unit] * 4 + [idx] * 4 + [iarea] * 2 + [unit] * 4 + [area] * 4]))
    before = _free()
    check(L.mom6h_hor_visc_set_options(cs, 1, 1, C.c_double(1e9), 0, *[D(i3)] * 4))
    check(L.mom6h_hor_visc_set_closures(cs, 1, 0, 0, D(aT), None, None, None, None))
    used = before - _free()
    print(f"[gpu hv scratch] {vary}: {used / 1e6:.1f} MB", flush=True)
    if vary == "nothing":
        assert used < field
    else:
        assert used >= 2 * field
    check(L.mom6h_hor_visc_end(cs))


@pytest.mark.parametrize("graph", [False, True])
def test_general_kernels_after_the_march(graph):
    from hackathon_mom6_miniapp_amd.model import Model

    cfg = Config(ni=40, nj=26, nk=3, bt_nsteps=4, bc_x=BC_PERIODIC, bc_y=BC_WALL, coriolis="betaplane", f0=1e-4,
                 beta=2e-11, Kh=20.0, biharmonic=True, Ah=1e9)
    case = make_case(cfg, init="seeded", seed=6)
    want, got = Model(cfg, case), Model(cfg, case, graph=graph)
    for m in (want, got):
        m.set_option("fused", 0)
    for q in range(4):
        got.set_option("general", q % 2)
        for m in (want, got):
            m.step(1)
            m.synchronize()
        for f in ("diffu", "diffv", "u", "v", "h"):
            assert np.array_equal(got.get(f), want.get(f)), (q, f)
    want.close()
    got.close()
