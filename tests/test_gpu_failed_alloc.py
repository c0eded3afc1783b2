"""An allocation that fails is reported by the call that asked for it, and not once
more by the next call that launches a kernel."""
import ctypes as C

import numpy as np
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, BC_WALL, Config, make_case

pytestmark = pytest.mark.gpu


def _hor_visc(cfg):
    """hor_visc on constant metrics (its byte masks are formed on the device)."""
    from hackathon_mom6_miniapp_amd._lib import lib

    cs, dx = C.c_void_p(), cfg.dx_km * 1000.0
    full = lambda x: np.full((cfg.n1, cfg.n2), x, order="F")  # noqa: E731
    unit, idx, iarea, area = full(1.0), full(1.0 / dx), full(dx ** -2), full(dx ** 2)
    rc = lib().mom6h_hor_visc_init(C.byref(cs), *cfg.bounds, cfg.nk, C.c_double(20.0), C.c_double(1e-3),
                                   *[a.ctypes.data_as(C.POINTER(C.c_double)) for a in
                                     [unit] * 4 + [idx] * 4 + [iarea] * 2 + [unit] * 4 + [area] * 4])
    return rc, cs


@pytest.mark.parametrize("failing", ["malloc", "fields"])
def test_next_call_succeeds(failing):
    from hackathon_mom6_miniapp_amd._lib import lib
    from hackathon_mom6_miniapp_amd.model import Model

    small = Config(ni=40, nj=26, nk=3, bt_nsteps=4, bc_x=BC_PERIODIC, bc_y=BC_WALL)
    case = make_case(small, init="seeded", seed=6)
    model, want = Model(small, case), Model(small, case)
    for m in (model, want):
        m.step(1)
        m.synchronize()
    want.step(1)
    want.synchronize()
    if failing == "malloc":
        p = C.c_void_p()
        assert lib().mom6h_malloc(C.byref(p), C.c_size_t(1 << 41)) != 0   # 2 TiB
    else:                                      # the work fields of a wide, deep grid: 1.6 TB each
        wide = Config(ni=2000, nj=2000, nk=50000, bt_nsteps=4, bc_x=BC_PERIODIC, bc_y=BC_WALL)
        rc, big = _hor_visc(wide)
        assert rc == 0
        i3 = np.full((wide.n1, wide.n2), 1e-12, order="F")
        i3[3, 3] *= 1.01                       # varying metrics: the general kernels
        d = i3.ctypes.data_as(C.POINTER(C.c_double))
        assert lib().mom6h_hor_visc_set_options(big, 1, 1, C.c_double(1e9), 0, *[d] * 4) != 0
        lib().mom6h_hor_visc_end(big)
    rc, cs = _hor_visc(small)
    assert rc == 0, lib().mom6h_last_error()
    lib().mom6h_hor_visc_end(cs)
    if failing == "malloc":
        assert lib().mom6h_malloc(C.byref(p), C.c_size_t(1 << 41)) != 0
    model.step(1)
    model.synchronize()
    for f in ("u", "v", "h"):
        assert np.array_equal(model.get(f), want.get(f)), f
    model.close()
    want.close()
