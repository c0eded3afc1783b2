"""The momentum tuner's choice, made right after set-up (the chip idle before),
is one of the fastest in a step: the momentum stage under it against every march
length, the candidates in turn, shortest of four times each.  8%: 1% that the
tuner grants the automatic length, 4% between launches timed back to back and
among a step's other kernels, 3% of noise (a wrong choice costs 13% here)."""
import pytest

from hackathon_mom6_miniapp_amd.state import BC_PERIODIC, BC_WALL, Config, make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_choice_is_among_the_fastest(precision):
    from hackathon_mom6_miniapp_amd.model import Model

    cfg = Config(ni=720, nj=720, nk=75, bt_nsteps=10, bc_x=BC_PERIODIC, bc_y=BC_WALL, coriolis="betaplane", f0=1e-4,
                 beta=2e-11, Kh=1e3, precision=precision)
    m = Model(cfg, make_case(cfg, init="seeded", seed=1, lazy3d=True))
    report = m.autotune(3)
    print(f"[gpu tuner] {precision} {report}", flush=True)
    chosen = report.rsplit(" ", 1)[1]
    lengths = {"128": (16, 1), "64": (8, 1), "32": (4, 1), "16": (4, 2), "8": (4, 4), "4": (4, 8)}
    best = {}
    m.set_option("serialize", 1)

    def momentum():
        m.set_option("profile", 1)
        m.step(2)
        m.synchronize()
        ms = m.stage_times()["momentum"] / 2
        m.set_option("profile", 0)
        return ms

    # the automatic length is timed as the tuner left it, before any option is set
    auto = [momentum() for _ in range(5)][1:] if chosen == "auto" else None
    for r in range(4):
        for name in (sorted(lengths) if r % 2 else sorted(lengths)[::-1]):
            m.set_option("momentum_tile", lengths[name][0])
            m.set_option("momentum_splits", lengths[name][1])
            best.setdefault(name, []).append(momentum())
    if auto:
        best["auto"] = auto
    best = {k: min(v) for k, v in best.items()}
    print(f"[gpu tuner] momentum ms per step: {best}, chosen {chosen}", flush=True)
    m.close()
    assert best[chosen] <= 1.08 * min(best.values()), (chosen, best)
