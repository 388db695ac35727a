"""Rounds of different budgets: with long lists a round of few particles ends
after fewer events per particle, with lists so short that the ions are held to
the round budget it does not.  Events and tallies are the same, single runs
and batches."""
import numpy as np
import pytest

import trekis_gpu as tg
from trekis_gpu.batch import Batch, IonContext

from gpu_helpers import first_mismatch, say, sort_trace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", ["test", "test_metal"])
def test_round_budget_changes_nothing(name, precision):
    out = []
    for capacity in (1 << 20, 2040):         # 2040 / 4 pairs of one ion a round: held to 512
        mat, ion, opt, run = tg.config_material(name)
        mat.prepare(tg.load_library())
        opt.precision, opt.gen_capacity = precision, capacity
        ctx = tg.Context(mat, ion, opt)
        ctx.build_tables()
        R, V = tg.radial_grid(30, run["Rmin"], run["Rmax"], mat.layer)
        t = ctx.run_mc(1, run["seed"], R, V, trace_cap=500_000)
        c = IonContext(ctx, ion)
        c.build_tables()
        b = Batch([c], R, V, capacity=capacity)
        b.run(run["seed"], 0, trace_cap=500_000)
        say(f"[rounds] {name} capacity {capacity}: events {t.n_events.tolist()}")
        out.append((t, sort_trace(t.trace), sort_trace(b.trace)))
    (a, ta, ba), (c, tc, bc) = out
    assert (a.n_events == c.n_events).all()
    for k in a.arrays:
        assert np.array_equal(a[k], c[k]), k
    for x in (tc, ba, bc):
        assert len(x) == len(ta) and first_mismatch(ta, x) is None


# The ion's collisions exceed a quarter of the short list by half and more, so
# it is held there and its rounds keep their 512 events, whatever the last
# digits of its path: oxygen in the oxide (480 collisions, the rounds differ by
# the budget alone), uranium in the metal and in the SiO2-like target.
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name,ion_of,capacity", [("test", None, 1200), ("test_metal", (92, 238.03, 1.0), 2040),
                                                  ("test_sio2", (92, 238.03, 1.0), 1500)])
def test_held_ions_keep_long_rounds(name, ion_of, capacity, precision):
    out = []
    for cap in (1 << 20, capacity):
        mat, ion, opt, run = tg.config_material(name)
        mat.prepare(tg.load_library())
        if ion_of:
            Z, M, E = ion_of
            ion.Zat, ion.Mass, ion.E = Z, M, E * 1e6 * M
        opt.precision, opt.gen_capacity = precision, cap
        ctx = tg.Context(mat, ion, opt)
        ctx.build_tables()
        R, V = tg.radial_grid(30, run["Rmin"], run["Rmax"], mat.layer)
        t = ctx.run_mc(1, run["seed"], R, V, trace_cap=500_000)
        c = IonContext(ctx, ion)
        c.build_tables()
        b = Batch([c], R, V, capacity=cap)
        (tb,) = b.run(run["seed"], 0, trace_cap=500_000)
        launches, rounds = ctx.timing()[2], b.timing()[2]
        say(f"[rounds] {name} capacity {cap}: {t.n_events[0]} collisions, {launches} launches, batch {rounds} rounds")
        out.append((t, tb, sort_trace(t.trace), sort_trace(b.trace), launches, rounds))
    (a, ab, ta, ba, la, ra), (c, cb, tc, bc, lc, rc) = out
    assert a.n_events[0] > 1.5 * (capacity / 4)
    assert la != lc and ra != rc
    assert (a.n_events == c.n_events).all()
    for k in a.arrays:
        assert np.array_equal(a[k], c[k]) and np.array_equal(ab[k], cb[k]), k
    for x in (tc, ba, bc):
        assert len(x) == len(ta) and first_mismatch(ta, x) is None
