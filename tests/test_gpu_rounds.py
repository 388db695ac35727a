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
