"""What a batch keeps from one run to the next: after a run that fails there
are no tallies to fetch, and a later good run gives its own again."""
import numpy as np
import pytest

import trekis_gpu as tg
from trekis_gpu.batch import Batch, IonContext

from gpu_helpers import say

pytestmark = pytest.mark.gpu


def _impact(name, ion_of=None):
    """(ion context, run values) on a target; ion_of: (Z, mass, MeV/u)"""
    mat, ion, opt, run = tg.config_material(name)
    mat.prepare(tg.load_library())
    ctx = tg.Context(mat, ion, opt)
    ctx.build_tables()
    if ion_of:
        Z, M, E = ion_of
        ion.Zat, ion.Mass, ion.E = Z, M, E * 1e6 * M
    c = IonContext(ctx, ion)
    c.build_tables()
    return c, run


def test_no_tallies_after_a_failed_run():
    # 2150 collisions of uranium in the metal: lists of 1500 hold the particles
    # of the one seed's history and not of the other's
    c, run = _impact("test_metal", (92, 238.03, 1.0))
    R, V = tg.radial_grid(30, run["Rmin"], run["Rmax"], 100.0)
    b = Batch([c], R, V, capacity=1500)
    good, full = 7, run["seed"]
    (a,) = b.run(good, 0)
    with pytest.raises(tg.TrekisError, match="capacity"):
        b.run(full, 0)
    say("[batch state] a failed run after a good one")
    with pytest.raises(tg.TrekisError, match="must run before"):
        b.fetch()
    b.run(good, 0, with_tallies=False)
    (f,) = b.fetch()
    for k in a.arrays:
        assert np.array_equal(a[k], f[k]), k


def test_round_budget_is_each_groups_own():
    # oxygen in the oxide (480 collisions, held to the round budget by lists of
    # 1200) beside lithium in the metal (run on, its rounds may be short): the
    # oxide's rounds are those it takes alone, whichever material comes first
    a, _ = _impact("test_metal", (3, 6.94, 0.5))
    b, run = _impact("test")
    R, V = tg.radial_grid(30, run["Rmin"], run["Rmax"], 100.0)
    rounds = []
    for impacts, first in (([b], 1), ([b, a], 1), ([a, b], 0)):       # the oxide's impact is iteration 1
        batch = Batch(impacts, R, V, capacity=1200)
        batch.run(run["seed"], first)
        rounds.append(batch.timing()[2])
    say(f"[batch state] rounds alone, first, second: {rounds}")
    assert rounds[0] == rounds[1] == rounds[2], rounds


def test_batches_on_two_host_threads():
    import threading
    impacts = [_impact("test"), _impact("test_metal", (10, 20.18, 0.4))]
    R, V = tg.radial_grid(30, 1.0, 300.0, 100.0)
    batches = [Batch([c, c], R, V, capacity=1 << 18) for c, _ in impacts]
    alone = [b.run(run["seed"], 0) for b, (_, run) in zip(batches, impacts)]
    got = [[], []]

    def work(i):
        for _ in range(4):
            got[i].append(batches[i].run(impacts[i][1]["seed"], 0))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    say("[batch state] two batches, four runs each, side by side")
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for want, runs in zip(alone, got):
        assert len(runs) == 4
        for tallies in runs:
            for x, y in zip(want, tallies):
                for k in x.arrays:
                    assert np.array_equal(x[k], y[k]), k
