"""Lists that overflow while the ions run on beyond the round budget and hold
the run with the ions kept to it: the second attempt gives the events, traces
and tallies of a run with long lists, bit for bit, and later runs of as much
work do not make the first attempt again.  Single runs, runs without
allocation and batches."""
import numpy as np
import pytest

import trekis_gpu as tg
from trekis_gpu.batch import Batch, IonContext

from gpu_helpers import first_mismatch, say, sort_trace

pytestmark = pytest.mark.gpu

# 4500 collisions of uranium in the metal.  With a cut-off of 4 eV its
# electrons take several hundred events each: rounds of 128 events keep more of
# them waiting than lists of 3300 hold, rounds of 512 do not.
CAPACITY = 3300


def _context(precision, capacity):
    mat, ion, opt, run = tg.config_material("test_metal")
    mat.layer, mat.cut_off = 100.0, 4.0
    mat.prepare(tg.load_library())
    ion.Zat, ion.Mass, ion.E = 92, 238.03, 1e6 * 238.03
    opt.precision, opt.gen_capacity = precision, capacity
    ctx = tg.Context(mat, ion, opt)
    ctx.build_tables()
    R, V = tg.radial_grid(30, run["Rmin"], run["Rmax"], mat.layer)
    return ctx, ion, run, R, V


def _attempts(capfd):
    """Transports of the first batch of iterations since the last call."""
    return capfd.readouterr().err.count("batch 0 round 1:")


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("precision", [0, 1])
def test_second_attempt_of_a_run(precision, noalloc, capfd, monkeypatch):
    long, _, run, R, V = _context(precision, 1 << 20)
    ctx, *_ = _context(precision, CAPACITY)
    monkeypatch.setenv("TRK_VERBOSE", "1")
    kw = {"noalloc": True} if noalloc else {"trace_cap": 500_000}
    for seed, attempts in ((run["seed"], 2), (7, 1), (run["seed"], 1)):
        a = long.run_mc(1, seed, R, V, trace_cap=500_000)
        assert _attempts(capfd) == 1
        t = ctx.run_mc(1, seed, R, V, **kw)
        n = _attempts(capfd)
        say(f"[overflow] precision {precision} noalloc {noalloc}: {n} attempts, events {t.n_events.tolist()}")
        assert n == attempts
        assert (t.n_events == a.n_events).all()
        for k in a.arrays:
            assert np.array_equal(a[k], t[k]), k
        if not noalloc:
            assert t.trace_total == a.trace_total == len(a.trace)
            assert first_mismatch(sort_trace(a.trace), sort_trace(t.trace)) is None


@pytest.mark.parametrize("precision", [0, 1])
def test_second_attempt_of_a_batch(precision):
    ctx, ion, run, R, V = _context(precision, 1 << 20)
    c = IonContext(ctx, ion)
    c.build_tables()
    long, short = Batch([c], R, V, capacity=1 << 20), Batch([c], R, V, capacity=CAPACITY)
    for seed in (run["seed"], 7):
        (a,) = long.run(seed, 0, trace_cap=500_000)
        (t,) = short.run(seed, 0, trace_cap=500_000)
        say(f"[overflow] batch, precision {precision}: rounds {long.timing()[2]} and {short.timing()[2]}")
        assert (long.timing()[1] == short.timing()[1]).all()
        assert long.trace_total == short.trace_total
        assert first_mismatch(sort_trace(long.trace), sort_trace(short.trace)) is None
        for k in a.arrays:
            assert np.array_equal(a[k], t[k]), k
