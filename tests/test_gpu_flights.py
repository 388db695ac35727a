"""Snapshot tallies of flights that cross many time nodes (a wave tallies a
long flight together, 64 nodes at a time; a lane its own short ones) and of
rounds with few particles (spread one or a few to a wave): the events and
tallies equal the oracle's on time steps from one node per several flights to
hundreds of nodes per flight, on fine and coarse radial grids."""
import numpy as np
import pytest

import trekis_gpu as tg
from trekis_gpu import abi
from trekis_gpu.batch import Batch, IonContext
from oracle import Oracle

from gpu_helpers import compare_tallies, first_mismatch, say, sort_trace

pytestmark = pytest.mark.gpu

SPECTRA = ("Out_Ee_vs_E", "Out_Eh_vs_E", "Out_theta", "Out_theta_h", "Out_Ne_Em", "Out_E_Em", "Out_Ee_vs_E_Em")


# flights of the test target's slow electrons and holes last ~0.2-2 fs: steps
# that give none or one node, about 4 (the limit between lane and wave), about
# 64 and several times 64; 1 and 3 bins (the last bin is open), 40 fine ones
@pytest.mark.parametrize("name,Tim,dt,NR", [("test", 60.0, 1.0, 3), ("test", 40.0, 0.25, 40), ("test", 12.0, 0.02, 40),
                                            ("test", 5.0, 0.004, 3), ("test_metal", 20.0, 0.05, 40)])
def test_flights_over_many_nodes(name, Tim, dt, NR):
    lib = tg.load_library()
    mat, ion, opt, run = tg.config_material(name)
    mat.prepare(lib)
    opt.Tim, opt.dt = Tim, dt
    ctx = tg.Context(mat, ion, opt)
    ctx.build_tables()
    orc = Oracle(mat, ion, opt)
    orc.inject_from(ctx)
    R, V = tg.radial_grid(NR, run["Rmin"], run["Rmax"], mat.layer)
    g = ctx.run_mc(1, run["seed"], R, V, trace_cap=500_000)
    c = orc.run_mc(1, run["seed"], R, V, tg.TallySet(orc.Nt, len(R), mat), trace_cap=500_000)
    say(f"[flights] {name} dt {dt}: {ctx.Nt} nodes, events {g.n_events.tolist()}")
    assert (g.n_events == c.n_events).all()
    assert first_mismatch(sort_trace(g.trace), sort_trace(c.trace)) is None
    assert not compare_tallies(g, c)


# The same histories on a grid whose nodes lie 2 fs apart, where lanes tally
# nearly every flight alone, and on one of 1/64 or 1/256 fs, where waves tally
# them: at the nodes that both have (sums of powers of two, so equal times)
# every tally is the same, bit for bit.  Three iterations, with the
# per-iteration spectra, and the three as impacts of a batch.
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name,ratio", [("test", 128), ("test_metal", 128), ("test_sio2", 512)])
def test_fine_and_coarse_nodes_agree(name, ratio, precision):
    lib = tg.load_library()
    out = []
    for dt in (2.0, 2.0 / ratio):
        mat, ion, opt, run = tg.config_material(name)
        mat.prepare(lib)
        opt.Tim, opt.dt, opt.precision = 16.0, dt, precision
        ctx = tg.Context(mat, ion, opt)
        ctx.build_tables()
        R, V = tg.radial_grid(40, run["Rmin"], run["Rmax"], mat.layer)
        t = ctx.run_mc(3, run["seed"], R, V, first_iter=5)
        c = IonContext(ctx, ion)
        c.build_tables()
        b = Batch([c, c, c], R, V, capacity=1 << 20)
        out.append((t, b.run(run["seed"], 5), ctx.Nt))
    (a, ab, na), (f, fb, nf) = out
    say(f"[flights] {name} precision {precision}: {na} and {nf} nodes, events {a.n_events.tolist()}")
    assert na == 8 and nf == na * ratio and (a.n_events == f.n_events).all()
    nodes = np.arange(1, na + 1) * ratio - 1
    skip = ("Out_Elat", "Out_diff_coeff")        # per node interval, a recurrence over the nodes
    for k in a.arrays:
        if k in skip:
            continue
        x, y = a[k], f[k]
        assert np.array_equal(x[:na], y[nodes]), k
        if k in SPECTRA:
            continue
        for xb, yb in zip(ab, fb):
            assert np.array_equal(xb[k], yb[k][nodes]), k
    assert a["Out_ne"].sum() > 0 and a["Out_E_at"][-1] > 0
