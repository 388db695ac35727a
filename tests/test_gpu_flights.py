"""Snapshot tallies of flights that cross many time nodes (a wave tallies a
long flight together, 64 nodes at a time; a lane its own short ones) and of
rounds with few particles (spread one or a few to a wave): the events and
tallies equal the oracle's on time steps from one node per several flights to
hundreds of nodes per flight, on fine and coarse radial grids."""
import pytest

import trekis_gpu as tg
from trekis_gpu import abi
from oracle import Oracle

from gpu_helpers import compare_tallies, first_mismatch, say, sort_trace

pytestmark = pytest.mark.gpu


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
