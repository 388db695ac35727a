"""The ion's chain looked ahead (shells chosen as at one energy, then checked
each at its own).  In FP64 its events equal the oracle's, for fast ions, where
nearly all choices hold, and for slow light ones that lose much of their
energy in 64 collisions or leave the energy grid; with a constant hole mass
and with masses from the density of states.  On both paths they equal those
of the chain taken collision by collision, which a batch runs for what an ion
has left after its first round."""
import pytest

import trekis_gpu as tg
from trekis_gpu import abi
from trekis_gpu.batch import Batch, IonContext
from oracle import Oracle

from gpu_helpers import first_mismatch, say, sort_trace

pytestmark = pytest.mark.gpu


# target, ion (Z, mass), MeV/u; the last two end inside the layer or are slow
# enough for the shells' shares to change along the track
@pytest.mark.parametrize("name,Z,M,E", [("test", 8, 16.0, 1.0), ("test_metal", 8, 16.0, 1.0), ("test_sio2", 18, 39.95, 2.0),
                                        ("test", 2, 4.0026, 0.08), ("test_metal", 3, 6.94, 0.06)])
def test_chain_equals_the_oracle(name, Z, M, E):
    mat, ion, opt, run = tg.config_material(name)
    mat.prepare(tg.load_library())
    ion.Zat, ion.Mass, ion.E = Z, M, E * 1e6 * M
    ctx = tg.Context(mat, ion, opt)
    ctx.build_tables()
    R, V = tg.radial_grid(20, run["Rmin"], run["Rmax"], mat.layer)
    g = ctx.run_mc(2, run["seed"], R, V, trace_cap=1_000_000)
    say(f"[chain] {name} Z {Z} {E} MeV/u: events {g.n_events.tolist()}")
    orc = Oracle(mat, ion, opt)
    orc.inject_from(ctx)
    c = orc.run_mc(2, run["seed"], R, V, tg.TallySet(orc.Nt, len(R), mat), trace_cap=1_000_000)
    assert g.trace_total == len(c.trace) and (g.n_events == c.n_events).all()
    assert first_mismatch(sort_trace(g.trace), sort_trace(c.trace)) is None


# an ion of ~2100 collisions: 1024 or 1500 of them in the first round (a quarter
# of the list), the others one by one
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("capacity", [4096, 6000])
def test_chain_equals_one_by_one(precision, capacity):
    mat, ion, opt, run = tg.config_material("test_sio2")
    mat.prepare(tg.load_library())
    opt.precision = precision
    ctx = tg.Context(mat, ion, opt)
    ctx.build_tables()
    R, V = tg.radial_grid(20, run["Rmin"], run["Rmax"], mat.layer)
    ahead = ctx.run_mc(1, run["seed"], R, V, trace_cap=500_000)
    assert ahead.n_events[abi.EVENT_NAMES.index("shi")] > 1600
    c = IonContext(ctx, ion)
    c.build_tables()
    b = Batch([c], R, V, capacity=capacity)
    b.run(run["seed"], 0, trace_cap=500_000)
    assert b.trace_total == ahead.trace_total
    assert first_mismatch(sort_trace(ahead.trace), sort_trace(b.trace)) is None
