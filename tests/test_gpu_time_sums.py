"""The running sums of the tallies along time, and their way to the caller's
arrays.  Sixteen waves of a workgroup share the time nodes of 64 columns:
fewer nodes than waves, as many, one more, a last piece that is short or
empty; 2, 64, 65 and more radial bins.  Tallies equal the
oracle's."""
import pytest

import trekis_gpu as tg
from oracle import Oracle

from gpu_helpers import compare_tallies, say

pytestmark = pytest.mark.gpu

_ORC = {}


def _pair(Tim, dt):
    if (Tim, dt) not in _ORC:
        mat, ion, opt, run = tg.config_material("test")
        mat.prepare(tg.load_library())
        opt.Tim, opt.dt = Tim, dt
        ctx = tg.Context(mat, ion, opt)
        ctx.build_tables()
        orc = Oracle(mat, ion, opt)
        orc.inject_from(ctx)
        _ORC[Tim, dt] = (ctx, orc, mat, run)
    return _ORC[Tim, dt]


@pytest.mark.parametrize("NR", [2, 3, 64, 65, 130])
@pytest.mark.parametrize("Tim,dt", [(3.0, 1.0), (15.0, 1.0), (16.0, 1.0), (33.0, 1.0), (64.0, 0.5)])
def test_sums_over_time(Tim, dt, NR):
    ctx, orc, mat, run = _pair(Tim, dt)
    say(f"[sums] {ctx.Nt} nodes, {NR} bins")
    R, V = tg.radial_grid(NR, run["Rmin"], run["Rmax"], mat.layer)
    g = ctx.run_mc(1, run["seed"], R, V)
    c = orc.run_mc(1, run["seed"], R, V, tg.TallySet(orc.Nt, len(R), mat))
    assert (g.n_events == c.n_events).all()
    assert not compare_tallies(g, c)
