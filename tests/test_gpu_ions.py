"""The ion kernel (one wave per ion, 64 collisions at a time): wherever an
ion's chain is cut -- by the collisions it may take in one round, which follow
from the list capacity, or by its end -- the events and tallies are those of
an uncut chain, bit for bit.  (Its events against the oracle's are
test_gpu_parity.test_mc_replay_bitwise.)"""
import numpy as np
import pytest

import trekis_gpu as tg
from trekis_gpu import abi

pytestmark = pytest.mark.gpu

_BASE = {}


def _run(precision, capacity):
    lib = tg.load_library()
    mat, ion, opt, run = tg.config_material("test_sio2")     # ~2100 collisions per ion
    mat.prepare(lib)
    opt.precision, opt.gen_capacity = precision, capacity
    ctx = tg.Context(mat, ion, opt)
    ctx.build_tables()
    R, V = tg.radial_grid(run["NR"], run["Rmin"], run["Rmax"], mat.layer)
    t = ctx.run_mc(2, run["seed"], R, V, trace_cap=500_000)
    return t


# list capacities that let 2 ions take 2048, 1500, 1024 and 750 collisions a
# round (a quarter of the list over the ions), the last ones not multiples of 64
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("capacity", [16384, 12000, 8192, 6001])
def test_ion_chain_cut_anywhere_is_the_same(precision, capacity):
    if precision not in _BASE:
        _BASE[precision] = _run(precision, 1 << 20)
    base = _BASE[precision]
    shi = base.trace[base.trace[:, 3] == abi.EVENT_NAMES.index("shi")]
    assert len(shi) == base.n_events[0] > 2 * 2048
    t = _run(precision, capacity)
    assert (t.n_events == base.n_events).all()
    for k in base.arrays:
        assert np.array_equal(base[k], t[k]), k

    def key(tr):
        return tr[np.lexsort((tr[:, 2], tr[:, 1].copy().view(np.uint64), tr[:, 0]))]
    assert np.array_equal(key(base.trace), key(t.trace), equal_nan=True)
    # every ion's collisions follow each other in time, to the end of the layer
    for it in (0.0, 1.0):
        c = key(shi[shi[:, 0] == it])
        assert np.array_equal(c[:, 2], np.arange(len(c)))
        assert np.array_equal(c[1:, 4], c[:-1, 10])
