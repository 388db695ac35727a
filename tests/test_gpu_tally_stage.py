"""The stage that a run's finished tallies pass through on their way to the
caller: it lies in the particle lists, so that asking for the tallies takes no
device memory; lists too short for it have a buffer beside them, and both give
the same values.  Single runs and batches."""
import numpy as np
import pytest
import torch

import trekis_gpu as tg
from trekis_gpu.batch import Batch, IonContext

from gpu_helpers import say

pytestmark = pytest.mark.gpu

NR = 3000          # 101 nodes x 3000 bins x 14 radial tallies: 34 MB of finished values
RADIAL = ("Out_ne", "Out_Ee", "Out_nphot", "Out_Ephot", "Out_Elat", "Out_nh", "Out_Eh", "Out_Ehkin")
SPECTRA = ("Out_Ee_vs_E", "Out_Eh_vs_E", "Out_theta", "Out_theta_h", "Out_diff_coeff", "Out_Ne_Em", "Out_E_Em",
           "Out_Ee_vs_E_Em")


def _context(capacity):
    mat, ion, opt, run = tg.config_material("test")
    mat.prepare(tg.load_library())
    opt.gen_capacity = capacity
    ctx = tg.Context(mat, ion, opt)
    ctx.build_tables()
    R, V = tg.radial_grid(NR, run["Rmin"], run["Rmax"], mat.layer)
    return ctx, ion, run, R, V


def _tallies(ctx, without):
    t = ctx.new_tallies(NR)
    for k in without:
        setattr(t.s, k, None)
    return t


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_tallies_of_a_run_take_no_device_memory():
    ctx, _, run, R, V = _context(1 << 20)
    ctx.run_mc(1, run["seed"], R, V, tallies=_tallies(ctx, RADIAL + SPECTRA))
    before = _free()
    a = ctx.run_mc(1, run["seed"], R, V, tallies=_tallies(ctx, SPECTRA))
    taken = before - _free()
    say(f"[stage] {taken} bytes taken by a run with all radial tallies")
    assert taken < 4 << 20
    # 600 particles in a list: a buffer of its own
    short, *_ = _context(600)
    b = short.run_mc(1, run["seed"], R, V, tallies=_tallies(short, SPECTRA))
    full = ctx.run_mc(1, run["seed"], R, V)
    for k in a.arrays:
        assert np.array_equal(a[k], b[k]), k
        if k not in SPECTRA:
            assert np.array_equal(a[k], full[k]), k
    assert a["Out_ne"].sum() > 0


def test_tallies_of_a_batch_take_no_device_memory():
    ctx, ion, run, R, V = _context(1 << 20)
    impacts = []
    for E in (1.0, 0.5, 0.75):
        other = type(ion).from_buffer_copy(ion)
        other.E = ion.E * E
        c = IonContext(ctx, other)
        c.build_tables()
        impacts.append(c)
    out = []
    for capacity in (1 << 20, 2000):
        b = Batch(impacts, R, V, capacity=capacity)
        b.run(run["seed"], 0, with_tallies=False)
        before = _free()
        t = b.fetch()
        taken = before - _free()
        again = b.run(run["seed"], 0)
        say(f"[stage] batch, lists of {capacity}: {taken} bytes taken by fetching the tallies")
        assert taken < 4 << 20 or capacity == 2000
        out += [t, again]
    for t in out[1:]:
        for x, y in zip(out[0], t):
            for k in x.arrays:
                assert np.array_equal(x[k], y[k]), k
    # each impact's own run, through the single run's stage
    for i, c in enumerate(impacts):
        s = c.run_mc(1, run["seed"], R, V, first_iter=i)
        for k in RADIAL:
            assert np.array_equal(s[k], out[0][i][k]), (i, k)
