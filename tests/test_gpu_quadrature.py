"""The inner loops of the table quadratures against the loss function written
out.  A shell (or the phonons) whose oscillators all have strengths and widths
of ordinary size is integrated in a loop made for its number of oscillators,
with the point's constants taken out of it; an oscillator of zero strength
sends the whole shell to the general loop, where it adds exactly 0 to every
sum (its position and width repeat another's, so the grids stay).  Both forms
round every operation alike: all tables and rows are equal bit for bit."""
import numpy as np
import pytest

import trekis_gpu as tg
from trekis_gpu import abi

from gpu_helpers import say

pytestmark = pytest.mark.gpu


def _tables(mat, ion, opt):
    ctx = tg.Context(mat, ion, opt)
    ctx.build_tables()
    out = {}
    for kind in (abi.TAB_E_INEL, abi.TAB_H_INEL, abi.TAB_E_EL, abi.TAB_H_EL, abi.TAB_SHI, abi.TAB_SHI_DIFF):
        for s in [0] if kind in (abi.TAB_E_EL, abi.TAB_H_EL) else range(sum(mat.n_shells)):
            E, L, D = ctx.table(kind, s)
            out[kind, s] = (E, L, D)
            if kind in (abi.TAB_SHI, abi.TAB_SHI_DIFF):
                continue
            for i in range(0, len(E), 7):
                try:
                    out[kind, s, i] = ctx.row(kind, s, i)
                except tg.TrekisError:
                    continue
    return out


def _pair(name, n, quadrature):
    """The target with n valence oscillators, and the same with zero-strength ones added."""
    built = []
    for zero in (False, True):
        mat, ion, opt, run = tg.config_material(name)
        if opt.quadrature != quadrature:
            opt.quadrature = quadrature
        for atom in mat.atoms:
            for k, sh in enumerate(atom.shells):
                if n and atom is mat.atoms[0] and k == len(atom.shells) - 1:
                    e, a, g = sh.osc[0]
                    sh.osc = [(e * (1.0 + 0.3 * i), a / (1.0 + i), g * (1.0 + 0.2 * i)) for i in range(n)]
                if zero:
                    sh.osc = list(sh.osc) + [(sh.osc[0][0], 0.0, sh.osc[0][2])]
        if zero and mat.phonon:
            mat.phonon = list(mat.phonon) + [(mat.phonon[0][0], 0.0, mat.phonon[0][2])]
        mat.prepare(tg.load_library())
        built.append(_tables(mat, ion, opt))
    return built


# 1 to 5 oscillators have loops of their own, 6 and 7 share one; a constant
# mass, the masses of a density of states, three phonons, a single-pole phonon
@pytest.mark.parametrize("name,n,quadrature", [("test", n, 0) for n in range(1, 8)] + [("test", n, 1) for n in (1, 2, 5, 6)] +
                         [("test_metal", 1, 0), ("test_metal", 3, 0), ("test_metal", 6, 0), ("test_sio2", 0, 0)])
def test_loop_forms_agree(name, n, quadrature):
    say(f"[quadrature] {name} {n} oscillators, quadrature {quadrature}")
    a, b = _pair(name, n, quadrature)
    assert a.keys() == b.keys() and len(a) > 50
    for k in a:
        for x, y in zip(a[k], b[k]):
            assert np.array_equal(x, y, equal_nan=True), (k, np.flatnonzero(x != y)[:5])


# an immobile hole given as an infinite mass: its momentum limits are infinite
# or NaN, every hole integral is empty, and the tables are the oracle's
def test_infinite_hole_mass_leaves_empty_integrals():
    from oracle import Oracle
    mat, ion, opt, run = tg.config_material("test_metal")        # electron masses from the density of states
    mat.hole_mass = float("inf")
    mat.prepare(tg.load_library())
    say("[quadrature] test_metal, infinite hole mass")
    ctx = tg.Context(mat, ion, opt)
    ctx.build_tables()
    orc = Oracle(mat, ion, opt)
    orc.build_tables(8)
    for kind in (abi.TAB_E_INEL, abi.TAB_H_INEL, abi.TAB_E_EL, abi.TAB_H_EL):
        for s in [0] if kind in (abi.TAB_E_EL, abi.TAB_H_EL) else range(sum(mat.n_shells)):
            for x, y in zip(ctx.table(kind, s), orc.table(kind, s)):
                assert np.array_equal(x, y, equal_nan=True), (kind, s)
    assert (ctx.table(abi.TAB_H_INEL, 0)[1] >= 1e15).all()
