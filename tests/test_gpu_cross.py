"""The cross-atom potentials against their own definition: V_k(p) = sum_lm Y_lm
S_{k,lm}(r) / r from the library's U_lm, with the oracle's spline and an
independent harmonics recurrence, over item and task shapes: one shell per item,
items that end inside a cell, tasks of one point up to two per lane, points below
the first and beyond the last knot, and every order of l up to the largest."""
import math

import numpy as np
import pytest

from dftcxx_amd import gridlib as G
from dftcxx_amd import molecule as M

from systems import core_guess

pytestmark = pytest.mark.gpu


def _harmonics(d, lmax):
    """|d| and the real harmonics [n, nlm] of the directions d [n, 3]."""
    r = np.sqrt((d * d).sum(1))
    ct = d[:, 2] / r
    az = np.arctan2(d[:, 1], d[:, 0])
    st = np.sqrt(np.maximum(0.0, 1.0 - ct * ct))
    Y = np.empty((len(d), (lmax + 1) ** 2))
    pmm = np.ones(len(d))
    for m in range(lmax + 1):
        p0, p1 = np.zeros(len(d)), pmm
        for l in range(m, lmax + 1):
            n = math.sqrt((2 * l + 1) / (4 * math.pi) * math.factorial(l - m) / math.factorial(l + m))
            n *= math.sqrt(2.0) if m else 1.0
            Y[:, l * l + l + m] = n * p1 * np.cos(m * az)
            if m:
                Y[:, l * l + l - m] = n * p1 * np.sin(m * az)
            p0, p1 = p1, ((2 * l + 1) * ct * p1 - (l + m) * p0) / (l + 1 - m)
        pmm = -(2 * m + 1) * st * pmm
    return r, Y


@pytest.mark.parametrize("make,nrad,nang,lmax", [
    (M.h2o, 5, 6, 0), (M.n2, 6, 590, 1), (M.co, 33, 26, 5), (M.ch4, 21, 110, 8), (M.benzene, 24, 302, 7),
    (M.h2o, 17, 146, 12)])
def test_cross_potentials_from_their_coefficients(make, nrad, nang, lmax):
    from oracle import oracle as O
    mol = make("sto3g")
    print(f"[case] {mol.name} {nrad}x{nang} lmax {lmax}", flush=True)
    g = G.MolecularGrid(mol, nrad, nang, lmax)
    g.set_density(core_guess(mol, *O.one_electron(mol)))
    g.correct_densities()
    g.calculate_hartree_potential()
    V, parts, xyz = g.get_hartree_potential(), g.get_hartree_parts(), g.get_positions()
    x = np.cos(math.pi / (nrad + 1) * np.arange(nrad, 0, -1))
    knots = (1 + x) / (1 - x)
    ref, size = parts["vcell"].copy(), np.abs(parts["vcell"])
    cell = nrad * nang
    for k in range(mol.natoms):
        r, Y = _harmonics(xyz - mol.xyz[k], lmax)
        other = np.arange(len(r)) // cell != k
        for lm in range((lmax + 1) ** 2):
            y = np.ascontiguousarray(parts["U_lm"][k, ::-1, lm])
            c = O.spline(knots, y).reshape(nrad - 1, 4)
            i = np.clip(np.searchsorted(knots, r), 1, nrad - 1) - 1
            t = r - knots[i]
            s = c[i, 0] + t * (c[i, 1] + t * (c[i, 2] + t * c[i, 3]))
            s = np.where(r < knots[0], y[0], np.where(r >= knots[-1], y[-1], s))
            ref[other] += (s * Y[:, lm] / r)[other]
            size[other] += np.abs(s * Y[:, lm] / r)[other]
    # the polynomials in cos(theta) cancel by at most (1 + sqrt 2)^lmax < 4e4 of a
    # term's size; 4e4 eps = 9e-12
    assert np.all(np.abs(V - ref) <= 1e-11 * size.max())
