"""Builds on chains longer than the reach of their functions (the density by the
number of tiles that count on a block, the contraction by point-block lists):
rho and XC against numpy on the library's own amplitudes, over 6 to 32 function
tiles, sizes with and without a density kernel of their own among them.

Each sum has at most (number of terms) roundings of 1.1e-16 of its sum of absolute
terms; 1e-12 of the largest such sum covers the up to 500 terms of the density
and the up to 4000 point-block partials of a matrix element."""
import numpy as np
import pytest

from dftcxx_amd import gridlib as G
from dftcxx_amd import molecule as M

from systems import random_density

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [G.PREC_FP64, G.PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("n_carbon", [7, 8, 9, 13, 21, 31, 38], ids=lambda n: f"c{n}")
def test_long_chain_against_its_amplitudes(n_carbon, precision):
    mol = M.alkane(n_carbon)
    print(f"[case] tile reach {mol.name} nbf={mol.nbf()} precision={precision}", flush=True)
    P = random_density(mol.nbf(), seed=n_carbon)
    g = G.MolecularGrid(mol, 9, 26, 2, precision=precision)
    phi = g.get_amplitudes()
    # an all-zero density first: what it leaves behind must not show in the next one
    g.set_density(np.zeros_like(P))
    g.correct_densities()
    g.set_density(P)
    rho = g.get_densities()
    ref = 2.0 * ((phi @ P) * phi).sum(1)
    assert np.abs(rho - ref).max() <= 1e-12 * (2.0 * ((np.abs(phi) @ np.abs(P)) * np.abs(phi)).sum(1)).max()
    if precision == G.PREC_MIXED:
        return
    g.correct_densities()
    XC, _ = g.calculate_exchange_correlation()
    _, wv = g.get_xc_parts()
    ref = phi.T @ (wv[:, None] * phi)
    assert np.abs(XC - ref).max() <= 1e-12 * (np.abs(phi).T @ (np.abs(wv)[:, None] * np.abs(phi))).max()
