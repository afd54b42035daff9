"""Functions and points at the edge of the reach beyond which function tiles are left
out of a build (bases of more than 80 functions, unscreened)."""
import numpy as np
import pytest

from dftcxx_amd import gridlib as G
from dftcxx_amd import molecule as M

from systems import random_density, with_d_shell

pytestmark = pytest.mark.gpu


def _results(mol, P, precision=G.PREC_FP64):
    with G.MolecularGrid(mol, 14, 38, 3, precision=precision) as g:
        g.set_density(P)
        g.correct_densities()
        rho = g.get_densities()
        J = g.calculate_hartree_potential()
        XC, exc = g.calculate_exchange_correlation()
        dP, grad = g.xc_adjoint()
    return rho, J, XC, exc, dP, grad


@pytest.mark.parametrize("make", [lambda: M.alkane(9), lambda: with_d_shell(M.alkane(7)),
                                  lambda: M.alkane(9, "p631")], ids=["s_p", "d", "p631"])
def test_basis_scaled_down(make):
    """Every function 2^-90 times itself and P 2^180 times: the same density, matrix
    elements 2^-180 times.  The products of both scalings are exact, so each result
    differs by no more than the roundings of sums in another order: 1e-12 of the
    largest value covers their some 1e3 terms of 1.1e-16."""
    mol = make()
    print(f"[case] scaled down {mol.name}", flush=True)
    table = mol.basis if isinstance(mol.basis, dict) else M.load_basis(mol.basis)
    small = M.Molecule(mol.Z, mol.xyz,
                       {z: [(L, a, [v * 2.0 ** -90 for v in c]) for L, a, c in sh] for z, sh in table.items()}, "small")
    P = random_density(mol.nbf(), 8)
    want, got = _results(mol, P), _results(small, P * 2.0 ** 180)
    for name, w, v, scale in zip(("rho", "J", "XC", "exc", "dEdP", "grad"), want, got, (1, 180, 180, 0, 180, 0)):
        v = np.asarray(v) * (2.0 ** 180 if scale == 180 else 1.0)
        assert np.abs(v - w).max() <= 1e-12 * max(np.abs(w).max(), 1.0 if name == "grad" else 0.0), name
