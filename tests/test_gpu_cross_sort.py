"""The sort of the cross potentials' points: batches in which some molecules are single
atoms and so have none, more than 64 spline intervals, several chunks of points to an
atom, few points to an interval; and a potential that does not depend on the order in
which an interval's points were found."""
import numpy as np
import pytest

from dftcxx_amd import gridlib as G
from dftcxx_amd import molecule as M

from systems import random_density

pytestmark = pytest.mark.gpu


def _atom(z, basis):
    return M.Molecule([z], np.array([[0.3, -0.2, 0.1]]), basis, f"Z{z}")


@pytest.mark.parametrize("nrad,nang,lmax", [(70, 50, 10), (130, 14, 2), (9, 302, 5)])
def test_batch_with_single_atoms(nrad, nang, lmax):
    mols = [_atom(2, "sto3g"), M.h2o("p631"), _atom(10, "p631"), _atom(3, "sto3g"), M.ethane(), M.n2(),
            _atom(2, "p631")]
    print(f"[case] batch with atoms {nrad}x{nang} lmax {lmax}", flush=True)
    Ps = [random_density(m.nbf(), i) for i, m in enumerate(mols)]
    J, XC, sc = G.Batch(mols, nrad, nang, lmax).build(Ps)
    for m, P, Jm, XCm, s in zip(mols, Ps, J, XC, sc):
        with G.MolecularGrid(m, nrad, nang, lmax) as g:
            g.set_density(P)
            g.correct_densities()
            J1 = g.calculate_hartree_potential()
            XC1, exc = g.calculate_exchange_correlation()
        assert np.abs(Jm - J1).max() <= 1e-12 * np.abs(J1).max(), m.name
        assert np.abs(XCm - XC1).max() <= 1e-12 * np.abs(XC1).max(), m.name
        assert abs(s[0] - exc) <= 1e-12 * abs(exc), m.name


@pytest.mark.parametrize("nrad,nang,lmax", [(75, 50, 8), (20, 302, 10)])
def test_potential_is_the_same_for_every_handle(nrad, nang, lmax):
    mol = M.alkane(4, "sto3g")
    print(f"[case] same potential {nrad}x{nang} lmax {lmax}", flush=True)
    P = random_density(mol.nbf(), 9)
    V = []
    for _ in range(3):
        with G.MolecularGrid(mol, nrad, nang, lmax) as g:
            g.set_density(P)
            g.correct_densities()
            g.calculate_hartree_potential()
            V.append(g.get_hartree_potential())
    assert np.array_equal(V[0], V[1]) and np.array_equal(V[0], V[2])
