"""The shell-quartet integrals: every class of s and p quartets, with contractions of
1 to 36 primitive pairs (each team width), zero and far separations (both branches of
the Boys function), p before s and s before p, and molecules that mix them with
d functions, against the oracle's Taketa-Huzinaga-O-ohata integrals."""
import numpy as np
import pytest

from dftcxx_amd import gridlib as G
from dftcxx_amd import molecule as M

from systems import random_density, with_d_shell

pytestmark = pytest.mark.gpu


def _mixed(far):
    """Two heavy atoms and a hydrogen; shells in the order p, s, p, s with 1, 2, 3 and 6 primitives."""
    table = {1: [(0, [3.4, 0.7, 0.17], [0.2, 0.6, 0.3])],
             6: [(1, [9.0, 1.9, 0.45], [0.1, 0.4, 0.6]),
                 (0, [3047.0, 457.0, 103.0, 29.0, 9.2, 3.1], [0.002, 0.014, 0.07, 0.23, 0.47, 0.36]),
                 (1, [0.17], [1.0]), (0, [0.8, 0.2], [0.5, 0.6])]}
    xyz = np.array([[0.0, 0.0, 0.0], [0.3, -1.1, far], [1.2, 0.9, -0.7]])
    return M.Molecule(np.array([6, 6, 1]), xyz, table, f"mixed {far}")


@pytest.mark.parametrize("make", [lambda: _mixed(2.3), lambda: _mixed(40.0), lambda: M.ch4("p631"),
                                  lambda: M.h2o("sto6g"), lambda: with_d_shell(M.co("sto3g"))])
def test_coulomb_against_oracle(make):
    from oracle import oracle as O
    mol = make()
    print(f"[case] ERI {mol.name}", flush=True)
    P = random_density(mol.nbf(), 5)
    J, Jo = G.Eri(mol).coulomb(P), O.eri_J(mol, P)
    assert np.abs(J - Jo).max() <= 1e-12 * np.abs(Jo).max()
