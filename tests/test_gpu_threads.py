"""Handles made, used and closed from several threads at a time, each on its own
stream: what one thread's handle leaves to the next must not show in any result."""
import threading

import numpy as np
import pytest

from dftcxx_amd import gridlib as G
from dftcxx_amd import molecule as M

from systems import random_density

pytestmark = pytest.mark.gpu


def _pass(n_carbon):
    mol = M.alkane(n_carbon)
    P = random_density(mol.nbf(), seed=n_carbon)
    with G.MolecularGrid(mol, 12, 50, 4) as g:
        g.set_density(P)
        g.correct_densities()
        J = g.calculate_hartree_potential()
        XC, exc = g.calculate_exchange_correlation()
    return J, XC, exc


def test_threads_share_the_memory_of_closed_handles():
    sizes = [2, 3, 9, 10]
    want = {n: _pass(n) for n in sizes}
    wrong = []

    def work(first):
        for k in range(6):
            n = sizes[(first + k) % len(sizes)]
            J, XC, exc = _pass(n)
            if not (np.array_equal(J, want[n][0]) and np.array_equal(XC, want[n][1]) and exc == want[n][2]):
                wrong.append(n)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
