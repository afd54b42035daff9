"""Results on device memory that holds NaN before the library writes it: a value
read before it is written would show."""
import pytest

import alloc_probe

pytestmark = pytest.mark.gpu

_ERI = """
probe.probe_fill(1)
for n in (1, 2, 126, 129):
    # n uncontracted s functions, two to an atom on a jittered lattice; with 1 or 126
    # (mod 128) functions the last pair is the first of its block of 64 and no row
    # follows it in the last chunk
    rng = np.random.default_rng(n)
    na = (n + 1) // 2
    xyz = np.array([[i % 5, i // 5 % 5, i // 25] for i in range(na)]) * 2.1 + 0.2 * rng.standard_normal((na, 3))
    one, two = [(0, [0.9], [1.0])], [(0, [0.9], [1.0]), (0, [0.3], [1.0])]
    mol = M.Molecule([1] * (n // 2) + [2] * (n % 2), xyz, {1: two, 2: one}, str(n))
    assert mol.nbf() == n
    P = random_density(n, n)
    e = G.Eri(mol)
    ints, J = e.integrals(), e.coulomb(P)
    i, j = np.tril_indices(n)
    v, Jp = np.where(i == j, P[i, j], 2.0 * P[i, j]), np.zeros(len(i))
    size = 0.0
    for K in range(len(i)):
        row = ints[K * (K + 1) // 2:(K + 1) * (K + 2) // 2]
        Jp[K] += row @ v[:K + 1]
        Jp[:K] += row[:K] * v[K]
        size = max(size, np.abs(row) @ np.abs(v[:K + 1]))
    # up to 8385 terms of at most 1.1e-16 of their size each, in both sums
    assert np.abs(J[i, j] - Jp).max() <= 2e-12 * size, n
    print("ok", n, flush=True)
"""


def test_coulomb_matrix_from_integrals(tmp_path):
    assert alloc_probe.run(tmp_path, _ERI).count("ok") == 4
