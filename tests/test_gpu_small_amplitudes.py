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


def test_last_points_in_a_nodal_plane():
    """The last block holds two points, both in the plane z = z_A of a p shell whose z
    function is alone in the last tile (113 functions): its amplitude there is 0, its
    gradient is not.  Gradient against the oracle at the tolerance of the other
    gradient tests."""
    from oracle import adjoint as AD
    h = [(0, [0.45 + 0.3 * k], [1.0]) for k in range(10)]
    o = [(0, [0.3 + 0.25 * k], [1.0]) for k in range(10)] + [(1, [0.15], [1.0])]
    rng = np.random.default_rng(2)
    xyz = np.vstack([[0.0, 0.0, 0.0], 2.5 * rng.standard_normal((9, 3)), [1.0, 0.5, 0.25]])
    mol = M.Molecule([8] + [1] * 10, xyz, {1: h, 8: o}, "nodal")
    assert mol.nbf() == 113 and 11 * 17 * 38 % 64 == 2
    with G.MolecularGrid(mol, 17, 38, 2) as g:  # the last points belong to the last atom
        z = g.get_positions()[-2:, 2]
    assert z[0] == z[1]
    mol.xyz[0, 2] = z[0]
    P = random_density(113, 6)
    print("[case] nodal plane", flush=True)
    with G.MolecularGrid(mol, 17, 38, 2) as g:
        assert np.all(g.get_amplitudes()[-2:, 112] == 0.0)
        g.set_density(P)
        g.correct_densities()
        g.calculate_exchange_correlation()
        dP, grad = g.xc_adjoint()
    _, dP_o, grad_o = AD.xc_adjoint(mol, 17, 38, 2, P)
    assert np.abs(dP - dP_o).max() < 1e-11 * np.abs(dP_o).max()
    assert np.abs(grad - grad_o).max() < 1e-10 * max(1.0, np.abs(grad_o).max())
