"""The routes that leave function tiles out, over 6 to 32 tiles: the contraction's
point-block lists in both precisions and with one and two outputs, T = Phi P by the
number of tiles that count, the force terms' own tile lists of screened handles, and
amplitudes that are not numbers."""
import numpy as np
import pytest

from dftcxx_amd import gridlib as G
from dftcxx_amd import molecule as M

from systems import random_density

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [G.PREC_FP64, G.PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("screen", [0.0, 1e-9], ids=["all", "screened"])
@pytest.mark.parametrize("n_carbon", [7, 9, 13, 21, 38], ids=lambda n: f"c{n}")
def test_matrices_against_their_weights(n_carbon, screen, precision):
    """J, XC and G = 2J + XC against numpy on the library's amplitudes and weights,
    element by element.  FP64: 1e-12 of the sum of absolute terms (some 4000 of 1.1e-16,
    mostly cancelling).  Mixed: a term has the roundings of two amplitudes, a weight and
    a product, and passes through at most 64 FP32 additions before its sum becomes FP64:
    68 of 2^-24.  Left-out terms: below 2^-106, or the screen, of one amplitude."""
    import torch
    mol = M.alkane(n_carbon)
    print(f"[case] {mol.name} screen={screen} precision={precision}", flush=True)
    P = random_density(mol.nbf(), seed=n_carbon)
    with G.MolecularGrid(mol, 9, 26, 2, precision=precision, screen=screen) as g:
        g.set_stream(torch.cuda.current_stream().cuda_stream)
        dP = torch.from_numpy(P).cuda()
        J, XC, F = (torch.empty_like(dP) for _ in range(3))
        g.build_device(dP.data_ptr(), J.data_ptr(), XC.data_ptr())
        g.build_fock_device(dP.data_ptr(), F.data_ptr())
        torch.cuda.synchronize()
        phi = g.get_amplitudes()
        _, wv = g.get_xc_parts()
        uJ = 0.5 * g.get_weights() * g.get_hartree_potential()
        XC1, _ = g.calculate_exchange_correlation()
        J1 = g.calculate_hartree_potential()
    rel = 1e-12 if precision == G.PREC_FP64 else 68 * 2.0 ** -24
    for name, got, u in (("J", J.cpu().numpy(), uJ), ("XC", XC.cpu().numpy(), wv), ("G", F.cpu().numpy(), 2 * uJ + wv),
                         ("J alone", J1, uJ), ("XC alone", XC1, wv)):
        want = phi.T @ (u[:, None] * phi)
        size = np.abs(phi).T @ (np.abs(u)[:, None] * np.abs(phi))
        left = max(screen, 2.0 ** -106) * 2.0 * np.abs(u).sum() * np.abs(phi).max()
        assert np.all(np.abs(got - want) <= rel * size + left + 1e-14 * size.max()), name


@pytest.mark.parametrize("n_carbon,screen", [(11, 0.0), (11, 1e-30), (19, 0.0)])
def test_gradient_of_chains(n_carbon, screen):
    """Chains longer than their functions reach against the oracle's gradient, which
    takes every function at every point; tolerances as in the other gradient tests.  A
    screen of 1e-30 changes nothing in the density that is above them."""
    from oracle import adjoint as AD
    mol = M.alkane(n_carbon)
    mol.xyz = mol.xyz + 0.05 * np.random.default_rng(n_carbon).standard_normal(mol.xyz.shape)
    print(f"[case] gradient {mol.name} screen={screen}", flush=True)
    P = random_density(mol.nbf(), seed=n_carbon)
    with G.MolecularGrid(mol, 5, 14, 1, screen=screen) as g:
        g.set_density(P)
        g.correct_densities()
        g.calculate_exchange_correlation()
        dP, grad = g.xc_adjoint()
    _, dP_o, grad_o = AD.xc_adjoint(mol, 5, 14, 1, P)
    assert np.abs(dP - dP_o).max() < 1e-11 * np.abs(dP_o).max()
    assert np.abs(grad - grad_o).max() < 1e-10 * max(1.0, np.abs(grad_o).max())


@pytest.mark.parametrize("screen", [0.0, 1e-9])
def test_amplitude_that_is_not_a_number_shows(screen):
    mol = M.alkane(9)
    s = M.load_basis(mol.basis)
    table = dict(s)
    table[6] = [(L, a, [float("nan")] + list(c[1:])) if i == 0 else (L, a, c) for i, (L, a, c) in enumerate(s[6])]
    bad = M.Molecule(mol.Z, mol.xyz, table, "nan")
    print(f"[case] NaN amplitudes screen={screen}", flush=True)
    with G.MolecularGrid(bad, 9, 26, 1, screen=screen) as g:
        g.set_density(random_density(mol.nbf(), 1))
        assert np.isnan(g.get_densities()).all()
