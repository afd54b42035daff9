"""A first gradient that runs out of device memory at any of its allocations: the
call fails, and the next one, with room again, gives what a handle gives that
never failed."""
import pytest

import alloc_probe

pytestmark = pytest.mark.gpu

# 121 functions: 8 tiles, so that T is formed by the number of tiles that count;
# screened handles make the force terms' own tile lists on the first gradient
_GRADIENT = """
mol = M.alkane(9)
P = random_density(mol.nbf(), 3)

def handle(screen):
    g = G.MolecularGrid(mol, 9, 26, 2, screen=screen)
    g.set_density(P)
    g.correct_densities()
    g.calculate_exchange_correlation()
    return g

kept = []  # open until the end: closed handles would leave memory that no allocation is made for
for screen in (0.0, 1e-9):
    kept.append(handle(screen))
    dP0, g0 = kept[-1].xc_adjoint()
    done = fails = 0
    while not done:
        g = handle(screen)
        kept.append(g)
        probe.probe_limit(fails)
        try:
            g.xc_adjoint()
            done = 1
        except G.DgError as e:
            assert "hipMalloc" in str(e), e
            fails += 1
        probe.probe_limit(-1)
        dP, gr = g.xc_adjoint()
        assert np.array_equal(dP, dP0) and np.array_equal(gr, g0), (screen, fails)
        print("screen", screen, "refused", fails, flush=True)
    assert fails >= 8, fails
print("whole")
"""


def test_gradient_after_a_failed_one(tmp_path):
    assert "whole" in alloc_probe.run(tmp_path, _GRADIENT)
