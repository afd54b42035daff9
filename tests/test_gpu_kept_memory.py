"""The device memory kept from closed grids on a device that is otherwise full: every
other allocation of the library gets it, and so does the process."""
import pytest

import alloc_probe

pytestmark = pytest.mark.gpu

_CODE = """
mol = M.ch4()
P = random_density(mol.nbf(), 2)
room = -1

def closed_grids():
    global room
    probe.probe_room(-1)
    for g in [G.MolecularGrid(mol, 20, 50, 4) for _ in range(3)]:
        g.close()
    kept = probe.probe_live()
    assert kept > 1 << 20
    probe.probe_room(kept)  # no room beside what is kept

J = G.Eri(mol).coulomb(P)
closed_grids()
assert np.array_equal(G.Eri(mol).coulomb(P), J)
print("integrals", flush=True)
for step in (G.STEP_HOST, G.STEP_DEVICE):
    closed_grids()
    e, res, _ = G.scf_run(mol, 20, 50, 4, density_step=step)
    print("scf", step, e[-1], flush=True)
closed_grids()
G.release_memory()
assert probe.probe_live() == 0
print("whole")
"""


def test_kept_memory_is_given_back(tmp_path):
    assert "whole" in alloc_probe.run(tmp_path, _CODE)
