"""Closing a grid while a graph captured from its build replays on another stream: the
replay's results are those of the build, whatever takes the grid's memory next."""
import pytest

from dftcxx_amd import gridlib as G
from dftcxx_amd import molecule as M

from systems import random_density

pytestmark = pytest.mark.gpu


def test_close_waits_for_replays_on_other_streams():
    import torch
    mol, other = M.ethane(), M.ethane()
    other.xyz = other.xyz * 1.2
    P = torch.from_numpy(random_density(mol.nbf(), 4)).cuda()
    out = torch.empty_like(P)
    build, replay = torch.cuda.Stream(), torch.cuda.Stream()
    g = G.MolecularGrid(mol, 30, 50, 6)
    g.set_stream(build.cuda_stream)
    with torch.cuda.stream(build):
        g.build_fock_device(P.data_ptr(), out.data_ptr())
    build.synchronize()
    want = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=build):
        g.build_fock_device(P.data_ptr(), out.data_ptr())
    g.set_stream(0)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        out.zero_()
    torch.cuda.synchronize()
    print("[case] closing with a replay pending", flush=True)
    with torch.cuda.stream(replay):
        torch.cuda._sleep(20_000_000)
        graph.replay()
        done = torch.cuda.Event()
        done.record()
    g.close()
    assert done.query()
    h = G.MolecularGrid(other, 30, 50, 6)  # on the memory just left
    h.set_density(P.cpu().numpy())
    h.correct_densities()
    h.calculate_hartree_potential()
    torch.cuda.synchronize()
    assert torch.equal(out, want)
