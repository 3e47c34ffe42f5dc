"""Recorded calls of the differentiable PM path, replayed after later calls on the same
context needed more memory: the graphs' buffers are kept (tests/test_growbuf.py has
their lifetime on the CPU), so every replay gives what the eager call gives.
"""
import pytest
import torch

from cube_nu_amd import pmdiff

pytestmark = pytest.mark.gpu


def _positions(m, n, seed):
    return torch.rand((m, 3), generator=torch.Generator().manual_seed(seed)).cuda() * n


def _more(pm, what):
    """A later call that needs larger buffers than any before."""
    if what == "density":
        pm.cic(_positions(70001, pm.n, 7), 96, 96 / pm.n)
    else:
        x = _positions(90001, pm.n, 8)
        pm.force_vjp(x, None, x)
    torch.cuda.synchronize()


@pytest.mark.parametrize("what", ["density", "particles"])
@pytest.mark.parametrize("n", [32, 50])
def test_recorded_force_after_larger_calls(n, what):
    pm, other = (pmdiff.PMForce(n, 1, 1.0) for _ in range(2))
    x, g = _positions(20011, n, 1), _positions(20011, 1, 2) - 0.5
    phi, phi_o = (torch.empty((1, n, n, n), device="cuda") for _ in range(2))
    pm.force_phi(x, phi)  # the buffers of both orders, so that the recorded calls sort
    pm.force_vjp_phi(x, phi, g)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        acc = pm.force_phi(x, phi)
        gx = pm.force_vjp_phi(x, phi, g)
    for k in range(3):
        if k:
            _more(pm, what if k == 1 else "density")
        y = _positions(20011, n, 10 + k)
        want = other.force_phi(y, phi_o)
        want_g = other.force_vjp_phi(y, phi_o, g)
        x.copy_(y)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(phi, phi_o) and torch.equal(acc, want) and torch.equal(gx, want_g), k
    pm.close()
    other.close()


@pytest.mark.parametrize("m", [5003, 70001])  # by atomics, in order
def test_recorded_density_after_larger_calls(m):
    pm, other = (pmdiff.PMForce(32, 1, 1.0) for _ in range(2))
    x = _positions(m, 32, 1)
    pm.cic(x, 40, 1.25)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rho = pm.cic(x, 40, 1.25)
    for k in range(3):
        if k:
            pm.cic(_positions(1003 if k == 1 else 150001, 32, 3), 72, 2.25)
            _more(pm, "particles")
        y = _positions(m, 32, 10 + k)
        want = other.cic(y, 40, 1.25)
        x.copy_(y)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(rho, want), k
    pm.close()
    other.close()


@pytest.mark.parametrize("nw", [40, 72])  # within the forces' accumulator (three meshes of 32^3), and beyond it
def test_recorded_density_of_more_particles_than_before(nw):
    """After one call with the mesh's size a recorded call takes any number of
    particles: the form by atomics needs no memory that depends on it."""
    pm, other = (pmdiff.PMForce(32, 1, 1.0) for _ in range(2))
    pm.cic(_positions(70001, 32, 1), nw, nw / 32)
    x = _positions(150001, 32, 2)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rho = pm.cic(x, nw, nw / 32)
    for k in range(3):
        y = _positions(150001, 32, 10 + k)
        want = other.cic(y, nw, nw / 32)
        x.copy_(y)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(rho, want), k
    pm.close()
    other.close()
