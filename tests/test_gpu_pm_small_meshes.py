"""Many particles on small meshes.  The sorted forms give a tile of 16 x 8 x 8 cells
to one workgroup, so on a mesh of a few tiles they would wait for a few
workgroups: such meshes take the form by atomics.

Times: never much above those of the other form (cube_pm_cic_noalloc; a force
recorded on a fresh context, which cannot allocate the order's buffers), with a
margin of one half for noise; in order, 300 000 particles on these meshes took
2.1 to 5.2 times as long.  Results: small meshes in batches of many have the tiles,
and stay the other form's bit for bit.
"""
import pytest
import torch

from cube_nu_amd import pmdiff

pytestmark = pytest.mark.gpu


def _time(f):
    f()
    best = []
    for _ in range(5):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(4):
            f()
        b.record()
        torch.cuda.synchronize()
        best.append(a.elapsed_time(b))
    return min(best)


def _positions(m, n, seed):
    return torch.rand((m, 3), generator=torch.Generator().manual_seed(seed)).cuda() * n


def _noalloc(pm, x, nw, scale, rho):
    rc = pm.lib.cube_pm_cic_noalloc(pm.ctx, pmdiff._ptr(x), pm._np(x), nw, scale, pmdiff._ptr(rho), pmdiff._stream())
    assert rc == 0


def _recorded(pm, x, phi):
    """A force by atomics, as a graph."""
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        acc = pm.force_phi(x, phi)
    return graph, acc


@pytest.mark.parametrize("nw,batch", [(8, 1), (9, 1), (16, 1), (20, 1), (16, 4)])
def test_density_on_a_few_tiles_takes_no_longer(nw, batch):
    pm = pmdiff.PMForce(16, batch, 1.0)
    x = _positions(300000, 16, nw)
    rho = torch.empty((batch, nw, nw, nw), device="cuda")
    assert _time(lambda: pm.cic(x, nw, nw / 16)) <= 1.5 * _time(lambda: _noalloc(pm, x, nw, nw / 16, rho))
    assert torch.equal(rho, pm.cic(x, nw, nw / 16))
    pm.close()


@pytest.mark.parametrize("n", [10, 12, 18])
def test_force_on_a_few_tiles_takes_no_longer(n):
    pm, few = (pmdiff.PMForce(n, 1, 1.0) for _ in range(2))
    x = _positions(300000, n, n)
    phi = [torch.empty((1, n, n, n), device="cuda") for _ in range(2)]
    graph, _ = _recorded(few, x, phi[1])
    assert _time(lambda: pm.force_phi(x, phi[0])) <= 1.5 * _time(graph.replay)
    assert torch.equal(*phi)
    pm.close()
    few.close()


@pytest.mark.parametrize("n,batch", [(8, 24), (10, 16), (18, 3), (22, 2)])
def test_batches_of_small_meshes_in_order(n, batch):
    pm, few = (pmdiff.PMForce(n, batch, 1.0) for _ in range(2))
    m = 16384 // batch + 11
    x = _positions(batch * m, n, n)
    x[::3] = torch.tensor([n - 0.4, 0.2, n / 2], device="cuda")
    phi = [torch.empty((batch, n, n, n), device="cuda") for _ in range(2)]
    graph, acc_few = _recorded(few, x, phi[1])
    acc = pm.force_phi(x, phi[0])
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(*phi)
    # 27 taps and 3 sums in FP32, each of relative rounding 2^-24, against the largest force
    assert float((acc - acc_few).abs().max()) <= 32 * 2.0 ** -24 * 27 * float(acc.abs().max())
    pm.close()
    few.close()


@pytest.mark.parametrize("nw,batch,m", [(8, 64, 65536), (17, 8, 65536), (28, 1, 262144), (29, 2, 65536), (33, 1, 65536)])
def test_batches_of_small_densities_in_order(nw, batch, m):
    pm = pmdiff.PMForce(16, batch, 1.0)
    x = _positions(batch * (m // batch), 16, nw)
    x[::3] = torch.tensor([15.9, 0.1, 8.0], device="cuda")
    rho = torch.empty((batch, nw, nw, nw), device="cuda")
    _noalloc(pm, x, nw, nw / 16, rho)
    assert torch.equal(rho, pm.cic(x, nw, nw / 16))
    pm.close()
