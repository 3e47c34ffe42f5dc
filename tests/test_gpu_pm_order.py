"""The two forms of the differentiable PM force: many particles, sorted and
gathered by tiles of 16 x 8 x 8 cells, and few, by global atomics.

Meshes of one ragged tile, of tiles that end in a remainder, with and without a
multiple of four points (quads); half of the particles crowded into one cell, so
that a tile's list is far longer than its workgroup.  Both forms add the same
integers, so their potentials are equal bit for bit; forces and adjoints agree
with the FP64 model within the bounds of test_pmdiff.py (rms 1e-5 and 1e-4), in
each form and with F, phi or neither given.  CIC densities take the sorted form
from 65536 particles on; cube_pm_cic_noalloc keeps the atomics, and the two are
equal bit for bit (17 and 33 points end in a tile of one cell).
"""
import pytest
import torch

from cube_nu_amd import pmdiff
from oracle import pm_torch as ref

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a.double().cpu() - b).norm() / b.norm())


@pytest.mark.parametrize("n,batch,lattice", [(8, 2, 0), (18, 1, 0), (24, 2, 0), (50, 1, 0), (40, 2, 32)])
def test_sorted_and_unsorted_forms_agree(n, batch, lattice):
    m = lattice ** 3 if lattice else 16384 // batch + 37
    gen = torch.Generator().manual_seed(n)
    x = torch.rand((batch * m, 3), generator=gen) * n
    x[::2] = torch.tensor([n - 0.6, 0.3, n / 2]) + 0.2 * torch.rand((len(x[::2]), 3), generator=gen)
    if lattice:  # displacements, a few lattice spacings at most
        x = (x - n / 2) * (3.0 / n)
    g = torch.randn(x.shape, generator=gen)
    xd, gd = x.cuda(), g.cuda()
    pm = pmdiff.PMForce(n, batch, 1.0, lattice=lattice)
    # a captured call cannot allocate the order's buffers: the unsorted form
    few = pmdiff.PMForce(n, batch, 1.0, lattice=lattice)
    phi = [torch.empty((batch, n, n, n), device="cuda") for _ in range(2)]
    acc = pm.force_phi(xd, phi[0])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        acc_few = few.force_phi(xd, phi[1])
        gx_few = few.force_vjp_phi(xd, phi[1], gd)
    for _ in range(2):
        phi[1].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(phi[0], phi[1])
    acc_F, F = pm.force(xd)
    assert torch.equal(acc_F, acc)
    gx = {"phi": pm.force_vjp_phi(xd, phi[0], gd), "F": pm.force_vjp(xd, F, gd), "none": pm.force_vjp(xd, None, gd),
          "few": gx_few}

    G = torch.from_numpy(pm.green()).double()
    xr = x.double()
    if lattice:
        xr = xr + pm.sites().repeat(batch, 1)
    xr.requires_grad_(True)
    acc_ref = ref.force(xr, G, batch, n)
    (gx_ref,) = torch.autograd.grad((acc_ref * g.double()).sum(), xr)
    assert _rel(acc, acc_ref.detach()) <= 1e-5 and _rel(acc_few, acc_ref.detach()) <= 1e-5
    for k, v in gx.items():
        assert _rel(v, gx_ref) <= 1e-4, k
    pm.close()
    few.close()


@pytest.mark.parametrize("nw,batch,lattice", [(8, 2, 0), (17, 1, 0), (24, 2, 0), (33, 1, 0), (50, 2, 32), (2, 1, 0)])
def test_sorted_cic_is_the_atomics_cic(nw, batch, lattice):
    n, m = 32, lattice ** 3 if lattice else 65536 // batch
    gen = torch.Generator().manual_seed(nw)
    x = (torch.rand((batch * m, 3), generator=gen) - 0.25) * 2 * n  # beyond the box on both sides
    x[::2] = torch.tensor([n - 0.2, 0.0, 0.5 * n]) + 0.3 * torch.rand((len(x[::2]), 3), generator=gen)
    x = x.cuda()
    pm = pmdiff.PMForce(n, batch, 1.0, lattice=lattice)
    rho, want = pm.cic(x, nw, nw / n), torch.empty((batch, nw, nw, nw), device="cuda")
    rc = pm.lib.cube_pm_cic_noalloc(pm.ctx, pmdiff._ptr(x), m, nw, nw / n, pmdiff._ptr(want), pmdiff._stream())
    assert rc == 0 and torch.equal(rho, want)
    assert torch.equal(pm.cic(x, nw, nw / n), want)  # counts and starts of a second call
    pm.close()
