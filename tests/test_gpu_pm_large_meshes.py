"""Meshes beyond 1024 points a side: three force meshes of 1152^3 have more than 2^32
cells, more than one launch dimension has threads.

Exact properties, so that no bound is needed: the potential does not depend on what
the context's memory held before it was created, nor on the calls before; adjoints
through the potential or without it are the same; and a cotangent twice as large,
whose fixed-point numbers are the same integers, has an adjoint twice as large.
"""
import pytest
import torch

from cube_nu_amd import pmdiff

pytestmark = pytest.mark.gpu

N = 1152


@pytest.mark.parametrize("m", [6007, 48056])
def test_adjoint_scales_and_memory_does_not_matter(m):
    gen = torch.Generator(device="cuda").manual_seed(m)
    x = torch.rand((m, 3), generator=gen, device="cuda") * N
    g = torch.randn(x.shape, generator=gen, device="cuda")
    got = []
    for junk in (0.0, 3.0):
        held = torch.full((24 << 30,), junk, device="cuda")  # memory the context is likely to get
        del held
        torch.cuda.empty_cache()
        pm = pmdiff.PMForce(N, 1, 1.0)
        phi = torch.empty((1, N, N, N), device="cuda")
        acc = pm.force_phi(x, phi)
        gx = pm.force_vjp_phi(x, phi, g)
        assert torch.equal(pm.force_vjp_phi(x, phi, 2 * g), 2 * gx)
        assert torch.equal(pm.force_vjp(x, None, g), gx)
        again = torch.empty_like(phi)
        assert torch.equal(pm.force_phi(x, again), acc) and torch.equal(again, phi)
        got.append((phi, acc, gx))
        pm.close()
        del again
    assert all(torch.equal(a, b) for a, b in zip(*got))
    del got, phi
    torch.cuda.empty_cache()


@pytest.mark.parametrize("n", [1040, 1050])  # with and without whole quads
def test_sorted_and_unsorted_forms_agree(n):
    """The order's cells past 1024 (32-bit cells of the mesh instead of bytes): the
    same integers are summed, so the potentials are equal bit for bit; forces
    and adjoints, 27 taps of FP32 rounding, to 27 * 2^-22 of the largest."""
    m = 20011
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = torch.rand((m, 3), generator=gen, device="cuda") * n
    x[::3] = n - 1.2 + 0.9 * torch.rand((len(x[::3]), 3), generator=gen, device="cuda")  # at the mesh's end
    g = torch.randn(x.shape, generator=gen, device="cuda")
    got = []
    for recorded in (False, True):  # a recorded call of a fresh context cannot make the order's buffers
        pm = pmdiff.PMForce(n, 1, 1.0)
        phi = torch.empty((1, n, n, n), device="cuda")
        graph = torch.cuda.CUDAGraph()
        if recorded:
            with torch.cuda.graph(graph):
                acc, gx = pm.force_phi(x, phi), pm.force_vjp_phi(x, phi, g)
            graph.replay()
        else:
            acc, gx = pm.force_phi(x, phi), pm.force_vjp_phi(x, phi, g)
        torch.cuda.synchronize()
        got.append((phi, acc.clone(), gx.clone()))
        pm.close()
    (phi, acc, gx), (phi_f, acc_f, gx_f) = got
    assert torch.equal(phi, phi_f)
    assert float((acc - acc_f).abs().max()) <= 27 * 2.0 ** -22 * float(acc_f.abs().max())
    assert float((gx - gx_f).abs().max()) <= 27 * 2.0 ** -22 * float(gx_f.abs().max())
    del got, phi, phi_f
    torch.cuda.empty_cache()
