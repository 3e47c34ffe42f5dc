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
