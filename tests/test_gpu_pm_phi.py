"""A potential at any address: arrays that are no multiple of 16 bytes hold the
same values, and give the same adjoint, as aligned ones."""
import pytest
import torch

from cube_nu_amd import pmdiff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(24, 20011), (18, 3001), (90, 20011)])
@pytest.mark.parametrize("at", [1, 2])
def test_potential_at_any_address(n, m, at):
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = torch.rand((m, 3), generator=gen, device="cuda") * n
    g = torch.randn(x.shape, generator=gen, device="cuda")
    pm = pmdiff.PMForce(n, 1, 1.0)
    phi = torch.empty((1, n, n, n), device="cuda")
    room = torch.full((n ** 3 + 8,), 5.0, device="cuda")
    odd = room[at:at + n ** 3].view(1, n, n, n)
    assert torch.equal(pm.force_phi(x, odd), pm.force_phi(x, phi))
    assert torch.equal(odd, phi) and bool((room[:at] == 5).all()) and bool((room[at + n ** 3:] == 5).all())
    # cells one at a time instead of four: the same operations in the same order
    assert torch.equal(pm.force_vjp_phi(x, odd, g), pm.force_vjp_phi(x, phi, g))
    pm.close()
