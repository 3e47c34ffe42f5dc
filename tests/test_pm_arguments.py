"""Sizes of the mesh and cotangent arguments of PMForce's methods: a tensor that is
shorter than what the library reads or writes is refused before the call (on the CPU,
with the library's entry points replaced)."""
import pytest

torch = pytest.importorskip("torch")

from cube_nu_amd import pmdiff  # noqa: E402


class _Library:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *a: self.calls.append(name) or 0


@pytest.fixture
def pm(monkeypatch):
    monkeypatch.setattr(pmdiff, "_ptr", lambda t: t.data_ptr())
    monkeypatch.setattr(pmdiff, "_stream", lambda: None)
    p = pmdiff.PMForce.__new__(pmdiff.PMForce)
    p.lib, p.ctx, p.n, p.batch, p.lattice = _Library(), None, 8, 2, 0
    return p


X = torch.zeros((2 * 5, 3))
CALLS = {
    "force": lambda p, mesh, g: p.force(X, mesh),
    "force_vjp": lambda p, mesh, g: p.force_vjp(X, mesh, g),
    "force_phi": lambda p, mesh, g: p.force_phi(X, mesh),
    "force_vjp_phi": lambda p, mesh, g: p.force_vjp_phi(X, mesh, g),
}


@pytest.mark.parametrize("name", CALLS)
def test_short_meshes_and_cotangents_are_refused(pm, name):
    meshes = 1 if name.endswith("phi") else 3
    whole, g = torch.zeros(2 * meshes * 512), torch.zeros_like(X)
    CALLS[name](pm, whole, g)
    CALLS[name](pm, None, g)
    assert pm.lib.calls == [f"cube_pm_{name}"] * 2
    with pytest.raises(ValueError, match="holds"):
        CALLS[name](pm, whole[1:], g)
    if "vjp" in name:
        with pytest.raises(ValueError, match="size of x"):
            CALLS[name](pm, whole, g[1:])
    assert len(pm.lib.calls) == 2
