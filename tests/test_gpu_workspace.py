"""Kicks under a workspace budget that holds the whole-image mesh and some of a level's
windows at a time: the windows of every batch are cut from the same mesh, so the
velocities are those of the automatic budget bit for bit, with one species and
with a second one whose density is added; and a budget below half of which the
mesh does not fit takes the deposits per window, with the same bits.
"""
import numpy as np
import pytest

from cube_nu_amd import P3M
from inputs import buffered_set

pytestmark = pytest.mark.gpu

NG = 64
IMAGE = 4 * (NG // 4 * 8) ** 3  # the sub-tile level's mesh of the whole image


@pytest.mark.parametrize("budget", [2 * IMAGE, 2 * IMAGE + 3000001, 2 * IMAGE - 1, 1])
@pytest.mark.parametrize("species", [1, 2])
def test_batches_under_a_budget(budget, species):
    got = []
    for b in (0, budget):
        p = P3M(NG, workspace_bytes=b)
        nu = P3M(NG) if species == 2 else None
        xp, vp, pid, rhoc = buffered_set(p.geo, seed=9, mean=5.0)
        p.upload(xp, vp, pid, rhoc)
        if nu:
            nu.upload(*buffered_set(nu.geo, seed=10, mean=1.0))
        out = []
        for _ in range(2):  # (a context's later kicks overlap their levels)
            out.append(p.kick_resident_nu(nu, a_mid=0.4, dt=0.2, nu_mass=0.05) if nu
                       else p.kick_resident(a_mid=0.4, dt=0.2))
        got.append((out, p.download()[1], nu.download()[1] if nu else None))
        p.close()
        if nu:
            nu.close()
    (o0, v0, n0), (o1, v1, n1) = got
    assert o0 == o1 and np.array_equal(v0, v1) and not np.array_equal(v0, vp)
    assert n0 is None or np.array_equal(n0, n1)
