"""PM1's interpolation where coarse cells hold more particles than a wavefront takes
alone (512; the rest is the workgroup's): counts around that edge and far above it,
on both block sizes (2^3 cells below 4096 blocks of 4^3, as at 64^3; 4^3 at 256^3),
against the oracle's coarse kick within the parity bound, rms 1e-5, from particles
at rest so that the velocities hold the kick alone.
"""
import numpy as np
import pytest

from cube_nu_amd import P3M
from inputs import buffered_set, oparams, rel_rms
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ng,izipx,mean", [(64, 2, 3.0), (64, 1, 3.0), (256, 2, 0.2)])
def test_cells_longer_than_a_wavefront(ng, izipx, mean):
    dense = [((1 + 2 * i, 3, i), n) for i, n in enumerate((511, 512, 513, 575, 767, 768, 769))] + [((15, 15, 15), 9001)]
    v = {}
    for precision in (32, 64):
        p = P3M(ng, izipx=izipx, precision=precision)
        xp, vp, _, rhoc = buffered_set(p.geo, seed=ng + izipx, mean=mean, dense=dense)
        v[precision] = np.zeros_like(vp)
        out = p.kick(xp, v[precision], rhoc, a_mid=0.5, dt=0.25, phase_mask=1)
        p.close()
    ref = np.zeros_like(vp)
    o, _, _ = orc.kick(oparams(p.geo), xp, ref, rhoc, orc.tf_default(oparams(p.geo)), 0.5, 0.25, phase_mask=1)
    assert rel_rms(v[32], ref) <= 1e-5 and rel_rms(v[64], ref) <= 1e-5
    assert abs(out["f2max_pm1"] / o["f2max_pm1"] - 1) <= 1e-5
