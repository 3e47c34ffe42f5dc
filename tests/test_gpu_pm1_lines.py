"""The coarse level's convolution by lines, at every size that the plane form holds
beyond 88 points, against the FP64 form (whose coarse meshes above 64 points take the
generic line passes) on the same particles at rest: the velocities hold the coarse
kick alone.

Tolerance: the force meshes carry FP32 rounding of 2e-6 (as in test_gpu_fft_sizes), the
interpolation 27 products of weights and forces that are rounded four times each,
4 eps/2 = 2.4e-7 of the sum of their sizes, within 4 times the kick's for white noise:
1e-6.  Taken together as 3e-6.
"""
import numpy as np
import pytest

from cube_nu_amd import P3M
from inputs import buffered_set, rel_rms

pytestmark = pytest.mark.gpu


# tilings whose other meshes are of lengths the transform takes
@pytest.mark.parametrize("nc,nnt,nns", [(96, 4, 4), (104, 2, 4), (112, 4, 4), (120, 3, 4), (128, 4, 4), (144, 4, 4),
                                        (160, 4, 4), (168, 4, 3), (176, 4, 4), (192, 4, 4)])
def test_coarse_kick_by_lines(nc, nnt, nns):
    v = {}
    for precision in (32, 64):
        p = P3M(4 * nc, nnt=nnt, nns=nns, precision=precision)
        if not v:
            xp, vp, _, rhoc = buffered_set(p.geo, seed=nc, mean=0.1)
        v[precision] = np.zeros_like(vp)
        p.kick(xp, v[precision], rhoc, a_mid=0.5, dt=0.25, phase_mask=1)
        p.close()
    err = rel_rms(v[32], v[64])
    print(f"nc={nc} rel {err:.2e}")
    assert err <= 3e-6
