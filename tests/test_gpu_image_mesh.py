"""Tile and sub-tile densities cut from the whole image's mesh against the
deposit per window (a context whose workspace holds one window at a time takes
the latter): the same integers are summed, so the kicked velocities agree bit
for bit.  Also with buffer cells that are not the periodic images they stand
for, which only the deposit per window can represent."""
import numpy as np
import pytest

from cube_nu_amd import P3M
from inputs import buffered_set

pytestmark = pytest.mark.gpu

CASES = [  # ng, nnt, nns, izipx, mean, dense cells (count puts their sub-tile at a finer level)
    (64, 4, 4, 2, 8.0, ()),
    (64, 4, 4, 1, 8.0, (((0, 0, 0), 3000), ((15, 15, 15), 1700), ((7, 8, 15), 400))),
    (128, 4, 4, 2, 3.0, (((31, 0, 16), 900),)),
    (192, 4, 4, 1, 2.0, ()),
    (48, 2, 2, 2, 8.0, (((11, 5, 0), 500),)),
    (96, 2, 2, 1, 6.0, ()),
    (16, 1, 2, 2, 20.0, ()),
]


def _pair(ng, nnt, nns, izipx):
    kw = dict(izipx=izipx, nnt=nnt, nns=nns, box=600.0 * ng / 512)
    return P3M(ng, **kw), P3M(ng, workspace_bytes=1, **kw)


@pytest.mark.parametrize("ng,nnt,nns,izipx,mean,dense", CASES)
def test_gpu_image_mesh_matches_windows(ng, nnt, nns, izipx, mean, dense):
    image, window = _pair(ng, nnt, nns, izipx)
    xp, vp, pid, rhoc = buffered_set(image.geo, seed=ng + izipx, mean=mean, dense=dense)
    for mask in (2, 4):
        a, b = vp.copy(), vp.copy()
        oa = image.kick(xp, a, rhoc, a_mid=0.4, dt=0.2, phase_mask=mask)
        ob = window.kick(xp, b, rhoc, a_mid=0.4, dt=0.2, phase_mask=mask)
        assert np.any(a != vp)
        assert np.array_equal(a, b) and oa == ob, (ng, mask)
    image.close()
    window.close()


def test_gpu_image_mesh_needs_periodic_buffers():
    ng = 64
    image, window = _pair(ng, 4, 4, 2)
    xp, vp, pid, rhoc = buffered_set(image.geo, seed=5, mean=6.0)
    first = int(np.argmax(rhoc.reshape(-1) > 0))  # a buffer cell: the corner of tile 0
    assert first < image.geo.ncb
    xp = xp.copy()
    xp[0, 1] ^= 0x4000
    for mask in (2, 4):
        a, b = vp.copy(), vp.copy()
        image.kick(xp, a, rhoc, a_mid=0.4, dt=0.2, phase_mask=mask)
        window.kick(xp, b, rhoc, a_mid=0.4, dt=0.2, phase_mask=mask)
        assert np.array_equal(a, b)
    image.close()
    window.close()
