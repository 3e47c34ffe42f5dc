"""The look at uploaded buffers where a wavefront for every extended cell is more
threads than a launch dimension has (1536^3: 72 million cells): a buffer particle
in a late tile that is no image of a physical one is seen, so the kick takes the
deposits per window, as a context without room for the whole-image mesh does.
"""
import numpy as np
import pytest

from cube_nu_amd import P3M

pytestmark = pytest.mark.gpu


def test_a_late_buffer_cell_is_looked_at():
    got = []
    for budget in (40 << 30, 1):
        p = P3M(1536, workspace_bytes=budget)
        g = p.geo
        assert g.nnt ** 3 * g.nte ** 3 * 64 > 2 ** 32
        rhoc = np.zeros(g.rhoc_shape, np.int32)
        row = rhoc.reshape(g.nnt ** 3, g.nte, g.nte, g.nte)[40, 50, 50]
        row[g.ncb - 1] = row[g.ncb] = 1  # the last buffer cell and the first physical one
        xp, v = np.zeros((2, 3), np.int16), np.zeros((2, 3), np.float32)
        p.kick(xp, v, rhoc, a_mid=0.4, dt=0.2, phase_mask=2)
        got.append(v)
        p.close()
    assert np.array_equal(*got) and got[0][1, 0] < -1e-5  # drawn to the buffer's particle
