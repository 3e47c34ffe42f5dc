"""The resident drift that visits only the source cells its shift bound reaches.

After a kick and buffer_v the buffers are images of the physical particles, and
a drift whose bound M is within the buffers takes the tile and M cells around it
as sources; without buffer_v, or beyond the buffers' depth, it takes every cell of
the extended tiles.  Sparse sets (most runs of cells empty), and dense ones (cells
of more particles than a wavefront has lanes), against the oracle's drift bit for
bit.
"""
import numpy as np
import pytest

from cube_nu_amd import P3M
from cube_nu_amd.p3m import Geometry
from inputs import buffered_set, oparams
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("izipx,nnt,mean", [(2, 4, 0.3), (1, 2, 70.0), (2, 2, 6.0)])
@pytest.mark.parametrize("cells,follow", [(0.4, True), (1.7, True), (3.6, True), (0.9, False)])
def test_drift_of_images_matches_oracle(izipx, nnt, mean, cells, follow):
    geo = Geometry(64, izipx=izipx, nnt=nnt, nns=2)
    xp, vp, pid, rhoc = buffered_set(geo, seed=int(10 * mean), mean=mean)
    vp = (vp * np.float32(3.0 / np.abs(vp).max())).astype(np.float32)
    p = P3M(64, izipx=izipx, nnt=nnt, nns=2)
    try:
        p.upload(xp, vp, pid, rhoc)
        k = p.kick_resident(a_mid=0.5, dt=0.001)
        if follow:
            p.buffer_v_resident()
        dt = cells * geo.ratio_cs / max(k["vmax"])
        xe, ve, pe, re = p.download()
        d = p.drift_resident(dt_old=dt, dt=dt, vz_max=k["vz_max"])
        xg, vg, pg, rg = p.download()
    finally:
        p.close()
    st, xo, vo, po, ro, oo = orc.drift(oparams(geo), xe, ve, pe, re, dt, dt, k["vz_max"])
    assert st == 0 and d["nlayer"] == oo["nlayer"] and d["nplocal"] == oo["nplocal"]
    assert np.array_equal(rg, ro)
    assert np.array_equal(xg, xo) and np.array_equal(vg, vo) and np.array_equal(pg, po)
