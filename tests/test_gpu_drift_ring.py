"""Which source cells a resident drift reads (drift_ring_last of the timing report: the
buffer cells around a tile), and the way back from the cut ring.

After buffer_v the ring is the bound of the shift, M cells; without it, or with M
beyond the buffers, the buffers whole.  A particle whose shift is within 1e-6 of
the bound cannot be told from one beyond it on all its images, so such a drift
starts again with a pass of its own over every cell: against the oracle, bit for
bit, like the others.
"""
import numpy as np
import pytest

from cube_nu_amd import P3M
from cube_nu_amd.p3m import Geometry
from inputs import buffered_set, oparams
from oracle import pyoracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("izipx,nnt", [(2, 4), (1, 2)])
@pytest.mark.parametrize("cells,follow,ring,again", [
    (0.4, True, 1, False), (1.7, True, 2, False), (2 - 1e-3, True, 2, False), (3.5, True, 4, False),
    (0.4, False, None, False), (4.5, True, None, False),  # the whole buffers
    (1 - 1e-7, True, None, True), (2 - 1e-7, True, None, True), (2.0, True, None, True)])
def test_ring_and_restart(izipx, nnt, cells, follow, ring, again):
    geo = Geometry(64, izipx=izipx, nnt=nnt, nns=2)
    xp, vp, pid, rhoc = buffered_set(geo, seed=int(10 * cells) + nnt, mean=5.0)
    vp = (vp * np.float32(3.0 / np.abs(vp).max())).astype(np.float32)
    p = P3M(64, izipx=izipx, nnt=nnt, nns=2)
    try:
        p.upload(xp, vp, pid, rhoc)
        k = p.kick_resident(a_mid=0.5, dt=0.001)
        if follow:
            p.buffer_v_resident()
        dt = cells * geo.ratio_cs / float(max(k["vmax"]))
        xe, ve, pe, re = p.download()
        p.timing(True)
        p.timing_reset()
        d = p.drift_resident(dt_old=dt, dt=dt, vz_max=k["vz_max"])
        rep = p.timing_report()
        xg, vg, pg, rg = p.download()
    finally:
        p.close()
    assert rep["drift_ring_last"]["calls"] == (geo.ncb if ring is None else ring)
    assert rep["drift_rank"]["calls"] == (2 if again else 1)
    assert rep.get("drift_shift", {"calls": 0})["calls"] == (1 if again else 0)
    st, xo, vo, po, ro, oo = orc.drift(oparams(geo), xe, ve, pe, re, dt, dt, k["vz_max"])
    assert st == 0 and d["nlayer"] == oo["nlayer"] and d["nplocal"] == oo["nplocal"]
    assert np.array_equal(rg, ro)
    assert np.array_equal(xg, xo) and np.array_equal(vg, vo) and np.array_equal(pg, po)


@pytest.mark.parametrize("rest", [(0, 0, 1), (1, 0, 1), (1, 1, 1)])
def test_axes_at_rest(rest):
    """Where nothing moves along an axis its bound is 0, and no particle is beyond it."""
    geo = Geometry(64, nnt=4, nns=2)
    xp, vp, pid, rhoc = buffered_set(geo, seed=8, mean=5.0)
    vp = vp * np.float32(3.0 / np.abs(vp).max()) * np.array([1 - r for r in rest], np.float32)
    p = P3M(64, nnt=4, nns=2)
    try:
        p.upload(xp, np.ascontiguousarray(vp), pid, rhoc)
        k = p.kick_resident(a_mid=0.5, dt=0.0)
        p.buffer_v_resident()
        xe, ve, pe, re = p.download()
        p.timing(True)
        p.timing_reset()
        dt = 0.4 * geo.ratio_cs / 3.0
        d = p.drift_resident(dt_old=dt, dt=dt, vz_max=k["vz_max"])
        rep = p.timing_report()
        xg, vg, pg, rg = p.download()
    finally:
        p.close()
    assert list(np.abs(ve).max(0) == 0) == [bool(r) for r in rest]
    assert rep["drift_ring_last"]["calls"] == (0 if all(rest) else 1)
    assert rep["drift_rank"]["calls"] == 1 and "drift_shift" not in rep
    st, xo, vo, po, ro, oo = orc.drift(oparams(geo), xe, ve, pe, re, dt, dt, k["vz_max"])
    assert st == 0 and d["nlayer"] == oo["nlayer"] and d["nplocal"] == oo["nplocal"]
    assert np.array_equal(rg, ro)
    assert np.array_equal(xg, xo) and np.array_equal(vg, vo) and np.array_equal(pg, po)
