"""Host arrays through the staged copies: pageable arrays of 8 MB and more pass
through pinned chunks of several threads, smaller and pinned ones directly; the
bytes are the same either way, and so is a kick through host arrays.
"""
import ctypes

import numpy as np
import pytest
import torch

from cube_nu_amd import P3M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ng,nnt,nns", [(48, 2, 2), (64, 4, 4), (96, 2, 2)])  # velocities of some MB to some 100 MB
def test_pageable_and_pinned_arrays_hold_the_same_state(ng, nnt, nns):
    p = P3M(ng, box=600.0 * ng / 512, nnt=nnt, nns=nns)
    q = P3M(ng, box=600.0 * ng / 512, nnt=nnt, nns=nns)
    try:
        p.make_ic(seed=3, z=1.0)
        xp, vp, pid, rhoc = p.download()
        n = xp.shape[0]
        pinned = [torch.zeros(a.shape, dtype=torch.from_numpy(a[:1].copy()).dtype, pin_memory=True)
                  for a in (xp, vp, pid, rhoc)]
        got = ctypes.c_int64()
        p._check(p.lib.cube_p3m_state_download(p.ctx, *[ctypes.c_void_p(t.data_ptr()) for t in pinned], n,
                                               ctypes.byref(got)))
        assert got.value == n
        for a, t in zip((xp, vp, pid, rhoc), pinned):
            assert np.array_equal(a, t.numpy())
        q.upload(xp, vp, pid, rhoc)
        for a, b in zip((xp, vp, pid, rhoc), q.download()):
            assert np.array_equal(a, b)
        v = vp.copy()
        k = q.kick(xp, v, rhoc, a_mid=0.5, dt=0.01)
        r = p.kick_resident(a_mid=0.5, dt=0.01)
        assert k["f2max_pp"] == r["f2max_pp"] and np.array_equal(v, p.download()[1])
    finally:
        p.close()
        q.close()
