"""A served underdamped job starts from the velocities it was submitted with:
sop_serve_submit copies the description, and the caller's arrays are its own
again when the call returns, however long the job is queued.  On device 0.
"""
import numpy as np
import pytest

import sop_amd as S
from sop_amd import serving

pytestmark = pytest.mark.gpu


def test_velocities_are_copied_at_submission():
    first = S.make_chain_system(641, 64)
    s = S.make_chain_system(642, 300)
    s.params.dynamics = S._abi.DYN_UNDERDAMPED
    s.params.h, s.params.zeta, s.params.T = 2.5e-3, 0.05, 0.6
    vel = np.random.default_rng(5).normal(0, 0.7, (s.n, 3)).astype(np.float32)
    s.vel = vel.copy()
    with S.Engine(0) as eng:
        srv = serving.Server(eng, max_jobs=1)
        try:
            a = srv.submit(first, 5000)  # holds the only slot while the next one is queued
            b = srv.submit(s, 100)
            s.vel[:] = 0.0
            assert srv.wait(a)[0]["status"] == 0
            r, x = srv.wait(b)
        finally:
            srv.stop()
    assert r["status"] == 0
    s.vel = vel
    with S.Engine(0) as e:
        i = e.add(s)
        e.run([i], 100)
        assert np.array_equal(x, e.coords(i))
