"""Calls that the thread driving the engine makes on a resident system while the
serve loop admits, steps and retires jobs beside it, on device 0: each returns
what it returns alone, and each job ends as it does alone.  The jobs grow the
pools and have new blocks captured meanwhile.
"""
import numpy as np
import pytest

import sop_amd as S
from sop_amd import serving

pytestmark = pytest.mark.gpu


def calls(e, i, x):
    """What a program may ask of a system between runs, whole."""
    e.set_coords(i, x)
    e.update_neighbor_list(i)
    e.update_pair_list(i)
    out = [e.coords(i), e.wrapped_coords(i), e.force_eval(i), e.energy_eval(i), np.array(e.observables(i))]
    out += [e.get_list(i, w) for w in range(4)]
    s = e.list_stats(i)
    return out + [np.array([s.nl_native, s.nl_rep, s.pl_native, s.pl_rep]), e.increments(i)]


def test_calls_beside_the_serve_loop():
    held = S.make_chain_system(660, 1700)
    moved = [held.xyz, held.xyz + np.float32(0.25)]
    jobs = [S.make_chain_system(661 + k, n) for k, n in enumerate([250, 900, 64, 3000, 6000, 400, 1500, 12000])]
    steps = [100 * (k % 4 + 1) for k in range(len(jobs))]
    with S.Engine(0) as e:
        i = e.add(held)
        want = [calls(e, i, x) for x in moved]
    with S.Engine(0) as eng:
        i = eng.add(held)
        srv = serving.Server(eng, max_jobs=4)
        try:
            ids = [srv.submit(s, n) for s, n in zip(jobs, steps)]
            rounds = 0
            while rounds < 6 or not all(srv.poll(j)[0] for j in ids):
                for x, w in zip(moved, want):
                    for k, (a, b) in enumerate(zip(calls(eng, i, x), w)):
                        assert np.array_equal(a, b), (rounds, k)
                rounds += 1
                assert rounds < 2000
            res = [srv.wait(j) for j in ids]
        finally:
            srv.stop()
        eng.remove(i)
    with S.Engine(0) as e:
        for s, n, (r, xs) in zip(jobs, steps, res):
            assert r["status"] == 0, s.n
            k = e.add(s)
            e.run([k], n)
            assert np.array_equal(xs, e.coords(k)), s.n
            assert np.array_equal(r["energies"], e.energy_eval(k)[:6]), s.n
            e.remove(k)
