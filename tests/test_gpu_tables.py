"""Batch tables kept between calls, on device 0: calls on other systems between
two runs of a batch, a system removed and another taking its slot and its
range, a batch in another order, tuned settings, row capacities moved, pools
grown -- each run gives what fresh engines give for its systems alone.
"""
import numpy as np
import pytest

import sop_amd as S
from sop_amd import workloads as W

pytestmark = pytest.mark.gpu


def make(seed, n):
    s = S.make_chain_system(seed, n)
    s.params.seed = W.philox_key(51, seed)
    return s


def alone(s, *steps):
    with S.Engine(0) as e:
        i = e.add(s)
        for k in steps:
            e.run([i], k)
        return e.coords(i)


def test_tables_follow_the_batch_and_the_systems():
    a, b, c, d = make(1, 700), make(2, 3000), make(3, 130), make(4, 701)
    with S.Engine(0) as e:
        ia, ib, ic = (e.add(s) for s in (a, b, c))
        e.run([ia, ib], 60)
        e.energy_eval(ic)
        e.force_eval(ib)
        e.update_pair_list(ic)
        e.run([ia, ib], 60)
        e.run([ib, ia], 30)
        assert np.array_equal(e.coords(ia), alone(a, 60, 60, 30))
        e.remove(ia)
        id_ = e.add(d)
        assert id_ == ia  # the same slot
        e.run([id_, ic], 75)
        assert np.array_equal(e.coords(id_), alone(d, 75))
        assert np.array_equal(e.coords(ic), alone(c, 75))
        e.tune_set({"lanes_per_bead": 4, "step_blocks": 0, "lds_beads_max": 5056, "bucket_max_beads": [1024, 3072, 10000],
                    "step_tiles": [4, 4, 4], "pl_shell": [3.0, 3.0, 3.0], "step_tail": 2})
        cap, _ = e.rows(id_)
        e.reserve_rows(id_, cap + 64)
        e.run([id_, ic], 25)
        more = [e.add(make(60 + k, 4000)) for k in range(8)]  # every pool grows
        e.run([id_, ic], 50)
        assert np.array_equal(e.coords(id_), alone(d, 75, 25, 50))
        assert np.array_equal(e.coords(ic), alone(c, 75, 25, 50))
        e.run(more, 20)
        assert np.array_equal(e.coords(more[5]), alone(make(65, 4000), 20))


def test_coordinates_forces_and_velocities_round_trip():
    for n in (1, 64, 65, 1000):
        s = make(70 + n, n)
        s.params.dynamics = S._abi.DYN_UNDERDAMPED
        s.vel = np.random.default_rng(n).normal(0, 0.5, (n, 3)).astype(np.float32)
        with S.Engine(0) as e:
            i = e.add(s)
            assert np.array_equal(e.coords(i), s.xyz) and np.array_equal(e.velocities(i), s.vel)
            x = (s.xyz + np.float32(0.25)).astype(np.float32)
            e.set_coords(i, x)
            assert np.array_equal(e.coords(i), x) and e.step_of(i) == 0
            e.update_pair_list(i)
            assert e.force_eval(i).shape == (n, 3)


def test_errors_are_reported_for_the_system_that_has_them():
    a, b = make(81, 200), make(82, 300)
    with S.Engine(0) as e:
        ia, ib = e.add(a), e.add(b)
        x = a.xyz.copy()
        x[100:] += 5.0  # one bond past its largest extension
        e.set_coords(ia, x)
        with pytest.raises(S.SopError) as err:
            e.run([ia, ib], 10)
        assert err.value.status == -5
        e.run([ib], 10)
        e.set_coords(ia, a.xyz)
        e.update_neighbor_list(ia)
        e.run([ia], 10)
