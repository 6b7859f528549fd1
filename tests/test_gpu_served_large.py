"""Served jobs on either side of the sizes at which the list kernels' grids
change (32,768 and 131,072 beads), with a small job beside them, on device 0:
each as it is run alone, bitwise.
"""
import numpy as np
import pytest

import sop_amd as S
from sop_amd import serving
from sop_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[32768, 6000], [32769, 6000, 5121], [131072, 300], [131073, 33000, 9000]])
def test_large_served_jobs_equal_alone(sizes):
    systems = [S.make_chain_system(680 + k, n) for k, n in enumerate(sizes)]
    for k, s in enumerate(systems):
        s.params.seed = W.philox_key(14, k)
    with S.Engine(0) as eng:
        srv = serving.Server(eng, hbm_budget_bytes=64 << 30)
        try:
            ids = [srv.submit(s, 60) for s in systems]
            res = [srv.wait(j) for j in ids]
        finally:
            srv.stop()
    with S.Engine(0) as e:
        for s, (r, x) in zip(systems, res):
            assert r["status"] == 0
            i = e.add(s)
            e.run([i], 60)
            assert np.array_equal(x, e.coords(i)), s.n
            assert np.array_equal(r["energies"], e.energy_eval(i)[:6]), s.n
            e.remove(i)
