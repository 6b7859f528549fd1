"""A served job is charged for what it holds, on device 0: per bead 185 bytes of
state and lists (seven 16-byte arrays, fourteen of 4 bytes, two of 8, one of 1)
and its rows, per tile of 64 beads 4 bytes of table and ten doubles of energy
sums, per cell 20 bytes; and those energy sums fit where they are kept, up to
the last tile of the pool.
"""
import numpy as np
import pytest

import sop_amd as S
from sop_amd import serving

pytestmark = pytest.mark.gpu


def test_a_job_is_charged_for_its_arrays():
    rows = 2 * 2 * 384  # two row segments of 16-bit entries at the starting capacity
    with S.Engine(0) as e:
        srv = serving.Server(e)
        try:
            sizes = [6400, 12800]
            charge = [srv.job_bytes(S.System(xyz=np.zeros((n, 3), np.float32), params=S.params_config()))
                      for n in sizes]
        finally:
            srv.stop()
    for n, c in zip(sizes, charge):
        assert c == n * (185 + rows) + n // 64 * 84 + 20 * (2 * n + 1)


def test_energies_of_a_full_pool():
    # 128 tiles, the pool's capacity (a power of two): systems in its last tiles
    # beside others, whose sums stay their own when it grows
    small = [S.make_chain_system(650 + k, 512) for k in range(16)]
    with S.Engine(0) as e, S.Engine(0) as one:
        ids = [e.add(s) for s in small]
        ids.append(e.add(S.make_chain_system(670, 3000)))
        for s, i in zip(small, ids):
            k = one.add(s)
            assert np.array_equal(e.energy_eval(i), one.energy_eval(k))
            one.remove(k)
