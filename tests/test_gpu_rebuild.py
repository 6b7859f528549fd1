"""List rebuilds at the sizes where their kernels change, on device 0.

Systems of up to 5,120 beads are decided and sorted by one block each; larger
ones by kernels that spread a system over the launch.  Lists are bit-exact
against the oracle on either side of that line, at the block's bead strides,
for clouds spread over more cells than beads, and after moves that force a
grid build; a batch that mixes the two kinds equals each system alone.
"""
import numpy as np
import pytest

import sop_amd as S
from sop_amd import workloads as W
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def pairs(a):
    return np.sort(np.ascontiguousarray(a, np.int32).reshape(-1, 2).view(np.int64).ravel())


def cloud(n, edge, seed):
    """Beads at random in a box: lists only, the bonds are far overstretched."""
    x = np.random.default_rng(seed).uniform(-edge / 2, edge / 2, (n, 3)).astype(np.float32)
    return S.System(xyz=x, params=S.params_config())


@pytest.mark.parametrize("n,edge", [(1, 10), (2, 10), (64, 60), (1023, 120), (1025, 500), (2049, 700), (5120, 420),
                                    (5120, 3000), (5121, 420), (5121, 3000), (8193, 250)])
def test_lists_at_the_rebuild_sizes(n, edge):
    s = cloud(n, edge, n + edge)
    o = Oracle(s)
    with S.Engine(0) as e:
        i = e.add(s)
        for x in (s.xyz, cloud(n, edge, n + edge + 1).xyz):
            e.set_coords(i, x)
            e.update_neighbor_list(i)
            e.update_pair_list(i)
            (_, nl), (_, pl) = o.lists(x)
            assert np.array_equal(pairs(e.get_list(i, S.LIST_PL_REP)), pairs(pl)), (n, edge)
            assert np.array_equal(pairs(e.get_list(i, S.LIST_NL_REP)), pairs(nl)), (n, edge)


def test_small_and_large_systems_in_one_batch_equal_alone():
    sizes = (5121, 70, 5120, 6000, 1024)
    systems = []
    for k, n in enumerate(sizes):
        s = S.make_chain_system(900 + k, n)
        s.params.seed = W.philox_key(31, k)
        systems.append(s)
    alone = []
    for s in systems:
        with S.Engine(0) as e:
            i = e.add(s)
            e.run([i], 130)
            alone.append(e.coords(i))
    with S.Engine(0) as e:
        ids = [e.add(s) for s in systems]
        e.run(ids, 130)
        for i, x in zip(ids, alone):
            assert np.array_equal(e.coords(i), x)
