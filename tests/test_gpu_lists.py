"""Half lists as the device counts, places and writes them, on device 0: one
bead, a broken group of sixteen beads, the blocks of 1,024 beads that the
places are summed over, cells of fewer and more members than the sort compares
at a time (eight), and a list that leaves in more than one window (4 Mi pairs)
from 32-bit rows.  Up to 2,100 beads against the FP64 oracle's lists;
the large one against a k-d tree: every pair nearer than its longest is in it,
or excluded.  In all of them the pairs come by bead, i < j, and a shorter buffer
gets the list's first entries and nothing behind them.
"""
import ctypes as C

import numpy as np
import pytest

import sop_amd as S
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def by_bead(got, n):
    assert np.all(got[:, 0] < got[:, 1]) and np.all(np.diff(got[:, 0]) >= 0)
    key = np.sort(got[:, 0].astype(np.int64) * n + got[:, 1])
    assert np.all(np.diff(key) > 0)  # none twice
    return key


def short_buffer(e, i, which, got, cap):
    buf = np.full((cap + 2, 2), -7, np.int32)
    n = C.c_int64()
    st = S.lib().sop_get_list(e._h, i, which, buf.ctypes.data_as(C.POINTER(C.c_int32)), cap, C.byref(n))
    assert st == 0 and n.value == len(got)
    assert np.array_equal(buf[:cap], got[:cap]) and np.all(buf[cap:] == -7)


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 17, 24, 1024, 1025, 2100])
def test_lists_against_the_oracle(n):
    s = S.make_chain_system(810 + n % 89, n)
    (nla, nlr), (pla, plr) = Oracle(s).lists(s.xyz, grid=False)
    nat = np.stack([s.nat_i, s.nat_j], 1).reshape(-1, 2)
    with S.Engine(0) as e:
        i = e.add(s)
        for which, ref in ((S.LIST_NL_NATIVE, nat[nla]), (S.LIST_NL_REP, nlr), (S.LIST_PL_NATIVE, nat[pla]),
                           (S.LIST_PL_REP, plr)):
            got = e.get_list(i, which)
            ref = np.asarray(ref, np.int64).reshape(-1, 2)
            assert np.array_equal(by_bead(got, n), np.sort(ref[:, 0] * n + ref[:, 1])), which
            if len(got) > 1:
                short_buffer(e, i, which, got, len(got) // 2)


def test_a_list_of_more_than_one_window():
    from scipy.spatial import cKDTree

    n = 90000
    s = S.make_chain_system(811, n, native_cutoff=4.0)
    with S.Engine(0) as e:
        i = e.add(s)
        got = e.get_list(i, S.LIST_PL_REP)
        assert len(got) > 4 << 20
        by_bead(got, n)
        x = s.xyz.astype(np.float64)
        d = np.sqrt(((x[got[:, 0]] - x[got[:, 1]]) ** 2).sum(1))
        r = float(d.max())
        tree = cKDTree(x)
        # pairs of other lists (bonds, angles, native contacts) are not in it
        listed = np.unique(got[:, 0].astype(np.int64) * n + got[:, 1])
        near = tree.query_pairs(r - 1e-4, output_type="ndarray").astype(np.int64)
        near = np.sort(near, axis=1)
        miss = np.setdiff1d(near[:, 0] * n + near[:, 1], listed)
        mi, mj = miss // n, miss % n
        nat = s.nat_i.astype(np.int64) * n + s.nat_j
        assert np.all((mj - mi <= 2) | np.isin(miss, nat))
        short_buffer(e, i, S.LIST_PL_REP, got, (4 << 20) + 5)
