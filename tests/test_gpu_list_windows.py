"""Half lists through the host buffer, on device 0: arrays shorter and far longer
than the list, ending at, before and behind the first window (64 Ki pairs of a
new engine) and the second, and again through the buffer those have left.  The
caller's array holds the list's first entries and is untouched behind them.
"""
import ctypes as C

import numpy as np
import pytest

import sop_amd as S

pytestmark = pytest.mark.gpu

FIRST = 64 << 10


@pytest.mark.parametrize("cap", [0, 1, FIRST - 1, FIRST, FIRST + 1, 2 * FIRST + 1, 10_000_000])
def test_windows_and_arrays_of_any_length(cap):
    s = S.make_chain_system(820, 1500)
    with S.Engine(0) as ref:
        want = ref.get_list(ref.add(s), S.LIST_NL_REP)
    assert len(want) > 2 * FIRST + 1
    buf = np.full((cap + 2, 2), -7, np.int32)
    n = C.c_int64()
    with S.Engine(0) as e:
        i = e.add(s)
        for _ in range(2):
            buf[:] = -7
            st = S.lib().sop_get_list(e._h, i, S.LIST_NL_REP, buf.ctypes.data_as(C.POINTER(C.c_int32)), cap, C.byref(n))
            assert st == 0 and n.value == len(want)
            m = min(cap, len(want))
            assert np.array_equal(buf[:m], want[:m]) and np.all(buf[m:] == -7)
        assert np.array_equal(e.get_list(i, S.LIST_NL_REP), want)
