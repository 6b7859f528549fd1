"""A system that is refused for want of a slot or of pool room leaves the pools
of the engine as they were, on device 0.
"""
import numpy as np
import pytest

import sop_amd as S

pytestmark = pytest.mark.gpu

SLOTS = 4096  # of an engine with fixed pools


def straight(n):
    x = np.zeros((n, 3), np.float32)
    x[:, 0] = 3.8 * np.arange(n)
    return S.System(xyz=x, params=S.params_config())


def test_refused_adds_give_their_ranges_back():
    # bead pool of two tiles a slot (capacities are powers of two): all slots
    # but two with a system of two tiles, those with one, two tiles free
    with S.Engine(0, pool_bytes=8 * 200 * 128 * SLOTS) as e:
        one, two = straight(4), straight(128)
        ids = [e.add(two) for _ in range(SLOTS - 2)] + [e.add(one) for _ in range(2)]
        for _ in range(5):
            with pytest.raises(S.SopError, match="slot") as err:
                e.add(one)
            assert err.value.status == S._abi.SOP_ERR_CAPACITY
        with pytest.raises(S.SopError, match="pool") as err:
            e.add(straight(129))
        assert err.value.status == S._abi.SOP_ERR_CAPACITY
        e.remove(ids.pop())
        e.remove(ids.pop())
        four = e.add(straight(256))  # the four tiles that are free now
        e.run([four, ids[0]], 3)
        with pytest.raises(S.SopError, match="pool") as err:  # a slot, but no room
            e.add(one)
        assert err.value.status == S._abi.SOP_ERR_CAPACITY
