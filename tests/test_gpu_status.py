"""The status of a call is the systems' state at that call, on device 0: error
bits stay until new coordinates clear them, and neither an earlier call's
status nor another system's comes back.
"""
import numpy as np
import pytest

import sop_amd as S

pytestmark = pytest.mark.gpu


def stretched(x):
    """The chain with bond 63-64 stretched by 3 A, beyond R0."""
    x = x.copy()
    u = (x[64] - x[63]) / np.linalg.norm(x[64] - x[63])
    x[64:] += (3.0 * u).astype(np.float32)
    return x


def status_of(call, *args):
    try:
        call(*args)
        return 0
    except S.SopError as ex:
        return ex.status


@pytest.mark.parametrize("steps", [0, 1])
def test_plain_run_reports_the_state_it_finds(steps):
    good, bad = S.make_chain_system(1, 128), S.make_chain_system(1, 128)
    bad.xyz = stretched(bad.xyz)
    with S.Engine(0) as e:
        b, g = e.add(bad), e.add(good)
        assert status_of(e.run, [b], 1) == S._abi.SOP_ERR_NUMERIC
        # the error bits stay, whatever another system's status is
        assert status_of(e.run_plain, [b, g], steps) == S._abi.SOP_ERR_NUMERIC
        assert status_of(e.run_plain, [g], steps) == 0
        # new coordinates clear them
        e.set_coords(b, good.xyz)
        assert status_of(e.run_plain, [g, b], steps) == 0
        assert e.step_of(b) == 1 + 2 * steps and e.step_of(g) == 3 * steps
