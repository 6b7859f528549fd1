"""Items that gather from global memory, several systems to a batch, on device
0: fewer items than XCDs, a last run that is short, a system cut by the end of
an XCD's run, more items than compute units, and 16- beside 32-bit rows.  Which
items a system is cut into, and where they run, is no part of a result: each
system as it is by itself, bitwise.
"""
import numpy as np
import pytest

import sop_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes, options", [
    ([300, 70], {"step_tiles": 16}),                       # two items
    ([900 + 13 * k for k in range(60)], {}),               # 60 items of one system each
    ([1000 + k for k in range(270)], {}),                  # more items than units
    ([4000, 12000, 5100, 12100, 4900, 16000, 3000], {}),   # cut by the runs
    ([11000, 66000], {}),                                  # 16- and 32-bit rows
])
def test_gathered_systems_together_equal_alone(sizes, options):
    systems = [S.make_chain_system(300 + k, n) for k, n in enumerate(sizes)]
    picked = sorted({0, len(sizes) // 2, len(sizes) - 1, int(np.argmax(sizes))})
    with S.Engine(0, lds_beads_max=-1, **options) as a, S.Engine(0) as b:
        ia = [a.add(s) for s in systems]
        a.run(ia, 20)
        for k in picked:
            ib = b.add(systems[k])
            b.run([ib], 20)
            assert np.array_equal(a.coords(ia[k]), b.coords(ib)), sizes[k]
            assert np.array_equal(a.force_eval(ia[k]), b.force_eval(ib)), sizes[k]
            b.remove(ib)


def test_a_large_system_beside_many():
    # more items than units: the large system's runs fill some XCDs, the others
    # go whole to the rest
    sizes = [66000] + [8000 + 100 * k for k in range(12)] + [11000, 25000, 30000]
    systems = [S.make_chain_system(380 + k, n) for k, n in enumerate(sizes)]
    with S.Engine(0, lds_beads_max=-1) as a, S.Engine(0) as b:
        ia = [a.add(s) for s in systems]
        a.run(ia, 20)
        for k in (0, 1, 12, 14, 15):
            ib = b.add(systems[k])
            b.run([ib], 20)
            assert np.array_equal(a.coords(ia[k]), b.coords(ib)), sizes[k]
            b.remove(ib)
