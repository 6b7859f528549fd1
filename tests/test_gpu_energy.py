"""Energies, virial, contacts and Rg^2 at the tile counts where their kernels
change, on device 0, against the FP64 oracle on the device's own pair list:
one bead, a full and a broken tile, more tiles than the reduction's threads,
more than the launch's blocks.  Tolerances as for the other energy checks:
each term within 2e-6 of the sum of magnitudes, contacts exact, Rg^2 1e-9.
"""
import numpy as np
import pytest

import sop_amd as S
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 64, 65, 16400, 33000])
def test_energies_at_the_tile_counts(n):
    s = S.make_chain_system(700 + n % 97, n)
    o = Oracle(s)
    with S.Engine(0) as e:
        i = e.add(s)
        rep = e.get_list(i, S.LIST_PL_REP)
        assert len(e.get_list(i, S.LIST_PL_NATIVE)) == len(s.nat_i)  # all within 16 A
        _, er, st = o.forces(s.xyz, (np.arange(len(s.nat_i), dtype=np.int32), rep))
        assert st == 0
        en = e.energy_eval(i)
        assert np.all(np.abs(en[:5] - er[:5]) <= 2e-6 * np.abs(er[:4]).sum() + 1e-12)
        assert abs(en[5] - er[5]) <= 2e-6 * max(abs(er[5]), np.abs(er[:4]).sum()) + 1e-12
        q, c, rg = e.observables(i)
        assert c == len(s.nat_i)
        x = s.xyz.astype(np.float64)
        assert abs(rg - ((x - x.mean(0)) ** 2).sum(1).mean()) <= 1e-9 * max(rg, 1.0)
