"""Step and shell filter with a block per tile against the item kernels, on device 0.

Small batches, and the few systems too large to stage, take a block per tile;
step_tiles asks for the item kernels instead.  Both run the same arithmetic in
the same order, so coordinates, forces and velocities are bitwise equal: at
tile remainders, with rows longer than one block of held chunks, native lists
longer than the held ones, no natives, two bead types, several chains, jobs
that end inside a block of steps, underdamped dynamics, every lane count, and
either side of the tile counts where the launch changes.  The filter's lists
come out in the same order, for shell, grid and neighbor-list builds.
"""
import numpy as np
import pytest

import sop_amd as S
from sop_amd import workloads as W

pytestmark = pytest.mark.gpu


def chain(seed, n, types=1, under=False, natives=True, chains=1):
    s = S.make_chain_system(seed, n)
    rng = np.random.default_rng(seed)
    s.params.seed = W.philox_key(41, seed)
    if types == 2:
        s.type = rng.integers(1, 3, n).astype(np.int32)
        for i in (1, 2):
            for j in (1, 2):
                s.params.sigma_rep[i][j] = 3.8 + 0.1 * (i + j - 2)
                s.params.eps_att[i][j] = 1.0 - 0.1 * (i + j - 2)
    if under:
        s.params.dynamics, s.params.h, s.params.zeta = S._abi.DYN_UNDERDAMPED, 2.5e-3, 0.05
        s.vel = rng.normal(0, 0.7, (n, 3)).astype(np.float32)
    if not natives:
        s.nat_i, s.nat_j, s.nat_r0 = (np.zeros(0, d) for d in (np.int32, np.int32, np.float32))
    if chains > 1:
        s.chain = np.sort(rng.integers(0, chains, n)).astype(np.int32)
        keep = ~((s.chain[s.nat_i] == s.chain[s.nat_j]) & (s.nat_j - s.nat_i <= 2))
        s.nat_i, s.nat_j, s.nat_r0 = s.nat_i[keep], s.nat_j[keep], s.nat_r0[keep]
    return s


def outputs(systems, steps, **opts):
    with S.Engine(0, **opts) as e:
        ids = [e.add(s) for s in systems]
        f0 = [e.force_eval(i, with_noise=k % 2 == 1) for k, i in enumerate(ids)]
        e.run(ids, steps)
        return f0 + [e.coords(i) for i in ids] + [e.velocities(i) for i in ids]


@pytest.mark.parametrize("systems,steps,lanes", [
    ([(1, 1), (2, 2), (3, 63), (4, 64), (5, 65)], 60, 4),
    ([(6, 700, 2)], 60, 4),
    ([(7, 700, 2, True), (8, 129)], 60, 4),
    ([(9, 900, 1, False, False)], 30, 4),
    ([(10, 900, 1, False, True, 5)], 55, 4),
    ([(11, 1500)], 30, 8),
    ([(12, 600, 2)], 30, 16),
    ([(13, 600)], 30, 32),
    ([(14, 11000)], 20, 4),
    ([(15, 65536, 1, False, False)], 12, 4),  # the largest system with 16-bit rows
    ([(16, 8000), (17, 3000), (18, 8000)], 12, 4),
])
def test_tile_step_equals_item_step(systems, steps, lanes):
    made = [chain(*a) for a in systems]
    got = outputs(made, steps, lanes_per_bead=lanes)
    want = outputs(made, steps, lanes_per_bead=lanes, step_tiles=16)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("sizes", [(49152,), (49153,), (66000,), (30000, 12000, 11000), (1000, 60000, 3000)])
def test_global_gather_items_by_count(sizes):
    """Items of the systems too large to stage, on either side of the last batch
    with a block per tile, against items of 16 tiles: 16- and 32-bit rows,
    several systems, and beside systems that are staged."""
    made = [chain(60 + k, n, 1, False, False) for k, n in enumerate(sizes)]
    for a, b in zip(outputs(made, 12), outputs(made, 12, step_tiles=16)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("systems,lanes", [
    ([(70, 2000)] * 14 + [(71, 12000)], 4),
    ([(72, 4500, 2)] * 8 + [(73, 11000, 2), (74, 64)], 4),
    ([(75, 130)] * 3 + [(76, 70000, 1, False, False)], 4),  # 32-bit rows
    ([(77, 700, 1, True)] * 30 + [(78, 20000, 1, True)], 8),
])
def test_staged_and_gathered_systems_in_one_launch(systems, lanes):
    """LDS and global-gather items of one launch, against each system alone."""
    made = [chain(*a) for a in systems]
    for k, s in enumerate(made):
        s.params.seed = W.philox_key(47, k)
    got = outputs(made, 20, lanes_per_bead=lanes)
    n = len(made)
    for k in (0, n - 2, n - 1):
        with S.Engine(0, lanes_per_bead=lanes) as e:
            i = e.add(made[k])
            assert np.array_equal(got[k], e.force_eval(i, with_noise=k % 2 == 1))
            e.run([i], 20)
            assert np.array_equal(got[n + k], e.coords(i))
            assert np.array_equal(got[2 * n + k], e.velocities(i))


@pytest.mark.parametrize("n,types,lanes", [(300, 1, 4), (1500, 2, 4), (700, 1, 8), (6000, 1, 4), (12000, 2, 4)])
def test_beads_on_one_another(n, types, lanes):
    """Pairs below the repulsion's guard, in the middle of rows and at their ends:
    the item kernels' loops meet them without the guard first."""
    s = chain(200 + n, n, types)
    rng = np.random.default_rng(n)
    on = rng.choice(np.arange(0, n - 4, 4), 40, replace=False)
    for a, b in zip(on[:20], on[20:]):
        s.xyz[a] = s.xyz[b]
    s.bond_r0[:-1] = np.linalg.norm(s.xyz[1:].astype(np.float64) - s.xyz[:-1], axis=1)  # bonds at rest
    f = []
    for tiles in (0, 16):
        with S.Engine(0, step_tiles=tiles, lanes_per_bead=lanes) as e:
            f.append(e.force_eval(e.add(s)))
    assert np.array_equal(*f) and np.all(np.isfinite(f[0]))


def test_dense_rows_and_many_natives():
    """Rows of several hundred partners and up to 40 natives a bead."""
    n = 1400
    s = chain(21, n)
    s.xyz = (s.xyz * np.float32(0.55)).astype(np.float32)
    s.bond_r0 = (s.bond_r0 * np.float32(0.55)).astype(np.float32)
    rng = np.random.default_rng(3)
    i, j = np.triu_indices(n, 3)
    pick = rng.random(len(i)) < 40.0 / n
    s.nat_i, s.nat_j = i[pick].astype(np.int32), j[pick].astype(np.int32)
    s.nat_r0 = np.linalg.norm(s.xyz[s.nat_i] - s.xyz[s.nat_j], axis=1).astype(np.float32)
    f = []
    for tiles in (0, 16):
        with S.Engine(0, step_tiles=tiles) as e:
            k = e.add(s)
            assert e.rows(k)[1] > 256
            f.append(e.force_eval(k))
    assert np.array_equal(*f)


@pytest.mark.parametrize("replicas,n", [(8, 4032), (8, 4096), (9, 4096)])
def test_either_side_of_the_tile_count(replicas, n):
    base = chain(31, n)
    made = []
    for r in range(replicas):
        t = S.System(xyz=base.xyz, params=S.copy_params(base.params), bond_r0=base.bond_r0, nat_i=base.nat_i,
                     nat_j=base.nat_j, nat_r0=base.nat_r0)
        t.params.seed = W.philox_key(43, r)
        made.append(t)
    got = outputs(made, 20)
    want = outputs(made, 20, step_tiles=16)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def lists_after_moves(s, tiles, moves):
    out = []
    rng = np.random.default_rng(5)
    with S.Engine(0, step_tiles=tiles) as e:
        i = e.add(s)
        x = s.xyz
        for d in moves:
            # (a larger move shifts the whole system: the bonds hold)
            x = x + rng.normal(0, 0.05, x.shape).astype(np.float32) + np.float32(d if d > 1 else 0.0)
            e.set_coords(i, x)
            e.update_pair_list(i)
            out += [e.get_list(i, w) for w in (S.LIST_PL_REP, S.LIST_PL_NATIVE)]
            st = e.list_stats(i)
            out.append(np.array([st.grid_builds, st.shell_builds, st.nl_builds, st.pl_rep, st.pl_native]))
            out.append(e.force_eval(i))
    return out


@pytest.mark.parametrize("n,types,scale,natives,skin,model", [
    (1, 1, 1.0, 8, 16.0, "config"), (63, 1, 1.0, 8, 16.0, "config"), (130, 2, 1.0, 8, 16.0, "config"),
    (1400, 1, 0.6, 8, 16.0, "config"),      # rows past two passes of 64
    (400, 1, 0.6, 300, 16.0, "config"),     # more than 128 natives a bead
    (700, 2, 1.0, 40, 16.0, "reference"),   # factor cutoffs
    (700, 1, 1.0, 8, 0.05, "config"),       # neighbor-list builds
    (12000, 1, 1.0, 8, 16.0, "config")])
def test_tile_filter_gives_the_item_filters_lists(n, types, scale, natives, skin, model):
    s = chain(100 + n, n, types)
    if model == "reference":
        p = S.params_reference()
        p.zeta, p.boxl, p.seed = 50.0, 0.0, 9
        s.params = p
    else:
        s.params.nl_abs = s.params.pl_abs + skin
    s.xyz = (s.xyz * np.float32(scale)).astype(np.float32)
    s.bond_r0 = (s.bond_r0 * np.float32(scale)).astype(np.float32)
    if natives != 8:
        rng = np.random.default_rng(n)
        i, j = np.triu_indices(n, 3)
        pick = rng.random(len(i)) < natives / n
        s.nat_i, s.nat_j = i[pick].astype(np.int32), j[pick].astype(np.int32)
        s.nat_r0 = np.linalg.norm(s.xyz[s.nat_i] - s.xyz[s.nat_j], axis=1).astype(np.float32)
    moves = (0.05, 0.05, 2.0, 0.05)  # shell builds, a grid build (or one from the snapshot), a shell build
    got, want = lists_after_moves(s, 0, moves), lists_after_moves(s, 16, moves)
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
