"""The work this engine is used for, as timed cases.

A case goes through the package's public entry points (sop_amd.Engine and
sop_amd.serving.Server) from what a program holds before the call -- systems
resident in an engine, or jobs on the host -- to the results on the host.

  run       systems advanced by `steps` in one batch, then read back as a
            trajectory row holds them: coordinates, and with `sample` the
            energies, native contacts and Rg^2, underdamped also the velocities
  evaluate  coordinates moved into the engine, both lists rebuilt there, and
            forces, energies and observables read back: a driver that keeps
            its own integrator, or the analysis of a stored trajectory
  lists     coordinates moved in, both lists rebuilt and the pair lists read
            back, as a driver that walks them itself does
  serve     a burst of jobs submitted to the serve loop, waited for one by one

Chains are the compact self-avoiding walks of the synthetic workloads; the
native map is taken from the generated state.  model "config" is the parameter
set of the benchmark workloads (absolute 32 A / 16 A cutoffs every 50 / 10
steps, no box), "reference" the reference program's defaults (3.2x / 2.5x
cutoffs, the pair list rebuilt at every step, a 500 A periodic box).
"""
import math

import numpy as np
import torch

import sop_amd as S
from sop_amd import workloads as W
from sop_amd.serving import Server


def listed():
    return [
        # one small chain, read back every 50 steps: launch latency and nothing else
        {"name": "chain_128", "kind": "run", "replicas": 1, "lo": 128, "hi": 128, "steps": 50, "model": "config",
         "under": False, "two_types": False, "sample": False},
        # one protein-sized chain sampled every 100 steps: energies, contacts, Rg^2
        {"name": "chain_1000_sampled", "kind": "run", "replicas": 1, "lo": 1000, "hi": 1000, "steps": 100,
         "model": "config", "under": False, "two_types": False, "sample": True},
        # the command-file driver's default: reference parameters, pair list at
        # every step, box, two bead types, underdamped, a row every 40 steps
        {"name": "reference_underdamped", "kind": "run", "replicas": 1, "lo": 701, "hi": 701, "steps": 40,
         "model": "reference", "under": True, "two_types": True, "sample": True},
        # the largest chain that is staged two to a compute unit, ragged at the last tile
        {"name": "chain_4999", "kind": "run", "replicas": 1, "lo": 4999, "hi": 4999, "steps": 50, "model": "config",
         "under": False, "two_types": False, "sample": False},
        # one 10,000-bead globule
        {"name": "globule_10000", "kind": "run", "replicas": 1, "lo": 10000, "hi": 10000, "steps": 50,
         "model": "config", "under": False, "two_types": False, "sample": False},
        # an ensemble of one small chain for statistics, sampled every 100 steps
        {"name": "ensemble_32x128", "kind": "run", "replicas": 32, "lo": 128, "hi": 128, "steps": 100,
         "model": "config", "under": False, "two_types": False, "sample": True},
        # the batched benchmark: 512 uneven replicas, a frame every 400 steps
        {"name": "batch_512", "kind": "run", "replicas": 512, "lo": 200, "hi": 5000, "steps": 400, "model": "config",
         "under": False, "two_types": False, "sample": False},
        # many chains in one system, above 65,536 beads (32-bit pair-list rows)
        {"name": "assembly_200k", "kind": "assembly", "chains": 400, "per": 500, "steps": 50},
        # a stored 5,000-bead trajectory evaluated frame by frame
        {"name": "evaluate_5000", "kind": "evaluate", "beads": 5000, "model": "config", "two_types": False},
        # a driver that takes the lists to the host
        {"name": "lists_1500", "kind": "lists", "beads": 1500, "model": "config", "two_types": False},
        # a burst of jobs of the served stream's size law
        {"name": "serve_96", "kind": "serve", "jobs": 96, "median": 1500, "top": 20000, "steps": 200},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["single", "single", "batch", "batch", "reference", "evaluate", "lists", "assembly", "serve"])
    if kind == "single":
        n = _log(rng, 100, 10112)
        return {"kind": "run", "replicas": 1, "lo": n, "hi": n, "steps": _log(rng, 20, 200), "model": "config",
                "under": False, "two_types": rng.random() < 0.2, "sample": rng.random() < 0.5}
    if kind == "batch":
        lo = _log(rng, 100, 1000)
        return {"kind": "run", "replicas": _log(rng, 8, 400), "lo": lo, "hi": _log(rng, lo, 5000),
                "steps": _log(rng, 50, 400), "model": "config", "under": False,
                "two_types": rng.random() < 0.2, "sample": False}
    if kind == "reference":
        n = _log(rng, 100, 5000)
        return {"kind": "run", "replicas": 1, "lo": n, "hi": n, "steps": _log(rng, 20, 100), "model": "reference",
                "under": rng.random() < 0.7, "two_types": rng.random() < 0.7, "sample": True}
    if kind == "evaluate":
        return {"kind": "evaluate", "beads": _log(rng, 100, 10112), "model": rng.choice(["config", "reference"]),
                "two_types": rng.random() < 0.3}
    if kind == "lists":
        return {"kind": "lists", "beads": _log(rng, 100, 5000), "model": rng.choice(["config", "reference"]),
                "two_types": rng.random() < 0.3}
    if kind == "assembly":
        return {"kind": "assembly", "chains": _log(rng, 24, 400), "per": 500, "steps": 50}
    return {"kind": "serve", "jobs": _log(rng, 8, 96), "median": _log(rng, 500, 1500), "top": 20000,
            "steps": rng.choice([100, 150, 200])}


# ------------------------------------------------------------------ systems

def _params(model, two_types, under=False):
    p = S.params_reference() if model == "reference" else S.params_config()
    if two_types:
        # two bead kinds that fit the walks' 4 A spacing; the reference's well depths
        for i in (1, 2):
            for j in (1, 2):
                p.sigma_rep[i][j] = 3.8 + 0.1 * (i + j - 2)
                p.eps_att[i][j] = (1.0, 0.8, 0.7)[i + j - 2]
    if model == "reference":
        p.zeta = 0.05 if under else 50.0
        if under:
            p.h = 2.5e-3
    if under:
        p.dynamics = S._abi.DYN_UNDERDAMPED
    return p


def _chain_system(seed, n, params, two_types, T, key):
    s = S.make_chain_system(seed, n, params=params)
    rng = np.random.default_rng(seed)
    if two_types:
        s.type = rng.integers(1, 3, n).astype(np.int32)
    s.params.T = T
    s.params.seed = key
    if s.params.dynamics == S._abi.DYN_UNDERDAMPED:
        s.vel = rng.normal(0, math.sqrt(T), (n, 3)).astype(np.float32)
    return s


def _assembly(seed, chains, per, spacing=72.0):
    """Chains on a cubic lattice wider than a confined walk, each turned at random."""
    rng = np.random.default_rng(seed)
    g = math.ceil(chains ** (1.0 / 3.0))
    xs, bs, nis, njs, nrs = [], [], [], [], []
    for c in range(chains):
        x, b = S.generate_chain(seed * 1000003 + c, per)
        q, r = np.linalg.qr(rng.normal(size=(3, 3)))
        site = np.array((c % g, (c // g) % g, c // (g * g)), np.float64)
        x = ((x - x.mean(0)).astype(np.float64) @ (q * np.sign(np.diag(r))) + spacing * site).astype(np.float32)
        b = b.copy()
        b[:-1] = np.linalg.norm(x[1:].astype(np.float64) - x[:-1], axis=1)
        ni, nj, nr = S.native_contacts(x, None, 8.0)
        xs.append(x)
        bs.append(b)
        nis.append(ni + c * per)
        njs.append(nj + c * per)
        nrs.append(nr)
    p = S.params_config()
    p.seed = W.philox_key(5, seed)
    return S.System(xyz=np.concatenate(xs), params=p, chain=np.repeat(np.arange(chains, dtype=np.int32), per),
                    bond_r0=np.concatenate(bs), nat_i=np.concatenate(nis), nat_j=np.concatenate(njs),
                    nat_r0=np.concatenate(nrs))


def _systems(case, seed):
    seed = int(seed)
    rng = np.random.default_rng(seed)  # temperatures; the sizes are the case's own
    law = np.random.default_rng(17)
    kind = case["kind"]
    if kind == "assembly":
        return [_assembly(seed, case["chains"], case["per"])]
    if kind in ("evaluate", "lists"):
        return [_chain_system(seed, case["beads"], _params(case["model"], case["two_types"]), case["two_types"], 0.6,
                              W.philox_key(1, seed))]
    if kind == "serve":
        sizes = np.clip(np.round(np.exp(law.normal(math.log(case["median"]), 0.9, case["jobs"]))), 100, case["top"])
        p = _params("config", False)
        return [_chain_system(seed * 1000003 + k, int(n), p, False, float(rng.uniform(0.5, 0.9)),
                              W.philox_key(4, seed * 4096 + k)) for k, n in enumerate(sizes)]
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    sizes = np.round(np.exp(law.uniform(lo, hi, case["replicas"]) if hi > lo else np.full(case["replicas"], lo)))
    p = _params(case["model"], case["two_types"], case["under"])
    return [_chain_system(seed * 1000003 + k, int(n), p, case["two_types"], float(rng.uniform(0.5, 0.9)),
                          W.philox_key(3, seed * 4096 + k)) for k, n in enumerate(sizes)]


def _frames(s, seed, count=4):
    """Frames of a trajectory: the state with every bead moved by about 0.1 A."""
    rng = np.random.default_rng([int(seed), 23])
    return [s.xyz + rng.normal(0, 0.06, s.xyz.shape).astype(np.float32) for _ in range(count)]


def prepare(case, seed):
    systems = _systems(case, seed)
    eng = S.Engine(0)
    st = {"case": case, "eng": eng}
    if case["kind"] == "serve":
        st["systems"] = systems
        st["srv"] = Server(eng, hbm_budget_bytes=32 << 30)
        return st
    st["ids"] = [eng.add(s) for s in systems]
    if case["kind"] in ("evaluate", "lists"):
        st["frames"], st["next"] = _frames(systems[0], seed), 0
        st["held"] = {w: np.zeros((k * case["beads"], 2), np.int32)
                      for w, k in ((S.LIST_PL_REP, 96), (S.LIST_PL_NATIVE, 12))}
    return st


def run(state):
    case, eng = state["case"], state["eng"]
    if case["kind"] == "serve":
        srv = state["srv"]
        jobs = [srv.submit(s, case["steps"]) for s in state["systems"]]
        out = [srv.wait(j) for j in jobs]
        return {"xyz": np.concatenate([x for _, x in out]),
                "energies": np.array([r["energies"] for r, _ in out], np.float32),
                "status": np.array([r["status"] for r, _ in out])}
    ids = state["ids"]
    if case["kind"] in ("run", "assembly"):
        eng.run(ids, case["steps"])
        row = {"xyz": np.concatenate([eng.coords(i) for i in ids])}
        if case.get("sample"):
            # a trajectory row: single precision, as the state it belongs to
            row["energies"] = np.array([eng.energy_eval(i) for i in ids], np.float32)
            obs = [eng.observables(i) for i in ids]
            row["contacts"] = np.array([o[1] for o in obs])
            row["rgsq"] = np.array([o[2] for o in obs], np.float32)
        if case.get("under"):
            row["vel"] = np.concatenate([eng.velocities(i) for i in ids])
        return row
    i = ids[0]
    eng.set_coords(i, state["frames"][state["next"] % len(state["frames"])])
    state["next"] += 1
    eng.update_neighbor_list(i)
    eng.update_pair_list(i)
    if case["kind"] == "lists":
        for which in (S.LIST_PL_REP, S.LIST_PL_NATIVE):
            ij = eng.get_list(i, which)
            held = state["held"][which]  # the driver's own arrays, as long as its longest list
            held[:len(ij)] = ij
            held[len(ij):] = -1
        return dict(zip(("rep", "native"), state["held"].values()))
    q, contacts, rgsq = eng.observables(i)
    return {"forces": eng.force_eval(i), "energies": eng.energy_eval(i), "q": q, "contacts": contacts, "rgsq": rgsq}


# --------------------------------------------------------------------- work

def _within(n, rc):
    """Expected partners of a bead within rc in a ball of n beads at 140 A^3 each
    (the distribution of distances in a ball)."""
    s = min(rc / (3.0 * 140.0 * n / (4.0 * math.pi)) ** (1.0 / 3.0), 2.0)
    return (n - 1) * s ** 3 * (1.0 - 9.0 * s / 16.0 + s ** 3 / 32.0)


def _sizes(case):
    """(beads, how many) of the case's systems; a size law by its quantiles."""
    if case["kind"] == "assembly":
        return [(case["per"], case["chains"])]
    if case["kind"] in ("evaluate", "lists"):
        return [(case["beads"], 1)]
    q = [(k + 0.5) / 16 for k in range(16)]
    if case["kind"] == "serve":
        z = [-1.86, -1.32, -1.01, -0.78, -0.58, -0.40, -0.24, -0.08, 0.08, 0.24, 0.40, 0.58, 0.78, 1.01, 1.32, 1.86]
        return [(min(max(case["median"] * math.exp(0.9 * v), 100.0), case["top"]), case["jobs"] / 16) for v in z]
    return [(case["lo"] * (case["hi"] / case["lo"]) ** v, case["replicas"] / 16) for v in q]


def work(case):
    """Per step: coordinates in and out (24 B a bead), bond lengths (4), the
    native (8) and non-native (4) half lists, some 30 operations a pair and 150 a
    bead for noise and move.  Per list rebuild: coordinates, and the neighbor
    half list read and the pair half list written."""
    ref = case.get("model") == "reference"
    rc_nl, rc_pl = (12.2, 9.5) if ref else (32.0, 16.0)
    n_nl, n_pl = (50, 1) if ref else (50, 10)
    nbytes = flops = 0.0
    for n, count in _sizes(case):
        nat = 4.6 * n
        pl = max(n * _within(n, rc_pl) / 2 - nat, 0.0)
        nl = max(n * _within(n, rc_nl) / 2 - nat, 0.0)
        step = 28.0 * n + 8.0 * nat + 4.0 * pl
        pair_list = 12.0 * n + 8.0 * nat + 4.0 * nl + 8.0 * nat + 4.0 * pl
        neigh_list = 28.0 * n + 8.0 * nat + 4.0 * nl
        pair_ops = 30.0 * (pl + nat)
        if case["kind"] in ("evaluate", "lists"):
            b = neigh_list + pair_list + 12.0 * n + (8.0 * (pl + nat) if case["kind"] == "lists" else 2 * step)
            f = 10.0 * (nl + pl) + (0.0 if case["kind"] == "lists" else 2 * pair_ops)
        else:
            b = case["steps"] * (step + pair_list / n_pl + neigh_list / n_nl) + 12.0 * n
            f = case["steps"] * (pair_ops + 150.0 * n + 10.0 * pl / n_pl + 10.0 * nl / n_nl)
            if case.get("sample"):
                b += step
                f += pair_ops
        nbytes += count * b
        flops += count * f
    return {"bytes": nbytes, "flops": flops}


# -------------------------------------------------------------------- exact

def _normals(key, n, step, dev):
    """Three normals per bead: Philox4x32-10 (Salmon et al., SC'11) keyed by the
    system, counter (bead, step), and Box-Muller in 64 bits."""
    m = 0xFFFFFFFF
    c = [torch.arange(n, device=dev), torch.full((n,), step & m, device=dev),
         torch.full((n,), (step >> 32) & m, device=dev), torch.zeros(n, dtype=torch.int64, device=dev)]
    k0, k1 = key & m, key >> 32
    mul = lambda a, x: ((x >> 16) * a, (x & 0xFFFF) * a)  # noqa: E731  32x32 bits in two 48-bit products
    for _ in range(10):
        (h0, l0), (h1, l1) = mul(0xD2511F53, c[0]), mul(0xCD9E8D57, c[2])
        t0, t1 = (h0 & m) * 65536 + l0, (h1 & m) * 65536 + l1
        hi0, lo0 = ((h0 >> 32) * 65536 + (t0 >> 32)) & m, t0 & m
        hi1, lo1 = ((h1 >> 32) * 65536 + (t1 >> 32)) & m, t1 & m
        c = [hi1 ^ c[1] ^ k0, lo1, hi0 ^ c[3] ^ k1, lo0]
        k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
    u = [((v >> 8) | 1).double() * 2.0 ** -24 for v in c]
    ra, rb = torch.sqrt(-2 * torch.log(u[0])), torch.sqrt(-2 * torch.log(u[2]))
    return torch.stack([ra * torch.cos(2 * math.pi * u[1]), ra * torch.sin(2 * math.pi * u[1]),
                        rb * torch.cos(2 * math.pi * u[3])], 1)


class _Exact:
    """One system in 64 bits: lists by the single-precision predicate at the
    current coordinates, everything else in double."""

    def __init__(self, s, dev):
        t = lambda a, d=torch.float64: torch.as_tensor(np.array(a), device=dev).to(d)  # noqa: E731
        p = s.params
        self.p, self.dev, self.n = p, dev, s.n
        self.x = t(s.xyz)
        self.chain, self.type = t(s.chain, torch.int64), t(s.type, torch.int64) - 1
        self.r0 = t(s.bond_r0)
        self.ni, self.nj, self.nr = t(s.nat_i, torch.int64), t(s.nat_j, torch.int64), t(s.nat_r0)
        self.nat_key = torch.sort(self.ni * s.n + self.nj).values
        tab = lambda f: t([[float(f(i, j)) for j in (1, 2)] for i in (1, 2)])  # noqa: E731
        self.ea, self.er = tab(lambda i, j: p.eps_att[i][j]), tab(lambda i, j: p.eps_rep[i][j])
        self.sg = tab(lambda i, j: p.sigma_rep[i][j])
        cut = lambda b: np.float32(p.pl_factor * float(b)) if p.pl_factor > 0 else np.float32(p.pl_abs)  # noqa: E731
        self.rc2 = tab(lambda i, j: cut(p.sigma_rep[i][j]) ** 2).float()
        self.nrc2 = t([cut(b) ** 2 for b in np.asarray(s.nat_r0)], torch.float32).reshape(-1)
        self.cand = None
        self.step = int(s.step0)
        self.v = t(s.vel) if s.vel is not None else torch.zeros_like(self.x)
        self.a, self.incr = None, None

    def _d2(self, x, i, j):
        d = x[j] - x[i]
        d = d * d
        return (d[:, 0] + d[:, 1]) + d[:, 2]

    def _candidates(self):
        """Master pairs within the largest cutoff and 2 A, in row chunks."""
        x, n = self.x.float(), self.n
        reach = float(self.rc2.max().sqrt()) + 2.0
        got = []
        rows = max(1, min(n, (1 << 26) // n))
        for a in range(0, n, rows):
            d2 = torch.zeros((min(rows, n - a), n), device=self.dev)
            for k in range(3):
                d = x[a:a + rows, k:k + 1] - x[None, :, k]
                d2 += d * d
            i, j = (d2 < reach * reach).nonzero(as_tuple=True)
            i = i + a
            keep = (j > i) & ~((self.chain[i] == self.chain[j]) & (j - i <= 2))
            i, j = i[keep], j[keep]
            key = i * n + j
            if len(self.nat_key):
                at = torch.searchsorted(self.nat_key, key).clamp(max=len(self.nat_key) - 1)
                keep = self.nat_key[at] != key
                i, j = i[keep], j[keep]
            got.append(torch.stack([i, j]))
        self.cand = torch.cat(got, 1)

    def lists(self):
        if self.cand is None:
            self._candidates()
        x = self.x.float()
        i, j = self.cand
        keep = self._d2(x, i, j) < self.rc2[self.type[i], self.type[j]]
        self.pi, self.pj = i[keep], j[keep]
        self.nk = self._d2(x, self.ni, self.nj) < self.nrc2

    def forces(self):
        p, x, n = self.p, self.x, self.n
        f = torch.zeros_like(x)
        e = {}

        def add(i, j, d, c):
            f.index_add_(0, i, c[:, None] * d)
            f.index_add_(0, j, -c[:, None] * d)

        b = torch.arange(n - 1, device=self.dev)
        b = b[self.chain[b] == self.chain[b + 1]]
        d = x[b + 1] - x[b]
        r = d.norm(dim=1)
        dev = r - self.r0[b]
        g = 1 - dev ** 2 / p.R0 ** 2
        c = p.k_bnd * dev / (r * g)
        add(b, b + 1, d, c)
        vir = -(c * r * r).sum()
        e["bond"] = (-0.5 * p.k_bnd * p.R0 ** 2 * torch.log(g)).sum()
        b = torch.arange(max(n - 2, 0), device=self.dev)
        b = b[self.chain[b] == self.chain[b + 2]]
        d = x[b + 2] - x[b]
        d2 = (d * d).sum(1)
        w = p.eps_ss * p.sigma_ss ** 6 / d2 ** 3
        add(b, b + 2, d, -6 * w / d2)
        vir = vir + (6 * w).sum()
        e["ang"] = w.sum()
        i, j, r0 = self.ni[self.nk], self.nj[self.nk], self.nr[self.nk]
        d = x[j] - x[i]
        d2 = (d * d).sum(1)
        q6 = (r0 * r0 / d2) ** 3
        ep = self.ea[self.type[i], self.type[j]]
        c = -12 * ep * q6 * (q6 - 1) / d2
        add(i, j, d, c)
        vir = vir - (c * d2).sum()
        e["nat"] = (ep * (q6 * q6 - 2 * q6)).sum()
        i, j = self.pi, self.pj
        d = x[j] - x[i]
        d2 = (d * d).sum(1)
        ti, tj = self.type[i], self.type[j]
        q6 = (self.sg[ti, tj] ** 2 / d2) ** 3
        ep = self.er[ti, tj]
        c = -ep * q6 * (12 * p.rep_c12 * q6 + 6 * p.rep_c6) / d2
        add(i, j, d, c)
        vir = vir - (c * d2).sum()
        e["rep"] = (ep * (p.rep_c12 * q6 * q6 + p.rep_c6 * q6)).sum()
        tot = e["bond"] + e["ang"] + e["nat"] + e["rep"]
        return f, torch.stack([e["bond"], e["ang"], e["nat"], e["rep"], tot, vir])

    def noisy(self):
        p = self.p
        var = math.sqrt(2 * p.T * p.zeta / p.h)
        return self.forces()[0] + var * _normals(int(p.seed), self.n, self.step, self.dev)

    def velocity(self, f):
        p, hz = self.p, self.p.h * self.p.zeta
        if self.incr is None:
            return self.v
        return (1 - hz / 2 + hz * hz / 4) / p.h * self.incr + p.h / 2 * (1 - hz / 2) * f

    def run(self, steps):
        p, hz = self.p, self.p.h * self.p.zeta
        for _ in range(steps):
            if self.step % p.n_pl == 0 or self.step % p.n_nl == 0:
                self.lists()
            f = self.noisy()
            if p.dynamics == S._abi.DYN_UNDERDAMPED:
                self.incr = p.h * (1 - hz / 2) * self.velocity(f) + p.h * p.h / 2 * f
                self.x = self.x + self.incr
            else:
                self.x = self.x + p.h / p.zeta * f
            self.step += 1

    def rgsq(self):
        return float(((self.x - self.x.mean(0)) ** 2).sum(1).mean())


def exact(case, seed):
    if case["kind"] in ("lists", "serve"):
        return None  # lists are whole numbers; a job is a run
    if case["kind"] == "run" and case["replicas"] > 64:
        return None  # too many systems one after another
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    systems = _systems(case, seed)
    if case["kind"] == "evaluate":
        s = systems[0]
        s.xyz = _frames(s, seed)[0]
        m = _Exact(s, dev)
        m.lists()
        f, e = m.forces()
        return {"forces": f.cpu().numpy(), "energies": e.cpu().numpy(), "q": None, "contacts": None, "rgsq": m.rgsq()}
    row = {"xyz": [], "energies": [], "rgsq": [], "vel": []}
    for s in systems:
        m = _Exact(s, dev)
        m.run(case["steps"])
        row["xyz"].append(m.x.cpu().numpy())
        if case.get("sample"):
            row["energies"].append(m.forces()[1].cpu().numpy())
            row["rgsq"].append(m.rgsq())
        if case.get("under"):
            row["vel"].append(m.velocity(m.noisy()).cpu().numpy())
    out = {"xyz": np.concatenate(row["xyz"])}
    if case.get("sample"):
        # the energies after a run carry the rounding of its single-precision
        # coordinates: an error that averages over an ensemble, and the throw of
        # a die for the six numbers of one system (its energies at given
        # coordinates are what "evaluate" compares)
        energies = np.array(row["energies"]) if len(systems) >= 16 else None
        out.update(energies=energies, contacts=None, rgsq=np.array(row["rgsq"]))
    if case.get("under"):
        out["vel"] = np.concatenate(row["vel"])
    return out
