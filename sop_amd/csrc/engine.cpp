// engine.cpp -- libsop host engine: device pools, systems, batch work tables,
// hipGraph step blocks and the C ABI of include/sop.h (device part).
#include "engine.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <sstream>
#include <unordered_map>
#include <utility>

using namespace sopk;

namespace sopk {

// ---------------------------------------------------------------- allocator

void RangeAlloc::init(int64_t cap) {
  cap_ = cap;
  used_ = 0;
  free_.clear();
  if (cap > 0) free_[0] = cap;
}

int64_t RangeAlloc::alloc(int64_t n, int64_t align) {
  if (n <= 0) n = 1;
  for (auto it = free_.begin(); it != free_.end(); ++it) {
    const int64_t off = it->first, len = it->second;
    const int64_t a = (off + align - 1) / align * align;
    if (a + n > off + len) continue;
    free_.erase(it);
    if (a > off) free_[off] = a - off;
    if (a + n < off + len) free_[a + n] = off + len - (a + n);
    used_ += n;
    return a;
  }
  return -1;
}

void RangeAlloc::release(int64_t off, int64_t n) {
  if (n <= 0) n = 1;
  used_ -= n;
  auto it = free_.emplace(off, n).first;
  auto nx = std::next(it);
  if (nx != free_.end() && it->first + it->second == nx->first) {
    it->second += nx->second;
    free_.erase(nx);
  }
  if (it != free_.begin()) {
    auto pv = std::prev(it);
    if (pv->first + pv->second == it->first) {
      pv->second += it->second;
      free_.erase(it);
    }
  }
}

void RangeAlloc::grow(int64_t new_cap) {
  if (new_cap <= cap_) return;
  release(cap_, new_cap - cap_);
  used_ += new_cap - cap_;  // release() subtracted it
  cap_ = new_cap;
}

sop_status set_error(sop_engine *e, sop_status st, const std::string &msg) {
  if (e) e->err = msg;
  return st;
}

sop_status hip_check(sop_engine *e, hipError_t h, const char *what) {
  if (h == hipSuccess) return SOP_OK;
  return set_error(e, SOP_ERR_HIP, std::string(what) + ": " + hipGetErrorString(h));
}

int grid_tiles(const sop_engine *e) {
  int g = e->opts.grid_blocks > 0 ? e->opts.grid_blocks : 8 * e->num_cu;
  g = std::max(8, g / 8 * 8);
  if (e->fixed_grids) return g;
  const int need = (e->cur_nwork + 7) / 8 * 8;
  return std::max(8, std::min(g, need));
}

int grid_sys(const sop_engine *e) {
  if (e->fixed_grids) return 1024;
  return std::max(1, std::min(e->cur_nsys, 2048));
}

// k_rebuild: a block per system of up to SORT_N_MAX beads (one that sorts is
// resident per compute unit, two that only decide)
static int grid_rebuild(const sop_engine *e) {
  if (e->fixed_grids) return 2 * e->num_cu;
  return std::min(e->cur_nsys - e->cur_nbig, 2048);
}

// The larger systems' kernels: blocks of 2,048 beads of the largest one, and
// one per system.  While serving, fixed grids whenever the batch has one, by
// the largest one's size, so that a few captured graphs serve every batch: up
// to 32,768 beads (the size law of served streams) one, and two more above.
// Served alone, per step with 8 blocks of beads whatever the size, and now:
// 60,000 beads 31.4 / 30.0 us, 200,000 52.5 / 48.3, 500,000 116 / 102 (95 outside
// serving).
static int grid_big_beads(const sop_engine *e) {
  if (e->cur_nbig == 0) return 0;
  if (e->fixed_grids) return e->cur_big_max <= 32768 ? 8 : e->cur_big_max <= 131072 ? 64 : 256;
  return std::min((e->cur_big_max + 2047) / 2048, 4 * e->num_cu);
}
static int grid_big_sys(const sop_engine *e) {
  if (e->cur_nbig == 0) return 0;
  if (e->fixed_grids) return e->cur_big_max <= 32768 ? 64 : e->cur_big_max <= 131072 ? 32 : 16;
  return std::min(e->cur_nbig, 1024);
}

// Launch grid of a persistent item kernel: `g` blocks (a multiple of 8, so
// that item k runs on XCD k mod 8), fewer when the batch has fewer items, none
// when it has none; with fixed grids (serving) g or none, so that a few
// captured graphs serve every batch.
static int items_grid(int g, bool fixed, int count) {
  g = std::max(8, g / 8 * 8);
  if (count == 0) return 0;  // no launch
  if (fixed) return g;
  return std::max(8, std::min(g, (count + 7) / 8 * 8));
}

// The step kernel's LDS launch: `step_blocks`, by default four blocks per
// compute unit for a batch (about one block per item of a large batch: two
// are resident per unit and the dispatcher starts each on whichever unit
// frees first; A/B on one box, 512 replicas: 6.61e9 -> 6.90e9 bead-steps/s
// against two per unit) and two while serving (fixed grids).
// (A mixed launch four in either: its items may be more than are resident, and
// a block that took two would double the step.)
int default_step_blocks(const sop_engine *e) { return (e->fixed_grids && !e->cur_mixed ? 2 : 4) * e->num_cu; }

int grid_items(const sop_engine *e) {
  return items_grid(e->step_blocks > 0 ? e->step_blocks : default_step_blocks(e), e->fixed_grids,
                    e->cur_nitems + (e->cur_mixed ? e->cur_nitems_far : 0));
}

int grid_items_far(const sop_engine *e) { return items_grid(2 * e->num_cu, e->fixed_grids, e->cur_nitems_far); }
// A block per tile; while serving a fixed grid whenever the batch has such
// tiles (two five-wave blocks of k_step_tile are resident per compute unit, one
// of nine waves, one of k_filter_tile; a block takes the rest in turn).
int grid_step_tiles(const sop_engine *e) {
  if (e->cur_ntiles == 0) return 0;
  return e->fixed_grids ? 4 * e->num_cu : e->cur_ntiles;
}

// Whole-CU LDS items: one block per compute unit (the block takes all of
// the unit's LDS).
static int items_grid_big(const sop_engine *e, int count) { return items_grid(e->num_cu, e->fixed_grids, count); }
int grid_items_big(const sop_engine *e) { return items_grid_big(e, e->cur_nitems_big); }

StepGrids step_grids(const sop_engine *e) {
  if (e->cur_mixed) return StepGrids{grid_items(e), 0, 0, e->cur_lds, 0, 0, true};
  return StepGrids{grid_items(e), grid_items_big(e), grid_items_far(e), e->cur_lds, e->cur_lds_big, grid_step_tiles(e), false};
}

// The shell filter's LDS launch: one block per item (a block leaves its
// compute unit after each item, so the cell-grid chain on the other stream
// finds units between the items); fixed grids (serving) as the step kernel's.
StepGrids filter_grids(const sop_engine *e) {
  const int g = e->step_blocks > 0 ? e->step_blocks : default_step_blocks(e);
  return StepGrids{items_grid(e->fixed_grids ? g : std::max(g, 8 * e->num_cu), e->fixed_grids, e->cur_nfitems),
                   items_grid_big(e, e->cur_nfitems_big),
                   items_grid(2 * e->num_cu, e->fixed_grids, e->cur_nfitems_far), e->cur_flds, e->cur_flds_big, grid_step_tiles(e), false};
}

ListGrids list_grids(const sop_engine *e) {
  // two streams when several systems, some built from the grid and some from
  // their shell rows, give the filter a quarter of the device's compute units
  // or more
  const bool split = e->cur_nsys > 1 && 4 * (e->cur_nfitems + e->cur_nfitems_big + e->cur_nfitems_far) > e->num_cu;
  return ListGrids{grid_tiles(e), std::min(16 * e->cur_nwork, 8 * e->num_cu), grid_rebuild(e), grid_big_beads(e), grid_big_sys(e), split, filter_grids(e)};
}

} // namespace sopk

#define HIPCK(expr)                                            \
  do {                                                         \
    sop_status _s = hip_check(e, (expr), #expr);               \
    if (_s != SOP_OK) return _s;                               \
  } while (0)

// ----------------------------------------------------------------- pools

static void bind_arrays(sop_engine *e) {
  DevPtrs &p = e->p;
  e->bead_arrays = {
      {(void **)&p.pos0, 16},      {(void **)&p.pos1, 16},       {(void **)&p.bond_r0, 4},
      {(void **)&p.pos_ref, 16},   {(void **)&p.pos_sorted, 16},
      {(void **)&p.nat_start, 4},  {(void **)&p.nat_cnt, 4},     {(void **)&p.nlatt_cnt, 4},
      {(void **)&p.platt_cnt, 4},  {(void **)&p.nlrep_cnt, 4},   {(void **)&p.plrep_cnt, 4},
      {(void **)&p.cell_of, 4},    {(void **)&p.cell_tmp, 4},    {(void **)&p.cell_sorted, 4},
      {(void **)&p.cell_pos, 4},   {(void **)&p.nat_sorted, 8},
      {(void **)&p.fout, 16},      {(void **)&p.vel, 16},
      {(void **)&p.tile_ord, 1},   {(void **)&p.slrep_cnt, 4},   {(void **)&p.pos_shell, 16},
      {(void **)&p.plrep_off, 4},  {(void **)&p.platt_off, 4},  {(void **)&p.plhead, 8}};
  e->nat_arrays = {{(void **)&p.nat_j, 4},    {(void **)&p.nat_r0, 4},  {(void **)&p.nlatt_j, 4},
                   {(void **)&p.nlatt_r0, 4}, {(void **)&p.platt, 8}};
  e->cell_arrays = {{(void **)&p.cell_cnt, 4}, {(void **)&p.cell_start, 4}, {(void **)&p.cell_cursor, 4},
                    {(void **)&p.cellitems, 8}};
}

static sop_status grow_array(sop_engine *e, void **ptr, size_t old_bytes, size_t new_bytes) {
  void *np = nullptr;
  HIPCK(hipMalloc(&np, std::max<size_t>(new_bytes, 256)));
  if (*ptr && old_bytes) HIPCK(hipMemcpy(np, *ptr, old_bytes, hipMemcpyDeviceToDevice));
  if (*ptr) HIPCK(hipFree(*ptr));
  *ptr = np;
  return SOP_OK;
}

namespace sopk {
// Pinned host memory of at least `bytes` (the stream is idle when it moves).
sop_status engine_io(sop_engine *e, HostBuf &b, size_t bytes) {
  if (b.bytes >= bytes) return SOP_OK;
  HIPCK(hipStreamSynchronize(e->stream));
  const size_t half = std::min(bytes / 2, (size_t)16 << 20);  // room for somewhat larger calls
  const size_t nb = std::max<size_t>(bytes + half, (size_t)64 << 10);
  void *q = nullptr;
  HIPCK(hipHostMalloc(&q, nb, hipHostMallocDefault));
  if (b.ptr) (void)hipHostFree(b.ptr);
  b.ptr = q;
  b.bytes = nb;
  return SOP_OK;
}
} // namespace sopk

static void invalidate_graphs(sop_engine *e) {
  for (auto &kv : e->graphs) (void)hipGraphExecDestroy(kv.second);
  e->graphs.clear();
}

// Grow pools so that the requested extra capacity fits (doubling).
static sop_status ensure_capacity(sop_engine *e, int64_t beads, int64_t nat, int64_t nl, int64_t pl,
                                  int64_t cells, int64_t slots) {
  Pools &c = e->cap;
  bool changed = false;
  auto next = [](int64_t cur, int64_t need) {
    int64_t v = std::max<int64_t>(cur, 1);
    while (v < need) v *= 2;
    return v;
  };
  HIPCK(hipStreamSynchronize(e->stream));
  if (beads > c.beads) {
    const int64_t nb = next(c.beads, beads);
    for (auto &a : e->bead_arrays) {
      sop_status s = grow_array(e, a.first, a.second * (size_t)c.beads, a.second * (size_t)nb);
      if (s) return s;
    }
    sop_status s = grow_array(e, (void **)&e->p.tile_sys, 4 * (size_t)(c.beads / TILE), 4 * (size_t)(nb / TILE));
    if (s) return s;
    s = grow_array(e, (void **)&e->p.epart, 0, 8 * TPART_N * (size_t)(nb / TILE));  // scratch of a call
    if (s) return s;
    e->a_beads.grow(nb);
    c.beads = nb;
    changed = true;
  }
  if (nat > c.nat) {
    const int64_t nn = next(c.nat, nat);
    for (auto &a : e->nat_arrays) {
      sop_status s = grow_array(e, a.first, a.second * (size_t)c.nat, a.second * (size_t)nn);
      if (s) return s;
    }
    e->a_nat.grow(nn);
    c.nat = nn;
    changed = true;
  }
  if (nl > c.nl) {
    const int64_t nn = next(c.nl, nl);
    sop_status s = grow_array(e, (void **)&e->p.nlrep_j, 4 * (size_t)c.nl, 4 * (size_t)nn);
    if (s) return s;
    c.nl = nn;
    changed = true;
  }
  if (pl > c.pl) {
    const int64_t nn = next(c.pl, pl);
    sop_status s = grow_array(e, (void **)&e->p.plrep_j, 4 * (size_t)c.pl, 4 * (size_t)nn);
    if (s) return s;
    s = grow_array(e, (void **)&e->p.slrep_j, 4 * (size_t)c.pl, 4 * (size_t)nn);
    if (s) return s;
    e->a_pl.grow(nn);
    c.pl = nn;
    changed = true;
  }
  if (cells > c.cells) {
    const int64_t nn = next(c.cells, cells);
    for (auto &a : e->cell_arrays) {
      sop_status s = grow_array(e, a.first, a.second * (size_t)c.cells, a.second * (size_t)nn);
      if (s) return s;
    }
    e->a_cells.grow(nn);
    c.cells = nn;
    changed = true;
  }
  if (slots > c.slots) {
    const int64_t nn = next(c.slots, slots);
    sop_status s = grow_array(e, (void **)&e->p.sys, sizeof(SysDev) * (size_t)c.slots, sizeof(SysDev) * (size_t)nn);
    if (s) return s;
    s = grow_array(e, (void **)&e->p.sysout, 8 * SYSOUT_N * (size_t)c.slots, 8 * SYSOUT_N * (size_t)nn);
    if (s) return s;
    s = grow_array(e, (void **)&e->p.syslist, 4 * (size_t)c.slots, 4 * (size_t)nn);
    if (s) return s;
    int4 *rep = nullptr;
    HIPCK(hipHostMalloc((void **)&rep, sizeof(int4) * (size_t)nn, hipHostMallocDefault));
    for (int64_t q = 0; q < nn; ++q) rep[q] = q < c.slots ? e->p.rep[q] : make_int4(0, 0, 0, 0);
    if (e->p.rep) (void)hipHostFree(e->p.rep);
    e->p.rep = rep;
    c.slots = nn;
    e->sys.resize((size_t)nn);
    changed = true;
  }
  if (changed) invalidate_graphs(e);
  return SOP_OK;
}

// Pool growth on demand: try to allocate, grow and retry once.
static int64_t alloc_or_grow(sop_engine *e, RangeAlloc &a, int64_t n, int64_t align, int which,
                             sop_status *st) {
  *st = SOP_OK;
  int64_t off = a.alloc(n, align);
  if (off >= 0) return off;
  if (e->fixed_pools) {
    *st = set_error(e, SOP_ERR_CAPACITY, "memory pool full");
    return -1;
  }
  const int64_t need = a.cap() + n + align;
  int64_t req[5] = {0, 0, 0, 0, 0};
  req[which] = need;
  *st = ensure_capacity(e, req[0], req[1], req[2], req[3], req[4], 0);
  if (*st) return -1;
  off = a.alloc(n, align);
  if (off < 0) *st = set_error(e, SOP_ERR_CAPACITY, "pool allocation failed after growth");
  return off;
}

// --------------------------------------------------------------- helpers

static float cutoff_host(double factor, float absval, float base) {
  return factor > 0.0 ? (float)(factor * (double)base) : absval;
}

static inline int32_t round_up(int32_t v, int32_t a) { return (v + a - 1) / a * a; }

// Row capacity of a system's shell rows and pair-list tiles (entries per
// bead): it starts at PL_CAP_START, is fitted to the longest row of the first
// build, and grows when a rebuild's longest row comes within an eighth of it,
// up to min(n - 1, pl_cap_max).  Growth moves the rows and changes no result.
constexpr int32_t PL_CAP_START = 384;

static int32_t pl_cap_limit(const sop_engine *e, int32_t n) {
  return round_up(std::max(1, std::min(n - 1, e->opts.pl_cap_max)), 16);
}
static int32_t pl_cap_start(const sop_engine *e, int32_t n) { return std::min(pl_cap_limit(e, n), PL_CAP_START); }
static int32_t pl_cap_target(const sop_engine *e, int32_t n, int32_t longest) {
  return std::min(pl_cap_limit(e, n), round_up(longest + longest / 4 + 32, 16));
}
static bool pl_cap_short(const sop_engine *e, const SysHost &h, int32_t longest) {
  return h.pl_cap < pl_cap_limit(e, h.n) && longest > h.pl_cap - h.pl_cap / 8;
}

namespace sopk {

// Pair-list shell of a system: rows within rc_pl + shell of pos_shell, valid
// while 2 max|x - pos_shell| < shell_ok (the shell less a 1e-4 margin, so the
// rounding of the shell cutoffs cannot matter); shell 0: no shell rows.  The
// rows are rebuilt from the cell grid at the next pair-list rebuild.
void shell_fields(const sop_params &P, float shell, SysDev &S) {
  float max_rcp = 0.0f;
  for (int q = 0; q < 4; ++q) {
    const int ti = q / 2 + 1, tj = q % 2 + 1;
    max_rcp = std::max(max_rcp, cutoff_host(P.pl_factor, P.pl_abs, P.sigma_rep[ti][tj]));
  }
  S.shell_ok = shell * (1.0f - 1.0e-4f);
  for (int q = 0; q < 4; ++q) {
    const int ti = q / 2 + 1, tj = q % 2 + 1;
    const double rs = (double)cutoff_host(P.pl_factor, P.pl_abs, P.sigma_rep[ti][tj]) + (double)shell;
    S.rc2_sl_rep[q] = (float)(rs * rs);
  }
  S.cell_min_edge_sl = std::max(1.0e-3f, (max_rcp + shell) * 1.001f);
  S.sl_valid = 0;
}

// Size bucket of a system of n beads in the tuned table (-1: none).
int engine_bucket(const sop_engine *e, int32_t n) {
  for (int b = 0; b < e->tune.nb; ++b)
    if (n <= e->tune.max_beads[b] || b == e->tune.nb - 1) return b;
  return -1;
}

float engine_shell_for(const sop_engine *e, int32_t n) {
  const int b = engine_bucket(e, n);
  return b >= 0 ? e->tune.shell[b] : e->opts.pl_shell;
}

sop_status engine_read_sys(sop_engine *e, int32_t slot, SysDev *out) {
  HIPCK(hipMemcpyAsync(out, e->p.sys + slot, sizeof(SysDev), hipMemcpyDeviceToHost, e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  return SOP_OK;
}

// Pool bytes of `beads` beads (whole tiles) and `cells` cells: the per-bead and
// per-cell arrays, and a tile's system slot and energy partials.
static int64_t pool_bytes(const sop_engine *e, int64_t beads, int64_t cells) {
  int64_t per_bead = 0, per_cell = 0;
  for (const auto &a : e->bead_arrays) per_bead += (int64_t)a.second;
  for (const auto &a : e->cell_arrays) per_cell += (int64_t)a.second;
  return beads * per_bead + beads / TILE * (4 + 8 * TPART_N) + cells * per_cell;
}

int64_t job_bytes_estimate(const sop_engine *e, const sop_system_desc *d) {
  const int64_t n = d->n_beads;
  const int64_t pl_cap = pl_cap_start(e, d->n_beads);
  const int64_t beads = (n + TILE - 1) / TILE * TILE;
  const int64_t cell_cap = std::min<int64_t>(e->opts.cell_cap_max, std::max<int64_t>(64, 2 * n)) + 1;
  // pair-list and shell-row segments (16-bit entries up to 65,536 beads); the
  // neighbor list is materialized only on request, in a scratch segment
  const int64_t esz = n <= 65536 ? 2 : 4;
  return pool_bytes(e, beads, cell_cap) + 24 * 2 * (int64_t)d->n_native + 2 * esz * n * pl_cap;
}

sop_status upload_drain(sop_engine *e, Upload *upl) {
  HIPCK(hipStreamSynchronize(upl->stream));
  upl->used = 0;
  return SOP_OK;
}

// Validate and upload one system, without its first lists (engine_init_lists).
sop_status engine_add_system_nolists(sop_engine *e, const sop_system_desc *d, int64_t step_end, int32_t *slot_out,
                                     Upload *upl) {
  const EngineLock lk(e->mu);
  hipStream_t up = upl ? upl->stream : nullptr;
  if (!d || d->n_beads < 1 || !d->xyz) return set_error(e, SOP_ERR_INVALID, "system: need n_beads >= 1 and xyz");
  const int32_t n = d->n_beads;
  const sop_params &P = d->params;
  if (P.n_nl < 1 || P.n_pl < 1) return set_error(e, SOP_ERR_INVALID, "n_nl and n_pl must be >= 1");
  if (P.dynamics != SOP_DYN_OVERDAMPED && P.dynamics != SOP_DYN_UNDERDAMPED)
    return set_error(e, SOP_ERR_INVALID, "dynamics must be SOP_DYN_OVERDAMPED or SOP_DYN_UNDERDAMPED");
  const bool under = P.dynamics == SOP_DYN_UNDERDAMPED;
  if (!(under ? P.zeta >= 0.0f : P.zeta > 0.0f) || !(P.h > 0.0f) || !(P.T >= 0.0f) || !(P.R0 > 0.0f))
    return set_error(e, SOP_ERR_INVALID, "need zeta > 0 (>= 0 underdamped), h > 0, T >= 0, R0 > 0");
  if (!(P.nl_factor > 0.0) && !(P.nl_abs > 0.0f)) return set_error(e, SOP_ERR_INVALID, "neighbor-list cutoff");
  if (!(P.pl_factor > 0.0) && !(P.pl_abs > 0.0f)) return set_error(e, SOP_ERR_INVALID, "pair-list cutoff");
  // chains and types
  std::vector<int32_t> chain(n, 0), type(n, 1);
  for (int i = 0; i < n; ++i) {
    if (d->chain) chain[i] = d->chain[i];
    if (d->type) type[i] = d->type[i];
    if (type[i] != 1 && type[i] != 2) return set_error(e, SOP_ERR_INVALID, "bead types must be 1 or 2");
    if (chain[i] < 0 || chain[i] >= (1 << 28)) return set_error(e, SOP_ERR_INVALID, "chain id out of range");
    if (i > 0 && chain[i] < chain[i - 1]) return set_error(e, SOP_ERR_INVALID, "chain ids must be non-decreasing");
  }
  // natives: validate, two-sided CSR sorted by partner
  const int32_t nn = d->n_native;
  if (nn < 0 || (nn > 0 && (!d->nat_i || !d->nat_j || !d->nat_r0)))
    return set_error(e, SOP_ERR_INVALID, "native arrays");
  std::vector<int32_t> nstart((size_t)n + 1, 0);
  for (int k = 0; k < nn; ++k) {
    const int i = d->nat_i[k], j = d->nat_j[k];
    if (i < 0 || j < 0 || i >= n || j >= n || i >= j)
      return set_error(e, SOP_ERR_INVALID, "native pair must satisfy 0 <= i < j < n");
    if (chain[i] == chain[j] && j - i <= 2)
      return set_error(e, SOP_ERR_INVALID, "native pair inside the |i-j| <= 2 exclusion");
    if (!(d->nat_r0[k] > 0.0f)) return set_error(e, SOP_ERR_INVALID, "native r0 must be > 0");
    ++nstart[(size_t)i + 1];
    ++nstart[(size_t)j + 1];
  }
  for (int i = 0; i < n; ++i) nstart[(size_t)i + 1] += nstart[i];
  std::vector<std::pair<int32_t, float>> nat((size_t)2 * nn);
  {
    // pairs sorted by (i, j) come out sorted by partner
    std::vector<int32_t> at(nstart.begin(), nstart.end() - 1);
    for (int k = 0; k < nn; ++k) {
      const int i = d->nat_i[k], j = d->nat_j[k];
      nat[(size_t)at[i]++] = {j, d->nat_r0[k]};
      nat[(size_t)at[j]++] = {i, d->nat_r0[k]};
    }
  }
  for (int i = 0; i < n; ++i) {
    const auto lo = nat.begin() + nstart[i], hi = nat.begin() + nstart[(size_t)i + 1];
    if (!std::is_sorted(lo, hi)) std::sort(lo, hi);
    for (auto q = lo; q < hi; ++q)
      if (q > lo && q->first == (q - 1)->first) return set_error(e, SOP_ERR_INVALID, "duplicate native pair");
    if (hi - lo > 65535) return set_error(e, SOP_ERR_CAPACITY, "more than 65535 native partners of one bead");
  }
  // the step kernel holds a native list's offset within its tile's native
  // slots in 16 bits
  for (int t0 = 0; t0 < n; t0 += TILE)
    if (nstart[std::min(n, t0 + TILE)] - nstart[t0] > 65535)
      return set_error(e, SOP_ERR_CAPACITY, "more than 65535 native partners in one 64-bead tile");
  // capacities
  const int32_t nl_cap = round_up(std::max(1, std::min(n - 1, e->opts.nl_cap_max)), 16);
  const int32_t pl_cap = pl_cap_start(e, n);
  // the step kernel addresses a system's pair-list rows with 32-bit byte
  // offsets, at any capacity they may grow to
  if ((int64_t)n * pl_cap_limit(e, n) * (n <= 65536 ? 2 : 4) > (int64_t)0xFFFFFFFF)
    return set_error(e, SOP_ERR_CAPACITY, "system's pair-list rows exceed 4 GiB (lower pl_cap_max)");
  const int32_t cell_cap = std::min(e->opts.cell_cap_max, std::max(64, 2 * n));
  int32_t dmax = 1;
  while ((int64_t)(dmax + 1) * (dmax + 1) * (dmax + 1) <= cell_cap) ++dmax;
  SysHost h;
  h.used = true;
  h.n = n;
  h.n_nat = nn;
  h.bead_len = round_up(n, TILE);
  h.nat_len = std::max(1, 2 * nn);
  h.nl_len = (int64_t)n * nl_cap;  // entries when materialized (scratch)
  h.pl_len = (int64_t)n * pl_cap / (n <= 65536 ? 2 : 1);  // 32-bit words: 16-bit entries pack two a word
  h.cell_len = cell_cap + 1;
  h.nl_cap = nl_cap;
  h.pl_cap = pl_cap;
  h.cell_cap = cell_cap;
  h.step = d->step0;
  h.parity = 0;
  h.params = P;
  // the upload: one pinned blob that a kernel unpacks (a copy from pageable
  // memory would wait for the engine stream)
  AddSystem up_a{};
  uint32_t words = 0;
  auto part = [&](uint32_t &off, size_t w) {
    off = words;
    words += (uint32_t)((w + 15) / 16 * 16);
  };
  part(up_a.xyz, 3 * (size_t)n);
  part(up_a.wbits, (size_t)n);
  part(up_a.bond, (size_t)n);
  part(up_a.nstart, (size_t)n + 1);
  part(up_a.natj, 2 * (size_t)nn);
  part(up_a.natr, 2 * (size_t)nn);
  part(up_a.vel, d->vel ? 3 * (size_t)n : 0);
  part(up_a.sys, sizeof(SysDev) / 4);
  const size_t stage_need = 4 * (size_t)words;
  if (up && stage_need > upl->stage_bytes) return SOP_ERR_BUSY;
  sop_status st;
  // with an upload stream, free ranges only: growing a pool reallocates
  // arrays that work in flight on the engine stream may be using
  auto alloc = [&](RangeAlloc &a, int64_t len, int64_t align, int which) -> int64_t {
    if (!up) return alloc_or_grow(e, a, len, align, which, &st);
    const int64_t off = a.alloc(len, align);
    st = off < 0 ? SOP_ERR_BUSY : SOP_OK;
    return off;
  };
  // ranges taken so far, given back by every return before the system exists
  struct Held {
    std::vector<std::pair<RangeAlloc *, std::pair<int64_t, int64_t>>> ranges;
    ~Held() {
      for (const auto &r : ranges) r.first->release(r.second.first, r.second.second);
    }
  } held;
  auto take = [&](RangeAlloc &a, int64_t len, int64_t align, int which, int64_t &off) {
    off = alloc(a, len, align, which);
    if (!st) held.ranges.push_back({&a, {off, len}});
    return st;
  };
  if (take(e->a_beads, h.bead_len, TILE, 0, h.bead_off)) return st;
  if (take(e->a_nat, h.nat_len, 1, 1, h.nat_off)) return st;
  if ((h.nat_off + h.nat_len) * 8 > (int64_t)0xFFFFFFFF)  // 32-bit byte offsets of the native pair list
    return set_error(e, SOP_ERR_CAPACITY, "native pool beyond 4 GiB");
  h.nl_off = 0;
  if (take(e->a_pl, h.pl_len, 16, 3, h.pl_off)) return st;
  if (take(e->a_cells, h.cell_len, 1, 4, h.cell_off)) return st;
  // slot
  int32_t slot = -1;
  for (size_t s = 0; s < e->sys.size(); ++s)
    if (!e->sys[s].used) { slot = (int32_t)s; break; }
  if (slot < 0 && up) return SOP_ERR_BUSY;
  if (slot < 0) {
    if (e->fixed_pools && (int64_t)e->sys.size() >= e->cap.slots && e->cap.slots > 0) {
      slot = -1;
    } else {
      const int64_t want = e->cap.slots + 1;
      st = ensure_capacity(e, 0, 0, 0, 0, 0, want);
      if (st) return st;
      for (size_t s = 0; s < e->sys.size(); ++s)
        if (!e->sys[s].used) { slot = (int32_t)s; break; }
    }
    if (slot < 0) return set_error(e, SOP_ERR_CAPACITY, "no free system slot");
  }
  const int64_t b0 = h.bead_off;
  if (up) {
    if (upl->used + stage_need > upl->stage_bytes && (st = upload_drain(e, upl))) return st;
  } else {
    HIPCK(hipStreamSynchronize(e->stream));  // the launch that read the staging buffer last has passed
    if ((st = engine_io(e, e->stage, stage_need))) return st;
  }
  uint32_t *blob = reinterpret_cast<uint32_t *>(up ? static_cast<char *>(upl->stage) + upl->used
                                                   : static_cast<char *>(e->stage.ptr));
  std::memcpy(blob + up_a.xyz, d->xyz, 12 * (size_t)n);
  std::memcpy(blob + up_a.nstart, nstart.data(), 4 * nstart.size());
  if (d->vel) std::memcpy(blob + up_a.vel, d->vel, 12 * (size_t)n);
  for (int i = 0; i < n; ++i) {
    const float r0 = d->bond_r0 ? d->bond_r0[i] : 3.8f;
    blob[up_a.wbits + i] = (uint32_t)((chain[i] << 2) | type[i]);
    std::memcpy(blob + up_a.bond + i, &r0, 4);
  }
  for (size_t k = 0; k < nat.size(); ++k) {
    blob[up_a.natj + k] = (uint32_t)nat[k].first;
    std::memcpy(blob + up_a.natr + k, &nat[k].second, 4);
  }
  SysDev S;
  // device descriptor
  std::memset(&S, 0, sizeof(S));
  S.bead_off = (int32_t)b0;
  S.n = n;
  S.nl_cap = nl_cap;
  S.pl_cap = pl_cap;
  S.idx16 = n <= 65536 ? 1 : 0;
  S.nl_base = 0;  // the neighbor-list scratch, when materialized
  S.pl_base = h.pl_off;
  S.cell_base = (int32_t)h.cell_off;
  S.cell_cap = cell_cap;
  S.dmax = dmax;
  S.parity = 0;
  S.step = d->step0;
  S.step_end = step_end > d->step0 ? step_end : d->step0;
  S.n_nl = P.n_nl;
  S.n_pl = P.n_pl;
  float a5, var;
  sop_params_derived(&P, &a5, &var);
  S.a5 = a5;
  S.dyn = under ? 1 : 0;
  S.vupd = P.T >= 1.0e-5f ? 1 : 0;  // sop.cu:475 (no velocity update for steepest descent)
  {
    float a[4];
    sop_params_underdamped(&P, a);
    S.a1 = a[0];
    S.a2 = a[1];
    S.a3 = a[2];
    S.a4 = a[3];
  }
  S.var = var;
  S.boxl = P.boxl;
  S.inv_boxl = P.boxl > 0.0f ? 1.0f / P.boxl : 0.0f;
  S.seed_lo = (uint32_t)P.seed;
  S.seed_hi = (uint32_t)(P.seed >> 32);
  S.k_bnd = P.k_bnd;
  S.inv_R0sq = 1.0f / (P.R0 * P.R0);
  S.half_k_R0sq = 0.5f * P.k_bnd * P.R0 * P.R0;
  const double s6 = std::pow((double)P.sigma_ss, 6.0);
  S.ss_e6 = (float)((double)P.eps_ss * s6);
  S.ss_f6 = (float)(6.0 * (double)P.eps_ss * s6);
  float max_rc = 0.0f;
  for (int ti = 1; ti <= 2; ++ti)
    for (int tj = 1; tj <= 2; ++tj) {
      const int q = (ti - 1) * 2 + (tj - 1);
      const float sg = P.sigma_rep[ti][tj], ep = P.eps_rep[ti][tj];
      S.eps_att[q] = P.eps_att[ti][tj];
      S.eps_rep[q] = ep;
      S.sig2_rep[q] = sg * sg;
      S.rep_guard[q] = sg * 1.0e-7f;
      S.rep_m12[q] = -12.0f * ep * P.rep_c12;
      S.rep_m6[q] = -6.0f * ep * P.rep_c6;
      const double s6q = std::pow((double)S.sig2_rep[q], 3.0);
      S.rep_a[q] = (float)((double)S.rep_m12[q] * s6q * s6q);
      S.rep_b[q] = (float)((double)S.rep_m6[q] * s6q);
      const float rn = cutoff_host(P.nl_factor, P.nl_abs, sg);
      const float rp = cutoff_host(P.pl_factor, P.pl_abs, sg);
      S.rc2_nl_rep[q] = rn * rn;
      S.rc2_pl_rep[q] = rp * rp;
      max_rc = std::max(max_rc, rn);
    }
  S.c12 = P.rep_c12;
  S.c6 = P.rep_c6;
  S.nl_factor = P.nl_factor;
  S.pl_factor = P.pl_factor;
  S.nl_abs = P.nl_abs;
  S.pl_abs = P.pl_abs;
  S.cell_min_edge = std::max(1.0e-3f, max_rc * 1.001f);
  // pair-list grid and list skin (the direct pair-list build is exact while
  // every bead stays within skin/2 of its neighbor-list snapshot)
  float skin = INFINITY;
  for (int q = 0; q < 4; ++q) {
    const int ti = q / 2 + 1, tj = q % 2 + 1;
    const float sg = P.sigma_rep[ti][tj];
    const float rn = cutoff_host(P.nl_factor, P.nl_abs, sg), rp = cutoff_host(P.pl_factor, P.pl_abs, sg);
    skin = std::min(skin, rn - rp);
  }
  for (int k = 0; k < nn; ++k) {
    const float r0 = d->nat_r0[k];
    skin = std::min(skin, cutoff_host(P.nl_factor, P.nl_abs, r0) - cutoff_host(P.pl_factor, P.pl_abs, r0));
  }
  S.skin = skin > 0.0f ? skin * (1.0f - 1.0e-5f) : 0.0f;
  h.shell = engine_shell_for(e, n);
  shell_fields(P, h.shell, S);
  S.build = BUILD_NONE;
  for (int k = 0; k < 8; ++k) S.acc[k] = k < 3 ? ACC_MIN : ACC_MAX;
  S.nl_valid = 0;
  int tmask = 0;
  for (int i = 0; i < n; ++i) tmask |= 1 << (type[i] - 1);
  S.type_mask = tmask;
  S.wrap_margin = 10.0f;
  S.dims[0] = S.dims[1] = S.dims[2] = 1;
  S.ncells = 1;
  S.wrap_free = 0;
  std::memcpy(blob + up_a.sys, &S, sizeof(SysDev));
  up_a.blob = blob;
  up_a.bead_off = (int32_t)b0;
  up_a.bead_len = (int32_t)h.bead_len;
  up_a.n = n;
  up_a.nat_off = (int32_t)h.nat_off;
  up_a.n_nat = 2 * nn;
  up_a.slot = slot;
  up_a.has_vel = d->vel ? 1 : 0;
  HIPCK(launch_add_system(e->p, up_a, up ? up : e->stream));
  if (up) upl->used += (stage_need + 255) / 256 * 256;
  held.ranges.clear();  // the system's own from here on
  e->sys[slot] = std::move(h);
  *slot_out = slot;
  return SOP_OK;
}

static sop_status read_sys_all(sop_engine *e, std::vector<SysDev> &sd) {
  sd.resize((size_t)e->cap.slots);
  HIPCK(hipMemcpy(sd.data(), e->p.sys, sizeof(SysDev) * sd.size(), hipMemcpyDeviceToHost));
  return SOP_OK;
}

// Resident bytes of one system (what job_bytes_estimate predicts for it).
int64_t engine_system_bytes(const sop_engine *e, int32_t slot) {
  const SysHost &h = e->sys[slot];
  return pool_bytes(e, h.bead_len, h.cell_len) + 24 * 2 * (int64_t)h.n_nat + 2 * 4 * h.pl_len;
}

// Move one system's shell rows and pair-list tiles to a segment of row
// capacity cap: with keep, the current rows are copied over (k_relayout);
// otherwise the caller builds them again.  Leaves the engine stream idle.
sop_status engine_resize_rows(sop_engine *e, int32_t slot, int32_t cap, bool keep) {
  SysHost &h = e->sys[slot];
  if (cap == h.pl_cap) return SOP_OK;
  const bool i16 = h.n <= 65536;
  const int64_t len = (int64_t)h.n * cap / (i16 ? 2 : 1);
  sop_status st = SOP_OK;
  const int64_t off = alloc_or_grow(e, e->a_pl, len, 16, 3, &st);
  if (st) return st;
  if (keep)
    HIPCK(launch_relayout(e->p, (int)h.bead_off, h.n, i16 ? 1 : 0, h.pl_off, h.pl_cap, off, cap, e->stream));
  const int64_t base = off;
  const int32_t c32 = cap, zero = 0;
  HIPCK(hipMemcpyAsync(&e->p.sys[slot].pl_base, &base, sizeof(base), hipMemcpyHostToDevice, e->stream));
  HIPCK(hipMemcpyAsync(&e->p.sys[slot].pl_cap, &c32, sizeof(c32), hipMemcpyHostToDevice, e->stream));
  if (!keep)  // no shell rows to filter: the next pair-list build comes from the cell grid
    HIPCK(hipMemcpyAsync(&e->p.sys[slot].sl_valid, &zero, sizeof(zero), hipMemcpyHostToDevice, e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  e->a_pl.release(h.pl_off, h.pl_len);
  h.pl_off = off;
  h.pl_len = len;
  h.pl_cap = cap;
  return SOP_OK;
}

// Systems whose longest row came within an eighth of their row capacity get
// a larger one; their rows move and no result changes.  With fixed pools a
// capacity that finds no room stays as it is (a row that outgrows it is
// reported as an overflow).  The engine stream must be idle; row_max[q] is the
// longest row of slots[q] so far.  *grown receives each system's added bytes.
sop_status engine_grow_rows(sop_engine *e, const int32_t *slots, int32_t n, const int32_t *row_max,
                            std::vector<int64_t> *grown) {
  if (grown) grown->assign((size_t)n, 0);
  if (!e->grow_rows) return SOP_OK;
  for (int32_t q = 0; q < n; ++q) {
    const int32_t s = slots[q];
    const SysHost &h = e->sys[s];
    const int32_t m = row_max[q];
    if (!pl_cap_short(e, h, m)) continue;
    const int64_t before = engine_system_bytes(e, s);
    const sop_status st = engine_resize_rows(e, s, pl_cap_target(e, h.n, m), true);
    if (st == SOP_ERR_CAPACITY && e->fixed_pools) continue;
    if (st) return st;
    if (grown) (*grown)[q] = engine_system_bytes(e, s) - before;
  }
  return SOP_OK;
}

// Before a system's shell widens to `shell`: a row capacity that the longest
// row so far, scaled by the volume of the wider shell (and a tenth more),
// would come within an eighth of grows now (rows moved, results unchanged),
// so the first rebuild with the new shell does not overflow.
sop_status engine_fit_shell(sop_engine *e, int32_t slot, float shell) {
  SysHost &h = e->sys[slot];
  if (!(shell > h.shell)) return SOP_OK;
  SysDev S;
  sop_status st = engine_read_sys(e, slot, &S);
  if (st) return st;
  float rc2 = 0.0f;
  for (int q = 0; q < 4; ++q) rc2 = std::max(rc2, S.rc2_pl_rep[q]);
  const double rc = std::sqrt((double)rc2);
  const double ratio = (rc + shell) / (rc + h.shell);
  const int32_t m = (int32_t)std::ceil((double)S.row_max * ratio * ratio * ratio * 1.1);
  if (S.row_max <= 0 || !pl_cap_short(e, h, m)) return SOP_OK;
  return engine_resize_rows(e, slot, pl_cap_target(e, h.n, m), true);
}

// After the first lists of newly added systems: a system whose longest row
// overflowed its starting capacity or comes within an eighth of it gets the
// fitted capacity, and its first lists are built again from the same
// coordinates (the lists a fitted first build gives); its build counts are
// set back to one build.  Capacities only grow, so a system never holds less
// than job_bytes_estimate charged for it.
// (From what the device reported after those lists.)
sop_status engine_fit_new(sop_engine *e, const int32_t *slots, int32_t n) {
  sop_status st = SOP_OK;
  std::vector<int32_t> redo;
  for (int32_t q = 0; q < n; ++q) {
    const int32_t s = slots[q];
    const SysHost &h = e->sys[s];
    const int32_t err = e->p.rep[s].x;
    if (err & ~ERR_PL_OVF) continue;  // failed for another reason: reported as it is
    const int32_t m = e->p.rep[s].y, want = pl_cap_target(e, h.n, m);
    const bool over = (err & ERR_PL_OVF) != 0;
    if (!over && !pl_cap_short(e, h, m)) continue;
    if (want == h.pl_cap || want < m) continue;  // at the limit: an overflow stands
    st = engine_resize_rows(e, s, want, false);
    if (st) return st;
    redo.push_back(s);
  }
  if (redo.empty()) return SOP_OK;
  std::vector<SysDev> sd;
  if ((st = read_sys_all(e, sd))) return st;
  const int32_t zero = 0;
  for (int32_t s : redo) {
    HIPCK(hipMemcpy(&e->p.sys[s].err, &zero, sizeof(zero), hipMemcpyHostToDevice));
    HIPCK(hipMemcpy(&e->p.sys[s].row_max, &zero, sizeof(zero), hipMemcpyHostToDevice));
  }
  st = engine_set_batch(e, redo.data(), (int32_t)redo.size());
  if (st) return st;
  HIPCK(launch_lists(e->p, list_grids(e), 0, FORCE_NL | FORCE_PL, e->stream));
  HIPCK(launch_report(e->p, e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  for (int32_t s : redo)
    HIPCK(hipMemcpy(e->p.sys[s].nbuild, sd[s].nbuild, sizeof(sd[s].nbuild), hipMemcpyHostToDevice));
  return SOP_OK;
}

// First neighbor and pair lists of newly added systems, in one launch
// sequence (the reference builds both before its step loop), with row
// capacities fitted.  status[q] receives each system's result; systems that
// fail are removed.
sop_status engine_init_lists(sop_engine *e, const int32_t *slots, int32_t n, sop_status *status) {
  if (n <= 0) return SOP_OK;
  sop_status st = engine_set_batch(e, slots, n);
  if (st) return st;
  HIPCK(launch_lists(e->p, list_grids(e), 0, FORCE_NL | FORCE_PL, e->stream));
  HIPCK(launch_report(e->p, e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  st = engine_fit_new(e, slots, n);
  if (st) return st;
  for (int32_t q = 0; q < n; ++q) {
    status[q] = engine_error_status(e, slots[q], e->p.rep[slots[q]].x);
    if (status[q]) engine_remove_system(e, slots[q]);
  }
  return SOP_OK;
}

sop_status engine_add_system(sop_engine *e, const sop_system_desc *d, int32_t *slot_out) {
  int32_t slot = -1;
  sop_status st = engine_add_system_nolists(e, d, 0, &slot);
  if (st) return st;
  sop_status one = SOP_OK;
  st = engine_init_lists(e, &slot, 1, &one);
  if (st) return st;
  if (one) return one;
  *slot_out = slot;
  return SOP_OK;
}

sop_status engine_remove_system(sop_engine *e, int32_t slot) {
  if (slot < 0 || slot >= (int32_t)e->sys.size() || !e->sys[slot].used)
    return set_error(e, SOP_ERR_INVALID, "no such system");
  SysHost &h = e->sys[slot];
  e->a_beads.release(h.bead_off, h.bead_len);
  e->a_nat.release(h.nat_off, h.nat_len);
  e->a_pl.release(h.pl_off, h.pl_len);
  if (e->nl_owner == slot) e->nl_owner = -1;
  e->a_cells.release(h.cell_off, h.cell_len);
  h = SysHost();
  return SOP_OK;
}

// Upload the work tables for a batch of systems.  Systems are spread over the
// 8 XCDs by bead count; entry k of the work list is processed by a block on
// XCD k % 8 (round-robin dispatch with a grid that is a multiple of 8), so all
// tiles of a system share one XCD's L2.
sop_status engine_set_batch(sop_engine *e, const int32_t *slots, int32_t nslots) {
  constexpr int NX = 8;
  // everything the tables are made from: while it is what it was, so are they
  std::vector<int64_t> key;
  key.reserve(20 + 3 * (size_t)nslots);
  for (int64_t v : {(int64_t)nslots, (int64_t)e->fixed_grids, (int64_t)e->opts.lanes_per_bead, (int64_t)e->opts.step_tiles,
                    (int64_t)e->opts.lds_beads_max, (int64_t)e->lds_limit, e->lds_big_cap, (int64_t)e->num_cu,
                    (int64_t)e->tune.nb, (int64_t)e->tune.tail})
    key.push_back(v);
  for (int b = 0; b < 3; ++b) {
    key.push_back(e->tune.max_beads[b]);
    key.push_back(e->tune.tiles[b]);
  }
  for (int32_t q = 0; q < nslots; ++q) {
    const SysHost &h = e->sys[slots[q]];
    key.push_back(slots[q]);
    key.push_back(h.bead_off);
    key.push_back(h.n);
  }
  if (key == e->batch_key) return SOP_OK;
  e->batch_key.clear();
  std::vector<int32_t> order(slots, slots + nslots);
  std::sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
    if (e->sys[a].bead_len != e->sys[b].bead_len) return e->sys[a].bead_len > e->sys[b].bead_len;
    return a < b;
  });
  std::vector<std::vector<int32_t>> bins(NX), bsys(NX);
  std::vector<int64_t> load(NX, 0);
  for (int32_t s : order) {
    const int x = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    const SysHost &h = e->sys[s];
    for (int64_t t = h.bead_off / TILE; t < (h.bead_off + h.n + TILE - 1) / TILE; ++t) {
      bins[x].push_back((int32_t)t);
      bsys[x].push_back(s);
    }
    load[x] += (h.n + TILE - 1) / TILE;
  }
  size_t mx = 0;
  for (auto &b : bins) mx = std::max(mx, b.size());
  e->h_work.assign(mx * NX, -1);
  for (int x = 0; x < NX; ++x)
    for (size_t m = 0; m < bins[x].size(); ++m) e->h_work[m * NX + x] = bins[x][m];
  // Work items of the step kernel and of the shell filter: {first tile, tiles
  // (| waves per tile << 8 for the step kernel), first staged bead or -1,
  // staged beads}.  Systems that fit the LDS budget are staged whole:
  // arena-adjacent small systems share an item (one staged range), a larger
  // system gets one item per `per` tiles, each staging the whole system.
  // Larger systems gather from global memory, their items in runs over all
  // XCDs.  The shell filter takes one wave per tile, STEP_WAVES tiles per item.
  // The step kernel's items hold `per` tiles and run each tile on
  // min(lanes_per_bead, STEP_WAVES / tiles) waves (power of two), each wave
  // taking that share of the tile's rounds: an item's duration shrinks with
  // its tile count, so small items do not leave waves idle while the big
  // ones finish.
  const int64_t lds_cap = e->opts.lds_beads_max > 0
                              ? std::min<int64_t>(e->opts.lds_beads_max, (int64_t)(e->lds_limit / 16))
                              : 0;
  std::vector<int32_t> by_arena(slots, slots + nslots);
  std::sort(by_arena.begin(), by_arena.end(),
            [&](int32_t a2, int32_t b2) { return e->sys[a2].bead_off < e->sys[b2].bead_off; });
  // tiles per step item: the option, or 16 while the batch's tiles fill the
  // wave slots of the LDS launch (two blocks of STEP_WAVES per compute unit),
  // 8 or 4 below that, so that a small batch still fills the device
  int64_t total_tiles = 0;
  for (int32_t q = 0; q < nslots; ++q) total_tiles += e->sys[slots[q]].bead_len / TILE;
  const int64_t slots_w = (int64_t)e->num_cu * STEP_WAVES;
  // systems above lds_cap that fit one compute unit's whole LDS take the
  // whole-CU tier (one block per unit) instead of global gathers.  While
  // serving only under load (more tiles than two LDS launches' wave slots):
  // there it raises the stream's capacity (3.8e9 -> 4.9e9 bead-steps/s at its
  // stated parameters), while under a light load the global-gather tier,
  // spread over more blocks, gives the shorter step (served p50 0.25 s
  // against 0.30 s)
  const int64_t big_cap = e->fixed_grids && total_tiles <= 2 * slots_w ? 0 : e->lds_big_cap;
  const int lpb = e->opts.lanes_per_bead;
  int32_t per_step = e->opts.step_tiles;
  if (per_step <= 0) per_step = total_tiles > slots_w ? STEP_WAVES : (2 * total_tiles > slots_w ? 8 : 4);
  e->cur_step_tiles = per_step;
  // the tiles with a block each in the step and the shell filter (k_step_tile,
  // k_filter_tile): all of a batch of up to
  // TILE_STEP_PER_CU tiles per compute unit; else the systems too large for
  // two LDS blocks per unit while theirs are that few, and the ones too large
  // for any LDS tier up to TILE_STEP_FAR_PER_CU.  Step times by tile against
  // the other kernel (us), on either side of the lines: 2 x 8,000 beads 7.7 /
  // 13.7 whole-CU, 4 x 8,000 12.6 / 14.1, 6 x 8,000 17.0 / 14.3; 8 x 4,000 11.2 /
  // 12.7 LDS, 12 x 4,000 16.4 / 13.0; 32 x 4,000 and 4 x 8,000 together 33.5 /
  // 40.3.  Against global-gather items, step, and run per step with its rebuilds:
  // 20,000 beads 11.7, 16.8 / 17.2, 24.8; 45,000 17.1, 26.1 / 18.3, 27.8; 60,000
  // 21.8, 32.8 / 18.7, 28.4; chains of 500 together, 40,000 13.2, 18.7 / 13.3,
  // 19.2; 60,000 17.1, 24.2 / 13.5, 19.4.
  const int64_t tile_cap = (int64_t)TILE_STEP_PER_CU * e->num_cu;
  int64_t mid_tiles = 0, far_tiles = 0;
  for (int32_t q = 0; q < nslots; ++q) {
    const int64_t len = e->sys[slots[q]].bead_len;
    if (len > lds_cap) (len > big_cap ? far_tiles : mid_tiles) += len / TILE;
  }
  const bool own_items = e->opts.step_tiles > 0;  // item size asked for
  const bool by_tile = total_tiles <= tile_cap && !own_items;
  const bool mid_by_tile = mid_tiles + far_tiles <= tile_cap && !own_items;
  const bool far_by_tile = far_tiles <= (int64_t)TILE_STEP_FAR_PER_CU * e->num_cu && !own_items;
  auto tile_filter = [&](const SysHost &h) {
    if (h.n > 65536) return false;  // 16-bit rows only
    return by_tile || (h.bead_len > lds_cap && (mid_by_tile || (far_by_tile && h.bead_len > big_cap)));
  };
  // a batch of LDS and global-gather systems alone steps in one launch of
  // items of both (k_step_mixed)
  e->cur_mixed = !by_tile && mid_tiles == 0 && far_tiles > 0 && far_tiles < total_tiles;
  auto tile_step = [&](const SysHost &h) { return !e->cur_mixed && tile_filter(h); };
  std::vector<int2> tiles;
  {
    // each XCD (tile k of the table runs on XCD k mod 8) a run of consecutive
    // tiles, whose gathers share much of their range of the coordinates
    std::vector<int2> all;
    for (int32_t sl : by_arena) {
      const SysHost &h = e->sys[sl];
      if (!tile_filter(h)) continue;
      for (int64_t t = h.bead_off / TILE; t < (h.bead_off + h.bead_len) / TILE; ++t)
        all.push_back(make_int2((int32_t)t, sl));
    }
    const size_t run = (all.size() + NX - 1) / NX;
    tiles.assign(run * NX, make_int2(-1, 0));
    for (size_t k = 0; k < all.size(); ++k) tiles[(k % run) * NX + k / run] = all[k];
  }
  struct Plan {
    std::vector<int4> items;
    int32_t n_lds = 0, n_big = 0, n_far = 0;
    size_t lds = 0, lds_big = 0;
  };
  // tiles per item of the global-gather systems: the fewest, 4 to 16, with at
  // most one item per compute unit (a wave's share of a tile repeats the tile's
  // chain terms and noise, and a second item on some of the units lasts as long
  // as on all).  Counted system by system: 200 systems of 16 tiles are 200
  // items of 16 tiles, and 400 of the 13 that their tiles over the units come
  // to (run 52.9 and 74.2 us per step).  Run per step for chains of 500 beads
  // by items of 4 / 8 / 16 tiles (us): 200,000 beads 56.5 / 49.4 / 46.0, by this
  // rule (13) 42.8; 100,000 beads 33.2 / 29.8 / 41.8, by this rule (7) 27.7.
  int32_t per_far = 4;
  for (; per_far < STEP_WAVES; ++per_far) {
    int64_t items = 0;
    for (int32_t q = 0; q < nslots; ++q) {
      const int64_t len = e->sys[slots[q]].bead_len;
      if (len > lds_cap && len > big_cap) items += (len / TILE + per_far - 1) / per_far;
    }
    if (items <= e->num_cu) break;
  }
  // in a mixed launch the fewest of 4, 8 or 16 tiles with which all items are
  // resident at once, two per unit (the batch's item size instead: 60 systems
  // of 1,500 beads and 3 of 18,000 60.8 us per step against 49.4, 120 and 8
  // 105 against 96)
  int32_t per_mixed = 4;
  while (per_mixed < STEP_WAVES &&
         (total_tiles - far_tiles) / per_step + far_tiles / per_mixed > 2 * (int64_t)e->num_cu)
    per_mixed *= 2;
  // tiles per item of a system: its size bucket's tuned value, else the rule's
  auto per_of = [&](const SysHost &h, int32_t otherwise) {
    const int b = engine_bucket(e, h.n);
    return b >= 0 && e->tune.tiles[b] > 0 ? e->tune.tiles[b] : otherwise;
  };
  auto plan = [&](int32_t per_fixed, bool split, Plan &out) {
    // waves per tile of an item of nt tiles
    auto waves = [&](int32_t nt) {
      int32_t w = 1;
      if (split)
        while (w * 2 <= lpb && nt * w * 2 <= STEP_WAVES) w *= 2;
      return w;
    };
    auto mk = [&](int32_t t0, int32_t nt, int32_t z, int32_t wlen) {
      return make_int4(t0, nt | (waves(nt) << 8), z, wlen);
    };
    std::vector<int4> lds_items, big_items;
    std::vector<std::vector<int4>> far_items;  // per non-LDS system
    int4 cur = make_int4(-1, 0, -1, 0);        // .y: tiles while the item grows
    int32_t cur_per = 0;                       // tiles per item of the systems in cur
    auto flush = [&]() {
      if (cur.x >= 0) lds_items.push_back(mk(cur.x, cur.y, cur.z, cur.w));
      cur = make_int4(-1, 0, -1, 0);
    };
    for (int32_t sl : by_arena) {
      const SysHost &h = e->sys[sl];
      if (split ? tile_step(h) : tile_filter(h)) continue;
      const int32_t t0 = (int32_t)(h.bead_off / TILE), nt = (int32_t)(h.bead_len / TILE);
      const int32_t per = per_fixed > 0 ? per_fixed : per_of(h, per_step);
      if (h.bead_len <= lds_cap) {
        out.lds = std::max(out.lds, (size_t)h.bead_len * 16);
        if (nt > per) {
          flush();
          for (int32_t k = 0; k < nt; k += per)
            lds_items.push_back(mk(t0 + k, std::min(per, nt - k), (int32_t)h.bead_off, (int32_t)h.bead_len));
          continue;
        }
        if (cur.x >= 0 && cur_per == per && (int64_t)cur.z + cur.w == h.bead_off && cur.y + nt <= per &&
            (int64_t)cur.w + h.bead_len <= lds_cap) {
          cur.y += nt;
          cur.w += (int32_t)h.bead_len;
          out.lds = std::max(out.lds, (size_t)cur.w * 16);
        } else {
          flush();
          cur = make_int4(t0, nt, (int32_t)h.bead_off, (int32_t)h.bead_len);
          cur_per = per;
        }
      } else if (h.bead_len <= big_cap) {
        flush();
        out.lds_big = std::max(out.lds_big, (size_t)h.bead_len * 16);
        for (int32_t k = 0; k < nt; k += per)
          big_items.push_back(mk(t0 + k, std::min(per, nt - k), (int32_t)h.bead_off, (int32_t)h.bead_len));
      } else {
        flush();
        std::vector<int4> v;
        const int32_t pf = own_items ? per : !split ? per_far : per_of(h, e->cur_mixed ? per_mixed : per_far);
        for (int32_t k = 0; k < nt; k += pf) v.push_back(mk(t0 + k, std::min(pf, nt - k), -1, 0));
        far_items.push_back(v);
      }
    }
    flush();
    // XCD bins by load (item k runs on XCD k mod 8): the LDS items, longest
    // first (an item lasts about one tile's rounds / its waves per tile)
    std::vector<std::vector<int4>> ibins(NX), bbins(NX), fbins(NX);
    std::vector<double> iload(NX, 0), bload(NX, 0);
    auto by_dur = [&](const int4 &u, const int4 &v) {
      const double du = 1.0 / item_split(u.y), dv = 1.0 / item_split(v.y);
      return du != dv ? du > dv : item_tiles(u.y) > item_tiles(v.y);
    };
    std::stable_sort(lds_items.begin(), lds_items.end(), by_dur);
    // the tail: items that start only after a first round of full-length
    // items (two LDS blocks per compute unit) are cut into pieces of at most
    // STEP_WAVES / tail tiles, each with more waves per tile, so that the last
    // round is short
    if (split && e->tune.tail > 1) {
      const size_t slots = 2 * (size_t)e->num_cu;
      size_t nfull = 0;
      while (nfull < lds_items.size() && item_split(lds_items[nfull].y) == 1) ++nfull;
      if (nfull > slots) {
        std::vector<int4> cut(lds_items.begin(), lds_items.begin() + slots);
        const int32_t pmax = std::max(1, STEP_WAVES / e->tune.tail);
        for (size_t k = slots; k < lds_items.size(); ++k) {
          const int4 it = lds_items[k];
          const int32_t nt = item_tiles(it.y);
          for (int32_t a = 0; a < nt; a += pmax)
            cut.push_back(mk(it.x + a, std::min(pmax, nt - a), it.z, it.w));
        }
        std::stable_sort(cut.begin() + slots, cut.end(), by_dur);
        lds_items.swap(cut);
      }
    }
    // the items that stage one range (one system's items) go to one XCD, so
    // that their stagings after the first read the range from that XCD's L2;
    // ranges by load, largest first, each to the least-loaded XCD, then each
    // XCD's items longest first
    auto bin_by_range = [&](const std::vector<int4> &items, std::vector<std::vector<int4>> &bins,
                            std::vector<double> &load) {
      std::vector<std::pair<double, std::vector<int4>>> ranges;
      std::unordered_map<int32_t, size_t> at;
      for (const int4 &it : items) {
        auto f = at.find(it.z);
        if (f == at.end()) {
          f = at.emplace(it.z, ranges.size()).first;
          ranges.emplace_back(0.0, std::vector<int4>());
        }
        ranges[f->second].first += (double)item_tiles(it.y);
        ranges[f->second].second.push_back(it);
      }
      std::stable_sort(ranges.begin(), ranges.end(),
                       [](const auto &u, const auto &v) { return u.first > v.first; });
      for (const auto &r : ranges) {
        const int x = (int)(std::min_element(load.begin(), load.end()) - load.begin());
        bins[x].insert(bins[x].end(), r.second.begin(), r.second.end());
        load[x] += r.first;
      }
      for (auto &bn : bins) std::stable_sort(bn.begin(), bn.end(), by_dur);
    };
    bin_by_range(lds_items, ibins, iload);
    std::stable_sort(big_items.begin(), big_items.end(), by_dur);
    bin_by_range(big_items, bbins, bload);
    std::sort(far_items.begin(), far_items.end(), [](const std::vector<int4> &u, const std::vector<int4> &v) {
      return u.size() != v.size() ? u.size() > v.size() : u[0].x < v[0].x;
    });
    // the global-gather items: each system's in contiguous runs of at most an
    // eighth of all items, to the XCD with the fewest, and no more to any than it
    // takes in as many rounds as all need, so that none holds a second round of
    // items while another has units free.  Step times
    // with each system whole on the least-loaded XCD, and now (us): 6 systems of
    // 30,000 beads 57.5, 44.5; 14 of 16,000 57.6, 49.8; 3 of 60,000 63.2, 48.1
    // (runs of at most an eighth, each whole to the least-loaded XCD, left two
    // on some: 67.8, 73.1 and 73.2)
    size_t n_far = 0;
    for (const auto &v : far_items) n_far += v.size();
    const size_t units = (size_t)std::max(1, e->num_cu / NX), share = (n_far + NX - 1) / NX;
    const size_t most = share <= units ? share : (share + units - 1) / units * units;
    for (const auto &v : far_items)
      for (size_t k = 0; k < v.size();) {
        auto &bn = *std::min_element(fbins.begin(), fbins.end(),
                                     [](const auto &u, const auto &w) { return u.size() < w.size(); });
        const size_t run = std::min({v.size() - k, share, most - bn.size()});
        bn.insert(bn.end(), v.begin() + k, v.begin() + k + run);
        k += run;
      }
    size_t imx = 0, bmx = 0, fmx = 0;
    for (auto &bn : ibins) imx = std::max(imx, bn.size());
    for (auto &bn : bbins) bmx = std::max(bmx, bn.size());
    for (auto &bn : fbins) fmx = std::max(fmx, bn.size());
    out.items.assign((imx + bmx + fmx) * NX, make_int4(-1, 0, -1, 0));
    for (int x = 0; x < NX; ++x) {
      for (size_t m = 0; m < ibins[x].size(); ++m) out.items[m * NX + x] = ibins[x][m];
      for (size_t m = 0; m < bbins[x].size(); ++m) out.items[(imx + m) * NX + x] = bbins[x][m];
      for (size_t m = 0; m < fbins[x].size(); ++m) out.items[(imx + bmx + m) * NX + x] = fbins[x][m];
    }
    out.n_lds = (int32_t)(imx * NX);
    out.n_big = (int32_t)(bmx * NX);
    out.n_far = (int32_t)(fmx * NX);
    // fixed grids (serving): the launches' LDS sizes too, so that one captured
    // graph serves every batch
    if (e->fixed_grids && lds_cap > 0) out.lds = (size_t)lds_cap * 16;
    if (e->fixed_grids && big_cap > 0) out.lds_big = (size_t)big_cap * 16;
  };
  Plan sp, fp;
  plan(0, true, sp);
  plan(STEP_WAVES, false, fp);
  e->h_items.swap(sp.items);
  e->h_fitems.swap(fp.items);
  e->cur_lds = sp.lds;
  e->cur_lds_big = sp.lds_big;
  e->cur_flds = fp.lds;
  e->cur_flds_big = fp.lds_big;
  // the systems too large for one block's rebuild first
  e->h_syslist.assign(slots, slots + nslots);
  const auto big_end = std::stable_partition(e->h_syslist.begin(), e->h_syslist.end(),
                                             [&](int32_t s) { return e->sys[s].n > SORT_N_MAX; });
  const int32_t nbig = (int32_t)(big_end - e->h_syslist.begin());
  e->cur_big_max = 0;
  for (int32_t q = 0; q < nbig; ++q) e->cur_big_max = std::max(e->cur_big_max, e->sys[e->h_syslist[q]].n);
  if ((int64_t)e->h_work.size() + 2 > e->work_cap) {
    HIPCK(hipStreamSynchronize(e->stream));
    int64_t nc = std::max<int64_t>(1024, (int64_t)e->h_work.size() * 2 + 2);
    if (e->p.work) HIPCK(hipFree(e->p.work));
    HIPCK(hipMalloc((void **)&e->p.work, 4 * (size_t)nc));
    e->work_cap = nc;
    invalidate_graphs(e);
  }
  if ((int64_t)tiles.size() > e->tiles_cap) {
    HIPCK(hipStreamSynchronize(e->stream));
    // (room for every block of the launch: a block reads its first entry at once)
    const int64_t nc = std::max<int64_t>(std::max(1024, 4 * e->num_cu), (int64_t)tiles.size() * 2);
    if (e->p.tiles) HIPCK(hipFree(e->p.tiles));
    HIPCK(hipMalloc((void **)&e->p.tiles, sizeof(int2) * (size_t)nc));
    e->tiles_cap = nc;
    invalidate_graphs(e);
  }
  if (!e->p.nwork) {
    HIPCK(hipMalloc((void **)&e->p.nwork, 256));
    e->p.nsys = e->p.nwork + 16;
    e->p.nbig = e->p.nwork + 24;
    e->p.ncellwork = e->p.nwork + 32;
    e->p.nlbuild = e->p.nwork + 40;
    e->p.nfitems = e->p.nwork + 44;
    e->p.nfitems_big = e->p.nwork + 45;
    e->p.nfitems_far = e->p.nwork + 46;
    e->p.nitems = e->p.nwork + 48;
    e->p.nitems_far = e->p.nwork + 56;
    e->p.ntiles = e->p.nwork + 57;
    e->p.nitems_big = e->p.nwork + 60;
    invalidate_graphs(e);
  }
  if ((int64_t)e->h_items.size() + 1 > e->items_cap) {
    HIPCK(hipStreamSynchronize(e->stream));
    const int64_t nc = std::max<int64_t>(1024, (int64_t)e->h_items.size() * 2 + 1);
    if (e->p.items) HIPCK(hipFree(e->p.items));
    HIPCK(hipMalloc((void **)&e->p.items, sizeof(int4) * (size_t)nc));
    e->items_cap = nc;
    invalidate_graphs(e);
  }
  if ((int64_t)e->h_fitems.size() + 1 > e->fitems_cap) {
    HIPCK(hipStreamSynchronize(e->stream));
    const int64_t nc = std::max<int64_t>(1024, (int64_t)e->h_fitems.size() * 2 + 1);
    if (e->p.fitems) HIPCK(hipFree(e->p.fitems));
    HIPCK(hipMalloc((void **)&e->p.fitems, sizeof(int4) * (size_t)nc));
    e->fitems_cap = nc;
    invalidate_graphs(e);
  }
  if (nslots > e->cap.slots) return set_error(e, SOP_ERR_INVALID, "batch larger than slot capacity");
  const int32_t nw = (int32_t)e->h_work.size(), ns = nslots;
  const int32_t ni = (int32_t)e->h_items.size(), nfi = (int32_t)e->h_fitems.size();
  // the counters: nwork[0] = work entries, [16] batch systems, [24] large
  // ones, [32] home cells and [40] neighbor-list builds of a rebuild (none
  // between rebuilds), [44..46] filter items, [48] / [56] / [60] step items
  // (LDS / far / whole-CU), [57] step tiles
  int32_t cnt[64] = {0};
  cnt[0] = nw;
  cnt[16] = ns;
  cnt[24] = nbig;
  cnt[44] = fp.n_lds;
  cnt[45] = fp.n_big;
  cnt[46] = fp.n_far;
  cnt[48] = sp.n_lds;
  cnt[56] = sp.n_far;
  cnt[57] = (int32_t)tiles.size();
  cnt[60] = sp.n_big;
  // all of it through the staging buffer, in one launch
  const std::pair<void *, std::pair<const void *, size_t>> parts[TABLE_PARTS] = {
      {e->p.nwork, {cnt, 64}},
      {e->p.work, {e->h_work.data(), (size_t)nw}},
      {e->p.syslist, {e->h_syslist.data(), (size_t)ns}},
      {e->p.items, {e->h_items.data(), 4 * (size_t)ni}},
      {e->p.fitems, {e->h_fitems.data(), 4 * (size_t)nfi}},
      {e->p.tiles, {tiles.data(), 2 * tiles.size()}}};
  size_t words = 0;
  for (const auto &q : parts) words += q.second.second;
  HIPCK(hipStreamSynchronize(e->stream));  // the launch that read the last tables has passed
  // room for a large system's upload, which the tables need none of, is given back
  constexpr size_t STAGE_KEEP = (size_t)96 << 20;
  if (e->stage.bytes > STAGE_KEEP && 4 * words <= STAGE_KEEP) {
    (void)hipHostFree(e->stage.ptr);
    e->stage = HostBuf();
  }
  sop_status st = engine_io(e, e->stage, 4 * words);
  if (st) return st;
  TableParts tp;
  tp.stage = static_cast<const uint32_t *>(e->stage.ptr);
  size_t at = 0;
  for (int k = 0; k < TABLE_PARTS; ++k) {
    const auto &q = parts[k];
    if (q.second.second) std::memcpy(static_cast<uint32_t *>(e->stage.ptr) + at, q.second.first, 4 * q.second.second);
    tp.part[k] = TablePart{static_cast<uint32_t *>(q.first), (uint32_t)at, (uint32_t)q.second.second};
    at += q.second.second;
  }
  HIPCK(launch_tables(tp, e->stream));
  e->cur_ntiles = (int32_t)tiles.size();
  e->cur_nwork = nw;
  e->cur_nsys = ns;
  e->cur_nbig = nbig;
  e->cur_nitems = sp.n_lds;
  e->cur_nitems_big = sp.n_big;
  e->cur_nitems_far = sp.n_far;
  e->cur_nfitems = fp.n_lds;
  e->cur_nfitems_far = fp.n_far;
  e->cur_nfitems_big = fp.n_big;
  e->batch_key.swap(key);
  return SOP_OK;
}

sop_status engine_error_status(sop_engine *e, int32_t s, int32_t err) {
  if (!err) return SOP_OK;
  std::ostringstream os;
  os << "system " << s << ":";
  sop_status st = SOP_ERR_STATE;
  if (err & ERR_NAN) { os << " non-finite coordinates;"; st = SOP_ERR_NUMERIC; }
  if (err & ERR_BOND) { os << " FENE bond stretched to |r-r0| >= R0;"; st = SOP_ERR_NUMERIC; }
  if (err & ERR_NL_OVF) { os << " neighbor list over capacity;"; st = SOP_ERR_CAPACITY; }
  if (err & ERR_PL_OVF) { os << " pair list over capacity;"; st = SOP_ERR_CAPACITY; }
  if (err & ERR_PBC) { os << " extent within 10 A of boxl/2 (open cell grid needs the minimum image to be the identity);"; st = SOP_ERR_PBC; }
  if (err & ERR_INTERNAL) { os << " inconsistent cell histogram;"; st = SOP_ERR_STATE; }
  return set_error(e, st, os.str());
}

// Status of the listed systems, which are the current batch's: reported by the
// device and read once the stream is done.
sop_status engine_check_errors(sop_engine *e, const int32_t *slots, int32_t nslots) {
  HIPCK(launch_report(e->p, e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  for (int q = 0; q < nslots; ++q) {
    const sop_status st = engine_error_status(e, slots[q], e->p.rep[slots[q]].x);
    if (st) return st;
  }
  return SOP_OK;
}

static std::string graph_key(const sop_engine *e, int G, int n_nl, int n_pl) {
  std::ostringstream os;
  os << G << '|' << n_nl << '|' << n_pl << '|' << e->opts.lanes_per_bead << '|' << grid_tiles(e) << '|'
     << grid_rebuild(e) << '|' << grid_big_beads(e) << '|' << grid_big_sys(e) << '|' << grid_items(e) << '|' << grid_items_big(e) << '|'
     << e->cur_lds << '|' << e->cur_lds_big;
  const StepGrids fg = filter_grids(e);
  os << '|' << e->cur_mixed << '|' << grid_step_tiles(e) << '|' << grid_items_far(e) << '|' << list_grids(e).split << '|' << fg.grid << '|' << fg.grid_big << '|' << fg.grid_far << '|' << fg.lds << '|' << fg.lds_big;
  return os.str();
}

constexpr int64_t GROW_BLOCKS = 20;

// One hipGraph replay = G steps of an aligned batch (every system's step is a
// multiple of n_nl): NL rebuild at k % n_nl == 0, PL filter at k % n_pl == 0,
// fused step kernel every k, step-counter advance at the end.
sop_status engine_run_block_graph(sop_engine *e, int32_t G) {
  const SysHost &h0 = e->sys[e->h_syslist[0]];
  const int n_nl = h0.params.n_nl, n_pl = h0.params.n_pl;
  const std::string key = graph_key(e, G, n_nl, n_pl);
  auto it = e->graphs.find(key);
  hipGraphExec_t exec;
  if (it == e->graphs.end()) {
    hipGraph_t graph;
    const int lpb = e->opts.lanes_per_bead;
    HIPCK(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal));
    for (int k = 0; k < G; ++k) {
      if (k % n_pl == 0 || k % n_nl == 0) (void)launch_lists(e->p, list_grids(e), k, 0, e->stream, &e->fork);
      (void)launch_step(e->p, MODE_STEP, lpb, step_grids(e), k, e->stream, &e->fork);
    }
    (void)launch_advance(e->p, G, e->stream);
    HIPCK(hipStreamEndCapture(e->stream, &graph));
    HIPCK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    HIPCK(hipGraphDestroy(graph));
    e->graphs[key] = exec;
  } else {
    exec = it->second;
  }
  HIPCK(hipGraphLaunch(exec, e->stream));
  return SOP_OK;
}

// Host-driven steps for the current batch: launches exactly the rebuilds some
// system is due for (the kernels check each system's own schedule).
sop_status engine_run_hostloop(sop_engine *e, int64_t nsteps) {
  if (nsteps <= 0) return SOP_OK;
  const int lpb = e->opts.lanes_per_bead;
  std::vector<int64_t> st;
  std::vector<int32_t> nnl, npl;
  for (int32_t s : e->h_syslist) {
    st.push_back(e->sys[s].step);
    nnl.push_back(e->sys[s].params.n_nl);
    npl.push_back(e->sys[s].params.n_pl);
  }
  for (int64_t k = 0; k < nsteps; ++k) {
    bool any_nl = false, any_pl = false;
    for (size_t q = 0; q < st.size(); ++q) {
      any_nl |= ((st[q] + k) % nnl[q]) == 0;
      any_pl |= ((st[q] + k) % npl[q]) == 0;
    }
    if (any_nl || any_pl) HIPCK(launch_lists(e->p, list_grids(e), (int)k, 0, e->stream, &e->fork));
    HIPCK(launch_step(e->p, MODE_STEP, lpb, step_grids(e), (int)k, e->stream, &e->fork));
  }
  HIPCK(launch_advance(e->p, (int)nsteps, e->stream));
  return SOP_OK;
}

static void mirror_advance(sop_engine *e, const int32_t *sys, int32_t nsys, int64_t nsteps) {
  for (int q = 0; q < nsys; ++q) {
    e->sys[sys[q]].step += nsteps;
    e->sys[sys[q]].parity = (int32_t)((e->sys[sys[q]].parity + nsteps) & 1);
  }
}

// Row capacities after steps, from what the last k_advance reported.
static sop_status grow_reported(sop_engine *e, const int32_t *sys, int32_t nsys) {
  std::vector<int32_t> longest((size_t)nsys);
  for (int32_t q = 0; q < nsys; ++q) longest[q] = e->p.rep[sys[q]].y;
  return engine_grow_rows(e, sys, nsys, longest.data(), nullptr);
}

// nsteps of the listed systems in one batch: hipGraph blocks of n_nl steps
// while the schedule is uniform and aligned, host-driven launches for the
// rest.  With events, ev0 is recorded after the batch's tables are set and
// ev1 after the last launch (device time of the steps).
sop_status engine_run(sop_engine *e, const int32_t *sys, int32_t nsys, int64_t nsteps, hipEvent_t ev0,
                      hipEvent_t ev1) {
  if (nsteps == 0) return SOP_OK;
  sop_status st = engine_set_batch(e, sys, nsys);
  if (st) return st;
  HIPCK(launch_begin(e->p, nsteps, e->stream));
  if (ev0) HIPCK(hipEventRecord(ev0, e->stream));
  // graph blocks need a uniform schedule and phase
  const sop_params &P0 = e->sys[sys[0]].params;
  bool uniform = e->opts.use_graphs != 0 && P0.n_nl % P0.n_pl == 0;
  const int64_t G = P0.n_nl;
  const int64_t r0 = e->sys[sys[0]].step % G;
  for (int q = 1; q < nsys && uniform; ++q) {
    const SysHost &h = e->sys[sys[q]];
    uniform = h.params.n_nl == P0.n_nl && h.params.n_pl == P0.n_pl && h.step % G == r0;
  }
  int64_t left = nsteps;
  if (uniform && G > 1) {
    const int64_t pre = std::min(left, (G - r0) % G);
    if (pre > 0) {
      st = engine_run_hostloop(e, pre);
      if (st) return st;
      mirror_advance(e, sys, nsys, pre);
      left -= pre;
    }
    int64_t blocks = 0;
    while (left >= G) {
      st = engine_run_block_graph(e, (int32_t)G);
      if (st) return st;
      mirror_advance(e, sys, nsys, G);
      left -= G;
      // row capacities checked every GROW_BLOCKS blocks of a long run
      if (++blocks % GROW_BLOCKS == 0 && left >= G && !ev1) {
        HIPCK(hipStreamSynchronize(e->stream));
        st = grow_reported(e, sys, nsys);
        if (st) return st;
      }
    }
  }
  if (left > 0) {
    st = engine_run_hostloop(e, left);
    if (st) return st;
    mirror_advance(e, sys, nsys, left);
  }
  if (ev1) HIPCK(hipEventRecord(ev1, e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  st = grow_reported(e, sys, nsys);
  if (st) return st;
  for (int32_t q = 0; q < nsys; ++q) {
    st = engine_error_status(e, sys[q], e->p.rep[sys[q]].x);
    if (st) return st;
  }
  return SOP_OK;
}

} // namespace sopk

// ================================================================ C ABI

extern "C" {

const char *sop_version(void) { return "sop-mi355x 0.1 (gfx950)"; }

double sop_clock_seconds(void) {
  using namespace std::chrono;
  return duration_cast<duration<double>>(steady_clock::now().time_since_epoch()).count();
}

void sop_engine_opts_default(sop_engine_opts *o) {
  std::memset(o, 0, sizeof(*o));
  o->nl_cap_max = 4096;
  o->pl_cap_max = 1024;
  o->cell_cap_max = 32768;
  o->lanes_per_bead = 4;
  o->grid_blocks = 0;
  o->use_graphs = 1;
  o->lds_beads_max = 5056;  // two 1024-thread step blocks per compute unit at 80,896 B each
  o->pl_shell = 3.0f;
  o->pool_bytes = 0;
  o->step_tail = 2;  // late step items cut to 8 tiles (6.12e9 against 6.02e9 bead-steps/s on 512 replicas)
}

sop_status sop_engine_create(int32_t device, const sop_engine_opts *opts, sop_engine **out) {
  if (!out) return SOP_ERR_INVALID;
  *out = nullptr;
  // the options first (refused before any device call)
  sop_engine_opts eo;
  sop_engine_opts_default(&eo);
  if (opts) {
    eo = *opts;
    sop_engine_opts def;
    sop_engine_opts_default(&def);
    if (eo.nl_cap_max <= 0) eo.nl_cap_max = def.nl_cap_max;
    if (eo.pl_cap_max <= 0) eo.pl_cap_max = def.pl_cap_max;
    if (eo.cell_cap_max <= 0) eo.cell_cap_max = def.cell_cap_max;
    if (eo.lanes_per_bead <= 0) eo.lanes_per_bead = def.lanes_per_bead;
    if (eo.lds_beads_max == 0) eo.lds_beads_max = def.lds_beads_max;
    if (eo.pl_shell == 0.0f) eo.pl_shell = def.pl_shell;
    if (!(eo.pl_shell > 0.0f) || eo.pl_shell > 8.0f) eo.pl_shell = 0.0f;
  }
  const int lpb = eo.lanes_per_bead;
  const int stt = eo.step_tiles;
  // the step kernel holds a bead's pair-list and native pair-list lengths in
  // 16 bits each, and a row's offset within its tile's region in 16 bits
  // (units of ROW_PAD entries): pl_cap_max <= 4095 (natives per bead and per
  // tile are checked at add)
  if ((lpb != 4 && lpb != 8 && lpb != 16 && lpb != 32) ||
      (stt != 0 && stt != 1 && stt != 2 && stt != 4 && stt != 8 && stt != 16) || eo.pl_cap_max > 4095)
    return SOP_ERR_INVALID;
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return SOP_ERR_NO_DEVICE;
  if (device < 0 || device >= count) return SOP_ERR_NO_DEVICE;
  (void)hipGetLastError();  // do not inherit an error left by earlier calls
  sop_engine *e = new sop_engine();
  e->opts = eo;
  e->device = device;
  if (hipSetDevice(device) != hipSuccess) {
    delete e;
    return SOP_ERR_NO_DEVICE;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) {
    delete e;
    return SOP_ERR_HIP;
  }
  e->num_cu = prop.multiProcessorCount;
  // the allocation-free entry point's scratch on this device (the device is current)
  if (noalloc_scratch(device, &e->scratch) != hipSuccess) {
    (void)hipGetLastError();
    e->scratch = nullptr;
  }
  e->step_blocks = e->opts.step_blocks > 0 ? e->opts.step_blocks : 0;
  e->tune.tail = e->opts.step_tail == 2 || e->opts.step_tail == 4 ? e->opts.step_tail : 0;
  // the step kernel keeps 1 KB of static LDS for the tile's forces
  e->lds_limit = prop.sharedMemPerBlock > 2048 ? prop.sharedMemPerBlock - 2048 : 0;
  if (step_lds_limit(e->lds_limit) != hipSuccess) {
    (void)hipGetLastError();
    e->lds_limit = 65536 - 2048;
  }
  // the shell filter's launches need their LDS sizes: no fallback
  if (filter_lds_init() != hipSuccess) {
    (void)hipGetLastError();
    delete e;
    return SOP_ERR_HIP;
  }
  {
    const int64_t whole = (int64_t)(e->lds_limit / 16) / TILE * TILE;
    e->lds_big_cap = e->opts.lds_beads_max > 0 && whole > e->opts.lds_beads_max ? whole : 0;
  }
  // A blocking stream: synchronous hipMemcpy calls on the null stream order
  // after the engine's kernels, so host reads never race device writes.
  if (hipStreamCreate(&e->stream) != hipSuccess) {
    delete e;
    return SOP_ERR_HIP;
  }
  if (hipStreamCreate(&e->fork.side) != hipSuccess ||
      hipEventCreateWithFlags(&e->fork.fork, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&e->fork.join, hipEventDisableTiming) != hipSuccess) {
    (void)hipGetLastError();
    sop_engine_destroy(e);
    return SOP_ERR_HIP;
  }
  bind_arrays(e);
  // Lane-layout self test of the DPP / swizzle / ballot helpers.
  int *d_out = nullptr;
  float *d_f = nullptr;
  int h_out[64] = {0};
  hipError_t h1 = hipMalloc((void **)&d_out, 64 * 4);
  hipError_t h2 = h1 == hipSuccess ? hipMalloc((void **)&d_f, 64 * 12) : h1;
  hipError_t h3 = h2 == hipSuccess ? launch_selftest(d_out, d_f, e->stream) : h2;
  hipError_t h3s = h3 == hipSuccess ? hipStreamSynchronize(e->stream) : h3;
  hipError_t h4 = h3s == hipSuccess ? hipMemcpy(h_out, d_out, 64 * 4, hipMemcpyDeviceToHost) : h3s;
  bool ok = h4 == hipSuccess;
  for (int k = 0; ok && k < 64; ++k) ok = h_out[k] == 0;
  if (d_out) (void)hipFree(d_out);
  if (d_f) (void)hipFree(d_f);
  if (!ok) {
    std::fprintf(stderr, "sop_engine_create: self test failed (%s / %s / %s / %s, lane0 bits %d)\n",
                 hipGetErrorString(h1), hipGetErrorString(h2), hipGetErrorString(h3), hipGetErrorString(h4),
                 h_out[0]);
    sop_engine_destroy(e);
    return SOP_ERR_HIP;
  }
  if (e->opts.pool_bytes > 0) {
    // fixed pools sized from the budget (serving): split by typical use (per
    // bead ~200 B + 2 * pl_cap entries of 2 B; the pair-list and shell-row
    // segments dominate); the neighbor-list scratch grows on request
    const int64_t B = e->opts.pool_bytes;
    const int64_t beads = std::max<int64_t>(4096, B / 8 / 200) / TILE * TILE;
    const int64_t nat = std::max<int64_t>(4096, B / 64 / 24);
    const int64_t pl = std::max<int64_t>(65536, B * 3 / 4 / 8);
    const int64_t cells = std::max<int64_t>(65536, B / 64 / 12);
    sop_status st = ensure_capacity(e, beads, nat, 0, pl, cells, 4096);
    if (st) {
      sop_engine_destroy(e);
      return st;
    }
    e->fixed_pools = true;
  }
  *out = e;
  return SOP_OK;
}

void sop_engine_destroy(sop_engine *e) {
  if (!e) return;
  if (e->serve) sop_serve_stop(e);
  hipError_t first = hipSuccess;
  const char *what = "";
  auto note = [&](hipError_t h, const char *w) {
    if (h != hipSuccess && first == hipSuccess) { first = h; what = w; }
  };
  note(hipSetDevice(e->device), "hipSetDevice");
  if (e->stream) note(hipStreamSynchronize(e->stream), "hipStreamSynchronize");
  for (auto &kv : e->graphs) note(hipGraphExecDestroy(kv.second), "hipGraphExecDestroy");
  for (auto &a : e->bead_arrays) if (*a.first) note(hipFree(*a.first), "hipFree(bead pool)");
  for (auto &a : e->nat_arrays) if (*a.first) note(hipFree(*a.first), "hipFree(native pool)");
  for (auto &a : e->cell_arrays) if (*a.first) note(hipFree(*a.first), "hipFree(cell pool)");
  void *others[] = {e->p.nlrep_j, e->p.plrep_j, e->p.slrep_j,  e->p.tile_sys, e->p.sys,  e->p.sysout,
                    e->p.syslist, e->p.work,    e->p.nwork,    e->p.items,
                    e->p.tiles,   e->p.epart};
  for (void *q : others) if (q) note(hipFree(q), "hipFree");
  for (void *q : {e->io.ptr, e->stage.ptr, (void *)e->p.rep}) if (q) note(hipHostFree(q), "hipHostFree");
  if (e->p.fitems) note(hipFree(e->p.fitems), "hipFree");
  if (e->fork.side) note(hipStreamSynchronize(e->fork.side), "hipStreamSynchronize");
  if (e->fork.fork) note(hipEventDestroy(e->fork.fork), "hipEventDestroy");
  if (e->fork.join) note(hipEventDestroy(e->fork.join), "hipEventDestroy");
  if (e->fork.side) note(hipStreamDestroy(e->fork.side), "hipStreamDestroy");
  if (e->stream) note(hipStreamDestroy(e->stream), "hipStreamDestroy");
  if (first != hipSuccess) std::fprintf(stderr, "sop_engine_destroy: %s: %s\n", what, hipGetErrorString(first));
  (void)hipGetLastError();
  delete e;
}

const char *sop_last_error(const sop_engine *e) { return e ? e->err.c_str() : "no engine"; }

sop_status sop_synchronize(sop_engine *e) {
  if (!e) return SOP_ERR_INVALID;
  const EngineLock lk(e->mu);
  return hip_check(e, hipStreamSynchronize(e->stream), "hipStreamSynchronize");
}

// The lock of a call, which may be given no engine.
static EngineLock call_lock(sop_engine *e) { return e ? EngineLock(e->mu) : EngineLock(); }

static bool valid_sys(sop_engine *e, int32_t s) {
  return e && s >= 0 && s < (int32_t)e->sys.size() && e->sys[s].used;
}

sop_status sop_system_add(sop_engine *e, const sop_system_desc *d, int32_t *sys) {
  if (!e || !sys) return SOP_ERR_INVALID;
  if (e->serve) return set_error(e, SOP_ERR_STATE, "engine is serving");
  return engine_add_system(e, d, sys);
}

sop_status sop_system_remove(sop_engine *e, int32_t sys) {
  if (!e) return SOP_ERR_INVALID;
  const EngineLock lk(e->mu);
  HIPCK(hipStreamSynchronize(e->stream));
  return engine_remove_system(e, sys);
}

sop_status sop_system_info(sop_engine *e, int32_t sys, int32_t *n_beads, int64_t *step) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys)) return set_error(e, SOP_ERR_INVALID, "no such system");
  if (n_beads) *n_beads = e->sys[sys].n;
  if (step) *step = e->sys[sys].step;
  return SOP_OK;
}

// The neighbor list is written only on request, into one scratch segment
// (grown to fit) that holds the rows of the last system materialized.
static sop_status nl_scratch_for(sop_engine *e, int32_t sys) {
  sop_status st = ensure_capacity(e, 0, 0, e->sys[sys].nl_len, 0, 0, 0);
  if (st) return st;
  if (e->nl_owner != sys) {  // the scratch holds another system's rows
    const int32_t zero = 0;
    HIPCK(hipMemcpy(&e->p.sys[sys].nl_valid, &zero, sizeof(zero), hipMemcpyHostToDevice));
  }
  e->nl_owner = sys;
  return SOP_OK;
}

sop_status sop_update_neighbor_list(sop_engine *e, int32_t sys) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys)) return set_error(e, SOP_ERR_INVALID, "no such system");
  sop_status st = nl_scratch_for(e, sys);
  if (st) return st;
  st = engine_set_batch(e, &sys, 1);
  if (st) return st;
  HIPCK(launch_lists(e->p, list_grids(e), 0, FORCE_NL, e->stream));
  return engine_check_errors(e, &sys, 1);
}

sop_status sop_update_pair_list(sop_engine *e, int32_t sys) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys)) return set_error(e, SOP_ERR_INVALID, "no such system");
  sop_status st = engine_set_batch(e, &sys, 1);
  if (st) return st;
  HIPCK(launch_lists(e->p, list_grids(e), 0, FORCE_PL, e->stream));
  return engine_check_errors(e, &sys, 1);
}

// The neighbor list is materialized on demand from its snapshot.
static sop_status materialize_nl(sop_engine *e, int32_t sys) {
  sop_status st = nl_scratch_for(e, sys);
  if (st) return st;
  st = engine_set_batch(e, &sys, 1);
  if (st) return st;
  HIPCK(launch_lists(e->p, list_grids(e), 0, MATERIALIZE_NL, e->stream));
  return engine_check_errors(e, &sys, 1);
}

sop_status sop_get_list(sop_engine *e, int32_t sys, int32_t which, int32_t *ij, int64_t cap, int64_t *n) {
  const EngineLock lk = call_lock(e);
  static_assert(LIST_NL_ATT == SOP_LIST_NL_NATIVE && LIST_NL_REP == SOP_LIST_NL_REP &&
                    LIST_PL_ATT == SOP_LIST_PL_NATIVE && LIST_PL_REP == SOP_LIST_PL_REP, "list ids");
  if (!valid_sys(e, sys) || !n) return set_error(e, SOP_ERR_INVALID, "bad arguments");
  if (which < LIST_NL_ATT || which > LIST_PL_REP) return set_error(e, SOP_ERR_INVALID, "unknown list");
  sop_status st = SOP_OK;
  if (which == SOP_LIST_NL_NATIVE || which == SOP_LIST_NL_REP) {
    st = materialize_nl(e, sys);
    if (st) return st;
  }
  const int32_t nb = e->sys[sys].n;
  // pairs go through the host buffer a window at a time, the total behind it;
  // the first window is written before the total is known, with one wait for
  // both, and is what the buffer holds (at least FIRST pairs): a caller's array
  // may be far longer than the list, and pinned memory for all of it costs 0.3
  // ms a MiB.  Later windows, for which the buffer grows, hold up to WINDOW
  constexpr int64_t WINDOW = (int64_t)4 << 20, FIRST = (int64_t)64 << 10;
  const int64_t room = ij ? std::max<int64_t>(cap, 0) : 0;
  int64_t m = std::min(room, std::clamp<int64_t>((int64_t)(e->io.bytes / 8) - 1, FIRST, WINDOW));
  int64_t total = 0;
  for (int64_t lo = 0;;) {
    if ((st = engine_io(e, e->io, 8 * (size_t)(m + 1)))) return st;
    int2 *const pairs = static_cast<int2 *>(e->io.ptr);
    int64_t *const count = static_cast<int64_t *>(e->io.ptr) + m;
    HIPCK(launch_list_places(e->p, sys, nb, which, lo, count, e->stream));
    if (m > 0) HIPCK(launch_list_write(e->p, sys, nb, which, pairs, (int)m, e->stream));
    HIPCK(hipStreamSynchronize(e->stream));
    total = *count;
    const int64_t want = std::min(total, room);
    if (want > lo) std::memcpy(ij + 2 * lo, pairs, 8 * (size_t)std::min(m, want - lo));
    lo += m;
    if (lo >= want) break;
    m = std::min(want - lo, WINDOW);
  }
  *n = total;
  return SOP_OK;
}

sop_status sop_system_rows(sop_engine *e, int32_t sys, int32_t *capacity, int32_t *longest) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys)) return set_error(e, SOP_ERR_INVALID, "no such system");
  HIPCK(hipStreamSynchronize(e->stream));
  SysDev S;
  const sop_status st = engine_read_sys(e, sys, &S);
  if (st) return st;
  if (capacity) *capacity = e->sys[sys].pl_cap;
  if (longest) *longest = S.row_max;
  return SOP_OK;
}

sop_status sop_system_reserve_rows(sop_engine *e, int32_t sys, int32_t capacity) {
  if (!valid_sys(e, sys) || capacity < 1) return set_error(e, SOP_ERR_INVALID, "bad arguments");
  if (e->serve) return set_error(e, SOP_ERR_STATE, "engine is serving");
  HIPCK(hipStreamSynchronize(e->stream));
  SysDev S;
  const sop_status st = engine_read_sys(e, sys, &S);
  if (st) return st;
  const SysHost &h = e->sys[sys];
  const int32_t cap = std::min(pl_cap_limit(e, h.n), std::max(round_up(capacity, 16), round_up(S.row_max, 16)));
  return engine_resize_rows(e, sys, cap, true);
}

sop_status sop_list_stats_get(sop_engine *e, int32_t sys, sop_list_stats *stt) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys) || !stt) return set_error(e, SOP_ERR_INVALID, "bad arguments");
  HIPCK(hipStreamSynchronize(e->stream));
  sop_status st = materialize_nl(e, sys);
  if (st) return st;
  const SysHost &h = e->sys[sys];
  std::vector<int32_t> c((size_t)h.n);
  int64_t tot[4];
  int32_t mx[4];
  int32_t *arrs[4] = {e->p.nlatt_cnt, e->p.nlrep_cnt, e->p.platt_cnt, e->p.plrep_cnt};
  for (int q = 0; q < 4; ++q) {
    HIPCK(hipMemcpy(c.data(), arrs[q] + h.bead_off, 4 * (size_t)h.n, hipMemcpyDeviceToHost));
    tot[q] = 0;
    mx[q] = 0;
    for (int32_t v : c) { tot[q] += v; mx[q] = std::max(mx[q], v); }
  }
  stt->nl_native = tot[0] / 2;
  stt->nl_rep = tot[1] / 2;
  stt->pl_native = tot[2] / 2;
  stt->pl_rep = tot[3] / 2;
  stt->nl_max_per_bead = mx[1];
  stt->pl_max_per_bead = mx[3];
  SysDev S;
  st = engine_read_sys(e, sys, &S);
  if (st) return st;
  stt->grid_builds = S.nbuild[0];
  stt->shell_builds = S.nbuild[1];
  stt->nl_builds = S.nbuild[2];
  return SOP_OK;
}

sop_status sop_force_eval(sop_engine *e, int32_t sys, int32_t with_noise) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys)) return set_error(e, SOP_ERR_INVALID, "no such system");
  sop_status st = engine_set_batch(e, &sys, 1);
  if (st) return st;
  HIPCK(launch_step(e->p, with_noise ? MODE_FORCE_NOISE : MODE_FORCE, e->opts.lanes_per_bead, step_grids(e), 0,
                    e->stream));
  return engine_check_errors(e, &sys, 1);
}

// Per-bead values of a system in the host buffer (after a 64-byte header),
// with the stream done.
static sop_status read_beads(sop_engine *e, int32_t sys, int what, const float **out, int64_t *step) {
  const SysHost &h = e->sys[sys];
  sop_status st = engine_io(e, e->io, 64 + 16 * (size_t)h.n);
  if (st) return st;
  float *f = reinterpret_cast<float *>(static_cast<char *>(e->io.ptr) + 64);
  HIPCK(launch_read(e->p, sys, h.n, what, f, static_cast<int64_t *>(e->io.ptr), e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  *out = f;
  if (step) *step = *static_cast<const int64_t *>(e->io.ptr);
  return SOP_OK;
}

sop_status sop_get_forces(sop_engine *e, int32_t sys, float *f3n) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys) || !f3n) return set_error(e, SOP_ERR_INVALID, "bad arguments");
  const float *f = nullptr;
  const sop_status st = read_beads(e, sys, READ_FORCES, &f, nullptr);
  if (st) return st;
  std::memcpy(f3n, f, 12 * (size_t)e->sys[sys].n);
  return SOP_OK;
}

static sop_status eval_energy(sop_engine *e, int32_t sys, double *out) {
  const SysHost &h = e->sys[sys];
  const sop_status st = engine_io(e, e->io, 8 * SYSOUT_N);
  if (st) return st;
  const int nt = (int)(h.bead_len / TILE);
  HIPCK(launch_energy_one(e->p, (int)(h.bead_off / TILE), nt, sys, std::min(nt, 2 * e->num_cu),
                          static_cast<double *>(e->io.ptr), e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  std::memcpy(out, e->io.ptr, 8 * 12);
  return SOP_OK;
}

sop_status sop_energy_eval(sop_engine *e, int32_t sys, double *energies) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys) || !energies) return set_error(e, SOP_ERR_INVALID, "bad arguments");
  double o[SYSOUT_N];
  sop_status st = eval_energy(e, sys, o);
  if (st) return st;
  for (int k = 0; k < SOP_E_COUNT; ++k) energies[k] = o[k];
  return SOP_OK;
}

sop_status sop_energy_eval_noalloc(sop_engine *e, int32_t sys, double *energies) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys) || !energies) return set_error(e, SOP_ERR_INVALID, "bad arguments");
  if (!e->scratch) return set_error(e, SOP_ERR_HIP, "sop_energy_eval_noalloc: no scratch address on this device");
  const SysHost &h = e->sys[sys];
  if (h.n > NOALLOC_BEADS) {
    std::ostringstream os;
    os << "sop_energy_eval_noalloc: system " << sys << " has " << h.n << " beads, above the scratch limit of "
       << NOALLOC_BEADS;
    return set_error(e, SOP_ERR_CAPACITY, os.str());
  }
  // the engine's arrays, with the partials and values in scratch
  DevPtrs q = e->p;
  char *b = static_cast<char *>(e->scratch);
  q.epart = reinterpret_cast<double *>(b);
  q.epart_base = (int32_t)h.bead_off;
  q.sysout = reinterpret_cast<double *>(b + NOALLOC_OFF_SYSOUT);
  q.sysout_base = sys;
  const int nt = (int)(h.bead_len / TILE);
  HIPCK(launch_energy_one(q, (int)(h.bead_off / TILE), nt, sys, std::min(nt, 2 * e->num_cu), nullptr, e->stream));
  double o[SYSOUT_N];
  HIPCK(hipMemcpyAsync(o, q.sysout, sizeof(o), hipMemcpyDeviceToHost, e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  for (int k = 0; k < SOP_E_COUNT; ++k) energies[k] = o[k];
  return SOP_OK;
}

sop_status sop_observables(sop_engine *e, int32_t sys, double *Q, int32_t *contacts, double *rgsq) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys)) return set_error(e, SOP_ERR_INVALID, "no such system");
  double o[SYSOUT_N];
  sop_status st = eval_energy(e, sys, o);
  if (st) return st;
  const int32_t c = (int32_t)std::llround(o[6]);
  if (contacts) *contacts = c;
  if (Q) *Q = e->sys[sys].n_nat > 0 ? (double)c / (double)e->sys[sys].n_nat : 0.0;
  if (rgsq) *rgsq = o[7];
  return SOP_OK;
}

static sop_status check_run_args(sop_engine *e, const int32_t *sys, int32_t nsys, int64_t nsteps) {
  if (!e || !sys || nsys <= 0 || nsteps < 0) return set_error(e, SOP_ERR_INVALID, "bad run arguments");
  if (e->serve) return set_error(e, SOP_ERR_STATE, "engine is serving");
  for (int q = 0; q < nsys; ++q) {
    if (!valid_sys(e, sys[q])) return set_error(e, SOP_ERR_INVALID, "no such system");
    for (int r = 0; r < q; ++r)
      if (sys[r] == sys[q]) return set_error(e, SOP_ERR_INVALID, "system listed twice");
  }
  return SOP_OK;
}

sop_status sop_run(sop_engine *e, const int32_t *sys, int32_t nsys, int64_t nsteps) {
  sop_status st = check_run_args(e, sys, nsys, nsteps);
  if (st) return st;
  return engine_run(e, sys, nsys, nsteps, nullptr, nullptr);
}

sop_status sop_run_plain(sop_engine *e, const int32_t *sys, int32_t nsys, int64_t nsteps) {
  sop_status st = check_run_args(e, sys, nsys, nsteps);
  if (st) return st;
  for (int q = 0; q < nsys; ++q) {
    st = engine_set_batch(e, &sys[q], 1);
    if (st) return st;
    HIPCK(launch_begin(e->p, nsteps, e->stream));
    st = engine_run_hostloop(e, nsteps);
    if (st) return st;
    if (nsteps == 0) HIPCK(launch_report(e->p, e->stream));  // no k_advance to report the state as it is now
    mirror_advance(e, &sys[q], 1, nsteps);
  }
  HIPCK(hipStreamSynchronize(e->stream));
  for (int q = 0; q < nsys; ++q) {  // as k_advance or k_report left them
    st = engine_error_status(e, sys[q], e->p.rep[sys[q]].x);
    if (st) return st;
  }
  return SOP_OK;
}

sop_status sop_get_coords(sop_engine *e, int32_t sys, float *xyz, int64_t *step) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys)) return set_error(e, SOP_ERR_INVALID, "no such system");
  const float *x = nullptr;
  const sop_status st = read_beads(e, sys, READ_COORDS, &x, step);
  if (st) return st;
  if (xyz) std::memcpy(xyz, x, 12 * (size_t)e->sys[sys].n);
  return SOP_OK;
}

sop_status sop_get_wrapped_coords(sop_engine *e, int32_t sys, float *xyz) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys) || !xyz) return set_error(e, SOP_ERR_INVALID, "bad arguments");
  const float *x = nullptr;
  const sop_status st = read_beads(e, sys, READ_COORDS, &x, nullptr);
  if (st) return st;
  const float boxl = e->sys[sys].params.boxl;
  const size_t m = 3 * (size_t)e->sys[sys].n;
  for (size_t k = 0; k < m; ++k) xyz[k] = boxl > 0.0f ? x[k] - boxl * rintf(x[k] / boxl) : x[k];
  return SOP_OK;
}

// Forces with noise of the current step (kstep 0) or of the last step taken
// (kstep -1: the other coordinate buffer and step - 1), three floats a bead.
static sop_status noisy_forces(sop_engine *e, int32_t sys, int kstep, std::vector<float> &f) {
  sop_status st = engine_set_batch(e, &sys, 1);
  if (st) return st;
  HIPCK(launch_step(e->p, MODE_FORCE_NOISE, e->opts.lanes_per_bead, step_grids(e), kstep, e->stream));
  st = engine_check_errors(e, &sys, 1);
  if (st) return st;
  const float *x = nullptr;
  st = read_beads(e, sys, READ_FORCES, &x, nullptr);
  if (st) return st;
  f.assign(x, x + 3 * (size_t)e->sys[sys].n);
  return SOP_OK;
}

static sop_status read_vel_state(sop_engine *e, int32_t sys, std::vector<float4> &v) {
  const float *x = nullptr;
  const sop_status st = read_beads(e, sys, READ_VEL, &x, nullptr);
  if (st) return st;
  v.resize((size_t)e->sys[sys].n);
  std::memcpy(v.data(), x, 16 * v.size());
  return SOP_OK;
}

static bool incr_flag(const float4 &s) {
  int32_t w;
  std::memcpy(&w, &s.w, 4);
  return w == 1;
}

sop_status sop_get_velocities(sop_engine *e, int32_t sys, float *v3n) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys) || !v3n) return set_error(e, SOP_ERR_INVALID, "bad arguments");
  const SysHost &h = e->sys[sys];
  if (h.params.dynamics != SOP_DYN_UNDERDAMPED) {
    std::fill(v3n, v3n + 3 * (size_t)h.n, 0.0f);
    return SOP_OK;
  }
  std::vector<float4> v;
  std::vector<float> f;
  sop_status st = read_vel_state(e, sys, v);
  if (st) return st;
  bool any = false;
  for (const auto &s : v) any |= incr_flag(s);
  if (any && (st = noisy_forces(e, sys, 0, f))) return st;
  float a[4];
  sop_params_underdamped(&h.params, a);
  for (int i = 0; i < h.n; ++i) {
    const float4 s = v[i];
    if (incr_flag(s)) {
      v3n[3 * i] = a[2] * s.x + a[3] * f[3 * i];
      v3n[3 * i + 1] = a[2] * s.y + a[3] * f[3 * i + 1];
      v3n[3 * i + 2] = a[2] * s.z + a[3] * f[3 * i + 2];
    } else {
      v3n[3 * i] = s.x;
      v3n[3 * i + 1] = s.y;
      v3n[3 * i + 2] = s.z;
    }
  }
  return SOP_OK;
}

sop_status sop_get_increments(sop_engine *e, int32_t sys, float *d3n) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys) || !d3n) return set_error(e, SOP_ERR_INVALID, "bad arguments");
  const SysHost &h = e->sys[sys];
  std::vector<float4> v;
  std::vector<float> f;
  sop_status st;
  if (h.params.dynamics == SOP_DYN_UNDERDAMPED) {
    if ((st = read_vel_state(e, sys, v))) return st;
    bool all = true;
    for (const auto &s : v) all &= incr_flag(s);
    if (!all && (st = noisy_forces(e, sys, -1, f))) return st;
    float a[4];
    sop_params_underdamped(&h.params, a);
    for (int i = 0; i < h.n; ++i) {
      const float4 s = v[i];
      if (incr_flag(s)) {
        d3n[3 * i] = s.x;
        d3n[3 * i + 1] = s.y;
        d3n[3 * i + 2] = s.z;
      } else {
        d3n[3 * i] = a[0] * s.x + a[1] * f[3 * i];
        d3n[3 * i + 1] = a[0] * s.y + a[1] * f[3 * i + 1];
        d3n[3 * i + 2] = a[0] * s.z + a[1] * f[3 * i + 2];
      }
    }
    return SOP_OK;
  }
  if ((st = noisy_forces(e, sys, -1, f))) return st;
  float a5, var;
  sop_params_derived(&h.params, &a5, &var);
  for (size_t k = 0; k < f.size(); ++k) d3n[k] = a5 * f[k];
  return SOP_OK;
}

sop_status sop_set_rng(sop_engine *e, int32_t sys, uint64_t seed, int64_t step) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys)) return set_error(e, SOP_ERR_INVALID, "no such system");
  if (step < 0) return set_error(e, SOP_ERR_INVALID, "step must be >= 0");
  SysDev S;
  sop_status st = engine_read_sys(e, sys, &S);
  if (st) return st;
  S.seed_lo = (uint32_t)seed;
  S.seed_hi = (uint32_t)(seed >> 32);
  S.step = step;
  S.step_end = step;
  HIPCK(hipMemcpy(e->p.sys + sys, &S, sizeof(SysDev), hipMemcpyHostToDevice));
  SysHost &h = e->sys[sys];
  h.params.seed = seed;
  h.step = step;
  return SOP_OK;
}

sop_status sop_set_coords(sop_engine *e, int32_t sys, const float *xyz) {
  const EngineLock lk = call_lock(e);
  if (!valid_sys(e, sys) || !xyz) return set_error(e, SOP_ERR_INVALID, "bad arguments");
  const size_t bytes = 12 * (size_t)e->sys[sys].n;
  sop_status st = engine_io(e, e->io, bytes);
  if (st) return st;
  std::memcpy(e->io.ptr, xyz, bytes);
  // new coordinates clear the system's sticky error bits
  HIPCK(launch_write_coords(e->p, sys, e->sys[sys].n, static_cast<const float *>(e->io.ptr), e->stream));
  HIPCK(hipStreamSynchronize(e->stream));  // the buffer is the next call's
  return SOP_OK;
}

sop_status sop_time_step_kernel(sop_engine *e, const int32_t *sys, int32_t nsys, int32_t reps, double *avg_ms) {
  sop_status st = check_run_args(e, sys, nsys, reps);
  if (st) return st;
  if (reps <= 0 || !avg_ms) return set_error(e, SOP_ERR_INVALID, "reps > 0 and avg_ms required");
  st = engine_set_batch(e, sys, nsys);
  if (st) return st;
  // Timing leaves no trace: coordinates and system descriptors are restored.
  const size_t pos_bytes = 16 * (size_t)e->cap.beads, sys_bytes = sizeof(SysDev) * (size_t)e->cap.slots;
  void *save = nullptr;
  HIPCK(hipMalloc(&save, 2 * pos_bytes + sys_bytes));
  char *sv = (char *)save;
  HIPCK(hipMemcpyAsync(sv, e->p.pos0, pos_bytes, hipMemcpyDeviceToDevice, e->stream));
  HIPCK(hipMemcpyAsync(sv + pos_bytes, e->p.pos1, pos_bytes, hipMemcpyDeviceToDevice, e->stream));
  HIPCK(hipMemcpyAsync(sv + 2 * pos_bytes, e->p.sys, sys_bytes, hipMemcpyDeviceToDevice, e->stream));
  HIPCK(launch_begin(e->p, reps, e->stream));
  hipEvent_t a, b;
  HIPCK(hipEventCreate(&a));
  HIPCK(hipEventCreate(&b));
  const int lpb = e->opts.lanes_per_bead;
  HIPCK(hipEventRecord(a, e->stream));
  for (int r = 0; r < reps; ++r) HIPCK(launch_step(e->p, MODE_STEP, lpb, step_grids(e), r, e->stream));
  HIPCK(hipEventRecord(b, e->stream));
  HIPCK(hipEventSynchronize(b));
  float ms = 0.0f;
  HIPCK(hipEventElapsedTime(&ms, a, b));
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  HIPCK(hipMemcpyAsync(e->p.pos0, sv, pos_bytes, hipMemcpyDeviceToDevice, e->stream));
  HIPCK(hipMemcpyAsync(e->p.pos1, sv + pos_bytes, pos_bytes, hipMemcpyDeviceToDevice, e->stream));
  HIPCK(hipMemcpyAsync(e->p.sys, sv + 2 * pos_bytes, sys_bytes, hipMemcpyDeviceToDevice, e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  HIPCK(hipFree(save));
  *avg_ms = ms / reps;
  return SOP_OK;
}

// Device self test for the tests: per-lane failure bits of the wave helpers
// and 64 x 3 device normals for (seed 0x9abcdef012345678, bead = lane,
// step = 1000 + lane).
sop_status sop_selftest(sop_engine *e, int32_t *bad64, float *normals192) {
  if (!e) return SOP_ERR_INVALID;
  int *d_out = nullptr;
  float *d_f = nullptr;
  HIPCK(hipMalloc((void **)&d_out, 64 * 4));
  HIPCK(hipMalloc((void **)&d_f, 64 * 12));
  HIPCK(launch_selftest(d_out, d_f, e->stream));
  HIPCK(hipStreamSynchronize(e->stream));
  HIPCK(hipMemcpy(bad64, d_out, 64 * 4, hipMemcpyDeviceToHost));
  HIPCK(hipMemcpy(normals192, d_f, 64 * 12, hipMemcpyDeviceToHost));
  (void)hipFree(d_out);
  (void)hipFree(d_f);
  return SOP_OK;
}

} // extern "C"
