// kernels.hip -- gfx950 kernels of the SOP overdamped hot path.
//
//   k_rebuild (k_big_skin / k_big_plan / k_cell_* for systems too large for
//   one block) / k_rows / k_shell_filter   list rebuilds: per-system open
//                cell grid, counting sort of beads into cells (histogram, DPP
//                wave scan, scatter, deterministic in-cell ranking), 27-cell
//                stencil with the exact FP32 predicates and ballot/mbcnt wave
//                compaction, pair-list rows filtered from shell rows and packed
//                per tile.  Replaces the reference's flag kernels + CUDPP
//                split/scan over the O(N^2) master list and its pair-list
//                filter (sop.cu:704-826, 835-920, 928-1262, 1456-1620,
//                1827-2608).
//   k_step       fused FENE + i,i+2 soft sphere + native LJ + non-native
//                repulsion gather (no atomics), group reduction over the lanes
//                of a bead, Philox4x32-10 random force, overdamped move
//                (energy.cu:81-167,228-604; sop.cu:487-520).
//   k_energy / k_sys_reduce   FP64 reductions of FP32 pair energies, virial,
//                native contacts and Rg^2 (energy.cu:194-442, sop.cu:528-611).
//
// Every kernel walks a device-resident work table with a grid-stride loop, so
// one launch covers any batch of systems and a captured graph stays valid when
// the batch changes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>

#include "sop_dev.h"

namespace sopk {

// ---------------------------------------------------------------- helpers

__device__ __forceinline__ int w_type(float w) { return __float_as_int(w) & 3; }
__device__ __forceinline__ int w_chain(float w) { return __float_as_int(w) >> 2; }

__device__ __forceinline__ const float4 *buf_in(const DevPtrs &p, int parity) {
  return (parity & 1) ? p.pos1 : p.pos0;
}
__device__ __forceinline__ float4 *buf_out(const DevPtrs &p, int parity) {
  return (parity & 1) ? p.pos0 : p.pos1;
}

// Exact FP32 predicate pieces, same operation order and rounding as the
// reference's single-precision list kernels; this file is compiled with
// -ffp-contract=off and correctly rounded division/sqrt.
__device__ __forceinline__ float mi_exact(float d, float boxl) {
  if (boxl > 0.0f) {
    float q = d / boxl;
    float r = rintf(q);
    float pr = boxl * r;
    d = d - pr;
  }
  return d;
}

__device__ __forceinline__ float dist2_exact(float4 a, float4 b, float boxl) {
  float dx = mi_exact(b.x - a.x, boxl);
  float dy = mi_exact(b.y - a.y, boxl);
  float dz = mi_exact(b.z - a.z, boxl);
  float p = dx * dx;
  float q = dy * dy;
  float r = dz * dz;
  return (p + q) + r;
}

__device__ __forceinline__ float cutoff_of(double factor, float absval, float base) {
  return factor > 0.0 ? (float)(factor * (double)base) : absval;
}

// Fast minimum image for forces (not used by any list predicate).
__device__ __forceinline__ float mi_fast(float d, float boxl, float inv_boxl) {
  return d - boxl * rintf(d * inv_boxl);
}

__device__ __forceinline__ float rcpf(float x) { return __builtin_amdgcn_rcpf(x); }

// DPP lane moves.  Controls: quad_perm [1,0,3,2] = 0xB1, [2,3,0,1] = 0x4E,
// row_half_mirror = 0x141, row_mirror = 0x140, row_shr:n = 0x110+n,
// row_bcast:15 = 0x142, row_bcast:31 = 0x143.
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

// Sum over aligned groups of W lanes; every lane of a group receives the sum.
template <int W>
__device__ __forceinline__ float group_sum(float v) {
  static_assert(W == 4 || W == 8 || W == 16 || W == 32 || W == 64, "group width");
  v += dpp_f<0xB1>(v);
  v += dpp_f<0x4E>(v);
  if (W >= 8) v += dpp_f<0x141>(v);
  if (W >= 16) v += dpp_f<0x140>(v);
  if (W >= 32) {
    // xor 16 inside each 32-lane half: ds_swizzle bit mode, and=0x1F, xor=0x10
    v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401F));
  }
  if (W >= 64) v += __shfl_xor(v, 32);
  return v;
}

__device__ __forceinline__ int wave_sum_i(int v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Maximum over the wave of values >= 0, in lane 63.
__device__ __forceinline__ float wave_max63(float v) {
  auto step = [&](int shifted) { v = fmaxf(v, __int_as_float(shifted)); };
  step(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xF, 0xF, false));
  step(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x112, 0xF, 0xF, false));
  step(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xF, 0xF, false));
  step(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x118, 0xF, 0xF, false));
  step(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x142, 0xA, 0xF, false));
  step(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x143, 0xC, 0xF, false));
  return v;
}

// Inclusive prefix sum across the 64 lanes of a wave with DPP: Hillis-Steele
// inside each 16-lane row (row_shr 1,2,4,8), then row_bcast15 / row_bcast31
// carry row totals into the rows above.
__device__ __forceinline__ int wave_incl_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);
  return v;
}

// Maximum over the wave's lanes (all lanes active).
__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = max(v, __shfl_xor(v, o));
  return v;
}

// Number of set bits of mask in lanes below this one (ballot prefix).
__device__ __forceinline__ int lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}

// Philox4x32-10 (Salmon et al., SC'11).
__device__ __forceinline__ uint4 philox10(uint4 c, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    // one 32x32->64 product per multiplier (v_mad_u64_u32) instead of
    // separate low and high multiplies
    const uint64_t p0 = (uint64_t)0xD2511F53u * c.x, p1 = (uint64_t)0xCD9E8D57u * c.z;
    c = make_uint4((uint32_t)(p1 >> 32) ^ c.y ^ k0, (uint32_t)p1, (uint32_t)(p0 >> 32) ^ c.w ^ k1, (uint32_t)p0);
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return c;
}

// 24-bit uniform in (0,1): odd multiples of 2^-24, exact in float.
__device__ __forceinline__ float u24(uint32_t r) {
  return (float)((r >> 8) | 1u) * 5.9604644775390625e-08f;
}

// Three standard normals for (seed, bead, step): Box-Muller on Philox output.
__device__ __forceinline__ void normals3(uint32_t k0, uint32_t k1, uint32_t bead, int64_t step,
                                         float &n0, float &n1, float &n2) {
  const uint4 r = philox10(make_uint4(bead, (uint32_t)step, (uint32_t)((uint64_t)step >> 32), 0u), k0, k1);
  const float ra = sqrtf(-2.0f * logf(u24(r.x)));
  const float rb = sqrtf(-2.0f * logf(u24(r.z)));
  float sa, ca, sb, cb;
  sincospif(2.0f * u24(r.y), &sa, &ca);
  sincospif(2.0f * u24(r.w), &sb, &cb);
  n0 = ra * ca;
  n1 = ra * sa;
  n2 = rb * cb;
}

// Loads through the scalar cache: one trip for all of a system's fields, where
// vector loads of values that steer the wave each wait in turn (three to eight
// trips to the L2 before a kernel's first bead).  For what no other block
// writes in the launch, and this one only after its reads.  Steps of one
// system: 128 beads 5.90 -> 5.51 us, 4,999 7.64 -> 7.04, 10,000 8.2 -> 7.6; 512
// replicas 69.6 -> 66.5 (the fields also leave the vector registers); the
// rebuild's decision 6.7 -> 5.7; rows, cells and filter of 200,000 beads 150
// -> 100 us a rebuild.
typedef const __attribute__((address_space(4))) SysDev SysConst;
__device__ __forceinline__ SysConst &sys_const(const DevPtrs &p, int s) { return *(SysConst *)(uintptr_t)(p.sys + s); }
__device__ __forceinline__ int sload(const int32_t *q) {
  return *(const __attribute__((address_space(4))) int *)(uintptr_t)q;
}
__device__ __forceinline__ int2 sload(const int2 *q) {
  typedef int v2 __attribute__((ext_vector_type(2)));
  const v2 v = *(const __attribute__((address_space(4))) v2 *)(uintptr_t)q;
  return make_int2(v.x, v.y);
}
__device__ __forceinline__ int4 sload(const int4 *q) {
  typedef int v4 __attribute__((ext_vector_type(4)));
  const v4 v = *(const __attribute__((address_space(4))) v4 *)(uintptr_t)q;
  return make_int4(v.x, v.y, v.z, v.w);
}

// Which rebuilds are due at step + kstep, or asked for by the flags.  The
// schedule's fields are read together (a short circuit between them would make
// each a round trip of its own), and steps below 2^32 take a 32-bit remainder.
struct Due {
  bool nl, pl;
};
__device__ __forceinline__ bool divides(int n, int64_t step) {
  return (uint64_t)step >> 32 ? step % n == 0 : (uint32_t)step % (uint32_t)n == 0;
}
template <typename Sys>
__device__ __forceinline__ Due rebuild_due(const Sys &S, int kstep, int flags) {
  const int64_t step = S.step + kstep, end = S.step_end;
  const int n_nl = S.n_nl, n_pl = S.n_pl;
  const bool mat = (flags & MATERIALIZE_NL) != 0, live = step < end;
  const bool nl = ((flags & FORCE_NL) != 0) | (live & divides(n_nl, step));
  const bool pl = ((flags & FORCE_PL) != 0) | (live & divides(n_pl, step));
  return Due{nl && !mat, pl && !mat};
}

template <typename G>
__device__ __forceinline__ int cell_index(const G &S, float4 x) {
  int cx = (int)floorf((x.x - S.org[0]) * S.inv_edge[0]);
  int cy = (int)floorf((x.y - S.org[1]) * S.inv_edge[1]);
  int cz = (int)floorf((x.z - S.org[2]) * S.inv_edge[2]);
  cx = min(max(cx, 0), S.dims[0] - 1);
  cy = min(max(cy, 0), S.dims[1] - 1);
  cz = min(max(cz, 0), S.dims[2] - 1);
  return (cz * S.dims[1] + cy) * S.dims[0] + cx;
}

// ------------------------------------------------------------ list rebuilds
//
// The neighbor list is defined by the snapshot pos_ref taken at its last
// rebuild: NL = master pairs with d2(pos_ref) < rc_nl^2, and the pair list is
// PL = NL pairs with d2(x) < rc_pl^2.  When every bead has moved less than
// skin/2 = (rc_nl - rc_pl)/2 since the snapshot, every pair with
// d(x) < rc_pl has d(pos_ref) < rc_pl + 2 max|dx| < rc_nl, so PL equals the
// master pairs with d2(x) < rc_pl^2: it is built straight from a cell grid of
// edge >= rc_pl (BUILD_DIRECT) and the neighbor list need not be written.
// Otherwise the neighbor list is materialized from pos_ref and filtered
// (BUILD_NL).  Both give the same set as the reference's two-level scheme.
//
// The direct build writes shell rows: master pairs with d(x) < rc_pl + shell,
// snapshot pos_shell = x, and the pair list is those rows filtered at x.  At a
// later direct-capable rebuild where every bead has moved less than shell/2
// since pos_shell, every pair with d(x) < rc_pl has d(pos_shell) < rc_pl +
// shell, so filtering the same rows again gives the same pair list without
// the cell grid (BUILD_SHELL).

// Systems whose rebuild sorts beads into a cell grid.
template <typename Sys>
__device__ __forceinline__ bool grid_build(const Sys &S) {
  return S.build != BUILD_NONE && S.build != BUILD_SHELL;
}

template <typename Sys>
__device__ __forceinline__ const float4 *build_src(const DevPtrs &p, const Sys &S, int kstep) {
  return S.build == BUILD_DIRECT ? buf_in(p, S.parity + kstep) : p.pos_ref;
}

// What a rebuild's decision reads, loaded with the system's other constants: in
// the deciding thread it would be one more round trip, behind the barrier.
struct BuildLimits {
  float skin, shell_ok;
  int32_t nl_valid, n_direct, n_shell, n_nl;
};

// A rebuild's decision for one system, from the largest displacements since
// the two snapshots (one thread).  Returns S.build.
__device__ __forceinline__ int decide_build(SysDev &S, const BuildLimits &lim, int flags, bool nl, bool pl,
                                            bool shell_chk, float d2max, float d2sh) {
  const float dmax = sqrtf(d2max), dsh = sqrtf(d2sh);
  int build = BUILD_NONE;
  if (flags & MATERIALIZE_NL) {
    build = lim.nl_valid ? BUILD_NONE : BUILD_NL_ONLY;
  } else {
    if (nl) S.nl_valid = 0;
    if (pl) {
      if (lim.skin > 0.0f && (nl || 2.0f * dmax < lim.skin))
        build = shell_chk && 2.0f * dsh < lim.shell_ok ? BUILD_SHELL : BUILD_DIRECT;
      else
        build = BUILD_NL;
    } else if (flags & FORCE_NL) {
      build = BUILD_NL_ONLY;
    }
  }
  S.build = build;
  if (build == BUILD_DIRECT) S.sl_valid = 1;
  if (build == BUILD_NL) S.sl_valid = 0;  // k_rows writes its rows into the shell-row slots
  if (build == BUILD_DIRECT) S.nbuild[0] = lim.n_direct + 1;
  if (build == BUILD_SHELL) S.nbuild[1] = lim.n_shell + 1;
  if (build == BUILD_NL) S.nbuild[2] = lim.n_nl + 1;
  return build;
}

// Cell grid of one axis range [a, b]: cells of the minimum edge, one more
// than fit in the extent so the grid covers it; when that exceeds dmax, dmax
// cells stretched over the extent (edge ext/dmax >= min_edge).  Stretching
// every cell to ext/floor(ext/min_edge) instead would make the 27-cell
// stencil up to 8x the volume it needs to be.
__device__ __forceinline__ void plan_axis(float a, float b, float min_edge, int dmax, int &dims, float &inv) {
  const float ext = b - a;
  dims = 1;
  inv = 0.0f;
  if (ext > 0.0f) {
    dims = (int)floorf(ext / min_edge) + 1;
    if (dims <= dmax) {
      inv = 1.0f / min_edge;
    } else {
      dims = dmax;
      inv = (float)dims / ext;
    }
  }
}

// The cell grid of a rebuild (one thread), from the bounding box mn..mx of
// the coordinates it sorts; a box too close to half the periodic box is
// refused (ERR_PBC).
struct CellGrid {
  float org[3], inv_edge[3];
  int dims[3];
};
__device__ __forceinline__ int plan_grid(SysDev &S, const float *mn, const float *mx, CellGrid &g) {
  const float min_edge = S.build == BUILD_DIRECT ? S.cell_min_edge_sl : S.cell_min_edge;
  const int dmax = S.dmax;
  float ext_max = 0.0f;
  int nc = 1;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    plan_axis(mn[d], mx[d], min_edge, dmax, g.dims[d], g.inv_edge[d]);
    g.org[d] = mn[d];
    nc *= g.dims[d];
    ext_max = fmaxf(ext_max, mx[d] - mn[d]);
    S.org[d] = g.org[d];
    S.inv_edge[d] = g.inv_edge[d];
    S.dims[d] = g.dims[d];
  }
  S.ncells = nc;
  int ok = 1;
  if (S.boxl > 0.0f) {
    ok = ext_max < 0.5f * S.boxl - S.wrap_margin;
    if (!ok) {
      atomicOr(&S.err, ERR_PBC);
      S.sl_valid = 0;
    }
  }
  S.wrap_free = ok;
  return nc;
}

// The entries s[st .. en) below b, eight at a time (s 16-byte aligned): the
// ranks read each cell once per member, bound by the block's one compute unit.
// Rebuild of 5,000 beads into 32 A cells of some 230 members: 75 us one entry
// at a time, 49 with eight comparisons a load, 38 with the packed ones.
__device__ __forceinline__ int count_below(const uint16_t *s, int st, int en, int b) {
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  int r = 0, m = st;
  for (const int a = min(en, (st + 7) & ~7); m < a; ++m) r += (int)s[m] < b;
  us2 acc = {0, 0};
  const us2 bb = {(unsigned short)b, (unsigned short)b}, one = {1, 1};
  for (; m + 8 <= en; m += 8) {
    const uint4 v = *reinterpret_cast<const uint4 *>(s + m);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {  // min(max(b - entry, 0), 1) in both halves
      uint32_t d;
      asm("v_pk_sub_u16 %0, %1, %2 clamp" : "=v"(d) : "v"(bb), "v"(w[k]));
      asm("v_pk_min_u16 %0, %1, %2" : "=v"(d) : "v"(d), "v"(one));
      acc += __builtin_bit_cast(us2, d);
    }
  }
  for (; m < en; ++m) r += (int)s[m] < b;
  return r + acc.x + acc.y;
}

// Rebuild of the systems whose cell sort fits one block's LDS (n <=
// SORT_N_MAX; at most 2 n cells, so every such system), one 1024-thread block
// per system.
//   PH_DECIDE  neighbor-list snapshot, displacements, which build it is
//   PH_GRID    for grid builds: bounding box, cell grid, the whole counting
//              sort in LDS -- cell of each bead, histogram, exclusive scan,
//              member lists, and the rank of each bead among its cell's
//              members by index, so the in-cell order is the index order --
//              the cell-ordered arrays, and the occupied cells appended to the
//              batch's home-cell list (in any order: each writes its own rows)
// What bounds it is latency: dependent round trips and block barriers of one
// block.  Both phases in one launch (a system's beads are loaded once) when
// the batch is small.  Run per step of one 128-bead system with lists at every
// step, by the chain of eleven kernels it replaced (most with nothing to do at
// most rebuilds) and by it: shell builds 46 and 18 us, grid builds 81 and 36.  A
// batch that fills the device launches the phases apart, the second on the side
// stream beside the shell builds' filter.  The sort's loads in flight take 128
// registers, one block per compute unit (and eight of them spill where both
// phases are one launch); the decision alone takes 63, two blocks.
constexpr int SORT_THREADS = 1024;
constexpr int PH_DECIDE = 1, PH_GRID = 2;

template <int PH>
__global__ __launch_bounds__(SORT_THREADS) void k_rebuild(DevPtrs p, int kstep, int flags) {
  constexpr int NW = SORT_THREADS / 64;
  constexpr int SB = SORT_N_MAX / SORT_THREADS;  // beads per thread
  __shared__ uint16_t s_cell[SORT_N_MAX];
  __shared__ __align__(16) uint16_t s_mem[SORT_N_MAX];
  __shared__ int s_cnt[SORT_C_MAX];  // counts, then end offsets
  __shared__ float s_red[6][NW];
  __shared__ int s_wsum[NW];
  __shared__ CellGrid s_grid;
  __shared__ int s_build, s_ncells, s_item0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nsys = *p.nsys;
  for (int q = *p.nbig + blockIdx.x; q < nsys; q += gridDim.x) {
    const int s = __builtin_amdgcn_readfirstlane(p.syslist[q]);
    SysDev &S = p.sys[s];
    // system constants in registers (the stores below may alias S)
    SysConst &C = sys_const(p, s);
    const int bo = C.bead_off, n = C.n;
    const float4 *x = buf_in(p, C.parity + kstep);
    float4 xs[SB];
    int build;
    bool loaded = false;
    if (PH & PH_DECIDE) {
      const BuildLimits lim{C.skin, C.shell_ok, C.nl_valid, C.nbuild[0], C.nbuild[1], C.nbuild[2]};
      const bool rows = C.sl_valid != 0;
      const Due due = rebuild_due(C, kstep, flags);
      const bool nl = due.nl, pl = due.pl, shell_chk = pl & rows;
      float d2max = 0.0f, d2sh = 0.0f;
      loaded = nl || pl;
      if (loaded) {
        // no branch on the bead count, so the loads issue together (a bead
        // past the end repeats the last one: the same snapshot store, the
        // same displacement)
#pragma unroll
        for (int u = 0; u < SB; ++u) xs[u] = x[bo + min(tid + u * SORT_THREADS, n - 1)];
        if (nl) {
#pragma unroll
          for (int u = 0; u < SB; ++u)
            if (u * SORT_THREADS < n) p.pos_ref[bo + min(tid + u * SORT_THREADS, n - 1)] = xs[u];
        }
        // (the fences keep each group of loads ahead of its uses)
        auto farthest = [&](const float4 *from) -> float {
          float4 r[SB];
          float m = 0.0f;
#pragma unroll
          for (int u = 0; u < SB; ++u) r[u] = from[bo + min(tid + u * SORT_THREADS, n - 1)];
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int u = 0; u < SB; ++u) {
            const float dx = xs[u].x - r[u].x, dy = xs[u].y - r[u].y, dz = xs[u].z - r[u].z;
            m = fmaxf(m, dx * dx + dy * dy + dz * dz);
          }
          return m;
        };
        if (!nl) d2max = farthest(p.pos_ref);
        if (shell_chk) d2sh = farthest(p.pos_shell);
        d2max = wave_max63(d2max);
        d2sh = wave_max63(d2sh);
      }
      if (lane == 63) {
        s_red[0][wave] = d2max;
        s_red[1][wave] = d2sh;
      }
      __syncthreads();
      if (tid == 0) {
        float m0 = 0.0f, m1 = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          m0 = fmaxf(m0, s_red[0][w]);
          m1 = fmaxf(m1, s_red[1][w]);
        }
        s_build = decide_build(S, lim, flags, nl, pl, shell_chk, m0, m1);
        if (s_build == BUILD_NL || s_build == BUILD_NL_ONLY) atomicOr(p.nlbuild, 1);
      }
      __syncthreads();
      build = s_build;
      if (build == BUILD_DIRECT) {  // the shell rows about to be built belong to these coordinates
#pragma unroll
        for (int u = 0; u < SB; ++u)
          if (u * SORT_THREADS < n) p.pos_shell[bo + min(tid + u * SORT_THREADS, n - 1)] = xs[u];
      }
    } else {
      build = S.build;
    }
    if ((PH & PH_GRID) == 0 || build == BUILD_NONE || build == BUILD_SHELL) {
      __syncthreads();  // the decision has been read before the next system's
      continue;
    }
    // ---- cell grid and counting sort
    const int cb = S.cell_base;
    if (!loaded || build != BUILD_DIRECT) {
      const float4 *src = build == BUILD_DIRECT ? x : p.pos_ref;
#pragma unroll
      for (int u = 0; u < SB; ++u) xs[u] = src[bo + min(tid + u * SORT_THREADS, n - 1)];
    }
    float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
#pragma unroll
    for (int u = 0; u < SB; ++u) {
      mn[0] = fminf(mn[0], xs[u].x); mx[0] = fmaxf(mx[0], xs[u].x);
      mn[1] = fminf(mn[1], xs[u].y); mx[1] = fmaxf(mx[1], xs[u].y);
      mn[2] = fminf(mn[2], xs[u].z); mx[2] = fmaxf(mx[2], xs[u].z);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        mn[d] = fminf(mn[d], __shfl_xor(mn[d], o));
        mx[d] = fmaxf(mx[d], __shfl_xor(mx[d], o));
      }
    }
    if (lane == 0) {
#pragma unroll
      for (int d = 0; d < 3; ++d) { s_red[d][wave] = mn[d]; s_red[3 + d][wave] = mx[d]; }
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
      for (int d = 0; d < 3; ++d)
        for (int w = 1; w < NW; ++w) {
          mn[d] = fminf(mn[d], s_red[d][w]);
          mx[d] = fmaxf(mx[d], s_red[3 + d][w]);
        }
      s_ncells = plan_grid(S, mn, mx, s_grid);
    }
    __syncthreads();
    const int nc = s_ncells;
    for (int c = tid; c < nc; c += SORT_THREADS) s_cnt[c] = 0;
    int cs[SB];
#pragma unroll
    for (int u = 0; u < SB; ++u) cs[u] = cell_index(s_grid, xs[u]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < SB; ++u) {
      const int b = tid + u * SORT_THREADS;
      if (b < n) {
        s_cell[b] = (uint16_t)cs[u];
        p.cell_of[bo + b] = cs[u];
        atomicAdd(&s_cnt[cs[u]], 1);
      }
    }
    __syncthreads();
    // exclusive scan of the counts, `per` consecutive cells per thread, with
    // the occupied cells counted in the upper half (beads <= 5120, occupied
    // cells <= beads: both fit 16 bits)
    const int per = (nc + SORT_THREADS - 1) / SORT_THREADS;
    int sum = 0;
    for (int u = 0; u < per; ++u) {
      const int c = tid * per + u;
      const int v = c < nc ? s_cnt[c] : 0;
      sum += v + (v > 0 ? 0x10000 : 0);
    }
    const int incl = wave_incl_scan(sum);
    if (lane == 63) s_wsum[wave] = incl;
    __syncthreads();
    int off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      off += w < wave ? s_wsum[w] : 0;
      tot += s_wsum[w];
    }
    if (tid == 0) {
      p.cell_start[cb + nc] = n;
      S.ncells_used = tot >> 16;
      s_item0 = build == BUILD_DIRECT ? atomicAdd(p.ncellwork, tot >> 16) : 0;
    }
    __syncthreads();
    const int item0 = s_item0;
    int run = off + incl - sum;
    for (int u = 0; u < per; ++u) {
      const int c = tid * per + u;
      if (c >= nc) break;
      const int v = s_cnt[c];
      p.cell_start[cb + c] = run & 0xFFFF;
      s_cnt[c] = run & 0xFFFF;  // cursor, ends at the cell's end offset
      if (v > 0 && build == BUILD_DIRECT) p.cellitems[item0 + (run >> 16)] = make_int2(q, c);
      run += v + (v > 0 ? 0x10000 : 0);
    }
    __syncthreads();
    for (int b = tid; b < n; b += SORT_THREADS) s_mem[atomicAdd(&s_cnt[s_cell[b]], 1)] = (uint16_t)b;
    // the loads of the output pass before its stores (a load issued after a
    // store would wait for it)
    int ns[SB], nn[SB];
#pragma unroll
    for (int u = 0; u < SB; ++u) {
      const int i = bo + min(tid + u * SORT_THREADS, n - 1);
      ns[u] = p.nat_start[i];
      nn[u] = p.nat_cnt[i];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < SB; ++u) {
      const int b = tid + u * SORT_THREADS;
      if (b < n) {
        const int c = s_cell[b];
        const int st = c > 0 ? s_cnt[c - 1] : 0, en = s_cnt[c];
        const int pos = st + count_below(s_mem, st, en, b);
        const int i = bo + b;
        p.cell_pos[i] = pos;
        p.cell_sorted[bo + pos] = i;
        p.pos_sorted[bo + pos] = xs[u];
        p.nat_sorted[bo + pos] = make_int2(ns[u], nn[u]);
      }
    }
    __syncthreads();
  }
}

// ---- systems of more than SORT_N_MAX beads (the first *nbig of the batch),
// each spread over many blocks: a 200,000-bead system's decision in one block
// took 174 us.  Grid: x blocks over a system's beads, y over the systems (64
// 8,000-bead systems one after another, each over the whole launch, took
// twice as long as side by side).

// Order-preserving unsigned image of a float, for atomic minima and maxima.
__device__ __forceinline__ uint32_t ord_u(float f) {
  const uint32_t b = __float_as_uint(f);
  return b ^ ((b >> 31) ? 0xFFFFFFFFu : 0x80000000u);
}
__device__ __forceinline__ float ord_f(uint32_t u) {
  return __uint_as_float(u ^ ((u >> 31) ? 0x80000000u : 0xFFFFFFFFu));
}

// Snapshot, displacements and bounding box of the coordinates: partial maxima
// of 2,048 beads per block into the system's accumulators (8 atomics a block).
constexpr int BIG_THREADS = 512;
__global__ __launch_bounds__(BIG_THREADS) void k_big_skin(DevPtrs p, int kstep, int flags) {
  constexpr int NW = BIG_THREADS / 64, U = 4;
  __shared__ float s_red[8][NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nbig = *p.nbig;
  for (int q = blockIdx.y; q < nbig; q += gridDim.y) {
    SysDev &S = p.sys[p.syslist[q]];
    const Due due = rebuild_due(S, kstep, flags);
    const bool nl = due.nl, pl = due.pl;
    if (!nl && !pl) continue;
    const int bo = S.bead_off, n = S.n;
    const float4 *x = buf_in(p, S.parity + kstep);
    const bool shell_chk = pl && S.sl_valid;
    float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[5] = {-INFINITY, -INFINITY, -INFINITY, 0.0f, 0.0f};
    bool any = false;
    for (int b0 = blockIdx.x * U * BIG_THREADS; b0 < n; b0 += gridDim.x * U * BIG_THREADS) {
      any = true;
      float4 xi[U], r[U], sh[U];
      int i[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        i[u] = bo + min(b0 + tid + u * BIG_THREADS, n - 1);  // past the end: the last bead again
        xi[u] = x[i[u]];
        r[u] = nl ? xi[u] : p.pos_ref[i[u]];
        sh[u] = shell_chk ? p.pos_shell[i[u]] : xi[u];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (nl) p.pos_ref[i[u]] = xi[u];
        const float dx = xi[u].x - r[u].x, dy = xi[u].y - r[u].y, dz = xi[u].z - r[u].z;
        mx[3] = fmaxf(mx[3], dx * dx + dy * dy + dz * dz);
        const float ex = xi[u].x - sh[u].x, ey = xi[u].y - sh[u].y, ez = xi[u].z - sh[u].z;
        mx[4] = fmaxf(mx[4], ex * ex + ey * ey + ez * ez);
        mn[0] = fminf(mn[0], xi[u].x); mx[0] = fmaxf(mx[0], xi[u].x);
        mn[1] = fminf(mn[1], xi[u].y); mx[1] = fmaxf(mx[1], xi[u].y);
        mn[2] = fminf(mn[2], xi[u].z); mx[2] = fmaxf(mx[2], xi[u].z);
      }
    }
    if (!any) continue;  // the same for the whole block
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
#pragma unroll
      for (int d = 0; d < 3; ++d) mn[d] = fminf(mn[d], __shfl_xor(mn[d], o));
#pragma unroll
      for (int d = 0; d < 5; ++d) mx[d] = fmaxf(mx[d], __shfl_xor(mx[d], o));
    }
    __syncthreads();  // the previous system's partials have been read
    if (lane == 0) {
#pragma unroll
      for (int d = 0; d < 3; ++d) s_red[d][wave] = mn[d];
#pragma unroll
      for (int d = 0; d < 5; ++d) s_red[3 + d][wave] = mx[d];
    }
    __syncthreads();
    if (tid < 8) {
      float v = s_red[tid][0];
      for (int w = 1; w < NW; ++w) v = tid < 3 ? fminf(v, s_red[tid][w]) : fmaxf(v, s_red[tid][w]);
      if (tid < 3) atomicMin(&S.acc[tid], ord_u(v));
      else atomicMax(&S.acc[tid], ord_u(v));
    }
  }
}

// Per big system: decision, cell grid, cleared histogram; the accumulators
// go back to their empty values for the next rebuild.
__global__ __launch_bounds__(1024) void k_big_plan(DevPtrs p, int kstep, int flags) {
  __shared__ int s_nc;
  const int tid = threadIdx.x;
  const int nbig = *p.nbig;
  for (int q = blockIdx.x; q < nbig; q += gridDim.x) {
    SysDev &S = p.sys[p.syslist[q]];
    if (tid == 0) {
      const Due due = rebuild_due(S, kstep, flags);
      const bool nl = due.nl, pl = due.pl;
      float mn[3], mx[3];
      for (int d = 0; d < 3; ++d) {
        mn[d] = ord_f(S.acc[d]);
        mx[d] = ord_f(S.acc[3 + d]);
      }
      const float d2max = nl || pl ? ord_f(S.acc[6]) : 0.0f, d2sh = nl || pl ? ord_f(S.acc[7]) : 0.0f;
      for (int d = 0; d < 8; ++d) S.acc[d] = d < 3 ? ACC_MIN : ACC_MAX;
      if (nl)  // the snapshot is these coordinates
        for (int d = 0; d < 3; ++d) {
          S.ref_box[d] = mn[d];
          S.ref_box[3 + d] = mx[d];
        }
      const BuildLimits lim{S.skin, S.shell_ok, S.nl_valid, S.nbuild[0], S.nbuild[1], S.nbuild[2]};
      const int build = decide_build(S, lim, flags, nl, pl, pl && S.sl_valid, d2max, d2sh);
      int nc = 0;
      if (build != BUILD_NONE && build != BUILD_SHELL) {
        if (build != BUILD_DIRECT)  // sorted at the snapshot
          for (int d = 0; d < 3; ++d) {
            mn[d] = S.ref_box[d];
            mx[d] = S.ref_box[3 + d];
          }
        CellGrid g;
        nc = plan_grid(S, mn, mx, g);
      }
      if (build == BUILD_NL || build == BUILD_NL_ONLY) atomicOr(p.nlbuild, 1);
      s_nc = nc;
    }
    __syncthreads();
    const int nc = s_nc, cb = S.cell_base;
    for (int c = tid; c < nc; c += blockDim.x) p.cell_cnt[cb + c] = 0;
    __syncthreads();
  }
}

// Per bead: cell id and histogram; the shell snapshot of a direct build.
__global__ __launch_bounds__(256) void k_cell_count(DevPtrs p, int kstep) {
  const int nbig = *p.nbig;
  for (int q = blockIdx.y; q < nbig; q += gridDim.y) {
    SysConst &S = sys_const(p, sload(p.syslist + q));
    if (!grid_build(S)) continue;
    const float4 *src = build_src(p, S, kstep);
    const bool direct = S.build == BUILD_DIRECT;
    const int bo = S.bead_off, n = S.n, cb = S.cell_base;
    for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < n; b += gridDim.x * blockDim.x) {
      const float4 x = src[bo + b];
      const int c = cell_index(S, x);
      p.cell_of[bo + b] = c;
      if (direct) p.pos_shell[bo + b] = x;
      atomicAdd(&p.cell_cnt[cb + c], 1);
    }
  }
}

// Per big system: exclusive scan of the histogram (DPP wave scan + wave
// totals), 4 consecutive cells per thread, and its occupied cells appended to
// the batch's home-cell list.
__global__ __launch_bounds__(1024) void k_cell_scan(DevPtrs p) {
  constexpr int NW = 16, PER = 4;
  __shared__ int wsum[NW], wused[NW], s_item0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nbig = *p.nbig;
  for (int q = blockIdx.x; q < nbig; q += gridDim.x) {
    SysDev &S = p.sys[p.syslist[q]];
    if (!grid_build(S)) continue;
    const int nc = S.ncells, cb = S.cell_base, n = S.n;
    const bool direct = S.build == BUILD_DIRECT;
    int carry = 0, used = 0;
    for (int c0 = 0; c0 < nc; c0 += 1024 * PER) {
      int v[PER], sum = 0, u = 0;
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int c = c0 + tid * PER + k;
        v[k] = c < nc ? p.cell_cnt[cb + c] : 0;
        sum += v[k];
        u += v[k] > 0;
      }
      const int incl = wave_incl_scan(sum), iused = wave_incl_scan(u);
      if (lane == 63) {
        wsum[wave] = incl;
        wused[wave] = iused;
      }
      __syncthreads();
      int off = 0, tot = 0, uoff = 0, utot = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        off += w < wave ? wsum[w] : 0;
        tot += wsum[w];
        uoff += w < wave ? wused[w] : 0;
        utot += wused[w];
      }
      if (tid == 0) s_item0 = direct ? atomicAdd(p.ncellwork, utot) : 0;
      __syncthreads();
      int run = carry + off + incl - sum, it = s_item0 + uoff + iused - u;
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int c = c0 + tid * PER + k;
        if (c < nc) {
          p.cell_start[cb + c] = run;
          p.cell_cursor[cb + c] = 0;
          if (direct && v[k] > 0) p.cellitems[it++] = make_int2(q, c);
        }
        run += v[k];
      }
      carry += tot;
      used += utot;
      __syncthreads();
    }
    if (tid == 0) {
      S.ncells_used = used;
      p.cell_start[cb + nc] = carry;
      if (carry != n) atomicOr(&S.err, ERR_INTERNAL);
    }
  }
}

// Per bead: scatter into its cell's segment (arbitrary in-cell order).
__global__ __launch_bounds__(256) void k_cell_scatter(DevPtrs p) {
  const int nbig = *p.nbig;
  for (int q = blockIdx.y; q < nbig; q += gridDim.y) {
    SysConst &S = sys_const(p, sload(p.syslist + q));
    if (!grid_build(S)) continue;
    const int bo = S.bead_off, n = S.n, cb = S.cell_base;
    for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < n; b += gridDim.x * blockDim.x) {
      const int c = p.cell_of[bo + b];
      const int slot = atomicAdd(&p.cell_cursor[cb + c], 1);
      const int pos = p.cell_start[cb + c] + slot;
      if (pos >= 0 && pos < n) p.cell_tmp[bo + pos] = bo + b;
    }
  }
}

// Per bead: rank among the beads of its cell by index -> sorted segment, with
// a cell-ordered copy of the coordinates.  The in-cell order, and with it every
// list, is independent of the order of the atomics above.
__global__ __launch_bounds__(256) void k_cell_rank(DevPtrs p, int kstep) {
  const int nbig = *p.nbig;
  for (int q = blockIdx.y; q < nbig; q += gridDim.y) {
    SysConst &S = sys_const(p, sload(p.syslist + q));
    if (!grid_build(S)) continue;
    const float4 *src = build_src(p, S, kstep);
    const int bo = S.bead_off, n = S.n, cb = S.cell_base;
    for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < n; b += gridDim.x * blockDim.x) {
      const int i = bo + b;
      const int c = p.cell_of[i];
      const int st = p.cell_start[cb + c], en = p.cell_start[cb + c + 1];
      int rank = 0;
      if (st >= 0 && en <= n) {
        for (int m = st; m < en; ++m) rank += p.cell_tmp[bo + m] < i;
        const int pos = st + rank;
        if (pos < n) {
          p.cell_pos[i] = pos;
          p.nat_sorted[bo + pos] = make_int2(p.nat_start[i], p.nat_cnt[i]);
          p.cell_sorted[bo + pos] = i;
          p.pos_sorted[bo + pos] = src[i];
        }
      }
    }
  }
}

__device__ __forceinline__ bool native_pair(const int32_t *nj, int nn, int j) {
  int lo = 0, hi = nn;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (nj[mid] < j) lo = mid + 1;
    else hi = mid;
  }
  return lo < nn && nj[lo] == j;
}

// Native partners of the current bead, as a wave-private LDS bitmap keyed by
// (local index mod 65536); a set bit is confirmed by the exact search unless
// the system is small enough for the key to be the index itself.
constexpr int NATBITS_WORDS = 2048;

__device__ __forceinline__ void natbits_mark(uint32_t *bits, const int32_t *natj, int nn, int bead_off, bool set) {
  const int lane = threadIdx.x & 63;
  for (int k = lane; k < nn; k += 64) {
    const int jl = (natj[k] - bead_off) & 0xFFFF;
    if (set) atomicOr(&bits[jl >> 5], 1u << (jl & 31));
    else bits[jl >> 5] = 0u;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Candidate scan of the 27 cells around xi as 9 rows of 3 contiguous cells,
// reading the cell-ordered copy of the coordinates.  Non-native master pairs
// with d2 below the cutoff of their type pair (rcA: tj = 1, rcB: tj = 2) are
// appended to out[0..cap) with ballot/mbcnt
// compaction; returns the count (which may exceed cap).
template <typename Extra, typename Emit>
__device__ __forceinline__ int scan_cells(const DevPtrs &p, SysConst &S, int i, float4 xi,
                                          float rcA, float rcB, int ns, int nn, uint32_t *bits, Extra extra,
                                          Emit emit) {
  const int lane = threadIdx.x & 63;
  const int wi = __float_as_int(xi.w), ci = wi >> 2;
  // (in registers: the emitted entries may alias S)
  const float boxl = S.boxl;
  const int bo = S.bead_off, n = S.n;
  const int cx = min(max((int)floorf((xi.x - S.org[0]) * S.inv_edge[0]), 0), S.dims[0] - 1);
  const int cy = min(max((int)floorf((xi.y - S.org[1]) * S.inv_edge[1]), 0), S.dims[1] - 1);
  const int cz = min(max((int)floorf((xi.z - S.org[2]) * S.inv_edge[2]), 0), S.dims[2] - 1);
  const int x0 = max(cx - 1, 0), x1 = min(cx + 1, S.dims[0] - 1);
  const int32_t *natj = p.nat_j + ns;
  const bool exact_key = S.n <= 65536;
  natbits_mark(bits, natj, nn, S.bead_off, true);
  int cnt = 0;
  for (int zz = max(cz - 1, 0); zz <= min(cz + 1, S.dims[2] - 1); ++zz)
    for (int yy = max(cy - 1, 0); yy <= min(cy + 1, S.dims[1] - 1); ++yy) {
      const int row = (zz * S.dims[1] + yy) * S.dims[0];
      const int st = max(p.cell_start[S.cell_base + row + x0], 0);
      const int en = min(p.cell_start[S.cell_base + row + x1 + 1], S.n);
      // U x 64 candidates' loads in flight together
      constexpr int U = 4;
      for (int m0 = st; m0 < en; m0 += 64 * U) {
        int jj[U];
        float4 xx[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int m = min(m0 + 64 * u + lane, en - 1);
          jj[u] = p.cell_sorted[bo + m];
          xx[u] = p.pos_sorted[bo + m];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (m0 + 64 * u >= en) break;
          const int j = jj[u];
          const float4 xj = xx[u];
          const int wj = __float_as_int(xj.w);
          const int dj = j - i;
          const bool excl = m0 + 64 * u + lane >= en || (j == i) || (((wj >> 2) == ci) && dj >= -2 && dj <= 2) ||
                            j < bo || j >= bo + n;
          bool pred = false;
          if (!excl && dist2_exact(xi, xj, boxl) < ((wj & 3) == 2 ? rcB : rcA)) {
            const int jl = (j - bo) & 0xFFFF;
            bool nat = (bits[jl >> 5] >> (jl & 31)) & 1u;
            if (nat && !exact_key) nat = native_pair(natj, nn, j);
            pred = !nat && extra(j, wj);
          }
          const uint64_t mk = __ballot(pred);
          if (pred) emit(cnt + lanes_below(mk), j);
          cnt += __popcll(mk);
        }
      }
    }
  natbits_mark(bits, natj, nn, S.bead_off, false);
  return cnt;
}

// Block per home cell: the shell rows of the cell's beads straight from the
// shell-cutoff grid.  The bounds of the 9 neighbor rows and all their
// candidates are staged in LDS together (CAND_MAX at a time); every home bead
// of the cell tests them.  Each bead's list comes out in row order, then
// cell-sorted order: the order of a per-bead scan of the same cells.
constexpr int HOME_MAX = 64;   // home beads per pass
constexpr int CAND_MAX = 1024; // candidates staged per pass (and bits of the exclusion bitmaps)
constexpr int EXCL_WORDS = CAND_MAX / 32;

// Pair-list rows are padded with the bead's own index up to a multiple of
// ROW_PAD entries, so the step kernel reads whole chunks without a count
// test: a self entry has d2 = 0, which the repulsion guard turns into zero
// force.  pl_cap is a multiple of 16, so a padded row fits its capacity.
constexpr int ROW_PAD = 4;
// 16-bit pair-list entries per step-kernel chunk load (4: 8 bytes; 8: 16
// bytes, which needs ROW_PAD 8): four entries per lane and load leave fewer
// lanes idle at the end of a row than eight
#ifndef STEP_CHUNK16
#define STEP_CHUNK16 4
#endif
static_assert(ROW_PAD % STEP_CHUNK16 == 0 && ROW_PAD % 4 == 0, "rows must hold whole chunks");
// LDS of one workgroup on gfx950, and the shell filter's row staging: per
// wave, 16 beads of a round x FILTER_SROW 16-bit entries (32-bit entries take
// twice the bytes; longer rows are completed by a second pass)
constexpr int LDS_BYTES_MAX = 160 * 1024;
constexpr int FILTER_SROW = 144;
constexpr int FILTER_STAGE_BYTES = STEP_WAVES * 16 * FILTER_SROW * 2;
// Buffer resource of `bytes` bytes at `base` (wave-uniform): loads through
// it take a 32-bit offset, and a load past the end returns zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *base, uint32_t bytes) {
  const uint64_t a = (uint64_t)base;
  const uint64_t u = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32) |
                     (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  return __builtin_amdgcn_make_buffer_rsrc((void *)u, (short)0, (int)__builtin_amdgcn_readfirstlane((int)bytes),
                                           0x00020000);
}

__device__ __forceinline__ uint4 load_b128(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}

__device__ __forceinline__ int2 load_i2(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0);
  return make_int2((int)v[0], (int)v[1]);
}

// Output row of one bead as a raw buffer of pl_cap entries: stores past the
// row's end are dropped by the buffer bounds check (the count still grows,
// which the caller reports as an overflow).  The caller's row address and
// size are wave-uniform; readfirstlane puts the descriptor in scalar registers.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(void *row, int bytes) {
  const uint64_t a = (uint64_t)row;
  const uint64_t u = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32) |
                     (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a);
  return __builtin_amdgcn_make_buffer_rsrc((void *)u, (short)0, __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

// The fast form of the home-bead scan: the staged candidates are padded to a
// multiple of 128 with coordinates no pair can reach, and the home bead's
// bitmap over candidate slots already excludes itself, its chain neighbours
// i +- 1, 2 and its native partners, so a candidate costs its loads, the
// distance, one bit test and, when kept, one buffer store.  No minimum image:
// a rebuild whose extent reaches boxl/2 - margin raises ERR_PBC, so every
// separation here is below boxl/2, where the minimum image is the identity.
// ONE: every bead has the home bead's type (one cutoff rcA).
template <bool ONE, bool IDX16>
__device__ __forceinline__ int pl_scan_fast(const float4 *s_cand, const int *s_cj, int ncp, float4 xi, float rcA,
                                            float rcB, const uint32_t *excl, __amdgpu_buffer_rsrc_t row, int bo,
                                            int lane, int cnt) {
  const uint32_t lbit = 1u << (lane & 31);
  for (int k0 = 0; k0 < ncp; k0 += 128) {
    int jj[2];
    float4 xj[2];
    uint32_t ew[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int ci = k0 + u * 64 + lane;
      jj[u] = s_cj[ci];
      xj[u] = s_cand[ci];
      ew[u] = excl[ci >> 5];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const float dx = xj[u].x - xi.x, dy = xj[u].y - xi.y, dz = xj[u].z - xi.z;
      const float d2 = (dx * dx + dy * dy) + dz * dz;
      const float rc = ONE ? rcA : ((__float_as_int(xj[u].w) & 3) == 2 ? rcB : rcA);
      const bool keep = (d2 < rc) & ((ew[u] & lbit) == 0u);
      const uint64_t mk = __ballot(keep);
      if (keep) {
        const int o = cnt + lanes_below(mk);
        if (IDX16) __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(jj[u] - bo), row, o * 2, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b32((unsigned int)jj[u], row, o * 4, 0, 0);
      }
      cnt += __popcll(mk);
    }
  }
  return cnt;
}

constexpr int PLC_BYTES = 16 * (CAND_MAX + HOME_MAX) + 4 * (CAND_MAX + HOME_MAX * (4 + EXCL_WORDS)) + 96;
__device__ __forceinline__ void pl_cells(const DevPtrs &p, int kstep, char *s_raw) {
  float4 *s_cand = reinterpret_cast<float4 *>(s_raw), *s_home = s_cand + CAND_MAX;
  int *s_cj = reinterpret_cast<int *>(s_home + HOME_MAX);
  int *s_hj = s_cj + CAND_MAX, *s_hcnt = s_hj + HOME_MAX, *s_hnn = s_hcnt + HOME_MAX, *s_hns = s_hnn + HOME_MAX;
  uint32_t(*s_excl)[EXCL_WORDS] = reinterpret_cast<uint32_t(*)[EXCL_WORDS]>(s_hns + HOME_MAX);  // per home bead:
                                                                                     // slots it must skip
  int *s_rst = reinterpret_cast<int *>(s_excl + HOME_MAX), *s_roff = s_rst + 9, *s_hrange = s_roff + 10;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int total = *p.ncellwork;
  for (int g = blockIdx.x; g < total; g += gridDim.x) {
    const int2 item = p.cellitems[g];
    const int s = sload(p.syslist + item.x);
    const int c = item.y;
    SysConst &S = sys_const(p, s);
    const int bo = S.bead_off, cb = S.cell_base, n = S.n;
    const int pl_cap = S.pl_cap;
    const int64_t pl_base = S.pl_base;
    const float rc2_11 = S.rc2_sl_rep[0], rc2_12 = S.rc2_sl_rep[1], rc2_21 = S.rc2_sl_rep[2],
                rc2_22 = S.rc2_sl_rep[3];
    const int d0 = S.dims[0], d1 = S.dims[1], d2 = S.dims[2];
    const int cx = c % d0, cy = (c / d0) % d1, cz = c / (d0 * d1);
    // bounds of the home cell and of the 3x3 neighbor rows (x-range cx-1..cx+1)
    if (tid < 9) {
      const int zz = cz + tid / 3 - 1, yy = cy + tid % 3 - 1;
      int st = 0, len = 0;
      if (zz >= 0 && zz < d2 && yy >= 0 && yy < d1) {
        const int row = (zz * d1 + yy) * d0;
        st = max(p.cell_start[cb + row + max(cx - 1, 0)], 0);
        len = max(min(p.cell_start[cb + row + min(cx + 1, d0 - 1) + 1], n) - st, 0);
      }
      s_rst[tid] = st;
      s_roff[tid + 1] = len;
    } else if (tid < 11) {
      s_hrange[tid - 9] = min(max(p.cell_start[cb + c + (tid - 9)], 0), n);
    }
    __syncthreads();
    if (tid == 0) {
      s_roff[0] = 0;
      for (int r = 1; r <= 9; ++r) s_roff[r] += s_roff[r - 1];
    }
    __syncthreads();
    const int hs = s_hrange[0], he = s_hrange[1];
    const int T = s_roff[9];
    if (hs >= he) {
      __syncthreads();  // everyone has read the bounds before the next cell rewrites them
      continue;
    }
    const bool exact = T > CAND_MAX;  // candidates staged in passes of CAND_MAX
    // stage the candidates [b0, b0 + nc), padded to a multiple of 128 with
    // coordinates no pair can reach
    auto stage = [&](int b0, int nc) {
      // CAND_MAX / 256 slots per thread, all loads before the LDS writes
      // (slots past nc load the last candidate and store the padding)
      constexpr int CS = CAND_MAX / 256;
      float4 xc[CS];
      int jc[CS];
#pragma unroll
      for (int u = 0; u < CS; ++u) {
        const int idx = b0 + min(tid + 256 * u, nc - 1);
        int r = 0;
#pragma unroll
        for (int q = 1; q < 9; ++q) r += s_roff[q] <= idx;
        const int m = s_rst[r] + (idx - s_roff[r]);
        xc[u] = p.pos_sorted[bo + m];
        jc[u] = p.cell_sorted[bo + m];
      }
      const int ncp = (nc + 127) & ~127;
#pragma unroll
      for (int u = 0; u < CS; ++u) {
        const int ci = tid + 256 * u;
        if (ci < nc) {
          s_cand[ci] = xc[u];
          s_cj[ci] = jc[u];
        } else if (ci < ncp) {
          s_cand[ci] = make_float4(INFINITY, INFINITY, INFINITY, 0.0f);
          s_cj[ci] = -1;
        }
      }
    };
    // the first home pass's beads load beside the candidate staging
    int2 ni0 = make_int2(0, 0);
    float4 xh0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    int jh0 = 0;
    if (tid < min(HOME_MAX, he - hs)) {
      ni0 = p.nat_sorted[bo + hs + tid];
      xh0 = p.pos_sorted[bo + hs + tid];
      jh0 = p.cell_sorted[bo + hs + tid];
    }
    if (!exact) stage(0, T);
    for (int h0 = hs; h0 < he; h0 += HOME_MAX) {
      const int nh = min(HOME_MAX, he - h0);
      if (tid < nh) {
        if (h0 != hs) {
          ni0 = p.nat_sorted[bo + h0 + tid];
          xh0 = p.pos_sorted[bo + h0 + tid];
          jh0 = p.cell_sorted[bo + h0 + tid];
        }
        s_home[tid] = xh0;
        s_hj[tid] = jh0;
        s_hcnt[tid] = 0;
        s_hns[tid] = ni0.x;
        s_hnn[tid] = ni0.y;
      }
      // candidate passes of CAND_MAX staged slots (one pass when they all fit,
      // staged above for every home pass)
      for (int b0 = 0; b0 < T; b0 += CAND_MAX) {
        const int nc = min(CAND_MAX, T - b0);
        if (exact) stage(b0, nc);
        if (tid < nh) {
#pragma unroll
          for (int w = 0; w < EXCL_WORDS; ++w) s_excl[tid][w] = 0u;
        }
        __syncthreads();
        // exclusion bitmaps over this pass's slots: the slot of each native
        // partner and of the bead itself and its chain neighbours i +- 1, 2,
        // from their cells in this rebuild's grid (the row) and sorted
        // positions (the offset)
        // four home beads per pass of a wave, 16 lanes each, so the dependent
        // loads of several beads are in flight together
        for (int t0 = 0; wave + 4 * t0 < nh; t0 += 4) {
          const int h = wave + 4 * (t0 + (lane >> 4));
          if (h >= nh) continue;
          const int ji = s_hj[h], ns = s_hns[h], nn = s_hnn[h];
          const int chi = __float_as_int(s_home[h].w) >> 2;
          for (int k = lane & 15; k < nn + 5; k += 16) {
            int cn, pos, jn;
            if (k < nn) {
              const int jp = p.nat_j[ns + k];  // native partner: its cell and place in the cell order
              cn = p.cell_of[jp];
              pos = p.cell_pos[jp];
              jn = -1;
            } else {
              jn = ji + (k - nn - 2);
              if (jn < bo || jn >= bo + n) continue;
              cn = p.cell_of[jn];
              pos = p.cell_pos[jn];
            }
            const int nx = cn % d0, ny = (cn / d0) % d1, nz = cn / (d0 * d1);
            if (abs(nx - cx) > 1 || abs(ny - cy) > 1 || abs(nz - cz) > 1) continue;
            const int r = (nz - cz + 1) * 3 + (ny - cy + 1);
            const int slot = s_roff[r] + (pos - s_rst[r]);
            if (slot < s_roff[r] || slot >= s_roff[r + 1]) continue;
            const int ls = slot - b0;  // staged position in this pass
            if (ls < 0 || ls >= nc) continue;
            if (jn >= 0 && (s_cj[ls] != jn || (__float_as_int(s_cand[ls].w) >> 2) != chi)) continue;
            atomicOr(&s_excl[h][ls >> 5], 1u << (ls & 31));
          }
        }
        __syncthreads();
        for (int h = wave; h < nh; h += 4) {
          const float4 xi = s_home[h];
          const int ji = s_hj[h];
          const int wi = __float_as_int(xi.w);
          const float rcA = (wi & 3) == 2 ? rc2_21 : rc2_11, rcB = (wi & 3) == 2 ? rc2_22 : rc2_12;
          int32_t *out = p.slrep_j + pl_base + (int64_t)(ji - bo) * pl_cap;
          uint16_t *out16 = S.idx16 ? (uint16_t *)(p.slrep_j + pl_base) + (int64_t)(ji - bo) * pl_cap : nullptr;
          const int ncp = (nc + 127) & ~127;
          const bool one = S.type_mask != 3;
          const float rc1 = S.type_mask == 2 ? rcB : rcA;
          void *row = S.idx16 ? (void *)out16 : (void *)out;
          const __amdgpu_buffer_rsrc_t rr = row_rsrc(row, pl_cap * (S.idx16 ? 2 : 4));
          const int c0 = s_hcnt[h];
          int cnt;
          if (one) cnt = S.idx16 ? pl_scan_fast<true, true>(s_cand, s_cj, ncp, xi, rc1, rc1, s_excl[h], rr, bo, lane, c0)
                                 : pl_scan_fast<true, false>(s_cand, s_cj, ncp, xi, rc1, rc1, s_excl[h], rr, bo, lane, c0);
          else cnt = S.idx16 ? pl_scan_fast<false, true>(s_cand, s_cj, ncp, xi, rcA, rcB, s_excl[h], rr, bo, lane, c0)
                             : pl_scan_fast<false, false>(s_cand, s_cj, ncp, xi, rcA, rcB, s_excl[h], rr, bo, lane, c0);
          if (lane == 0) s_hcnt[h] = cnt;
        }
        __syncthreads();  // the next pass restages and clears the bitmaps
      }
      __syncthreads();
      if (tid < nh) {
        const int j = s_hj[tid], cr = s_hcnt[tid];
        p.slrep_cnt[j] = min(cr, pl_cap);
        if (cr > pl_cap) {
          atomicOr(&p.sys[s].err, ERR_PL_OVF);
          p.sys[s].sl_valid = 0;  // truncated rows must not be filtered again
        }
      }
      if (wave == 0) {  // the longest row of this pass, for the host's capacity check
        const int cr = lane < nh ? s_hcnt[lane] : 0;
        const int mx = wave_max(cr);
        if (lane == 0) atomicMax(&p.sys[s].row_max, mx);
      }
      __syncthreads();
    }
  }
}

// Wave per bead, from the cell grid of the neighbor-list snapshot pos_ref.
// BUILD_NL_ONLY: materialize the neighbor list (pairs within rc_nl at
// pos_ref) into the neighbor-list scratch.  BUILD_NL: the pair list of the
// reference's two-level scheme, neighbor-list pairs within rc_pl at x, in one
// pass without materializing the neighbor list: the native pair list in each
// bead's native slots, the non-native rows in the shell-row slots (the shell
// filter packs them into the pair list), which therefore stop holding shell
// rows (decide_build clears sl_valid).
__device__ __forceinline__ void nl_build(const DevPtrs &p, int kstep, char *s_raw) {
  uint32_t(*s_bits)[NATBITS_WORDS] = reinterpret_cast<uint32_t(*)[NATBITS_WORDS]>(s_raw);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int k = lane; k < NATBITS_WORDS; k += 64) s_bits[wave][k] = 0u;
  __builtin_amdgcn_wave_barrier();
  // a wave scans a bead's 27 cells one load batch after another, so the beads
  // go out over as many waves as the launch has (a wave took sixteen: 860 us for
  // the neighbor list of 5,000 beads)
  const int nbead = *p.nwork * TILE;
  for (int w = blockIdx.x * 4 + wave; w < nbead; w += gridDim.x * 4) {
    const int t = sload(p.work + w / TILE);
    if (t < 0) continue;
    const int s = sload(p.tile_sys + t);
    SysConst &S = sys_const(p, s);
    if (S.build != BUILD_NL && S.build != BUILD_NL_ONLY) continue;
    const bool plb = S.build == BUILD_NL;
    const float4 *ref = p.pos_ref;
    const float4 *pin = buf_in(p, S.parity + kstep);
    const float boxl = S.boxl;
    const int bend = min(t * TILE + TILE, S.bead_off + S.n);
    const int i = t * TILE + w % TILE;
    if (i >= bend) continue;
    const float4 xi = ref[i];
    const float4 xn = pin[i];
    const int ti = __float_as_int(xi.w) & 3;
    const int ns = p.nat_start[i], nn = p.nat_cnt[i];
    int cnt = 0;
    for (int k0 = 0; k0 < nn; k0 += 64) {
      const int k = k0 + lane;
      bool pred = false;
      int j = 0;
      float r0 = 0.0f;
      if (k < nn) {
        j = p.nat_j[ns + k];
        r0 = p.nat_r0[ns + k];
        const float rc = cutoff_of(S.nl_factor, S.nl_abs, r0);
        pred = dist2_exact(xi, ref[j], boxl) < rc * rc;
        if (plb && pred) {
          const float rp = cutoff_of(S.pl_factor, S.pl_abs, r0);
          pred = dist2_exact(xn, pin[j], boxl) < rp * rp;
        }
      }
      const uint64_t m = __ballot(pred);
      if (pred) {
        const int o = ns + cnt + lanes_below(m);
        if (plb) {
          p.platt[o] = make_int2(j, __float_as_int(r0));
        } else {
          p.nlatt_j[o] = j;
          p.nlatt_r0[o] = r0;
        }
      }
      cnt += __popcll(m);
    }
    const float rcA = S.rc2_nl_rep[(ti - 1) * 2], rcB = S.rc2_nl_rep[(ti - 1) * 2 + 1];
    if (plb) {
      if (lane == 0) {
        p.platt_cnt[i] = cnt;
        p.platt_off[i] = ns;  // in the bead's own native slots
      }
      const float pA = S.rc2_pl_rep[(ti - 1) * 2], pB = S.rc2_pl_rep[(ti - 1) * 2 + 1];
      const int64_t row = (int64_t)(i - S.bead_off) * S.pl_cap;  // the bead's shell-row slot
      uint16_t *r16 = (uint16_t *)(p.slrep_j + S.pl_base) + row;
      int32_t *r32 = p.slrep_j + S.pl_base + row;
      const int cap = S.pl_cap, bo = S.bead_off;
      const bool i16 = S.idx16 != 0;
      const int cr = scan_cells(
          p, S, i, xi, rcA, rcB, ns, nn, s_bits[wave],
          [&](int j, int wj) { return dist2_exact(xn, pin[j], boxl) < ((wj & 3) == 2 ? pB : pA); },
          [&](int o, int j) {
            if (o < cap) {
              if (i16) r16[o] = (uint16_t)(j - bo);
              else r32[o] = j;
            }
          });
      if (lane == 0) {
        p.slrep_cnt[i] = min(cr, cap);
        if (cr > cap) atomicOr(&p.sys[s].err, ERR_PL_OVF);
        atomicMax(&p.sys[s].row_max, cr);
      }
    } else {
      if (lane == 0) p.nlatt_cnt[i] = cnt;
      int32_t *out = p.nlrep_j + S.nl_base + (int64_t)(i - S.bead_off) * S.nl_cap;
      const int cap = S.nl_cap;
      const int cr = scan_cells(p, S, i, xi, rcA, rcB, ns, nn, s_bits[wave], [](int, int) { return true; },
                                [&](int o, int j) {
                                  if (o < cap) out[o] = j;
                                });
      if (lane == 0) {
        p.nlrep_cnt[i] = min(cr, cap);
        if (cr > cap) atomicOr(&p.sys[s].err, ERR_NL_OVF);
        p.sys[s].nl_valid = 1;
      }
    }
  }
}

// Rows of one rebuild: the home cells of the batch's grid builds, then the
// neighbor-list builds, which are rare (one launch: a kernel of their own cost
// 5 us a rebuild with nothing to do).
__global__ __launch_bounds__(256) void k_rows(DevPtrs p, int kstep) {
  constexpr int NLB_BYTES = 4 * 4 * NATBITS_WORDS;
  __shared__ __align__(16) char s_raw[PLC_BYTES > NLB_BYTES ? PLC_BYTES : NLB_BYTES];
  pl_cells(p, kstep, s_raw);
  if (*p.nlbuild != 0) {
    __syncthreads();
    nl_build(p, kstep, s_raw);
  }
}

// ----------------------------------------------- fused force + integrate

// Partner coordinates come from the LDS copy of the item's arena range
// (LDS = true, base = first staged bead) or from global memory.
template <bool LDS>
__device__ __forceinline__ float4 partner(const float4 *__restrict__ pin, const float4 *s_pos, int base, int j) {
  return LDS ? s_pos[j - base] : pin[j];
}

// The same by 32-bit byte offsets, for the pair loops: one instruction per
// partner for its address.  at0 is arena bead 0's, modulo 2^32.  In LDS the
// offset is the LDS address itself; global coordinates go through a buffer
// resource at the system's first bead (a system's rows are below 4 GiB, so its
// coordinates are too, whatever the arena holds).
typedef float vf4 __attribute__((ext_vector_type(4)));
typedef float vf3 __attribute__((ext_vector_type(3)));
template <bool LDS>
struct PosAt {
  uint32_t at0;
  __amdgpu_buffer_rsrc_t r;
  // first: the first staged bead (LDS), or the system's
  __device__ __forceinline__ PosAt(const float4 *__restrict__ pin, const float4 *s_pos, int first) {
    at0 = 0u - 16u * (uint32_t)first;
    if constexpr (LDS) at0 += (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) float4 *)s_pos;
    else r = buf_rsrc(pin + first, 0xFFFFFFFFu);
  }
  template <bool XYZ>
  __device__ __forceinline__ float4 get(uint32_t off) const {
    if constexpr (LDS && XYZ) {
      const vf3 v = *(const __attribute__((address_space(3))) vf3 *)off;
      return make_float4(v.x, v.y, v.z, 0.0f);
    } else if constexpr (LDS) {
      const vf4 v = *(const __attribute__((address_space(3))) vf4 *)off;
      return make_float4(v.x, v.y, v.z, v.w);
    } else if constexpr (XYZ) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b96(r, (int)off, 0, 0);
      return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), 0.0f);
    } else {
      const uint4 v = load_b128(r, off);
      return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
    }
  }
};

// base + 16 * the low or high half of w
template <bool HI>
__device__ __forceinline__ uint32_t mad16(uint32_t w, uint32_t base) {
  uint32_t o;
  if constexpr (HI) asm("v_mad_u32_u16 %0, %1, 16, %2 op_sel:[1,0,0,0]" : "=v"(o) : "v"(w), "v"(base));
  else asm("v_mad_u32_u16 %0, %1, 16, %2" : "=v"(o) : "v"(w), "v"(base));
  return o;
}

// Force of the chain terms on bead b0 + lane of a tile, one bead per lane.
template <bool LDS>
__device__ __forceinline__ float3 chain_force(const DevPtrs &p, SysConst &S, int s, int b0,
                                              const float4 *__restrict__ pin, const float4 *s_pos, int lds0, float t_br,
                                              float br_before) {
  const int lane = threadIdx.x & 63;
  const int bead_off = S.bead_off, n = S.n;
  const int bend = min(b0 + TILE, bead_off + n);
  // Chain terms, each pair once, over the tile's lanes: lane m computes the
  // FENE bond (i, i+1) and the i,i+2 soft sphere of its bead i = b0 + m (the
  // force on i; the partner takes the opposite), and takes the partner halves
  // of the bond (i-1, i) and the pair (i-2, i) from lanes m-1 and m-2.  The
  // pairs that start before the tile come from lanes 0 and 1 themselves.
  const int i = b0 + lane;
  const int send = bead_off + n;
  float4 xc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (i < bend) xc = partner<LDS>(pin, s_pos, lds0, i);
  // force on a from the pair (a, b) of chain offset off (1: FENE bond of
  // length r0, 2: soft sphere); zero across chains
  auto chain_pair = [&](float4 xa, int ja, int off, float r0, float &ox, float &oy, float &oz) {
    ox = oy = oz = 0.0f;
    const int jb = ja + off;
    if (ja < bead_off || jb >= send) return;
    const float4 xb = partner<LDS>(pin, s_pos, lds0, jb);
    if ((__float_as_int(xb.w) >> 2) != (__float_as_int(xa.w) >> 2)) return;
    const float dx = xb.x - xa.x, dy = xb.y - xa.y, dz = xb.z - xa.z;
    const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
    float c;
    if (off == 1) {
      const float d = sqrtf(d2);
      const float dev = d - r0;
      const float gg = 1.0f - dev * dev * S.inv_R0sq;
      c = S.k_bnd * dev * rcpf(d * gg);
      if (gg <= 0.0f) atomicOr(&p.sys[s].err, ERR_BOND);
    } else {
      const float ir2 = rcpf(d2);
      const float ir4 = ir2 * ir2;
      c = -S.ss_f6 * (ir4 * ir4);
    }
    ox = c * dx;
    oy = c * dy;
    oz = c * dz;
  };
  float bx, by, bz, sx, sy, sz;
  chain_pair(xc, i < bend ? i : send, 1, t_br, bx, by, bz);
  chain_pair(xc, i < bend ? i : send, 2, 0.0f, sx, sy, sz);
  // the partner halves from lanes m-1 (bond) and m-2 (soft sphere)
  const int m1 = lane >= 1 ? lane - 1 : 0, m2 = lane >= 2 ? lane - 2 : 0;
  float pbx = __shfl(bx, m1), pby = __shfl(by, m1), pbz = __shfl(bz, m1);
  float psx = __shfl(sx, m2), psy = __shfl(sy, m2), psz = __shfl(sz, m2);
  if (lane < 2 && i < bend) {  // pairs that start before the tile
    float ex, ey, ez;
    const float4 xp2 = i - 2 >= bead_off ? partner<LDS>(pin, s_pos, lds0, i - 2) : xc;
    chain_pair(xp2, i - 2 >= bead_off ? i - 2 : send, 2, 0.0f, ex, ey, ez);
    psx = ex; psy = ey; psz = ez;
    if (lane == 0) {
      const float4 xp1 = i - 1 >= bead_off ? partner<LDS>(pin, s_pos, lds0, i - 1) : xc;
      chain_pair(xp1, i - 1 >= bead_off ? i - 1 : send, 1, br_before, ex, ey, ez);
      pbx = ex; pby = ey; pbz = ez;
    }
  }
  return make_float3((bx + sx) - (pbx + psx), (by + sy) - (pby + psy), (bz + sz) - (pbz + psz));
}

// The move of bead b0 + lane (or the force output) from its force mf without
// noise and its three normals n0, n1, n2 of this step.
template <bool LDS>
__device__ __forceinline__ void integrate(const DevPtrs &p, SysConst &S, int s, int i, int mode,
                                          const float4 *__restrict__ pin, float4 *__restrict__ pout,
                                          const float4 *s_pos, int lds0, float mfx, float mfy, float mfz, float n0,
                                          float n1, float n2) {
  if (mode == MODE_FORCE) {
    p.fout[i] = make_float4(mfx, mfy, mfz, 0.0f);
    return;
  }
  const float var = S.var;
  const float ftx = mfx + n0 * var, fty = mfy + n1 * var, ftz = mfz + n2 * var;
  if (mode == MODE_FORCE_NOISE) {
    p.fout[i] = make_float4(ftx, fty, ftz, 0.0f);
    return;
  }
  float4 x = partner<LDS>(pin, s_pos, lds0, i);
  if (S.dyn == 0) {
    // overdamped (sop.cu:487-520): x += (h/zeta) F
    const float a5 = S.a5;
    x.x = x.x + a5 * ftx;
    x.y = x.y + a5 * fty;
    x.z = x.z + a5 * ftz;
  } else {
    // underdamped (sop.cu:421-484): the reference's velocity update after its
    // force evaluation, v = a3 incr + a4 F, happens here at the start of the
    // next step, then incr = a1 v + a2 F, x += incr
    const float4 st = p.vel[i];
    float vx2 = st.x, vy2 = st.y, vz2 = st.z;
    if (__float_as_int(st.w) == 1) {
      vx2 = S.a3 * st.x + S.a4 * ftx;
      vy2 = S.a3 * st.y + S.a4 * fty;
      vz2 = S.a3 * st.z + S.a4 * ftz;
    }
    const float ix = S.a1 * vx2 + S.a2 * ftx, iy = S.a1 * vy2 + S.a2 * fty, iz = S.a1 * vz2 + S.a2 * ftz;
    x.x = x.x + ix;
    x.y = x.y + iy;
    x.z = x.z + iz;
    p.vel[i] = S.vupd ? make_float4(ix, iy, iz, __int_as_float(1)) : make_float4(vx2, vy2, vz2, 0.0f);
  }
  pout[i] = x;
  if (!(isfinite(x.x) && isfinite(x.y) && isfinite(x.z))) atomicOr(&p.sys[s].err, ERR_NAN);
}

// One wave, one tile of 64 beads.  LPB lanes per bead gather its partners and
// reduce with DPP; GPW = 64 / LPB beads per round, LPB rounds.  After each
// round, lane m picks up the force of bead m of the tile from the group that
// computed it, so the random force and the move run on all 64 lanes, one bead
// per lane, with no block barrier.  ONE: every bead of the system has the
// same type, so the force-field constants are wave-uniform (scalar registers).
// GB partners are asked for together.
template <int LPB, int MODE, bool LDS, bool IDX16, bool ONE, int GB>
__device__ __forceinline__ void wave_tile(const DevPtrs &p, SysConst &S, int s, int t, int kstep,
                                          const float4 *__restrict__ pin, float4 *__restrict__ pout,
                                          const float4 *s_pos, int lds0, int r0, int r1) {
  constexpr int GPW = 64 / LPB;
  const int lane = threadIdx.x & 63;
  const int g = lane / LPB, l = lane % LPB;
  const int bead_off = S.bead_off, n = S.n;
  const int b0 = t * TILE;
  const int bend = min(b0 + TILE, bead_off + n);
  // No minimum image: a state whose extent reaches boxl/2 - margin is refused
  // at each rebuild (ERR_PBC), so every separation here is below boxl/2.
  const int q1 = S.type_mask == 2 ? 3 : 0;  // type-pair index of a one-type system
  // slot q of the tile's order (tile_ord) is computed in round q / GPW by
  // group q % GPW; lane m's own bead b0 + m sits in slot qm
  const int ordm = p.tile_ord[b0 + lane];
  const int qm = __builtin_amdgcn_ds_permute(ordm << 2, lane);
  const int src = (qm % GPW) * LPB, rm = qm / GPW;
  // per-bead list heads of the whole tile in one coalesced load each; a
  // round picks its beads' values up by shuffles
  // (native pair-list length | pair-list length << 16: both below 2^16, which
  // the host checks)
  int t_ns = 0, t_cn = 0, t_po = 0;
  float t_br = 0.0f;  // r0 of bond (b0 + lane, b0 + lane + 1)
  // (from the bead's list head: rows from the tile's region start, native
  // lists from the native slots of the tile's first bead)
  const int nat0 = p.nat_start[b0], reg0 = (b0 - bead_off) * S.pl_cap;
  if (b0 + lane < bend) {
    const uint2 hd = p.plhead[b0 + lane];
    t_cn = (int)hd.x;
    t_po = reg0 + ROW_PAD * (int)(hd.y & 0xFFFFu);
    t_ns = nat0 + (int)(hd.y >> 16);
    t_br = p.bond_r0[b0 + lane];
  }
  const float br_before = b0 > bead_off ? p.bond_r0[b0 - 1] : 0.0f;  // bond (b0 - 1, b0)
  // the non-native rows in chunks of E entries: STEP_CHUNK16 16-bit entries
  // (8 or 4: one 16- or 8-byte load) or 4 32-bit ones
  constexpr int E = IDX16 ? STEP_CHUNK16 : 4;
  constexpr uint32_t ESZ = IDX16 ? 2u : 4u;
  constexpr uint32_t CB = (uint32_t)E * ESZ;  // chunk bytes
  using chunk_t = uint4;
  auto load_chunk = [&](__amdgpu_buffer_rsrc_t r, uint32_t off) -> chunk_t {
    if constexpr (CB == 16) {
      return load_b128(r, off);
    } else {
      const int2 v = load_i2(r, off);
      return make_uint4((uint32_t)v.x, (uint32_t)v.y, 0u, 0u);
    }
  };
  // buffer resources in scalar registers: this system's pair-list segment
  // (rows packed per tile, plrep_off) and the native pair list, addressed by
  // 32-bit offsets
  const __amdgpu_buffer_rsrc_t rrow =
      buf_rsrc(p.plrep_j + S.pl_base, (uint32_t)S.n * (uint32_t)S.pl_cap * ESZ);
  const __amdgpu_buffer_rsrc_t rnat = buf_rsrc(p.platt, 0xFFFFFFFFu);
  const PosAt<LDS> pos(pin, s_pos, LDS ? lds0 : bead_off);
  const uint32_t row0 = pos.at0 + 16u * (uint32_t)bead_off;  // of row index 0
  float mfx = 0.0f, mfy = 0.0f, mfz = 0.0f;  // force on bead b0 + lane
  bool exact = false;                        // this round takes the guard at every pair
  for (int r = r0; r < r1; ++r) {
    const int li = __shfl(ordm, r * GPW + g);
    const int i = b0 + li;
    const int ns = __shfl(t_ns, li), cn = __shfl(t_cn, li), po = __shfl(t_po, li);
    const int nc = cn & 0xFFFF, nr = cn >> 16;
    float fx = 0.0f, fy = 0.0f, fz = 0.0f;
    uint32_t dmin = ~0u, gmax = 0u;  // least d2 of the unguarded pairs, the guard (as bits)
    if (i < bend) {
      // first loads of the native and non-native loops, issued before any
      // gather: the lane's first row chunk and first two native entries
      // ({partner, bits of r0})
      const uint32_t rowoff = (uint32_t)po * ESZ;
      const int nch = (nr + E - 1) / E;
      chunk_t q = {};
      if (l < nch) q = load_chunk(rrow, rowoff + CB * (uint32_t)l);
      int2 na = make_int2(0, 0), nb2 = make_int2(0, 0);
      if (l < nc) na = load_i2(rnat, 8u * (uint32_t)(ns + l));
      if (l + LPB < nc) nb2 = load_i2(rnat, 8u * (uint32_t)(ns + l + LPB));
      const float4 xi = partner<LDS>(pin, s_pos, lds0, i);
      const int wi = __float_as_int(xi.w);
      const int row = ONE ? q1 : ((wi & 3) - 1) * 2;
      // native LJ over the native pair list (the first two entries per lane loaded above)
      {
        // c = -12 eps u q6 (q6 - 1) with u = 1/d2, q6 = (r0^2 u)^3, as
        // fma(t, q6, -t) with t = -12 eps u q6
        const float eA = -12.0f * S.eps_att[row], eB = ONE ? eA : -12.0f * S.eps_att[row + 1];
        for (int k = l; k < nc; k += LPB) {
          int2 en;
          if (k == l) en = na;
          else if (k == l + LPB) en = nb2;
          else en = load_i2(rnat, 8u * (uint32_t)(ns + k));
          const int j = en.x;
          const float r0 = __int_as_float(en.y);
          const float4 xj = pos.template get<ONE>(pos.at0 + 16u * (uint32_t)j);
          float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
          const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
          const float eps = ONE ? eA : (w_type(xj.w) == 2 ? eB : eA);
          const float r02 = r0 * r0;
          const float ir2 = rcpf(d2);
          const float q2 = r02 * ir2;
          const float q6 = q2 * q2 * q2;
          const float t = eps * ir2 * q6;
          float c = fmaf(t, q6, -t);
          c = d2 > 1.0e-7f * r02 ? c : 0.0f;
          fx = fmaf(c, dx, fx);
          fy = fmaf(c, dy, fy);
          fz = fmaf(c, dz, fz);
        }
      }
      // non-native repulsion: lane l takes chunks l, l + LPB, ... of the row,
      // one load per E pairs, the next chunk's load issued before the current
      // chunk's gathers; the row's padding entries are the bead itself and
      // contribute nothing (d2 = 0 fails the guard)
      {
        // c = u q6 (m12 q6 + m6) with u = 1/d2, q6 = (sigma^2 u)^3, as
        // u^4 (a u^3 + b) with a = m12 sigma^12, b = m6 sigma^6
        const float aA = S.rep_a[row], aB = ONE ? aA : S.rep_a[row + 1];
        const float bA = S.rep_b[row], bB = ONE ? bA : S.rep_b[row + 1];
        const float gA = S.rep_guard[row], gB = ONE ? gA : S.rep_guard[row + 1];
        auto rep = [&](float4 xj, auto guarded) -> float {
          float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
          const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
          const bool tb = !ONE && w_type(xj.w) == 2;
          const float u = rcpf(d2);
          const float u2 = u * u;
          float c = (u2 * u2) * fmaf(tb ? aB : aA, u2 * u, tb ? bB : bA);
          if constexpr (guarded) c = d2 > (tb ? gB : gA) ? c : 0.0f;
          fx = fmaf(c, dx, fx);
          fy = fmaf(c, dy, fy);
          fz = fmaf(c, dz, fz);
          return d2;
        };
        // the E partners of one chunk; the next chunk's load goes out first,
        // without a condition: past the row it reads the rows after it, or
        // zeros past the segment (buffer range check)
        auto chunk = [&](int c, auto guarded) {
          const chunk_t cur = q;
          q = load_chunk(rrow, rowoff + CB * (uint32_t)(c + LPB));
          const uint32_t w[4] = {cur.x, cur.y, cur.z, cur.w};
          float d2[E];
#pragma unroll
          for (int e0 = 0; e0 < E; e0 += GB) {
            float4 x[GB];
#pragma unroll
            for (int g = 0; g < GB; ++g) {
              const int e = e0 + g;
              uint32_t off;
              if constexpr (!IDX16) off = pos.at0 + 16u * w[e % 4];
              else if (e % 2) off = mad16<true>(w[e / 2], row0);
              else off = mad16<false>(w[e / 2], row0);
              x[g] = pos.template get<ONE>(off);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < GB; ++g) d2[e0 + g] = rep(x[g], guarded);
            __builtin_amdgcn_sched_barrier(0);
          }
          if constexpr (!guarded) {
#pragma unroll
            for (int e = 0; e < E; e += 2)
              dmin = min(min(dmin, __float_as_uint(d2[e])), __float_as_uint(d2[e + 1]));
          }
        };
        // Every pair whose d2 is not above the guard contributes nothing.  The
        // guard is taken at each pair of a lane's last chunk, which alone can
        // hold padding; before it only the least d2 is kept (a sum of squares:
        // its bits order as it does), and a round that met one at or below the
        // larger guard is done again with the guard at every pair.  Not
        // unrolled: a lane's chunk counts in a round differ by one, and the odd
        // chunk of a loop of pairs cost every round half a chunk.  The vector
        // ALUs issue in nine of ten cycles, and LDS, half of them conflicts, in
        // six: 17.8 vector instructions a pair instead of 19.6 and a 1/11 fewer
        // in all take 69.2 us instead of 70.3 for 512 replicas (the clock falls
        // to 2.05 GHz in either), 40.4 instead of 42.8 for 200 of two bead
        // types, and 32.4 instead of 33.8 for 200,000 beads gathered from
        // global memory, where four partners asked for together count more.
        gmax = max(__float_as_uint(gA), __float_as_uint(gB));
        const int nfast = exact ? 0 : nch - LPB;
        int c = l;
#pragma unroll 1
        for (; c < nfast; c += LPB) chunk(c, std::false_type());
#pragma unroll 1
        for (; c < nch; c += LPB) chunk(c, std::true_type());
      }
    }
    if (!exact && __ballot(dmin <= gmax)) {
      exact = true;
      --r;
      continue;
    }
    exact = false;
    fx = group_sum<LPB>(fx);
    fy = group_sum<LPB>(fy);
    fz = group_sum<LPB>(fz);
    const float vx = __shfl(fx, src), vy = __shfl(fy, src), vz = __shfl(fz, src);
    if (rm == r) {
      mfx = vx;
      mfy = vy;
      mfz = vz;
    }
  }
  const float3 ch = chain_force<LDS>(p, S, s, b0, pin, s_pos, lds0, t_br, br_before);
  if (b0 + lane >= bend || rm < r0 || rm >= r1) return;  // (a split tile's other beads are its other waves')
  float n0 = 0.0f, n1 = 0.0f, n2 = 0.0f;
  if (MODE != MODE_FORCE)
    normals3(S.seed_lo, S.seed_hi, (uint32_t)(b0 + lane - bead_off), S.step + kstep, n0, n1, n2);
  integrate<LDS>(p, S, s, b0 + lane, MODE, pin, pout, s_pos, lds0, mfx + ch.x, mfy + ch.y, mfz + ch.z, n0, n1, n2);
}

// Stage an item's arena beads [z, z + w) (whole tiles) into LDS.  Wave v
// copies tiles v, v + STEP_WAVES, ...: lane j first looks up the coordinate
// buffer of tile v + STEP_WAVES * j (one dependent chain per wave instead of
// one per bead), then each batch of copies issues all its loads before its
// LDS writes.
__device__ __forceinline__ void stage_item(const DevPtrs &p, int z, int w, int kstep, float4 *s_pos, int wave,
                                           int lane) {
  const int t0 = z / TILE, nt = w / TILE;
  const int mt = wave + STEP_WAVES * lane;
  int par = 0;
  if (mt < nt) par = p.sys[p.tile_sys[t0 + mt]].parity + kstep;
  constexpr int JB = 5;
  if (wave >= nt) return;
  const int jl = (nt - 1 - wave) / STEP_WAVES;  // this wave's last tile is wave + STEP_WAVES * jl
  for (int j0 = 0; j0 <= jl; j0 += JB) {
    // no conditions, so every load issues before the first write: past its
    // last tile the wave copies that tile again (same data, same buffer)
    float4 v[JB];
    int k[JB];
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      const int jj = min(j0 + j, jl);
      k[j] = wave + STEP_WAVES * jj;
      const int pj = __shfl(par, jj);
      v[j] = buf_in(p, pj)[z + k[j] * TILE + lane];
    }
#pragma unroll
    for (int j = 0; j < JB; ++j) s_pos[k[j] * TILE + lane] = v[j];
  }
}

// Work items of one launch: LDS items (tier 0), whole-CU LDS items (tier 1),
// the items that gather from global memory (KLDS = false), or the LDS items and
// then those (TIER_MIXED: a batch with no whole-CU items).
constexpr int TIER_MIXED = 2;
template <bool KLDS, bool FILTER>
__device__ __forceinline__ void item_range(const DevPtrs &p, int tier, int &w0, int &w1) {
  const int n0 = FILTER ? *p.nfitems : *p.nitems, n1 = FILTER ? *p.nfitems_big : *p.nitems_big;
  if (!KLDS) {
    w0 = n0 + n1;
    w1 = w0 + (FILTER ? *p.nfitems_far : *p.nitems_far);
  } else if (tier == TIER_MIXED) {
    w0 = 0;
    w1 = n0 + n1 + *p.nitems_far;
  } else if (tier == 0) {
    w0 = 0;
    w1 = n0;
  } else {
    w0 = n0;
    w1 = n0 + n1;
  }
}

// Fused step over work items {first tile, tiles | waves per tile << 8, first
// staged bead or -1, staged beads}: with s waves per tile, waves s k .. s k +
// s - 1 of the block share tile first + k, each taking LPB / s consecutive
// rounds (tiles * s <= STEP_WAVES).  The LDS kernel (KLDS) takes the items
// whose systems fit in LDS and first copies the staged arena beads (whole
// systems, each from its own coordinate buffer) into dynamic LDS, so every
// partner gather is an LDS read; the other kernel takes the items that gather
// from global memory (items[nitems .. nitems + nitems_far)).  The result is
// identical either way, and k_step_tile's.
template <int LPB, int MODE, bool KLDS, bool MIXED = false>
__device__ __forceinline__ void step_items(const DevPtrs &p, int kstep, float4 *s_pos, int tier) {
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: system data in scalar registers
  int w0, w1;
  item_range<KLDS, false>(p, tier, w0, w1);
  for (int w = w0 + blockIdx.x; w < w1; w += gridDim.x) {
    const int4 it = sload(p.items + w);
    if (it.x < 0) continue;
    const bool staged = KLDS && (!MIXED || it.z >= 0);
    if (staged) {
      __syncthreads();  // the previous item's reads are done
      stage_item(p, it.z, it.w, kstep, s_pos, wave, tid & 63);
      __syncthreads();
    }
    // split tiles: waves ns*k .. ns*k + ns - 1 share tile k of the item, each
    // taking LPB / ns consecutive rounds
    const int ns = __builtin_amdgcn_readfirstlane(item_split(it.y));
    const int tw = wave / ns;
    const int r0 = (wave % ns) * (LPB / ns), r1 = r0 + LPB / ns;
    if (tw >= item_tiles(it.y)) continue;
    const int t = it.x + tw;
    const int s = sload(p.tile_sys + t);
    SysConst &S = sys_const(p, s);
    const int par = S.parity + kstep;
    const float4 *__restrict__ pin = buf_in(p, par);
    float4 *__restrict__ pout = buf_out(p, par);
    if (MODE == MODE_STEP && S.step + kstep >= S.step_end) {
      // finished inside this block of steps: carry the coordinates over
      const int i = t * TILE + (tid & 63);
      if (r0 == 0 && i < S.bead_off + S.n) pout[i] = pin[i];
      continue;
    }
    const bool one = S.type_mask != 3;
    if (staged) {  // (small enough for 16-bit rows)
      if (one) wave_tile<LPB, MODE, KLDS, true, true, 2>(p, S, s, t, kstep, pin, pout, s_pos, it.z, r0, r1);
      else wave_tile<LPB, MODE, KLDS, true, false, 2>(p, S, s, t, kstep, pin, pout, s_pos, it.z, r0, r1);
    } else if constexpr (!KLDS || MIXED) {
      constexpr int GB = MIXED ? 2 : 4;  // (the mixed launch has half the registers)
      if (S.idx16) {
        if (one) wave_tile<LPB, MODE, false, true, true, GB>(p, S, s, t, kstep, pin, pout, s_pos, 0, r0, r1);
        else wave_tile<LPB, MODE, false, true, false, GB>(p, S, s, t, kstep, pin, pout, s_pos, 0, r0, r1);
      } else {
        if (one) wave_tile<LPB, MODE, false, false, true, GB>(p, S, s, t, kstep, pin, pout, s_pos, 0, r0, r1);
        else wave_tile<LPB, MODE, false, false, false, GB>(p, S, s, t, kstep, pin, pout, s_pos, 0, r0, r1);
      }
    }
  }
}

// The tile's bead order for the filter and the step kernel: decreasing row
// length (shell-row length + the last native pair-list length), ties by
// index, so that the beads one round of lane groups takes together run loops
// of similar length.  Computed at grid and neighbor-list builds (before this
// pass rewrites platt_cnt): shell builds keep the order of the grid build that
// made their shell rows (row lengths change little between them).  The order
// only groups beads into rounds; no result depends on it.  Returns the bead of
// slot `lane`; beads past the system's end come last.
__device__ __forceinline__ int tile_order(const DevPtrs &p, int t, int build, bool tin, int nr, bool write) {
  const int lane = threadIdx.x & 63;
  if (build == BUILD_SHELL) return p.tile_ord[t * TILE + lane];
  const int key = tin ? nr + p.platt_cnt[t * TILE + lane] : -1;
  int rank = 0;
  for (int j = 0; j < TILE; ++j) {
    const int kj = __builtin_amdgcn_readlane(key, j);
    rank += (kj > key) | ((kj == key) & (j < lane));
  }
  if (write) p.tile_ord[t * TILE + rank] = (uint8_t)lane;
  return __builtin_amdgcn_ds_permute(rank << 2, lane);  // slot lane holds the bead of that rank
}

// Pair list of one tile's beads = their shell rows filtered at x with the
// reference's exact predicate (d2 < rc_pl^2, squares summed in order without
// contraction), for grid and shell builds, and the native pair list from the
// native CSR.  Neighbor-list builds: k_rows has left the filtered rows in
// the shell-row slots and written the native pair list; the rows are packed
// here as they are.  4 lanes per bead, 16 beads per round: lane l
// takes 4-entry chunks l, l + 4, ... of the row, kept entries are compacted
// per chunk position, so a row comes out in (chunk pass, position, lane)
// order.  The rows are packed per tile (plrep_off): a round's row starts
// follow from its kept counts, so a round first stages up to FILTER_SROW
// entries per row in LDS (STAGE) and writes them out once the starts are
// known; the entries past FILTER_SROW, and every entry without staging, come
// from a second pass over the round's rows, which repeats the first's
// compaction order.  Rows are padded to ROW_PAD entries for the step kernel.
// Bound by latency and memory together: a staging block has a compute unit to
// itself (three waves per SIMD at work on average), reads 0.3 GB of shell rows
// and natives and writes 0.2 GB of lists for 512 replicas, with the vector ALUs
// at half and LDS at 43 %.  Addresses by one multiply-add an entry, the row's
// end tested only in chunks that reach it, and one word of keep bits per chunk
// took it from 229 to 209 us.
template <bool LDS, bool IDX16, bool STAGE, bool ONE>
__device__ __forceinline__ void filter_tile(const DevPtrs &p, SysConst &S, int s, int t,
                                            const float4 *__restrict__ pin, const float4 *s_pos, int lds0,
                                            void *s_stage) {
  using ent_t = typename std::conditional<IDX16, uint16_t, uint32_t>::type;
  using chunk_t = typename std::conditional<IDX16, uint2, uint4>::type;
  const int lane = threadIdx.x & 63, g = lane >> 2, l = lane & 3;
  const uint32_t lb = 1u << l, below = lb - 1u;
  // system constants in registers: the stores below may alias SysDev as far
  // as the compiler knows, and a reload would wait for every earlier store
  const int bo = S.bead_off, pl_cap = S.pl_cap;
  const int64_t pl_base = S.pl_base;
  const int bend = min(t * TILE + TILE, bo + S.n);
  const bool nlb = S.build == BUILD_NL;  // neighbor-list build: rows already filtered (k_rows)
  // cutoffs as wave-uniform values (a per-lane indexed load would be a vector
  // load, and waiting for it would also wait for the earlier stores)
  const float rc11 = S.rc2_pl_rep[0], rc12 = S.rc2_pl_rep[1], rc21 = S.rc2_pl_rep[2], rc22 = S.rc2_pl_rep[3];
  // row lengths of the whole tile in one load, picked up by shuffles; beads
  // in the tile's order (tile_ord), slot q = 16 r + g
  const bool tin = t * TILE + lane < bend;
  const int t_nr = tin ? p.slrep_cnt[t * TILE + lane] : 0;
  const int t_ns = tin ? p.nat_start[t * TILE + lane] : 0, t_nn = tin ? p.nat_cnt[t * TILE + lane] : 0;
  const int ordm = tile_order(p, t, S.build, tin, t_nr, true);
  const double plf = S.pl_factor;
  const float pla = S.pl_abs;
  ent_t *const seg = reinterpret_cast<ent_t *>(p.plrep_j + pl_base);
  const PosAt<LDS> pos(pin, s_pos, LDS ? lds0 : bo);
  const uint32_t row0 = pos.at0 + 16u * (uint32_t)bo;  // of row index 0
  // this tile's region of the segment, and the rows packed so far; the same
  // for the native pair list, whose region is the tile's native CSR range
  const int region = (t * TILE - bo) * pl_cap;
  int packed = 0;
  const int nat_region = __shfl(t_ns, 0);
  int nat_packed = 0;
  for (int r = 0; r < 4; ++r) {
    const int li = __shfl(ordm, r * 16 + g);
    const int i = t * TILE + li;
    const bool act = i < bend;
    const int self = act ? i : bend - 1;  // a bead of this tile: safe to gather
    const int nr = __shfl(t_nr, li);
    // shuffles outside any condition: a lane that a condition turns off does
    // not provide its value to the lanes reading from it
    const int ns = __shfl(t_ns, li), nn_all = __shfl(t_nn, li);
    const int nn = act && !nlb ? nn_all : 0;
    // the bead's first NB natives per lane, loaded with the row's first batch
    constexpr int NB = 4;
    int nj[NB];
    float nr0[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int k = l + 4 * b;
      nj[b] = self;
      nr0[b] = 0.0f;
      if (k < nn) {
        nj[b] = p.nat_j[ns + k];
        nr0[b] = p.nat_r0[ns + k];
      }
    }
    const float4 xi = partner<LDS>(pin, s_pos, lds0, self);
    const bool t2 = (__float_as_int(xi.w) & 3) == 2;
    // the cutoffs by the partner's type (one-type systems: the one of their type)
    const float rcA = ONE ? (t2 ? rc22 : rc11) : (t2 ? rc21 : rc11), rcB = t2 ? rc22 : rc12;
    const uint32_t self_off = pos.at0 + 16u * (uint32_t)self;
    const chunk_t *src = reinterpret_cast<const chunk_t *>(
        reinterpret_cast<const ent_t *>(p.slrep_j + pl_base) + (int64_t)(self - bo) * pl_cap);
    ent_t *s_row = STAGE ? reinterpret_cast<ent_t *>(s_stage) + g * FILTER_SROW : nullptr;  // this group's staged row
    // One pass over the first m entries of the row (m = 0: the group takes
    // no part): kept entries in (chunk batch, position, lane) order, put(o, j)
    // for the o-th.  Chunks in batches of CB per lane, all loads of a batch
    // issued before its stores (a load issued after a store waits for the
    // store as well).  The order does not depend on CB.
    auto pass = [&](int m, auto put) -> int {
      constexpr int CB = IDX16 ? 8 : 4;  // 64 bytes of row loads in flight per lane
      const int nch = (m + 3) >> 2;
      const int clast = max(nch - 1, 0);
      int cnt = 0;
      // one chunk of each lane; full: no lane's is past its row's end.  Staged
      // positions: the keep bits of a group's four lanes, position-major as
      // the row's order, meet in one word, and entry (e, l) goes behind the
      // bits below 4 e + l; gathered ones are decided as each arrives (waiting
      // for all four cost 2 us of 67 for 200,000 beads).
      auto chunk = [&](const chunk_t &ch, int c, auto full) {
        ent_t v[4];
        uint32_t off[4];
        if constexpr (IDX16) {
          v[0] = (ent_t)ch.x; v[1] = (ent_t)(ch.x >> 16); v[2] = (ent_t)ch.y; v[3] = (ent_t)(ch.y >> 16);
          off[0] = mad16<false>(ch.x, row0); off[1] = mad16<true>(ch.x, row0);
          off[2] = mad16<false>(ch.y, row0); off[3] = mad16<true>(ch.y, row0);
        } else {
          v[0] = ch.x; v[1] = ch.y; v[2] = ch.z; v[3] = ch.w;
#pragma unroll
          for (int e = 0; e < 4; ++e) off[e] = pos.at0 + 16u * v[e];
        }
        float4 xj[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // (an entry past the row's end reads the bead itself)
          if constexpr (!full) off[e] = 4 * c + e < m ? off[e] : self_off;
          xj[e] = pos.template get<ONE>(off[e]);
        }
        bool keep[4];
        uint32_t bits = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // the reference's predicate without the minimum image, which is the
          // identity here (a grid build whose extent reaches boxl/2 - margin
          // raises ERR_PBC, and beads move less than the margin before the next)
          const float dx = xj[e].x - xi.x, dy = xj[e].y - xi.y, dz = xj[e].z - xi.z;
          const float rc = ONE ? rcA : (w_type(xj[e].w) == 2 ? rcB : rcA);
          keep[e] = ((dx * dx + dy * dy) + dz * dz) < rc;
          if (nlb) keep[e] = true;
          if constexpr (!full) keep[e] = keep[e] & (4 * c + e < m);
          if constexpr (LDS) {
            bits |= keep[e] ? lb << (4 * e) : 0u;
          } else {
            const uint32_t eb = (uint32_t)(__builtin_amdgcn_ballot_w64(keep[e]) >> (4 * g)) & 0xFu;
            if (keep[e]) put(cnt + __popc(eb & below), v[e]);
            cnt += __popc(eb);
          }
        }
        if constexpr (!LDS) return;
        bits |= (uint32_t)__builtin_amdgcn_mov_dpp((int)bits, 0xB1, 0xF, 0xF, true);
        bits |= (uint32_t)__builtin_amdgcn_mov_dpp((int)bits, 0x4E, 0xF, 0xF, true);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (keep[e]) put(cnt + __popc(bits & ((lb << (4 * e)) - 1u)), v[e]);
        cnt += __popc(bits);
      };
      for (int m0 = 0; __ballot(l + 4 * m0 < nch) != 0; m0 += CB) {
        chunk_t ch[CB];
#pragma unroll
        for (int b = 0; b < CB; ++b) ch[b] = src[min(l + 4 * (m0 + b), clast)];
#pragma unroll
        for (int b = 0; b < CB; ++b) {
          const int c = l + 4 * (m0 + b);
          if (__ballot(c < nch) == 0) break;
          if (LDS && __ballot(4 * c + 4 > m) == 0) chunk(ch[b], c, std::true_type());
          else chunk(ch[b], c, std::false_type());
        }
      }
      return cnt;
    };
    const int mrow = act ? nr : 0;
    int cnt;
    if constexpr (STAGE) {
      cnt = pass(mrow, [&](int o, ent_t v) {
        if (o < FILTER_SROW) s_row[o] = v;
      });
    } else {
      cnt = pass(mrow, [](int, ent_t) {});
    }
    // native pair list: natives within their pair cutoff, in native order,
    // packed per tile like the rows (platt_off): the keep decisions first,
    // kept as one bit per entry of the lane (up to 32), then the entries at
    // the round's starts.  A batch past the first is loaded again for the
    // writes; a bead with more than 128 natives (4 lanes x 32) has its
    // decisions made again.
    int h_ncnt = 0, h_noff = 0;  // the bead's native pair-list length and offset in the tile's slots
    if (nlb) {
      if (act) {
        h_ncnt = p.platt_cnt[i];
        h_noff = p.platt_off[i] - nat_region;
      }
    } else {
      const bool multi = __ballot(nn > 4 * NB) != 0, huge = __ballot(nn > 4 * 32) != 0;
      uint32_t km = 0;  // keep bits: bit m0 + b for the lane's entry l + 4 (m0 + b)
      auto nat_pass = [&](bool wr, int o0) -> int {
        int ncnt = 0;
        for (int m0 = 0; __ballot(l + 4 * m0 < nn) != 0; m0 += NB) {
          if (m0 > 0 || (wr && multi)) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
              const int k = l + 4 * (m0 + b);
              nj[b] = self;
              nr0[b] = 0.0f;
              if (k < nn) {
                nj[b] = p.nat_j[ns + k];
                nr0[b] = p.nat_r0[ns + k];
              }
            }
          }
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            bool keep;
            const int bit = m0 + b;
            if (wr && !huge) {
              keep = (km >> bit) & 1u;
            } else {
              const int k = l + 4 * (m0 + b);
              const float4 xj = partner<LDS>(pin, s_pos, lds0, nj[b]);
              const float rc = cutoff_of(plf, pla, nr0[b]);
              // the reference's predicate without the minimum image (see above)
              const float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
              keep = (k < nn) & (((dx * dx + dy * dy) + dz * dz) < rc * rc);
              if (!wr && bit < 32 && keep) km |= 1u << bit;
            }
            const uint32_t bits = (uint32_t)(__ballot(keep) >> (4 * g)) & 0xFu;
            if (wr && keep) p.platt[o0 + ncnt + __popc(bits & below)] = make_int2(nj[b], __float_as_int(nr0[b]));
            ncnt += __popc(bits);
          }
        }
        return ncnt;
      };
      const int ncnt = nat_pass(false, 0);
      const int nincl = wave_incl_scan(l == 0 ? ncnt : 0);
      const int nstart = nat_region + nat_packed + nincl - ncnt;
      nat_packed += __shfl(nincl, 63);
      nat_pass(true, nstart);
      if (act && l == 0) {
        p.platt_cnt[i] = ncnt;
        p.platt_off[i] = nstart;
      }
      h_ncnt = ncnt;
      h_noff = nstart - nat_region;
    }
    // row starts: the round's rows follow the rows packed so far, in slot order
    const int c = act ? min(cnt, pl_cap) : 0;
    const int len = (c + ROW_PAD - 1) & ~(ROW_PAD - 1);
    const int incl = wave_incl_scan(l == 0 ? len : 0);
    const int start = region + packed + incl - len;
    packed += __shfl(incl, 63);
    ent_t *dst = seg + start;
    if (act && l == 0) {
      p.plrep_cnt[i] = c;
      p.plrep_off[i] = start;
      p.plhead[i] = make_uint2((uint32_t)h_ncnt | ((uint32_t)c << 16),
                               (uint32_t)((start - region) / ROW_PAD) | ((uint32_t)h_noff << 16));
      if (cnt > pl_cap) atomicOr(&p.sys[s].err, ERR_PL_OVF);
    }
    // pad to a multiple of ROW_PAD with the bead itself (its d2 = 0 fails the
    // step kernel's repulsion guard)
    const ent_t me = (ent_t)(IDX16 ? i - bo : i);
    for (int k = c + l; k < len; k += 4) {
      if (STAGE && k < FILTER_SROW) s_row[k] = me;
      else dst[k] = me;
    }
    if constexpr (STAGE) {
      // the staged part of each row to global memory in 8-byte chunks (row
      // starts are multiples of ROW_PAD entries from a 64-byte aligned segment)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      constexpr int PER8 = 8 / (int)sizeof(ent_t);
      const int nst = min(len, FILTER_SROW) / PER8;
      const uint2 *srow2 = reinterpret_cast<const uint2 *>(s_row);
      uint2 *drow2 = reinterpret_cast<uint2 *>(dst);
      for (int k = l; k < nst; k += 4) drow2[k] = srow2[k];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // the entries not staged: a second pass over the rows that have them
    const int lo = STAGE ? FILTER_SROW : 0;
    if (__ballot(c > lo) != 0) {
      pass(c > lo ? mrow : 0, [&](int o, ent_t v) {
        if (o >= lo && o < c) dst[o] = v;
      });
    }
  }
}

// Shell filter over its own work items (the step kernel's LDS staging, one
// wave per tile): wave w of the block takes tile first + w of its item.
// stage_off >= 0: rows are staged in LDS at this byte offset (FILTER_SROW
// entries per bead of a round, per wave), for systems whose entries fit
// stage_bytes (16-bit entries need FILTER_STAGE_BYTES, 32-bit twice that).
template <bool KLDS>
__global__ __launch_bounds__(STEP_THREADS) void k_shell_filter(DevPtrs p, int kstep, int tier, int stage_off,
                                                               int stage_bytes, int builds) {
  extern __shared__ float4 s_pos[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  char *s_stage = reinterpret_cast<char *>(s_pos) + stage_off;
  // the filter of the grid builds runs after their rows: the rebuild's work
  // counters go back to empty for the next one
  if (blockIdx.x == 0 && tid == 0 && ((builds >> BUILD_DIRECT) & 1)) {
    *p.ncellwork = 0;
    *p.nlbuild = 0;
  }
  int w0, w1;
  item_range<KLDS, true>(p, tier, w0, w1);
  for (int w = w0 + blockIdx.x; w < w1; w += gridDim.x) {
    const int4 it = sload(p.fitems + w);
    if (it.x < 0) continue;
    // one wave per tile (the tile order it computes first must come from one
    // wave); a tile is filtered when its system's build is one of `builds`
    // (bit per build kind).  Every wave reads the whole item's decisions, so
    // an item with nothing to filter is skipped by the whole block (no
    // staging) without a block-wide vote.
    const int lane = tid & 63;
    bool mine = false;
    if (lane < item_tiles(it.y)) mine = ((builds >> p.sys[p.tile_sys[it.x + lane]].build) & 1) != 0;
    const uint64_t tiles_mine = __ballot(mine);
    if (tiles_mine == 0) continue;
    if (KLDS) {
      __syncthreads();  // the previous item's reads are done
      stage_item(p, it.z, it.w, kstep, s_pos, wave, lane);
      __syncthreads();
    }
    if (((tiles_mine >> wave) & 1) == 0) continue;
    const int t = it.x + wave;
    const int s = sload(p.tile_sys + t);
    SysConst &S = sys_const(p, s);
    const float4 *pin = buf_in(p, S.parity + kstep);
    const int lds0 = KLDS ? it.z : 0;
    // each wave owns stage_bytes / STEP_WAVES bytes whatever the entry width
    // of the system it filters: the waves of a global-gather block move on to
    // their next item without a barrier, so one wave may stage 16-bit rows
    // while another stages 32-bit ones
    char *wst = s_stage + wave * (stage_bytes / STEP_WAVES);
    const bool st16 = stage_off >= 0 && stage_bytes >= FILTER_STAGE_BYTES;
    const bool st32 = stage_off >= 0 && stage_bytes >= 2 * FILTER_STAGE_BYTES;
    // one-type systems: every partner has the bead's type (one cutoff)
    const bool one = S.type_mask != 3;
    if (KLDS || S.idx16) {  // (staged systems have 16-bit rows)
      if (st16) {
        if (one) filter_tile<KLDS, true, true, true>(p, S, s, t, pin, s_pos, lds0, wst);
        else filter_tile<KLDS, true, true, false>(p, S, s, t, pin, s_pos, lds0, wst);
      } else {
        filter_tile<KLDS, true, false, false>(p, S, s, t, pin, s_pos, lds0, nullptr);
      }
    } else if constexpr (!KLDS) {
      if (!st32) filter_tile<false, false, false, false>(p, S, s, t, pin, s_pos, lds0, nullptr);
      else if (one) filter_tile<false, false, true, true>(p, S, s, t, pin, s_pos, lds0, wst);
      else filter_tile<false, false, true, false>(p, S, s, t, pin, s_pos, lds0, wst);
    }
  }
}

// ---- the same by a block per tile
//
// The filter of the systems that step with a block per tile.  One wave per
// tile is a chain of some 40 dependent round trips (the rounds' row batches,
// gathers, natives and write passes): 25 us for a 4,999-bead system, 46 for
// 10,000, in which most compute units stood empty.  Here eight waves take eight
// rows each, a row 64 entries per pass -- all their entries loaded, then all
// their partners gathered, at once -- and four waves the natives of sixteen
// beads each; one exchange of the waves' totals gives every list its place,
// and the kept entries are written from registers.  Lane 16 q + 4 e + l takes
// entry 16 q + 4 l + e of its pass: a row's kept entries come out in the order
// of the item kernel.  The native lists are packed in bead order.  What a lane
// holds takes 125 registers: one block per compute unit, so two or three tiles a
// unit go through in as many rounds.
constexpr int FILTER_ROW_WAVES = 8, FILTER_NAT_WAVES = 4;
constexpr int FILTER_TILE_THREADS = 64 * (FILTER_ROW_WAVES + FILTER_NAT_WAVES);

template <bool ONE>
__device__ __forceinline__ void filter_rows(const DevPtrs &p, SysConst &S, int b0, int nb, int wave,
                                            const float4 *__restrict__ pin, int *s_len, const int *s_nlen,
                                            const int2 *s_nat) {
  constexpr int R = TILE / FILTER_ROW_WAVES, NP = 2;  // rows of the wave, passes held in registers
  constexpr uint32_t PAST = 0xFFFFFF00u;  // beyond any segment: a load returns 0, a store is dropped
  const int lane = threadIdx.x & 63;
  const int bo = S.bead_off, pl_cap = S.pl_cap;
  const bool nlb = S.build == BUILD_NL;
  const uint32_t bytes = (uint32_t)S.n * (uint32_t)pl_cap * 2u;  // 16-bit entries
  const __amdgpu_buffer_rsrc_t rin = buf_rsrc(p.slrep_j + S.pl_base, bytes), rout = buf_rsrc(p.plrep_j + S.pl_base, bytes);
  const uint32_t region = (uint32_t)(b0 - bo) * (uint32_t)pl_cap;  // this tile's first entry
  auto load = [&](uint32_t entry, bool on) -> int {
    return (int)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rin, (int)(on ? 2u * entry : PAST), 0, 0);
  };
  auto store = [&](uint32_t entry, bool on, int v) {
    __builtin_amdgcn_raw_buffer_store_b16((unsigned short)v, rout, (int)(on ? 2u * entry : PAST), 0, 0);
  };
  const bool tin = lane < nb;
  const int t_nr = tin ? p.slrep_cnt[b0 + lane] : 0;
  const int ordm = tile_order(p, b0 / TILE, S.build, tin, t_nr, wave == 0);
  const int o_nr = __shfl(t_nr, ordm);  // by slot
  const int eo = (lane & 48) + 4 * (lane & 3) + ((lane >> 2) & 3);
  const float4 *__restrict__ base = pin + bo;
  const int vself = b0 - bo;  // a lane without an entry gathers a bead of the system
  int nr[R], li[R], e[R][NP];
#pragma unroll
  for (int g = 0; g < R; ++g) {
    nr[g] = __builtin_amdgcn_readlane(o_nr, R * wave + g);
    li[g] = __builtin_amdgcn_readlane(ordm, R * wave + g);
#pragma unroll
    for (int u = 0; u < NP; ++u)
      e[g][u] = load(region + (uint32_t)(li[g] * pl_cap + 64 * u + eo), 64 * u + eo < nr[g]);
  }
  const float rc11 = S.rc2_pl_rep[0], rc12 = S.rc2_pl_rep[1], rc21 = S.rc2_pl_rep[2], rc22 = S.rc2_pl_rep[3];
  float4 xi[R];
#pragma unroll
  for (int g = 0; g < R; ++g) xi[g] = pin[b0 + min(li[g], nb - 1)];
  // the reference's predicate without the minimum image, which is the identity
  // here (a grid build whose extent reaches boxl/2 - margin raises ERR_PBC, and
  // beads move less than the margin before the next)
  auto kept = [&](int g, bool valid, float4 xj) {
    const bool t2 = w_type(xi[g].w) == 2;
    const float rcA = ONE ? (t2 ? rc22 : rc11) : (t2 ? rc21 : rc11), rcB = t2 ? rc22 : rc12;
    const float dx = xj.x - xi[g].x, dy = xj.y - xi[g].y, dz = xj.z - xi[g].z;
    const float rc = ONE ? rcA : (w_type(xj.w) == 2 ? rcB : rcA);
    return valid & (nlb | (((dx * dx + dy * dy) + dz * dz) < rc));
  };
  uint64_t m[R][NP];
#pragma unroll
  for (int h = 0; h < R; h += R / 2) {  // half the wave's rows gathered at a time
    float4 xj[R / 2][NP];
#pragma unroll
    for (int g = 0; g < R / 2; ++g)
#pragma unroll
      for (int u = 0; u < NP; ++u) xj[g][u] = base[64 * u + eo < nr[h + g] ? e[h + g][u] : vself];
#pragma unroll
    for (int g = 0; g < R / 2; ++g)
#pragma unroll
      for (int u = 0; u < NP; ++u)
        m[h + g][u] = __builtin_amdgcn_ballot_w64(kept(h + g, 64 * u + eo < nr[h + g], xj[g][u]));
  }
  // passes past the held ones: counted now, filtered again when written
  auto tail = [&](int g, bool write, int at) {
    int c = 0;
    for (int m0 = 64 * NP; m0 < nr[g]; m0 += 64) {
      const bool valid = m0 + eo < nr[g];
      const int v = load(region + (uint32_t)(li[g] * pl_cap + m0 + eo), valid);
      const bool k = kept(g, valid, base[valid ? v : vself]);
      const uint64_t mk = __builtin_amdgcn_ballot_w64(k);
      if (write) store(region + (uint32_t)(at + c + lanes_below(mk)), k, v);
      c += __popcll(mk);
    }
    return c;
  };
  int cnt[R], sum = 0;
#pragma unroll
  for (int g = 0; g < R; ++g) {
    cnt[g] = tail(g, false, 0);
#pragma unroll
    for (int u = 0; u < NP; ++u) cnt[g] += __popcll(m[g][u]);
    sum += (cnt[g] + ROW_PAD - 1) & ~(ROW_PAD - 1);
  }
  if (lane == 0) s_len[wave] = sum;
  __syncthreads();
  int packed = 0;
  for (int v = 0; v < wave; ++v) packed += s_len[v];
  int c_q = 0, s_q = 0;
#pragma unroll
  for (int g = 0; g < R; ++g) {
    int at = packed;
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      store(region + (uint32_t)(at + lanes_below(m[g][u])), (m[g][u] >> lane) & 1, e[g][u]);
      at += __popcll(m[g][u]);
    }
    if (nr[g] > 64 * NP) at += tail(g, true, at);
    // padded to a multiple of ROW_PAD with the bead itself (its d2 = 0 fails the
    // step kernel's repulsion guard)
    const int len = (cnt[g] + ROW_PAD - 1) & ~(ROW_PAD - 1);
    store(region + (uint32_t)(at + lane), lane < len - cnt[g], b0 - bo + li[g]);
    c_q = lane == g ? cnt[g] : c_q;
    s_q = lane == g ? packed : s_q;
    packed += len;
  }
  const int lb = __shfl(ordm, R * wave + (lane & (R - 1)));
  if (lane < R && lb < nb) {
    int2 nat = s_nat[lb];  // {length, offset within its wave's sixteen beads}
    if (!nlb)
      for (int v = 0; v < lb / 16; ++v) nat.y += s_nlen[v];
    const int i = b0 + lb;
    p.plrep_cnt[i] = c_q;
    p.plrep_off[i] = (int)region + s_q;
    p.plhead[i] = make_uint2((uint32_t)nat.x | ((uint32_t)c_q << 16), (uint32_t)(s_q / ROW_PAD) | ((uint32_t)nat.y << 16));
  }
}

// Natives within their pair cutoff of sixteen beads, four lanes each: keep
// decisions and counts, then the entries at the lists' places.  Keep bits hold
// 32 batches of four (128 natives of a bead); past them the decision is made
// again for the writes, and batches past the first NB are loaded again.
__device__ __forceinline__ void filter_nats(const DevPtrs &p, SysConst &S, int b0, int nb, int wave,
                                            const float4 *__restrict__ pin, int *s_nlen, int2 *s_nat) {
  constexpr int NB = 4;
  const int lane = threadIdx.x & 63, g = lane >> 2, l = lane & 3;
  const uint32_t below = (1u << l) - 1u;
  const int lb = 16 * wave + g;
  const bool act = lb < nb, nlb = S.build == BUILD_NL;
  const int i = b0 + min(lb, nb - 1);
  const int nat0 = p.nat_start[b0];
  const int ns = p.nat_start[i], nn = act && !nlb ? p.nat_cnt[i] : 0;
  if (nlb) {  // k_rows has left the lists in the beads' own slots
    if (act && l == 0) s_nat[lb] = make_int2(p.platt_cnt[i], p.platt_off[i] - nat0);
    __syncthreads();
    return;
  }
  const double plf = S.pl_factor;
  const float pla = S.pl_abs;
  int j[NB];
  float r0[NB];
  auto load = [&](int m0) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int k = l + 4 * (m0 + b);
      j[b] = i;
      r0[b] = 0.0f;
      if (k < nn) {
        j[b] = p.nat_j[ns + k];
        r0[b] = p.nat_r0[ns + k];
      }
    }
  };
  load(0);
  const float4 xi = pin[i];
  const bool multi = __ballot(nn > 4 * NB) != 0;
  uint32_t km = 0;  // keep bits: bit m0 + b for the lane's entry l + 4 (m0 + b)
  auto pass = [&](bool wr, int o0) {
    int c = 0;
    for (int m0 = 0; __ballot(l + 4 * m0 < nn) != 0; m0 += NB) {
      if (m0 > 0 || (wr && multi)) load(m0);
      float4 xj[NB];
      const bool test = !wr || m0 >= 32;
      if (test) {
#pragma unroll
        for (int b = 0; b < NB; ++b) xj[b] = pin[j[b]];
      }
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int bit = m0 + b;
        bool keep;
        if (test) {
          const float rc = cutoff_of(plf, pla, r0[b]);
          const float dx = xj[b].x - xi.x, dy = xj[b].y - xi.y, dz = xj[b].z - xi.z;
          keep = (l + 4 * bit < nn) & (((dx * dx + dy * dy) + dz * dz) < rc * rc);
          if (!wr && bit < 32 && keep) km |= 1u << bit;
        } else {
          keep = (km >> bit) & 1u;
        }
        const uint32_t bits = (uint32_t)(__ballot(keep) >> (4 * g)) & 0xFu;
        if (wr && keep) p.platt[o0 + c + __popc(bits & below)] = make_int2(j[b], __float_as_int(r0[b]));
        c += __popc(bits);
      }
    }
    return c;
  };
  const int c = pass(false, 0);
  const int incl = wave_incl_scan(l == 0 ? c : 0);
  if (lane == 63) s_nlen[wave] = incl;
  if (act && l == 0) s_nat[lb] = make_int2(c, incl - c);
  __syncthreads();
  int off = incl - c;
  for (int v = 0; v < wave; ++v) off += s_nlen[v];
  pass(true, nat0 + off);
  if (act && l == 0) {
    p.platt_cnt[i] = c;
    p.platt_off[i] = nat0 + off;
  }
}

__global__ __launch_bounds__(FILTER_TILE_THREADS) void k_filter_tile(DevPtrs p, int kstep, int builds) {
  __shared__ int s_len[FILTER_ROW_WAVES], s_nlen[FILTER_NAT_WAVES];
  __shared__ int2 s_nat[TILE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the filter of the grid builds runs after their rows: the rebuild's work
  // counters go back to empty for the next one
  if (blockIdx.x == 0 && threadIdx.x == 0 && ((builds >> BUILD_DIRECT) & 1)) {
    *p.ncellwork = 0;
    *p.nlbuild = 0;
  }
  // (the table has room for every block of the grid)
  const int ntiles = sload(p.ntiles);
  int2 it = sload(p.tiles + blockIdx.x);
  for (int w = blockIdx.x; w < ntiles; w += gridDim.x) {
    if (w != (int)blockIdx.x) {
      __syncthreads();  // the previous tile's totals have been read
      it = sload(p.tiles + w);
    }
    if (it.x < 0) continue;
    SysConst &S = sys_const(p, it.y);
    if (((builds >> S.build) & 1) == 0) continue;
    const int b0 = it.x * TILE, nb = min(TILE, S.bead_off + S.n - b0);
    const float4 *__restrict__ pin = buf_in(p, S.parity + kstep);
    if (wave >= FILTER_ROW_WAVES) {
      filter_nats(p, S, b0, nb, wave - FILTER_ROW_WAVES, pin, s_nlen, s_nat);
    } else if (S.type_mask != 3) {
      filter_rows<true>(p, S, b0, nb, wave, pin, s_len, s_nlen, s_nat);
    } else {
      filter_rows<false>(p, S, b0, nb, wave, pin, s_len, s_nlen, s_nat);
    }
  }
}

// 8 waves per SIMD: two blocks per compute unit
template <int LPB, int MODE>
__global__ __launch_bounds__(STEP_THREADS, 8) void k_step(DevPtrs p, int kstep, int tier) {
  extern __shared__ float4 s_pos[];
  step_items<LPB, MODE, true>(p, kstep, s_pos, tier);
}

// The LDS items and the global-gather ones in one launch, at two blocks per
// compute unit.  Two launches on two streams cost the graph a fork and a join,
// 9 us a step, and the gathering blocks got the registers of one per unit.
// Run per step, two launches / one: 12 systems of 1,500 beads and one of
// 18,000 40.1 / 33.5 us, 60 and 3 59.2 / 49.4, 120 and 1 62.6 / 48.7, 120 and 8
// 102.5 / 96.0.
template <int LPB, int MODE>
__global__ __launch_bounds__(STEP_THREADS, 8) void k_step_mixed(DevPtrs p, int kstep) {
  extern __shared__ float4 s_pos[];
  step_items<LPB, MODE, true, true>(p, kstep, s_pos, TIER_MIXED);
}

template <int LPB, int MODE>
__global__ __launch_bounds__(STEP_THREADS) void k_step_far(DevPtrs p, int kstep) {
  step_items<LPB, MODE, false>(p, kstep, nullptr, 0);
}

// ---- a block per tile
//
// The step of a small batch (at most TILE_STEP_PER_CU tiles per compute unit)
// and of the systems too large to stage in LDS.  A small batch is bound by
// latency, not by the vector ALUs: each compute unit has a handful of waves,
// and with whole systems staged in LDS a 4,999-bead step spent 18,000 of its
// 26,000 cycles waiting for the 80 KB copies of 79 blocks.  So nothing is
// staged -- the positions are in the L2s, and a wave's gathers are issued in
// batches of sixteen -- and a tile's work is spread over as many waves as it
// has parts:
//   - up to 8 waves take the rounds (64 / LPB beads each): heads, the row's
//     chunks and native entries, gathers, forces, left in LDS;
//   - one more wave draws the tile's noise and computes its chain terms beside
//     them, then adds the forces up and moves the beads.
// The arithmetic of a bead and its order are those of the item kernels:
// results are identical.

// The lane's bead of round r and its list ranges, from the tile's heads.
struct RoundAt {
  int li, i, ns, nc, nr;
  uint32_t row;  // first entry of the row in the system's segment
};
template <int LPB>
__device__ __forceinline__ RoundAt round_at(int r, int b0, int bend, int ordm, uint2 hd, int nat0, int reg0) {
  constexpr int GPW = 64 / LPB;
  RoundAt a;
  a.li = __shfl(ordm, r * GPW + (int)(threadIdx.x & 63) / LPB);
  const uint32_t cn = (uint32_t)__shfl((int)hd.x, a.li), po = (uint32_t)__shfl((int)hd.y, a.li);
  a.i = b0 + a.li;
  const bool in = a.i < bend;
  a.nc = in ? (int)(cn & 0xFFFFu) : 0;
  a.nr = in ? (int)(cn >> 16) : 0;
  a.ns = nat0 + (int)(po >> 16);
  a.row = (uint32_t)reg0 + (uint32_t)ROW_PAD * (po & 0xFFFFu);
  return a;
}

// Gathered native and non-native force on the lane group's bead.
template <int LPB, bool ONE>
__device__ __forceinline__ float3 tile_round(const DevPtrs &p, SysConst &S, const float4 *__restrict__ pin, int self,
                                             const RoundAt &a) {
  const int l = (int)(threadIdx.x & 63) % LPB;
  // buffer resources in scalar registers: the system's pair-list segment
  // (16-bit entries) and the natives
  const __amdgpu_buffer_rsrc_t rrow = buf_rsrc(p.plrep_j + S.pl_base, (uint32_t)S.n * (uint32_t)S.pl_cap * 2u);
  const __amdgpu_buffer_rsrc_t rnat = buf_rsrc(p.platt, 0xFFFFFFFFu);
  constexpr int D = 8;   // chunks of four entries held per lane
  constexpr int NB = 4;  // natives held per lane
  uint32_t q[2 * D];
  auto load_chunks = [&](int c0) {  // without a condition: past the segment a buffer load returns zeros
#pragma unroll
    for (int k = 0; k < D; ++k) {
      const int2 v = load_i2(rrow, 2u * a.row + 8u * (uint32_t)(l + LPB * (c0 + k)));
      q[2 * k] = (uint32_t)v.x;
      q[2 * k + 1] = (uint32_t)v.y;
    }
  };
  int2 en[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    en[b] = make_int2(self, 0);  // past the list: the bead itself, which contributes nothing
    if (l + LPB * b < a.nc) en[b] = load_i2(rnat, 8u * (uint32_t)(a.ns + l + LPB * b));
  }
  load_chunks(0);
  const float4 xi = pin[self];
  const int bead_off = S.bead_off;
  const int row = ONE ? (S.type_mask == 2 ? 3 : 0) : (w_type(xi.w) - 1) * 2;  // type-pair index
  const int nch = (a.nr + 3) >> 2;
  const uint32_t sv = (uint32_t)(self - bead_off) * 0x10001u;
  const float4 *__restrict__ base = pin + bead_off;
  // the four partners of chunk position k (a lane past its row: the bead
  // itself, whose d2 = 0 fails the guard)
  auto gather = [&](int k, bool on, float4 *x) {
    const uint32_t w0 = on ? q[2 * k] : sv, w1 = on ? q[2 * k + 1] : sv;
    x[0] = base[w0 & 0xFFFFu];
    x[1] = base[w0 >> 16];
    x[2] = base[w1 & 0xFFFFu];
    x[3] = base[w1 >> 16];
  };
  constexpr int R = 4;  // chunks in flight
  float4 xn[NB], xr[R][4];
#pragma unroll
  for (int b = 0; b < NB; ++b) xn[b] = pin[en[b].x];
#pragma unroll
  for (int k = 0; k < R; ++k)
    if (__ballot(l + LPB * k < nch) != 0) gather(k, l + LPB * k < nch, xr[k]);
  float fx = 0.0f, fy = 0.0f, fz = 0.0f;
  // native LJ: c = -12 eps u q6 (q6 - 1) with u = 1/d2, q6 = (r0^2 u)^3, as
  // fma(t, q6, -t) with t = -12 eps u q6
  {
    const float eA = -12.0f * S.eps_att[row], eB = ONE ? eA : -12.0f * S.eps_att[row + 1];
    auto nat = [&](float4 xj, float r0) {
      const float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
      const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
      const float eps = ONE ? eA : (w_type(xj.w) == 2 ? eB : eA);
      const float r02 = r0 * r0;
      const float ir2 = rcpf(d2);
      const float q2 = r02 * ir2;
      const float q6 = q2 * q2 * q2;
      const float t = eps * ir2 * q6;
      float c = fmaf(t, q6, -t);
      c = d2 > 1.0e-7f * r02 ? c : 0.0f;
      fx = fmaf(c, dx, fx);
      fy = fmaf(c, dy, fy);
      fz = fmaf(c, dz, fz);
    };
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (__ballot(l + LPB * b < a.nc) != 0) nat(xn[b], __int_as_float(en[b].y));
    for (int k = l + NB * LPB; k < a.nc; k += LPB) {
      const int2 e = load_i2(rnat, 8u * (uint32_t)(a.ns + k));
      nat(pin[e.x], __int_as_float(e.y));
    }
  }
  // non-native repulsion: c = u q6 (m12 q6 + m6) with u = 1/d2, q6 =
  // (sigma^2 u)^3, as u^4 (a u^3 + b) with a = m12 sigma^12, b = m6 sigma^6
  {
    const float aA = S.rep_a[row], aB = ONE ? aA : S.rep_a[row + 1];
    const float bA = S.rep_b[row], bB = ONE ? bA : S.rep_b[row + 1];
    const float gA = S.rep_guard[row], gB = ONE ? gA : S.rep_guard[row + 1];
    auto rep = [&](const float4 *x) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float4 xj = x[e];
        const float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
        const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        const bool tb = !ONE && w_type(xj.w) == 2;
        const float u = rcpf(d2);
        const float u2 = u * u;
        float c = (u2 * u2) * fmaf(tb ? aB : aA, u2 * u, tb ? bB : bA);
        c = d2 > (tb ? gB : gA) ? c : 0.0f;
        fx = fmaf(c, dx, fx);
        fy = fmaf(c, dy, fy);
        fz = fmaf(c, dz, fz);
      }
    };
    for (int c0 = 0;;) {
#pragma unroll
      for (int k = 0; k < D; ++k) {
        if (__ballot(l + LPB * (c0 + k) < nch) == 0) break;
        rep(xr[k % R]);
        if (k + R < D && __ballot(l + LPB * (c0 + k + R) < nch) != 0)
          gather(k + R, l + LPB * (c0 + k + R) < nch, xr[k % R]);
      }
      c0 += D;
      if (__ballot(l + LPB * c0 < nch) == 0) break;
      load_chunks(c0);  // rows of more than D chunks a lane
#pragma unroll
      for (int k = 0; k < R; ++k) gather(k, l + LPB * (c0 + k) < nch, xr[k]);
    }
  }
  return make_float3(group_sum<LPB>(fx), group_sum<LPB>(fy), group_sum<LPB>(fz));
}

// waves of a tile's rounds: one round each for up to 8 lanes per bead
constexpr int tile_waves(int lpb) { return lpb < 8 ? lpb : 8; }

template <int LPB>
__global__ __launch_bounds__(64 * (tile_waves(LPB) + 1)) void k_step_tile(DevPtrs p, int kstep, int mode) {
  constexpr int W = tile_waves(LPB);
  __shared__ float s_f[3][TILE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform: system data in scalar registers
  // (the table has room for every block of the grid)
  const int ntiles = sload(p.ntiles);
  int2 it = sload(p.tiles + blockIdx.x);
  for (int w = blockIdx.x; w < ntiles; w += gridDim.x) {
    if (w != (int)blockIdx.x) {
      __syncthreads();  // the previous tile's forces have been read
      it = sload(p.tiles + w);
    }
    if (it.x < 0) continue;
    const int t = it.x, s = it.y;
    const int b0 = t * TILE;
    SysConst &S = sys_const(p, s);
    if (wave < W) {
      const int ordm = p.tile_ord[b0 + lane];
      const uint2 hd = p.plhead[b0 + lane];
      const int nat0 = p.nat_start[b0];
      const int bead_off = S.bead_off;
      const int bend = min(b0 + TILE, bead_off + S.n);
      const float4 *__restrict__ pin = buf_in(p, S.parity + kstep);
      if (mode != MODE_STEP || S.step + kstep < S.step_end) {
        for (int r = wave; r < LPB; r += W) {
          const RoundAt a = round_at<LPB>(r, b0, bend, ordm, hd, nat0, (b0 - bead_off) * S.pl_cap);
          const int self = a.i < bend ? a.i : b0;  // a bead of this system: safe to gather
          const float3 f = S.type_mask != 3 ? tile_round<LPB, true>(p, S, pin, self, a) : tile_round<LPB, false>(p, S, pin, self, a);
          if (lane % LPB == 0) {
            s_f[0][a.li] = f.x;
            s_f[1][a.li] = f.y;
            s_f[2][a.li] = f.z;
          }
        }
      }
      __syncthreads();
    } else {
      const float br = p.bond_r0[b0 + lane], brb = p.bond_r0[max(b0 - 1, 0)];
      const int bead_off = S.bead_off;
      const int bend = min(b0 + TILE, bead_off + S.n);
      const int par = S.parity + kstep;
      const int64_t step = S.step + kstep;
      const float4 *__restrict__ pin = buf_in(p, par);
      float4 *__restrict__ pout = buf_out(p, par);
      const int i = b0 + lane;
      const bool over = mode == MODE_STEP && step >= S.step_end;
      float n0 = 0.0f, n1 = 0.0f, n2 = 0.0f;
      float3 ch = make_float3(0.0f, 0.0f, 0.0f);
      if (over) {
        // finished inside this block of steps: carry the coordinates over
        if (i < bend) pout[i] = pin[i];
      } else {
        ch = chain_force<false>(p, S, s, b0, pin, nullptr, 0, i < bend ? br : 0.0f, b0 > bead_off ? brb : 0.0f);
        if (mode != MODE_FORCE) normals3(S.seed_lo, S.seed_hi, (uint32_t)(i - bead_off), step, n0, n1, n2);
      }
      __syncthreads();
      if (!over && i < bend)
        integrate<false>(p, S, s, i, mode, pin, pout, nullptr, 0, s_f[0][lane] + ch.x, s_f[1][lane] + ch.y,
                         s_f[2][lane] + ch.z, n0, n1, n2);
    }
  }
}

// ------------------------------------------------ energies / observables

// 16 lanes per bead; FP32 pair energies, FP64 accumulation; pairs are seen
// from both beads and weighted 1/2.  Native contacts (d/r0 < 1.25 over all
// natives) are counted from the lower index.  A block of 16 waves takes a tile,
// every bead at once (four waves took sixteen rounds of load chains: 17 us for
// 701 beads, 6 now), and leaves the tile's sums: its 6 energy partials, then
// sum x, y, z, |r|^2.  nt > 0: tiles t0 .. t0 + nt - 1 (one system, no work
// table); else the work table's tiles.
constexpr int ENERGY_THREADS = 1024;
__global__ __launch_bounds__(ENERGY_THREADS) void k_energy(DevPtrs p, int t0, int nt) {
  constexpr int LPB = 16;
  __shared__ double sh[ENERGY_THREADS / 64][TPART_N];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane / LPB, l = lane % LPB;
  const int nwork = nt > 0 ? nt : *p.nwork;
  for (int w = blockIdx.x; w < nwork; w += gridDim.x) {
    const int t = nt > 0 ? t0 + w : sload(p.work + w);
    if (t < 0) continue;
    const int s = sload(p.tile_sys + t);
    SysConst &S = sys_const(p, s);
    const int bead_off = S.bead_off, n = S.n;
    const int b0 = t * TILE;
    const int bend = min(b0 + TILE, bead_off + n);
    const float4 *pin = buf_in(p, S.parity);
    const float boxl = S.boxl, inv_boxl = S.inv_boxl;
    const bool wrapf = S.wrap_free != 0 || boxl <= 0.0f;
    {
      const int i = b0 + wave * (64 / LPB) + g;
      float4 xi = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      double eb = 0.0, ea = 0.0, en = 0.0, er = 0.0, vir = 0.0, con = 0.0;
      if (i < bend) {
        xi = pin[i];
        const int wi = __float_as_int(xi.w);
        const int row = ((wi & 3) - 1) * 2;
        if (l < 4) {
          const int off = l < 2 ? l - 2 : l - 1;
          const int j = i + off;
          if (j >= bead_off && j < bead_off + n) {
            const float4 xj = pin[j];
            if ((__float_as_int(xj.w) >> 2) == (wi >> 2)) {
              float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
              if (!wrapf) {
                dx = mi_fast(dx, boxl, inv_boxl);
                dy = mi_fast(dy, boxl, inv_boxl);
                dz = mi_fast(dz, boxl, inv_boxl);
              }
              const float d2 = dx * dx + dy * dy + dz * dz;
              if (off == 1 || off == -1) {
                const float r0 = p.bond_r0[off < 0 ? j : i];
                const float d = sqrtf(d2);
                const float dev = d - r0;
                const float gg = 1.0f - dev * dev * S.inv_R0sq;
                eb += 0.5 * (double)(-S.half_k_R0sq * log1pf(-dev * dev * S.inv_R0sq));
                const float c = S.k_bnd * dev / (d * gg);
                vir += 0.5 * (double)(-c * d2);
              } else {
                const float ir2 = 1.0f / d2;
                const float ir6 = ir2 * ir2 * ir2;
                ea += 0.5 * (double)(S.ss_e6 * ir6);
                vir += 0.5 * (double)(S.ss_f6 * ir6);
              }
            }
          }
        }
        const int ns = p.nat_start[i], po = p.platt_off[i];
        const int nc = p.platt_cnt[i];
        for (int k = l; k < nc; k += LPB) {
          const int2 pe = p.platt[po + k];
          const int j = pe.x;
          const float r0 = __int_as_float(pe.y);
          const float4 xj = pin[j];
          float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
          if (!wrapf) {
            dx = mi_fast(dx, boxl, inv_boxl);
            dy = mi_fast(dy, boxl, inv_boxl);
            dz = mi_fast(dz, boxl, inv_boxl);
          }
          const float d2 = dx * dx + dy * dy + dz * dz;
          const float eps = w_type(xj.w) == 2 ? S.eps_att[row + 1] : S.eps_att[row];
          const float r02 = r0 * r0;
          const float q2 = r02 / d2;
          const float q6 = q2 * q2 * q2;
          en += 0.5 * (double)(eps * (q6 * q6 - 2.0f * q6));
          if (d2 > 1.0e-7f * r02) vir += 0.5 * (double)(12.0f * eps * q6 * (q6 - 1.0f));
        }
        // contacts over all natives, counted once (partner index above i)
        const int nn = p.nat_cnt[i];
        for (int k = l; k < nn; k += LPB) {
          const int j = p.nat_j[ns + k];
          if (j > i) {
            const float d = sqrtf(dist2_exact(xi, pin[j], boxl));
            if (d / p.nat_r0[ns + k] < 1.25f) con += 1.0;
          }
        }
        const int64_t pb = S.pl_base + p.plrep_off[i];
        const int nr = p.plrep_cnt[i];
        for (int k = l; k < nr; k += LPB) {
          const int j = S.idx16 ? bead_off + ((const uint16_t *)(p.plrep_j + S.pl_base))[pb - S.pl_base + k]
                                : p.plrep_j[pb + k];
          const float4 xj = pin[j];
          float dx = xj.x - xi.x, dy = xj.y - xi.y, dz = xj.z - xi.z;
          if (!wrapf) {
            dx = mi_fast(dx, boxl, inv_boxl);
            dy = mi_fast(dy, boxl, inv_boxl);
            dz = mi_fast(dz, boxl, inv_boxl);
          }
          const float d2 = dx * dx + dy * dy + dz * dz;
          const bool tb = w_type(xj.w) == 2;
          const float q2 = (tb ? S.sig2_rep[row + 1] : S.sig2_rep[row]) / d2;
          const float q6 = q2 * q2 * q2;
          const float ep = tb ? S.eps_rep[row + 1] : S.eps_rep[row];
          er += 0.5 * (double)(ep * (S.c12 * q6 * q6 + S.c6 * q6));
          if (d2 > (tb ? S.rep_guard[row + 1] : S.rep_guard[row]))
            vir += 0.5 * (double)(-((tb ? S.rep_m12[row + 1] : S.rep_m12[row]) * q6 +
                                    (tb ? S.rep_m6[row + 1] : S.rep_m6[row])) * q6);
        }
      }
#pragma unroll
      for (int o = LPB / 2; o >= 1; o >>= 1) {
        eb += __shfl_xor(eb, o);
        ea += __shfl_xor(ea, o);
        en += __shfl_xor(en, o);
        er += __shfl_xor(er, o);
        vir += __shfl_xor(vir, o);
        con += __shfl_xor(con, o);
      }
      // the wave's four beads, then the block's sixteen waves in order
      double v[TPART_N] = {eb, ea, en, er, vir, con, 0.0, 0.0, 0.0, 0.0};
      if (i < bend) {
        v[6] = xi.x;
        v[7] = xi.y;
        v[8] = xi.z;
        v[9] = (double)xi.x * xi.x + (double)xi.y * xi.y + (double)xi.z * xi.z;
      }
#pragma unroll
      for (int k = 0; k < TPART_N; ++k) {
        v[k] += __shfl_xor(v[k], 16);
        v[k] += __shfl_xor(v[k], 32);
      }
      __syncthreads();  // the previous tile's sums have been read
      if (lane == 0) {
#pragma unroll
        for (int k = 0; k < TPART_N; ++k) sh[wave][k] = v[k];
      }
      __syncthreads();
      if (tid < TPART_N) {
        double a = 0.0;
        for (int q = 0; q < ENERGY_THREADS / 64; ++q) a += sh[q][tid];
        p.epart[(int64_t)(t - p.epart_base / TILE) * TPART_N + tid] = a;
      }
    }
  }
}

// Per system, fixed-order sum of the tile partials plus Rg^2 from the centroid
// form (1/N) sum |r|^2 - |r_cm|^2, identical to the reference's pair sum / N^2
// (sop.cu:564-580).  slot >= 0: that system alone; else the batch's systems.
// The values also to out (when not null), in batch order.
__global__ __launch_bounds__(256) void k_sys_reduce(DevPtrs p, int slot, double *out) {
  __shared__ double sh[4][TPART_N];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nsys = slot >= 0 ? 1 : *p.nsys;
  for (int q = blockIdx.x; q < nsys; q += gridDim.x) {
    const int s = slot >= 0 ? slot : sload(p.syslist + q);
    SysConst &S = sys_const(p, s);
    const int nt = (S.n + TILE - 1) / TILE;
    const double *e = p.epart + (int64_t)(S.bead_off - p.epart_base) / TILE * TPART_N;
    double acc[TPART_N];
#pragma unroll
    for (int k = 0; k < TPART_N; ++k) acc[k] = 0.0;
    for (int b = tid; b < nt; b += 256) {
#pragma unroll
      for (int k = 0; k < TPART_N; ++k) acc[k] += e[b * TPART_N + k];
    }
#pragma unroll
    for (int k = 0; k < TPART_N; ++k) acc[k] = wave_sum_d(acc[k]);
    if (lane == 0)
      for (int k = 0; k < TPART_N; ++k) sh[wave][k] = acc[k];
    __syncthreads();
    if (tid == 0) {
      double tot[TPART_N];
      for (int k = 0; k < TPART_N; ++k) tot[k] = sh[0][k] + sh[1][k] + sh[2][k] + sh[3][k];
      double o[SYSOUT_N] = {0.0};
      o[0] = tot[0]; o[1] = tot[1]; o[2] = tot[2]; o[3] = tot[3];
      o[4] = tot[0] + tot[1] + tot[2] + tot[3];
      o[5] = tot[4];
      o[6] = tot[5];
      const double inv = 1.0 / (double)S.n;
      const double cx = tot[6] * inv, cy = tot[7] * inv, cz = tot[8] * inv;
      o[7] = tot[9] * inv - (cx * cx + cy * cy + cz * cz);
      o[8] = tot[6]; o[9] = tot[7]; o[10] = tot[8];
      o[11] = (double)S.n;
      double *d = p.sysout + (int64_t)(s - p.sysout_base) * SYSOUT_N;
      for (int k = 0; k < 12; ++k) {
        d[k] = o[k];
        if (out) out[(slot >= 0 ? 0 : q) * SYSOUT_N + k] = o[k];
      }
    }
    __syncthreads();
  }
}

// ---- the host's end of a call
//
// A call's tables come from one pinned host buffer and its results go to
// another, both read and written by kernels in stream order: a call is its
// launches and one wait for the stream (7 synchronous copies of tables and 2
// of results, 15 us each, were 120 us of every call).

// Tables of a batch from the pinned staging buffer to their device arrays.
__global__ __launch_bounds__(256) void k_tables(TableParts tp) {
  const int k = blockIdx.y;
  const uint32_t *src = tp.stage + tp.part[k].src;
  uint32_t *dst = tp.part[k].dst;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < tp.part[k].words; i += gridDim.x * 256) dst[i] = src[i];
}

// A system's state, for the host.
__device__ __forceinline__ void report(const DevPtrs &p, int s, const SysDev &S) {
  p.rep[s] = make_int4(S.err, S.row_max, S.step >= S.step_end ? 1 : 0, 0);
}
__global__ void k_report(DevPtrs p) {
  const int nsys = *p.nsys;
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < nsys; q += gridDim.x * blockDim.x)
    report(p, p.syslist[q], p.sys[p.syslist[q]]);
}

// A new system unpacked from its upload: every array of its ranges in one
// launch (21 copies of host-made arrays, half of them zeros, took 300 us a
// system, half a served job's admission).
__global__ __launch_bounds__(256) void k_add_system(DevPtrs p, AddSystem a) {
  const int id = blockIdx.x * 256 + threadIdx.x, stride = gridDim.x * 256;
  const float *xyz = reinterpret_cast<const float *>(a.blob + a.xyz), *bond = reinterpret_cast<const float *>(a.blob + a.bond);
  const float *vel = reinterpret_cast<const float *>(a.blob + a.vel);
  const int *wb = reinterpret_cast<const int *>(a.blob + a.wbits), *ns = reinterpret_cast<const int *>(a.blob + a.nstart);
  for (int k = id; k < a.bead_len; k += stride) {
    const int i = a.bead_off + k;
    const bool in = k < a.n;
    const float4 x = in ? make_float4(xyz[3 * k], xyz[3 * k + 1], xyz[3 * k + 2], __int_as_float(wb[k]))
                        : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    p.pos0[i] = x;
    p.pos1[i] = x;
    p.bond_r0[i] = in ? bond[k] : 0.0f;
    p.nat_start[i] = a.nat_off + (in ? ns[k] : 0);
    p.nat_cnt[i] = in ? ns[k + 1] - ns[k] : 0;
    p.nlatt_cnt[i] = p.platt_cnt[i] = p.nlrep_cnt[i] = p.plrep_cnt[i] = p.plrep_off[i] = p.platt_off[i] = 0;
    // underdamped state: the velocities entering the first step (w = 0)
    p.vel[i] = in && a.has_vel ? make_float4(vel[3 * k], vel[3 * k + 1], vel[3 * k + 2], 0.0f)
                               : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    p.tile_ord[i] = (uint8_t)(k % TILE);  // identity bead order until the first pair list orders it
    if (k % TILE == 0) p.tile_sys[i / TILE] = a.slot;
  }
  const int *nj = reinterpret_cast<const int *>(a.blob + a.natj);
  const float *nr = reinterpret_cast<const float *>(a.blob + a.natr);
  for (int k = id; k < a.n_nat; k += stride) {
    p.nat_j[a.nat_off + k] = a.bead_off + nj[k];
    p.nat_r0[a.nat_off + k] = nr[k];
  }
  uint32_t *d = reinterpret_cast<uint32_t *>(p.sys + a.slot);
  for (int k = id; k < (int)(sizeof(SysDev) / 4); k += stride) d[k] = a.blob[a.sys + k];
}

// Per-bead values of one system to the host buffer: the current coordinates or
// the forces, three floats a bead, or the underdamped state, four; step: the
// system's completed steps (when not null).
__global__ __launch_bounds__(256) void k_read(DevPtrs p, int slot, int what, float *out, int64_t *step) {
  const SysDev &S = p.sys[slot];
  const float4 *src = what == READ_COORDS ? buf_in(p, S.parity) : (what == READ_FORCES ? p.fout : p.vel);
  const float *f = reinterpret_cast<const float *>(src + S.bead_off);
  const int w = what == READ_VEL ? 4 : 3, m = S.n * w;
  for (int k = blockIdx.x * 256 + threadIdx.x; k < m; k += gridDim.x * 256) out[k] = f[4 * (k / w) + k % w];
  if (step && blockIdx.x == 0 && threadIdx.x == 0) *step = S.step;
}

// Half lists for the host (pairs i < j, by bead and row order): 16 lanes per
// bead count the entries above the bead, one block turns the counts into
// places, and the pairs of a window of the list are written to pinned memory.
// Bound by the calls' round trips.  The two pair lists of 1,500 beads, each
// asked for its length and then fetched: 105 us, against 720 with the row
// segments copied to the host and walked there (all four lists 470 and 4,100).
struct ListRow {
  int64_t at;   // first entry
  int cnt;
};
__device__ __forceinline__ ListRow list_row(const DevPtrs &p, const SysDev &S, int which, int i) {
  if (which == LIST_NL_ATT) return ListRow{p.nat_start[i], p.nlatt_cnt[i]};
  if (which == LIST_PL_ATT) return ListRow{p.platt_off[i], p.platt_cnt[i]};
  if (which == LIST_NL_REP) return ListRow{S.nl_base + (int64_t)(i - S.bead_off) * S.nl_cap, p.nlrep_cnt[i]};
  return ListRow{p.plrep_off[i], p.plrep_cnt[i]};
}
__device__ __forceinline__ int list_entry(const DevPtrs &p, const SysDev &S, int which, int64_t k) {
  if (which == LIST_NL_ATT) return p.nlatt_j[k];
  if (which == LIST_PL_ATT) return p.platt[k].x;
  if (which == LIST_NL_REP) return p.nlrep_j[k];
  return S.idx16 ? S.bead_off + reinterpret_cast<const uint16_t *>(p.plrep_j + S.pl_base)[k] : p.plrep_j[S.pl_base + k];
}

__global__ __launch_bounds__(256) void k_list_count(DevPtrs p, int slot, int which) {
  const SysDev &S = p.sys[slot];
  const int bo = S.bead_off, n = S.n, l = threadIdx.x & 15;
  for (int b = blockIdx.x * 16 + (threadIdx.x >> 4); b < n; b += gridDim.x * 16) {
    const ListRow r = list_row(p, S, which, bo + b);
    int c = 0;
    for (int k = l; k < r.cnt; k += 16) c += list_entry(p, S, which, r.at + k) > bo + b;
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) c += __shfl_xor(c, o);
    if (l == 0) p.cell_tmp[bo + b] = c;
  }
}

__global__ __launch_bounds__(1024) void k_list_places(DevPtrs p, int slot, int64_t lo, int64_t *total) {
  __shared__ int wsum[16];
  const SysDev &S = p.sys[slot];
  const int bo = S.bead_off, n = S.n, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int64_t carry = 0;
  for (int b0 = 0; b0 < n; b0 += 1024) {
    const int v = b0 + tid < n ? p.cell_tmp[bo + b0 + tid] : 0;
    const int incl = wave_incl_scan(v);
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int off = 0, tot = 0;
    for (int w = 0; w < 16; ++w) {
      off += w < wave ? wsum[w] : 0;
      tot += wsum[w];
    }
    // relative to the window, and held to 30 bits: far outside is outside
    const int64_t at = carry + off + incl - v - lo;
    if (b0 + tid < n) p.cell_tmp[bo + b0 + tid] = (int)min(max(at, -((int64_t)1 << 30)), (int64_t)1 << 30);
    carry += tot;
    __syncthreads();
  }
  if (tid == 0) *total = carry;
}

__global__ __launch_bounds__(256) void k_list_write(DevPtrs p, int slot, int which, int2 *out, int m) {
  const SysDev &S = p.sys[slot];
  const int bo = S.bead_off, n = S.n, l = threadIdx.x & 15;
  const int shift = threadIdx.x & 48;  // the group's first lane of its wave
  for (int b = blockIdx.x * 16 + (threadIdx.x >> 4); b < n; b += gridDim.x * 16) {
    const ListRow r = list_row(p, S, which, bo + b);
    int at = p.cell_tmp[bo + b];
    for (int k0 = 0; k0 < r.cnt; k0 += 16) {
      const int j = k0 + l < r.cnt ? list_entry(p, S, which, r.at + k0 + l) - bo : -1;
      const uint32_t bits = (uint32_t)(__ballot(j > b) >> shift) & 0xFFFFu;
      const int o = at + __popc(bits & ((1u << l) - 1u));
      if (j > b && o >= 0 && o < m) out[o] = make_int2(b, j);
      at += __popc(bits);
    }
  }
}

// New coordinates of one system from the host buffer (type and chain stay),
// and its error bits cleared.
__global__ __launch_bounds__(256) void k_write_coords(DevPtrs p, int slot, const float *in) {
  SysDev &S = p.sys[slot];
  float4 *x = const_cast<float4 *>(buf_in(p, S.parity)) + S.bead_off;
  const int n = S.n;
  for (int b = blockIdx.x * 256 + threadIdx.x; b < n; b += gridDim.x * 256) {
    const float4 o = x[b];
    x[b] = make_float4(in[3 * b], in[3 * b + 1], in[3 * b + 2], o.w);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) S.err = 0;
}

// Per system: open a run of nsteps (the step kernel moves a system while
// step < step_end).
__global__ void k_begin(DevPtrs p, int64_t nsteps) {
  const int nsys = *p.nsys;
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < nsys; q += gridDim.x * blockDim.x) {
    SysDev &S = p.sys[p.syslist[q]];
    S.step_end = S.step + nsteps;
  }
}

// One system's shell rows and packed pair-list rows moved to a segment of
// another row capacity (wave per tile): each row keeps its entries and its
// place in the tile's order, so the lists, and every result computed from
// them, are unchanged.  The two segments do not overlap.
template <typename T>
__device__ __forceinline__ void relayout_tile(const DevPtrs &p, int bo, int n, int t, int64_t ob, int oc, int64_t nb,
                                              int nc) {
  const int lane = threadIdx.x & 63;
  const T *so = reinterpret_cast<const T *>(p.slrep_j + ob);
  T *sn = reinterpret_cast<T *>(p.slrep_j + nb);
  const T *po = reinterpret_cast<const T *>(p.plrep_j + ob);
  T *pn = reinterpret_cast<T *>(p.plrep_j + nb);
  const int shift = t * TILE * (nc - oc);  // the tile's region moves with the capacity
  for (int q = 0; q < TILE; ++q) {
    const int li = t * TILE + q;
    if (li >= n) break;
    const int i = bo + li;
    const int cs = p.slrep_cnt[i];
    for (int k = lane; k < cs; k += 64) sn[(int64_t)li * nc + k] = so[(int64_t)li * oc + k];
    const int off = p.plrep_off[i];
    const int len = (p.plrep_cnt[i] + ROW_PAD - 1) & ~(ROW_PAD - 1);
    for (int k = lane; k < len; k += 64) pn[off + shift + k] = po[off + k];
    if (lane == 0) p.plrep_off[i] = off + shift;
  }
}

__global__ __launch_bounds__(64) void k_relayout(DevPtrs p, int bo, int n, int idx16, int64_t ob, int oc, int64_t nb,
                                                 int nc) {
  const int t = blockIdx.x;
  if (idx16) relayout_tile<uint16_t>(p, bo, n, t, ob, oc, nb, nc);
  else relayout_tile<uint32_t>(p, bo, n, t, ob, oc, nb, nc);
}

// Per system: advance the step counter after a block of kernel steps, and
// report to the host.
__global__ void k_advance(DevPtrs p, int nsteps) {
  const int nsys = *p.nsys;
  for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < nsys; q += gridDim.x * blockDim.x) {
    SysDev &S = p.sys[p.syslist[q]];
    const int64_t st = S.step + nsteps;
    S.step = st < S.step_end ? st : (S.step_end > S.step ? S.step_end : S.step);
    S.parity = (S.parity + nsteps) & 1;
    report(p, p.syslist[q], S);
  }
}

// ------------------------------------------------------------ self test
// Lane-layout checks of the DPP / swizzle helpers against shuffles, and of
// the device normal generator; run by the GPU tests before the engine.
__global__ void k_selftest(int *out, float *fout) {
  const int lane = threadIdx.x;
  const int v = (lane * 7 + 3) % 11;
  int ref = 0;
  for (int k = 0; k <= lane; ++k) ref += (k * 7 + 3) % 11;
  const int sc = wave_incl_scan(v);
  int bad = sc != ref;
  const float fv = (float)((lane * 5) % 13);
  float r4 = 0, r8 = 0, r16 = 0, r32 = 0, r64 = 0;
  for (int k = 0; k < 64; ++k) {
    const float x = (float)((k * 5) % 13);
    if (k / 4 == lane / 4) r4 += x;
    if (k / 8 == lane / 8) r8 += x;
    if (k / 16 == lane / 16) r16 += x;
    if (k / 32 == lane / 32) r32 += x;
    r64 += x;
  }
  bad |= (group_sum<4>(fv) != r4) << 1;
  bad |= (group_sum<8>(fv) != r8) << 2;
  bad |= (group_sum<16>(fv) != r16) << 3;
  bad |= (group_sum<32>(fv) != r32) << 4;
  bad |= (group_sum<64>(fv) != r64) << 5;
  const uint64_t m = __ballot(lane % 3 == 0);
  int below = 0;
  for (int k = 0; k < lane; ++k) below += (k % 3 == 0);
  bad |= (lanes_below(m) != below) << 6;
  out[lane] = bad;
  float n0, n1, n2;
  normals3(0x12345678u, 0x9abcdef0u, (uint32_t)lane, 1000 + lane, n0, n1, n2);
  fout[3 * lane] = n0;
  fout[3 * lane + 1] = n1;
  fout[3 * lane + 2] = n2;
}

// --------------------------------------------------------------- launchers

#define SOPK_LAUNCH_CHECK() hipGetLastError()

// Fork (the side stream waits for st) and join (st waits for the side
// stream).  Under graph capture these become two graph branches.
static hipError_t fork_begin(const StepFork *fk, hipStream_t st) {
  hipError_t h = hipEventRecord(fk->fork, st);
  if (h == hipSuccess) h = hipStreamWaitEvent(fk->side, fk->fork, 0);
  return h;
}

static hipError_t fork_end(const StepFork *fk, hipStream_t st) {
  hipError_t h = hipEventRecord(fk->join, fk->side);
  if (h == hipSuccess) h = hipStreamWaitEvent(st, fk->join, 0);
  return h;
}

// The shell filter's launches (LDS items, whole-CU items, global-gather
// items) on one stream, for the systems whose build is one of `builds`.
static void launch_filter(const DevPtrs &p, const StepGrids &sg, int kstep, int builds, hipStream_t st) {
  // row staging after the staged positions where LDS has room for it
  const bool stage0 = sg.lds + FILTER_STAGE_BYTES <= LDS_BYTES_MAX;
  if (sg.tiles > 0)
    hipLaunchKernelGGL(k_filter_tile, dim3(sg.tiles), dim3(FILTER_TILE_THREADS), 0, st, p, kstep, builds);
  if (sg.grid > 0)
    hipLaunchKernelGGL(k_shell_filter<true>, dim3(sg.grid), dim3(STEP_THREADS),
                       sg.lds + (stage0 ? FILTER_STAGE_BYTES : 0), st, p, kstep, 0, stage0 ? (int)sg.lds : -1,
                       stage0 ? FILTER_STAGE_BYTES : 0, builds);
  if (sg.grid_big > 0)
    hipLaunchKernelGGL(k_shell_filter<true>, dim3(sg.grid_big), dim3(STEP_THREADS), sg.lds_big, st, p, kstep, 1,
                       -1, 0, builds);
  // global-gather items stage no coordinates: room for 32-bit rows
  if (sg.grid_far > 0)
    hipLaunchKernelGGL(k_shell_filter<false>, dim3(sg.grid_far), dim3(STEP_THREADS), 2 * FILTER_STAGE_BYTES, st,
                       p, kstep, 0, 0, 2 * FILTER_STAGE_BYTES, builds);
}

// One list-rebuild point for the current batch: decision, cell grid and
// counting sort, the rows of grid and neighbor-list builds, then the filter.
// lg.split (and fk): the systems whose pair list comes from their shell rows
// need nothing from the cell grid, so their filter runs beside the grid chain,
// and the filter of the grid-built systems follows the chain on the second
// stream (the two filters take disjoint systems).  A batch whose filter does
// not fill the device gains nothing from that and pays for the fork and for
// the launches with nothing to do: it runs the whole rebuild in three launches
// on one stream.
hipError_t launch_lists(const DevPtrs &p, const ListGrids &lg, int kstep, int flags, hipStream_t st,
                        const StepFork *fk) {
  constexpr int ALL = (1 << BUILD_DIRECT) | (1 << BUILD_SHELL) | (1 << BUILD_NL);
  constexpr int SHELL_ONLY = 1 << BUILD_SHELL;
  const bool split = fk && lg.split;
  if (lg.grid_big > 0) {
    hipLaunchKernelGGL(k_big_skin, dim3(lg.grid_big, lg.grid_nbig), dim3(BIG_THREADS), 0, st, p, kstep, flags);
    hipLaunchKernelGGL(k_big_plan, dim3(lg.grid_nbig), dim3(1024), 0, st, p, kstep, flags);
  }
  hipStream_t cs = st;  // the grid chain's stream
  if (split) {
    if (lg.grid_sys > 0)
      hipLaunchKernelGGL(k_rebuild<PH_DECIDE>, dim3(lg.grid_sys), dim3(SORT_THREADS), 0, st, p, kstep, flags);
    const hipError_t h = fork_begin(fk, st);
    if (h != hipSuccess) return h;
    cs = fk->side;
    if (lg.grid_sys > 0)
      hipLaunchKernelGGL(k_rebuild<PH_GRID>, dim3(lg.grid_sys), dim3(SORT_THREADS), 0, cs, p, kstep, flags);
  } else if (lg.grid_sys > 0) {
    hipLaunchKernelGGL(k_rebuild<PH_DECIDE | PH_GRID>, dim3(lg.grid_sys), dim3(SORT_THREADS), 0, cs, p, kstep, flags);
  }
  if (lg.grid_big > 0) {
    hipLaunchKernelGGL(k_cell_count, dim3(4 * lg.grid_big, lg.grid_nbig), dim3(256), 0, cs, p, kstep);
    hipLaunchKernelGGL(k_cell_scan, dim3(lg.grid_nbig), dim3(1024), 0, cs, p);
    hipLaunchKernelGGL(k_cell_scatter, dim3(4 * lg.grid_big, lg.grid_nbig), dim3(256), 0, cs, p);
    hipLaunchKernelGGL(k_cell_rank, dim3(4 * lg.grid_big, lg.grid_nbig), dim3(256), 0, cs, p, kstep);
  }
  // the neighbor list asked for: a wave per bead
  const int grid_rows = flags == FORCE_NL || (flags & MATERIALIZE_NL) ? lg.grid_nl : lg.grid_tiles;
  hipLaunchKernelGGL(k_rows, dim3(grid_rows), dim3(256), 0, cs, p, kstep);
  if (split) {
    launch_filter(p, lg.fg, kstep, ALL & ~SHELL_ONLY, cs);
    launch_filter(p, lg.fg, kstep, SHELL_ONLY, st);
    const hipError_t h = fork_end(fk, st);
    if (h != hipSuccess) return h;
  } else {
    launch_filter(p, lg.fg, kstep, ALL, st);
  }
  return SOPK_LAUNCH_CHECK();
}

template <int MODE>
static void launch_step_lds(const DevPtrs &p, int lpb, int grid, size_t lds, int kstep, int tier, hipStream_t st) {
  const dim3 g(grid), b(STEP_THREADS);
  switch (lpb) {
    case 4: hipLaunchKernelGGL((k_step<4, MODE>), g, b, lds, st, p, kstep, tier); break;
    case 8: hipLaunchKernelGGL((k_step<8, MODE>), g, b, lds, st, p, kstep, tier); break;
    case 32: hipLaunchKernelGGL((k_step<32, MODE>), g, b, lds, st, p, kstep, tier); break;
    default: hipLaunchKernelGGL((k_step<16, MODE>), g, b, lds, st, p, kstep, tier); break;
  }
}

template <int MODE>
static void launch_step_mixed(const DevPtrs &p, int lpb, int grid, size_t lds, int kstep, hipStream_t st) {
  const dim3 g(grid), b(STEP_THREADS);
  switch (lpb) {
    case 4: hipLaunchKernelGGL((k_step_mixed<4, MODE>), g, b, lds, st, p, kstep); break;
    case 8: hipLaunchKernelGGL((k_step_mixed<8, MODE>), g, b, lds, st, p, kstep); break;
    case 32: hipLaunchKernelGGL((k_step_mixed<32, MODE>), g, b, lds, st, p, kstep); break;
    default: hipLaunchKernelGGL((k_step_mixed<16, MODE>), g, b, lds, st, p, kstep); break;
  }
}

template <int MODE>
static hipError_t launch_step_mode(const DevPtrs &p, int lpb, const StepGrids &sg, int kstep, hipStream_t st,
                                   const StepFork *fk) {
  if (sg.mixed) {
    launch_step_mixed<MODE>(p, lpb, sg.grid, sg.lds, kstep, st);
    return SOPK_LAUNCH_CHECK();
  }
  // the whole-CU and per-tile launches beside the two-blocks-per-unit one
  const bool fork = fk && sg.grid > 0 && (sg.grid_big > 0 || sg.grid_far > 0 || sg.tiles > 0);
  if (fork) {
    const hipError_t h = fork_begin(fk, st);
    if (h != hipSuccess) return h;
  }
  const hipStream_t far_st = fork ? fk->side : st;
  for (int tier = 0; tier < 2; ++tier) {
    const int grid = tier ? sg.grid_big : sg.grid;
    if (grid > 0) launch_step_lds<MODE>(p, lpb, grid, tier ? sg.lds_big : sg.lds, kstep, tier, tier ? far_st : st);
  }
  if (sg.grid_far > 0) {
    const dim3 g(sg.grid_far), b(STEP_THREADS);
    switch (lpb) {
      case 4: hipLaunchKernelGGL((k_step_far<4, MODE>), g, b, 0, far_st, p, kstep); break;
      case 8: hipLaunchKernelGGL((k_step_far<8, MODE>), g, b, 0, far_st, p, kstep); break;
      case 32: hipLaunchKernelGGL((k_step_far<32, MODE>), g, b, 0, far_st, p, kstep); break;
      default: hipLaunchKernelGGL((k_step_far<16, MODE>), g, b, 0, far_st, p, kstep); break;
    }
  }
  if (sg.tiles > 0) {
    const dim3 g(sg.tiles), b(64 * (tile_waves(lpb) + 1));
    switch (lpb) {
      case 4: hipLaunchKernelGGL(k_step_tile<4>, g, b, 0, far_st, p, kstep, MODE); break;
      case 8: hipLaunchKernelGGL(k_step_tile<8>, g, b, 0, far_st, p, kstep, MODE); break;
      case 32: hipLaunchKernelGGL(k_step_tile<32>, g, b, 0, far_st, p, kstep, MODE); break;
      default: hipLaunchKernelGGL(k_step_tile<16>, g, b, 0, far_st, p, kstep, MODE); break;
    }
  }
  hipError_t h = SOPK_LAUNCH_CHECK();
  if (fork && h == hipSuccess) h = fork_end(fk, st);
  return h;
}

hipError_t launch_step(const DevPtrs &p, int mode, int lpb, const StepGrids &sg, int kstep, hipStream_t st,
                       const StepFork *fk) {
  if (mode == MODE_FORCE) return launch_step_mode<MODE_FORCE>(p, lpb, sg, kstep, st, fk);
  if (mode == MODE_FORCE_NOISE) return launch_step_mode<MODE_FORCE_NOISE>(p, lpb, sg, kstep, st, fk);
  return launch_step_mode<MODE_STEP>(p, lpb, sg, kstep, st, fk);
}

// Allow the step kernels dynamic LDS up to `bytes`.
hipError_t step_lds_limit(size_t bytes) {
  hipError_t h = hipSuccess;
  auto allow = [&](auto *k) {
    if (h == hipSuccess)
      h = hipFuncSetAttribute(reinterpret_cast<const void *>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  };
#define SOPK_LDS_ATTR(L)                                                                            \
  allow(&k_step<L, MODE_STEP>), allow(&k_step<L, MODE_FORCE>), allow(&k_step<L, MODE_FORCE_NOISE>),   \
      allow(&k_step_mixed<L, MODE_STEP>), allow(&k_step_mixed<L, MODE_FORCE>),                        \
      allow(&k_step_mixed<L, MODE_FORCE_NOISE>);
  SOPK_LDS_ATTR(4) SOPK_LDS_ATTR(8) SOPK_LDS_ATTR(16) SOPK_LDS_ATTR(32)
#undef SOPK_LDS_ATTR
  return h;
}

// Allow the shell filter the dynamic LDS its launches take (a compute unit's
// whole LDS for the LDS items, row staging for the global-gather ones).
hipError_t filter_lds_init() {
  hipError_t h = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_shell_filter<true>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES_MAX);
  if (h == hipSuccess)
    h = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_shell_filter<false>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)(2 * FILTER_STAGE_BYTES));
  return h;
}

hipError_t launch_relayout(const DevPtrs &p, int bo, int n, int idx16, int64_t old_base, int old_cap,
                           int64_t new_base, int new_cap, hipStream_t st) {
  hipLaunchKernelGGL(k_relayout, dim3((n + TILE - 1) / TILE), dim3(64), 0, st, p, bo, n, idx16, old_base, old_cap,
                     new_base, new_cap);
  return SOPK_LAUNCH_CHECK();
}

hipError_t launch_energy(const DevPtrs &p, int grid_tiles, int grid_sys, double *out, hipStream_t st) {
  hipLaunchKernelGGL(k_energy, dim3(std::min(grid_tiles, 512)), dim3(ENERGY_THREADS), 0, st, p, 0, 0);
  hipLaunchKernelGGL(k_sys_reduce, dim3(grid_sys), dim3(256), 0, st, p, -1, out);
  return SOPK_LAUNCH_CHECK();
}

// One system (tiles t0 .. t0 + nt - 1, slot), without a work table.
hipError_t launch_energy_one(const DevPtrs &p, int t0, int nt, int slot, int grid_tiles, double *out, hipStream_t st) {
  hipLaunchKernelGGL(k_energy, dim3(grid_tiles), dim3(ENERGY_THREADS), 0, st, p, t0, nt);
  hipLaunchKernelGGL(k_sys_reduce, dim3(1), dim3(256), 0, st, p, slot, out);
  return SOPK_LAUNCH_CHECK();
}

hipError_t launch_tables(const TableParts &tp, hipStream_t st) {
  uint32_t most = 1;
  for (const TablePart &q : tp.part) most = std::max(most, q.words);
  hipLaunchKernelGGL(k_tables, dim3(std::min(64u, (most + 255) / 256), TABLE_PARTS), dim3(256), 0, st, tp);
  return SOPK_LAUNCH_CHECK();
}

hipError_t launch_add_system(const DevPtrs &p, const AddSystem &a, hipStream_t st) {
  const int m = std::max(a.bead_len, a.n_nat);
  hipLaunchKernelGGL(k_add_system, dim3(std::max(1, std::min(1024, (m + 255) / 256))), dim3(256), 0, st, p, a);
  return SOPK_LAUNCH_CHECK();
}

hipError_t launch_report(const DevPtrs &p, hipStream_t st) {
  hipLaunchKernelGGL(k_report, dim3(4), dim3(256), 0, st, p);
  return SOPK_LAUNCH_CHECK();
}

hipError_t launch_read(const DevPtrs &p, int slot, int n, int what, float *out, int64_t *step, hipStream_t st) {
  hipLaunchKernelGGL(k_read, dim3(std::max(1, std::min(512, (4 * n + 255) / 256))), dim3(256), 0, st, p, slot, what,
                     out, step);
  return SOPK_LAUNCH_CHECK();
}

hipError_t launch_list_places(const DevPtrs &p, int slot, int n, int which, int64_t lo, int64_t *total, hipStream_t st) {
  hipLaunchKernelGGL(k_list_count, dim3(std::min(4096, (n + 15) / 16)), dim3(256), 0, st, p, slot, which);
  hipLaunchKernelGGL(k_list_places, dim3(1), dim3(1024), 0, st, p, slot, lo, total);
  return SOPK_LAUNCH_CHECK();
}

hipError_t launch_list_write(const DevPtrs &p, int slot, int n, int which, int2 *out, int m, hipStream_t st) {
  hipLaunchKernelGGL(k_list_write, dim3(std::min(4096, (n + 15) / 16)), dim3(256), 0, st, p, slot, which, out, m);
  return SOPK_LAUNCH_CHECK();
}

hipError_t launch_write_coords(const DevPtrs &p, int slot, int n, const float *in, hipStream_t st) {
  hipLaunchKernelGGL(k_write_coords, dim3(std::max(1, std::min(512, (n + 255) / 256))), dim3(256), 0, st, p, slot, in);
  return SOPK_LAUNCH_CHECK();
}

hipError_t launch_advance(const DevPtrs &p, int nsteps, hipStream_t st) {
  hipLaunchKernelGGL(k_advance, dim3(4), dim3(256), 0, st, p, nsteps);
  return SOPK_LAUNCH_CHECK();
}

hipError_t launch_begin(const DevPtrs &p, int64_t nsteps, hipStream_t st) {
  hipLaunchKernelGGL(k_begin, dim3(4), dim3(256), 0, st, p, nsteps);
  return SOPK_LAUNCH_CHECK();
}

// ------------------------------------------ allocation-free energy entry point
//
// The energy partials and values of sop_energy_eval_noalloc live in this
// file-scope array instead of memory the library allocates.
// Host code never passes the array's name to a kernel or a copy (in host
// code it stands for no device address): the address of each device's copy
// comes from hipGetSymbolAddress, once per device, and only that address is
// used.  Every call on one device shares that device's copy: calls that
// overlap on one device race.
static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

namespace {
std::mutex g_scratch_mu;
std::map<int, void *> g_scratch_ptr;  // device ordinal -> address of its copy of scratch
}  // namespace

// The device address of `device`'s copy of scratch; the device must be current.
hipError_t noalloc_scratch(int device, void **ptr) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  auto it = g_scratch_ptr.find(device);
  if (it != g_scratch_ptr.end()) {
    *ptr = it->second;
    return hipSuccess;
  }
  void *p = nullptr;
  const hipError_t h = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (h != hipSuccess) return h;
  g_scratch_ptr[device] = p;
  *ptr = p;
  return hipSuccess;
}

hipError_t launch_selftest(int *out, float *fout, hipStream_t st) {
  hipLaunchKernelGGL(k_selftest, dim3(1), dim3(64), 0, st, out, fout);
  return SOPK_LAUNCH_CHECK();
}

} // namespace sopk
