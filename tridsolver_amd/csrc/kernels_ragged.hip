// kernels_ragged.hip - ragged batch: S independent systems of uneven lengths
// stored back to back (system s = rows offsets[s] .. offsets[s+1]-1 of a, b,
// c, d). No counterpart in the reference, whose API needs equal lengths; per
// system the result is the plain solve's.
//
// Plan (four tiny kernels, all stream-ordered and capturable):
//   reset     zero the class counters, the work counter and the error flag
//   classify  class(s) = log2 of the lanes a system needs, P = next_pow2(ceil(L/M));
//             counted per workgroup in LDS, one global atomic per class
//   prefix    per class: first list slot and first work item; items are
//             ordered longest class first (largest-first scheduling)
//   scatter   list[slot] = s, slots reserved per workgroup and class
// Solve: an item is W systems of one class, P lanes each, the Thomas-PCR hybrid of
// hybrid_core.hpp. By default each item is a 256-thread workgroup of its own
// (rg_solve_each): the hardware keeps as many resident as registers and LDS
// allow and starts the next as one ends. Forced or tuned shapes run it as a
// resident grid of T-thread workgroups, `per_cu` per CU, that stride through the
// items (rg_solve), in one launch or in two: systems needing more than T/2 lanes,
// then the rest in T/2-thread workgroups. The mixed-precision solves take items
// from an atomic counter. Systems longer than M*T set the error flag and are
// skipped.

#include <algorithm>
#include <atomic>

#include "../../include/tridsolver_hip.h"
#include "hybrid_core.hpp"
#include "mixed_core.hpp"
#include "trid_internal.h"

namespace trid {
namespace {

constexpr int RG_CLASSES = 11;  // P = 1, 2, 4, ..., 1024

struct RaggedPlan {
  int counts[RG_CLASSES];
  int cursor[RG_CLASSES];
  int64_t sys_prefix[RG_CLASSES + 1];
  int64_t item_prefix[RG_CLASSES + 1];  // in scheduling order (longest first)
  int work;       // next item of the long-system launch
  int work_short; // next item of the short-system launch
  int error;
  int total_items;
  int long_items;  // items [0, long_items) need more than Tshort lanes
};

__global__ void rg_reset(RaggedPlan *plan) {
  const int t = threadIdx.x;
  if (t < RG_CLASSES) {
    plan->counts[t] = 0;
    plan->cursor[t] = 0;
  }
  if (t == 0) {
    plan->work = 0;
    plan->work_short = 0;
    plan->long_items = 0;
    plan->error = 0;
    plan->total_items = 0;
  }
}

__device__ __forceinline__ int rg_class(int64_t L, int M, int Tmax) {
  if (L <= 0) return -1;
  const int64_t need = (L + M - 1) / M;
  if (need > Tmax) return -2;
  int c = 0;
  while ((int64_t(1) << c) < need) ++c;
  return c;
}

// Counting and scattering aggregate per workgroup in LDS first: one global
// atomic per class and workgroup instead of one per system (systems of one
// class would otherwise serialise on a single counter).
constexpr int RG_PLAN_BLOCK = 256;

__global__ __launch_bounds__(RG_PLAN_BLOCK) void rg_classify(const int64_t *__restrict__ off,
                                                             int64_t S, int M, int Tmax,
                                                             RaggedPlan *plan) {
  __shared__ int cnt[RG_CLASSES];
  const int t = threadIdx.x;
  if (t < RG_CLASSES) cnt[t] = 0;
  __syncthreads();
  const int64_t s = (int64_t)blockIdx.x * RG_PLAN_BLOCK + t;
  if (s < S) {
    const int c = rg_class(off[s + 1] - off[s], M, Tmax);
    if (c >= 0) atomicAdd(&cnt[c], 1);
    else if (c == -2) atomicOr(&plan->error, 1);
  }
  __syncthreads();
  if (t < RG_CLASSES && cnt[t] > 0) atomicAdd(&plan->counts[t], cnt[t]);
}

// Systems of class c in a work item: one where they need more than Tshort
// lanes, as many as fit Tshort lanes else.
__host__ __device__ __forceinline__ int rg_systems(int c, int Tshort) {
  return (1 << c) > Tshort ? 1 : Tshort >> c;
}

__global__ void rg_prefix(RaggedPlan *plan, int Tshort) {
  if (threadIdx.x != 0) return;
  int64_t sp = 0;
  for (int c = 0; c < RG_CLASSES; ++c) {
    plan->sys_prefix[c] = sp;
    sp += plan->counts[c];
  }
  plan->sys_prefix[RG_CLASSES] = sp;
  // item_prefix[k] for scheduling slot k = class RG_CLASSES-1-k
  int64_t ip = 0;
  int long_items = 0;
  for (int k = 0; k < RG_CLASSES; ++k) {
    const int c = RG_CLASSES - 1 - k;
    plan->item_prefix[k] = ip;
    const int W = rg_systems(c, Tshort);
    const int64_t items = (plan->counts[c] + W - 1) / W;
    ip += items;
    if ((1 << c) > Tshort) long_items += (int)items;
  }
  plan->item_prefix[RG_CLASSES] = ip;
  plan->total_items = (int)ip;
  plan->long_items = long_items;
}

__global__ __launch_bounds__(RG_PLAN_BLOCK) void rg_scatter(const int64_t *__restrict__ off,
                                                            int64_t S, int M, int Tmax,
                                                            RaggedPlan *plan,
                                                            int *__restrict__ list) {
  __shared__ int cnt[RG_CLASSES], first[RG_CLASSES];
  const int t = threadIdx.x;
  if (t < RG_CLASSES) cnt[t] = 0;
  __syncthreads();
  const int64_t s = (int64_t)blockIdx.x * RG_PLAN_BLOCK + t;
  int c = -1, pos = 0;
  if (s < S) {
    c = rg_class(off[s + 1] - off[s], M, Tmax);
    if (c >= 0) pos = atomicAdd(&cnt[c], 1);  // position among this block's class-c systems
  }
  __syncthreads();
  if (t < RG_CLASSES && cnt[t] > 0) first[t] = atomicAdd(&plan->cursor[t], cnt[t]);
  __syncthreads();
  if (c >= 0) list[plan->sys_prefix[c] + first[c] + pos] = (int)s;
}

// One lane's view of work item `item`: the class (P lanes per system, W
// systems), and the lane's system (offset, length) if it has one. The list
// and offset loads depend on each other, so the persistent loops below decode
// the next item while the current one is being solved.
struct RgMeta {
  int cls;
  bool active;
  int N;  // listed systems passed rg_class: N <= M * Tmax
  int64_t base;
};

// The plan's class prefixes, copied into LDS once per workgroup at the start
// of a solve launch (rg_prefix has written them before it): item decoding
// then reads them from LDS, with no chain of dependent global loads.
struct RgPlanView {
  int64_t sys_prefix[RG_CLASSES + 1];
  int64_t item_prefix[RG_CLASSES + 1];
};

// Call with every thread before the launch's first barrier.
__device__ __forceinline__ void rg_view_load(RgPlanView &v, const RaggedPlan *plan, int t) {
  if (t <= RG_CLASSES) {
    v.sys_prefix[t] = plan->sys_prefix[t];
    v.item_prefix[t] = plan->item_prefix[t];
  }
}

// Its first part: everything but the system's offset and length, with the list
// entry (0 where the lane has no system).
__device__ __forceinline__ RgMeta rg_entry(const RgPlanView &v, const int *__restrict__ list,
                                           int item, int t, int Tmax, int *sys) {
  RgMeta m;
  // scheduling slot k: the last one whose first item is <= item (the
  // prefixes do not decrease, so that is the count of k >= 1 whose first
  // item is <= item; independent LDS reads)
  int k = 0;
#pragma unroll
  for (int j = 1; j < RG_CLASSES; ++j) k += v.item_prefix[j] <= item ? 1 : 0;
  m.cls = RG_CLASSES - 1 - k;
  const int P = 1 << m.cls, W = max(1, Tmax >> m.cls);
  const int64_t first = v.sys_prefix[m.cls] + (int64_t)(item - v.item_prefix[k]) * W;
  const int64_t slot = first + t / P;
  m.active = slot < v.sys_prefix[m.cls + 1];
  *sys = m.active ? list[slot] : 0;
  m.base = 0;
  m.N = 0;
  return m;
}

// The second part, from the list entry.
__device__ __forceinline__ void rg_locate(RgMeta &m, const int64_t *__restrict__ off, int sys) {
  if (m.active) {
    m.base = off[sys];
    m.N = (int)(off[sys + 1] - m.base);
  }
}

__device__ __forceinline__ RgMeta rg_meta(const RgPlanView &v, const int *__restrict__ list,
                                          const int64_t *__restrict__ off, int item, int t,
                                          int Tmax) {
  int sys;
  RgMeta m = rg_entry(v, list, item, t, Tmax, &sys);
  rg_locate(m, off, sys);
  return m;
}

__device__ __forceinline__ hyb::Lane rg_lane(const RgMeta &m, int t, int Tmax) {
  hyb::Lane L;
  L.P = 1 << m.cls;
  L.W = Tmax >> m.cls;
  L.T = Tmax;
  L.t = t;
  L.p = t % L.P;
  L.w = t / L.P;
  L.pstep = 1;
  L.stride = 1;
  L.active = m.active;
  L.base = m.base;
  L.N = m.N;
  L.i0 = 0;
  L.i1 = 0;
  return L;
}

// Threads per workgroup: 1024 for the M = 4/8 variants, 512 for M = 16 (FP64
// M = 16 needs that register budget; FP32 M = 16 at 1024 threads would spill,
// and 512 threads of 16 rows cover the same 8192 rows with half the lanes).
template <typename REAL, int M>
struct RgBounds {
  static constexpr int threads = M >= 16 ? 512 : 1024;
};

// Threads of rg_solve_each's workgroups (per_cu 0).
constexpr int RG_SMALL_T = 256;

// One work item of rg_solve: W systems of one class, P lanes each, in T
// threads (hyb::wave_solve). issued() runs once the loads are issued, loaded()
// once they have arrived: the caller decodes its next item in the two.
template <typename REAL, int M, bool INC, int T, typename OnIssued, typename OnLoaded>
__device__ __forceinline__ void rg_item(const RgMeta &cur, unsigned char *smem_raw,
                                        const REAL *__restrict__ a, const REAL *__restrict__ b,
                                        const REAL *__restrict__ c, const REAL *d, REAL *u,
                                        OnIssued issued, OnLoaded loaded) {
  const int t = threadIdx.x;
  const hyb::Lane L = rg_lane(cur, t, T);
  REAL *tile = reinterpret_cast<REAL *>(smem_raw);
  hyb::Ring ring{smem_raw + sizeof(REAL) * (size_t)T * (M + 1), (int)(3 * sizeof(REAL) * T), 0};
  if (cur.cls >= 6)
    hyb::wave_solve<REAL, M, INC, true>(L, tile, ring, a, b, c, d, u, issued, loaded);
  else
    hyb::wave_solve<REAL, M, INC, false>(L, tile, ring, a, b, c, d, u, issued, loaded);
}

// Waves per SIMD that the registers are held to: FP32 at 16 rows per lane needs
// 134 without a bound, which would leave three waves.
template <typename REAL, int M>
constexpr int rg_waves() {
  return sizeof(REAL) == 4 && M == 16 ? 4 : M == 16 ? 2 : 4;
}

// Workgroup k takes items k, k + grid, ... of its range, largest systems first.
// `body(cur, issued, loaded)` solves one item; the next one's list entry is
// loaded once the item's loads are issued, its offset and length once they have
// arrived.
template <typename Entry, typename Body>
__device__ __forceinline__ void rg_items(int lo, int total, const int64_t *__restrict__ off,
                                         Entry entry, Body body) {
  int item = lo + (int)blockIdx.x, sys = 0;
  if (item >= total) return;
  RgMeta cur = entry(item, &sys);
  rg_locate(cur, off, sys);
  for (;;) {
    const int nxt = item + (int)gridDim.x;
    RgMeta next{};
    body(
        item, cur, [&] { if (nxt < total) next = entry(nxt, &sys); },
        [&] { if (nxt < total) rg_locate(next, off, sys); });
    if (nxt >= total) return;
    item = nxt;
    cur = next;
    hyb::lds_barrier();  // the next item's LDS use starts after this one's
  }
}

// A resident grid over a range of items: LONG = the items whose systems
// need more than Tshort lanes (workgroups of T = Tmax threads, one per CU),
// else the rest (T = Tshort, two workgroups per CU, so that one loads while
// the other computes). A single launch plans with Tshort = Tmax: no item is
// long, and the LONG = false launch at T = Tmax takes them all.
template <typename REAL, int M, bool INC, int T, bool LONG>
__global__ __launch_bounds__(T, (rg_waves<REAL, M>())) void rg_solve(
    const REAL *__restrict__ a, const REAL *__restrict__ b, const REAL *__restrict__ c,
    const REAL *d, REAL *u, const int64_t *__restrict__ off, const int *__restrict__ list,
    const RaggedPlan *plan) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ RgPlanView s_view;
  const int t = threadIdx.x;
  const int lo = LONG ? 0 : plan->long_items;
  const int total = LONG ? plan->long_items : plan->total_items;
  if (lo + (int)blockIdx.x >= total) return;
  rg_view_load(s_view, plan, t);
  __syncthreads();
  rg_items(
      lo, total, off,
      [&](int item, int *sys) { return rg_entry(s_view, list, item, t, T, sys); },
      [&](int, const RgMeta &cur, auto issued, auto loaded) {
        rg_item<REAL, M, INC, T>(cur, smem_raw, a, b, c, d, u, issued, loaded);
      });
}

// Segments of RG_SMALL_T * M rows in the longest system that a shape's plan lists.
template <typename REAL, int M>
constexpr int rg_segments() {
  return RgBounds<REAL, M>::threads / RG_SMALL_T;
}
// LDS elements of rg_item_segments behind the tile: the equations of all segments
// but the last, and the first-row forms of the waves' first chunks.
template <typename REAL, int M>
constexpr int rg_segment_reals() {
  return 3 * RG_SMALL_T * (rg_segments<REAL, M>() - 1) + 3 * (RG_SMALL_T / 64) * rg_segments<REAL, M>();
}

// A system of more rows than RG_SMALL_T lanes of M hold, in one such workgroup:
// what is left over where the shape was chosen for a max_len that the caller
// understated. Its segments of T * M rows are swept one after the other (lane t of
// segment j has chunk j * T + t), the reduced system of all their chunks is solved
// by PCR in LDS, and the segments are read and swept again for x. Bound by the two
// readings: 9765 systems of 4096 rows, FP64, 0.50 ms where max_len says 2048, 0.29
// where it says 4096 (2.16 with every lane's rows read straight from memory, 0.41 in
// one 1024-thread workgroup per CU, which every other batch paid for).
template <typename REAL, int M, bool INC>
__device__ __forceinline__ void rg_item_segments(const RgMeta &cur, unsigned char *smem_raw,
                                                 const REAL *__restrict__ a,
                                                 const REAL *__restrict__ b,
                                                 const REAL *__restrict__ c, const REAL *d,
                                                 REAL *u) {
  constexpr int T = RG_SMALL_T, ROWS = T * M, Q = rg_segments<REAL, M>();
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));  // (what is formed from it is not held across the items)
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int N = __builtin_amdgcn_readfirstlane(cur.N), nseg = (N + ROWS - 1) / ROWS;
  const int64_t base = hyb::wave_uniform(cur.base);
  REAL *tile = reinterpret_cast<REAL *>(smem_raw), *eqs = tile + T * (M + 1);
  REAL *edge = eqs + 3 * T * (Q - 1);
  // the equations [A, C, D][T] of segment j; the last one's in the tile
  auto block = [&](int j) { return j == nseg - 1 ? tile : eqs + 3 * T * j; };
  hyb::Lane L{};
  L.P = T; L.W = 1; L.T = T; L.t = t; L.p = t; L.pstep = 1; L.stride = 1; L.active = true;

  REAL rb[M], rc[M], rd[M], e[3];
  auto sweep = [&](int j, REAL (&f)[3]) {
    REAL ra[M];
    L.t = t;
    asm volatile("" : "+v"(L.t));  // (nor are the loads' addresses across the segments)
    L.p = L.t;
    L.base = base + (int64_t)j * ROWS;
    L.N = N - j * ROWS;
    hyb::wave_rows<REAL, M, true>(L, tile, j == 0, a, b, c, d, ra, rb, rc, rd, [] {}, [] {});
    hyb::sweep_carry<REAL, M>([&](int r) { return ra[r]; }, rb, rc, rd, f[0], f[1], f[2]);
  };
  // a chunk's equation from its last row (al, ga, de) and the next chunk's first row
  // (f_d, f_a, f_g), as in hyb::reduced_solve
  auto close = [&](REAL nd, REAL na, REAL ng) {
    const REAL inv = REAL(1) / (REAL(1) - e[1] * na);
    e[2] = (e[2] - e[1] * nd) * inv;
    e[0] = e[0] * inv;
    e[1] = -e[1] * ng * inv;
  };
  auto put = [&](int j) {
#pragma unroll
    for (int k = 0; k < 3; ++k) block(j)[k * T + t] = e[k];
  };
  for (int j = 0; j < nseg; ++j) {
    REAL f[3], nx[3];
    sweep(j, f);
    e[0] = rb[M - 1]; e[1] = rc[M - 1]; e[2] = rd[M - 1];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if ((t & 63) == 0) edge[3 * (j * (T / 64) + wv) + k] = f[k];
      nx[k] = hyb::wave_read(f[k], (t & 63) + 1);
    }
    if ((t & 63) != 63) close(nx[0], nx[1], nx[2]);
    if (j < nseg - 1) put(j);
  }
  hyb::lds_barrier();  // the edges are there, the tile is free
  put(nseg - 1);
  if ((t & 63) == 63) {
    for (int j = 0; j < nseg; ++j) {
      const int w = j * (T / 64) + wv + 1;  // the next wave's first chunk
      const bool last = w == nseg * (T / 64);
#pragma unroll
      for (int k = 0; k < 3; ++k) e[k] = block(j)[k * T + t];
      close(last ? REAL(0) : edge[3 * w], last ? REAL(0) : edge[3 * w + 1],
            last ? REAL(0) : edge[3 * w + 2]);
      put(j);
    }
  }
  hyb::lds_barrier();
  for (int h = 1; h < nseg * T; h <<= 1) {
    REAL v[Q][3];
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      if (j >= nseg) break;
      const int lo = j * T + t - h, hi = j * T + t + h;
      const REAL *own = block(j) + t, *below = block(lo >= 0 ? lo / T : 0) + lo % T;
      const REAL *above = block(hi < nseg * T ? hi / T : 0) + hi % T;
      REAL m[3] = {}, q[3] = {};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        if (lo >= 0) m[k] = below[k * T];
        if (hi < nseg * T) q[k] = above[k * T];
      }
      const REAL A = own[0], C = own[T], D = own[2 * T];
      const REAL inv = REAL(1) / (REAL(1) - A * m[1] - C * q[0]);
      v[j][0] = -inv * A * m[0];
      v[j][1] = -inv * C * q[1];
      v[j][2] = inv * (D - A * m[2] - C * q[2]);
    }
    hyb::lds_barrier();
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      if (j >= nseg) break;
#pragma unroll
      for (int k = 0; k < 3; ++k) block(j)[k * T + t] = v[j][k];
    }
    hyb::lds_barrier();
  }
  // x of the lane's chunks' last rows and of those before them, out of the tile's way
  static_assert(2 * Q * T <= std::max(6 * T, rg_segment_reals<REAL, M>()), "LDS behind the tile");
  {
    REAL y[Q][2] = {};
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      if (j >= nseg) break;
      const int k = j * T + t - 1;
      y[j][0] = block(j)[2 * T + t];
      if (k >= 0) y[j][1] = block(k / T)[2 * T + k % T];
    }
    hyb::lds_barrier();
#pragma unroll
    for (int j = 0; j < Q; ++j) {
      if (j >= nseg) break;
      eqs[2 * T * j + t] = y[j][0];
      eqs[2 * T * j + T + t] = y[j][1];
    }
  }
  for (int j = 0; j < nseg; ++j) {
    REAL f[3];
    sweep(j, f);
    const REAL y = eqs[2 * T * j + t], ym = eqs[2 * T * j + T + t];
    hyb::substitute_back<REAL, M>(rb, rc, rd, y, ym);
    hyb::wave_put<REAL, M, INC, true>(L, tile, d, u, rd);
  }
}

// One launch of RG_SMALL_T-thread workgroups over every item, one each, planned with
// Tshort = RG_SMALL_T. The items [0, long_items), single systems that need more
// lanes, come first: LONG32 (M = 16: 4097-8192 rows) takes them by
// hyb::long32_solve, 32 rows per lane in 256 threads with `a` moved HBM->LDS in
// chunk order; otherwise there are none but misdeclared ones (rg_item_segments). Bound by
// HBM: with the plan's four launches (19 us), FP64, 40 M unknowns in systems of
// 4096 rows 291 us, of 2048 (M = 8) 286; lengths of 2049-4096 at random 153 us for
// 17.7 M unknowns, of 4097-8192 206 us for 23.6 M. What is left over the floor is
// idle lanes (a system fills its power of two of lanes to 3/4 on average; 40 M FP64
// unknowns in systems of 4096 / 3072 / 2064 rows, max_len 8192: 291 / 334 / 457 us)
// and the plan. One 512- or 1024-thread workgroup per CU that took items
// from an atomic counter: 412 and 406 us for the first two.
template <typename REAL, int M, bool LONG32>
constexpr size_t rg_each_lds_bytes() {
  if (LONG32) return hyb::long32_lds_bytes<REAL>();
  // the tile, and the ring or what rg_item_segments keeps
  return sizeof(REAL) * (size_t)RG_SMALL_T * (M + 1) +
         std::max(hyb::ring_bytes<REAL>(RG_SMALL_T, 3), sizeof(REAL) * (size_t)rg_segment_reals<REAL, M>());
}

template <typename REAL, int M, bool INC, bool LONG32>
__global__ __launch_bounds__(RG_SMALL_T, (LONG32 ? 2 : rg_waves<REAL, M>())) void rg_solve_each(
    const REAL *__restrict__ a, const REAL *__restrict__ b, const REAL *__restrict__ c,
    const REAL *d, REAL *u, const int64_t *__restrict__ off, const int *__restrict__ list,
    const RaggedPlan *plan) {
  static_assert(!LONG32 || (M == 16 && hyb::LONG32_T == RG_SMALL_T), "long32_solve's shape");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ RgPlanView s_view;
  const int t = threadIdx.x;
  const int nlong = plan->long_items, total = plan->total_items;
  if ((int)blockIdx.x >= total) return;
  rg_view_load(s_view, plan, t);
  __syncthreads();
  rg_items(
      0, total, off,
      [&](int i, int *sys) { return rg_entry(s_view, list, i, t, RG_SMALL_T, sys); },
      [&](int i, const RgMeta &cur, auto issued, auto loaded) {
        if (i >= nlong) {
          rg_item<REAL, M, INC, RG_SMALL_T>(cur, smem_raw, a, b, c, d, u, issued, loaded);
        } else if constexpr (LONG32) {
          hyb::long32_solve<REAL, INC, RG_SMALL_T>(hyb::wave_uniform(cur.base),
                                                   __builtin_amdgcn_readfirstlane(cur.N),
                                                   smem_raw, a, b, c, d, u, issued, loaded);
        } else {
          rg_item_segments<REAL, M, INC>(cur, smem_raw, a, b, c, d, u);
          issued();
          loaded();
        }
      });
}

// The four planning launches: work items of at most Tmax lanes.
void launch_plan(const int64_t *off, int64_t S, int M, int Tmax, int Tshort, void *ws,
                 hipStream_t st) {
  RaggedPlan *plan = static_cast<RaggedPlan *>(ws);
  int *list = reinterpret_cast<int *>(static_cast<unsigned char *>(ws) + RAGGED_PLAN_HEADER_BYTES);
  hipLaunchKernelGGL(rg_reset, dim3(1), dim3(64), 0, st, plan);
  const unsigned nb = (unsigned)((S + RG_PLAN_BLOCK - 1) / RG_PLAN_BLOCK);
  if (nb > 0) {
    hipLaunchKernelGGL(rg_classify, dim3(nb), dim3(RG_PLAN_BLOCK), 0, st, off, S, M, Tmax,
                       plan);
  }
  hipLaunchKernelGGL(rg_prefix, dim3(1), dim3(64), 0, st, plan, Tshort);
  if (nb > 0) {
    hipLaunchKernelGGL(rg_scatter, dim3(nb), dim3(RG_PLAN_BLOCK), 0, st, off, S, M, Tmax,
                       plan, list);
  }
}

// Workgroups of a launch that gives every item one of its own: there are at most
// S items, known only on the device, and workgroups past the last leave at once.
// Above this many, workgroups take several.
constexpr int64_t RG_GRID_MOST = 16384;

template <typename REAL, int M, bool INC, bool LONG32>
hipError_t launch_each(const REAL *a, const REAL *b, const REAL *c, REAL *d, REAL *u,
                       const int64_t *off, int64_t S, void *ws, hipStream_t st) {
  RaggedPlan *plan = static_cast<RaggedPlan *>(ws);
  int *list = reinterpret_cast<int *>(static_cast<unsigned char *>(ws) + RAGGED_PLAN_HEADER_BYTES);
  launch_plan(off, S, M, RgBounds<REAL, M>::threads, RG_SMALL_T, ws, st);
  auto kern = rg_solve_each<REAL, M, INC, LONG32>;
  static LdsGrant lds_granted;
  constexpr size_t lds = rg_each_lds_bytes<REAL, M, LONG32>();
  hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), lds, lds_granted);
  if (e != hipSuccess) return e;
  const unsigned blocks = (unsigned)std::min<int64_t>(std::max<int64_t>(S, 1), RG_GRID_MOST);
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(RG_SMALL_T), lds, st, a, b, c, d, INC ? u : d, off,
                     list, plan);
  return hipGetLastError();
}

// One rg_solve launch of `blocks` T-thread workgroups.
template <typename REAL, int M, bool INC, int T, bool LONG>
hipError_t launch_range(const REAL *a, const REAL *b, const REAL *c, REAL *d, REAL *u,
                        const int64_t *off, const int *list, const RaggedPlan *plan,
                        unsigned blocks, hipStream_t st) {
  const size_t lds = sizeof(REAL) * (size_t)T * (M + 1) + hyb::ring_bytes<REAL>(T, 3);
  auto kern = rg_solve<REAL, M, INC, T, LONG>;
  static LdsGrant lds_granted;
  hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), lds, lds_granted);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(T), lds, st, a, b, c, d, INC ? u : d, off, list,
                     plan);
  return hipGetLastError();
}

template <typename REAL, int M, bool INC>
hipError_t launch_m(const REAL *a, const REAL *b, const REAL *c, REAL *d, REAL *u,
                    const int64_t *off, int64_t S, int per_cu, int launches, void *ws,
                    hipStream_t st, int dev) {
  constexpr int Tmax = RgBounds<REAL, M>::threads;
  constexpr int Tshort = Tmax / 2;
  RaggedPlan *plan = static_cast<RaggedPlan *>(ws);
  int *list = reinterpret_cast<int *>(static_cast<unsigned char *>(ws) + RAGGED_PLAN_HEADER_BYTES);
  if (launches == 3 && M != 16) return hipErrorInvalidValue;
  if constexpr (M == 16) {  // the long systems at 32 rows per lane
    if (launches == 3) return launch_each<REAL, M, INC, true>(a, b, c, d, u, off, S, ws, st);
  }
  if (per_cu == 0) return launch_each<REAL, M, INC, false>(a, b, c, d, u, off, S, ws, st);
  int cus = 256;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const unsigned wgs = (unsigned)(cus * std::max(1, per_cu));
  if (launches == 1) {  // every item in one launch of Tmax-thread workgroups
    launch_plan(off, S, M, Tmax, Tmax, ws, st);
    return launch_range<REAL, M, INC, Tmax, false>(a, b, c, d, u, off, list, plan, wgs, st);
  }
  launch_plan(off, S, M, Tmax, Tshort, ws, st);
  if (launches == 2) {  // the long systems first (an empty range exits at once)
    const hipError_t e =
        launch_range<REAL, M, INC, Tmax, true>(a, b, c, d, u, off, list, plan, wgs, st);
    if (e != hipSuccess) return e;
  }
  return launch_range<REAL, M, INC, Tshort, false>(a, b, c, d, u, off, list, plan, 2 * wgs, st);
}

// FP64 systems by FP32 sweeps plus FP64 refinement (mixed_core.hpp): the
// same work queue, 512-thread workgroups (P <= 2^MIXED_MAX_STEPS lanes).
constexpr int RG_MIXED_THREADS = 512;

template <int M>
__global__ __launch_bounds__(RG_MIXED_THREADS) void rg_solve_mixed(
    const double *__restrict__ a, const double *__restrict__ b, const double *__restrict__ c,
    double *__restrict__ d, const int64_t *__restrict__ off, const int *__restrict__ list,
    RaggedPlan *plan, int refine) {
  constexpr int Tmax = RG_MIXED_THREADS;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ int s_next;
  __shared__ RgPlanView s_view;
  rg_view_load(s_view, plan, threadIdx.x);
  const int t = threadIdx.x;
  const int total = plan->total_items;
  if (t == 0) s_next = atomicAdd(&plan->work, 1);
  __syncthreads();
  int item = s_next;
  RgMeta cur = item < total ? rg_meta(s_view, list, off, item, t, Tmax) : RgMeta{};
  for (;;) {
    __syncthreads();  // every thread has read s_next
    if (item >= total) break;
    if (t == 0) s_next = atomicAdd(&plan->work, 1);
    const hyb::Lane L = rg_lane(cur, t, Tmax);
    double *tile = reinterpret_cast<double *>(smem_raw) + (size_t)L.w * L.P * (M + 1);
    hyb::Ring ring{smem_raw + sizeof(double) * (size_t)Tmax * (M + 1),
                   (int)(3 * sizeof(double) * Tmax), 0};
    double A[M], B[M], Cc[M], D[M];
    hyb::fetch_abcd<M, true>(L, a, b, c, d, A, B, Cc, D);
    hyb::to_chunk<M, true>(L, A, tile);
    const int nxt = s_next;
    const RgMeta next = nxt < total ? rg_meta(s_view, list, off, nxt, t, Tmax) : RgMeta{};
    hyb::to_chunk<M, true>(L, B, tile);
    hyb::to_chunk<M, true>(L, Cc, tile);
    hyb::to_chunk<M, true>(L, D, tile);
    double X[M];
    mixed_chunk<M>(L, ring, A, B, Cc, D, refine, X);
    hyb::to_fetch<M, true>(L, X, tile);
    hyb::store<M, true>(L, d, X);
    item = nxt;
    cur = next;
  }
}

// FP64 solution of FP32-stored systems (the arithmetic of kernels_mixed32.hip):
// FP32 a, b, c, d in, FP64 x out (d is not written); 16 rows per lane in
// 512 threads, so systems up to 8192 rows; ONE: at most one refinement. The
// LDS tile holds doubles for x's transpose; the FP32 operands go through its
// first half. AC_LDS keeps a and c in the tile (its two FP32 halves) for the
// solve, 32 registers a lane fewer: the general refinement loop needs that
// to fit the register file.
constexpr int RG_M32_M = 16;

// T threads, LONG as in rg_solve (the range of a two-launch split).
template <bool ONE, bool AC_LDS, int T, bool LONG>
__global__ __launch_bounds__(T) void rg_solve_mixed32(
    const float *__restrict__ a, const float *__restrict__ b, const float *__restrict__ c,
    const float *__restrict__ d, double *__restrict__ x, const int64_t *__restrict__ off,
    const int *__restrict__ list, RaggedPlan *plan, int refine) {
  constexpr int M = RG_M32_M, Tmax = T;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ int s_next;
  __shared__ RgPlanView s_view;
  rg_view_load(s_view, plan, threadIdx.x);
  const int t = threadIdx.x;
  int *counter = LONG ? &plan->work : &plan->work_short;
  const int lo = LONG ? 0 : plan->long_items;
  const int total = LONG ? plan->long_items : plan->total_items;
  if (t == 0) s_next = lo + atomicAdd(counter, 1);
  __syncthreads();
  int item = s_next;
  RgMeta cur = item < total ? rg_meta(s_view, list, off, item, t, Tmax) : RgMeta{};
  for (;;) {
    __syncthreads();  // every thread has read s_next
    if (item >= total) break;
    if (t == 0) s_next = lo + atomicAdd(counter, 1);
    const hyb::Lane L = rg_lane(cur, t, Tmax);
    double *dtile = reinterpret_cast<double *>(smem_raw) + (size_t)L.w * L.P * (M + 1);
    float *ftile = reinterpret_cast<float *>(dtile);
    hyb::Ring ring{smem_raw + sizeof(double) * (size_t)Tmax * (M + 1),
                   (int)(2 * sizeof(double) * Tmax), 0};
    float A[M], B[M], Cc[M], D[M];
    hyb::fetch_abcd<M, true>(L, a, b, c, d, A, B, Cc, D);
    hyb::to_chunk<M, true>(L, B, ftile);  // has barriers: s_next is visible below
    const int nxt = s_next;
    const RgMeta next = nxt < total ? rg_meta(s_view, list, off, nxt, t, Tmax) : RgMeta{};
    hyb::to_chunk<M, true>(L, D, ftile);
    double X[M];
    if constexpr (AC_LDS) {
      float *tC = ftile + L.P * (M + 1);
#pragma unroll
      for (int r = 0; r < M; ++r) {
        const int e = hyb::skew<M>(L.p + L.P * r);
        ftile[e] = A[r];
        tC[e] = Cc[r];
      }
      __syncthreads();
      const float *ca = ftile + L.p * (M + 1), *cc = tC + L.p * (M + 1);
      mixed_solve<M, MIXED_MAX_STEPS, ONE, false>(
          L, ring, [&](int r) { return ca[r]; }, B, [&](int r) { return cc[r]; }, D, refine, X);
      __syncthreads();  // a and c are read to the end before x overwrites the tile
    } else {
      hyb::to_chunk<M, true>(L, A, ftile);
      hyb::to_chunk<M, true>(L, Cc, ftile);
      mixed_solve<M, MIXED_MAX_STEPS, ONE, false>(
          L, ring, [&](int r) { return A[r]; }, B, [&](int r) { return Cc[r]; }, D, refine, X);
    }
    hyb::to_fetch<M, true>(L, X, dtile);
    hyb::store<M, true>(L, x, X);
    item = nxt;
    cur = next;
  }
}

template <bool ONE, bool AC_LDS, int T, bool LONG>
hipError_t launch_mixed32_range(const float *a, const float *b, const float *c, const float *d,
                                double *x, const int64_t *off, RaggedPlan *plan, int *list,
                                unsigned blocks, int refine, hipStream_t st) {
  const size_t lds = sizeof(double) * (size_t)T * (RG_M32_M + 1) + hyb::ring_bytes<double>(T, 2);
  auto kern = rg_solve_mixed32<ONE, AC_LDS, T, LONG>;
  static LdsGrant lds_granted;
  {
    hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), lds, lds_granted);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(T), lds, st, a, b, c, d, x, off, list, plan,
                     refine);
  return hipGetLastError();
}

// One launch of 512-thread workgroups, or two: the systems needing more than
// 256 lanes in 512-thread workgroups, then the rest in 256-thread ones, two
// per CU.
template <bool ONE, bool AC_LDS>
hipError_t launch_mixed32_one(const float *a, const float *b, const float *c, const float *d,
                              double *x, const int64_t *off, int64_t S, int per_cu,
                              int launches, int refine, void *ws, hipStream_t st, int dev) {
  constexpr int Tmax = RG_MIXED_THREADS, Tshort = Tmax / 2;
  RaggedPlan *plan = static_cast<RaggedPlan *>(ws);
  int *list = reinterpret_cast<int *>(static_cast<unsigned char *>(ws) + RAGGED_PLAN_HEADER_BYTES);
  int cus = 256;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const unsigned per = (unsigned)std::max(1, per_cu);
  if (launches == 1) {  // no long range: the LONG = false launch takes every item
    launch_plan(off, S, RG_M32_M, Tmax, Tmax, ws, st);
    return launch_mixed32_range<ONE, AC_LDS, Tmax, false>(a, b, c, d, x, off, plan, list,
                                                          cus * per, refine, st);
  }
  launch_plan(off, S, RG_M32_M, Tmax, Tshort, ws, st);
  hipError_t e = launch_mixed32_range<ONE, AC_LDS, Tmax, true>(a, b, c, d, x, off, plan, list,
                                                               cus * per, refine, st);
  if (e != hipSuccess) return e;
  return launch_mixed32_range<ONE, AC_LDS, Tshort, false>(a, b, c, d, x, off, plan, list,
                                                          2 * cus * per, refine, st);
}

template <int M>
hipError_t launch_mixed_m(const double *a, const double *b, const double *c, double *d,
                          const int64_t *off, int64_t S, int per_cu, int refine, void *ws,
                          hipStream_t st, int dev) {
  constexpr int Tmax = RG_MIXED_THREADS;
  RaggedPlan *plan = static_cast<RaggedPlan *>(ws);
  int *list = reinterpret_cast<int *>(static_cast<unsigned char *>(ws) + RAGGED_PLAN_HEADER_BYTES);
  launch_plan(off, S, M, Tmax, Tmax, ws, st);  // one launch: no long range
  const size_t lds =
      sizeof(double) * (size_t)Tmax * (M + 1) + hyb::ring_bytes<double>(Tmax, 3);
  auto kern = rg_solve_mixed<M>;
  static LdsGrant lds_granted;
  {
    hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), lds, lds_granted);
    if (e != hipSuccess) return e;
  }
  int cus = 256;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  hipLaunchKernelGGL(kern, dim3((unsigned)(cus * std::max(1, per_cu))), dim3(Tmax), lds, st,
                     a, b, c, d, off, list, plan, refine);
  return hipGetLastError();
}

// M = 16 with the FP64 a and c operands in LDS (mixed_contig_lds): 8192 rows
// in 512 threads. One launch of 512-thread workgroups, one per CU, or the
// FP64 solve's split: systems needing more than 256 lanes by that launch, the
// rest by 256-thread workgroups, two per CU (LDS 2 tiles x T*(M+1) doubles +
// 2 ring slots of 2 doubles per thread: 152 KiB at 512 threads, 76 KiB at
// 256).
constexpr int RG_MIXED_LDS_M = 16;

template <int T>
constexpr size_t rg_mixed_lds_bytes() {
  return 2 * sizeof(double) * (size_t)T * (RG_MIXED_LDS_M + 1) + hyb::ring_bytes<double>(T, 2);
}

// Two waves per SIMD in both shapes (the 256-thread workgroups run two per
// CU), i.e. at most 256 VGPRs.
template <int T, bool LONG>
__global__ __launch_bounds__(T, 2) void rg_solve_mixed_lds(
    const double *__restrict__ a, const double *__restrict__ b, const double *__restrict__ c,
    double *__restrict__ d, const int64_t *__restrict__ off, const int *__restrict__ list,
    RaggedPlan *plan, int refine) {
  constexpr int M = RG_MIXED_LDS_M;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  __shared__ int s_next;
  __shared__ RgPlanView s_view;
  // each thread's system offset of the current item, read again for the
  // stores: with the next item decoded during the solve, holding both in
  // registers across it would spill
  __shared__ int64_t s_base[T];
  rg_view_load(s_view, plan, threadIdx.x);
  const int t = threadIdx.x;
  int *counter = LONG ? &plan->work : &plan->work_short;
  const int lo = LONG ? 0 : plan->long_items;
  const int total = LONG ? plan->long_items : plan->total_items;
  if (t == 0) s_next = lo + atomicAdd(counter, 1);
  __syncthreads();
  int item = s_next;
  RgMeta cur = item < total ? rg_meta(s_view, list, off, item, t, T) : RgMeta{};
  double *tiles = reinterpret_cast<double *>(smem_raw);
  hyb::Ring ring{smem_raw + 2 * sizeof(double) * (size_t)T * (M + 1),
                 (int)(2 * sizeof(double) * T), 0};
  for (;;) {
    __syncthreads();  // every thread has read s_next
    if (item >= total) break;
    // claim the following item now; its id is read after the first transpose
    if (t == 0) s_next = lo + atomicAdd(counter, 1);
    s_base[t] = cur.base;
    const hyb::Lane L = rg_lane(cur, t, T);
    double *tA = tiles + (size_t)L.w * L.P * (M + 1);
    double *tC = tA + (size_t)T * (M + 1);
    int nxt = 0;
    RgMeta next{};
    // at most T lanes per system: log2(T) PCR steps
    mixed_contig_lds<M, T == 512 ? 9 : 8, false>(L, ring, a, b, c, d, tA, tC, refine, [&] {
      nxt = s_next;
      if (nxt < total) next = rg_meta(s_view, list, off, nxt, t, T);
    }, [&] { return s_base[t]; });
    item = nxt;
    cur = next;
  }
}

template <int T, bool LONG>
hipError_t launch_rg_mixed_lds(const double *a, const double *b, const double *c, double *d,
                               const int64_t *off, int *list, RaggedPlan *plan, unsigned blocks,
                               int refine, hipStream_t st) {
  auto kern = rg_solve_mixed_lds<T, LONG>;
  static LdsGrant lds_granted;
  hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), rg_mixed_lds_bytes<T>(),
                            lds_granted);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(T), rg_mixed_lds_bytes<T>(), st, a, b, c, d, off,
                     list, plan, refine);
  return hipGetLastError();
}

hipError_t launch_mixed_lds(const double *a, const double *b, const double *c, double *d,
                            const int64_t *off, int64_t S, int per_cu, int launches, int refine,
                            void *ws, hipStream_t st, int dev) {
  constexpr int Tmax = 512, Tshort = 256;
  RaggedPlan *plan = static_cast<RaggedPlan *>(ws);
  int *list = reinterpret_cast<int *>(static_cast<unsigned char *>(ws) + RAGGED_PLAN_HEADER_BYTES);
  int cus = 256;
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  const int per = std::max(1, per_cu);
  if (launches == 1) {  // no long range: the LONG = false launch takes every item
    launch_plan(off, S, RG_MIXED_LDS_M, Tmax, Tmax, ws, st);
    return launch_rg_mixed_lds<Tmax, false>(a, b, c, d, off, list, plan,
                                            (unsigned)(cus * per), refine, st);
  }
  launch_plan(off, S, RG_MIXED_LDS_M, Tmax, Tshort, ws, st);
  hipError_t e = launch_rg_mixed_lds<Tmax, true>(a, b, c, d, off, list, plan,
                                                 (unsigned)(cus * per), refine, st);
  if (e != hipSuccess) return e;
  return launch_rg_mixed_lds<Tshort, false>(a, b, c, d, off, list, plan,
                                            (unsigned)(2 * cus * per), refine, st);
}

}  // namespace

int ragged_mixed32_max_len() { return RG_M32_M * RG_MIXED_THREADS; }

hipError_t launch_ragged_mixed32(const float *a, const float *b, const float *c, const float *d,
                                 double *x, const int64_t *off, int64_t S, int per_cu,
                                 int launches, int refine, void *ws, hipStream_t st, int dev) {
  if (launches != 1 && launches != 2) return hipErrorInvalidValue;
  return refine <= 1 ? launch_mixed32_one<true, false>(a, b, c, d, x, off, S, per_cu, launches,
                                                       refine, ws, st, dev)
                     : launch_mixed32_one<false, true>(a, b, c, d, x, off, S, per_cu, launches,
                                                       refine, ws, st, dev);
}

int ragged_mixed_max_len(int M) {
  if (M == RG_MIXED_LDS_M) return M * 512;
  return (M == 4 || M == 8) ? M * RG_MIXED_THREADS : 0;
}

hipError_t launch_ragged_mixed(int M, const double *a, const double *b, const double *c,
                               double *d, const int64_t *off, int64_t S, int per_cu,
                               int launches, int refine, void *ws, hipStream_t st, int dev) {
  if (launches != 1 && launches != 2) return hipErrorInvalidValue;
  switch (M) {
    case 4: return launch_mixed_m<4>(a, b, c, d, off, S, per_cu, refine, ws, st, dev);
    case 8: return launch_mixed_m<8>(a, b, c, d, off, S, per_cu, refine, ws, st, dev);
    case RG_MIXED_LDS_M:
      return launch_mixed_lds(a, b, c, d, off, S, per_cu, launches, refine, ws, st, dev);
    default: return hipErrorInvalidValue;
  }
}

size_t ragged_workspace_bytes(int64_t S) {
  return RAGGED_PLAN_HEADER_BYTES + sizeof(int) * (size_t)std::max<int64_t>(S, 1);
}

int ragged_max_len(int fp64, int M) {
  (void)fp64;  // the same shapes at both precisions
  if (M != 4 && M != 8 && M != 16) return 0;
  return M * (M >= 16 ? 512 : 1024);
}

template <typename REAL, bool INC>
hipError_t launch_ragged(int M, const REAL *a, const REAL *b, const REAL *c, REAL *d, REAL *u,
                         const int64_t *off, int64_t S, int per_cu, int launches, void *ws,
                         hipStream_t st, int dev) {
  static_assert(sizeof(RaggedPlan) <= RAGGED_PLAN_HEADER_BYTES, "plan header");
  if (launches < 1 || launches > 3) return hipErrorInvalidValue;
  switch (M) {
    case 4: return launch_m<REAL, 4, INC>(a, b, c, d, u, off, S, per_cu, launches, ws, st, dev);
    case 8: return launch_m<REAL, 8, INC>(a, b, c, d, u, off, S, per_cu, launches, ws, st, dev);
    case 16:
      return launch_m<REAL, 16, INC>(a, b, c, d, u, off, S, per_cu, launches, ws, st, dev);
    default: return hipErrorInvalidValue;
  }
}

// Reads the plan's error flag (after the stream has completed).
hipError_t ragged_error_flag(void *ws, int *flag) {
  RaggedPlan *plan = static_cast<RaggedPlan *>(ws);
  return hipMemcpy(flag, &plan->error, sizeof(int), hipMemcpyDeviceToHost);
}

#define TRID_RG_INST(REAL, INC)                                                              \
  template hipError_t launch_ragged<REAL, INC>(int, const REAL *, const REAL *, const REAL *, \
                                               REAL *, REAL *, const int64_t *, int64_t, int, \
                                               int, void *, hipStream_t, int);
TRID_RG_INST(float, false)
TRID_RG_INST(float, true)
TRID_RG_INST(double, false)
TRID_RG_INST(double, true)

}  // namespace trid
