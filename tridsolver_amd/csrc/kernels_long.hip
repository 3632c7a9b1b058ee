// kernels_long.hip - batched solve of systems longer than one workgroup holds
// (contiguous: above 16384 rows; strided: above 2048 FP64 / 4096 FP32 rows),
// by the Thomas-PCR hybrid with its reduced system solved outside the
// workgroups.
//
// The hybrid (hybrid_core.hpp, kernels_solve.hip) cuts a system into chunks
// of M rows, reduces every chunk to one equation in its last unknown y_k
//     A_k y_{k-1} + y_k + C_k y_{k+1} = D_k,
// solves that reduced system by PCR inside the workgroup and substitutes back.
// A longer system does not fit one workgroup, so here:
//   1. long_reduce_kernel: workgroups take segments of SEG = P * M rows (P
//      lanes per system segment), sweep every chunk and write its reduced
//      equation; only the last chunk of a segment needs a value of another
//      workgroup (the next segment's first chunk), which
//   2. long_join_kernel completes, one thread per segment;
//   3. the reduced systems (ceil(N / M) rows each) are solved by the batched
//      hybrid itself -- or, when still too long, by this path again;
//   4. long_subst_kernel: the segments are read again, the sweep recomputed (the
//      same arithmetic, so the same values), and x written (or added to u).
// HBM traffic: a, b, c, d read twice (64 B per point at FP64), x written once,
// 4 reals per M rows of reduced equations: about 74 B per point
// against the one-workgroup hybrid's 40, and the reduced solve. It replaces
// the per-lane Thomas kernel, whose one recurrence per system leaves the GPU
// idle at a few thousand long systems.
// Both passes are bound by HBM: at 4096 x 4096 rows along y, FP64, reduce 111 us
// (4.8 TB/s), join 5, reduced solve 13, substitution 131 us (5.1 TB/s). With a forward
// and a backward sweep after all loads, six reals per chunk in a record of their own
// and 512-thread workgroups it was 119, 15 and 135 us; 777 x 6001 rows (misaligned) 156 us
// in all against 85, 1000 x 5000 FP32 84 against 42.
//
// Reduced equations live in the caller's workspace, laid out so
// that lanes write consecutive addresses: contiguous systems [system][chunk]
// (the reduced solve is contiguous), strided ones [chunk][system] (the
// reduced solve is strided, x-neighbouring systems adjacent).

#include <algorithm>
#include <atomic>

#include "hybrid_core.hpp"
#include "trid_internal.h"
#include "trid_tune.h"
#include "wide_core.hpp"

namespace trid {
namespace {

constexpr int LONG_M = 16;  // rows per lane

// Lanes per system segment and systems per workgroup: contiguous systems one
// system, 512 lanes (8192-row segments); strided ones 128-byte rows of
// x-neighbours, 256 threads (FP64: 256-row segments, three workgroups per CU).
template <typename REAL, bool CONTIG>
struct LongShape {
  static constexpr int W = CONTIG ? 1 : 128 / (int)sizeof(REAL);
  static constexpr int P = CONTIG ? 512 : 256 / W;
  static constexpr int T = W * P;
  static constexpr int64_t SEG = (int64_t)P * LONG_M;
};

// LDS: contiguous systems' transposes; the reduce kernel's exchange behind them.
template <typename REAL, bool CONTIG>
constexpr size_t long_tile_bytes() {
  using S = LongShape<REAL, CONTIG>;
  return CONTIG ? sizeof(REAL) * (size_t)S::T * (LONG_M + 1) : 0;
}
template <typename REAL, bool CONTIG>
constexpr size_t long_reduce_lds_bytes() {
  return long_tile_bytes<REAL, CONTIG>() + 3 * sizeof(REAL) * (size_t)LongShape<REAL, CONTIG>::T;
}

// The lane of segment `seg` of its system. Chunk k = seg * P + p of the system
// owns rows k*M .. k*M+M-1; L.base and L.N are relative to the segment, so
// the shared fetch order and masks apply inside it.
template <typename REAL, bool CONTIG>
__device__ __forceinline__ hyb::Lane long_lane(const Geom &g, int64_t nseg, int64_t *seg_out,
                                               int64_t *sys_out) {
  using S = LongShape<REAL, CONTIG>;
  hyb::Lane L;
  L.T = S::T;
  L.t = threadIdx.x;
  L.P = S::P;
  L.W = S::W;
  L.p = CONTIG ? L.t : L.t / S::W;
  L.w = CONTIG ? 0 : L.t % S::W;
  L.pstep = CONTIG ? 1 : S::W;
  const int64_t nb0 = (g.n0 + S::W - 1) / S::W;
  // contiguous systems: segment by segment in plain order; strided ones: the groups
  // of a row of segments in turn, dealt to the XCDs in 8 ranges, so that neighbouring
  // groups, which share lines where rows are misaligned, run on one XCD (300 x 20000
  // rows, FP64, 108 us against 131 with a group's segments in turn, 200 x 100000 338 against
  // 380, 1000 x 5000 81 against 94; 4096 x 4096 272 against 271)
  const int64_t ngrp = nb0 * g.n1;
  const int64_t bid = CONTIG ? blockIdx.x : hyb::xcd_remap(blockIdx.x, gridDim.x, 8);
  const int64_t seg = CONTIG ? bid % nseg : bid / ngrp;
  const int64_t grp = CONTIG ? bid / nseg : bid % ngrp;  // system group: (i0 block, i1)
  const int64_t i0 = (grp % nb0) * S::W + L.w;
  const int64_t i1 = grp / nb0;
  L.active = i0 < g.n0;
  L.i0 = i0;
  L.i1 = i1;
  L.stride = g.stride;
  L.base = i0 * g.st0 + i1 * g.st1 + seg * S::SEG * g.stride;
  const int64_t left = g.N - seg * S::SEG;
  L.N = left < S::SEG ? left : S::SEG;
  *seg_out = seg;
  *sys_out = i0 + g.n0 * i1;
  return L;
}

// Phases (i) and (ii) on the lane's chunk: on return (al, ga, de) of its rows in (rb,
// rc, rd) and the chunk's first unknown's form, as hyb::sweep_carry. a is 0 only at
// the system's first row and c only at its last; rows past N are identity rows.
// Strided systems: the loads are issued row by row, from rows and systems clamped
// into the array, and the sweep follows them; only a short last segment waits for all of
// them. NT: nontemporal loads (each pass reads the arrays once).
template <typename REAL, bool CONTIG, bool NT>
__device__ __forceinline__ void long_sweep(const Geom &g, const hyb::Lane &L, bool first_seg,
                                           bool last_seg, const REAL *a, const REAL *b,
                                           const REAL *c, const REAL *d, REAL *tile,
                                           REAL (&rb)[LONG_M], REAL (&rc)[LONG_M],
                                           REAL (&rd)[LONG_M], REAL &f_d, REAL &f_a, REAL &f_g) {
  constexpr int M = LONG_M;
  REAL ra[M];
  if constexpr (CONTIG) {
    hyb::fetch<M, CONTIG, NT>(L, a, ra, REAL(0), 0, first_seg ? 1 : 0, L.N);
    hyb::fetch<M, CONTIG, NT>(L, b, rb, REAL(1), 0, 0, L.N);
    hyb::fetch<M, CONTIG, NT>(L, c, rc, REAL(0), 0, 0, last_seg ? L.N - 1 : L.N);
    hyb::fetch<M, CONTIG, NT>(L, d, rd, REAL(0), 0, 0, L.N);
    hyb::to_chunk<M, CONTIG>(L, ra, tile);
    hyb::to_chunk<M, CONTIG>(L, rb, tile);
    hyb::to_chunk<M, CONTIG>(L, rc, tile);
    hyb::to_chunk<M, CONTIG>(L, rd, tile);
  } else {
    const int N = (int)L.N, row0 = L.p * M;
    const int64_t base = L.base - (L.active ? 0 : (L.i0 - (g.n0 - 1)) * g.st0);
    const bool whole = N == LongShape<REAL, CONTIG>::SEG;
#pragma unroll
    for (int r = 0; r < M; ++r) {
      const int row = row0 + r;
      const int64_t e = base + (int64_t)(row < N ? row : N - 1) * g.stride;
      ra[r] = hyb::ld<NT>(a + e);
      rb[r] = hyb::ld<NT>(b + e);
      rc[r] = hyb::ld<NT>(c + e);
      rd[r] = hyb::ld<NT>(d + e);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!whole) {  // the last segment
#pragma unroll
      for (int r = 0; r < M; ++r) {
        const int row = row0 + r;
        ra[r] = row < N ? ra[r] : REAL(0);
        rb[r] = row < N ? rb[r] : REAL(1);
        rc[r] = row + 1 < N ? rc[r] : REAL(0);
        rd[r] = row < N ? rd[r] : REAL(0);
      }
    }
    if (first_seg && L.p == 0) ra[0] = REAL(0);
  }
  hyb::sweep_carry<REAL, M>([&](int r) { return ra[r]; }, rb, rc, rd, f_d, f_a, f_g);
  // (c of the system's last row is not used; ga of the row is not read before this)
  if (!CONTIG && last_seg && L.p == L.P - 1) rc[M - 1] = REAL(0);
}

// Index of chunk k of system s in the reduced arrays.
template <bool CONTIG>
__device__ __forceinline__ int64_t long_idx(int64_t s, int64_t k, int64_t nsys, int64_t nchunk) {
  return CONTIG ? s * nchunk + k : k * nsys + s;
}

// The reduced equation of a chunk, normalised as in hyb::reduced_solve, from its last
// row's forward values and the next chunk's first row.
template <typename REAL>
__device__ __forceinline__ void long_equation(REAL al_e, REAL ga_e, REAL de_e, REAL nd, REAL na,
                                              REAL ng, REAL &A, REAL &Cc, REAL &D) {
  const REAL inv = REAL(1) / (REAL(1) - ga_e * na);
  A = al_e * inv;
  Cc = -ga_e * ng * inv;
  D = (de_e - ga_e * nd) * inv;
}

// A_k, 1, C_k, D_k of every chunk but the segments' last ones, whose next chunk is
// another workgroup's: those get (al, 1, ga, de), and the segments' first chunks'
// forms go to `edge` for long_join_kernel.
template <typename REAL, bool CONTIG, bool NT>
__global__ __launch_bounds__((LongShape<REAL, CONTIG>::T)) void long_reduce_kernel(
    Geom g, int64_t nseg, const REAL *__restrict__ a, const REAL *__restrict__ b,
    const REAL *__restrict__ c, const REAL *__restrict__ d, REAL *__restrict__ qa,
    REAL *__restrict__ qb, REAL *__restrict__ qc, REAL *__restrict__ qd,
    REAL *__restrict__ edge) {
  using S = LongShape<REAL, CONTIG>;
  constexpr int M = LONG_M;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int64_t seg, sys;
  const hyb::Lane L = long_lane<REAL, CONTIG>(g, nseg, &seg, &sys);
  REAL *tile = reinterpret_cast<REAL *>(smem_raw);
  REAL rb[M], rc[M], rd[M], f[3], n[3];
  long_sweep<REAL, CONTIG, NT>(g, L, seg == 0, seg == nseg - 1, a, b, c, d, tile, rb, rc, rd,
                               f[0], f[1], f[2]);
  hyb::Ring ring{smem_raw + long_tile_bytes<REAL, CONTIG>(), (int)(3 * sizeof(REAL) * S::T), 0, 1};
  hyb::from_above<3>(L, ring, false, f, n);
  REAL A = rb[M - 1], Cc = rc[M - 1], D = rd[M - 1];
  const bool open = L.p == L.P - 1;
  if (!open) long_equation(A, Cc, D, n[0], n[1], n[2], A, Cc, D);
  if (!L.active) return;
  const int64_t nsys = g.nsys(), nchunk = nseg * S::P;
  const int64_t i = long_idx<CONTIG>(sys, seg * S::P + L.p, nsys, nchunk);
  qa[i] = A;
  qb[i] = REAL(1);
  qc[i] = Cc;
  qd[i] = D;
  if (L.p == 0) {
    const int64_t E = nseg * nsys, e = seg * nsys + sys;
    edge[e] = f[0];
    edge[E + e] = f[1];
    edge[2 * E + e] = f[2];
  }
}

// The equations of the segments' last chunks, one thread each.
template <typename REAL, bool CONTIG>
__global__ __launch_bounds__(256) void long_join_kernel(int64_t nsys, int64_t nseg,
                                                        REAL *__restrict__ qa,
                                                        REAL *__restrict__ qc,
                                                        REAL *__restrict__ qd,
                                                        const REAL *__restrict__ edge) {
  using S = LongShape<REAL, CONTIG>;
  const int64_t E = nseg * nsys, e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= E) return;
  const int64_t seg = e / nsys, sys = e - seg * nsys;
  const int64_t i = long_idx<CONTIG>(sys, seg * S::P + S::P - 1, nsys, nseg * S::P);
  REAL nd = 0, na = 0, ng = 0;
  if (seg + 1 < nseg) {
    nd = edge[e + nsys];
    na = edge[E + e + nsys];
    ng = edge[2 * E + e + nsys];
  }
  REAL A, Cc, D;
  long_equation(qa[i], qc[i], qd[i], nd, na, ng, A, Cc, D);
  qa[i] = A;
  qc[i] = Cc;
  qd[i] = D;
}

template <typename REAL, bool CONTIG, bool INC, bool NT>
__global__ __launch_bounds__((LongShape<REAL, CONTIG>::T)) void long_subst_kernel(
    Geom g, int64_t nseg, const REAL *__restrict__ a, const REAL *__restrict__ b,
    const REAL *__restrict__ c, const REAL *d, REAL *u, const REAL *__restrict__ y) {
  using S = LongShape<REAL, CONTIG>;
  constexpr int M = LONG_M;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int64_t seg, sys;
  const hyb::Lane L = long_lane<REAL, CONTIG>(g, nseg, &seg, &sys);
  REAL *tile = reinterpret_cast<REAL *>(smem_raw);
  const int64_t nsys = g.nsys(), nchunk = nseg * S::P;
  const int64_t k = seg * S::P + L.p;
  REAL yk = 0, ym = 0;
  if (L.active) {
    yk = y[long_idx<CONTIG>(sys, k, nsys, nchunk)];
    if (k > 0) ym = y[long_idx<CONTIG>(sys, k - 1, nsys, nchunk)];
  }
  REAL rb[M], rc[M], rd[M], f_d, f_a, f_g;
  long_sweep<REAL, CONTIG, NT>(g, L, seg == 0, seg == nseg - 1, a, b, c, d, tile, rb, rc, rd,
                               f_d, f_a, f_g);
  hyb::substitute_back<REAL, M>(rb, rc, rd, yk, ym);
  hyb::to_fetch<M, CONTIG>(L, rd, tile);
  if (INC) hyb::store_add<M, CONTIG>(L, u, rd);
  else hyb::store<M, CONTIG, NT>(L, u, rd);  // u == d for a solve in place
}

template <typename REAL>
int64_t long_segments(const Geom &g) {
  const int64_t seg = g.stride == 1 ? LongShape<REAL, true>::SEG : LongShape<REAL, false>::SEG;
  return (g.N + seg - 1) / seg;
}
template <typename REAL>
int64_t long_chunks(const Geom &g) {
  return long_segments<REAL>(g) *
         (g.stride == 1 ? LongShape<REAL, true>::P : LongShape<REAL, false>::P);
}
// Workspace reals of one level: the four reduced arrays and the segments' edges
// (in whole 256-byte lines, so that the next level's arrays are as aligned).
template <typename REAL>
int64_t long_level_reals(const Geom &g) {
  return ((4 * long_chunks<REAL>(g) + 3 * long_segments<REAL>(g)) * g.nsys() + 63) / 64 * 64;
}

// Geometry of the reduced systems of g (nchunk rows per system).
Geom reduced_geom(const Geom &g, int64_t nchunk) {
  Geom r;
  const int64_t nsys = g.nsys();
  r.N = nchunk;
  if (g.stride == 1) {  // [system][chunk]
    r.stride = 1; r.n0 = nsys; r.n1 = 1; r.st0 = nchunk; r.st1 = nsys * nchunk;
  } else {              // [chunk][system]
    r.stride = nsys; r.n0 = nsys; r.n1 = 1; r.st0 = 1; r.st1 = nsys;
  }
  return r;
}

// The reduced equations of g's chunks: q = the four arrays and the edges.
template <typename REAL, bool CONTIG, bool NT>
hipError_t launch_long_reduce(const Geom &g, const REAL *a, const REAL *b, const REAL *c,
                              const REAL *d, REAL *q, hipStream_t st) {
  using S = LongShape<REAL, CONTIG>;
  const int64_t nseg = long_segments<REAL>(g), nsys = g.nsys(), R = nseg * S::P * nsys;
  const int64_t blocks = nseg * ((g.n0 + S::W - 1) / S::W) * g.n1;
  const int64_t jblocks = (nseg * nsys + 255) / 256;
  if (blocks > (int64_t)UINT32_MAX / S::T || jblocks > (int64_t)UINT32_MAX)
    return hipErrorInvalidValue;
  constexpr size_t lds = long_reduce_lds_bytes<REAL, CONTIG>();
  auto kern = long_reduce_kernel<REAL, CONTIG, NT>;
  static LdsGrant granted;
  hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), lds, granted);
  if (e != hipSuccess) return e;
  REAL *edge = q + 4 * R;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(S::T), lds, st, g, nseg, a, b, c, d, q,
                     q + R, q + 2 * R, q + 3 * R, edge);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL((long_join_kernel<REAL, CONTIG>), dim3((unsigned)jblocks), dim3(256), 0, st,
                     nsys, nseg, q, q + 2 * R, q + 3 * R, edge);
  return hipGetLastError();
}

template <typename REAL, bool CONTIG, bool INC, bool NT>
hipError_t launch_long_subst(const Geom &g, const REAL *a, const REAL *b, const REAL *c, REAL *d,
                             REAL *u, const REAL *y, hipStream_t st) {
  using S = LongShape<REAL, CONTIG>;
  const int64_t nseg = long_segments<REAL>(g);
  const int64_t blocks = nseg * ((g.n0 + S::W - 1) / S::W) * g.n1;
  constexpr size_t lds = long_tile_bytes<REAL, CONTIG>();
  auto kern = long_subst_kernel<REAL, CONTIG, INC, NT>;
  static LdsGrant granted;
  hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), lds, granted);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(S::T), lds, st, g, nseg, a, b, c, d,
                     u ? u : d, y);
  return hipGetLastError();
}

}  // namespace

template <typename REAL>
size_t long_workspace_bytes(const Geom &g) {
  size_t total = 0;
  Geom cur = g;
  // levels until the reduced systems fit one workgroup of the hybrid
  for (int level = 0; level < 8; ++level) {
    const int64_t nchunk = long_chunks<REAL>(cur);
    total += sizeof(REAL) * (size_t)long_level_reals<REAL>(cur);
    Geom r = reduced_geom(cur, nchunk);
    HybridCfg cfg;
    if (hybrid_default_cfg<REAL>(r, &cfg)) break;
    cur = r;
  }
  return total;
}

template <typename REAL, bool INC>
hipError_t launch_long(int dev, const Geom &g, const REAL *a, const REAL *b, const REAL *c,
                       REAL *d, REAL *u, void *ws, size_t ws_bytes, hipStream_t st) {
  const bool contig = g.stride == 1;
  // nontemporal where the rows of a strided batch are 128-byte aligned
  const bool nt =
      contig || wide::wide_rows_aligned<REAL>(
                    g, reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) |
                           reinterpret_cast<uintptr_t>(c) | reinterpret_cast<uintptr_t>(d) |
                           reinterpret_cast<uintptr_t>(u));
  const int64_t nchunk = long_chunks<REAL>(g);
  const int64_t R = nchunk * g.nsys(), level = long_level_reals<REAL>(g);
  if (ws_bytes < sizeof(REAL) * (size_t)level) return hipErrorInvalidValue;
  REAL *q = static_cast<REAL *>(ws);
  REAL *ra = q, *rb = q + R, *rc = q + 2 * R, *rd = q + 3 * R;
  hipError_t e = contig ? launch_long_reduce<REAL, true, true>(g, a, b, c, d, q, st)
                 : nt   ? launch_long_reduce<REAL, false, true>(g, a, b, c, d, q, st)
                        : launch_long_reduce<REAL, false, false>(g, a, b, c, d, q, st);
  if (e != hipSuccess) return e;
  // the reduced systems: the batched hybrid (tuned shape if one is cached),
  // or this path again with the rest of the workspace
  const Geom r = reduced_geom(g, nchunk);
  HybridCfg cfg;
  if (tuned_config<REAL, false>(dev, r, &cfg) || hybrid_default_cfg<REAL>(r, &cfg)) {
    e = for_each_grid_chunk(r, cfg.W, cfg.W * cfg.P, [&](const Geom &sub, int64_t o) {
      return launch_hybrid<REAL, false>(sub, cfg, ra + o, rb + o, rc + o, rd + o, nullptr, st);
    });
  } else {
    e = launch_long<REAL, false>(dev, r, ra, rb, rc, rd, nullptr, q + level,
                                 ws_bytes - sizeof(REAL) * (size_t)level, st);
  }
  if (e != hipSuccess) return e;
  return contig ? launch_long_subst<REAL, true, INC, true>(g, a, b, c, d, u, rd, st)
         : nt   ? launch_long_subst<REAL, false, INC, true>(g, a, b, c, d, u, rd, st)
                : launch_long_subst<REAL, false, INC, false>(g, a, b, c, d, u, rd, st);
}

#define TRID_LONG_INST(REAL)                                                                  \
  template size_t long_workspace_bytes<REAL>(const Geom &);                                  \
  template hipError_t launch_long<REAL, false>(int, const Geom &, const REAL *, const REAL *, \
                                               const REAL *, REAL *, REAL *, void *, size_t,  \
                                               hipStream_t);                                  \
  template hipError_t launch_long<REAL, true>(int, const Geom &, const REAL *, const REAL *,  \
                                              const REAL *, REAL *, REAL *, void *, size_t,   \
                                              hipStream_t);
TRID_LONG_INST(float)
TRID_LONG_INST(double)

}  // namespace trid
