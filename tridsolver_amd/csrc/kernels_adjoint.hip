// kernels_adjoint.hip - adjoint of the batched solve (no counterpart in the
// reference).
//
// For every system A x = d (A = tridiag(a, b, c), a[0] and c[N-1] unused) and
// an incoming gradient w = dL/dx, the adjoint solves
//     A^T lam = w,   A^T = tridiag(sub = c[n-1], diag = b[n], sup = a[n+1]),
// and forms
//     dL/dd = lam,  dL/da[n] = -lam[n] x[n-1] (0 at n = 0),
//     dL/db[n] = -lam[n] x[n],  dL/dc[n] = -lam[n] x[n+1] (0 at n = N-1),
// with x the forward solution. The transpose is solved by the same Thomas-PCR
// hybrid as the forward solve (hybrid_core.hpp): the shifted coefficients are
// fetched directly (row n of the transpose reads c at n-1 and a at n+1, so
// every element is still read once), and the neighbour chunks' boundary x
// values come through LDS. HBM traffic: read a, b, c, w, x; write lam and
// each requested gradient (72 B per point at FP64 with all three gradients).
// When no coefficient gradient is requested (GRAD false) x is not read: the
// solve for lam alone moves the forward solve's 40 B per point.
// Systems longer than adjoint_kernel holds take three steps instead: the
// transpose's off-diagonals written out (adj_transpose_kernel), A^T lam = w
// solved by the batched solve, which takes any length, and the gradients
// (adj_grad_kernel): about 128 B per point with all three gradients.

#include <algorithm>
#include <atomic>

#include "../../include/tridsolver_hip.h"
#include "hybrid_core.hpp"
#include "trid_internal.h"
#include "wide_core.hpp"

namespace trid {
namespace {

template <typename REAL, int M>
struct AdjBounds {
  static constexpr int threads = sizeof(REAL) * M >= 64 ? 512 : 1024;
};

template <typename REAL, int M, bool CONTIG, bool GRAD, bool NT>
__global__ __launch_bounds__((AdjBounds<REAL, M>::threads)) void adjoint_kernel(
    Geom g, int P, int W, int G, const REAL *__restrict__ a, const REAL *__restrict__ b,
    const REAL *__restrict__ c, const REAL *__restrict__ x, const REAL *__restrict__ w,
    REAL *__restrict__ lam, REAL *__restrict__ ga, REAL *__restrict__ gb,
    REAL *__restrict__ gc) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const hyb::Lane L = hyb::lane_of<CONTIG>(g, P, W, G);
  const size_t tile_bytes = CONTIG ? sizeof(REAL) * (size_t)W * P * (M + 1) : 0;
  REAL *tile = reinterpret_cast<REAL *>(smem_raw) + (size_t)L.w * P * (M + 1);
  hyb::Ring ring{smem_raw + tile_bytes, (int)(3 * sizeof(REAL) * L.T), 0};

  REAL ra[M], rb[M], rc[M], rd[M], rx[M];
  hyb::fetch<M, CONTIG, NT>(L, c, ra, REAL(0), -1, 0, L.N);  // sub of A^T: c[n-1]
  hyb::fetch<M, CONTIG, NT>(L, b, rb, REAL(1), 0, 0, L.N);
  hyb::fetch<M, CONTIG, NT>(L, a, rc, REAL(0), +1, 1, L.N);  // sup of A^T: a[n+1]
  hyb::fetch<M, CONTIG, NT>(L, w, rd, REAL(0), 0, 0, L.N);
  if (GRAD) hyb::fetch<M, CONTIG, NT>(L, x, rx, REAL(0), 0, 0, L.N);
  hyb::to_chunk<M, CONTIG>(L, ra, tile);
  hyb::to_chunk<M, CONTIG>(L, rb, tile);
  hyb::to_chunk<M, CONTIG>(L, rc, tile);
  hyb::to_chunk<M, CONTIG>(L, rd, tile);
  if (GRAD) hyb::to_chunk<M, CONTIG>(L, rx, tile);
  REAL l[M];
  hyb::solve_chunk<REAL, M, CONTIG>(L, ring, ra, rb, rc, rd, l);
  if (!GRAD) {
    hyb::to_fetch<M, CONTIG>(L, l, tile);
    hyb::store<M, CONTIG, NT>(L, lam, l);
    return;
  }

  // x of the neighbouring chunks' boundary rows
  REAL xprev = 0, xnext = 0;
  {
    REAL *q = ring.next<REAL>();
    q[L.t] = rx[0];
    q[L.T + L.t] = rx[M - 1];
    __syncthreads();
    if (L.p > 0) xprev = q[L.T + L.t - L.pstep];
    if (L.p + 1 < L.P) xnext = q[L.t + L.pstep];
  }
  const int64_t row0 = (int64_t)L.p * M;  // global row of chunk slot 0
  // Outputs go through the tile one at a time (contiguous systems).
  if (ga) {
    REAL v[M];
#pragma unroll
    for (int r = 0; r < M; ++r) {
      const REAL xl = r > 0 ? rx[r - 1] : xprev;
      v[r] = (row0 + r == 0) ? REAL(0) : -l[r] * xl;
    }
    hyb::to_fetch<M, CONTIG>(L, v, tile);
    hyb::store<M, CONTIG, NT>(L, ga, v);
  }
  if (gb) {
    REAL v[M];
#pragma unroll
    for (int r = 0; r < M; ++r) v[r] = -l[r] * rx[r];
    hyb::to_fetch<M, CONTIG>(L, v, tile);
    hyb::store<M, CONTIG, NT>(L, gb, v);
  }
  if (gc) {
    REAL v[M];
#pragma unroll
    for (int r = 0; r < M; ++r) {
      const REAL xr = r < M - 1 ? rx[r + 1] : xnext;
      v[r] = (row0 + r >= L.N - 1) ? REAL(0) : -l[r] * xr;
    }
    hyb::to_fetch<M, CONTIG>(L, v, tile);
    hyb::store<M, CONTIG, NT>(L, gc, v);
  }
  hyb::to_fetch<M, CONTIG>(L, l, tile);
  hyb::store<M, CONTIG, NT>(L, lam, l);
}

// The strided adjoint with the operand below the transpose's diagonal, c[n-1],
// staged in LDS and the sweep following the loads (wide_core.hpp; what bounds a
// strided solve and why this split: kernels_wide.hip). x's rows take c's place
// in the tile during the PCR, so that the gradients' operands arrive while
// nothing else is loaded and hold no registers; the rows next to the chunk's
// come in two registers. The four outputs are written one array after the other
// (256^3 FP64 y 231 against 237 us with all four row by row). Every output
// stream is as long as an input's: with all gradients, nine streams at 256^3
// FP64, y / z run at 5.3 / 5.0 TB/s, 227 / 241 us, against 234 / 262 with every
// operand in registers (adjoint_kernel); lam alone at 6.2 TB/s (z 108 us against 147).
template <typename REAL, int M, int SEG, bool GRAD, bool NT>
__global__ __launch_bounds__((wide::WideBounds<REAL, M>::threads)) void adjoint_wide_kernel(
    Geom g, int P, int G, int slots, const REAL *__restrict__ a, const REAL *__restrict__ b,
    const REAL *__restrict__ c, const REAL *__restrict__ x, const REAL *__restrict__ w,
    REAL *__restrict__ lam, REAL *__restrict__ ga, REAL *__restrict__ gb,
    REAL *__restrict__ gc) {
  constexpr int W = wide::WideShape<REAL, SEG>::W;
  constexpr int CH = 64 / W;  // chunks per wave
  constexpr int PITCH = wide::wide_chunk_bytes(M, SEG);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const hyb::Lane L = hyb::lane_of<false>(g, P, W, G);
  hyb::Ring ring{smem_raw + (size_t)P * PITCH, (int)(3 * sizeof(REAL) * L.T), 0, slots};
  const int lane = L.t & 63, wv = __builtin_amdgcn_readfirstlane(L.t >> 6);
  const int N = (int)L.N;
  const uint32_t tile = hyb::lds_address(smem_raw) + wv * CH * PITCH;
  const int64_t first = hyb::wave_uniform(L.i0 - L.w);
  const int64_t base0 = first + hyb::wave_uniform(L.i1) * g.st1, nsys = g.n0 - first;
  const uint32_t os = (uint32_t)(L.stride * (int64_t)sizeof(REAL));
  const int row0 = L.p * M;
  const int rows = L.active ? N - row0 : 0;
  const uint32_t ob = (uint32_t)(L.base + row0 * L.stride) * (uint32_t)sizeof(REAL);
  REAL *xs = reinterpret_cast<REAL *>(reinterpret_cast<char *>(smem_raw) + L.p * PITCH) + L.w;
  const bool whole = __all(rows >= M);
  REAL rb[M], rc[M], rd[M], f_d, f_a, f_g;
  if (whole)
    wide::wide_sweep<REAL, M, SEG, CH, true, NT, 1>(c + base0, tile, wv * CH * M, lane, N, nsys,
                                                    os, ob, row0, rows, xs, b, a, w, rb, rc, rd,
                                                    f_d, f_a, f_g);
  else
    wide::wide_sweep<REAL, M, SEG, CH, false, NT, 1>(c + base0, tile, wv * CH * M, lane, N, nsys,
                                                     os, ob, row0, rows, xs, b, a, w, rb, rc, rd,
                                                     f_d, f_a, f_g);
  REAL xprev = 0, xnext = 0;
  uint32_t obs = ob;
  asm volatile("" : "+v"(obs));  // offsets formed here, not held from the loads
  if (GRAD) {
    int ln = lane;
    asm volatile("" : "+v"(ln));
    if (whole)
      wide::wide_stage<REAL, M, SEG, CH, true>(x + base0, tile, wv * CH * M, ln, os, N, nsys);
    else
      wide::wide_stage<REAL, M, SEG, CH, false>(x + base0, tile, wv * CH * M, ln, os, N, nsys);
    const char *xb = reinterpret_cast<const char *>(x);
    if (row0 > 0 && rows > 0) xprev = *reinterpret_cast<const REAL *>(xb + (obs - os));
    if (rows > M) xnext = *reinterpret_cast<const REAL *>(xb + (obs + (uint32_t)M * os));
  }
  REAL y, ym;
  hyb::reduced_solve<REAL>(L, ring, rb[M - 1], rc[M - 1], rd[M - 1], f_d, f_a, f_g, y, ym);
  if (GRAD) {
    // every wave has its x rows before any wave stores (an output may be one
    // of the inputs)
    hyb::stage_wait_all();
    __syncthreads();
  }
  if (!L.active) return;
  hyb::substitute_back<REAL, M>(rb, rc, rd, y, ym);
  auto put = [&](REAL *p, uint32_t off, REAL v) {
    hyb::st<NT>(reinterpret_cast<REAL *>(reinterpret_cast<char *>(p) + off), v);
  };
#pragma unroll
  for (int r = 0; r < M; ++r)
    if (r < rows) put(lam, obs + (uint32_t)r * os, rd[r]);
  if (GRAD) {
    if (ga) {
#pragma unroll
      for (int r = 0; r < M; ++r)
        if (r < rows)
          put(ga, obs + (uint32_t)r * os,
              row0 + r == 0 ? REAL(0) : -rd[r] * (r > 0 ? xs[(r - 1) * W] : xprev));
    }
    if (gb) {
#pragma unroll
      for (int r = 0; r < M; ++r)
        if (r < rows) put(gb, obs + (uint32_t)r * os, -rd[r] * xs[r * W]);
    }
    if (gc) {
#pragma unroll
      for (int r = 0; r < M; ++r)
        if (r < rows)
          put(gc, obs + (uint32_t)r * os,
              r + 1 < rows ? -rd[r] * (r + 1 < M ? xs[(r + 1) * W] : xnext) : REAL(0));
    }
  }
}

template <typename REAL, int M, int SEG, bool GRAD, bool NT>
hipError_t launch_adjoint_wide_nt(const Geom &g, const HybridCfg &cfg, const REAL *a,
                                  const REAL *b, const REAL *c, const REAL *x, const REAL *w,
                                  REAL *lam, REAL *ga, REAL *gb, REAL *gc, hipStream_t st) {
  const int slots = wide::wide_slots<REAL>(M, cfg.P, SEG);
  const size_t lds = wide::wide_lds_bytes<REAL>(M, cfg.P, SEG, slots);
  auto kern = adjoint_wide_kernel<REAL, M, SEG, GRAD, NT>;
  static LdsGrant lds_granted;
  {
    hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), lds, lds_granted);
    if (e != hipSuccess) return e;
  }
  const int64_t blocks = (g.n0 + cfg.W - 1) / cfg.W * g.n1;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(cfg.W * cfg.P), lds, st, g, cfg.P, cfg.G,
                     slots, a, b, c, x, w, lam, ga, gb, gc);
  return hipGetLastError();
}

template <typename REAL, int M, int SEG>
hipError_t launch_adjoint_wide(const Geom &g, const HybridCfg &cfg, const REAL *a, const REAL *b,
                               const REAL *c, const REAL *x, const REAL *w, REAL *lam, REAL *ga,
                               REAL *gb, REAL *gc, hipStream_t st) {
  const bool grad = ga || gb || gc;
  uintptr_t low = (uintptr_t)a | (uintptr_t)b | (uintptr_t)w | (uintptr_t)lam;
  if (grad) low |= (uintptr_t)x | (uintptr_t)ga | (uintptr_t)gb | (uintptr_t)gc;
  const bool nt = wide::wide_rows_aligned<REAL>(g, low);
#define TRID_ADJ_WIDE(GRAD, NT)                                                          \
  return launch_adjoint_wide_nt<REAL, M, SEG, GRAD, NT>(g, cfg, a, b, c, x, w, lam, ga, gb, gc, st)
  if (grad && nt) TRID_ADJ_WIDE(true, true);
  if (grad) TRID_ADJ_WIDE(true, false);
  if (nt) TRID_ADJ_WIDE(false, true);
  TRID_ADJ_WIDE(false, false);
#undef TRID_ADJ_WIDE
}

// Nontemporal loads and stores except for strided systems whose rows are
// 64 KiB or more apart (256^3 FP64, all gradients: x / y 0.233 / 0.233 ms
// with them against 0.242 / 0.252, z 0.294 against 0.282).
template <typename REAL, int M, bool CONTIG, bool GRAD, bool NT>
hipError_t launch_adjoint_nt(const Geom &g, const HybridCfg &cfg, const REAL *a,
                             const REAL *b, const REAL *c, const REAL *x, const REAL *w,
                             REAL *lam, REAL *ga, REAL *gb, REAL *gc, hipStream_t st) {
  const int T = cfg.W * cfg.P;
  size_t lds = hyb::ring_bytes<REAL>(T, 3);
  if (CONTIG) lds += sizeof(REAL) * (size_t)T * (M + 1);
  auto kern = adjoint_kernel<REAL, M, CONTIG, GRAD, NT>;
  static LdsGrant lds_granted;
  {
    hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), lds, lds_granted);
    if (e != hipSuccess) return e;
  }
  const int64_t blocks = (g.n0 + cfg.W - 1) / cfg.W * g.n1;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(T), lds, st, g, cfg.P, cfg.W, cfg.G,
                     a, b, c, x, w, lam, ga, gb, gc);
  return hipGetLastError();
}

template <typename REAL, int M, bool CONTIG, bool GRAD>
hipError_t launch_adjoint_m(const Geom &g, const HybridCfg &cfg, const REAL *a,
                            const REAL *b, const REAL *c, const REAL *x, const REAL *w,
                            REAL *lam, REAL *ga, REAL *gb, REAL *gc, hipStream_t st) {
  if (CONTIG || g.stride * (int64_t)sizeof(REAL) < (64 << 10))
    return launch_adjoint_nt<REAL, M, CONTIG, GRAD, true>(g, cfg, a, b, c, x, w, lam, ga, gb,
                                                          gc, st);
  return launch_adjoint_nt<REAL, M, CONTIG, GRAD, false>(g, cfg, a, b, c, x, w, lam, ga, gb,
                                                         gc, st);
}

template <typename REAL>
int adj_max_threads(int M) {
  switch (M) {
    case 1: return AdjBounds<REAL, 1>::threads;
    case 2: return AdjBounds<REAL, 2>::threads;
    case 4: return AdjBounds<REAL, 4>::threads;
    case 8: return AdjBounds<REAL, 8>::threads;
    case 16: return AdjBounds<REAL, 16>::threads;
    default: return 0;
  }
}

// ---- systems longer than the adjoint kernel holds -------------------------
// The transpose's off-diagonals in the layout of the inputs, sub[n] = c[n-1]
// and sup[n] = a[n+1] (0 where the row has none), and lam = w, the right-hand
// side the batched solve then overwrites with the solution of A^T lam = w.
template <typename REAL, bool CONTIG>
__global__ __launch_bounds__(256) void adj_transpose_kernel(
    Geom g, const REAL *__restrict__ a, const REAL *__restrict__ c, const REAL *__restrict__ w,
    REAL *__restrict__ sub, REAL *__restrict__ sup, REAL *__restrict__ lam) {
  const int64_t total = g.nsys() * g.N;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * 256) {
    int64_t k;
    const int64_t i = hyb::batch_elem<CONTIG>(g, e, &k);
    sub[i] = k > 0 ? c[i - g.stride] : REAL(0);
    sup[i] = k + 1 < g.N ? a[i + g.stride] : REAL(0);
    lam[i] = w[i];
  }
}

// dL/da[n] = -lam[n] x[n-1] (0 at n = 0), dL/db[n] = -lam[n] x[n],
// dL/dc[n] = -lam[n] x[n+1] (0 at n = N-1), each where its output is given.
template <typename REAL, bool CONTIG>
__global__ __launch_bounds__(256) void adj_grad_kernel(Geom g, const REAL *__restrict__ x,
                                                       const REAL *__restrict__ lam,
                                                       REAL *__restrict__ ga,
                                                       REAL *__restrict__ gb,
                                                       REAL *__restrict__ gc) {
  const int64_t total = g.nsys() * g.N;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * 256) {
    int64_t k;
    const int64_t i = hyb::batch_elem<CONTIG>(g, e, &k);
    const REAL l = lam[i];
    if (ga) ga[i] = k > 0 ? -l * x[i - g.stride] : REAL(0);
    if (gb) gb[i] = -l * x[i];
    if (gc) gc[i] = k + 1 < g.N ? -l * x[i + g.stride] : REAL(0);
  }
}

}  // namespace

template <typename REAL>
hipError_t launch_adjoint_transpose(const Geom &g, const REAL *a, const REAL *c, const REAL *w,
                                    REAL *sub, REAL *sup, REAL *lam, hipStream_t st) {
  if (g.stride == 1)
    hipLaunchKernelGGL((adj_transpose_kernel<REAL, true>), dim3(batch_elem_blocks(g)), dim3(256),
                       0, st, g, a, c, w, sub, sup, lam);
  else
    hipLaunchKernelGGL((adj_transpose_kernel<REAL, false>), dim3(batch_elem_blocks(g)),
                       dim3(256), 0, st, g, a, c, w, sub, sup, lam);
  return hipGetLastError();
}

template <typename REAL>
hipError_t launch_adjoint_grads(const Geom &g, const REAL *x, const REAL *lam, REAL *ga,
                                REAL *gb, REAL *gc, hipStream_t st) {
  if (g.stride == 1)
    hipLaunchKernelGGL((adj_grad_kernel<REAL, true>), dim3(batch_elem_blocks(g)), dim3(256), 0,
                       st, g, x, lam, ga, gb, gc);
  else
    hipLaunchKernelGGL((adj_grad_kernel<REAL, false>), dim3(batch_elem_blocks(g)), dim3(256), 0,
                       st, g, x, lam, ga, gb, gc);
  return hipGetLastError();
}

// Variant 3 on a shape that wide kernels hold takes adjoint_wide_kernel; every
// other variant number, and variant 3 on another shape, adjoint_kernel.
template <typename REAL>
static bool adjoint_wide(const Geom &g, const HybridCfg &c) {
  return c.V == 3 && wide::wide_shape_fits<REAL>(g, c);
}

template <typename REAL>
bool adjoint_cfg_valid(const Geom &g, const HybridCfg &c) {
  if (adjoint_wide<REAL>(g, c)) return true;
  // FP64 M = 16 on contiguous systems spills a few registers; not offered.
  if (sizeof(REAL) == 8 && c.M == 16 && g.stride == 1) return false;
  const int maxT = adj_max_threads<REAL>(c.M);
  if (maxT == 0 || c.P < 1 || c.W < 1 || c.G < 1) return false;
  if ((int64_t)c.P * c.M < g.N) return false;
  const int64_t T = (int64_t)c.W * c.P;
  if (T > maxT) return false;
  size_t lds = hyb::ring_bytes<REAL>((int)T, 3);
  if (g.stride == 1) lds += sizeof(REAL) * (size_t)T * (c.M + 1);
  return lds <= 160 * 1024;
}

// The most 128-byte rows of strided systems that adjoint_kernel solves: with few
// groups the chip is idle either way and what counts is one workgroup's time, which
// the wide kernel's staged tile, whole waves and serial outputs lengthen; it pays once
// workgroups follow each other on a CU. More so where the system fills its waves
// (N a multiple of 64 rows in FP64, 32 in FP32, at 16 rows per lane), less so on
// short systems. adjoint_kernel against the wide one, us, on lines of one group: FP64,
// all gradients, 16 rows, 512 groups 5.0 / 9.5; 96 rows, 512 groups 10.1 / 12.0, 1024
// 20.8 / 19.3; 64 rows, 256 groups 6.6 / 7.3, 512 10.6 / 7.8; 400 rows, 256 groups 21.3 /
// 23.2, 512 56 / 49; 1000 rows, 64 groups 22.3 / 28.2, 128 39.6 / 34.7; lambda alone, 64 rows
// 5.8 / 5.0 at 256 groups, 1000 rows 23.2 / 24.4 at 128, 32.3 / 24.5 at 192. FP32, all
// gradients, 40 rows, 512 groups 7.9 / 8.5, 768 11.6 / 9.1; 800 rows, 32 groups 20.2 / 22.7,
// 64 32.8 / 27.8; 592 rows of a z line of 56 18.5 / 22.5, 32 rows of 312 7.8 / 9.1.
// By the lines' shape too: on lines of at most half a segment the wide kernel leaves half
// its systems out (half: 8 x 1000 x 512 FP64 y, lambda alone, 38 against 50; 16 x 512 x 512
// FP32 20.5 against 23.0; a quarter, lambda alone, 8 x 621 x 309 FP32 17.5 / 23.4), and whole waves count for less where rows are misaligned
// (33 x 128 x 62 FP64 y, lambda alone, 5.9 against 6.9, on aligned lines 5.8 against 5.1).
// One long misaligned line of FP64 systems of up to 256 rows stays with adjoint_kernel,
// all gradients (32763 x 256 z 151 against 165, 601 x 404 x 136 z 580 against 597; 16379 x
// 300 z 94 against 92, 199 x 123 x 200 z, 1530 groups, 102 against 91).
template <typename REAL>
static int64_t adjoint_plain_most(const Geom &g, bool grads) {
  const int64_t N = g.N;
  const bool fp64 = sizeof(REAL) == 8, whole = N % (fp64 ? 64 : 32) == 0;
  const bool half = g.n0 * (int64_t)sizeof(REAL) <= 64;
  const bool aligned = !half && wide::wide_rows_aligned<REAL>(g, 0);
  if (N <= 16) return fp64 ? INT64_MAX : 16384 / N;
  if (half && (fp64 ? N > 512 : N > 256 && N <= 512)) return INT64_MAX;
  if (fp64 && grads && !aligned && g.n1 == 1 && N <= 256 && g.n0 > 28000) return INT64_MAX;
  if (!fp64 && N > 512 && g.n0 <= 8) return grads ? 80 : 256;
  if (N > 512) return fp64 ? (grads ? 96 : 128) : grads ? 60 : 64;
  if (N > 256) return !fp64 ? 128 : !whole ? 256 : half ? 160 : 0;
  if (!whole) {
    if (!grads) return N < 64 ? 512 : aligned ? 256 : 300;
    return N < (fp64 ? 64 : 32) ? 1024 : fp64 || N <= 192 ? 512 : 384;
  }
  if (!grads)
    return aligned ? 0 : N < 64 ? 300 : N <= 192 ? (fp64 ? 256 : 160) : half ? 160 : 32;
  if (N <= 96) return (fp64 ? !aligned : N < 64) ? 512 : 256;
  if (N <= 192) return aligned ? 512 : half ? 384 : fp64 ? 300 : 224;
  if (half) return 160;
  return fp64 ? (aligned ? 0 : 64) : aligned ? 384 : 128;
}

// Whether contiguous systems take the fewest rows per lane that keep a system in one
// wave (hybrid_fewest_rows_cfg). At more rows a wave's accesses spread over more lines
// each, which nine streams feel on short systems: us at the fewest rows / at the
// solve's shape, all gradients, FP32: 8 x 262144 21 / 41, 16 x 65536 13 / 17, 24 x 65536 21 /
// 25, 24 x 16384 7.9 / 7.4, 100 x 65536 58 / 64, 100 x 8192 10.7 / 9.2, 64 x 2048 5.5 / 5.9, 64 x
// 4096 6.6 / 6.1; FP64: 16 x 65536 17.9 / 19.7, 16 x 16384 7.9 / 6.8. lambda alone, FP32, 8 x
// 16384 4.1 / 4.6.
// Rows or planes apart from each other have more lines: sooner there (FP64, 8 / 16 rows, 600000
// elements, 2 apart, as at 750000: 0.70 / 0.77 of the time; FP32 12 rows, 400000, 0.76).
template <typename REAL>
static bool adjoint_fewest_rows(const Geom &g, bool grads) {
  const int64_t N = g.N, n = N * g.nsys();
  const bool apart = g.st0 != N || (g.n1 > 1 && g.st1 != g.n0 * N), pow2 = (N & (N - 1)) == 0;
  if (sizeof(REAL) == 8) {
    if (!grads) return false;
    if (N <= 24) return n >= 750000 || (apart && g.nsys() >= 30000);
    return apart && N <= 50 && n >= (N <= 32 ? 750000 : 2500000);
  }
  if (!grads) return N == 8;
  if (N < 4 || (pow2 && N <= 32)) return true;
  if (N <= 16) return g.nsys() >= 16500;
  if (N <= 24) return n >= 750000;
  if (pow2) return N <= 128 && (n <= 200000 || (g.st0 % 4 != 0 && n >= 2500000));
  return N <= 100 && n >= (N <= 64 && g.st0 % 4 != 0 ? 750000 : 2500000);
}

template <typename REAL>
bool adjoint_default_cfg(const Geom &g, bool grads, HybridCfg *cfg) {
  // Strided systems: the forward solve's wide shape, unless they are few
  // (adjoint_plain_most). Otherwise the same shapes as the forward solve where
  // they fit the adjoint's register budget, else the next valid one.
  HybridCfg c;
  // (128-byte groups of the lines; two lines of at most half a group count as one)
  const int64_t line = g.n0 * (int64_t)sizeof(REAL);
  const int64_t rows = line <= 64 ? (g.n1 * line + 127) / 128 : (line + 127) / 128 * g.n1;
  if (g.stride != 1 && rows > adjoint_plain_most<REAL>(g, grads) &&
      hybrid_wide_default_cfg<REAL>(g, &c) && adjoint_wide<REAL>(g, c)) {
    if (sizeof(REAL) == 4 && g.N <= 512 && wide::wide_many_groups<REAL>(g) &&
        wide::wide_whole_segments<REAL>(g)) {
      // nine streams of 128-byte rows want more bytes per row than the
      // solve's five: 256-byte rows at every length (256^3 FP32 y / z 108 /
      // 113 against 114 / 127 us, 203 x 170 x 300 z 117 against 128)
      c.M = g.N > 256 ? 32 : 16;
      c.W = 64;
      c.P = (int)((g.N + c.M - 1) / c.M);
    }
    if (sizeof(REAL) == 8 && g.N > 192 && g.N <= 512 && wide::wide_many_groups<REAL>(g, 160) &&
        wide::wide_whole_segments<REAL>(g)) {
      // 256-byte rows of long systems from fewer workgroups on than in the solve (64 x 256
      // x 80 y 17.9 against 22.7 us, lambda alone, x 128 14.9 / 15.5; 64 x 400 x 64, 128
      // workgroups, 26.8 against 23.3)
      c.W = 32;
      c.P = (int)(g.N + 31) / 32 * 2;
    }
    // plain workgroup order for short ones on aligned lines (64 x 128 x 1024 y 94.7 against
    // 104.3 us, 192^3 y 86.8 / 90.0; 512 x 512 x 64 y the other way, 230.6 / 216.9)
    if (sizeof(REAL) == 8 && g.N <= 192 && wide::wide_rows_aligned<REAL>(g, 0)) c.G = 1;
    *cfg = c;
    return true;
  }
  if (g.stride == 1 && adjoint_fewest_rows<REAL>(g, grads) &&
      hybrid_fewest_rows_cfg<REAL>(g, &c) && adjoint_cfg_valid<REAL>(g, c)) {
    *cfg = c;
    return true;
  }
  if (g.stride == 1 && sizeof(REAL) == 8 && g.N > 32 && g.N <= 256) {
    // fewer rows per lane than the solve takes at these lengths: with nine
    // streams the loads in flight matter more than the PCR (all gradients, 100
    // / 200 rows: 125 / 85 against 137 / 89 us)
    c.M = g.N <= 128 ? 2 : 4;
    c.P = (int)((g.N + c.M - 1) / c.M);
    c.W = std::max(1, 256 / c.P);
    c.G = 1;
    c.V = 0;
    if (adjoint_cfg_valid<REAL>(g, c)) { *cfg = c; return true; }
  }
  if (hybrid_plain_cfg<REAL>(g, &c)) {
    // (a workgroup each for a few longer systems: 1000 rows x 64 FP64 8.5 against 9.9 us)
    if (g.stride == 1 && sizeof(REAL) == 8 && g.N > 512 && g.nsys() <= 256) c.W = 1;
    for (int k = 0; k < 4 && !adjoint_cfg_valid<REAL>(g, c); ++k) {
      if (g.stride == 1 && c.W > 1) c.W /= 2;
      else if (c.M < 16) { c.M *= 2; c.P = (int)((g.N + c.M - 1) / c.M); }
    }
    if (adjoint_cfg_valid<REAL>(g, c)) { *cfg = c; return true; }
  }
  static const int Ms[] = {8, 4, 16, 2, 1};
  for (int W = g.stride == 1 ? 1 : 128 / (int)sizeof(REAL); W >= 1; W /= 2)
    for (int M : Ms) {
      c.M = M;
      c.P = (int)((g.N + M - 1) / M);
      c.W = W;
      c.G = 8;
      if (adjoint_cfg_valid<REAL>(g, c)) { *cfg = c; return true; }
    }
  return false;
}

template <typename REAL>
hipError_t launch_adjoint(const Geom &g, const HybridCfg &cfg, const REAL *a, const REAL *b,
                          const REAL *c, const REAL *x, const REAL *w, REAL *lam, REAL *ga,
                          REAL *gb, REAL *gc, hipStream_t st) {
  const bool contig = g.stride == 1, grad = ga || gb || gc;
  if (adjoint_wide<REAL>(g, cfg)) {
    const bool s256 = cfg.W * (int)sizeof(REAL) == 256;
    if (cfg.M == 16)
      return s256 ? launch_adjoint_wide<REAL, 16, 256>(g, cfg, a, b, c, x, w, lam, ga, gb, gc, st)
                  : launch_adjoint_wide<REAL, 16, 128>(g, cfg, a, b, c, x, w, lam, ga, gb, gc, st);
    return s256 ? launch_adjoint_wide<REAL, 32, 256>(g, cfg, a, b, c, x, w, lam, ga, gb, gc, st)
                : launch_adjoint_wide<REAL, 32, 128>(g, cfg, a, b, c, x, w, lam, ga, gb, gc, st);
  }
#define TRID_ADJ_CASE(MM)                                                                  \
  case MM:                                                                                 \
    if (grad)                                                                              \
      return contig ? launch_adjoint_m<REAL, MM, true, true>(g, cfg, a, b, c, x, w, lam, ga, \
                                                             gb, gc, st)                   \
                    : launch_adjoint_m<REAL, MM, false, true>(g, cfg, a, b, c, x, w, lam, \
                                                              ga, gb, gc, st);             \
    return contig ? launch_adjoint_m<REAL, MM, true, false>(g, cfg, a, b, c, x, w, lam, ga, \
                                                            gb, gc, st)                    \
                  : launch_adjoint_m<REAL, MM, false, false>(g, cfg, a, b, c, x, w, lam, ga, \
                                                             gb, gc, st);
  switch (cfg.M) {
    TRID_ADJ_CASE(1)
    TRID_ADJ_CASE(2)
    TRID_ADJ_CASE(4)
    TRID_ADJ_CASE(8)
    TRID_ADJ_CASE(16)
    default:
      return hipErrorInvalidValue;
  }
#undef TRID_ADJ_CASE
}

template bool adjoint_cfg_valid<float>(const Geom &, const HybridCfg &);
template bool adjoint_cfg_valid<double>(const Geom &, const HybridCfg &);
template bool adjoint_default_cfg<float>(const Geom &, bool, HybridCfg *);
template bool adjoint_default_cfg<double>(const Geom &, bool, HybridCfg *);
template hipError_t launch_adjoint<float>(const Geom &, const HybridCfg &, const float *,
                                          const float *, const float *, const float *,
                                          const float *, float *, float *, float *, float *,
                                          hipStream_t);
template hipError_t launch_adjoint<double>(const Geom &, const HybridCfg &, const double *,
                                           const double *, const double *, const double *,
                                           const double *, double *, double *, double *,
                                           double *, hipStream_t);
#define TRID_ADJ_LONG_INST(REAL)                                                            \
  template hipError_t launch_adjoint_transpose<REAL>(const Geom &, const REAL *, const REAL *, \
                                                     const REAL *, REAL *, REAL *, REAL *,     \
                                                     hipStream_t);                             \
  template hipError_t launch_adjoint_grads<REAL>(const Geom &, const REAL *, const REAL *,    \
                                                 REAL *, REAL *, REAL *, hipStream_t);
TRID_ADJ_LONG_INST(float)
TRID_ADJ_LONG_INST(double)
#undef TRID_ADJ_LONG_INST

}  // namespace trid
