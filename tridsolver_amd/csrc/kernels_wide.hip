// kernels_wide.hip - strided Thomas-PCR hybrid with 128- or 256-byte row
// segments.
//
// A workgroup solves W = SEG / sizeof(REAL) x-neighbouring systems, so each row
// it reads is one contiguous segment of SEG bytes. For z solves every row lies
// in its own page; 256-byte segments halve the address translations per byte
// moved against 128-byte ones.
//
// What bounds it: HBM, as long as the arithmetic hides behind the loads. At
// 256-byte rows of 512 FP64 rows a CU holds one workgroup (its operands fill
// the register file and most of the LDS), so whatever a workgroup does after
// its last load has arrived and before its last store is issued leaves the CU
// without traffic. The kernel therefore keeps that part short:
//   - `a` goes HBM->LDS by global->LDS loads (global_load_lds_dword, no
//     registers), every wave fetching the rows of its own chunks, so no
//     workgroup barrier stands between the loads and the sweep; b, c and d go to
//     registers behind it, row by row.
//   - (i) the forward sweep takes each row as soon as it has arrived. Row i
//     becomes al_i x_{s-1} + x_i + ga_i x_{i+1} = de_i; al overwrites b's
//     register (a row's b is dead once its pivot is formed), ga c's, de d's.
//   - (ii) the chunk's first unknown in terms of x_{s-1} and x_{i+1},
//     x_s = F - Fa x_{s-1} - Fg x_{i+1}, is carried along the same sweep
//     (F -= Fg de_i, Fa -= Fg al_i, Fg = -Fg ga_i): no backward sweep.
//   - (iii) the reduced system in y_k = x_{e_k}, by PCR (hyb::reduced_solve).
//   - (iv) back substitution from the chunk's end, x_i = de_i - al_i x_{s-1} -
//     ga_i x_{i+1}, in registers. For Inc, u's rows come into the LDS tile
//     (which `a` has left) during (iii).
// 512^3 FP64 z: 0.91-0.94 ms, 5.7-5.9 TB/s (1.05-1.09 ms, 4.9-5.1 TB/s, with
// every load awaited before the sweep, a backward sweep and al / ap kept in the
// LDS tile); 400 x 360 x 300 FP32 y, u += x: 0.221 against 0.253 ms.
//
// LDS: P chunks of M rows x SEG bytes (plus SEG bytes a chunk for 128-byte
// rows, so that a half wave's two or more chunks read different banks), and the
// PCR ring (3 values per thread per slot, two slots when they fit).

#include <algorithm>
#include <atomic>

#include "trid_internal.h"
#include "wide_core.hpp"

namespace trid {
namespace {

using namespace wide;

// Waves per SIMD that the registers are held to: at FP32, 16 rows of 128 bytes, two of
// the largest workgroups (1024 threads) share a CU at 64 VGPRs, which the compiler
// exceeds by two without the bound (32 x 500 x 2048 y 101 against 120 us).
template <typename REAL, int M, int SEG>
constexpr int wide_waves() {
  return sizeof(REAL) == 4 && M == 16 && SEG == 128 ? 8 : 1;
}

template <typename REAL, int M, int SEG, bool INC, bool NT>
__global__ __launch_bounds__((WideBounds<REAL, M>::threads), (wide_waves<REAL, M, SEG>()))
void hybrid_wide_kernel(
    Geom g, int P, int G, int slots, const REAL *__restrict__ a, const REAL *__restrict__ b,
    const REAL *__restrict__ c, const REAL *d, REAL *u) {
  constexpr int W = WideShape<REAL, SEG>::W;
  constexpr int CH = 64 / W;  // chunks per wave
  constexpr int PITCH = wide_chunk_bytes(M, SEG);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const hyb::Lane L = hyb::lane_of<false>(g, P, W, G);
  const int T = L.T;
  hyb::Ring ring{smem_raw + (size_t)P * PITCH, (int)(3 * sizeof(REAL) * T), 0, slots};
  const int lane = L.t & 63, wv = __builtin_amdgcn_readfirstlane(L.t >> 6);
  const int N = (int)L.N;
  const uint32_t tile = hyb::lds_address(smem_raw) + wv * CH * PITCH;  // the wave's first chunk
  // Addresses are 32-bit byte offsets from uniform bases (extent < 4 GiB,
  // checked by wide_cfg_valid).
  const int64_t first = hyb::wave_uniform(L.i0 - L.w);  // x index of the workgroup's system 0
  const int64_t base0 = first + hyb::wave_uniform(L.i1) * g.st1, nsys = g.n0 - first;
  const uint32_t os = (uint32_t)(L.stride * (int64_t)sizeof(REAL));
  const int row0 = L.p * M;
  const int rows = L.active ? N - row0 : 0;  // rows of the system from this chunk on
  const uint32_t ob = (uint32_t)(L.base + row0 * L.stride) * (uint32_t)sizeof(REAL);
  // as[r * W]: the lane's row r in the tile
  REAL *as = reinterpret_cast<REAL *>(reinterpret_cast<char *>(smem_raw) + L.p * PITCH) + L.w;
  const bool whole = __all(rows >= M);
  REAL rb[M], rc[M], rd[M], f_d, f_a, f_g;
  if (whole)
    wide_sweep<REAL, M, SEG, CH, true, NT>(a + base0, tile, wv * CH * M, lane, N, nsys, os, ob, row0,
                                       rows, as, b, c, d, rb, rc, rd, f_d, f_a, f_g);
  else
    wide_sweep<REAL, M, SEG, CH, false, NT>(a + base0, tile, wv * CH * M, lane, N, nsys, os, ob, row0,
                                        rows, as, b, c, d, rb, rc, rd, f_d, f_a, f_g);
  if (INC) {  // the wave has read its rows of a: u's take their place
    int ln = lane;
    asm volatile("" : "+v"(ln));  // offsets formed here, not held from the first staging
    if (whole) wide_stage<REAL, M, SEG, CH, true>(u + base0, tile, wv * CH * M, ln, os, N, nsys);
    else wide_stage<REAL, M, SEG, CH, false>(u + base0, tile, wv * CH * M, ln, os, N, nsys);
  }
  // (iii)
  REAL y, ym;
  hyb::reduced_solve<REAL>(L, ring, rb[M - 1], rc[M - 1], rd[M - 1], f_d, f_a, f_g, y, ym);
  // (iv). The lane's rows and offsets are formed here again from a thread index that
  // the compiler cannot match with the first (empty asm), so that none of them is held
  // in registers across the whole kernel.
  int ts = L.t;
  asm volatile("" : "+v"(ts));
  const int p = ts / W, w = ts % W;
  if (w >= nsys) return;
  if (INC) hyb::stage_wait_all();
  hyb::substitute_back<REAL, M>(rb, rc, rd, y, ym);
  const uint32_t obs = (uint32_t)(base0 + w + (int64_t)p * M * L.stride) * (uint32_t)sizeof(REAL);
  const REAL *us = reinterpret_cast<REAL *>(smem_raw + p * PITCH) + w;
  char *dst = reinterpret_cast<char *>(u);  // u == d for a solve in place
#pragma unroll
  for (int r = 0; r < M; ++r) {
    if (p * M + r < N) {
      REAL *q = reinterpret_cast<REAL *>(dst + obs + (uint32_t)r * os);
      if (INC) hyb::st<NT>(q, us[r * W] + rd[r]);
      else hyb::st<NT>(q, rd[r]);
    }
  }
}

template <typename REAL, int M, int SEG, bool INC, bool NT>
hipError_t launch_wide_nt(const Geom &g, const HybridCfg &cfg, const REAL *a, const REAL *b,
                         const REAL *c, REAL *d, REAL *u, hipStream_t st) {
  constexpr int W = WideShape<REAL, SEG>::W;
  const int T = W * cfg.P;
  const int slots = wide_slots<REAL>(M, cfg.P, SEG);
  const size_t lds = wide_lds_bytes<REAL>(M, cfg.P, SEG, slots);
  auto kern = hybrid_wide_kernel<REAL, M, SEG, INC, NT>;
  static LdsGrant lds_granted;
  {
    hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), lds, lds_granted);
    if (e != hipSuccess) return e;
  }
  const int64_t blocks = (g.n0 + W - 1) / W * g.n1;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(T), lds, st, g, cfg.P, cfg.G, slots, a,
                     b, c, d, u ? u : d);
  return hipGetLastError();
}

// Nontemporal or plain access by the rows' alignment (wide_rows_aligned).
template <typename REAL, int M, int SEG, bool INC>
hipError_t launch_wide_m(const Geom &g, const HybridCfg &cfg, const REAL *a, const REAL *b,
                         const REAL *c, REAL *d, REAL *u, hipStream_t st) {
  const uintptr_t low = (uintptr_t)b | (uintptr_t)c | (uintptr_t)d | (uintptr_t)(u ? u : d);
  if (wide_rows_aligned<REAL>(g, low))
    return launch_wide_nt<REAL, M, SEG, INC, true>(g, cfg, a, b, c, d, u, st);
  return launch_wide_nt<REAL, M, SEG, INC, false>(g, cfg, a, b, c, d, u, st);
}

}  // namespace

template <typename REAL>
bool wide_cfg_valid(const Geom &g, const HybridCfg &c) {
  return wide_shape_fits<REAL>(g, c);
}

template <typename REAL, bool INC>
hipError_t launch_wide(const Geom &g, const HybridCfg &cfg, const REAL *a, const REAL *b,
                       const REAL *c, REAL *d, REAL *u, hipStream_t st) {
  const bool s256 = cfg.W * (int)sizeof(REAL) == 256;
  if (cfg.M == 16)
    return s256 ? launch_wide_m<REAL, 16, 256, INC>(g, cfg, a, b, c, d, u, st)
                : launch_wide_m<REAL, 16, 128, INC>(g, cfg, a, b, c, d, u, st);
  if (cfg.M == 32)
    return s256 ? launch_wide_m<REAL, 32, 256, INC>(g, cfg, a, b, c, d, u, st)
                : launch_wide_m<REAL, 32, 128, INC>(g, cfg, a, b, c, d, u, st);
  return hipErrorInvalidValue;
}

#define TRID_WIDE_INST(REAL)                                                                  \
  template bool wide_cfg_valid<REAL>(const Geom &, const HybridCfg &);                        \
  template hipError_t launch_wide<REAL, false>(const Geom &, const HybridCfg &, const REAL *,  \
                                               const REAL *, const REAL *, REAL *, REAL *,     \
                                               hipStream_t);                                  \
  template hipError_t launch_wide<REAL, true>(const Geom &, const HybridCfg &, const REAL *,   \
                                              const REAL *, const REAL *, REAL *, REAL *,      \
                                              hipStream_t);
TRID_WIDE_INST(float)
TRID_WIDE_INST(double)

}  // namespace trid
