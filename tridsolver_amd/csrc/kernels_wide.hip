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

#include "hybrid_core.hpp"
#include "trid_internal.h"

namespace trid {
namespace {

// SEG: bytes of one row segment (W * sizeof(REAL)), 128 or 256.
template <typename REAL, int SEG>
struct WideShape {
  static constexpr int W = SEG / (int)sizeof(REAL);
};
// Threads per workgroup the register file allows: FP64 M = 32 holds 3 x 64
// VGPRs of b, c, d (512 threads); everything else fits 1024.
template <typename REAL, int M>
struct WideBounds {
  static constexpr int threads = (sizeof(REAL) == 8 && M == 32) ? 512 : 1024;
};
constexpr size_t WIDE_LDS = 160 * 1024;

// Bytes of one chunk's tile: M rows, and a row's worth of padding for
// 128-byte rows.
constexpr int wide_chunk_bytes(int M, int seg) { return M * seg + (seg < 256 ? seg : 0); }

// PCR exchange slots: two (one barrier per step) where they cost no
// workgroup per CU, else one (two barriers per step).
template <typename REAL>
size_t wide_lds_bytes(int M, int P, int seg, int slots) {
  const int T = seg / (int)sizeof(REAL) * P;
  return (size_t)P * wide_chunk_bytes(M, seg) + (size_t)slots * 3 * sizeof(REAL) * (size_t)T;
}
template <typename REAL>
int wide_slots(int M, int P, int seg) {
  const size_t one = wide_lds_bytes<REAL>(M, P, seg, 1), two = wide_lds_bytes<REAL>(M, P, seg, 2);
  return WIDE_LDS / two == WIDE_LDS / one ? 2 : 1;
}

// Rows of the wave's own chunks, src[row] -> tile, by global->LDS loads: one
// wave instruction moves 256 bytes (lane l: bytes 4l..4l+3), i.e. K = 256 / SEG
// rows of one chunk. The wave's chunks are rows row0 .. row0 + CH*M - 1, taken
// in the order the forward sweep reads them. src is the address of the
// workgroup's first system, tile that of the wave's first chunk. Without WHOLE,
// lanes whose row is >= N or whose system is past the last (nsys systems from
// src on) are masked off.
template <typename REAL, int M, int SEG, int CH, bool WHOLE>
__device__ __forceinline__ void wide_stage(const REAL *src, uint32_t tile, int row0, int lane,
                                           uint32_t row_bytes, int N, int64_t nsys) {
  constexpr int K = 256 / SEG;
  const int sub = (lane * 4) / SEG;
  const uint32_t byte = (uint32_t)(lane * 4) % SEG;
  if constexpr (WHOLE) {
    const uint32_t o = (uint32_t)(row0 + sub) * row_bytes + byte;
#pragma unroll
    for (int r = 0; r < M; r += K)
#pragma unroll
      for (int q = 0; q < CH; ++q)
        hyb::stage_dword(tile + q * wide_chunk_bytes(M, SEG) + r * SEG, src,
                         o + (uint32_t)(q * M + r) * row_bytes);
  } else {
    if ((int)byte / (int)sizeof(REAL) >= nsys) return;
    for (int r = 0; r < M; r += K)
      for (int q = 0; q < CH; ++q) {
        const int row = row0 + q * M + r + sub;
        if (row < N)
          hyb::stage_dword(tile + q * wide_chunk_bytes(M, SEG) + r * SEG, src,
                           (uint32_t)row * row_bytes + byte);
      }
  }
}

// (i) and (ii) on one wave's chunks, loads included: (b, c, d) -> (al, ga, de)
// of the lane's M rows, and x_s = f_d - f_a x_{s-1} - f_g x_e. WHOLE: every row
// of every lane lies inside an existing system, so every load is unmasked and
// the sweep of row r waits for the loads of rows 0..r only (global->LDS and
// register loads complete in order; the `a` rows come first). Otherwise rows
// past N, and systems past n0, become identity rows (their tile slots, which no
// global->LDS load writes, are set to 0 here).
template <typename REAL, int M, int SEG, int CH, bool WHOLE, bool NT>
__device__ __forceinline__ void wide_sweep(const REAL *a0, uint32_t tile, int wave_row0, int lane,
                                           int N, int64_t nsys, uint32_t os, uint32_t ob,
                                           int row0, int rows, REAL *as,
                                           const REAL *__restrict__ b,
                                           const REAL *__restrict__ c,
                                           const REAL *__restrict__ d, REAL (&rb)[M],
                                           REAL (&rc)[M], REAL (&rd)[M], REAL &f_d, REAL &f_a,
                                           REAL &f_g) {
  constexpr int W = WideShape<REAL, SEG>::W;
  wide_stage<REAL, M, SEG, CH, WHOLE>(a0, tile, wave_row0, lane, os, N, nsys);
  ob = hyb::loads_after_stage(ob);
  auto at = [](const REAL *p, uint32_t off) -> REAL {
    return hyb::ld<NT>(reinterpret_cast<const REAL *>(reinterpret_cast<const char *>(p) + off));
  };
#pragma unroll
  for (int r = 0; r < M; ++r) {
    const uint32_t o = ob + (uint32_t)r * os;
    if constexpr (WHOLE) {
      rb[r] = at(b, o);
      rc[r] = at(c, o);
      rd[r] = at(d, o);
      __builtin_amdgcn_sched_barrier(0);  // the loads stay in row order
    } else {
      rb[r] = r < rows ? at(b, o) : REAL(1);
      rc[r] = r + 1 < rows ? at(c, o) : REAL(0);
      rd[r] = r < rows ? at(d, o) : REAL(0);
      if (r >= rows) as[r * W] = REAL(0);
    }
  }
  if constexpr (WHOLE) hyb::stage_done(rb[0]);
  else hyb::stage_wait_all();
  // one row at a time (scheduling barriers), the next row's a read from LDS
  // ahead of it
  f_d = 0; f_a = 0; f_g = -1;
  REAL ar = as[0], al = 0;
  if (row0 == 0) ar = REAL(0);  // a of the system's first row is not used
#pragma unroll
  for (int r = 0; r < M; ++r) {
    REAL anext = 0;
    if (r + 1 < M) anext = as[(r + 1) * W];
    if (r == 0) {
      const REAL inv = REAL(1) / rb[0];
      al = ar * inv;
      rc[0] = rc[0] * inv;
      rd[0] = rd[0] * inv;
      if (M >= 2) { f_d = rd[0]; f_a = al; f_g = rc[0]; }
    } else {
      const REAL inv = REAL(1) / (rb[r] - ar * rc[r - 1]);
      al = -ar * al * inv;
      // c of the system's last row is not used
      rc[r] = (WHOLE && r == M - 1 && rows == M) ? REAL(0) : rc[r] * inv;
      rd[r] = (rd[r] - ar * rd[r - 1]) * inv;
      if (r < M - 1) {
        f_d = f_d - f_g * rd[r];
        f_a = f_a - f_g * al;
        f_g = -f_g * rc[r];
      }
    }
    rb[r] = al;
    ar = anext;
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <typename REAL, int M, int SEG, bool INC, bool NT>
__global__ __launch_bounds__((WideBounds<REAL, M>::threads)) void hybrid_wide_kernel(
    Geom g, int P, int G, int slots, const REAL *__restrict__ a, const REAL *__restrict__ b,
    const REAL *__restrict__ c, REAL *__restrict__ d, REAL *__restrict__ u) {
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
  if (!L.active) return;
  // (iv)
  if (INC) hyb::stage_wait_all();
  rd[M - 1] = y;
#pragma unroll
  for (int r = M - 2; r >= 0; --r) rd[r] = rd[r] - rb[r] * ym - rc[r] * rd[r + 1];
  // The store offsets are recomputed here (the empty asm hides that they
  // equal the load offsets, which would otherwise be kept live in registers
  // across the whole kernel).
  uint32_t obs = ob;
  asm volatile("" : "+v"(obs));
  char *dst = reinterpret_cast<char *>(INC ? u : d);
#pragma unroll
  for (int r = 0; r < M; ++r) {
    if (r < rows) {
      REAL *q = reinterpret_cast<REAL *>(dst + obs + (uint32_t)r * os);
      if (INC) hyb::st<NT>(q, as[r * W] + rd[r]);
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
                     b, c, d, u);
  return hipGetLastError();
}

// Nontemporal access where every row starts on a 128-byte line, plain access
// where rows are misaligned: a workgroup's segments then share lines with
// the neighbouring workgroups', and only plain stores let an XCD's L2 join the two
// partial lines (777 x 300 x 250 FP64 along y: 560 MB written with nontemporal
// stores, 472 with plain ones, 466 algorithmic).
template <typename REAL, int M, int SEG, bool INC>
hipError_t launch_wide_m(const Geom &g, const HybridCfg &cfg, const REAL *a, const REAL *b,
                         const REAL *c, REAL *d, REAL *u, hipStream_t st) {
  const uintptr_t low = (uintptr_t)b | (uintptr_t)c | (uintptr_t)d | (uintptr_t)(INC ? u : d) |
                        (uintptr_t)(g.stride * (int64_t)sizeof(REAL)) |
                        (uintptr_t)(g.n1 > 1 ? g.st1 * (int64_t)sizeof(REAL) : 0);
  if (low % 128 == 0) return launch_wide_nt<REAL, M, SEG, INC, true>(g, cfg, a, b, c, d, u, st);
  return launch_wide_nt<REAL, M, SEG, INC, false>(g, cfg, a, b, c, d, u, st);
}

}  // namespace

// Rows per lane compiled for the wide variant.
bool wide_m_supported(int M) { return M == 16 || M == 32; }

template <typename REAL>
bool wide_cfg_valid(const Geom &g, const HybridCfg &c) {
  const int seg = c.W * (int)sizeof(REAL);
  if (g.stride == 1 || g.st0 != 1) return false;  // x-neighbouring strided systems
  if (!wide_m_supported(c.M) || (seg != 128 && seg != 256) || c.P < 1 || c.G < 1)
    return false;
  if ((int64_t)c.P * c.M < g.N) return false;
  const int W = c.W;
  const int64_t T = (int64_t)W * c.P;
  const int maxT = c.M == 32 ? WideBounds<REAL, 32>::threads : WideBounds<REAL, 16>::threads;
  if (T > maxT || T % 64 != 0) return false;  // whole waves
  // 32-bit byte offsets: every address a lane forms lies below 4 GiB
  const int64_t nb0 = (g.n0 + W - 1) / W * W;
  const int64_t last = (nb0 - 1) + (g.n1 - 1) * g.st1 + ((int64_t)c.P * c.M - 1) * g.stride;
  if ((last + 1) * (int64_t)sizeof(REAL) > (int64_t)0xFFFFFFFFll) return false;
  return wide_lds_bytes<REAL>(c.M, c.P, seg, 1) <= WIDE_LDS;
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
