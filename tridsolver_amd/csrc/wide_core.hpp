// wide_core.hpp - device and host parts shared by the strided kernels that stage
// one operand in LDS (kernels_wide.hip, the adjoint in kernels_adjoint.hip).
// What bounds such a kernel, and why it is split as it is, stands at the top of
// kernels_wide.hip.
#pragma once

#include "hybrid_core.hpp"
#include "trid_internal.h"

namespace trid {
namespace wide {

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
// src on) are masked off. SHIFT 1: tile row r gets src's row r - 1 (row 0, of
// which the system has none, its own row 0).
template <typename REAL, int M, int SEG, int CH, bool WHOLE, int SHIFT = 0>
__device__ __forceinline__ void wide_stage(const REAL *src, uint32_t tile, int row0, int lane,
                                           uint32_t row_bytes, int N, int64_t nsys) {
  constexpr int K = 256 / SEG;
  const hyb::Stage stage;
  const int sub = (lane * 4) / SEG;
  const uint32_t byte = (uint32_t)(lane * 4) % SEG;
  if constexpr (WHOLE) {
    const uint32_t o = (uint32_t)(row0 + sub) * row_bytes + byte;
#pragma unroll
    for (int r = 0; r < M; r += K)
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        uint32_t off = o + (uint32_t)(q * M + r) * row_bytes;
        if (SHIFT) off -= r == 0 && q == 0 && row0 + sub == 0 ? 0u : row_bytes;
        stage.dword(tile + q * wide_chunk_bytes(M, SEG) + r * SEG, src, off);
      }
  } else {
    if ((int)byte / (int)sizeof(REAL) >= nsys) return;
    for (int r = 0; r < M; r += K)
      for (int q = 0; q < CH; ++q) {
        const int row = row0 + q * M + r + sub;
        if (row < N)
          stage.dword(tile + q * wide_chunk_bytes(M, SEG) + r * SEG, src,
                      (uint32_t)(SHIFT && row > 0 ? row - 1 : row) * row_bytes + byte);
      }
  }
}

// (i) and (ii) on one wave's chunks, loads included: (b, c, d) -> (al, ga, de)
// of the lane's M rows, and x_s = f_d - f_a x_{s-1} - f_g x_e. WHOLE: every row
// of every lane lies inside an existing system, so every load is unmasked and
// the sweep of row r waits for the loads of rows 0..r only (global->LDS and
// register loads complete in order; the `a` rows come first). Otherwise rows
// past N, and systems past n0, become identity rows (their tile slots, which no
// global->LDS load writes, are set to 0 here). SHIFT 0: the system of a (below
// the diagonal), b, c (above it). SHIFT 1: that of the transpose of a matrix
// with upper diagonal a0 and lower diagonal c, i.e. row n has a0[n-1] below and
// c[n+1] above the diagonal.
template <typename REAL, int M, int SEG, int CH, bool WHOLE, bool NT, int SHIFT = 0>
__device__ __forceinline__ void wide_sweep(const REAL *a0, uint32_t tile, int wave_row0, int lane,
                                           int N, int64_t nsys, uint32_t os, uint32_t ob,
                                           int row0, int rows, REAL *as,
                                           const REAL *__restrict__ b,
                                           const REAL *__restrict__ c, const REAL *d,
                                           REAL (&rb)[M],
                                           REAL (&rc)[M], REAL (&rd)[M], REAL &f_d, REAL &f_a,
                                           REAL &f_g) {
  constexpr int W = WideShape<REAL, SEG>::W;
  wide_stage<REAL, M, SEG, CH, WHOLE, SHIFT>(a0, tile, wave_row0, lane, os, N, nsys);
  ob = hyb::loads_after_stage(ob);
  auto at = [](const REAL *p, uint32_t off) -> REAL {
    return hyb::ld<NT>(reinterpret_cast<const REAL *>(reinterpret_cast<const char *>(p) + off));
  };
#pragma unroll
  for (int r = 0; r < M; ++r) {
    const uint32_t o = ob + (uint32_t)r * os;
    if constexpr (WHOLE) {
      rb[r] = at(b, o);
      // (c of the system's last row is not used: no row below it is read)
      rc[r] = at(c, !SHIFT ? o : r < M - 1 || rows > M ? o + os : o);
      rd[r] = at(d, o);
      __builtin_amdgcn_sched_barrier(0);  // the loads stay in row order
    } else {
      rb[r] = r < rows ? at(b, o) : REAL(1);
      rc[r] = r + 1 < rows ? at(c, SHIFT ? o + os : o) : REAL(0);
      rd[r] = r < rows ? at(d, o) : REAL(0);
      if (r >= rows) as[r * W] = REAL(0);
    }
  }
  if constexpr (WHOLE) hyb::stage_done(rb[0]);
  else hyb::stage_wait_all();
  // (a of the system's first row is not used, nor c of its last)
  hyb::sweep_carry<REAL, M>(
      [&](int r) { return r == 0 && row0 == 0 ? REAL(0) : as[r * W]; }, rb, rc, rd, f_d, f_a, f_g);
  if (WHOLE && rows == M) rc[M - 1] = REAL(0);
}

// Whether a workgroup of the shape holds the system: whole waves of W
// x-neighbouring strided systems, 32-bit byte offsets (every address a lane
// forms lies below 4 GiB), the tile and a one-slot ring within LDS.
template <typename REAL>
bool wide_shape_fits(const Geom &g, const HybridCfg &c) {
  const int seg = c.W * (int)sizeof(REAL);
  if (g.stride == 1 || g.st0 != 1) return false;
  if ((c.M != 16 && c.M != 32) || (seg != 128 && seg != 256) || c.P < 1 || c.G < 1) return false;
  if ((int64_t)c.P * c.M < g.N) return false;
  const int64_t T = (int64_t)c.W * c.P;
  const int maxT = c.M == 32 ? WideBounds<REAL, 32>::threads : WideBounds<REAL, 16>::threads;
  if (T > maxT || T % 64 != 0) return false;
  const int64_t nb0 = (g.n0 + c.W - 1) / c.W * c.W;
  const int64_t last = (nb0 - 1) + (g.n1 - 1) * g.st1 + ((int64_t)c.P * c.M - 1) * g.stride;
  if ((last + 1) * (int64_t)sizeof(REAL) > (int64_t)0xFFFFFFFFll) return false;
  return wide_lds_bytes<REAL>(c.M, c.P, seg, 1) <= WIDE_LDS;
}

// Whether workgroups of 256-byte rows are enough to keep the CUs busy: half a
// workgroup more than one per CU (130 x 100 x 280 FP64 z, 500 of them: 37 us
// against 46 with 128-byte rows; 130 x 512 x 64 y, 320: 52 against 47; 64 x 500 x
// 150 y, 300: 45 against 39).
template <typename REAL>
bool wide_many_groups(const Geom &g, int64_t least = 384) {
  return (g.n0 * (int64_t)sizeof(REAL) + 255) / 256 * g.n1 >= least;
}

// Whether 256-byte rows suit the lines: not where a line is an odd number of 128-byte
// segments, so that its last 256-byte group is half empty, and that counts: lines of
// one or three, and of up to 23 with systems whose 256-byte group fills a CU (256
// against 128 bytes, FP64: 16 x 500 x 1100 y 93 against 61 us, 48 x 400 x 550 y 92 against 72,
// 104 x 500 x 275 y 153 against 128; 130 x 100 x 280 z the other way, 37 against 46; FP32:
// 32 x 300 x 1100 y 62 against 42, 224 x 300 x 275 y 79 against 69, 288 x 500 x 220 y 110
// against 122). FP64 systems of up to 32 rows leave half the lanes of a 128-byte group
// idle as well (16 x 32 x 1100 y 8.3 against 8.8).
template <typename REAL>
bool wide_whole_segments(const Geom &g) {
  const int64_t segs = (g.n0 * (int64_t)sizeof(REAL) + 127) / 128;
  if (segs % 2 == 0) return true;
  if (sizeof(REAL) == 8) return g.N <= 32 || segs >= 25 || (segs >= 5 && g.N <= 320);
  return segs >= 9 || (segs >= 5 && g.N > 384);
}

// Whether every row of the batch starts on a 128-byte line, with `low` the
// arrays' addresses or-ed together. Kernels take nontemporal access then, and
// plain access where rows are misaligned: a workgroup's segments share lines
// with the neighbouring workgroups' there, and only plain stores let an XCD's L2
// join the two partial lines (777 x 300 x 250 FP64 along y: 560 MB written with
// nontemporal stores, 472 with plain ones, 466 algorithmic).
template <typename REAL>
bool wide_rows_aligned(const Geom &g, uintptr_t low) {
  low |= (uintptr_t)(g.stride * (int64_t)sizeof(REAL));
  if (g.n1 > 1) low |= (uintptr_t)(g.st1 * (int64_t)sizeof(REAL));
  return low % 128 == 0;
}

}  // namespace wide
}  // namespace trid
