// kernels_adi.hip - the ADI heat-diffusion caller of the batched solve.
//
// The reference app (apps/adi/src/adi_cuda.cu:282-326) runs, per timestep,
//   preproc -> tridXmtsvStridedBatch(solvedim 0) -> (solvedim 1)
//           -> tridXmtsvStridedBatchInc(solvedim 2, u += x),
// with a device synchronisation inside every solve. Here the step is four
// stream-ordered launches with no host synchronisation, so a whole step can be
// captured once into a hipGraph and replayed (tridAdiRun*). Unless the caller
// chooses the solves, the array step's sweeps compute the coefficients instead
// of reading them back (array_step_matrix_free).
//
// preproc (reference apps/adi/src/preproc.cu:40-90, CPU apps/adi/src/preproc.hpp:172-214):
//   boundary points:  d = 0, a = 0, b = 1, c = 0
//   interior points:  d = lambda * (sum of the 6 neighbours - 6 u),
//                     a = c = -0.5 lambda, b = 1 + lambda.
// The reference writes the same a, b, c into nine arrays (x, y and z); the
// kernel writes each distinct output pointer once, so a caller may pass one
// coefficient set for all three directions (4 arrays written instead of 10).
// Each thread owns one (i, j) column and walks a chunk of k with the three
// planes k-1, k, k+1 of u in registers.

#include <algorithm>

#include "../../include/tridsolver.h"
#include "../../include/tridsolver_adi.h"
#include "../../include/tridsolver_hip.h"
#include "hybrid_core.hpp"
#include "trid_internal.h"
#include "trid_tune.h"

namespace trid {
namespace {

constexpr int PRE_BX = 64, PRE_BY = 4, PRE_KCHUNK = 16;

template <typename REAL>
struct Coef {
  REAL *a, *b, *c;
};

// Right-hand side at an interior point, from u at the point (c) and its six
// neighbours; the one expression both the preproc kernel and the x sweep
// that computes its own right-hand side evaluate, so they agree bit for bit.
template <typename REAL>
__device__ __forceinline__ REAL adi_rhs(REAL lambda, REAL xm, REAL xp, REAL ym, REAL yp,
                                        REAL zm, REAL zp, REAL c) {
  // lambda * (u[-1] + u[+1] + u[-nx] + u[+nx] + u[-nx*ny] + u[+nx*ny] - 6 u)
  return lambda * (xm + xp + ym + yp + zm + zp - REAL(6) * c);
}

template <typename REAL>
__global__ __launch_bounds__(PRE_BX *PRE_BY) void adi_preproc_kernel(
    REAL lambda, const REAL *__restrict__ u, REAL *__restrict__ du, Coef<REAL> c0,
    Coef<REAL> c1, Coef<REAL> c2, int nx, int ny, int nz) {
  const int i = blockIdx.x * PRE_BX + threadIdx.x;
  const int j = blockIdx.y * PRE_BY + threadIdx.y;
  const int k0 = blockIdx.z * PRE_KCHUNK;
  if (i >= nx || j >= ny || k0 >= nz) return;
  const int k1 = min(nz, k0 + PRE_KCHUNK);
  const int64_t sx = 1, sy = nx, sz = (int64_t)nx * ny;
  const bool edge_ij = (i == 0 || i == nx - 1 || j == 0 || j == ny - 1);
  int64_t ind = (int64_t)k0 * sz + (int64_t)j * sy + i;
  REAL um = 0, uc = u[ind], up = 0;
  if (!edge_ij && k0 > 0) um = u[ind - sz];
  const REAL ca = REAL(-0.5) * lambda, cb = REAL(1) + lambda;
  for (int k = k0; k < k1; ++k, ind += sz) {
    const bool inner = !edge_ij && k > 0 && k < nz - 1;
    if (!edge_ij && k < nz - 1) up = u[ind + sz];
    REAL d, a, b, c;
    if (inner) {
      d = adi_rhs(lambda, u[ind - sx], u[ind + sx], u[ind - sy], u[ind + sy], um, up, uc);
      a = ca;
      b = cb;
      c = ca;
    } else {
      d = 0; a = 0; b = 1; c = 0;
    }
    du[ind] = d;
    if (c0.a) { c0.a[ind] = a; c0.b[ind] = b; c0.c[ind] = c; }
    if (c1.a) { c1.a[ind] = a; c1.b[ind] = b; c1.c[ind] = c; }
    if (c2.a) { c2.a[ind] = a; c2.b[ind] = b; c2.c[ind] = c; }
    um = uc;
    uc = up;
  }
}

template <typename REAL>
tridStatus_t preproc(REAL lambda, const REAL *u, REAL *du, REAL *ax, REAL *bx, REAL *cx,
                     REAL *ay, REAL *by, REAL *cy, REAL *az, REAL *bz, REAL *cz, int nx,
                     int ny, int nz) {
  const bool x_null = !ax && !bx && !cx;  // du only (matrix-free step)
  if (!u || !du || nx < 1 || ny < 1 || nz < 1 || (!x_null && (!ax || !bx || !cx)))
    return TRID_STATUS_INVALID_VALUE;
  // A direction whose three pointers are NULL, or equal to an earlier set,
  // is not written again.
  auto same = [](REAL *p, REAL *q, REAL *r, REAL *P, REAL *Q, REAL *R) {
    return p == P && q == Q && r == R;
  };
  Coef<REAL> c0{ax, bx, cx}, c1{nullptr, nullptr, nullptr}, c2{nullptr, nullptr, nullptr};
  const bool y_null = !ay && !by && !cy, z_null = !az && !bz && !cz;
  if ((!y_null && (!ay || !by || !cy)) || (!z_null && (!az || !bz || !cz)))
    return TRID_STATUS_INVALID_VALUE;
  if (x_null && (!y_null || !z_null)) return TRID_STATUS_INVALID_VALUE;
  if (!y_null && !same(ay, by, cy, ax, bx, cx)) c1 = {ay, by, cy};
  if (!z_null && !same(az, bz, cz, ax, bx, cx) && !same(az, bz, cz, ay, by, cy))
    c2 = {az, bz, cz};
  int dev = 0;
  tridStatus_t s = check_device(&dev);
  if (s != TRID_STATUS_SUCCESS) return s;
  dim3 grid((nx + PRE_BX - 1) / PRE_BX, (ny + PRE_BY - 1) / PRE_BY,
            (nz + PRE_KCHUNK - 1) / PRE_KCHUNK);
  hipLaunchKernelGGL(adi_preproc_kernel<REAL>, grid, dim3(PRE_BX, PRE_BY), 0,
                     current_stream(), lambda, u, du, c0, c1, c2, nx, ny, nz);
  return hipGetLastError() == hipSuccess ? TRID_STATUS_SUCCESS
                                         : TRID_STATUS_EXECUTION_FAILED;
}

// ---------------------------------------------------------------------------
// Matrix-free sweeps for the ADI step. The coefficients preproc would store
// are functions of the grid position only (interior: a = c = -0.5 lambda,
// b = 1 + lambda; any boundary point: a = 0, b = 1, c = 0), so each sweep
// computes them from (i, j, k) with the same expressions in the same
// precision, and reads only du (and u for the z sweep): 16 B per point
// per sweep instead of 40 (FP64). The solve is the Thomas-PCR hybrid of
// hybrid_core.hpp.
// ---------------------------------------------------------------------------
template <typename REAL>
struct AdiCoef {
  REAL lambda;
  int nx, ny, nz, sd;  // sd: direction of the sweep
};

// Coefficients of chunk-order rows r = 0..M-1 of the lane's system.
template <typename REAL, int M, bool CONTIG>
__device__ __forceinline__ void adi_coefs(const hyb::Lane &L, const AdiCoef<REAL> &k,
                                          REAL (&ra)[M], REAL (&rb)[M], REAL (&rc)[M]) {
  const REAL ca = REAL(-0.5) * k.lambda, cb = REAL(1) + k.lambda;
  // the contiguous sweep is the x sweep
  const int sd = CONTIG ? 0 : k.sd;
  // coordinates of the system; the row index runs along direction sd
  int ci, cj, ck;
  if (sd == 0) { cj = (int)L.i0; ck = (int)L.i1; ci = 0; }
  else if (sd == 1) { ci = (int)L.i0; ck = (int)L.i1; cj = 0; }
  else { ci = (int)L.i0; cj = (int)L.i1; ck = 0; }
#pragma unroll
  for (int r = 0; r < M; ++r) {
    const int64_t row = (int64_t)L.p * M + r;
    int i = ci, j = cj, kk = ck;
    if (sd == 0) i = (int)row;
    else if (sd == 1) j = (int)row;
    else kk = (int)row;
    const bool pad = !L.active || row >= L.N;
    const bool edge = i == 0 || i == k.nx - 1 || j == 0 || j == k.ny - 1 || kk == 0 ||
                      kk == k.nz - 1;
    const bool inner = !pad && !edge;
    ra[r] = inner ? ca : REAL(0);
    rb[r] = inner ? cb : REAL(1);
    rc[r] = inner ? ca : REAL(0);
  }
}

template <typename REAL, int M>
struct AdiBounds {  // same register budget as the array-based hybrid kernel
  static constexpr int threads = sizeof(REAL) * M > 64 ? 512 : 1024;
};

// RHS (x sweep only): the right-hand side is not read from d but computed
// from u, as the preproc kernel does: the line's own u through the LDS tile
// for the x neighbours, the four neighbour lines (j +- 1, k +- 1) loaded
// alongside (coalesced; at 256^3 u stays in the last-level cache). d is
// written only.
template <typename REAL, int M, bool INC, bool CONTIG, bool RHS>
__global__ __launch_bounds__((AdiBounds<REAL, M>::threads)) void adi_solve_kernel(
    Geom g, int P, int W, int G, AdiCoef<REAL> kc, REAL *__restrict__ d,
    REAL *__restrict__ u) {
  static_assert(!RHS || (CONTIG && !INC), "right-hand side from u: x sweep only");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const hyb::Lane L = hyb::lane_of<CONTIG>(g, P, W, G);
  const size_t tile_bytes = CONTIG ? sizeof(REAL) * (size_t)W * P * (M + 1) : 0;
  REAL *tile = reinterpret_cast<REAL *>(smem_raw) + (size_t)L.w * P * (M + 1);
  hyb::Ring ring{smem_raw + tile_bytes, (int)(3 * sizeof(REAL) * L.T), 0};
  REAL ra[M], rb[M], rc[M], rd[M];
  if constexpr (RHS) {
    // Every lane loads all of its rows unconditionally, from addresses kept
    // inside the grid: rows past N read row N-1, lanes past the last line
    // read line 0, and lines on the boundary read their own line as the
    // "neighbours". Those values only feed rows whose right-hand side is 0
    // below, so no load needs a branch around it.
    // Offsets are 32-bit byte offsets from u (the launch checks that the
    // grid is below 4 GiB).
    REAL uc[M], ym[M], yp[M], zm[M], zp[M];
    const int j = (int)L.i0, k = (int)L.i1;  // the x line (j, k)
    const bool line_inner = L.active && j > 0 && j < kc.ny - 1 && k > 0 && k < kc.nz - 1;
    const uint32_t sy = line_inner ? (uint32_t)(kc.nx * sizeof(REAL)) : 0u;
    const uint32_t sz = line_inner ? (uint32_t)((uint32_t)kc.nx * kc.ny * sizeof(REAL)) : 0u;
    const uint32_t lbase = L.active ? (uint32_t)L.base : 0u;
    const int n = (int)L.N;
    const char *ub = reinterpret_cast<const char *>(u);
    auto ld = [ub](uint32_t off) { return *reinterpret_cast<const REAL *>(ub + off); };
#pragma unroll
    for (int r = 0; r < M; ++r) {
      const int row = (int)hyb::fetch_row<M, true>(L, r);
      const uint32_t o = (lbase + (uint32_t)(row < n ? row : n - 1)) * (uint32_t)sizeof(REAL);
      uc[r] = ld(o);
      ym[r] = ld(o - sy);
      yp[r] = ld(o + sy);
      zm[r] = ld(o - sz);
      zp[r] = ld(o + sz);
    }
    // x neighbours: the line's u in the tile, row order
#pragma unroll
    for (int r = 0; r < M; ++r) tile[hyb::skew<M>(L.p + L.P * r)] = uc[r];
    __syncthreads();
    const int last = P * M - 1;
#pragma unroll
    for (int r = 0; r < M; ++r) {
      const int row = L.p + L.P * r;
      const bool inner = line_inner && row > 0 && row < L.N - 1;
      const REAL xm = tile[hyb::skew<M>(row > 0 ? row - 1 : 0)];
      const REAL xp = tile[hyb::skew<M>(row < last ? row + 1 : last)];
      rd[r] = inner ? adi_rhs(kc.lambda, xm, xp, ym[r], yp[r], zm[r], zp[r], uc[r]) : REAL(0);
    }
    __syncthreads();  // the tile is reused below
  } else {
    hyb::fetch<M, CONTIG>(L, d, rd, REAL(0), 0, 0, L.N);
  }
  hyb::to_chunk<M, CONTIG>(L, rd, tile);
  adi_coefs<REAL, M, CONTIG>(L, kc, ra, rb, rc);
  REAL x[M];
  hyb::solve_chunk<REAL, M, CONTIG>(L, ring, ra, rb, rc, rd, x);
  hyb::to_fetch<M, CONTIG>(L, x, tile);
  if constexpr (RHS) {  // 32-bit byte offsets, as the loads
    if (!L.active) return;
    const int n = (int)L.N;
    const uint32_t lbase = (uint32_t)L.base;
    char *db = reinterpret_cast<char *>(d);
    auto st = [&](int r) {
      const uint32_t row = (uint32_t)hyb::fetch_row<M, true>(L, r);
      *reinterpret_cast<REAL *>(db + (lbase + row) * (uint32_t)sizeof(REAL)) = x[r];
    };
    if ((int64_t)P * M == L.N) {  // every row of every lane lies inside the line
#pragma unroll
      for (int r = 0; r < M; ++r) st(r);
    } else {
#pragma unroll
      for (int r = 0; r < M; ++r)
        if ((int)hyb::fetch_row<M, true>(L, r) < n) st(r);
    }
  } else if (INC) {
    hyb::store_add<M, CONTIG>(L, u, x);
  } else {
    hyb::store<M, CONTIG>(L, d, x);
  }
}

// ---- sweeps along y and z, several lines per lane ----------------------------
// Every line away from the grid's boundary has the same coefficients, and the lines
// on it have a right-hand side of zeros (the x sweep leaves du = 0 there), which any
// regular coefficients solve to zeros. So a lane takes V neighbouring lines, one 16-byte
// vector per row, and forms the pivots, the forward factors and the reduced
// system's coefficients once for all of them: per point, the right-hand side's
// four multiply-adds and 1/V of the rest (one division per row). Against a line per
// lane (adi_solve_kernel, which was bound by that arithmetic): 200 x 168 x 147, FP32,
// whose arrays the last-level cache holds, y 14.4 to 10.6 us, z 21.5 to 12.1; FP64
// 20.5 to 15.8 and 29.8 to 21.4; 256^3 FP32 28.6 to 22.4 and 57.6 to 32.8, FP64 43.4 to
// 40.3 and 65.9 to 62.1 (402 MB in the z sweep: 6.5 TB/s).
// Lines along y: V x-neighbours of one k. Along z: the plane's lines in memory
// order, n0 = nx * ny (the launch folds them).
constexpr int ADI_VEC_T = 512;  // most threads of a workgroup

// The solve of one chunk of V lines: x[e][r] the right-hand sides in, the solution
// out. middle() runs once the forward sweep is done. WAVE: the lines lie in one wave
// (no ring).
template <typename REAL, int M, int V, bool WAVE, typename Middle>
__device__ __forceinline__ void adi_lines(const hyb::Lane &L, hyb::Ring &ring, REAL lambda, int n,
                                          int row0, REAL (&x)[V][M], Middle middle) {
  // factors: al_r x_{s-1} + x_r + ga_r x_{r+1} = de_r, the chunk's first unknown
  // x_s = f_d - f_a x_{s-1} - f_g x_{r+1} after row r (as hyb::sweep_carry)
  const REAL ca = REAL(-0.5) * lambda, cb = REAL(1) + lambda;
  REAL al[M], ga[M], s[2 + V], m[2 + V], q[2 + V];
  s[0] = 0;
  s[1] = -1;
#pragma unroll
  for (int e = 0; e < V; ++e) s[2 + e] = 0;
#pragma unroll
  for (int r = 0; r < M; ++r) {
    const int row = row0 + r;
    const bool inner = row > 0 && row < n - 1;
    const REAL a = inner ? ca : REAL(0), b = inner ? cb : REAL(1);
    const REAL inv = REAL(1) / (r > 0 ? b - a * ga[r - 1] : b);
    al[r] = r > 0 ? -a * al[r - 1] * inv : a * inv;
    ga[r] = a * inv;
#pragma unroll
    for (int e = 0; e < V; ++e) {
      const REAL v = row < n ? x[e][r] : REAL(0);
      x[e][r] = (r > 0 ? v - a * x[e][r - 1] : v) * inv;
      if (r < M - 1) s[2 + e] = s[2 + e] - s[1] * x[e][r];
    }
    if (r < M - 1) {
      s[0] = s[0] - s[1] * al[r];
      s[1] = -s[1] * ga[r];
    }
  }
  middle();
  // reduced system, as hyb::reduced_solve with V right-hand sides
  hyb::from_above<2 + V>(L, ring, WAVE, s, q);
  {
    const REAL inv = REAL(1) / (REAL(1) - ga[M - 1] * q[0]);
    s[0] = al[M - 1] * inv;
    s[1] = -ga[M - 1] * q[1] * inv;
#pragma unroll
    for (int e = 0; e < V; ++e) s[2 + e] = (x[e][M - 1] - ga[M - 1] * q[2 + e]) * inv;
  }
  for (int h = 1; h < L.P; h <<= 1) {
    hyb::from_both<2 + V>(L, ring, WAVE, h, s, m, q);
    const REAL A = s[0], C = s[1];
    const REAL inv = REAL(1) / (REAL(1) - A * m[1] - C * q[0]);
    s[0] = -inv * A * m[0];
    s[1] = -inv * C * q[1];
#pragma unroll
    for (int e = 0; e < V; ++e) s[2 + e] = inv * (s[2 + e] - A * m[2 + e] - C * q[2 + e]);
  }
  REAL y[V], ym[V];
#pragma unroll
  for (int e = 0; e < V; ++e) y[e] = s[2 + e];
  hyb::from_below<V>(L, ring, WAVE, y, ym);
#pragma unroll
  for (int e = 0; e < V; ++e) x[e][M - 1] = y[e];
#pragma unroll
  for (int r = M - 2; r >= 0; --r) {
#pragma unroll
    for (int e = 0; e < V; ++e) x[e][r] = x[e][r] - al[r] * ym[e] - ga[r] * x[e][r + 1];
  }
}

template <typename REAL, int M, bool INC>
__global__ __launch_bounds__(ADI_VEC_T) void adi_vec_kernel(Geom g, int P, int W, int G,
                                                            REAL lambda, REAL *__restrict__ d,
                                                            REAL *__restrict__ u) {
  constexpr int V = 16 / (int)sizeof(REAL);
  typedef REAL vec __attribute__((ext_vector_type(V)));
  extern __shared__ __align__(16) unsigned char smem_raw[];
  hyb::Lane L{};
  L.P = P; L.W = W; L.T = P * W;
  L.t = threadIdx.x;
  L.p = L.t / W;
  L.w = L.t - L.p * W;
  L.pstep = W;
  hyb::Ring ring{smem_raw, (int)((2 + V) * sizeof(REAL) * L.T), 0};
  const uint32_t groups = (uint32_t)((g.n0 + W * V - 1) / (W * V));
  const uint32_t id = hyb::xcd_remap(blockIdx.x, gridDim.x, G);
  const uint32_t k = id / groups, i0 = ((id - k * groups) * W + L.w) * V;
  const int n = (int)g.N, row0 = L.p * M;
  const bool active = i0 < (uint32_t)g.n0;
  // 32-bit byte offsets (the launch checks the extent); rows past N and lines past
  // n0 are read from inside the array and not stored
  const uint32_t stride = (uint32_t)g.stride * (uint32_t)sizeof(REAL);
  const uint32_t o = ((active ? i0 : 0u) + k * (uint32_t)g.st1) * (uint32_t)sizeof(REAL);
  auto at = [&](REAL *base, int r) {
    const int row = row0 + r;
    return reinterpret_cast<vec *>(reinterpret_cast<char *>(base) + o +
                                   (uint32_t)(row < n ? row : n - 1) * stride);
  };
  REAL x[V][M];
#pragma unroll
  for (int r = 0; r < M; ++r) {
    const vec v = *at(d, r);
#pragma unroll
    for (int e = 0; e < V; ++e) x[e][r] = v[e];
  }

  // u's rows arrive during the reduced solve
  vec uv[INC ? M : 1];
  adi_lines<REAL, M, V, false>(L, ring, lambda, n, row0, x, [&] {
    if (INC) {
#pragma unroll
      for (int r = 0; r < M; ++r) uv[r] = *at(u, r);
    }
  });
  if (!active) return;
#pragma unroll
  for (int r = 0; r < M; ++r) {
    if (row0 + r >= n) break;
    vec v;
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = x[e][r];
    if (INC) *at(u, r) = uv[r] + v;
    else *at(d, r) = v;
  }
}

// Shape of adi_vec_kernel for the sweep along sd = 1 or 2, or false where it does
// not apply: lines in whole vectors, 16-byte aligned, arrays below 4 GiB, a line
// within a workgroup. Eight lanes' vectors a row are a 128-byte line (four: 200 x 168 x
// 147 FP64 66 against 68 us a step, 300^3 412 against 389; sixteen 409). 16 rows per lane
// for the longer lines (us a step at 16 / 8 rows: FP64 300^3 389 / 413, 256^3 150 / 153, 128 x
// 320^2 120 / 133, 64 x 400^2 98 / 110, 128 x 480 x 200 113 / 119; FP32 300^3 139 / 143, 128 x 448
// x 256 71.5 / 73.1, 64 x 400^2 55.5 / 56.5; below the line FP32 256 x 176^2 45.6 / 44.1, 512 x
// 144^2 58.7 / 56.2, FP64 256 x 160^2 70.0 / 70.0).
template <typename REAL>
bool adi_vec_cfg(const REAL *d, const REAL *u, int nx, int ny, int nz, int sd, Geom *g,
                 HybridCfg *cfg) {
  constexpr int V = 16 / (int)sizeof(REAL);
  const int64_t plane = (int64_t)nx * ny, points = plane * nz;
  if (sd == 1) *g = Geom{ny, nx, nx, nz, 1, plane};
  else *g = Geom{nz, plane, plane, 1, 1, 0};
  if (g->n0 % V != 0 || points * (int64_t)sizeof(REAL) > (int64_t)0xffffffff) return false;
  if (((reinterpret_cast<uintptr_t>(d) | reinterpret_cast<uintptr_t>(u)) & 15) != 0) return false;
  cfg->M = g->N > (sizeof(REAL) == 8 ? 192 : 256) ? 16 : 8;
  cfg->P = (int)std::min<int64_t>((g->N + cfg->M - 1) / cfg->M, ADI_VEC_T);
  cfg->W = 8 * cfg->P <= ADI_VEC_T ? 8 : 4;
  cfg->G = 8;
  cfg->V = 0;
  // (HIP grids hold 2^32 work-items)
  const int64_t blocks = (g->n0 + cfg->W * V - 1) / (cfg->W * V) * g->n1;
  return cfg->W * cfg->P <= ADI_VEC_T && (int64_t)cfg->P * cfg->M >= g->N &&
         blocks <= (int64_t)UINT32_MAX / (cfg->W * cfg->P);
}

template <typename REAL, int M, bool INC>
hipError_t launch_adi_vec(const Geom &g, const HybridCfg &cfg, REAL lambda, REAL *d, REAL *u,
                          hipStream_t st) {
  constexpr int V = 16 / (int)sizeof(REAL);
  const int T = cfg.W * cfg.P;
  const size_t lds = hyb::ring_bytes<REAL>(T, 2 + V);
  const int64_t blocks = (g.n0 + cfg.W * V - 1) / (cfg.W * V) * g.n1;
  hipLaunchKernelGGL((adi_vec_kernel<REAL, M, INC>), dim3((unsigned)blocks), dim3(T), lds, st, g,
                     cfg.P, cfg.W, cfg.G, lambda, d, u);
  return hipGetLastError();
}


// The x sweep the same way, every access in chunk order: a lane takes M rows (32
// bytes: two vectors) of LN lines j0 .. j0 + LN - 1 of one k, P lanes of one wave a
// line, 64 / P groups of lines a wave. The right-hand side's neighbours: along x from the
// lanes p-1 and p+1 by ds_bpermute, along y the lines themselves and one on either
// side, along z two more lines each. No LDS tile, no transpose, no barrier. LN = 4 in
// FP64, 2 in FP32 (256^3 step: FP64 LN = 1, 2, 4 172, 154.5, 150 us; FP32 84.5, 80.9, 83.9).
// Against the tiled sweep, FP64, and one line per lane, FP32: 256^3 64.0 to 46.3 and 28.1
// to 24.1 us; 200 x 168 x 147 28.8 to 21.9 and 14.3 to 12.9.
template <typename REAL, int M, int LN>
__global__ __launch_bounds__(64) void adi_xvec_kernel(int nx, int ny, int nz, int P, int G,
                                                      REAL lambda, REAL *__restrict__ d,
                                                      const REAL *__restrict__ u) {
  constexpr int V = 16 / (int)sizeof(REAL), Q = M / V;
  typedef REAL vec __attribute__((ext_vector_type(V)));
  const int W = 64 / P;
  hyb::Lane L{};
  L.P = P; L.W = W; L.T = 64;
  L.t = threadIdx.x;
  L.w = L.t / P;
  L.p = L.t - L.w * P;
  L.pstep = 1;
  hyb::Ring ring{nullptr, 0, 0};  // not used: the systems are wave-local
  const uint32_t groups = (uint32_t)((ny + W * LN - 1) / (W * LN));
  const uint32_t id = hyb::xcd_remap(blockIdx.x, gridDim.x, G);
  const int k = (int)(id / groups);
  const int j0 = ((int)(id - (uint32_t)k * groups) * W + L.w) * LN;
  const bool active = L.w < W && j0 < ny;  // (64 - W * P lanes have no line)
  const bool k_inner = k > 0 && k < nz - 1;
  const int row0 = L.p * M;

  // vector q of line j, plane k + dk: lines and rows outside are read from inside the
  // grid; they feed right-hand sides that are 0 below, or no stored value
  auto ldv = [&](int j, int dk, int q) {
    const int jj = j < 0 ? 0 : j < ny ? j : ny - 1;
    const int row = row0 + q * V < nx ? row0 + q * V : nx - V;
    const uint32_t e = ((uint32_t)(k + dk) * (uint32_t)ny + (uint32_t)jj) * (uint32_t)nx + (uint32_t)row;
    return *reinterpret_cast<const vec *>(reinterpret_cast<const char *>(u) +
                                          e * (uint32_t)sizeof(REAL));
  };
  const int dz = k_inner ? 1 : 0;
  REAL c[LN + 2][M], zm[LN][M], zp[LN][M];
#pragma unroll
  for (int l = 0; l < LN + 2; ++l) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const vec v = ldv(j0 - 1 + l, 0, q);
#pragma unroll
      for (int e = 0; e < V; ++e) c[l][q * V + e] = v[e];
    }
  }
#pragma unroll
  for (int l = 0; l < LN; ++l) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const vec v = ldv(j0 + l, -dz, q), w = ldv(j0 + l, dz, q);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        zm[l][q * V + e] = v[e];
        zp[l][q * V + e] = w[e];
      }
    }
  }

  REAL x[LN][M];
  {
    REAL edge[2 * LN], lo[2 * LN], hi[2 * LN];
#pragma unroll
    for (int l = 0; l < LN; ++l) {
      edge[2 * l] = c[l + 1][M - 1];
      edge[2 * l + 1] = c[l + 1][0];
    }
    hyb::exchange<3, 2 * LN>(L, ring, true, edge, 1, L.p > 0, lo, 1, L.p + 1 < P, hi);
#pragma unroll
    for (int l = 0; l < LN; ++l) {
      const bool line_inner = k_inner && j0 + l > 0 && j0 + l < ny - 1;
#pragma unroll
      for (int r = 0; r < M; ++r) {
        const bool inner = line_inner && row0 + r > 0 && row0 + r < nx - 1;
        const REAL xm = r > 0 ? c[l + 1][r - 1] : lo[2 * l];
        const REAL xp = r < M - 1 ? c[l + 1][r + 1] : hi[2 * l + 1];
        x[l][r] = inner ? adi_rhs(lambda, xm, xp, c[l][r], c[l + 2][r], zm[l][r], zp[l][r],
                                  c[l + 1][r])
                        : REAL(0);
      }
    }
  }
  adi_lines<REAL, M, LN, true>(L, ring, lambda, nx, row0, x, [] {});
  if (!active) return;
#pragma unroll
  for (int l = 0; l < LN; ++l) {
    if (j0 + l >= ny) break;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (row0 + q * V >= nx) break;
      vec v;
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = x[l][q * V + e];
      const uint32_t e = ((uint32_t)k * (uint32_t)ny + (uint32_t)(j0 + l)) * (uint32_t)nx +
                         (uint32_t)(row0 + q * V);
      *reinterpret_cast<vec *>(reinterpret_cast<char *>(d) + e * (uint32_t)sizeof(REAL)) = v;
    }
  }
}

// Lines per lane, and workgroups (one wave each), at M rows per lane.
template <typename REAL>
constexpr int adi_xvec_lines(int M) {
  return sizeof(REAL) == 8 && M == 4 ? 4 : 2;
}
template <typename REAL>
int64_t adi_xvec_blocks(int M, int nx, int ny, int nz) {
  const int lines = 64 / ((nx + M - 1) / M) * adi_xvec_lines<REAL>(M);
  return (int64_t)((ny + lines - 1) / lines) * nz;
}

// Rows per lane of adi_xvec_kernel: 32 bytes, twice that for lines that 64 lanes
// of 32 do not hold; 0 where it does not apply: lines of whole 16-byte vectors,
// aligned, within a wave, arrays below 4 GiB, 2^32 work-items (HIP's grids).
template <typename REAL>
int adi_xvec_rows(const REAL *d, const REAL *u, int nx, int ny, int nz) {
  constexpr int V = 16 / (int)sizeof(REAL);
  if (nx % V != 0 || nx > 64 * 4 * V ||
      (uint64_t)nx * (uint64_t)ny * (uint64_t)nz * sizeof(REAL) > 0xffffffffull ||
      ((reinterpret_cast<uintptr_t>(d) | reinterpret_cast<uintptr_t>(u)) & 15) != 0)
    return 0;
  const int M = nx > 64 * 2 * V ? 4 * V : 2 * V;
  return adi_xvec_blocks<REAL>(M, nx, ny, nz) <= (int64_t)UINT32_MAX / 64 ? M : 0;
}

template <typename REAL, int M, int LN>
hipError_t launch_adi_xvec(REAL lambda, REAL *d, const REAL *u, int nx, int ny, int nz,
                           hipStream_t st) {
  static_assert(LN == adi_xvec_lines<REAL>(M), "the grid is the one that was checked");
  const int P = (nx + M - 1) / M;
  const int64_t blocks = adi_xvec_blocks<REAL>(M, nx, ny, nz);
  hipLaunchKernelGGL((adi_xvec_kernel<REAL, M, LN>), dim3((unsigned)blocks), dim3(64), 0, st, nx,
                     ny, nz, P, 8, lambda, d, u);
  return hipGetLastError();
}

template <typename REAL, int M, bool INC, bool CONTIG, bool RHS = false>
hipError_t launch_adi_solve_m(const Geom &g, const HybridCfg &cfg, const AdiCoef<REAL> &kc,
                              REAL *d, REAL *u, hipStream_t st) {
  const int T = cfg.W * cfg.P;
  size_t lds = hyb::ring_bytes<REAL>(T, 3);
  if (CONTIG) lds += sizeof(REAL) * (size_t)T * (M + 1);
  auto kern = adi_solve_kernel<REAL, M, INC, CONTIG, RHS>;
  static LdsGrant lds_granted;
  {
    hipError_t e = ensure_lds(reinterpret_cast<const void *>(kern), lds, lds_granted);
    if (e != hipSuccess) return e;
  }
  const int64_t blocks = (g.n0 + cfg.W - 1) / cfg.W * g.n1;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(T), lds, st, g, cfg.P, cfg.W, cfg.G,
                     kc, d, u);
  return hipGetLastError();
}

// Shape: the one the array-based solve of this geometry uses (tuned or
// default), with plain loads. Systems longer than one workgroup covers are
// not supported here.
template <typename REAL, bool INC>
bool adi_cfg(int dev, const Geom &g, HybridCfg *cfg) {
  if (!tuned_config<REAL, INC>(dev, g, cfg)) return false;
  if (cfg->V != 0) {
    // a variant shape: keep its chunking (M, P: same arithmetic) with plain
    // loads of 16 systems per workgroup (128-byte FP64 rows, 64-byte FP32
    // rows), which suit a sweep that reads only d. Measured on the 256^3
    // matrix-free step over W in {8, 16, 32, 64} and G in {1, 8, 16}: FP32
    // 0.123 ms at W = 16 against 0.134 at 32 (128-byte rows) and 0.143 at 64;
    // FP64 0.198-0.200 ms at W = 16, 0.205 at 8, 0.24 at 32.
    HybridCfg c = *cfg;
    c.V = 0;
    c.W = 16;
    if (hybrid_cfg_valid<REAL>(g, c)) {
      *cfg = c;
      return true;
    }
    return hybrid_plain_cfg<REAL>(g, cfg);
  }
  return hybrid_cfg_valid<REAL>(g, *cfg) || hybrid_plain_cfg<REAL>(g, cfg);
}

// Shape of the array step's x solve and of the matrix-free x sweep that takes the lines
// adi_xvec_kernel does not. An x line
// fits one workgroup easily; what costs is the PCR across its lanes (a
// division per step and lane), so fewer lanes of more rows than the general
// contiguous default (up to 64 lanes of 4 rows at 256 rows) pay off. Measured
// on 256^3 steps over M in {4, 8, 16}, T in {64, 128, 256}, G in {1, 8}:
// 8 rows per lane, one 64-thread wave per workgroup (matrix-free step FP64
// 0.217 against 0.229-0.233 ms at M = 4; FP32 0.149 against 0.159-0.162).
// G = 1 and 8 time alike; with G = 8 neighbouring x lines run on one XCD,
// so the halo lines the right-hand side reads (j +- 1) hit in its L2
// instead of being fetched again. Re-measured with the branch-free
// right-hand-side loads: M = 16 / T = 64, M = 8 / T = 128, M = 16 / T = 128
// and M = 4 / T = 64 take the FP64 step to 0.206-0.215 ms against 0.200, and
// the FP32 step to 0.134-0.160 ms against 0.133.
template <typename REAL>
struct AdiX {
  static constexpr int M = 8;
  static constexpr int T = 64;
  static constexpr int G = 8;
};

template <typename REAL>
bool adi_x_cfg(const Geom &g, HybridCfg *cfg) {
  HybridCfg c;
  c.M = AdiX<REAL>::M;
  c.P = (int)((g.N + c.M - 1) / c.M);
  c.W = (int)std::max<int64_t>(1, AdiX<REAL>::T / c.P);
  c.G = AdiX<REAL>::G;
  c.V = 0;
  if (g.stride != 1 || !hybrid_cfg_valid<REAL>(g, c)) return false;
  *cfg = c;
  return true;
}

// The x solve of the array step, in the ADI x shape unless the caller has
// forced a shape of its own.
template <typename REAL>
tridStatus_t x_solve(const TridParams *p, const REAL *a, const REAL *b, const REAL *c, REAL *d,
                     const int *dims) {
  Geom g;
  bool empty = false;
  HybridCfg xc;
  const bool shape = forced_config().M == 0 &&
                     make_geom(3, 0, dims, dims, &g, &empty) == TRID_STATUS_SUCCESS &&
                     !empty && adi_x_cfg<REAL>(g, &xc);
  if (shape) tridHipForceHybridConfig(xc.M, xc.P, xc.W, xc.G, xc.V);
  tridStatus_t s;
  if constexpr (sizeof(REAL) == 8) s = tridDmtsvStridedBatch(p, a, b, c, d, 3, 0, dims, dims);
  else s = tridSmtsvStridedBatch(p, a, b, c, d, 3, 0, dims, dims);
  if (shape) tridHipForceHybridConfig(0, 0, 0, 0, 0);
  return s;
}

// The shape of the sweep along sd, or false where no workgroup holds a line or
// the grid of workgroups is too large. The sweep forms coefficients from grid
// coordinates, so it is not split into sub-batches: its grid must fit HIP's
// 2^32 work-items (about 2^35 points at 8 rows per lane, beyond a GPU's
// memory for two arrays).
template <typename REAL, bool INC>
bool adi_sweep_cfg(int dev, const Geom &g, int sd, HybridCfg *cfg) {
  if (!(sd == 0 && adi_x_cfg<REAL>(g, cfg)) && !adi_cfg<REAL, INC>(dev, g, cfg)) return false;
  return (g.n0 + cfg->W - 1) / cfg->W * g.n1 <= (int64_t)UINT32_MAX / (cfg->W * cfg->P);
}

template <typename REAL, bool INC, bool RHS = false>
tridStatus_t adi_sweep(int dev, REAL lambda, REAL *d, REAL *u, int nx, int ny, int nz,
                       int sd) {
  static_assert(!RHS || !INC, "right-hand side from u: x sweep only");
  const int dims[3] = {nx, ny, nz};
  Geom g;
  bool empty = false;
  tridStatus_t s = make_geom(3, sd, dims, dims, &g, &empty);
  if (s != TRID_STATUS_SUCCESS || empty) return s;
  AdiCoef<REAL> kc{lambda, nx, ny, nz, sd};
  hipStream_t st = current_stream();
  const bool contig = sd == 0;
  hipError_t e;
  if (RHS && !contig) return TRID_STATUS_INTERNAL_ERROR;
  // the kernels with several lines per lane choose their own shape; only the general
  // sweep behind them asks for a tuned one
  if constexpr (RHS) {
    constexpr int M = 32 / (int)sizeof(REAL), LN = adi_xvec_lines<REAL>(M);
    const int rows = adi_xvec_rows<REAL>(d, u, nx, ny, nz);
    if (rows != 0) {
      e = rows == M ? launch_adi_xvec<REAL, M, LN>(lambda, d, u, nx, ny, nz, st)
                    : launch_adi_xvec<REAL, 2 * M, adi_xvec_lines<REAL>(2 * M)>(lambda, d, u, nx, ny, nz, st);
      if (e != hipSuccess) {
        record_hip_error(e);
        return TRID_STATUS_EXECUTION_FAILED;
      }
      return TRID_STATUS_SUCCESS;
    }
  } else {
    Geom vg;
    HybridCfg vc;
    if (!contig && adi_vec_cfg<REAL>(d, INC ? u : d, nx, ny, nz, sd, &vg, &vc)) {
      e = vc.M == 16 ? launch_adi_vec<REAL, 16, INC>(vg, vc, lambda, d, u, st)
                     : launch_adi_vec<REAL, 8, INC>(vg, vc, lambda, d, u, st);
      if (e != hipSuccess) {
        record_hip_error(e);
        return TRID_STATUS_EXECUTION_FAILED;
      }
      return TRID_STATUS_SUCCESS;
    }
  }
  HybridCfg cfg;
  if (!adi_sweep_cfg<REAL, INC>(dev, g, sd, &cfg)) return TRID_STATUS_INVALID_VALUE;
  // The right-hand side is computed in the sweep unless FP32 x lines are
  // at 16 rows per lane (they would spill) or the grid is 4 GiB or more (the
  // sweep's loads use 32-bit byte offsets): there preproc writes du and the
  // plain sweep reads it.
  constexpr bool RHS16 = RHS && sizeof(REAL) == 8;
  const bool grid32 =
      (uint64_t)nx * (uint64_t)ny * (uint64_t)nz * sizeof(REAL) < (uint64_t(1) << 32);
  const bool rhs_here = RHS && grid32 && (cfg.M != 16 || RHS16);
  if (RHS && !rhs_here) {
    tridStatus_t sp = preproc<REAL>(lambda, u, d, nullptr, nullptr, nullptr, nullptr, nullptr,
                                    nullptr, nullptr, nullptr, nullptr, nx, ny, nz);
    if (sp != TRID_STATUS_SUCCESS) return sp;
  }
#define TRID_ADI_CASE(MM)                                                                  \
  case MM:                                                                                 \
    if (contig && rhs_here)                                                                \
      e = launch_adi_solve_m<REAL, MM, INC, true, (MM == 16 ? RHS16 : RHS)>(g, cfg, kc, d, \
                                                                              u, st);      \
    else if (contig)                                                                       \
      e = launch_adi_solve_m<REAL, MM, INC, true, false>(g, cfg, kc, d, u, st);            \
    else                                                                                   \
      e = launch_adi_solve_m<REAL, MM, INC, false>(g, cfg, kc, d, u, st);                  \
    break;
  switch (cfg.M) {
    TRID_ADI_CASE(1)
    TRID_ADI_CASE(2)
    TRID_ADI_CASE(4)
    TRID_ADI_CASE(8)
    TRID_ADI_CASE(16)
    default:
      return TRID_STATUS_INVALID_VALUE;
  }
#undef TRID_ADI_CASE
  if (e != hipSuccess) {
    record_hip_error(e);
    return TRID_STATUS_EXECUTION_FAILED;
  }
  return TRID_STATUS_SUCCESS;
}

// Matrix-free step: du = solve_x(rhs(u)) (the right-hand side computed in
// the x sweep); du = solve_y(du); u += solve_z(du). 56 B per point at FP64:
// u read + du written, du read + written, du and u read + u written.
template <typename REAL>
tridStatus_t step_fused(REAL lambda, REAL *u, REAL *du, int nx, int ny, int nz) {
  int dev = 0;
  tridStatus_t s = check_device(&dev);
  if (s == TRID_STATUS_SUCCESS && (nx < 1 || ny < 1 || nz < 1)) s = TRID_STATUS_INVALID_VALUE;
  if (s == TRID_STATUS_SUCCESS)
    s = adi_sweep<REAL, false, true>(dev, lambda, du, u, nx, ny, nz, 0);
  if (s == TRID_STATUS_SUCCESS) s = adi_sweep<REAL, false>(dev, lambda, du, u, nx, ny, nz, 1);
  if (s == TRID_STATUS_SUCCESS) s = adi_sweep<REAL, true>(dev, lambda, du, u, nx, ny, nz, 2);
  return s;
}

// The three coefficient arrays alone, as the preproc kernel writes them: a
// write-bound kernel (24 B per point at FP64), V consecutive points per thread
// as one 16-byte vector per array (VEC: arrays 16-byte aligned; the last
// points, and unaligned arrays, one element at a time).
template <typename REAL, bool VEC>
__global__ __launch_bounds__(256) void adi_coef_kernel(REAL lambda, REAL *__restrict__ a,
                                                       REAL *__restrict__ b,
                                                       REAL *__restrict__ c, int nx, int ny,
                                                       int nz) {
  constexpr int V = VEC ? 16 / (int)sizeof(REAL) : 1;
  const int64_t total = (int64_t)nx * ny * nz;
  const REAL ca = REAL(-0.5) * lambda, cb = REAL(1) + lambda;
  for (int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V; e < total;
       e += (int64_t)gridDim.x * 256 * V) {
    // the first point's coordinates (32-bit divisions where they suffice),
    // the rest by counting on
    int i, j, k;
    if ((uint64_t)e >> 32 == 0) {
      const uint32_t r = (uint32_t)e / (uint32_t)nx;
      i = (int)((uint32_t)e - r * (uint32_t)nx);
      k = (int)(r / (uint32_t)ny);
      j = (int)(r - (uint32_t)k * (uint32_t)ny);
    } else {
      const int64_t r = e / nx;
      i = (int)(e - r * nx);
      k = (int)(r / ny);
      j = (int)(r - (int64_t)k * ny);
    }
    REAL va[V], vb[V];
#pragma unroll
    for (int q = 0; q < V; ++q) {
      const bool inner = i > 0 && i < nx - 1 && j > 0 && j < ny - 1 && k > 0 && k < nz - 1;
      va[q] = inner ? ca : REAL(0);
      vb[q] = inner ? cb : REAL(1);
      if (++i == nx) {
        i = 0;
        if (++j == ny) { j = 0; ++k; }
      }
    }
    if constexpr (VEC) {
      typedef REAL vec __attribute__((ext_vector_type(V)));
      if (e + V <= total) {
        vec x, y;
#pragma unroll
        for (int q = 0; q < V; ++q) { x[q] = va[q]; y[q] = vb[q]; }
        __builtin_nontemporal_store(x, reinterpret_cast<vec *>(a + e));
        __builtin_nontemporal_store(y, reinterpret_cast<vec *>(b + e));
        __builtin_nontemporal_store(x, reinterpret_cast<vec *>(c + e));
        continue;
      }
    }
#pragma unroll
    for (int q = 0; q < V; ++q) {
      if (e + q < total) {
        a[e + q] = va[q];
        b[e + q] = vb[q];
        c[e + q] = va[q];
      }
    }
  }
}

template <typename REAL>
tridStatus_t write_coefs(REAL lambda, REAL *a, REAL *b, REAL *c, int nx, int ny, int nz) {
  auto al16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const bool vec = al16(a) && al16(b) && al16(c);
  const int64_t per = 256 * (vec ? 16 / (int64_t)sizeof(REAL) : 1);
  const int64_t blocks =
      std::min<int64_t>(((int64_t)nx * ny * nz + per - 1) / per, int64_t(1) << 22);
  if (vec)
    hipLaunchKernelGGL((adi_coef_kernel<REAL, true>), dim3((unsigned)blocks), dim3(256), 0,
                       current_stream(), lambda, a, b, c, nx, ny, nz);
  else
    hipLaunchKernelGGL((adi_coef_kernel<REAL, false>), dim3((unsigned)blocks), dim3(256), 0,
                       current_stream(), lambda, a, b, c, nx, ny, nz);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    record_hip_error(e);
    return TRID_STATUS_EXECUTION_FAILED;
  }
  return TRID_STATUS_SUCCESS;
}

// Whether the array step runs as the coefficient arrays written once, then
// matrix-free sweeps: the coefficients that preproc stores are functions of
// the grid position, so sweeps that compute them need not read them back, and
// the x sweep computes the right-hand side that preproc would store. u, du,
// a, b and c end as preproc and the three array solves leave them, for 24 B per
// point once per call and 56 per step (FP64) instead of 168 per step. Calls
// that choose the solves' algorithm or shape (ctx->opts 1 or 2, a forced
// shape), grids with a line that no workgroup holds, and calls the argument
// checks refuse keep preproc and the array solves.
template <typename REAL>
bool array_step_matrix_free(const TridParams *ctx, const REAL *u, const REAL *du, const REAL *a,
                            const REAL *b, const REAL *c, int nx, int ny, int nz) {
  if (!u || !du || !a || !b || !c || nx < 1 || ny < 1 || nz < 1) return false;
  if (forced_config().M != 0) return false;
  for (int k = 0; ctx && k < 3; ++k)
    if (ctx->opts[k] == 1 || ctx->opts[k] == 2) return false;
  int dev = 0;
  if (check_device(&dev) != TRID_STATUS_SUCCESS) return false;
  const int dims[3] = {nx, ny, nz};
  for (int sd = 0; sd < 3; ++sd) {
    Geom g;
    HybridCfg cfg;
    bool empty = false;
    if (make_geom(3, sd, dims, dims, &g, &empty) != TRID_STATUS_SUCCESS || empty) return false;
    // (as adi_sweep chooses)
    Geom vg;
    if (sd == 0 ? adi_xvec_rows<REAL>(du, u, nx, ny, nz) != 0
                : adi_vec_cfg<REAL>(du, sd == 2 ? u : du, nx, ny, nz, sd, &vg, &cfg))
      continue;
    const bool ok = sd == 2 ? adi_sweep_cfg<REAL, true>(dev, g, sd, &cfg)
                            : adi_sweep_cfg<REAL, false>(dev, g, sd, &cfg);
    if (!ok) return false;
  }
  return true;
}

template <typename REAL, bool INC>
tridStatus_t array_solve(const TridParams *p, const REAL *a, const REAL *b, const REAL *c,
                         REAL *d, REAL *u, int sd, const int *dims) {
  return solve<REAL, INC>(p, a, b, c, d, u, 3, sd, dims, dims);
}

// One step by preproc and the three array solves, stream-ordered, no host
// synchronisation (ctx->sync forced to 0 for the solves; the caller decides
// when to wait).
template <typename REAL>
tridStatus_t step_arrays(const TridParams *ctx, REAL lambda, REAL *u, REAL *du, REAL *a, REAL *b,
                         REAL *c, int nx, int ny, int nz) {
  TridParams p = ctx ? *ctx : TridParams{nullptr, {0, 0, 0}, 0};
  p.sync = 0;
  const int dims[3] = {nx, ny, nz};
  tridStatus_t s = preproc<REAL>(lambda, u, du, a, b, c, nullptr, nullptr, nullptr, nullptr,
                                 nullptr, nullptr, nx, ny, nz);
  if (s == TRID_STATUS_SUCCESS) s = x_solve<REAL>(&p, a, b, c, du, dims);
  if (s == TRID_STATUS_SUCCESS)
    s = array_solve<REAL, false>(&p, a, b, c, du, nullptr, 1, dims);
  if (s == TRID_STATUS_SUCCESS) s = array_solve<REAL, true>(&p, a, b, c, du, u, 2, dims);
  return s;
}

template <typename REAL>
tridStatus_t step(const TridParams *ctx, REAL lambda, REAL *u, REAL *du, REAL *a, REAL *b,
                  REAL *c, int nx, int ny, int nz) {
  if (!array_step_matrix_free<REAL>(ctx, u, du, a, b, c, nx, ny, nz))
    return step_arrays<REAL>(ctx, lambda, u, du, a, b, c, nx, ny, nz);
  const tridStatus_t s = write_coefs<REAL>(lambda, a, b, c, nx, ny, nz);
  return s == TRID_STATUS_SUCCESS ? step_fused<REAL>(lambda, u, du, nx, ny, nz) : s;
}

template <typename REAL>
tridStatus_t run(const TridParams *ctx, REAL lambda, REAL *u, REAL *du, REAL *a, REAL *b,
                 REAL *c, int nx, int ny, int nz, int iters, int use_graph) {
  // a == NULL selects the matrix-free step. The array step's coefficient
  // arrays do not change from step to step: where its sweeps are matrix-free,
  // they are written once before the steps. 256^3, per step, against
  // preproc and the array solves in every step: FP64 0.150 against 0.605 ms,
  // FP32 0.081 against 0.276; a call of 20 FP64 steps 3.10 against 12.3 ms.
  if (iters < 0) return TRID_STATUS_INVALID_VALUE;
  hipStream_t st = current_stream();
  tridStatus_t s = TRID_STATUS_SUCCESS;
  const bool arrays = a && !(iters > 0 && array_step_matrix_free<REAL>(ctx, u, du, a, b, c, nx,
                                                                      ny, nz));
  auto one_step = [&]() {
    return arrays ? step_arrays<REAL>(ctx, lambda, u, du, a, b, c, nx, ny, nz)
                  : step_fused<REAL>(lambda, u, du, nx, ny, nz);
  };
  if (a && !arrays) {
    s = write_coefs<REAL>(lambda, a, b, c, nx, ny, nz);
    if (s != TRID_STATUS_SUCCESS) return s;
  }
  const bool sync = ctx == nullptr || ctx->sync != 0;
  // use_graph: a step of array solves is captured once and replayed. The
  // matrix-free sweeps are launched in either case: at three launches a step
  // the replays are no faster (32^3 FP32, 200 steps: 4.54 ms with one step
  // captured and replayed, 3.37 with graphs of 20 steps, 3.27 launched; 256^3
  // FP64, 20 steps 3.66 against 3.47 ms), and capturing costs about 110 us a
  // call. The call waits for the steps as it does for replays.
  if (!use_graph || iters == 0 || !arrays) {
    for (int it = 0; it < iters && s == TRID_STATUS_SUCCESS; ++it) s = one_step();
    if (use_graph && iters > 0 && hipStreamSynchronize(st) != hipSuccess &&
        s == TRID_STATUS_SUCCESS)
      s = TRID_STATUS_EXECUTION_FAILED;
  } else {
    // Capture one step on a private stream (the null stream cannot be
    // captured), replay it `iters` times on the caller's stream.
    int dev = 0;
    if ((s = check_device(&dev)) != TRID_STATUS_SUCCESS) return s;
    hipStream_t cap = nullptr;
    if (hipStreamCreateWithFlags(&cap, hipStreamNonBlocking) != hipSuccess)
      return TRID_STATUS_EXECUTION_FAILED;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    void *prev = nullptr;
    tridHipGetStream(&prev);
    {
      // Solves that take the per-lane path (ctx->opts 1 or 2, or systems
      // longer than one workgroup holds) need a workspace, which cannot be
      // allocated during capture: reserve it for the capture stream now.
      const int dims[3] = {nx, ny, nz};
      size_t need = 0;
      HybridCfg xc;
      Geom gx;
      bool empty = false;
      const bool x_forced = forced_config().M == 0 &&
                            make_geom(3, 0, dims, dims, &gx, &empty) == TRID_STATUS_SUCCESS &&
                            !empty && adi_x_cfg<REAL>(gx, &xc);
      if (!x_forced) need = lane_workspace_need<REAL, false>(dev, ctx, 3, 0, dims, dims);
      need = std::max(need, lane_workspace_need<REAL, false>(dev, ctx, 3, 1, dims, dims));
      need = std::max(need, lane_workspace_need<REAL, true>(dev, ctx, 3, 2, dims, dims));
      void *ws = nullptr;
      if (need > 0) s = get_workspace(dev, cap, need, &ws);
    }
    if (s == TRID_STATUS_SUCCESS) {
      if (hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal) != hipSuccess) {
        s = TRID_STATUS_EXECUTION_FAILED;
      } else {
        tridHipSetStream(cap);
        tridStatus_t s_step = one_step();
        tridHipSetStream(prev);
        hipError_t e = hipStreamEndCapture(cap, &graph);
        if (s_step != TRID_STATUS_SUCCESS) s = s_step;
        else if (e != hipSuccess) s = TRID_STATUS_EXECUTION_FAILED;
      }
    }
    if (s == TRID_STATUS_SUCCESS &&
        hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess)
      s = TRID_STATUS_EXECUTION_FAILED;
    for (int it = 0; it < iters && s == TRID_STATUS_SUCCESS; ++it)
      if (hipGraphLaunch(exec, st) != hipSuccess) s = TRID_STATUS_EXECUTION_FAILED;
    // Wait for the replays before the executable graph is destroyed.
    if (exec) {
      if (hipStreamSynchronize(st) != hipSuccess && s == TRID_STATUS_SUCCESS)
        s = TRID_STATUS_EXECUTION_FAILED;
      (void)hipGraphExecDestroy(exec);
    }
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipStreamDestroy(cap);
    drop_stream_workspaces(dev, cap);
  }
  if (s == TRID_STATUS_SUCCESS && sync && hipStreamSynchronize(st) != hipSuccess)
    s = TRID_STATUS_EXECUTION_FAILED;
  return s;
}

}  // namespace
}  // namespace trid

using namespace trid;

EXTERN_C tridStatus_t tridAdiPreprocD(double lambda, const double *u, double *du,
                                      double *ax, double *bx, double *cx, double *ay,
                                      double *by, double *cy, double *az, double *bz,
                                      double *cz, int nx, int ny, int nz) {
  return preproc<double>(lambda, u, du, ax, bx, cx, ay, by, cy, az, bz, cz, nx, ny, nz);
}

EXTERN_C tridStatus_t tridAdiPreprocS(float lambda, const float *u, float *du, float *ax,
                                      float *bx, float *cx, float *ay, float *by,
                                      float *cy, float *az, float *bz, float *cz, int nx,
                                      int ny, int nz) {
  return preproc<float>(lambda, u, du, ax, bx, cx, ay, by, cy, az, bz, cz, nx, ny, nz);
}

EXTERN_C tridStatus_t tridAdiStepD(const TridParams *ctx, double lambda, double *u,
                                   double *du, double *a, double *b, double *c, int nx,
                                   int ny, int nz) {
  tridStatus_t s = step<double>(ctx, lambda, u, du, a, b, c, nx, ny, nz);
  if (s == TRID_STATUS_SUCCESS && (ctx == nullptr || ctx->sync != 0) &&
      hipStreamSynchronize(current_stream()) != hipSuccess)
    s = TRID_STATUS_EXECUTION_FAILED;
  return s;
}

EXTERN_C tridStatus_t tridAdiStepS(const TridParams *ctx, float lambda, float *u, float *du,
                                   float *a, float *b, float *c, int nx, int ny, int nz) {
  tridStatus_t s = step<float>(ctx, lambda, u, du, a, b, c, nx, ny, nz);
  if (s == TRID_STATUS_SUCCESS && (ctx == nullptr || ctx->sync != 0) &&
      hipStreamSynchronize(current_stream()) != hipSuccess)
    s = TRID_STATUS_EXECUTION_FAILED;
  return s;
}

EXTERN_C tridStatus_t tridAdiStepFusedD(double lambda, double *u, double *du, int nx, int ny,
                                        int nz) {
  if (!u || !du) return TRID_STATUS_INVALID_VALUE;
  return step_fused<double>(lambda, u, du, nx, ny, nz);
}

EXTERN_C tridStatus_t tridAdiStepFusedS(float lambda, float *u, float *du, int nx, int ny,
                                        int nz) {
  if (!u || !du) return TRID_STATUS_INVALID_VALUE;
  return step_fused<float>(lambda, u, du, nx, ny, nz);
}

EXTERN_C tridStatus_t tridAdiRunFusedD(const TridParams *ctx, double lambda, double *u,
                                       double *du, int nx, int ny, int nz, int iters,
                                       int use_graph) {
  if (!u || !du) return TRID_STATUS_INVALID_VALUE;
  return run<double>(ctx, lambda, u, du, nullptr, nullptr, nullptr, nx, ny, nz, iters,
                     use_graph);
}

EXTERN_C tridStatus_t tridAdiRunFusedS(const TridParams *ctx, float lambda, float *u, float *du,
                                       int nx, int ny, int nz, int iters, int use_graph) {
  if (!u || !du) return TRID_STATUS_INVALID_VALUE;
  return run<float>(ctx, lambda, u, du, nullptr, nullptr, nullptr, nx, ny, nz, iters,
                    use_graph);
}

EXTERN_C tridStatus_t tridAdiRunD(const TridParams *ctx, double lambda, double *u,
                                  double *du, double *a, double *b, double *c, int nx,
                                  int ny, int nz, int iters, int use_graph) {
  if (!a || !b || !c) return TRID_STATUS_INVALID_VALUE;
  return run<double>(ctx, lambda, u, du, a, b, c, nx, ny, nz, iters, use_graph);
}

EXTERN_C tridStatus_t tridAdiRunS(const TridParams *ctx, float lambda, float *u, float *du,
                                  float *a, float *b, float *c, int nx, int ny, int nz,
                                  int iters, int use_graph) {
  if (!a || !b || !c) return TRID_STATUS_INVALID_VALUE;
  return run<float>(ctx, lambda, u, du, a, b, c, nx, ny, nz, iters, use_graph);
}
