// svd.hip -- batched Jacobi SVD of the Casorati matrices (arma::svd_econ at
// src/svt.hpp:111).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <limits>

#include "common.hpp"
#include "kernels.hpp"
#include "lanes.hpp"
#include "shapes.hpp"

namespace pgsvt {

// --------------------------------------------------- batched Jacobi SVD --
// One-sided (Hestenes) Jacobi on the m x n Casorati matrix of each patch
// (arma::svd_econ at src/svt.hpp:111).  Output per patch, sorted by
// descending singular value: V^T (n x n), W^T = (X V)^T (n x m) and s (n).
// A group of L lanes holds one matrix; lane l owns rows l, l + L, l + 2L ...
// of X (R rows), so the rotation parameters, which every lane of the group
// computes, are shared by R rows.  Column dot products
// are a sum over the lane's rows, then a butterfly across the group (DPP
// inside a 16-lane row, lane swaps for 32/64-lane groups).  Every lane ends
// the butterfly with the bit-identical sum, so all lanes apply the same
// rotation.  Column norms are carried through the sweep with the exact
// Jacobi update (a -= t c, b += t c) and refreshed at the start of every
// sweep, so a pair costs one butterfly.  V is not accumulated: after
// convergence V = X^T W S^-2 (X reloaded), row by row.  Its error in a
// reconstruction d_r w_r v_r^T stays at eps * s_max (that of v_r is
// eps * s_max / s_r, times |w_r| = s_r); ranks with s_r <= eps * s_max get
// v_r = 0, below that level too.
// reciprocal, square root and reciprocal square root: the hardware
// approximations in FP32, IEEE-correct operations in FP64
__device__ __forceinline__ float rcp_(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double rcp_(double x) { return 1.0 / x; }
__device__ __forceinline__ float sqrt_(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ double sqrt_(double x) { return sqrt(x); }
__device__ __forceinline__ float rsq_(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double rsq_(double x) { return 1.0 / sqrt(x); }

// RT: the window length n = nw is known at run time only (n <= N): the
// matrix is held as N columns, the last N - n zero, and every loop stops at
// n (uniform branches); the stored layout follows n.
template <int BS, int N, int L, class T, bool RT = false>
__global__ __launch_bounds__(256) void k_svd(const T* __restrict__ u32, const int32_t* __restrict__ pos,
                                             const uint32_t* __restrict__ sel, uint32_t nvar, uint32_t nvar_stored,
                                             uint32_t p_sel, uint32_t p_all, uint32_t nr, uint32_t fs, uint32_t nw,
                                             uint32_t vol, uint32_t lim, uint32_t fstride, int max_sweeps, T tol2,
                                             T* __restrict__ factors, uint32_t* __restrict__ stats) {
  constexpr int M = BS * BS, R = (M + L - 1) / L, SRN = (N + 3) & ~3;
  const int n = RT ? (int)nw : N;
  const int SR = RT ? ((n + 3) & ~3) : SRN;
  const uint32_t b = blockIdx.y;
  const int lane = threadIdx.x % L;
  const uint32_t g = (blockIdx.x * blockDim.x + threadIdx.x) / L;
  const uint32_t var = g / p_sel, p = g % p_sel;
  const bool valid = var < nvar;  // uniform per group
  const uint32_t it = valid ? (p_sel == p_all ? p : sel[p]) : 0;  // step 1: identity selection

  const T* U = u32 + ((size_t)b * nvar_stored + (valid ? var : 0)) * vol;
  // the lane's rows of the Casorati matrix X (column k: frame k's patch)
  auto load_x = [&](T (&y)[R][N]) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const bool kin = !RT || k < n;
      const int32_t pk = (valid && kin) ? pos[((size_t)b * nw + k) * p_all + it] : 0;
      const uint32_t row = min((uint32_t)(pk & 0xffff), lim), col = min((uint32_t)(pk >> 16), lim);
#pragma unroll
      for (int h = 0; h < R; ++h) {
        const int q = lane + L * h;
        y[h][k] = (valid && kin && q < M) ? U[(size_t)k * fs + (row + q % BS) + (size_t)nr * (col + q / BS)] : T(0);
      }
    }
  };
  T x[R][N];
  load_x(x);

  T a[N];
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      T t = x[0][k] * x[0][k];
#pragma unroll
      for (int h = 1; h < R; ++h) t = fma(x[h][k], x[h][k], t);
      a[k] = group_sum<L>(t);
    }
    // sum of t^2 over the sweep: zero exactly when no pair rotated.  A
    // floating-point chain (never reassociated) keeps this in one register.
    T tsum = T(0);
#pragma unroll
    for (int i = 0; i < N - 1; ++i) {
      if (RT && i + 1 >= n) break;
#pragma unroll
      for (int j = i + 1; j < N; ++j) {
        if (RT && j >= n) break;
        // rotation zeroing the (i, j) inner product: zeta = (b - a) / 2c,
        // t = sign(zeta) / (|zeta| + sqrt(1 + zeta^2)), cs = 1/sqrt(1+t^2)
        T cp = x[0][i] * x[0][j];
#pragma unroll
        for (int h = 1; h < R; ++h) cp = fma(x[h][i], x[h][j], cp);
        const T c = group_sum<L>(cp);
        const bool rot = c * c > tol2 * a[i] * a[j];
        // Late in the iteration most pairs rotate in none of the wave's
        // matrices; the update is then the identity (t = 0, cs = 1, sn = 0
        // reproduce every value exactly) and is skipped for the whole wave.
        if (!__any(rot)) continue;
        const T zeta = (a[j] - a[i]) * rcp_(c + c);
        const T den = fabs(zeta) + sqrt_(fma(zeta, zeta, T(1)));
        const T t = rot ? copysign(rcp_(den), zeta) : T(0);
        const T cs = rsq_(fma(t, t, T(1)));
        const T sn = cs * t;
#pragma unroll
        for (int h = 0; h < R; ++h) {
          const T xi = x[h][i], xj = x[h][j];
          x[h][i] = cs * xi - sn * xj;
          x[h][j] = sn * xi + cs * xj;
        }
        a[i] = fma(-t, c, a[i]);
        a[j] = fma(t, c, a[j]);
        tsum = fma(t, t, tsum);
      }
    }
    if (!__any(tsum > T(0))) break;
  }
  if (stats && lane == 0 && valid) atomicMax(stats, (uint32_t)sweep + 1);
  // final column norms (identical in every lane of the group)
#pragma unroll
  for (int k = 0; k < N; ++k) {
    T t = x[0][k] * x[0][k];
#pragma unroll
    for (int h = 1; h < R; ++h) t = fma(x[h][k], x[h][k], t);
    a[k] = group_sum<L>(t);
  }
  if (!valid) return;
  // Store in descending singular-value order, transposed: row r of V^T is
  // the right singular vector of the r-th largest singular value (row
  // stride SR, padded with zeros), row r of W^T is the matching column of
  // W = X V = U S (the rotated Casorati columns), then the sorted values.
  // rank(l) counts the values that sort before column l (ties by index).
  T* F = factors + (((size_t)b * nvar_stored + var) * p_sel + p) * fstride;
  T* FW = F + n * SR;
  T* FS = FW + n * M;
  // ranks (< N <= 32) packed in bytes, four per register: the epilogue
  // keeps X, 1/s^2 and the ranks live, and unpacked ranks would cost the
  // kernel a wave per SIMD
  uint32_t rk8[(N + 3) / 4];
#pragma unroll
  for (int i = 0; i < (N + 3) / 4; ++i) rk8[i] = 0u;
  auto rank_of = [&](int l) -> int { return (int)((rk8[l / 4] >> (8 * (l % 4))) & 0xffu); };
  T inv[N];
  T amax = a[0];
#pragma unroll
  for (int k = 1; k < N; ++k) amax = fmax(amax, a[k]);
  constexpr T eps = std::numeric_limits<T>::epsilon();
#pragma unroll
  for (int l = 0; l < N; ++l) {
    // (RT: the zero columns past n rank after every real one)
    uint32_t rl = 0;
#pragma unroll
    for (int m = 0; m < N; ++m) rl += (a[m] > a[l] || (a[m] == a[l] && m < l)) ? 1u : 0u;
    rk8[l / 4] |= rl << (8 * (l % 4));
    inv[l] = a[l] > eps * eps * amax ? T(1) / a[l] : T(0);
    if (RT && l >= n) continue;
#pragma unroll
    for (int h = 0; h < R; ++h) {
      const int q = lane + L * h;
      if (q < M) FW[rl * M + q] = x[h][l];
    }
    if (lane == 0) FS[rl] = sqrt(a[l]);
  }

  // V^T, column by column: element k of v_l = X^T w_l / s_l^2 from column
  // k of X (reloaded), stored by lane k % L
#pragma unroll
  for (int k = 0; k < SRN; ++k) {
    if (RT && k >= SR) break;
    if (k < n) {
      const int32_t pk = pos[((size_t)b * nw + k) * p_all + it];
      const uint32_t row = min((uint32_t)(pk & 0xffff), lim), col = min((uint32_t)(pk >> 16), lim);
      T xk[R];
#pragma unroll
      for (int h = 0; h < R; ++h) {
        const int q = lane + L * h;
        xk[h] = q < M ? U[(size_t)k * fs + (row + q % BS) + (size_t)nr * (col + q / BS)] : T(0);
      }
#pragma unroll
      for (int l = 0; l < N; ++l) {
        if (RT && l >= n) break;  // uniform: the zero columns
        T pv = xk[0] * x[0][l];
#pragma unroll
        for (int h = 1; h < R; ++h) pv = fma(xk[h], x[h][l], pv);
        const T vk = group_sum<L>(pv) * inv[l];
        const int rl = rank_of(l);
        if (lane == k % L) F[rl * SR + k] = vk;
      }
    } else {
#pragma unroll
      for (int l = 0; l < N; ++l)
        if ((!RT || l < n) && lane == k % L) F[rank_of(l) * SR + k] = T(0);
    }
  }
}

uint32_t svd_lanes(uint32_t bs, uint32_t nw, int which) {
#define PG_L1(B, N, LE, L) \
  if (which == 0 && bs == B && nw == N) return L;
  PG_SHAPES(PG_L1)
#undef PG_L1
#define PG_L2(B, N, L) \
  if (which == 1 && bs == B && nw == N) return L;
  PG_SVD_ALT(PG_L2)
#undef PG_L2
  return 0;
}

hipError_t launch_svd(const void* uvar, const int32_t* pos, const uint32_t* sel, uint32_t nb, uint32_t nvar,
                      uint32_t nvar_stored, const Shape& sh, void* factors, int max_sweeps, double tol,
                      uint32_t* stats, hipStream_t s, int mapping) {
  if (nvar > nvar_stored) return hipErrorInvalidValue;
  const uint32_t lim = sh.nr - sh.bs;
  const uint32_t groups = nvar * sh.p_sel;
#define PG_SVD_F32(B, N, L)                                                                                      \
  {                                                                                                            \
    const dim3 grid((groups * L + 255) / 256, nb);                                                             \
    hipLaunchKernelGGL((k_svd<B, N, L, float>), grid, dim3(256), 0, s, (const float*)uvar, pos, sel, nvar,     \
                       nvar_stored, sh.p_sel, sh.p_all, sh.nr, sh.fs, sh.nw, sh.vol, lim, sh.fstride, max_sweeps,            \
                       (float)(tol * tol), (float*)factors, stats);                                                \
    return hipGetLastError();                                                                                  \
  }
#define PG_SVD(B, N, LE, L)                                                                                      \
  if (sh.bs == B && sh.nw == N && (sh.fp64 || mapping == 0)) {                                                 \
    if (sh.fp64) {                                                                                             \
      /* FP64: at least 16 lanes per matrix (fewer rows per lane fit the registers); the 64-row matrices     \
         of patch 8 take 32 (15 frames) and 64 (31 frames) */                                                  \
      constexpr int LD = (B == 8 && N == 31) ? 64 : (B == 8 && N == 15) ? 32 : (L < 16 ? 16 : L);            \
      const dim3 grid((groups * LD + 255) / 256, nb);                                                          \
      hipLaunchKernelGGL((k_svd<B, N, LD, double>), grid, dim3(256), 0, s, (const double*)uvar, pos, sel, nvar, \
                         nvar_stored, sh.p_sel, sh.p_all, sh.nr, sh.fs, sh.nw, sh.vol, lim, sh.fstride, max_sweeps, tol * tol, \
                         (double*)factors, stats);                                                               \
      return hipGetLastError();                                                                                \
    }                                                                                                          \
    PG_SVD_F32(B, N, L)                                                                                        \
  }
  PG_SHAPES(PG_SVD)
#undef PG_SVD
#define PG_SVD2(B, N, L)                                                                                         \
  if (sh.bs == B && sh.nw == N && mapping == 1) PG_SVD_F32(B, N, L)
  PG_SVD_ALT(PG_SVD2)
#undef PG_SVD2
  // an exact shape without an alternative mapping: the primary one
#define PG_SVD3(B, N, LE, L)                                                                                     \
  if (sh.bs == B && sh.nw == N && !sh.fp64) PG_SVD_F32(B, N, L)
  PG_SHAPES(PG_SVD3)
#undef PG_SVD3
#undef PG_SVD_F32
  if (sh.fp64) return hipErrorInvalidValue;
  const uint32_t nm = shape_generic(sh.bs, sh.nw);
#define PG_SVDG(B, NM, L, LE)                                                                                    \
  if (sh.bs == B && nm == NM) {                                                                                \
    const dim3 grid((groups * L + 255) / 256, nb);                                                             \
    hipLaunchKernelGGL((k_svd<B, NM, L, float, true>), grid, dim3(256), 0, s, (const float*)uvar, pos, sel,    \
                       nvar, nvar_stored, sh.p_sel, sh.p_all, sh.nr, sh.fs, sh.nw, sh.vol, lim, sh.fstride, max_sweeps,      \
                       (float)(tol * tol), (float*)factors, stats);                                                \
    return hipGetLastError();                                                                                  \
  }
  PG_GENERIC(PG_SVDG)
#undef PG_SVDG
  return hipErrorInvalidValue;
}

}  // namespace pgsvt
