// svd.hip -- batched Jacobi SVD of the Casorati matrices (arma::svd_econ at
// src/svt.hpp:111).
#include <hip/hip_runtime.h>

#include <cstdint>
#include <limits>
#include <type_traits>
#include <utility>

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

// The pairs of a sweep in groups of two: anti-diagonals i + j = 1 .. 2 N - 3,
// neighbours (i, j) and (i + 1, j - 1) of one anti-diagonal together, a last
// odd one alone (k >= l).
struct PairGroup {
  int i, j, k, l;
};
template <int N>
struct Sweep {
  static constexpr int first(int d) { return d > N - 1 ? d - (N - 1) : 0; }
  static constexpr int pairs(int d) { return (d - 1) / 2 - first(d) + 1; }
  static constexpr int count() {
    int c = 0;
    for (int d = 1; d < 2 * N - 2; ++d) c += (pairs(d) + 1) / 2;
    return c;
  }
  static constexpr int kGroups = count();
  static constexpr PairGroup group(int g) {
    int d = 1;
    for (; g >= (pairs(d) + 1) / 2; ++d) g -= (pairs(d) + 1) / 2;
    const int i = first(d) + 2 * g;
    return {i, d - i, i + 1, d - i - 1};
  }
};
template <class F, int... G>
__device__ __forceinline__ void for_all(std::integer_sequence<int, G...>, F&& f) {
  (f(std::integral_constant<int, G>{}), ...);
}

// xi, xj = cs xi - sn xj, sn xi + cs xj, in place.  The FP32 form is written
// out because the update is skipped where no matrix of the wave rotates: left
// to itself the compiler forms the new xi beside the old one and copies it
// home for the join, 4 of the 46 vector instructions of a pair (16 x 15
// matrices, 4 rows a lane; 55.0 -> 53.6 ms for 19.2 M of them).  Both round as
// the compiler contracts the expressions: fma(cs, xi, -(sn xj)) and
// fma(sn, xi, cs xj).
__device__ __forceinline__ void rotate1(float& xi, float& xj, float cs, float sn) {
  float t;
  asm("v_mul_f32 %2, %4, %1\n\t"
      "v_mul_f32 %1, %3, %1\n\t"
      "v_fmac_f32 %1, %4, %0\n\t"
      "v_fma_f32 %0, %3, %0, -%2"
      : "+v"(xi), "+v"(xj), "=&v"(t)
      : "v"(cs), "v"(sn));
}
__device__ __forceinline__ void rotate2(float& xi, float& xj, float& yi, float& yj, float cs, float sn) {
  float t, u;
  asm("v_mul_f32 %4, %7, %1\n\t"
      "v_mul_f32 %5, %7, %3\n\t"
      "v_mul_f32 %1, %6, %1\n\t"
      "v_mul_f32 %3, %6, %3\n\t"
      "v_fmac_f32 %1, %7, %0\n\t"
      "v_fmac_f32 %3, %7, %2\n\t"
      "v_fma_f32 %0, %6, %0, -%4\n\t"
      "v_fma_f32 %2, %6, %2, -%5"
      : "+v"(xi), "+v"(xj), "+v"(yi), "+v"(yj), "=&v"(t), "=&v"(u)
      : "v"(cs), "v"(sn));
}
__device__ __forceinline__ void rotate1(double& xi, double& xj, double cs, double sn) {
  const double a = xi, b = xj;
  xi = cs * a - sn * b;
  xj = sn * a + cs * b;
}
__device__ __forceinline__ void rotate2(double& xi, double& xj, double& yi, double& yj, double cs, double sn) {
  rotate1(xi, xj, cs, sn);
  rotate1(yi, yj, cs, sn);
}

// RT: the window length n = nw is known at run time only (n <= N): the
// matrix is held as N columns, the last N - n zero, and every loop stops at
// n (uniform branches); the stored layout follows n.
// Waves per SIMD the register allocator is held to: 130 registers would leave
// the 64 x 15 matrices of patch 8 three; 31 columns, left alone, 172 for two
// (64 x 31, 1.36 M matrices: 158 ms with two waves, 152 with three).
template <int BS, int N, int L, class T>
constexpr int svd_min_waves() {
  if (sizeof(T) != 4) return 1;
  return N > 16 ? 3 : (BS == 8 && N == 15 && L == 16) ? 4 : 1;
}

template <int BS, int N, int L, class T, bool RT = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(svd_min_waves<BS, N, L, T>()))) void k_svd(
    const T* __restrict__ u32, const int32_t* __restrict__ pos, const uint32_t* __restrict__ sel, uint32_t nvar,
    uint32_t nvar_stored, uint32_t p_sel, uint32_t p_all, uint32_t nr, uint32_t fs, uint32_t nw, uint32_t vol,
    uint32_t lim, uint32_t fstride, int max_sweeps, T tol2, T* __restrict__ factors, uint32_t* __restrict__ stats) {
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

  // inner product of columns i and j, in every lane of the group
  auto column_dot = [&](int i, int j) __attribute__((always_inline)) {
    T t = x[0][i] * x[0][j];
#pragma unroll
    for (int h = 1; h < R; ++h) t = fma(x[h][i], x[h][j], t);
    return group_sum<L>(t);
  };

  T a[N];
  int sweep = 0;
  for (; sweep < max_sweeps; ++sweep) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      a[k] = column_dot(k, k);
    }
    // sum of t^2 over the sweep: zero exactly when no pair rotated.  A
    // floating-point chain (never reassociated) keeps this in one register.
    T tsum = T(0);
    // rotation zeroing the (i, j) inner product c: zeta = (b - a) / 2c,
    // t = sign(zeta) / (|zeta| + sqrt(1 + zeta^2)), cs = 1/sqrt(1+t^2)
    auto tangent = [&](int i, int j, T c, bool rot) __attribute__((always_inline)) {
      const T zeta = (a[j] - a[i]) * rcp_(c + c);
      const T den = fabs(zeta) + sqrt_(fma(zeta, zeta, T(1)));
      return rot ? copysign(rcp_(den), zeta) : T(0);
    };
    auto turn = [&](int i, int j, T cs, T sn) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h + 1 < R; h += 2) rotate2(x[h][i], x[h][j], x[h + 1][i], x[h + 1][j], cs, sn);
      if constexpr (R % 2 == 1) rotate1(x[R - 1][i], x[R - 1][j], cs, sn);
    };
    // Late in the iteration most pairs rotate in none of the wave's
    // matrices; the update is then the identity (t = 0, cs = 1, sn = 0
    // reproduce every value exactly) and is skipped for the whole wave.
    auto one = [&](int i, int j) __attribute__((always_inline)) {
      const T c = column_dot(i, j);
      const bool rot = c * c > tol2 * a[i] * a[j];
      if (!__any(rot)) return;
      const T t = tangent(i, j, c, rot), cs = rsq_(fma(t, t, T(1)));
      a[i] = fma(-t, c, a[i]);
      a[j] = fma(t, c, a[j]);
      tsum = fma(t, t, tsum);
      turn(i, j, cs, cs * t);
    };
    auto two = [&](int i, int j, int k, int l) __attribute__((always_inline)) {
      const T c = column_dot(i, j), e = column_dot(k, l);
      const bool rc = c * c > tol2 * a[i] * a[j], re = e * e > tol2 * a[k] * a[l];
      if (!__any(rc || re)) return;
      const T t = tangent(i, j, c, rc), u = tangent(k, l, e, re);
      const T cs = rsq_(fma(t, t, T(1))), du = rsq_(fma(u, u, T(1)));
      a[i] = fma(-t, c, a[i]);
      a[j] = fma(t, c, a[j]);
      a[k] = fma(-u, e, a[k]);
      a[l] = fma(u, e, a[l]);
      tsum = fma(t, t, tsum);
      tsum = fma(u, u, tsum);
      turn(i, j, cs, cs * t);
      turn(k, l, du, du * u);
    };
    // The sweep's order is row-cyclic, (0, 1), (0, 2) .. (1, 2) ..  A pair
    // depends on those before it that share a column, so the pairs of one
    // anti-diagonal i + j = d, taken after every smaller d, give the same
    // bits, and are independent of each other.  Matrices of 31 columns leave
    // three waves a SIMD: there two pairs go at a time, one's chain (dot
    // product, reciprocals and roots, update) in the other's waits (64 x 31:
    // 179 -> 169 ms for 1.36 M matrices).  With more waves it costs: a pair
    // that does not rotate is skipped only with its neighbour (16 x 15: 53.6
    // -> 55.8 ms for 19.2 M).
    // A run-time window length goes by the list as well: a loop that breaks at
    // n is not unrolled, and X would live in scratch memory.
    constexpr bool PAIRS = N > 16 && sizeof(T) == 4;
    if constexpr (PAIRS || RT) {
      for_all(std::make_integer_sequence<int, Sweep<N>::kGroups>{}, [&](auto gc) __attribute__((always_inline)) {
        constexpr PairGroup q = Sweep<N>::group(decltype(gc)::value);
        const bool in = !RT || q.j < n;  // (uniform)
        if constexpr (q.k >= q.l) {
          if (in) one(q.i, q.j);
        } else if constexpr (PAIRS) {
          if (in)
            two(q.i, q.j, q.k, q.l);
          else if (q.l < n)
            one(q.k, q.l);
        } else {
          if (in) one(q.i, q.j);
          if (!RT || q.l < n) one(q.k, q.l);
        }
      });
    } else {
#pragma unroll
      for (int i = 0; i < N - 1; ++i)
#pragma unroll
        for (int j = i + 1; j < N; ++j) one(i, j);
    }
    if (!__any(tsum > T(0))) break;
  }
  if (stats && lane == 0 && valid) atomicMax(stats, (uint32_t)sweep + 1);
  // final column norms (identical in every lane of the group)
#pragma unroll
  for (int k = 0; k < N; ++k) {
    a[k] = column_dot(k, k);
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

  // V^T, KG columns at a time: element k of v_l = X^T w_l / s_l^2 from column
  // k of X (reloaded), lane z < KG taking and storing column k0 + z.  With
  // 4 lanes that is one store and one scaling for four elements (16 x 15,
  // 19.2 M matrices: 53.6 -> 51.4 ms), at 31 columns fewer addresses (64 x 31:
  // 169 -> 165 ms); at 16 lanes the selects cost more than they save (36 x 15
  // in a batch: 17.6 -> 21.1 ms).
  constexpr int KG = (L == 4 || N > 16) ? 4 : 1;
#pragma unroll
  for (int k0 = 0; k0 < SRN; k0 += KG) {
    if (RT && k0 >= SR) continue;  // (uniform)
    if constexpr (KG > 1) {
      // the ranks anew: the row addresses of all N ranks, kept from one
      // group of columns to the next, would cost a wave per SIMD or two
#pragma unroll
      for (int i = 0; i < (N + 3) / 4; ++i) asm volatile("" : "+v"(rk8[i]));
    }
    T xk[KG][R];
#pragma unroll
    for (int z = 0; z < KG; ++z) {
      const int k = k0 + z;
      const bool kin = k < N && (!RT || k < n);
      const int32_t pk = kin ? pos[((size_t)b * nw + k) * p_all + it] : 0;
      const uint32_t row = min((uint32_t)(pk & 0xffff), lim), col = min((uint32_t)(pk >> 16), lim);
#pragma unroll
      for (int h = 0; h < R; ++h) {
        const int q = lane + L * h;
        xk[z][h] = kin && q < M ? U[(size_t)k * fs + (row + q % BS) + (size_t)nr * (col + q / BS)] : T(0);
      }
    }
#pragma unroll
    for (int l = 0; l < N; ++l) {
      if (RT && l >= n) continue;  // uniform: the zero columns
      T mine = T(0);
#pragma unroll
      for (int z = 0; z < KG; ++z) {
        T pv = xk[z][0] * x[0][l];
#pragma unroll
        for (int h = 1; h < R; ++h) pv = fma(xk[z][h], x[h][l], pv);
        const T t = group_sum<L>(pv);
        mine = KG == 1 || lane % KG == z ? t : mine;
      }
      const T vk = mine * inv[l];
      const int at = KG == 1 ? k0 : k0 + lane;
      const bool real = (!RT && k0 + KG <= N) || at < n;  // (the row's padding is zero)
      if (KG == 1 ? lane == k0 % L : L == KG || lane < KG) F[rank_of(l) * SR + at] = real ? vk : T(0);
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
    const dim3 grid((groups * L + 255) / 256, nb);                                                            \
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
    const dim3 grid((groups * L + 255) / 256, nb);                                                            \
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
