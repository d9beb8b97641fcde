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

// The pairs of a sweep in groups of at most four that share no column, with
// the bits of the row-cyclic order (0, 1), (0, 2) .. (1, 2) ..: there column c
// meets the others in ascending order, so a pair is due when each of its
// columns is the other's next.  Of those due the lowest anti-diagonals go
// first.
struct PairGroup {
  int n = 0, i[4] = {0, 0, 0, 0}, j[4] = {0, 0, 0, 0};
};
template <int N>
struct Sweep {
  struct Table {
    PairGroup g[N * (N - 1) / 2];
    int groups = 0;
  };
  static constexpr Table make() {
    Table t{};
    int next[N] = {};  // the column that column c meets next (N: none)
    next[0] = 1;
    for (int left = N * (N - 1) / 2; left > 0;) {
      PairGroup q{};
      for (; q.n < 4; ++q.n) {
        int bi = -1;
        for (int i = 0; i < N; ++i) {
          const int k = next[i];
          if (k <= i || k >= N || next[k] != i) continue;
          bool in = false;
          for (int z = 0; z < q.n; ++z) in = in || q.i[z] == i;
          if (!in && (bi < 0 || i + k < bi + next[bi])) bi = i;
        }
        if (bi < 0) break;
        q.i[q.n] = bi;
        q.j[q.n] = next[bi];
      }
      for (int z = 0; z < q.n; ++z) {
        const int i = q.i[z], k = q.j[z];
        next[i] = k + 1;
        next[k] = i + 1 == k ? k + 1 : i + 1;
      }
      t.g[t.groups++] = q;
      left -= q.n;
    }
    return t;
  }
  static constexpr Table kTable = make();
  // every pair once, each column's partners in ascending order, no column
  // twice in a group
  static constexpr bool sound() {
    int last[N] = {}, pairs = 0;
    for (int c = 0; c < N; ++c) last[c] = -1;
    for (int g = 0; g < kTable.groups; ++g) {
      const PairGroup& q = kTable.g[g];
      if (q.n < 1 || q.n > 4) return false;
      for (int z = 0; z < q.n; ++z, ++pairs) {
        const int i = q.i[z], k = q.j[z];
        if (i < 0 || i >= k || k >= N || k <= last[i] || i <= last[k]) return false;
        for (int y = 0; y < z; ++y)
          if (q.i[y] == i || q.j[y] == i || q.i[y] == k || q.j[y] == k) return false;
        last[i] = k;
        last[k] = i;
      }
    }
    return pairs == N * (N - 1) / 2;
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
      : "+&v"(xi), "+&v"(xj), "=&v"(t)
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
      : "+&v"(xi), "+&v"(xj), "+&v"(yi), "+&v"(yj), "=&v"(t), "=&v"(u)
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
template <int BS, int N, int L, class T, bool RT>
constexpr int svd_min_waves() {
  if (sizeof(T) != 4 || RT) return 1;
  return N > 16 ? 3 : (BS == 8 && N == 15 && L == 16) ? 4 : 1;
}

// whether a sweep takes four pairs at a time
template <int N, int L, class T>
constexpr bool quads() {
  return sizeof(T) == 4 && L >= 4 && N > 8;
}

template <int BS, int N, int L, class T, bool RT = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(svd_min_waves<BS, N, L, T, RT>()))) void k_svd(
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
    // Up to four pairs that share no column.  Lane l of a group works out the
    // rotation of pair l % 4 and hands it to its neighbours, where each lane
    // had worked out every pair's: the reciprocals and roots take four times a
    // plain instruction's slot, and were most of what a pair cost beside its
    // dot product and update.
    auto quad = [&](auto qc) __attribute__((always_inline)) {
      constexpr PairGroup q = Sweep<N>::kTable.g[decltype(qc)::value];
      const bool odd = lane & 1, high = lane & 2;
      auto mine = [&](float v0, float v1, float v2, float v3) __attribute__((always_inline)) {
        return high ? (odd ? v3 : v2) : (odd ? v1 : v0);
      };
      float c;
      if constexpr (L == 4) {
        // each lane ends with its own pair's sum, added as group_sum does
        float d[4];
        static_for<0, 4>([&](auto zc) __attribute__((always_inline)) {
          constexpr int z = decltype(zc)::value;
          d[z] = 0.f;
          if constexpr (z < q.n) {
            d[z] = x[0][q.i[z]] * x[0][q.j[z]];
#pragma unroll
            for (int h = 1; h < R; ++h) d[z] = fma(x[h][q.i[z]], x[h][q.j[z]], d[z]);
            asm("" : "+v"(d[z]));  // (rounded before the sum)
          }
        });
        const float s01 = (odd ? d[1] : d[0]) + dpp_f<0xB1>(odd ? d[0] : d[1]);
        const float s23 = (odd ? d[3] : d[2]) + dpp_f<0xB1>(odd ? d[2] : d[3]);
        c = (high ? s23 : s01) + dpp_f<0x4E>(high ? s01 : s23);
      } else {
        float d[4] = {0.f, 0.f, 0.f, 0.f};
        static_for<0, 4>([&](auto zc) __attribute__((always_inline)) {
          constexpr int z = decltype(zc)::value;
          if constexpr (z < q.n) d[z] = column_dot(q.i[z], q.j[z]);
        });
        c = mine(d[0], d[1], d[2], d[3]);
      }
      float ai = mine(a[q.i[0]], a[q.i[1]], a[q.i[2]], a[q.i[3]]);
      float aj = mine(a[q.j[0]], a[q.j[1]], a[q.j[2]], a[q.j[3]]);
      const bool rot = c * c > tol2 * ai * aj;
      const uint64_t rotates = __ballot(rot);
      if (!rotates) return;
      const float zeta = (aj - ai) * rcp_(c + c);
      const float den = fabs(zeta) + sqrt_(fma(zeta, zeta, 1.f));
      const float t = rot ? copysign(rcp_(den), zeta) : 0.f;
      const float cs = rsq_(fma(t, t, 1.f)), sn = cs * t;
      ai = fma(-t, c, ai);
      aj = fma(t, c, aj);
      tsum = fma(t, t, tsum);
      static_for<0, 4>([&](auto zc) __attribute__((always_inline)) {
        constexpr int z = decltype(zc)::value, kFrom = z * 0x55;  // quad_perm [z, z, z, z]
        if constexpr (z < q.n) {
          if (rotates & (0x1111111111111111ull << z)) {
            a[q.i[z]] = dpp_f<kFrom>(ai);
            a[q.j[z]] = dpp_f<kFrom>(aj);
            turn(q.i[z], q.j[z], dpp_f<kFrom>(cs), dpp_f<kFrom>(sn));
          }
        }
      });
    };
    // Groups pay where they are full for most of a sweep (16 x 15, 19.2 M
    // matrices: 51.4 -> 45.3 ms; 64 x 15, 1.14 M: 12.8 -> 11.5; 64 x 31, 1.36 M:
    // 152 -> 130); 7 columns have two pairs to a group (16 x 7, 31 M: 25.9 ms a
    // pair at a time, 26.1 in groups).
    if constexpr (quads<N, L, T>() && !RT) {
      static_assert(Sweep<N>::sound(), "a pair missing, repeated or out of order");
      for_all(std::make_integer_sequence<int, Sweep<N>::kTable.groups>{}, quad);
    } else {
#pragma unroll
      for (int i = 0; i < N - 1; ++i) {
        if (RT && i >= n - 1) break;  // uniform
#pragma unroll
        for (int j = i + 1; j < N; ++j) {
          if (RT && j >= n) break;
          one(i, j);
        }
      }
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
  constexpr int KG = !RT && (L == 4 || N > 16) ? 4 : 1;
#pragma unroll
  for (int k0 = 0; k0 < SRN; k0 += KG) {
    if (RT && k0 >= SR) break;  // uniform
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
      if (RT && l >= n) break;  // uniform: the zero columns
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
