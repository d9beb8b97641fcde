// noise_gpu.hip -- quadtree leaf statistics of the noise estimator on the GPU
// (src/noise.hpp:55-100, 173-271, 395-458), with the host estimator's
// rounding.
//
// Items: (frame, scale) pairs, each normalised once into Z [items][n n].
// Split tests: one workgroup per candidate block of an item (every block of
// the complete quadtree whose size has an F-table entry); the host replays
// the reference's recursion with the decisions.  Leaf statistics: one
// workgroup per distinct leaf (1,024 threads above 64 x 64), one wave per
// leaf up to 16 x 16.
//
// The reference sums even- and odd-indexed terms one after the other.  The
// GPU keeps those sums: most waves of a workgroup form a tile of terms in
// LDS while one wave adds the tile before it up, a lane per chain, so the
// robust mean and the split statistics round as the host's do.  What bounds
// them is that chain: half an element's FP64 add latency per element and
// sum, 0.11 ms a pass of a 256 x 256 block, beside which everything else is
// hidden.  Order statistics are exact in any order: a radix walk over the
// values' bit patterns, or ranks counted within a wave.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "kernels.hpp"

namespace pgsvt {
namespace {

// sum over the 256 threads of the workgroup, returned to every thread
// (red: 4 doubles of LDS, free again when the function returns to all)
__device__ double wg_sum(double v, double* red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();  // the previous sum's readers are done with red
  if ((threadIdx.x & 63) == 0) red[threadIdx.x / 64] = v;
  __syncthreads();
  return ((red[0] + red[1]) + red[2]) + red[3];
}

// totally ordered 64-bit key of a double (negative values reversed)
__device__ __forceinline__ uint64_t order_key(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
__device__ __forceinline__ double from_key(uint64_t k) {
  return __builtin_bit_cast(double, (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k);
}


// ------------------------------------------------------ ordered sums --
// K sums of N terms each, every sum as two chains (even and odd indices) in
// index order.  Tiles of T elements: the waves after the first load tile
// t + 1 (load(e)) and form tile t's terms (terms(value, x): the K terms)
// while lanes 0 .. 2K-1 of the first wave add tile t - 1 up.  NT threads.
// even / odd: the chains' ends, in every thread.
template <int K, int NT>
struct ChainLds {
  static constexpr int E = NT == 1024 ? 1 : 3, T = E * (NT - 64);  // E elements a filling thread and tile
  double t[2][2 * K][T / 2 + 2];
  double end[2 * K];
};

template <int K, int NT, class Load, class Terms>
__device__ void chain_sums(uint32_t N, Load load, Terms terms, ChainLds<K, NT>& L, double (&even)[K],
                           double (&odd)[K]) {
#pragma clang fp contract(off)
  constexpr uint32_t T = ChainLds<K, NT>::T, E = ChainLds<K, NT>::E, F = NT - 64;
  const uint32_t tiles = (N + T - 1) / T, wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  decltype(load(0u)) next[E];
  const uint32_t own = threadIdx.x - 64;  // (filling threads)
  if (wave > 0) {
#pragma unroll
    for (uint32_t i = 0; i < E; ++i)
      if (own + i * F < N) next[i] = load(own + i * F);
  }
  double acc = 0.0;
  // the decomposition's waves share the SIMD: the chain goes first
  __builtin_amdgcn_s_setprio(3);
  for (uint32_t t = 0; t <= tiles; ++t) {
    if (wave > 0) {
      if (t < tiles) {
        decltype(load(0u)) now[E];
#pragma unroll
        for (uint32_t i = 0; i < E; ++i) {
          now[i] = next[i];
          const uint32_t e = (t + 1) * T + own + i * F;
          if (e < N) next[i] = load(e);
        }
#pragma unroll
        for (uint32_t i = 0; i < E; ++i) {
          const uint32_t r = own + i * F;
          if (t * T + r < N) {
            double x[K];
            terms(now[i], x);
#pragma unroll
            for (int q = 0; q < K; ++q) L.t[t & 1][2 * q + (r & 1)][r / 2] = x[q];  // (T is even)
          }
        }
      }
    } else if (t > 0 && lane < 2 * K) {
      const uint32_t len = min(T, N - (t - 1) * T), steps = (len + 1 - (lane & 1)) / 2;
      const double* p = L.t[(t - 1) & 1][lane];
      uint32_t i = 0;
      for (; i + 16 <= steps; i += 16) {
        double2 v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = *reinterpret_cast<const double2*>(p + i + 2 * q);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          acc += v[q].x;
          acc += v[q].y;
        }
      }
      for (; i < steps; ++i) acc += p[i];
    }
    __syncthreads();
  }
  __builtin_amdgcn_s_setprio(0);
  if (wave == 0 && lane < 2 * K) L.end[lane] = acc;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < K; ++q) {
    even[q] = L.end[2 * q];
    odd[q] = L.end[2 * q + 1];
  }
  __syncthreads();  // L is rewritten by the next call
}

// -------------------------------------------------- order statistics --
// LDS of the selection: two 256-bin histograms, the wave totals of their
// prefix sums, the chosen prefixes and remaining ranks
struct SelectLds {
  uint32_t hist[2][256];
  uint32_t wtot[4];
  uint64_t prefix[2];
  uint32_t k[2];
};

// Count `bin` of the active lanes that match: the lanes of the first one's
// bin add once (the leading bytes of a leaf's values are nearly all equal).
__device__ __forceinline__ void count_bin(uint32_t* hist, bool match, uint32_t bin) {
  if (!match) return;
  const uint32_t b0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)bin);
  const uint64_t same = __ballot(bin == b0);
  if (bin != b0)
    atomicAdd(&hist[bin], 1u);
  else if ((threadIdx.x & 63) == (uint32_t)__ffsll((unsigned long long)same) - 1)
    atomicAdd(&hist[bin], (uint32_t)__popcll(same));
}

// The elements of ranks k0 and k1 (0-based, ascending) of the values each
// thread visits (each(f) calls f(value) for the thread's elements): eight
// passes, each a 256-bin histogram of the next key byte among the values
// that match the bytes chosen so far, one histogram while both ranks share
// them.  Every thread of the workgroup calls it.
template <class Each>
__device__ void wg_select2(uint32_t k0, uint32_t k1, Each each, SelectLds& L, double& out0, double& out1) {
  uint64_t prefix[2] = {0, 0}, mask = 0;
  uint32_t kk[2] = {k0, k1};
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int shift = 56; shift >= 0; shift -= 8) {
    const bool one = prefix[0] == prefix[1];
    if (threadIdx.x < 256) L.hist[0][threadIdx.x] = L.hist[1][threadIdx.x] = 0u;
    __syncthreads();
    each([&](double x) {
      const uint64_t key = order_key(x);
      const uint32_t bin = (uint32_t)(key >> shift) & 255u;
      count_bin(L.hist[0], (key & mask) == prefix[0], bin);
      if (!one) count_bin(L.hist[1], (key & mask) == prefix[1], bin);
    });
    __syncthreads();
    for (int h = 0; h < 2; ++h) {
      // inclusive prefix sum over the 256 bins
      const uint32_t c = threadIdx.x < 256 ? L.hist[one ? 0 : h][threadIdx.x] : 0u;
      uint32_t incl = c;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(incl, o, 64);
        incl += lane >= (uint32_t)o ? y : 0u;
      }
      if (lane == 63 && w < 4) L.wtot[w] = incl;
      __syncthreads();
      if (threadIdx.x < 256) {
        for (uint32_t q = 0; q < w; ++q) incl += L.wtot[q];
        const uint32_t excl = incl - c;
        if (excl <= kk[h] && kk[h] < incl) {  // exactly one thread: the bin of rank k
          L.prefix[h] = prefix[h] | ((uint64_t)threadIdx.x << shift);
          L.k[h] = kk[h] - excl;
        }
      }
      __syncthreads();
    }
    prefix[0] = L.prefix[0];
    prefix[1] = L.prefix[1];
    kk[0] = L.k[0];
    kk[1] = L.k[1];
    mask |= 0xffull << shift;
    __syncthreads();  // L is rewritten by the next pass
  }
  out0 = from_key(prefix[0]);
  out1 = from_key(prefix[1]);
}

// Elements of rank k0 and k1 of a wave's N <= 64 C values (value e in lane
// e % 64, slot e / 64): ranks counted against every value.
__device__ __forceinline__ double lane_value(double x, int l) {
  const int2 h = __builtin_bit_cast(int2, x);
  int2 o;
  o.x = __builtin_amdgcn_readlane(h.x, l);
  o.y = __builtin_amdgcn_readlane(h.y, l);
  return __builtin_bit_cast(double, o);
}
template <int C>
__device__ void wave_select2(uint32_t k0, uint32_t k1, const double (&v)[C], uint32_t N, double& out0, double& out1) {
  uint32_t less[C], upto[C];
#pragma unroll
  for (int c = 0; c < C; ++c) less[c] = upto[c] = 0;
#pragma unroll
  for (int d = 0; d < C; ++d) {
    const int cnt = (int)min(64u, N - min(N, 64u * d));
    for (int l = 0; l < cnt; ++l) {
      const double x = lane_value(v[d], l);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        less[c] += x < v[c] ? 1u : 0u;
        upto[c] += x <= v[c] ? 1u : 0u;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const bool live = (threadIdx.x & 63) + 64 * c < N;
    const uint64_t m0 = __ballot(live && less[c] <= k0 && k0 < upto[c]);
    const uint64_t m1 = __ballot(live && less[c] <= k1 && k1 < upto[c]);
    if (m0) out0 = lane_value(v[c], __ffsll((unsigned long long)m0) - 1);
    if (m1) out1 = lane_value(v[c], __ffsll((unsigned long long)m1) - 1);
  }
}

// ----------------------------------------------------------- kernels --
// Z [items][n n] = the items' frames over their scales (true division, as
// u /= uMax)
__global__ __launch_bounds__(256) void k_normalise(const double* __restrict__ X, uint32_t fs,
                                                   const uint32_t* __restrict__ frames,
                                                   const double* __restrict__ scales, double* __restrict__ Z) {
  const double* F = X + (size_t)frames[blockIdx.y] * fs;
  const double sc = scales[blockIdx.y];
  double* O = Z + (size_t)blockIdx.y * fs;
  for (uint32_t e = blockIdx.x * 256 + threadIdx.x; e < fs; e += gridDim.x * 256) O[e] = F[e] / sc;
}

// SplitBlockQ (src/noise.hpp:182-221) statistics of block (i0, j0, N) of
// item blockIdx.y: the F statistic max(Sz, Se) / min(Sz, Se) of the values
// and of their 5-point residuals (wrap-around within the block), element
// k = y + N x.  ORDERED: the sums in the host's order; otherwise as
// workgroup sums, which may change a decision only when F lies within their
// rounding of its threshold (the learned path's).
template <bool ORDERED>
__global__ __launch_bounds__(256) void k_split_stats(const double* __restrict__ Z, uint32_t n,
                                                     const uint32_t* __restrict__ blocks, uint32_t nblocks,
                                                     double* __restrict__ stat) {
#pragma clang fp contract(off)
  __shared__ double red[4];
  __shared__ ChainLds<ORDERED ? 2 : 1, 256> L;
  const uint32_t bi = blockIdx.x, it = blockIdx.y;
  const uint32_t i0 = blocks[3 * bi], j0 = blocks[3 * bi + 1], N = blocks[3 * bi + 2];
  const double* F = Z + (size_t)it * n * n;
  const uint32_t R = N * N, lg = 31 - __clz((int)N);  // sizes with a threshold are powers of two
  const double sq = sqrt((double)(5 * 5 + 5));
  auto val = [&](uint32_t y, uint32_t x) { return F[(i0 + y) + (size_t)n * (j0 + x)]; };
  auto res = [&](uint32_t y, uint32_t x) {
    const uint32_t yp = (y + 1 == N) ? 1 : y + 1, ym = (y == 0) ? N - 2 : y - 1;
    const uint32_t xp = (x + 1 == N) ? 1 : x + 1, xm = (x == 0) ? N - 2 : x - 1;
    return (5.0 * val(y, x) - (((val(yp, x) + val(ym, x)) + val(y, xm)) + val(y, xp))) / sq;
  };
  const double OoR = 1.0 / R, OoRm1 = 1.0 / (R - 1);
  double Sz, Se;
  if constexpr (ORDERED) {
    double ev[2], od[2];
    auto load = [&](uint32_t e) {
      return make_double2(val(e & (N - 1), e >> lg), res(e & (N - 1), e >> lg));
    };
    chain_sums<2, 256>(
        R, load,
        [](double2 v, double (&x)[2]) {
          x[0] = v.x;
          x[1] = v.y;
        },
        L, ev, od);
    const double accuZ = (ev[0] + od[0]) * OoR, accuR = (ev[1] + od[1]) * OoR;
    chain_sums<2, 256>(
        R, load,
        [accuZ, accuR](double2 v, double (&x)[2]) {
#pragma clang fp contract(off)
          const double t = v.x - accuZ, u = v.y - accuR;
          x[0] = t * t;
          x[1] = u * u;
        },
        L, ev, od);
    Sz = (ev[0] + od[0]) * OoRm1;
    Se = (ev[1] + od[1]) * OoRm1;
  } else {
    double sa = 0.0, sr = 0.0;
    for (uint32_t e = threadIdx.x; e < R; e += 256) {
      sa += val(e & (N - 1), e >> lg);
      sr += res(e & (N - 1), e >> lg);
    }
    const double accuZ = wg_sum(sa, red) * OoR;
    const double accuR = wg_sum(sr, red) * OoR;
    double ss = 0.0, se = 0.0;
    for (uint32_t e = threadIdx.x; e < R; e += 256) {
      const double t = val(e & (N - 1), e >> lg) - accuZ, u = res(e & (N - 1), e >> lg) - accuR;
      ss += t * t;
      se += u * u;
    }
    Sz = wg_sum(ss, red) * OoRm1;
    Se = wg_sum(se, red) * OoRm1;
  }
  if (threadIdx.x == 0) stat[(size_t)it * nblocks + bi] = (Sz > Se) ? Sz / Se : Se / Sz;
}

// leaves of at most kWaveLeaf values take a wave, of at most kLeafCache 256
// values a workgroup that holds them in registers, larger ones a workgroup
// of 1,024 threads that reads them again at every pass
constexpr uint32_t kWaveLeaf = 256, kLeafCache = 16;

// Leaf element e = r + s c (column-major) of leaf (item, i0, j0, s): its
// value and its 9-point Laplacian from the wrapped 3 x 3 neighbourhood
// within the leaf, in the host's order (even terms, odd terms, their sum).
struct LeafView {
  const double* F;
  uint32_t n, s, lg;  // lg: log2 of s, or 32 where s (a frame's side) is not a power of two
  __device__ LeafView(const double* Z, uint32_t n_, const uint32_t* Lf)
      : F(Z + (size_t)Lf[0] * n_ * n_ + Lf[1] + (size_t)n_ * Lf[2]), n(n_), s(Lf[3]) {
    lg = (s & (s - 1)) ? 32u : 31u - (uint32_t)__clz((int)s);
  }
  __device__ uint32_t col(uint32_t e) const { return lg < 32 ? e >> lg : e / s; }
  __device__ double val(uint32_t e) const {
    const uint32_t c = col(e);
    return F[(e - s * c) + (size_t)n * c];
  }
  __device__ double lap(uint32_t e) const {
#pragma clang fp contract(off)
    const double ne = (1.0 * 0.125) * -1.0, nm = -1.0 * -1.0;
    const uint32_t x = col(e), y = e - s * x;
    const uint32_t xp = (x + 1 == s) ? 1 : x + 1, xm = (x == 0) ? s - 2 : x - 1;
    const uint32_t yp = (y + 1 == s) ? 1 : y + 1, ym = (y == 0) ? s - 2 : y - 1;
    auto I = [&](uint32_t r, uint32_t c) { return F[r + (size_t)n * c]; };
    double a1 = 0.0, a2 = 0.0;
    a1 += I(xm, ym) * ne;
    a2 += I(xm, y) * ne;
    a1 += I(xm, yp) * ne;
    a2 += I(x, ym) * ne;
    a1 += I(x, y) * nm;
    a2 += I(x, yp) * ne;
    a1 += I(xp, ym) * ne;
    a2 += I(xp, y) * ne;
    a1 += I(xp, yp) * ne;
    return a1 + a2;
  }
};

// Laplacians of the leaves above the register cache, computed once: leaf
// big[q] into laps from element boff[q].
__global__ __launch_bounds__(256) void k_leaf_prep(const double* __restrict__ Z, uint32_t n,
                                                   const uint32_t* __restrict__ leaves,
                                                   const uint64_t* __restrict__ boff, double* __restrict__ laps) {
  const LeafView v(Z, n, leaves + 4 * (size_t)blockIdx.y);
  const uint32_t N = v.s * v.s;
  const uint64_t o = boff[blockIdx.y];
  for (uint32_t e = blockIdx.x * 256 + threadIdx.x; e < N; e += gridDim.x * 256) laps[o + e] = v.lap(e);
}

// RobustMeanEstimate (src/noise.hpp:238-271): Huber IRLS from the mean, the
// scale from the interquartile distance (its two order statistics a_hi, a_lo
// of A fixed: sorted(A - m) is sorted(A) - m, rounding being monotone).
// sums(first, m, inv, ev, od): the chains of sum |A - m|, sum w A and sum w
// with the weights at (m, inv), all 1 when first.
template <class Sums>
__device__ double robust_mean(uint32_t N, double a_hi, double a_lo, Sums sums) {
#pragma clang fp contract(off)
  const double tol = 1e-6, eps = 1e-12;
  double ev[3], od[3];
  sums(true, 0.0, 0.0, ev, od);
  double wa = ev[1] + od[1], ws = (double)((N + 1) / 2) + (double)(N / 2);
  double m = 0, m0 = 1e12;
  for (uint32_t it = 0; it < 10000; ++it) {
    m = (fabs(ws) < eps) ? m0 : wa / ws;
    const double d = ((a_hi - m) - (a_lo - m)) + eps;
    sums(false, m, 1. / d, ev, od);
    const double err = (ev[0] + od[0]) / (double)N;
    wa = ev[1] + od[1];
    ws = ev[2] + od[2];
    // (a mean that is not a number stays one: the host's further passes end
    // at the same value)
    if (fabs(m0 - m) < tol || err < tol || m != m) break;
    m0 = m;
  }
  return m;
}

// one element's terms of those sums
__device__ __forceinline__ void mean_terms(bool first, double m, double inv, double A, double (&x)[3]) {
#pragma clang fp contract(off)
  if (first) {
    x[0] = 0.0;
    x[1] = A;
    x[2] = 1.0;
    return;
  }
  const double r = A - m, a = fabs(r * inv);
  const double wq = (a < 0.75) ? 1. : 0.75 / a;
  x[0] = fabs(r);
  x[1] = wq * A;
  x[2] = wq;
}

__device__ __forceinline__ uint32_t mean_rank(uint32_t N) { return ((N + 1) / 2 + 1) / 2; }

// median as the host averages it
__device__ __forceinline__ double mid_of(uint32_t N, double o0, double o1) {
  return (N % 2 == 0) ? o0 + (o1 - o0) / 2.0 : o0;
}

// Robust mean and variance (RobustVarianceEstimate of the 9-point Laplacian,
// src/noise.hpp:232-236, 395-417) of leaf blockIdx.x: out [leaf][2].  BIG:
// values from Z and Laplacians from laps at every pass; otherwise both in
// registers (element threadIdx.x + 256 i in slot i) and the values once more
// in LDS, where the filling waves find them.
template <bool BIG>
__global__ __launch_bounds__(BIG ? 1024 : 256) void k_leaf_stats(const double* __restrict__ Z, uint32_t n,
                                                                 const uint32_t* __restrict__ leaves,
                                                                 const uint64_t* __restrict__ boff,
                                                                 const double* __restrict__ laps,
                                                                 double* __restrict__ out) {
#pragma clang fp contract(off)
  constexpr uint32_t NT = BIG ? 1024 : 256;
  __shared__ SelectLds sel;
  __shared__ ChainLds<3, NT> L;
  const LeafView lv(Z, n, leaves + 4 * (size_t)blockIdx.x);
  const uint32_t N = lv.s * lv.s;
  const double* Lp = BIG ? laps + boff[blockIdx.x] : nullptr;
  double cv[BIG ? 1 : kLeafCache], cl[BIG ? 1 : kLeafCache];
  if constexpr (!BIG) {
#pragma unroll
    for (uint32_t i = 0; i < kLeafCache; ++i) {
      const uint32_t e = threadIdx.x + 256 * i;
      cv[i] = e < N ? lv.val(e) : 0.0;
      cl[i] = e < N ? lv.lap(e) : 0.0;
    }
  }
  // visit the thread's values (or Laplacians, through g)
  auto each_of = [&](bool of_lap, auto g) {
    return [&, of_lap, g](auto f) {
      if constexpr (!BIG) {
#pragma unroll
        for (uint32_t i = 0; i < kLeafCache; ++i)
          if (threadIdx.x + 256 * i < N) f(g(of_lap ? cl[i] : cv[i]));
      } else {
        // eight loads in flight
        uint32_t e = threadIdx.x;
        for (; e + 7 * NT < N; e += 8 * NT) {
          double x[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) x[q] = of_lap ? Lp[e + q * NT] : lv.val(e + q * NT);
#pragma unroll
          for (int q = 0; q < 8; ++q) f(g(x[q]));
        }
        for (; e < N; e += NT) f(g(of_lap ? Lp[e] : lv.val(e)));
      }
    };
  };
  auto ident = [](double x) { return x; };
  const uint32_t mq = mean_rank(N);
  double a_hi, a_lo;
  wg_select2(N - mq - 1, mq - 1, each_of(false, ident), sel, a_hi, a_lo);
  const double m = robust_mean(N, a_hi, a_lo, [&](bool first, double mm, double inv, double (&ev)[3], double (&od)[3]) {
    chain_sums<3, (int)NT>(
        N, [&](uint32_t e) { return lv.val(e); },
        [=](double A, double (&x)[3]) { mean_terms(first, mm, inv, A, x); }, L, ev, od);
  });
  // robust variance: (1.4826 median |lap - median(lap)|)^2
  const uint32_t half = N / 2, other = N % 2 == 0 ? half - 1 : half;
  double o0, o1;
  wg_select2(half, other, each_of(true, ident), sel, o0, o1);
  const double med = mid_of(N, o0, o1);
  wg_select2(half, other, each_of(true, [med](double x) { return fabs(x - med); }), sel, o0, o1);
  const double sig = 1.4826 * mid_of(N, o0, o1);
  if (threadIdx.x == 0) {
    out[2 * (size_t)blockIdx.x] = m;
    out[2 * (size_t)blockIdx.x + 1] = sig * sig;
  }
}

// The same for leaves of at most 256 values, a wave each.
__global__ __launch_bounds__(256) void k_leaf_wave(const double* __restrict__ Z, uint32_t n,
                                                   const uint32_t* __restrict__ leaves, uint32_t nleaves,
                                                   double* __restrict__ out) {
#pragma clang fp contract(off)
  constexpr int C = kWaveLeaf / 64;
  __shared__ double terms[4][6][kWaveLeaf / 2 + 2];
  const uint32_t w = threadIdx.x / 64, lane = threadIdx.x % 64;
  const uint32_t leaf = min(blockIdx.x * 4 + w, nleaves - 1);  // the last block's spare waves repeat a leaf
  const LeafView lv(Z, n, leaves + 4 * (size_t)leaf);
  const uint32_t N = lv.s * lv.s;
  double v[C], l[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const uint32_t e = lane + 64 * c;
    v[c] = e < N ? lv.val(e) : 0.0;
    l[c] = e < N ? lv.lap(e) : 0.0;
  }
  auto select2 = [&](uint32_t k0, uint32_t k1, const double (&x)[C], double& o0, double& o1) {
    if (N <= 64) {
      const double y[1] = {x[0]};
      wave_select2<1>(k0, k1, y, N, o0, o1);
    } else {
      wave_select2<C>(k0, k1, x, N, o0, o1);
    }
  };
  const uint32_t mq = mean_rank(N);
  double a_hi = 0, a_lo = 0;
  select2(N - mq - 1, mq - 1, v, a_hi, a_lo);
  const double m = robust_mean(N, a_hi, a_lo, [&](bool first, double mm, double inv, double (&ev)[3], double (&od)[3]) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const uint32_t e = lane + 64 * c;
      if (e < N) {
        double x[3];
        mean_terms(first, mm, inv, v[c], x);
#pragma unroll
        for (int q = 0; q < 3; ++q) terms[w][2 * q + (e & 1)][e / 2] = x[q];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    double acc = 0.0;
    if (lane < 6) {
      const uint32_t steps = (N + 1 - (lane & 1)) / 2;
      const double* p = terms[w][lane];
      uint32_t i = 0;
      for (; i + 8 <= steps; i += 8) {
        double2 t[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) t[q] = *reinterpret_cast<const double2*>(p + i + 2 * q);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc += t[q].x;
          acc += t[q].y;
        }
      }
      for (; i < steps; ++i) acc += p[i];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      ev[q] = lane_value(acc, 2 * q);
      od[q] = lane_value(acc, 2 * q + 1);
    }
  });
  const uint32_t half = N / 2, other = N % 2 == 0 ? half - 1 : half;
  double o0 = 0, o1 = 0;
  select2(half, other, l, o0, o1);
  const double med = mid_of(N, o0, o1);
  double d[C];
#pragma unroll
  for (int c = 0; c < C; ++c) d[c] = fabs(l[c] - med);
  select2(half, other, d, o0, o1);
  const double sig = 1.4826 * mid_of(N, o0, o1);
  if (lane == 0 && blockIdx.x * 4 + w < nleaves) {
    out[2 * (size_t)leaf] = m;
    out[2 * (size_t)leaf + 1] = sig * sig;
  }
}

}  // namespace

hipError_t launch_normalise(const double* X, uint32_t fs, const uint32_t* frames, const double* scales,
                            uint32_t items, double* Z, hipStream_t s) {
  if (items == 0) return hipSuccess;
  hipLaunchKernelGGL(k_normalise, dim3(std::min((fs + 255) / 256, 64u), items), dim3(256), 0, s, X, fs, frames,
                     scales, Z);
  return hipGetLastError();
}

hipError_t launch_split_stats(const double* Z, uint32_t n, uint32_t items, const uint32_t* blocks, uint32_t nblocks,
                              bool ordered, double* stat, hipStream_t s) {
  if (nblocks == 0 || items == 0) return hipSuccess;
  if (ordered)
    hipLaunchKernelGGL(k_split_stats<true>, dim3(nblocks, items), dim3(256), 0, s, Z, n, blocks, nblocks, stat);
  else
    hipLaunchKernelGGL(k_split_stats<false>, dim3(nblocks, items), dim3(256), 0, s, Z, n, blocks, nblocks, stat);
  return hipGetLastError();
}

uint32_t leaf_class(uint32_t s) { return s * s <= kWaveLeaf ? 0 : s * s <= 256 * kLeafCache ? 1 : 2; }

hipError_t launch_leaf_stats(const double* Z, uint32_t n, const uint32_t* leaves, const uint32_t count[3],
                             const uint64_t* boff, double* laps, double* out, hipStream_t s) {
  const uint32_t small = count[0], mid = count[1], big = count[2];
  // the longest first
  if (big > 0) {
    const uint32_t* Lf = leaves + 4 * (size_t)(small + mid);
    hipLaunchKernelGGL(k_leaf_prep, dim3(std::min<uint32_t>((n * n + 255) / 256, 64), big), dim3(256), 0, s, Z, n, Lf,
                       boff, laps);
    hipLaunchKernelGGL(k_leaf_stats<true>, dim3(big), dim3(1024), 0, s, Z, n, Lf, boff, laps,
                       out + 2 * (size_t)(small + mid));
  }
  if (mid > 0)
    hipLaunchKernelGGL(k_leaf_stats<false>, dim3(mid), dim3(256), 0, s, Z, n, leaves + 4 * (size_t)small, nullptr,
                       nullptr, out + 2 * (size_t)small);
  if (small > 0)
    hipLaunchKernelGGL(k_leaf_wave, dim3((small + 3) / 4), dim3(256), 0, s, Z, n, leaves, small, out);
  return hipGetLastError();
}

}  // namespace pgsvt
