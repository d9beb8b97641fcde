// overlap.hip -- overlap-add of the thresholded patches (src/svt.hpp:121-167)
// and its bookkeeping: patches binned by column, cover counts, the leading
// singular vectors by patch, and the sums of the risk.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "common.hpp"
#include "kernels.hpp"
#include "lanes.hpp"

namespace pgsvt {

namespace {

// Strip of a frame that one workgroup of the overlap-add owns: tr rows x tc
// columns, accumulated in LDS.  Column-major frames make a strip of whole
// columns one run of memory and the patches that reach it one run of the
// column bins, so strips take every row; only frames above 2,048 rows are
// cut.  From 192 rows, up to 6,144 cells (48 KB, 3 workgroups a CU) and 512
// threads: wide strips repeat little halo (bs - 1 columns), 24 waves a CU
// cover the loads (searches, ms a call for 8, 12, 16 and 24 columns: 256 rows
// 35.5, 32.2, 29.6, 28.4, with 256 threads 30.1, 28.8, 30.9, 35.4; 512 rows
// 12 columns 24.2, with 256 threads and 8 columns 30.8).  Smaller frames take
// 256 threads and fewer columns a strip, so that a call of a few windows
// still has a workgroup for every CU (128 rows: 16 columns 3.9, 12 4.1, 8
// 4.4); patches above 4 x 4, with a wider halo, more.
struct Strips {
  uint32_t tr, tc, ld, nr, nc, threads;  // ld: column stride in LDS; nr x nc strips a frame
};
Strips strips_of(uint32_t n, uint32_t bs) {
  Strips s;
  s.tr = std::min(n, 2048u);
  if (n >= 192) {
    s.threads = 512;
    s.tc = (s.tr <= 1024 ? 6144 : 7600) / s.tr;
  } else {
    s.threads = 256;
    s.tc = bs <= 4 ? std::min(16u, std::max(4u, n / 8)) : std::min({4096 / n, 32u, std::max(8u, n / 4)});
  }
  // 8 lanes of a half-wave's row group and the 4 patch columns of a row
  // meet in distinct banks when the stride is 8 mod 32 cells
  s.ld = ((s.tr + 23) / 32) * 32 + 8;
  s.nr = (n + s.tr - 1) / s.tr;
  s.nc = (n + s.tc - 1) / s.tc;
  return s;
}
// cells a thread holds at a time where a strip is summed by magnitude
constexpr int kCellsHeld = 8;
// strips of the cover counts: their two LDS arrays stay within 60 KB
Strips cover_strips(uint32_t n, uint32_t bs) {
  Strips s{};
  s.tc = std::min(n, 16u);
  const uint32_t most = (60 * 256 / (s.tc + bs - 1) - bs) / 2;
  s.tr = n <= most ? n : std::min(most, 256u);
  s.nr = (n + s.tr - 1) / s.tr;
  s.nc = (n + s.tc - 1) / s.tc;
  return s;
}

// column bins of a frame: one per patch column, or 2^shift columns a bin
// where a frame has more columns than the counters in LDS
constexpr uint32_t kMaxBins = 8192;
uint32_t bin_shift(uint32_t n1) {
  uint32_t sh = 0;
  while (((n1 - 1) >> sh) + 1 > kMaxBins) ++sh;
  return sh;
}

// as in kernels.hip: workgroups go to the 8 XCDs round-robin by linear id;
// each XCD gets one contiguous range of logical blocks
__device__ __forceinline__ void xcd_block(uint32_t& bx, uint32_t& by) {
  constexpr uint32_t kXcd = 8;
  const uint32_t total = gridDim.x * gridDim.y;
  const uint32_t lin = blockIdx.y * gridDim.x + blockIdx.x;
  const uint32_t x = lin % kXcd, idx = lin / kXcd, q = total / kXcd, r = total % kXcd;
  const uint32_t logical = x * q + min(x, r) + idx;
  bx = logical % gridDim.x;
  by = logical / gridDim.x;
}

// ------------------------------------------------------------- binning --
// Counting sort of one frame's patches by the column of their position, one
// workgroup per (window, frame): recs [nb][nw][p_sel] = (position, patch)
// by column, off [nb][nw][bins + 1].  The order inside a column is left to
// the LDS atomics: every sum over the records is one of integers (the
// overlap-add, the cover counts), which no order changes.
__global__ __launch_bounds__(1024) void k_bin_columns(const int32_t* __restrict__ pos, const uint32_t* __restrict__ sel,
                                                      uint32_t p_sel, uint32_t p_all, uint32_t nw, uint32_t n1,
                                                      uint32_t bins, uint32_t shift, int32_t* __restrict__ off,
                                                      int2* __restrict__ recs) {
  __shared__ int32_t h[kMaxBins];
  __shared__ int32_t wsum[16];
  const size_t tab = (size_t)blockIdx.y * nw + blockIdx.x;
  const int32_t* P = pos + tab * p_all;
  const bool all = p_sel == p_all;  // step 1: identity selection
  for (uint32_t i = threadIdx.x; i < bins; i += 1024) h[i] = 0;
  __syncthreads();
  auto bin_of = [&](int32_t pk) { return min((uint32_t)pk >> 16, n1 - 1) >> shift; };
  for (uint32_t p = threadIdx.x; p < p_sel; p += 1024) atomicAdd(&h[bin_of(P[all ? p : sel[p]])], 1);
  __syncthreads();
  // exclusive scan: thread t owns `per` consecutive bins
  const uint32_t per = (bins + 1023) / 1024, lane = threadIdx.x % 64, w = threadIdx.x / 64;
  const uint32_t lo = min(threadIdx.x * per, bins), hi = min(lo + per, bins);
  int32_t sum = 0;
  for (uint32_t i = lo; i < hi; ++i) sum += h[i];
  int32_t incl = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t y = __shfl_up(incl, o, 64);
    incl += lane >= (uint32_t)o ? y : 0;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  int32_t at = incl - sum;
  for (uint32_t k = 0; k < w; ++k) at += wsum[k];
  int32_t* O = off + tab * (bins + 1);
  for (uint32_t i = lo; i < hi; ++i) {
    const int32_t c = h[i];
    O[i] = at;
    h[i] = at;
    at += c;
  }
  if (threadIdx.x == 0) O[bins] = (int32_t)p_sel;
  __syncthreads();
  int2* R = recs + tab * p_sel;
  for (uint32_t p = threadIdx.x; p < p_sel; p += 1024) {
    const int32_t pk = P[all ? p : sel[p]];
    const int32_t slot = atomicAdd(&h[bin_of(pk)], 1);
    const uint32_t r = min((uint32_t)pk & 0xffffu, n1 - 1), c = min((uint32_t)pk >> 16, n1 - 1);
    R[slot] = make_int2((int32_t)(r | c << 16), (int32_t)p);
  }
}

// --------------------------------------------------------------- cover --
// W of src/svt.hpp:157-163, the number of patches over each voxel, as 1/W
// (FP64, 0 where nothing covers it) and, for the divergence sum, delta2/W.
// One workgroup per strip and frame: a histogram of the patch positions in
// LDS, then box sums down and across.  wstat[b (2 + nw) + 2 + k]: the largest W
// of frame k (the overlap-add's headroom).
__global__ __launch_bounds__(256) void k_cover(const int2* __restrict__ recs, const int32_t* __restrict__ off,
                                               const uint8_t* __restrict__ d2, uint32_t n, uint32_t nw, uint32_t n1,
                                               uint32_t bs, uint32_t p_sel, uint32_t bins, uint32_t shift, Strips st,
                                               double d2neg, double d2pos, double* __restrict__ invw,
                                               float* __restrict__ dw, uint32_t* __restrict__ wstat) {
  extern __shared__ int32_t cells[];
  __shared__ int32_t wmax[4];
  const uint32_t hr = st.tr + bs - 1, hc = st.tc + bs - 1;  // positions that reach the strip
  int32_t* H = cells;            // [hc][hr] positions
  int32_t* S = cells + hr * hc;  // [hc][tr] sums down a patch column
  const uint32_t b = blockIdx.y, k = blockIdx.x % nw, strip = blockIdx.x / nw;
  const int r0 = (int)((strip % st.nr) * st.tr), c0 = (int)((strip / st.nr) * st.tc);
  const uint32_t rows = min(st.tr, n - r0), cols = min(st.tc, n - c0);
  const size_t tab = (size_t)b * nw + k;
  for (uint32_t i = threadIdx.x; i < hr * hc; i += blockDim.x) H[i] = 0;
  __syncthreads();
  const int pr0 = r0 - (int)bs + 1, pc0 = c0 - (int)bs + 1;  // first position
  const int32_t* O = off + tab * (bins + 1);
  const int32_t lo = O[(uint32_t)max(pc0, 0) >> shift];
  const int32_t hi = O[(min((uint32_t)c0 + cols - 1, n1 - 1) >> shift) + 1];
  const int2* R = recs + tab * p_sel;
  for (int32_t j = lo + (int32_t)threadIdx.x; j < hi; j += (int32_t)blockDim.x) {
    const int32_t pk = R[j].x;
    const uint32_t r = (uint32_t)((pk & 0xffff) - pr0), c = (uint32_t)(((pk >> 16) & 0xffff) - pc0);
    if (r < hr && c < hc) atomicAdd(&H[c * hr + r], 1);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < rows * hc; i += blockDim.x) {
    const uint32_t c = i / rows, r = i % rows;
    int32_t s = 0;
    for (uint32_t q = 0; q < bs; ++q) s += H[c * hr + r + q];
    S[c * st.tr + r] = s;
  }
  __syncthreads();
  int32_t most = 0;
  for (uint32_t i = threadIdx.x; i < rows * cols; i += blockDim.x) {
    const uint32_t c = i / rows, r = i % rows;
    int32_t w = 0;
    for (uint32_t q = 0; q < bs; ++q) w += S[(c + q) * st.tr + r];
    most = max(most, w);
    const uint32_t pv = k * n * n + (uint32_t)(r0 + r) + n * (uint32_t)(c0 + c);
    const double iw = w > 0 ? 1.0 / (double)w : 0.0;
    invw[(size_t)b * nw * n * n + pv] = iw;
    if (dw) dw[(size_t)b * nw * n * n + pv] = (float)((d2[pv] ? d2neg : d2pos) * iw);
  }
  for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o));
  if (threadIdx.x % 64 == 0) wmax[threadIdx.x / 64] = most;
  __syncthreads();
  if (threadIdx.x == 0)
    atomicMax(&wstat[b * (2 + nw) + 2 + k], (uint32_t)max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])));
}

// ---------------------------------------------------- leading vectors --
// By patch, from the U variant's factors: w_0 (w0 [nb][p_sel][m], may be
// null) and v_0 as one plane per frame (v0 [nb][nw][p_sel]), and the window's
// largest finite s_0 and the complement of its smallest above 0 (wstat[b (2 +
// nw)] and the next word, as the bits of a float).  A workgroup takes 64
// patches: 16 lanes read a patch's vectors, v_0 turns in LDS, so that both
// sides move whole lines.
__global__ __launch_bounds__(256) void k_lead(const float* __restrict__ factors, uint32_t nvar_stored, uint32_t p_sel,
                                              uint32_t nw, uint32_t m, uint32_t fstride, float* __restrict__ w0,
                                              float* __restrict__ v0, uint32_t* __restrict__ wstat) {
  __shared__ float tv[32][65];
  __shared__ uint32_t top[4], low[4];
  const uint32_t b = blockIdx.y, p0 = blockIdx.x * 64, SR = (nw + 3) & ~3u;
  const uint32_t g = threadIdx.x / 16, l = threadIdx.x % 16;
  uint32_t s = 0, c = 0;
  for (uint32_t q = 0; q < 4; ++q) {
    const uint32_t pl = q * 16 + g, p = p0 + pl;
    if (p >= p_sel) continue;
    const float* F = factors + ((size_t)b * nvar_stored * p_sel + p) * fstride;
    const float* FW = F + nw * SR;
    if (w0)
      for (uint32_t i = l; i < m; i += 16) w0[((size_t)b * p_sel + p) * m + i] = FW[i];
    for (uint32_t k = l; k < nw; k += 16) tv[k][pl] = F[k];
    if (l == 0) {
      const uint32_t u = __float_as_uint(FW[nw * m]);
      s = max(s, u < 0x7f800000u ? u : 0u);
      c = max(c, u - 1u < 0x7f7fffffu ? ~u : 0u);
    }
  }
  __syncthreads();
  for (uint32_t e = threadIdx.x; e < nw * 64; e += 256) {
    const uint32_t k = e / 64, pl = e % 64;
    if (p0 + pl < p_sel) v0[((size_t)b * nw + k) * p_sel + p0 + pl] = tv[k][pl];
  }
  for (int o = 32; o > 0; o >>= 1) {
    s = max(s, (uint32_t)__shfl_xor((int)s, o));
    c = max(c, (uint32_t)__shfl_xor((int)c, o));
  }
  if (threadIdx.x % 64 == 0) {
    top[threadIdx.x / 64] = s;
    low[threadIdx.x / 64] = c;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicMax(&wstat[b * (2 + nw)], max(max(top[0], top[1]), max(top[2], top[3])));
    atomicMax(&wstat[b * (2 + nw) + 1], max(max(low[0], low[1]), max(low[2], low[3])));
  }
}

// --------------------------------------------------------- overlap-add --
struct OverlapArgs {
  const float *factors, *dr, *rows, *w0, *v0;
  const int2* recs;
  const int32_t* off;
  const double *invw, *u64;
  const WinMeta* meta;
  const uint32_t *wl, *wstat;
  double *out, *partial;
  uint32_t n, nw, n1, p_sel, fstride, nvar_stored, nk, bins, shift;
  int mode;
  Strips st;
};

// BS consecutive floats, as wide as their alignment allows (the start is a
// multiple of BS floats into a block of M floats that is 16-byte aligned)
template <int BS>
__device__ __forceinline__ void load_run(const float* __restrict__ p, float (&x)[BS]) {
  if constexpr (BS % 4 == 0) {
#pragma unroll
    for (int i = 0; i < BS / 4; ++i) {
      const float4 t = reinterpret_cast<const float4*>(p)[i];
      x[4 * i] = t.x;
      x[4 * i + 1] = t.y;
      x[4 * i + 2] = t.z;
      x[4 * i + 3] = t.w;
    }
  } else if constexpr (BS % 2 == 0) {
#pragma unroll
    for (int i = 0; i < BS / 2; ++i) {
      const float2 t = reinterpret_cast<const float2*>(p)[i];
      x[2 * i] = t.x;
      x[2 * i + 1] = t.y;
    }
  } else {
#pragma unroll
    for (int i = 0; i < BS; ++i) x[i] = p[i];
  }
}

// A strip's sums with a quantum for each class of 2^27 in magnitude, in FP64
// bits into the cells; each(f) calls f(x, cell, row) for every column of the
// thread's records.  The first walk finds the largest column and the cells that
// NaN or infinities reach (a cell's bits 1, 2, 4), each further one adds up
// the columns of one class (by the sum of their finite |x|) and finds the
// largest below it; the classes' sums are added from the largest down.  Every
// column is held to 2^-25 of its own |x|, in any order, and a strip costs a few
// walks (256 x 256 x 3, half of it 1e-20 of the rest, plain threshold 0: 0.25 ms
// a lambda, 0.08 where no strip comes here; a walk of the strip's records for
// each cell that is not finite 6.4).  The sums between the classes stay in
// registers, kCellsHeld a thread, so a strip of more cells takes its parts one
// after the other; and the cells' places are worked out anew at each use:
// registers held here cost the whole kernel waves (16 sums a thread and their
// addresses: four waves per SIMD for 4 x 4, 16 sums alone six for 8 x 8
// against seven).
template <int BS, bool CUT, class Each>
__device__ __forceinline__ void sum_by_magnitude(unsigned long long* acc, const Strips& st, uint32_t rows,
                                                 uint32_t cols, int head, Each each) {
  __shared__ unsigned long long top;  // the largest column left (bits of a non-negative double)
  const uint32_t part = (uint32_t)kCellsHeld * blockDim.x;
#pragma unroll 1
  for (uint32_t v0 = 0; v0 < rows * cols; v0 += part) {
    double run[kCellsHeld];
    // the part's cells: count of acc from first
    const uint32_t first = v0 / rows * st.ld + v0 % rows;
    const uint32_t v1 = v0 + part, count = (v1 < rows * cols ? v1 / rows * st.ld + v1 % rows : cols * st.ld) - first;
    auto own = [&](auto f) {
      uint32_t t = v0 + threadIdx.x;
      asm volatile("" : "+v"(t));
#pragma unroll
      for (int i = 0; i < kCellsHeld; ++i) {
        const uint32_t v = t + (uint32_t)i * blockDim.x;
        if (v < rows * cols) f(i, acc[v / rows * st.ld + v % rows]);
      }
    };
    auto clear = [&] {
      for (uint32_t c = threadIdx.x; c < count; c += blockDim.x) acc[first + c] = 0ull;
      if (threadIdx.x == 0) top = 0ull;
      __syncthreads();
    };
    auto inside = [&](uint32_t cell, int row) { return (!CUT || (uint32_t)row < rows) && cell - first < count; };
    auto magnitude = [](const float(&x)[BS]) {
      double m = 0.0;
      for (int q = 0; q < BS; ++q) m += __builtin_isfinite(x[q]) ? fabs((double)x[q]) : 0.0;
      return m;
    };
    double most = 0.0;
    clear();
    each([&](const float(&x)[BS], uint32_t cell, int row) {
      most = fmax(most, magnitude(x));
      for (int q = 0; q < BS; ++q)
        if (!__builtin_isfinite(x[q]) && inside(cell + q, row + q))
          atomicOr(&acc[cell + q], x[q] != x[q] ? 1ull : x[q] > 0.f ? 2ull : 4ull);
    });
    atomicMax(&top, __builtin_bit_cast(unsigned long long, most));
    __syncthreads();
    own([&](int i, unsigned long long bits) {
      run[i] = (bits & 1ull) || (bits & 6ull) == 6ull ? __builtin_nan("")
               : bits & 2ull                          ? __builtin_inf()
               : bits & 4ull                          ? -__builtin_inf()
                                                      : 0.0;
    });
    for (;;) {
      const double t = __builtin_bit_cast(double, top);
      __syncthreads();
      if (!(t > 0.0)) break;  // (each class starts below the one before: 48 at most)
      clear();
      const int e = ilogb(t) + 1;
      const double quantum = ldexp(1.0, e - 51 + head), magic = 1.5 * ldexp(1.0, e + 1 + head);
      const double high = ldexp(1.0, e), low = ldexp(1.0, e - 27 + head);
      most = 0.0;
      each([&](const float(&x)[BS], uint32_t cell, int row) {
        const double m = magnitude(x);
        if (m < low) most = fmax(most, m);
        if (!(m >= low && m < high)) return;
        for (int q = 0; q < BS; ++q) {
          const unsigned long long y = __builtin_bit_cast(unsigned long long, (double)x[q] + magic) -
                                       __builtin_bit_cast(unsigned long long, magic);
          if (__builtin_isfinite(x[q]) && inside(cell + q, row + q)) atomicAdd(&acc[cell + q], y);
        }
      });
      atomicMax(&top, __builtin_bit_cast(unsigned long long, most));
      __syncthreads();
      own([&](int i, unsigned long long bits) { run[i] += (double)(long long)bits * quantum; });
    }
    own([&](int i, unsigned long long& cell) { cell = __builtin_bit_cast(unsigned long long, run[i]); });
  }
}

// Uhat = (sum of the patches' rows over each voxel) / W.  The row of patch p
// in frame k is B[q][k] = d_0 w_0[q] v_0[k] (lead_product) where the patch
// keeps rank 0 alone (d_0 > 0, by patch, from k_round_prep), and the row that
// k_rows stored where it keeps more (d_0 < 0).
//
// A workgroup owns a strip of one frame and walks the records of the patches
// that reach it, one lane per patch column of BS elements, adding each
// element to the strip's cells in LDS as a 64-bit integer: x is
// rounded to a multiple of a quantum q (x + 1.5 2^52 q leaves the multiple
// in the low bits of the double) and the integers are added by ds_add_u64.
// Integer sums are the same in every order, so the result is reproducible
// without a sort.  q = 2^(e - 51) with 2^e above the sum of any column's
// |x| (the window's largest s_0 bounds the 2-norm of a row), raised where
// more than 2^11 patches pile on a voxel of the frame (without motion
// estimation every patch of the other frames lies on (0, 0); the output frame's
// sums must not pay for them): an FP32 contribution of at least
// 2^-24 of the window's largest s_0 is held exactly, a smaller one to 2^-48
// of it, which is 2^-25 of its own patch's s_0 or finer in every window whose
// s_0 stay within a factor of 2^24 (16-bit counts do).  Strips with a column
// that this does not hold, one whose |x| reach 2^e or are no numbers, or,
// in a window of wider s_0, one whose |x| sum to less than 2^24 q, are
// summed again by magnitude (sum_by_magnitude).
//
// Bound: instruction issue (355 vector instructions per 64 voxels, 17.1 of the
// 26.0 ms of 1.9 G voxels) and the LDS atomics (about 10 ms), then memory (28
// bytes a voxel).  256 x 256 x 15 windows at searched lambdas: 13.7 ps a voxel.
// The
// form before (rows of a 32 x 8 tile staged in LDS from bucket-sorted rows,
// each voxel reading its 16 positions and looping over further patches of a
// position) issued 1,197 vector instructions per 64 voxels, at 4 cycles each
// all of its 33 ps.  Further ranks formed here, as a row needs them, instead
// of by k_rows: 128 x 128 x 30 over 64 lambdas 50.9 ms a call instead of 31.7
// (every frame reads each kept rank's w_r again).
//   mode 0: risk sums per block: sum Uhat^2, sum Uhat, sum Uhat U, sum U, sum U^2
//   mode 1: final frame: Y(:,:,out) = uMax * Uhat(:,:,ref)
//   mode 2: whole window volume of slot 0 into out
// CUT: strips that do not hold every row of the frame.
template <int BS, bool CUT>
__global__ __launch_bounds__(512) void k_overlap(const OverlapArgs a) {
  constexpr int M = BS * BS, LG = BS <= 2 ? 2 : BS <= 4 ? 4 : BS <= 8 ? 8 : 16;
  constexpr int U = BS <= 4 ? 4 : BS <= 8 ? 2 : 1;  // rows in flight per lane group
  // 2^LOGC bounds sum |x| of a column over its 2-norm (sqrt(BS)), once doubled
  constexpr int LOGC = BS <= 4 ? 3 : 4;
  extern __shared__ unsigned long long acc[];  // [tc][ld] cells
  __shared__ double sm[5][8];
  __shared__ uint32_t beyond;  // a column the quantum does not hold
  const Strips st = a.st;
  uint32_t bx, slot;
  xcd_block(bx, slot);
  const uint32_t b = a.wl[slot];
  const uint32_t mref = a.meta[b].ref;
  const uint32_t nk = a.mode == 1 ? 1 : a.nk, i = bx % nk, strip = bx / nk;
  // mode 0 covers nk frames of the window: all, or nk spread over it
  // (k_i = i (nw - 1) / (nk - 1)); mode 1 the reference frame
  const uint32_t k = a.mode == 1 ? mref : (nk == a.nw ? i : (nk > 1 ? i * (a.nw - 1) / (nk - 1) : a.nw / 2));
  const uint32_t n = a.n;
  const int r0 = CUT ? (int)((strip % st.nr) * st.tr) : 0;
  const int c0 = (int)((CUT ? strip / st.nr : strip) * st.tc);
  const uint32_t rows = CUT ? min(st.tr, n - r0) : n, cols = min(st.tc, n - c0);
  const size_t tab = (size_t)b * a.nw + k;
  const int32_t* O = a.off + tab * (a.bins + 1);
  const int32_t lo = O[(uint32_t)max(c0 - BS + 1, 0) >> a.shift];
  const int32_t hi = O[(min((uint32_t)c0 + cols - 1, a.n1 - 1) >> a.shift) + 1];
  // quantum and bound (see above)
  const uint32_t* fig = a.wstat + b * (2 + a.nw);
  const float smax = __uint_as_float(fig[0]), smin = __uint_as_float(~fig[1]);  // (NaN: no s_0 above 0)
  const uint32_t wmax = fig[2 + k];
  const int e = (smax > 0.f ? ilogbf(smax) : 0) + LOGC;
  const int head = max(0, (int)(32 - __clz((int)wmax | 1)) - 11);
  const double quantum = ldexp(1.0, e - 51 + head), magic = 1.5 * ldexp(1.0, e + 1 + head);
  const uint32_t bound = __float_as_uint(ldexpf(1.f, min(e, 127)));
  const float dim = ldexpf(1.f, min(e - 27 + head, 127));
  const uint32_t least = smin < dim ? min(__float_as_uint(dim), bound) : 0u, span = bound - least;
  const uint32_t mhi = (uint32_t)(__double_as_longlong(magic) >> 32);
  const uint32_t cells = st.tc * st.ld;
  for (uint32_t c = threadIdx.x; c < cells; c += blockDim.x) acc[c] = 0ull;
  if (threadIdx.x == 0) beyond = 0;
  __syncthreads();

  const int2* R = a.recs + tab * a.p_sel;
  const float* D = a.dr + (size_t)slot * a.nw * a.p_sel;  // [rank][patch]
  const float* V = a.v0 + tab * a.p_sel;
  const int cb = (int)(threadIdx.x % LG), grp = (int)(threadIdx.x / LG), G = (int)(blockDim.x / LG);
  const uint32_t sr = (a.nw + 3) & ~3u;
  const float* Fu = a.factors + (size_t)b * a.nvar_stored * a.p_sel * a.fstride;  // the U variant
  // w_0 by patch: a 4 x 4 patch's 64 bytes share a cache line with its
  // neighbour's in w0, larger ones fill their lines in the factors
  const float* W = BS <= 4 ? a.w0 + (size_t)b * a.p_sel * M : Fu + a.nw * sr;
  const size_t wst = BS <= 4 ? M : a.fstride;
  // stored rows of frame k
  const float* S = a.rows + ((size_t)slot * a.nw + k) * a.p_sel * M;
  // Three stages in flight: the records of the rows after the next ones, d_0
  // and v_0 of the next ones (by their patch), the row or w_0 of this one
  // (by its d_0), so that a round of rows waits for memory once.
  auto fetch = [&](int32_t j0, int2 (&r)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) r[u] = R[min(j0 + u * G, hi - 1)];
  };
  // column and row of the record's first element in the strip; false: the
  // lane's column lies outside it
  auto place = [&](int32_t j, int2 r, int& col, int& row) {
    col = ((r.x >> 16) & 0xffff) + cb - c0;
    row = (r.x & 0xffff) - r0;
    return j < hi && (LG == BS || cb < BS) && (uint32_t)col < cols && (!CUT || (row < (int)rows && row + BS > 0));
  };
  auto lead = [&](int32_t j0, const int2 (&r)[U], float (&d)[U], float (&v)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int col, row;
      d[u] = 0.f;
      v[u] = 0.f;
      if (place(j0 + u * G, r[u], col, row)) {
        d[u] = D[(uint32_t)r[u].y];
        v[u] = V[(uint32_t)r[u].y];
      }
    }
  };
  int2 rec[U], rec1[U];
  float d0[U], v[U];
  int32_t j0 = lo + grp;
  if (j0 < hi) {
    fetch(j0, rec);
    fetch(j0 + U * G, rec1);
    lead(j0, rec, d0, v);
  }
  for (; j0 < hi; j0 += U * G) {
    float x[U][BS];
    uint32_t cell[U], id[U];
    int row[U];  // (used by cut strips only)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int col;
      (void)place(j0 + u * G, rec[u], col, row[u]);
      cell[u] = (uint32_t)col * st.ld + (uint32_t)row[u];
      id[u] = (uint32_t)rec[u].y;
      if (d0[u] != 0.f) load_run<BS>((d0[u] < 0.f ? S + (size_t)id[u] * M : W + (size_t)id[u] * wst) + cb * BS, x[u]);
    }
    int2 rec2[U];
    float d1[U], v1[U];
    fetch(j0 + 2 * U * G, rec2);
    lead(j0 + U * G, rec1, d1, v1);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < BS; ++q) x[u][q] = d0[u] < 0.f ? x[u][q] : lead_product<(BS <= 4)>(d0[u], x[u][q], v[u]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (d0[u] == 0.f) continue;  // nothing kept, or outside the strip
      float mag = fabsf(x[u][0]);
#pragma unroll
      for (int q = 1; q < BS; ++q) mag += fabsf(x[u][q]);
      if (__float_as_uint(mag) - least >= span) {  // (NaN and infinity among them)
        if (mag != 0.f) beyond = 1;
        continue;
      }
#pragma unroll
      for (int q = 0; q < BS; ++q) {
        const double y = (double)x[u][q] + magic;
        uint2 h = __builtin_bit_cast(uint2, y);
        h.y -= mhi;
        if (!CUT || (uint32_t)(row[u] + q) < rows)
          __hip_atomic_fetch_add(&acc[cell[u] + q], __builtin_bit_cast(unsigned long long, h), __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      rec[u] = rec1[u];
      rec1[u] = rec2[u];
      d0[u] = d1[u];
      v[u] = v1[u];
    }
  }
  __syncthreads();

  const double umax = a.meta[b].uMax;
  const size_t oslice = (size_t)a.meta[b].out * n * n;
  const size_t base = tab * n * n + (size_t)r0 + (size_t)n * c0;
  const bool wide = beyond != 0;
  if (__builtin_expect(wide, 0))
    sum_by_magnitude<BS, CUT>(acc, st, rows, cols, head, [&](auto f) {
      for (int32_t j = lo + grp; j < hi; j += G) {
        const int2 r = R[j];
        int col, row;
        if (!place(j, r, col, row)) continue;
        const uint32_t id = (uint32_t)r.y;
        const float d = D[id], v0 = V[id];
        if (d == 0.f) continue;
        float x[BS];
        load_run<BS>((d < 0.f ? S + (size_t)id * M : W + (size_t)id * wst) + cb * BS, x);
        if (d > 0.f)
          for (int q = 0; q < BS; ++q) x[q] = lead_product<(BS <= 4)>(d, x[q], v0);
        f(x, (uint32_t)col * st.ld + (uint32_t)row, row);
      }
    });
  // cell of the strip's v-th voxel: column v / rows
  const uint32_t inv = (uint32_t)(((1ull << 32) + rows - 1) / rows);
  double s_q = 0, s_h = 0, s_hu = 0, s_u = 0, s_u2 = 0;
  for (uint32_t v = threadIdx.x; v < rows * cols; v += blockDim.x) {
    const uint32_t c = CUT ? v / rows : __umulhi(v, inv), r = v - c * rows;  // exact: rows * cols < 2^16
    const size_t at = base + (CUT ? r + (size_t)n * c : v);
    const uint32_t cell = c * st.ld + r;
    const double sum = wide ? __builtin_bit_cast(double, acc[cell]) : (double)(long long)acc[cell] * quantum;
    const double uh = sum * a.invw[at];
    if (a.mode == 0) {
      const double u = a.u64[at];
      s_q = fma(uh, uh, s_q);
      s_h += uh;
      s_hu = fma(uh, u, s_hu);
      s_u += u;
      s_u2 = fma(u, u, s_u2);
    } else if (a.mode == 1) {
      a.out[oslice + (at - tab * n * n)] = uh * umax;
    } else {
      a.out[at - (size_t)b * a.nw * n * n] = uh;
    }
  }
  if (a.mode != 0) return;
  for (int o = 32; o > 0; o >>= 1) {
    s_q += __shfl_xor(s_q, o);
    s_h += __shfl_xor(s_h, o);
    s_hu += __shfl_xor(s_hu, o);
    s_u += __shfl_xor(s_u, o);
    s_u2 += __shfl_xor(s_u2, o);
  }
  const int wv = (int)threadIdx.x / 64, waves = (int)blockDim.x / 64;
  if ((threadIdx.x & 63) == 0) {
    sm[0][wv] = s_q;
    sm[1][wv] = s_h;
    sm[2][wv] = s_hu;
    sm[3][wv] = s_u;
    sm[4][wv] = s_u2;
  }
  __syncthreads();
  if (threadIdx.x < 5) {
    double t = sm[threadIdx.x][0];
    for (int w = 1; w < waves; ++w) t += sm[threadIdx.x][w];
    a.partial[((size_t)slot * gridDim.x + bx) * 5 + threadIdx.x] = t;
  }
}

}  // namespace

uint32_t column_bins(const Shape& sh) { return ((sh.n1 - 1) >> bin_shift(sh.n1)) + 1; }

hipError_t launch_bins(const int32_t* pos, const uint32_t* sel, uint32_t nb, const Shape& sh, int32_t* off,
                       int2* recs, hipStream_t s) {
  hipLaunchKernelGGL(k_bin_columns, dim3(sh.nw, nb), dim3(1024), 0, s, pos, sel, sh.p_sel, sh.p_all, sh.nw, sh.n1,
                     column_bins(sh), bin_shift(sh.n1), off, recs);
  return hipGetLastError();
}

hipError_t launch_cover(const int32_t* off, const int2* recs, const uint8_t* d2, uint32_t nb, const Shape& sh,
                        double d2neg, double d2pos, double* invw, float* dw, uint32_t* wstat, hipStream_t s) {
  const Strips st = cover_strips(sh.nr, sh.bs);
  const size_t hr = st.tr + sh.bs - 1, hc = st.tc + sh.bs - 1;
  hipLaunchKernelGGL(k_cover, dim3(st.nr * st.nc * sh.nw, nb), dim3(256), (hr + st.tr) * hc * 4, s, recs, off, d2,
                     sh.nr, sh.nw, sh.n1, sh.bs, sh.p_sel, column_bins(sh), bin_shift(sh.n1), st, d2neg, d2pos, invw,
                     dw, wstat);
  return hipGetLastError();
}

hipError_t launch_lead(const float* factors, uint32_t nb, uint32_t nvar_stored, const Shape& sh, float* w0, float* v0,
                       uint32_t* wstat, hipStream_t s) {
  hipLaunchKernelGGL(k_lead, dim3((sh.p_sel + 63) / 64, nb), dim3(256), 0, s, factors, nvar_stored, sh.p_sel, sh.nw,
                     sh.m, sh.fstride, w0, v0, wstat);
  return hipGetLastError();
}

uint32_t overlap_blocks(const Shape& sh, int mode, uint32_t nk) {
  const Strips st = strips_of(sh.nr, sh.bs);
  return st.nr * st.nc * (mode == 1 ? 1 : (nk == 0 || nk > sh.nw ? sh.nw : nk));
}

hipError_t launch_overlap(const OverlapSrc& src, const double* invw, const double* u64, const WinMeta* meta,
                          const uint32_t* wl, uint32_t na, const Shape& sh, int mode, double* out, double* partial,
                          hipStream_t s, uint32_t nk) {
  const Strips st = strips_of(sh.nr, sh.bs);
  OverlapArgs a;
  a.factors = src.factors;
  a.dr = src.dr;
  a.rows = src.rows;
  a.w0 = src.w0;
  a.v0 = src.v0;
  a.recs = src.recs;
  a.off = src.off;
  a.invw = invw;
  a.u64 = u64;
  a.meta = meta;
  a.wl = wl;
  a.wstat = src.wstat;
  a.out = out;
  a.partial = partial;
  a.n = sh.nr;
  a.nw = sh.nw;
  a.n1 = sh.n1;
  a.p_sel = sh.p_sel;
  a.fstride = sh.fstride;
  a.nvar_stored = src.nvar_stored;
  a.nk = nk == 0 || nk > sh.nw ? sh.nw : nk;
  a.bins = column_bins(sh);
  a.shift = bin_shift(sh.n1);
  a.mode = mode;
  a.st = st;
  const dim3 grid(overlap_blocks(sh, mode, nk), na);
  const size_t lds = (size_t)st.tc * st.ld * 8;
#define PG_OV(B)                                                                                   \
  case B:                                                                                          \
    if (st.nr > 1)                                                                                 \
      hipLaunchKernelGGL((k_overlap<B, true>), grid, dim3(st.threads), lds, s, a);                 \
    else                                                                                           \
      hipLaunchKernelGGL((k_overlap<B, false>), grid, dim3(st.threads), lds, s, a);                \
    return hipGetLastError();
  switch (sh.bs) {
    PG_OV(2) PG_OV(3) PG_OV(4) PG_OV(5) PG_OV(6) PG_OV(7) PG_OV(8) PG_OV(16)
    default: return hipErrorInvalidValue;
  }
#undef PG_OV
}

}  // namespace pgsvt
