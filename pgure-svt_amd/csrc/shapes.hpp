// shapes.hpp -- the (patch size, window length) shapes the kernels are
// instantiated for.
#pragma once

#include <cstdint>

namespace pgsvt {

// shape table of the instantiated SVD / evaluation kernels (patch size,
// window frames, lanes per patch in the evaluation, lanes per matrix in the
// SVD)
#define PG_SHAPES(X) \
  X(4, 3, 16, 4) X(4, 5, 16, 4) X(4, 7, 16, 4) X(4, 9, 16, 4) X(4, 11, 16, 4) X(4, 13, 16, 4) X(4, 15, 16, 4) \
  X(2, 3, 16, 4) X(3, 3, 16, 4) X(3, 5, 16, 4) X(3, 7, 16, 4) X(3, 9, 16, 4) \
  X(6, 7, 64, 16) X(6, 15, 64, 16) X(6, 31, 64, 32) X(8, 7, 64, 16) X(8, 15, 64, 16) X(8, 31, 64, 32)

// second lanes-per-matrix mapping of the SVD for each shape, timed against
// the first by the autotuner of the batched path
#define PG_SVD_ALT(X) \
  X(4, 3, 8) X(4, 5, 8) X(4, 7, 8) X(4, 9, 8) X(4, 11, 8) X(4, 13, 8) X(4, 15, 8) \
  X(2, 3, 2) X(3, 3, 8) X(3, 5, 8) X(3, 7, 8) X(3, 9, 8) \
  X(6, 7, 32) X(6, 15, 32) X(6, 31, 64) X(8, 7, 32) X(8, 15, 32) X(8, 31, 64)

// Every other shape, FP32 only: the window length is known at run time
// (the kernels' RT form) up to NM frames.  (patch size, NM, lanes per
// matrix in the SVD, lanes per patch in the divergence factors and, for
// patches above 4 x 4, the evaluation; patches up to 4 x 4 evaluate fused,
// one thread per patch)
#define PG_GENERIC(X) \
  X(2, 16, 4, 16) X(3, 16, 4, 16) X(4, 16, 4, 16) \
  X(5, 16, 16, 64) X(5, 32, 16, 64) X(6, 16, 16, 64) X(6, 32, 32, 64) X(7, 16, 16, 64) X(7, 32, 32, 64) \
  X(8, 16, 32, 64) X(8, 32, 64, 64) X(16, 16, 64, 64)

inline bool shape_exact(uint32_t bs, uint32_t nw) {
#define PG_CHK(B, N, L, LS) \
  if (bs == B && nw == N) return true;
  PG_SHAPES(PG_CHK)
#undef PG_CHK
  return false;
}

// the generic family that runs a shape: its NM, or 0
inline uint32_t shape_generic(uint32_t bs, uint32_t nw) {
  if (nw < 1) return 0;
#define PG_GCHK(B, NM, L, LE) \
  if (bs == B && nw <= NM) return NM;
  PG_GENERIC(PG_GCHK)
#undef PG_GCHK
  return 0;
}

}  // namespace pgsvt
