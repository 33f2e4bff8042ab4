// Undecimated periodic 2D wavelet transform (analysis / synthesis passes).
#pragma once

#include "shx_common.h"

namespace shx {

constexpr int RDWT_MAX_TAPS = 32;

// Per-tap coefficients of the two filters one pass applies.
struct RdwtFilt {
  int lh;
  float f0[RDWT_MAX_TAPS];
  float f1[RDWT_MAX_TAPS];
};

// x (nimg x m x n) -> yl (nimg x m x n), yh (nimg x m x 3nL); f holds the
// analysis taps (a0, a1); tmp: 2*m*n floats per image.
hipError_t rdwt_analysis(const float* x, float* yl, float* yh, float* tmp, int m, int n, int L, const RdwtFilt& f,
                         int nimg, hipStream_t s);
// yl, yh -> x; f holds the synthesis taps (g0, g1).  th (rdwt_fused only): 1 + 3 L
// device thresholds (yl first); the bands are soft-thresholded as they are read.
hipError_t rdwt_synthesis(const float* yl, const float* yh, float* x, float* tmp, int m, int n, int L,
                          const RdwtFilt& f, int nimg, hipStream_t s, const float* th = nullptr);
// Whether a transform of rows of n, L levels and lh taps runs its levels fused.
bool rdwt_fused(int n, int L, int lh);
// Backward of the soft-thresholded bands of b under the synthesis' output gradient
// g (rdwt_fused only): gyl, gyh = the synthesis' transpose of g masked by
// |bands of b| > th, gth += the threshold gradients.  f: analysis taps; tmp:
// 4*m*n floats per image.
hipError_t rdwt_shrink_mask(const float* b, const float* g, float* gyl, float* gyh, float* tmp, int m, int n, int L,
                            const RdwtFilt& f, const float* th, float* gth, int nimg, hipStream_t s);

}  // namespace shx
