// Undecimated (redundant) periodic 2D wavelet transform, Rice Wavelet Toolbox
// semantics, as the reference's mrdwt/mirdwt (shearcuda/src/mrdwt_r.h:70-207,
// mirdwt_r.h:92-218; GPU shearcuda/src_cuda/mrdwt_cuda.cpp:220-253,
// mirdwt_cuda.cpp:210-255).
//
// Row-major m x n images; yh is m x 3nL, level l (1-based) in columns
// [3n(l-1), 3nl) as [lh hl hh] (first letter: filtering along a row).
// Level l uses dilation sf = 2^(l-1) and periodic indexing.
//   analysis  (mrdwt):  out[i] = sum_j in[(i + j*sf) mod n] * a[j]
//             a0[j] = h[j],  a1[j] = h[lh-1-j] * (-1 if lh-1-j is even)
//             rows: A = a0 (x) yl, B = a1 (x) yl; columns: yl = a0 A,
//             lh = a1 A, hl = a0 B, hh = a1 B
//   synthesis (mirdwt): out[i] = sum_t d[(i - t*sf) mod n] * g[t]
//             g0[t] = h[t]/2,  g1[t] = h[lh-1-t]/2 * (-1 if t is odd)
//             columns: X = g0 x + g1 lh, XH = g0 hl + g1 hh; rows:
//             x = g0 X + g1 XH
// The adjoint of the analysis is the synthesis with filters 2g and the adjoint
// of the synthesis is the analysis with filters a/2 (host side picks them).
#include "rdwt.h"

#include <type_traits>

namespace shx {

__device__ __forceinline__ int wrap(int i, int n) {
  i %= n;
  return i < 0 ? i + n : i;
}

// analysis along rows: A, B from yl
__global__ void k_rdwt_rows_an(const float* __restrict__ yl, float* __restrict__ A, float* __restrict__ B, int m,
                               int n, int sf, RdwtFilt f, long long img_stride, long long tmp_stride) {
  const int img = blockIdx.z;
  const int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (c >= n) return;
  const float* row = yl + (size_t)img * img_stride + (size_t)r * n;
  float a = 0.f, b = 0.f;
  for (int j = 0; j < f.lh; ++j) {
    const float v = row[wrap(c + j * sf, n)];
    a = fmaf(f.f0[j], v, a);
    b = fmaf(f.f1[j], v, b);
  }
  const size_t o = (size_t)img * tmp_stride + (size_t)r * n + c;
  A[o] = a;
  B[o] = b;
}

// analysis along columns: yl, lh, hl, hh of level `lev` from A, B
__global__ void k_rdwt_cols_an(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ yl,
                               float* __restrict__ yh, int m, int n, int sf, int L, int lev, RdwtFilt f,
                               long long img_stride, long long yh_stride, long long tmp_stride) {
  const int img = blockIdx.z;
  const int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (c >= n) return;
  const float* a = A + (size_t)img * tmp_stride + c;
  const float* b = B + (size_t)img * tmp_stride + c;
  float ll = 0.f, lh = 0.f, hl = 0.f, hh = 0.f;
  for (int j = 0; j < f.lh; ++j) {
    const int rr = wrap(r + j * sf, m);
    const float va = a[(size_t)rr * n], vb = b[(size_t)rr * n];
    ll = fmaf(f.f0[j], va, ll);
    lh = fmaf(f.f1[j], va, lh);
    hl = fmaf(f.f0[j], vb, hl);
    hh = fmaf(f.f1[j], vb, hh);
  }
  yl[(size_t)img * img_stride + (size_t)r * n + c] = ll;
  float* yr = yh + (size_t)img * yh_stride + (size_t)r * 3 * n * L + (size_t)3 * n * (lev - 1);
  yr[c] = lh;
  yr[n + c] = hl;
  yr[2 * n + c] = hh;
}

// synthesis along columns: X, XH from x and the level's (lh, hl, hh)
__global__ void k_rdwt_cols_syn(const float* __restrict__ x, const float* __restrict__ yh, float* __restrict__ X,
                                float* __restrict__ XH, int m, int n, int sf, int L, int lev, RdwtFilt f,
                                long long img_stride, long long yh_stride, long long tmp_stride) {
  const int img = blockIdx.z;
  const int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (c >= n) return;
  const float* xi = x + (size_t)img * img_stride + c;
  const float* yb = yh + (size_t)img * yh_stride + (size_t)3 * n * (lev - 1) + c;
  const size_t yrow = (size_t)3 * n * L;
  float s0 = 0.f, s1 = 0.f;
  for (int t = 0; t < f.lh; ++t) {
    const int rr = wrap(r - t * sf, m);
    const float* yr = yb + (size_t)rr * yrow;
    s0 = fmaf(f.f0[t], xi[(size_t)rr * n], s0);
    s0 = fmaf(f.f1[t], yr[0], s0);
    s1 = fmaf(f.f0[t], yr[n], s1);
    s1 = fmaf(f.f1[t], yr[2 * n], s1);
  }
  const size_t o = (size_t)img * tmp_stride + (size_t)r * n + c;
  X[o] = s0;
  XH[o] = s1;
}

// synthesis along rows: x from X, XH
__global__ void k_rdwt_rows_syn(const float* __restrict__ X, const float* __restrict__ XH, float* __restrict__ x,
                                int m, int n, int sf, RdwtFilt f, long long img_stride, long long tmp_stride) {
  const int img = blockIdx.z;
  const int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (c >= n) return;
  const float* a = X + (size_t)img * tmp_stride + (size_t)r * n;
  const float* b = XH + (size_t)img * tmp_stride + (size_t)r * n;
  float s = 0.f;
  for (int t = 0; t < f.lh; ++t) {
    const int cc = wrap(c - t * sf, n);
    s = fmaf(f.f0[t], a[cc], s);
    s = fmaf(f.f1[t], b[cc], s);
  }
  x[(size_t)img * img_stride + (size_t)r * n + c] = s;
}

// ---- fused levels (filters of at most 8 taps) -----------------------------------
// One launch per level.  Row and column passes commute, so the column pass
// goes first: a thread owns one column and walks down the rows of one phase
// (rows ph, ph + sf, ...: the dilated taps of a row are its neighbours there),
// keeping the taps' values in registers, and the two filtered rows pass
// through LDS to the row pass.  Every input value is read once per strip of K
// rows (plus the taps' LH - 1 rows of warm-up) and the intermediate planes of
// the separate passes, 4 planes of traffic per level, never reach memory.
// The separate passes below read every tap from global memory behind an
// integer remainder: calls of 295 and 345 us for the 3-level analysis and synthesis
// of 4 x 1000 x 1496 with 8 taps against 80 and 100 us here, 3.3 and 2.6 TB/s of
// the values that have to move (the transform's input and bands; bound by loads in
// flight).
struct RdwtLevel {
  const float* in;   // low band of the level (analysis: its input)
  float* out;        // analysis: next low band; synthesis: result
  float* yh;         // the level's [lh hl hh] rows: column 3n(lev-1) of yh
  int m, n, sf;
  int M;             // rows of a phase, m / sf
  int W;             // output columns per block
  int halo;          // columns before (synthesis) or after them that only feed taps; 0: the block holds whole rows
  long long ldh, is, ys;  // row stride of yh; image strides of in/out and yh
  // thresholded forms: thresholds of the level's three bands, of the low band
  // (the last level; else NULL), their gradients
  const float* th;
  const float* th_ll;
  float* gth;
  float* gth_ll;
  // the dual form: the second transform's low bands
  const float* in2;
  float* out2;
};
template <int LH>
struct RdwtTaps {
  float f0[LH], f1[LH];
};
constexpr int RT = 512;  // most columns a block holds

// Rows of a phase in order, wrapping at M.
struct PhaseRow {
  int r, M, sf, ph;
  __device__ __forceinline__ PhaseRow(int r0, const RdwtLevel& a, int phase) : r(r0 % a.M), M(a.M), sf(a.sf), ph(phase) {
    if (r < 0) r += M;
  }
  __device__ __forceinline__ int next() {
    const int g = r * sf + ph;
    r = r + 1 == M ? 0 : r + 1;
    return g;
  }
};

template <int LH, int K>
__global__ void __launch_bounds__(RT) k_rdwt_level_an(RdwtLevel a, RdwtTaps<LH> f) {
  __shared__ float lu[2][4][RT], lv[2][4][RT];
  const int i = threadIdx.x, ph = blockIdx.y % a.sf, r0 = (blockIdx.y / a.sf) * K;
  const int c = (blockIdx.x * a.W + i) % a.n;
  const bool put = i < a.W && (int)blockIdx.x * a.W + i < a.n;
  int at[LH];
#pragma unroll
  for (int j = 0; j < LH; ++j) at[j] = a.halo ? min(i + j * a.sf, RT - 1) : (i + j * a.sf) % a.n;
  const float* in = a.in + (size_t)blockIdx.z * a.is + c;
  float* out = a.out + (size_t)blockIdx.z * a.is + c;
  float* yh = a.yh + (size_t)blockIdx.z * a.ys + c;
  PhaseRow row(r0, a, ph);
  float w[LH + 3];
#pragma unroll
  for (int j = 0; j < LH - 1; ++j) w[j] = in[(size_t)row.next() * a.n];
#pragma unroll
  for (int s = 0; s < K / 4; ++s) {
#pragma unroll
    for (int q = 0; q < 4; ++q) w[LH - 1 + q] = in[(size_t)row.next() * a.n];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float u = 0.f, v = 0.f;
#pragma unroll
      for (int j = 0; j < LH; ++j) {
        u = fmaf(f.f0[j], w[q + j], u);
        v = fmaf(f.f1[j], w[q + j], v);
      }
      lu[s & 1][q][i] = u;
      lv[s & 1][q][i] = v;
    }
#pragma unroll
    for (int j = 0; j < LH - 1; ++j) w[j] = w[j + 4];
    __syncthreads();  // the two buffers alternate: one barrier per step
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = r0 + 4 * s + q;
      float ll = 0.f, lh = 0.f, hl = 0.f, hh = 0.f;
#pragma unroll
      for (int j = 0; j < LH; ++j) {
        const float u = lu[s & 1][q][at[j]], v = lv[s & 1][q][at[j]];
        ll = fmaf(f.f0[j], u, ll);
        lh = fmaf(f.f0[j], v, lh);
        hl = fmaf(f.f1[j], u, hl);
        hh = fmaf(f.f1[j], v, hh);
      }
      if (put && r < a.M) {
        const size_t g = (size_t)(r * a.sf + ph);
        out[g * a.n] = ll;
        float* y = yh + g * a.ldh;
        y[0] = lh;
        y[a.n] = hl;
        y[2 * a.n] = hh;
      }
    }
  }
}

// SOFT: the bands are soft-thresholded as they are read (8 x 512^2, 3 levels,
// 4 taps: 38 us of kernels; with a pass of its own over the bands 88).
template <int LH, int K, bool SOFT>
__global__ void __launch_bounds__(RT) k_rdwt_level_syn(RdwtLevel a, RdwtTaps<LH> f) {
  __shared__ float lu[2][4][RT], lv[2][4][RT];
  const int i = threadIdx.x, ph = blockIdx.y % a.sf, r0 = (blockIdx.y / a.sf) * K;
  const int c0 = blockIdx.x * a.W - a.halo + i;
  int c = c0 % a.n;
  if (c < 0) c += a.n;
  const bool put = i >= a.halo && i < a.halo + a.W && c0 < a.n;
  int at[LH];
#pragma unroll
  for (int j = 0; j < LH; ++j) {
    at[j] = a.halo ? max(i - j * a.sf, 0) : (i - j * a.sf) % a.n;
    if (at[j] < 0) at[j] += a.n;
  }
  const float* in = a.in + (size_t)blockIdx.z * a.is + c;
  float* out = a.out + (size_t)blockIdx.z * a.is + c;
  const float* yh = a.yh + (size_t)blockIdx.z * a.ys + c;
  PhaseRow row(r0 - (LH - 1), a, ph);
  float t0 = 0.f, t1 = 0.f, t2 = 0.f, tl = 0.f;
  const bool soft_ll = SOFT && a.th_ll;
  if constexpr (SOFT) {
    t0 = a.th[0];
    t1 = a.th[1];
    t2 = a.th[2];
    if (soft_ll) tl = a.th_ll[0];
  }
  float w[4][LH + 3];
  const auto load = [&](int k) {
    const size_t g = (size_t)row.next();
    const float* y = yh + g * a.ldh;
    w[0][k] = in[g * a.n];
    w[1][k] = y[0];
    w[2][k] = y[a.n];
    w[3][k] = y[2 * a.n];
    if constexpr (SOFT) {
      if (soft_ll) w[0][k] = soft_keep(w[0][k], tl);
      w[1][k] = soft_keep(w[1][k], t0);
      w[2][k] = soft_keep(w[2][k], t1);
      w[3][k] = soft_keep(w[3][k], t2);
    }
  };
#pragma unroll
  for (int j = 0; j < LH - 1; ++j) load(j);
#pragma unroll
  for (int s = 0; s < K / 4; ++s) {
#pragma unroll
    for (int q = 0; q < 4; ++q) load(LH - 1 + q);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float u = 0.f, v = 0.f;
#pragma unroll
      for (int t = 0; t < LH; ++t) {
        const int k = LH - 1 + q - t;
        u = fmaf(f.f0[t], w[0][k], u);
        u = fmaf(f.f1[t], w[1][k], u);
        v = fmaf(f.f0[t], w[2][k], v);
        v = fmaf(f.f1[t], w[3][k], v);
      }
      lu[s & 1][q][i] = u;
      lv[s & 1][q][i] = v;
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int j = 0; j < LH - 1; ++j) w[b][j] = w[b][j + 4];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = r0 + 4 * s + q;
      float x = 0.f;
#pragma unroll
      for (int t = 0; t < LH; ++t) {
        x = fmaf(f.f0[t], lu[s & 1][q][at[t]], x);
        x = fmaf(f.f1[t], lv[s & 1][q][at[t]], x);
      }
      if (put && r < a.M) out[(size_t)(r * a.sf + ph) * a.n] = x;
    }
  }
}

// Backward of a soft-thresholded level: the analysis of two images at once, b (the
// forward's input, for the masks) and g (the output gradient, taps f2 = f/2):
//   bands of g * 1[|bands of b| > t] to yh, gth += sum -sign(b) 1[|b| > t] g,
// and the low bands of both on (of g masked at the last level).  The bands of b are
// never stored; separate passes wrote both stacks and read them back for the mask
// (8 x 512^2, 3 levels, 4 taps: 164 us of kernels against 68).
template <int LH, int K>
__global__ void __launch_bounds__(RT) k_rdwt_level_mask(RdwtLevel a, RdwtTaps<LH> f, RdwtTaps<LH> f2) {
  __shared__ float lb[2][4][2][RT], lg[2][4][2][RT];
  __shared__ float part[4][RT / 64];
  const int i = threadIdx.x, ph = blockIdx.y % a.sf, r0 = (blockIdx.y / a.sf) * K;
  const int c = (blockIdx.x * a.W + i) % a.n;
  const bool put = i < a.W && (int)blockIdx.x * a.W + i < a.n;
  int at[LH];
#pragma unroll
  for (int j = 0; j < LH; ++j) at[j] = a.halo ? min(i + j * a.sf, RT - 1) : (i + j * a.sf) % a.n;
  const float* ib = a.in + (size_t)blockIdx.z * a.is + c;
  const float* ig = a.in2 + (size_t)blockIdx.z * a.is + c;
  // the last level's low band of b is not needed by anyone
  float* ob = a.out ? a.out + (size_t)blockIdx.z * a.is + c : nullptr;
  float* og = a.out2 + (size_t)blockIdx.z * a.is + c;
  float* yh = a.yh + (size_t)blockIdx.z * a.ys + c;
  const bool last = a.th_ll != nullptr;
  const float t[4] = {last ? a.th_ll[0] : 0.f, a.th[0], a.th[1], a.th[2]};
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  PhaseRow row(r0, a, ph);
  float wb[LH + 3], wg[LH + 3];
#pragma unroll
  for (int j = 0; j < LH - 1; ++j) {
    const size_t o = (size_t)row.next() * a.n;
    wb[j] = ib[o];
    wg[j] = ig[o];
  }
#pragma unroll
  for (int s = 0; s < K / 4; ++s) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const size_t o = (size_t)row.next() * a.n;
      wb[LH - 1 + q] = ib[o];
      wg[LH - 1 + q] = ig[o];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float ub = 0.f, vb = 0.f, ug = 0.f, vg = 0.f;
#pragma unroll
      for (int j = 0; j < LH; ++j) {
        ub = fmaf(f.f0[j], wb[q + j], ub);
        vb = fmaf(f.f1[j], wb[q + j], vb);
        ug = fmaf(f2.f0[j], wg[q + j], ug);
        vg = fmaf(f2.f1[j], wg[q + j], vg);
      }
      lb[s & 1][q][0][i] = ub;
      lb[s & 1][q][1][i] = vb;
      lg[s & 1][q][0][i] = ug;
      lg[s & 1][q][1][i] = vg;
    }
#pragma unroll
    for (int j = 0; j < LH - 1; ++j) {
      wb[j] = wb[j + 4];
      wg[j] = wg[j + 4];
    }
    __syncthreads();  // the two buffers alternate: one barrier per step
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = r0 + 4 * s + q;
      float b[4] = {0.f, 0.f, 0.f, 0.f}, g[4] = {0.f, 0.f, 0.f, 0.f};  // ll, lh, hl, hh
#pragma unroll
      for (int j = 0; j < LH; ++j) {
        const float ub = lb[s & 1][q][0][at[j]], vb = lb[s & 1][q][1][at[j]];
        const float ug = lg[s & 1][q][0][at[j]], vg = lg[s & 1][q][1][at[j]];
        b[0] = fmaf(f.f0[j], ub, b[0]);
        b[1] = fmaf(f.f0[j], vb, b[1]);
        b[2] = fmaf(f.f1[j], ub, b[2]);
        b[3] = fmaf(f.f1[j], vb, b[3]);
        g[0] = fmaf(f2.f0[j], ug, g[0]);
        g[1] = fmaf(f2.f0[j], vg, g[1]);
        g[2] = fmaf(f2.f1[j], ug, g[2]);
        g[3] = fmaf(f2.f1[j], vg, g[3]);
      }
      if (put && r < a.M) {
        const size_t gr = (size_t)(r * a.sf + ph);
        if (ob) ob[gr * a.n] = b[0];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (k == 0 && !last) continue;
          const bool keep = fabsf(b[k]) > t[k];
          acc[k] += keep ? (b[k] > 0.f ? -g[k] : g[k]) : 0.f;
          g[k] = keep ? g[k] : 0.f;
        }
        og[gr * a.n] = g[0];
        float* y = yh + gr * a.ldh;
        y[0] = g[1];
        y[a.n] = g[2];
        y[2 * a.n] = g[3];
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    for (int o = 32; o > 0; o >>= 1) acc[k] += __shfl_xor(acc[k], o);
    if ((i & 63) == 0) part[k][i >> 6] = acc[k];
  }
  __syncthreads();
  if (i < 4 && (i > 0 || last)) {
    float s = 0.f;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += part[i][w];
    if (s != 0.f) atomicAdd(i ? a.gth + (i - 1) : a.gth_ll, s);
  }
}

// Whether every level of a transform has a fused form: filters whose windows
// fit the registers, and rows that fit a block or halos of at most half of it
// (past that more than half of the block's columns would only feed taps).
bool rdwt_fused(int n, int L, int lh) {
  return lh <= 8 && lh % 2 == 0 && (n <= RT || (lh - 1) * (1 << (L - 1)) <= RT / 2);
}

// Columns and rows per block.  A row of at most RT columns goes to one block
// whole (it wraps inside LDS, no column is read twice); longer rows split
// evenly.  Strips of 16 rows re-read LH - 1 rows per 16; where that leaves
// fewer than 1024 blocks (4 per CU), shorter strips.
static int level_shape(RdwtLevel& a, int lh, int nimg, dim3& grid, dim3& blk) {
  a.halo = a.n <= RT ? 0 : (lh - 1) * a.sf;
  const int nb = a.n <= RT ? 1 : (a.n + RT - a.halo - 1) / (RT - a.halo);
  a.W = (a.n + nb - 1) / nb;
  int K = 16;
  while (K > 4 && (long long)nb * ((a.M + K - 1) / K) * a.sf * nimg < 1024) K /= 2;
  grid = dim3(nb, ((a.M + K - 1) / K) * a.sf, nimg);
  blk = dim3((a.W + a.halo + 63) / 64 * 64);
  return K;
}

enum LevelForm { LEVEL_AN, LEVEL_SYN, LEVEL_SYN_SOFT, LEVEL_MASK };

template <int LH, LevelForm FORM>
static hipError_t launch_level(RdwtLevel a, const RdwtFilt& f, int nimg, hipStream_t s) {
  RdwtTaps<LH> t;
  for (int j = 0; j < LH; ++j) t.f0[j] = f.f0[j], t.f1[j] = f.f1[j];
  dim3 grid, blk;
  const int K = level_shape(a, LH, nimg, grid, blk);
  const auto go = [&](auto k) {
    if constexpr (FORM == LEVEL_AN) {
      hipLaunchKernelGGL((k_rdwt_level_an<LH, k.value>), grid, blk, 0, s, a, t);
    } else if constexpr (FORM == LEVEL_MASK) {
      RdwtTaps<LH> t2;  // the transpose of the synthesis: analysis with half the taps
      for (int j = 0; j < LH; ++j) t2.f0[j] = 0.5f * f.f0[j], t2.f1[j] = 0.5f * f.f1[j];
      hipLaunchKernelGGL((k_rdwt_level_mask<LH, k.value>), grid, blk, 0, s, a, t, t2);
    } else {
      hipLaunchKernelGGL((k_rdwt_level_syn<LH, k.value, FORM == LEVEL_SYN_SOFT>), grid, blk, 0, s, a, t);
    }
  };
  if (K == 16)
    go(std::integral_constant<int, 16>{});
  else if (K == 8)
    go(std::integral_constant<int, 8>{});
  else
    go(std::integral_constant<int, 4>{});
  return hipGetLastError();
}

template <LevelForm FORM>
static hipError_t launch_level(const RdwtLevel& a, const RdwtFilt& f, int nimg, hipStream_t s) {
  switch (f.lh) {
    case 2: return launch_level<2, FORM>(a, f, nimg, s);
    case 4: return launch_level<4, FORM>(a, f, nimg, s);
    case 6: return launch_level<6, FORM>(a, f, nimg, s);
    default: return launch_level<8, FORM>(a, f, nimg, s);
  }
}

hipError_t rdwt_analysis(const float* x, float* yl, float* yh, float* tmp, int m, int n, int L, const RdwtFilt& f,
                         int nimg, hipStream_t s) {
  const long long is = (long long)m * n, ys = (long long)m * 3 * n * L, ts = 2LL * m * n;
  const dim3 blk(256), grid((n + 255) / 256, m, nimg);
  hipError_t e = hipSuccess;
  if (rdwt_fused(n, L, f.lh)) {
    // a level cannot run in place: the low bands alternate between tmp's halves
    float* t[2] = {tmp, tmp + is * nimg};
    const float* in = x;
    if (yl == x && L == 1) {
      if ((e = hipMemcpyAsync(t[1], x, sizeof(float) * is * nimg, hipMemcpyDeviceToDevice, s)) != hipSuccess) return e;
      in = t[1];
    }
    for (int lev = 1; lev <= L; ++lev) {
      float* out = lev == L ? yl : t[lev & 1];
      const int sf = 1 << (lev - 1);
      const RdwtLevel a{in, out, yh + 3LL * n * (lev - 1), m, n, sf, m / sf, 0, 0, 3LL * n * L, is, ys};
      if ((e = launch_level<LEVEL_AN>(a, f, nimg, s)) != hipSuccess) return e;
      in = out;
    }
    return hipSuccess;
  }
  if (yl != x && (e = hipMemcpyAsync(yl, x, sizeof(float) * is * nimg, hipMemcpyDeviceToDevice, s)) != hipSuccess)
    return e;
  int sf = 1;
  for (int lev = 1; lev <= L; ++lev, sf *= 2) {
    hipLaunchKernelGGL(k_rdwt_rows_an, grid, blk, 0, s, yl, tmp, tmp + is, m, n, sf, f, is, ts);
    hipLaunchKernelGGL(k_rdwt_cols_an, grid, blk, 0, s, tmp, tmp + is, yl, yh, m, n, sf, L, lev, f, is, ys, ts);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t rdwt_synthesis(const float* yl, const float* yh, float* x, float* tmp, int m, int n, int L,
                          const RdwtFilt& f, int nimg, hipStream_t s, const float* th) {
  const long long is = (long long)m * n, ys = (long long)m * 3 * n * L, ts = 2LL * m * n;
  const dim3 blk(256), grid((n + 255) / 256, m, nimg);
  hipError_t e = hipSuccess;
  if (rdwt_fused(n, L, f.lh)) {
    float* t[2] = {tmp, tmp + is * nimg};
    const float* in = yl;
    if (yl == x && L == 1) {
      if ((e = hipMemcpyAsync(t[1], yl, sizeof(float) * is * nimg, hipMemcpyDeviceToDevice, s)) != hipSuccess) return e;
      in = t[1];
    }
    for (int lev = L; lev >= 1; --lev) {
      float* out = lev == 1 ? x : t[lev & 1];
      const int sf = 1 << (lev - 1);
      RdwtLevel a{in, out, const_cast<float*>(yh) + 3LL * n * (lev - 1), m, n, sf, m / sf, 0, 0, 3LL * n * L, is, ys};
      if (th) {
        a.th = th + 1 + 3 * (lev - 1);
        a.th_ll = lev == L ? th : nullptr;
        e = launch_level<LEVEL_SYN_SOFT>(a, f, nimg, s);
      } else {
        e = launch_level<LEVEL_SYN>(a, f, nimg, s);
      }
      if (e != hipSuccess) return e;
      in = out;
    }
    return hipSuccess;
  }
  if (th) return hipErrorInvalidValue;
  if (x != yl && (e = hipMemcpyAsync(x, yl, sizeof(float) * is * nimg, hipMemcpyDeviceToDevice, s)) != hipSuccess)
    return e;
  int sf = 1 << (L - 1);
  for (int lev = L; lev >= 1; --lev, sf /= 2) {
    hipLaunchKernelGGL(k_rdwt_cols_syn, grid, blk, 0, s, x, yh, tmp, tmp + is, m, n, sf, L, lev, f, is, ys, ts);
    hipLaunchKernelGGL(k_rdwt_rows_syn, grid, blk, 0, s, tmp, tmp + is, x, m, n, sf, f, is, ts);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t rdwt_shrink_mask(const float* b, const float* g, float* gyl, float* gyh, float* tmp, int m, int n, int L,
                            const RdwtFilt& f, const float* th, float* gth, int nimg, hipStream_t s) {
  if (!rdwt_fused(n, L, f.lh)) return hipErrorInvalidValue;
  const long long is = (long long)m * n, ys = (long long)m * 3 * n * L;
  float* t[4] = {tmp, tmp + is * nimg, tmp + 2 * is * nimg, tmp + 3 * is * nimg};
  for (int lev = 1; lev <= L; ++lev) {
    const bool last = lev == L;
    const int sf = 1 << (lev - 1);
    float *ob = last ? nullptr : t[lev & 1], *og = last ? gyl : t[2 + (lev & 1)];
    RdwtLevel a{b, ob, gyh + 3LL * n * (lev - 1), m, n, sf, m / sf, 0, 0, 3LL * n * L, is, ys};
    a.in2 = g;
    a.out2 = og;
    a.th = th + 1 + 3 * (lev - 1);
    a.gth = gth + 1 + 3 * (lev - 1);
    a.th_ll = last ? th : nullptr;
    a.gth_ll = gth;
    const hipError_t e = launch_level<LEVEL_MASK>(a, f, nimg, s);
    if (e != hipSuccess) return e;
    b = ob;
    g = og;
  }
  return hipSuccess;
}

}  // namespace shx
