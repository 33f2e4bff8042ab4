// Median absolute deviation of every plane of a stack, on the device.
//
// The noise scalars of the denoise (shearlet_toolbox_1/nsst_scalars.m:28-45,
// demo_denoise/shearcuda/shearcuda.cpp:205-271) are MAD/0.6745 of each band of
// the transform of unit white noise.  The reference copies every band to the
// host and takes two medians there; here the order statistics are found by radix
// selection over monotone integer keys of the values (one workgroup per plane, or
// histograms split over many where a workspace is given and planes are large), so
// the result is the exact median of the data, as a sort gives it.
//
// Two arithmetic conventions, each reproducing one caller bit for bit:
//   SHX_MAD_FP64  values widened to double: m = (a + b) / 2 of the two middle
//                 values (even count), deviations |v - m| in double, their
//                 median the same way, / 0.6745 (MATLAB's median on the double
//                 transform of nsst_scalars.m:36-44; numpy's median).
//   SHX_MAD_FP32  float arithmetic as in the demo: m = (a + b) / 2 in float,
//                 |v - m| in float, median in float, then / .6745 in double
//                 (shearcuda.cpp:165-181, 246-252).
// Inputs must be finite.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "api_err.h"

namespace shx {
namespace {

constexpr int MT = 1024;                // threads per plane
constexpr int MBITS = 11;               // key bits resolved per histogram pass
constexpr int MBINS = 1 << MBITS;       // == 2 * MT: two bins per thread in the scan
static_assert(MBINS == 2 * MT, "scan assumes two bins per thread");

// Order-preserving key of a float: negative values flipped, sign bit set on
// the others, so that unsigned comparison of keys orders the values.
__device__ __forceinline__ uint32_t f32_key(float v) {
  const uint32_t b = __float_as_uint(v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float f32_unkey(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Keys of the three selections.  Deviations are non-negative, so their bit
// patterns already order them.
struct KeyValue {
  static constexpr int W = 32;
  __device__ uint64_t operator()(float v) const { return f32_key(v); }
};
struct KeyDev64 {
  static constexpr int W = 64;
  double m;
  __device__ uint64_t operator()(float v) const { return (uint64_t)__double_as_longlong(fabs((double)v - m)); }
};
struct KeyDev32 {
  static constexpr int W = 32;
  float m;
  __device__ uint64_t operator()(float v) const { return __float_as_uint(fabsf(v - m)); }
};

// Calls fn(v) for every element of p[0, n) over the block's NT threads.
// U: float4 loads in flight (fn's LDS atomics keep the compiler from moving the next
// load above them); one for planes of a few thousand elements, which have no more
// (16384 planes of 1024: 472 us, four 499; 49 planes of 1024^2, four 702 us, one 962).
template <bool VEC, int NT, int U, class F>
__device__ __forceinline__ void each_value(const float* __restrict__ p, int n, F&& fn) {
  if constexpr (VEC) {
    const float4* p4 = reinterpret_cast<const float4*>(p);
    const int n4 = n >> 2;
    int i = threadIdx.x;
    if constexpr (U > 1) {
      for (; i + (U - 1) * NT < n4; i += U * NT) {
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = p4[i + u * NT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          fn(v[u].x);
          fn(v[u].y);
          fn(v[u].z);
          fn(v[u].w);
        }
      }
    }
    for (; i < n4; i += NT) {
      const float4 v = p4[i];
      fn(v.x);
      fn(v.y);
      fn(v.z);
      fn(v.w);
    }
    const int rest = n & 3;
    if ((int)threadIdx.x < rest) fn(p[n - rest + threadIdx.x]);
  } else {
    // unsigned: the step past the end of a plane of 2^31 - 1 elements exceeds an int
    for (uint32_t i = threadIdx.x; i < (uint32_t)n; i += NT) fn(p[i]);
  }
}

struct SelShared {
  uint32_t hist[MBINS];
  uint32_t wsum[MT / 64];
  uint32_t res[3];
  uint64_t wmin[MT / 64], wmax[MT / 64];
};

// Rank search in a histogram held by `sh`, two bins per thread: the bin that
// holds rank krem, the elements before it and in it go to sh.res.
__device__ __forceinline__ void find_bin(SelShared& sh, uint32_t krem) {
  const int t = threadIdx.x;
  const uint32_t h0 = sh.hist[2 * t], h1 = sh.hist[2 * t + 1], s = h0 + h1;
  uint32_t inc = s;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(inc, o, 64);
    if ((t & 63) >= o) inc += y;
  }
  if ((t & 63) == 63) sh.wsum[t >> 6] = inc;
  __syncthreads();
  uint32_t before = inc - s;
  for (int w = 0; w < (t >> 6); ++w) before += sh.wsum[w];
  if (krem >= before && krem < before + h0) {
    sh.res[0] = 2 * t;
    sh.res[1] = before;
    sh.res[2] = h0;
  } else if (krem >= before + h0 && krem < before + s) {
    sh.res[0] = 2 * t + 1;
    sh.res[1] = before + h0;
    sh.res[2] = h1;
  }
  __syncthreads();
}

__device__ __forceinline__ uint64_t shfl_xor64(uint64_t v, int o) {
  const uint32_t lo = __shfl_xor((uint32_t)v, o, 64), hi = __shfl_xor((uint32_t)(v >> 32), o, 64);
  return ((uint64_t)hi << 32) | lo;
}

// Smallest and largest of the block's values.
__device__ __forceinline__ void block_minmax(uint64_t& mn, uint64_t& mx, SelShared& sh) {
  const int t = threadIdx.x;
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t a = shfl_xor64(mn, o), b = shfl_xor64(mx, o);
    mn = a < mn ? a : mn;
    mx = b > mx ? b : mx;
  }
  if ((t & 63) == 0) sh.wmin[t >> 6] = mn, sh.wmax[t >> 6] = mx;
  __syncthreads();
  mn = sh.wmin[0], mx = sh.wmax[0];
  for (int w = 1; w < MT / 64; ++w) {
    mn = sh.wmin[w] < mn ? sh.wmin[w] : mn;
    mx = sh.wmax[w] > mx ? sh.wmax[w] : mx;
  }
  __syncthreads();
}

// Key of the element of rank k (0-based) of p[0, n) under kf, all of whose keys agree
// above their low `top` bits (there: `above`); *after_eq is the number of elements with
// the same key ranked after it.  W: `top` at compile time (whole planes, whose passes
// then unroll with constant masks: 4096 planes of 4096 331 -> 216 us), or 0.
template <bool VEC, int U, int W, class K>
__device__ uint64_t block_select(const float* __restrict__ p, int n, uint32_t k, const K& kf, int top, uint64_t above,
                                 SelShared& sh, uint32_t* after_eq) {
  const int t = threadIdx.x;
  if constexpr (W > 0) top = W, above = 0;
  uint64_t prefix = above, pmask = W > 0 || top == 64 ? 0 : ~0ull << top;
  uint32_t krem = k, cnt = (uint32_t)n;
  for (int left = top; left > 0;) {
    const int d = left < MBITS ? left : MBITS;
    const int shift = left - d;
    const uint32_t dmask = (1u << d) - 1u;
    sh.hist[2 * t] = 0;
    sh.hist[2 * t + 1] = 0;
    __syncthreads();
    each_value<VEC, MT, U>(p, n, [&](float v) {
      const uint64_t key = kf(v);
      if ((key & pmask) == prefix) atomicAdd(&sh.hist[(uint32_t)(key >> shift) & dmask], 1u);
    });
    __syncthreads();
    find_bin(sh, krem);
    krem -= sh.res[1];
    cnt = sh.res[2];
    prefix |= (uint64_t)sh.res[0] << shift;
    pmask |= (uint64_t)dmask << shift;
    left = shift;
    __syncthreads();  // hist and res are rewritten by the next pass
  }
  *after_eq = cnt - krem - 1;
  return prefix;
}

// Smallest key of p[0, n) past lo, at most `above`.
template <bool VEC, int U, class K>
__device__ uint64_t block_min_past(const float* __restrict__ p, int n, uint64_t lo, uint64_t above, const K& kf,
                                   SelShared& sh) {
  uint64_t mn = above;
  each_value<VEC, MT, U>(p, n, [&](float v) {
    const uint64_t key = kf(v);
    if (key > lo && key < mn) mn = key;
  });
  uint64_t none = 0;
  block_minmax(mn, none, sh);
  return mn;
}

// The two middle keys of a whole plane (equal for an odd count), keys of W bits.
template <bool VEC, int U, int W, class K>
__device__ void block_middle(const float* __restrict__ p, int n, const K& kf, SelShared& sh, uint64_t* lo,
                             uint64_t* hi) {
  uint32_t after = 0;
  *lo = *hi = block_select<VEC, U, W>(p, n, (uint32_t)((n - 1) / 2), kf, W, 0, sh, &after);
  if (!(n & 1) && after == 0) *hi = block_min_past<VEC, U>(p, n, *lo, ~0ull, kf, sh);
}

// Median of the values from its two middle keys.
template <bool FP32>
__device__ __forceinline__ double value_median(uint64_t a, uint64_t b, int n) {
  const float fa = f32_unkey((uint32_t)a), fb = f32_unkey((uint32_t)b);
  if constexpr (FP32) return (n & 1) ? fa : (fa + fb) / 2.0f;
  return (n & 1) ? (double)fa : ((double)fa + (double)fb) / 2.0;
}
// MAD / 0.6745 from the two middle deviation keys.
template <bool FP32>
__device__ __forceinline__ double dev_mad(uint64_t a, uint64_t b, int n) {
  if constexpr (FP32) {
    const float da = __uint_as_float((uint32_t)a), db = __uint_as_float((uint32_t)b);
    const float md = (n & 1) ? da : (da + db) / 2.0f;
    return (double)md / 0.6745;
  }
  const double da = __longlong_as_double((long long)a), db = __longlong_as_double((long long)b);
  const double md = (n & 1) ? da : (da + db) / 2.0;
  return md / 0.6745;
}
template <bool FP32>
__device__ __forceinline__ auto dev_key(double m) {
  if constexpr (FP32)
    return KeyDev32{(float)m};
  else
    return KeyDev64{m};
}

// One block per plane, which reads it once per pass: planes of at most MCAP elements
// (their passes come from the caches, two blocks to a CU: 4096 planes of 4096 216 us;
// a copy in LDS fills a CU with one block: 404), and planes of any size where the
// caller has no workspace.
constexpr int MCAP = 32768;  // values kept in LDS by a selecting block (128 KiB of the CU's 160)

template <bool VEC, bool FP32, int U>
__global__ void __launch_bounds__(MT, 8) k_band_mad(const float* __restrict__ planes, long long stride, int n,
                                                 double* __restrict__ mad) {
  __shared__ SelShared sh;
  const float* p = planes + (size_t)blockIdx.x * (size_t)stride;
  uint64_t a, b;
  block_middle<VEC, U, KeyValue::W>(p, n, KeyValue{}, sh, &a, &b);
  const double m = value_median<FP32>(a, b, n);
  const auto dev = dev_key<FP32>(m);
  block_middle<VEC, U, decltype(dev)::W>(p, n, dev, sh, &a, &b);
  if (threadIdx.x == 0) mad[blockIdx.x] = dev_mad<FP32>(a, b, n);
}

// ---- large planes: the passes over the plane split over many blocks -------------
// One block per plane leaves most CUs idle (49 planes on 256 CUs) and reads the
// plane ten times through one CU: 447 us for 49 planes of 512^2, 0.12 TB/s.
// Here each of the two medians takes
//   k_mad_hist    histogram of the keys' top 12 bits, per block
//   k_mad_find    one block per plane: the bin of the middle rank
//   k_mad_hist    the next 11 bits inside that bin; returns at once for a plane
//                 whose bin already fits the candidate buffer.  A bin is an eighth
//                 of an octave and holds 3 to 5% of a Gaussian plane at the median
//                 of its deviations: planes of up to 512^2 fit, 1024^2 planes and
//                 128^3 bands mostly do not.
//   k_mad_find    the bin among those 11 bits (where find2_in_gather is false; else
//                 every block of the gather finds it itself)
//   k_mad_gather  values of the bin to the candidate buffer, and the smallest
//                 key above the bin
//   k_mad_select  one block per plane: exact selection among the candidates,
//                 in LDS
// so the plane is read two or three times per median, by all CUs: 92 us for the same
// planes, bound by the latency of ten short dependent launches (the four
// streaming ones read 51 MB in 11-15 us each).  The 64-bit deviations
// are binned by their float rounding, which keeps their order, and compared
// exactly in the last step.  A plane with more candidates than the buffer
// takes (more than MCAP elements equal in their leading 23 bits) is selected
// from global memory by its one block.
constexpr int HBITS = 12, HBINS = 1 << HBITS;        // first histogram
constexpr int H2BITS = 11, H2BINS = 1 << H2BITS;     // second
constexpr int ST = 512;                              // threads of the streaming kernels
constexpr int SCHUNK = 16384, GCHUNK = 8192;         // elements per block
static_assert(HBINS == 4 * MT && H2BINS == 2 * MT && ST == MT / 2, "bin scans of the streaming kernels");

struct MadState {
  uint32_t prefix, shift;   // bin of the middle rank: the keys with key >> shift == prefix
  uint32_t rank;            // the rank inside the bin
  uint32_t rank2;           // the rank inside the gathered bin
  uint32_t second, ncand;   // the second histogram was needed; candidates
  double m;                 // out: the median of the values
};

// Blocks of a plane's histogram and gather passes (planes of up to 2^31 - 1 elements,
// so the rounding is done in 64 bits).
struct MadBlocks {
  int gh, gg;
  constexpr explicit MadBlocks(long long n)
      : gh((int)((n + SCHUNK - 1) / SCHUNK)), gg((int)((n + GCHUNK - 1) / GCHUNK)) {}
  // workspace bytes of one plane
  constexpr size_t bytes() const {
    return 2 * sizeof(MadState) + sizeof(float) * MCAP + sizeof(uint16_t) * HBINS * (size_t)gh +
           sizeof(uint64_t) * (size_t)gg;
  }
};
static_assert(MadBlocks(0x7fffffff).gh == 131072 && MadBlocks(0x7fffffff).gg == 262144, "the largest plane");

// Planes that go through the passes together; the groups of a stack share one
// workspace (128 KB and an eighth of its bytes a plane), so it takes at most 268 MB and
// an eighth of MAD_GROUP planes, whatever the stack.  Even groups of at most MAD_GROUP:
// 8192 planes of 65536 2461 us in one group, 2499 in four; 1100 planes of 33000 236 us,
// 296 in groups of 512.
constexpr int MAD_GROUP = 2048;
inline int mad_group(int nplanes) {
  const int groups = nplanes / MAD_GROUP + (nplanes % MAD_GROUP > 0);
  return nplanes / groups + (nplanes % groups > 0);
}

struct MadPlanes {
  const float* p;
  long long stride;
  int n;
  MadState* st;    // two per plane: values, deviations
  float* cand;     // MCAP per plane
  uint16_t* part;  // a histogram per block of the histogram pass, gh blocks per plane
  uint64_t* above; // smallest key above the bin, per block of the gather, gg blocks per plane
  int gh, gg;
};

// The 32-bit binning key of a stage, and the exact key its order refines to.
template <int STAGE, bool FP32>
struct MadKey {
  static constexpr int W = STAGE && !FP32 ? 64 : 32;
  double m;
  __device__ uint64_t exact(float v) const {
    if constexpr (STAGE == 0) return KeyValue{}(v);
    return dev_key<FP32>(m)(v);
  }
  __device__ uint32_t bin(float v) const {
    if constexpr (STAGE == 0) return f32_key(v);
    if constexpr (FP32) return __float_as_uint(fabsf(v - (float)m));
    return __float_as_uint((float)fabs((double)v - m));
  }
};

// The bin of `rank` among the plane's bins (NB consecutive ones per thread),
// summed over its blocks' histograms: every thread finds (bin, elements before
// it, elements in it) in res.
template <int NB>
__device__ __forceinline__ void find_bin_parts(const uint16_t* part, int nparts, uint32_t rank, uint32_t* wsum,
                                               uint32_t* res) {
  const int t = threadIdx.x;
  uint32_t h[NB] = {}, s = 0;
  using V = __attribute__((ext_vector_type(NB))) uint16_t;
#pragma unroll 4
  for (int b = 0; b < nparts; ++b) {
    const V v = *reinterpret_cast<const V*>(part + (size_t)b * HBINS + NB * t);
#pragma unroll
    for (int i = 0; i < NB; ++i) h[i] += v[i];
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) s += h[i];
  uint32_t inc = s;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(inc, o, 64);
    if ((t & 63) >= o) inc += y;
  }
  if ((t & 63) == 63) wsum[t >> 6] = inc;
  __syncthreads();
  uint32_t before = inc - s;
  for (int w = 0; w < (t >> 6); ++w) before += wsum[w];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if (rank >= before && rank < before + h[i]) {
      res[0] = NB * t + i;
      res[1] = before;
      res[2] = h[i];
    }
    before += h[i];
  }
  __syncthreads();
}

// The blocks' histograms go to the workspace whole (16-bit counts: a block has
// SCHUNK elements) and one block per plane adds them up (k_mad_find).  Adding
// them with a global atomic per occupied bin, or in the plane's last block to
// finish (whose fence writes the L2 back in every block), took 137 and 160 us
// for 49 planes of 512^2.
template <int STAGE, bool VEC, bool FP32, bool SECOND>
__global__ void __launch_bounds__(ST) k_mad_hist(MadPlanes io) {
  constexpr int NB = SECOND ? H2BINS : HBINS;
  static_assert(SCHUNK < 65536, "16-bit counts");
  __shared__ uint32_t hist[NB];
  const MadState* st = io.st + 2 * blockIdx.y + STAGE;
  if (SECOND && !st->second) return;
  const MadKey<STAGE, FP32> kf{STAGE ? io.st[2 * blockIdx.y].m : 0.0};
  const uint32_t prefix = SECOND ? st->prefix : 0;
  for (int i = threadIdx.x; i < NB; i += ST) hist[i] = 0;
  __syncthreads();
  const int at = blockIdx.x * SCHUNK;
  each_value<VEC, ST, 4>(io.p + (size_t)blockIdx.y * io.stride + at, min(SCHUNK, io.n - at), [&](float v) {
    const uint32_t key = kf.bin(v);
    if constexpr (SECOND) {
      if (key >> (32 - HBITS) == prefix) atomicAdd(&hist[(key >> (32 - HBITS - H2BITS)) & (H2BINS - 1)], 1u);
    } else {
      atomicAdd(&hist[key >> (32 - HBITS)], 1u);
    }
  });
  __syncthreads();
  uint32_t* mine = reinterpret_cast<uint32_t*>(io.part + ((size_t)blockIdx.y * io.gh + blockIdx.x) * HBINS);
  for (int i = threadIdx.x; i < NB / 2; i += ST) mine[i] = hist[2 * i] | (hist[2 * i + 1] << 16);
}

// The bin of the plane's middle rank, and the start values of the gather; SECOND:
// the bin inside that one.
template <int STAGE, bool SECOND>
__global__ void __launch_bounds__(ST) k_mad_find(MadPlanes io) {
  __shared__ uint32_t wsum[ST / 64], res[3];
  MadState* st = io.st + 2 * blockIdx.x + STAGE;
  const uint16_t* part = io.part + (size_t)blockIdx.x * io.gh * HBINS;
  if constexpr (SECOND) {
    if (!st->second) return;
    const uint32_t rank = st->rank;
    find_bin_parts<H2BINS / ST>(part, io.gh, rank, wsum, res);
    if (threadIdx.x == 0) {
      st->prefix = (st->prefix << H2BITS) | res[0];
      st->shift -= H2BITS;
      st->rank = rank - res[1];
    }
  } else {
    const uint32_t rank = (uint32_t)((io.n - 1) / 2);
    find_bin_parts<HBINS / ST>(part, io.gh, rank, wsum, res);
    if (threadIdx.x == 0) {
      st->prefix = res[0];
      st->shift = 32 - HBITS;
      st->rank = rank - res[1];
      st->second = res[2] > (uint32_t)MCAP;
      st->ncand = 0;
    }
  }
}

// FIND2: a block adds up the plane's second histograms itself instead of a launch of
// k_mad_find before the gather.
template <int STAGE, bool VEC, bool FP32, bool FIND2>
__global__ void __launch_bounds__(ST) k_mad_gather(MadPlanes io) {
  __shared__ float buf[GCHUNK];
  __shared__ uint32_t cnt, base;
  __shared__ uint64_t mn[ST / 64];
  MadState* st = io.st + 2 * blockIdx.y + STAGE;
  const MadKey<STAGE, FP32> kf{STAGE ? io.st[2 * blockIdx.y].m : 0.0};
  uint32_t prefix = st->prefix, rank = st->rank, shift = st->shift;
  if constexpr (FIND2) {
    __shared__ uint32_t wsum[ST / 64], res[3];
    if (st->second) {
      find_bin_parts<H2BINS / ST>(io.part + (size_t)blockIdx.y * io.gh * HBINS, io.gh, rank, wsum, res);
      prefix = (prefix << H2BITS) | res[0];
      rank -= res[1];
      shift -= H2BITS;
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) st->rank2 = rank;
  if (threadIdx.x == 0) cnt = 0;
  __syncthreads();
  const int at = blockIdx.x * GCHUNK;
  uint64_t above = ~0ull;
  uint32_t abin = ~0u;  // binning key of `above`: exact keys are made only for values not past it
  each_value<VEC, ST, 4>(io.p + (size_t)blockIdx.y * io.stride + at, min(GCHUNK, io.n - at), [&](float v) {
    const uint32_t bin = kf.bin(v), b = bin >> shift;
    if (b > prefix) {
      if (bin > abin) return;
      const uint64_t key = kf.exact(v);
      abin = bin;
      above = key < above ? key : above;
    } else if (b == prefix) {
      buf[atomicAdd(&cnt, 1u)] = v;
    }
  });
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t a = shfl_xor64(above, o);
    above = a < above ? a : above;
  }
  if ((threadIdx.x & 63) == 0) mn[threadIdx.x >> 6] = above;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < ST / 64; ++w) above = mn[w] < above ? mn[w] : above;
    io.above[(size_t)blockIdx.y * io.gg + blockIdx.x] = above;
  }
  if (threadIdx.x == 0 && cnt) base = atomicAdd(&st->ncand, cnt);
  __syncthreads();
  float* out = io.cand + (size_t)blockIdx.y * MCAP;
  for (uint32_t i = threadIdx.x; i < cnt; i += ST)
    if (base + i < (uint32_t)MCAP) out[base + i] = buf[i];
}

template <int STAGE, bool VEC, bool FP32>
__global__ void __launch_bounds__(MT) k_mad_select(MadPlanes io, double* __restrict__ mad) {
  __shared__ SelShared sh;
  __shared__ float buf[MCAP];
  MadState* st = io.st + 2 * blockIdx.x + STAGE;
  const MadKey<STAGE, FP32> kf{STAGE ? io.st[2 * blockIdx.x].m : 0.0};
  const auto exact = [&](float v) { return kf.exact(v); };
  const uint32_t nc = st->ncand;
  const bool two = !(io.n & 1);
  uint64_t a, b;
  if (nc <= (uint32_t)MCAP) {
    const float* c = io.cand + (size_t)blockIdx.x * MCAP;
    uint64_t mn = ~0ull, mx = 0;
    for (uint32_t i = threadIdx.x; i < nc; i += MT) {
      const float v = c[i];
      const uint64_t key = exact(v);
      buf[i] = v;
      mn = key < mn ? key : mn;
      mx = key > mx ? key : mx;
    }
    block_minmax(mn, mx, sh);
    // the smallest key past the bin, used if the rank is the bin's last
    uint64_t above = ~0ull, none = 0;
    if (two && st->rank2 + 1 == nc) {
      for (int i = threadIdx.x; i < io.gg; i += MT) {
        const uint64_t key = io.above[(size_t)blockIdx.x * io.gg + i];
        above = key < above ? key : above;
      }
      block_minmax(above, none, sh);
    }
    // the candidates' keys lie in [mn, mx]: only the bits in which these differ are open
    const int top = mn == mx ? 0 : 64 - __clzll((long long)(mn ^ mx));
    uint32_t after = 0;
    a = b = block_select<false, 4, 0>(buf, (int)nc, st->rank2, exact, top, top == 64 ? 0 : mn & (~0ull << top), sh, &after);
    if (two && after == 0) b = block_min_past<false, 4>(buf, (int)nc, a, above, exact, sh);
  } else {
    block_middle<VEC, 4, MadKey<STAGE, FP32>::W>(io.p + (size_t)blockIdx.x * io.stride, io.n, exact, sh, &a, &b);
  }
  if (threadIdx.x == 0) {
    if constexpr (STAGE == 0)
      st->m = value_median<FP32>(a, b, io.n);
    else
      mad[blockIdx.x] = dev_mad<FP32>(a, b, io.n);
  }
}

// Whether the gather's blocks each add up the plane's second histograms (gh of 4 KB).
// A launch of k_mad_find instead costs 2-3 us, also where no plane needs the second
// histogram; the sums of all blocks grow with the square of a plane's size.  In the
// gather / by a launch, us: 49 normal planes of 400000 115 / 118, of 800000 180 / 182,
// of 1024^2 (which need it) 280 / 217; one plane of 128^3 91 / 94, four 121 / 109, 192
// 2964 / 1670; 2^27 elements 31.6 / 3.9 ms.  In the gather for planes of up to 50
// histograms (819200 elements, from where normal planes begin to need them) and while
// all sums are at most 128 MB.
bool find2_in_gather(const MadPlanes& io, int nplanes) {
  return io.gh <= 50 || (long long)io.gh * io.gg * nplanes <= 32768;
}

template <int STAGE, bool VEC, bool FP32>
void launch_mad_stage(const MadPlanes& io, int nplanes, double* mad, hipStream_t s) {
  const dim3 gh(io.gh, nplanes), gg(io.gg, nplanes);
  hipLaunchKernelGGL((k_mad_hist<STAGE, VEC, FP32, false>), gh, dim3(ST), 0, s, io);
  hipLaunchKernelGGL((k_mad_find<STAGE, false>), dim3(nplanes), dim3(ST), 0, s, io);
  hipLaunchKernelGGL((k_mad_hist<STAGE, VEC, FP32, true>), gh, dim3(ST), 0, s, io);
  if (find2_in_gather(io, nplanes)) {
    hipLaunchKernelGGL((k_mad_gather<STAGE, VEC, FP32, true>), gg, dim3(ST), 0, s, io);
  } else {
    hipLaunchKernelGGL((k_mad_find<STAGE, true>), dim3(nplanes), dim3(ST), 0, s, io);
    hipLaunchKernelGGL((k_mad_gather<STAGE, VEC, FP32, false>), gg, dim3(ST), 0, s, io);
  }
  hipLaunchKernelGGL((k_mad_select<STAGE, VEC, FP32>), dim3(nplanes), dim3(MT), 0, s, io, mad);
}

// Whether a call with a workspace splits its planes over blocks or gives each to one,
// where many planes fill the chip by themselves.  Split / one block, us, 33000 elements:
//   FP32  1 plane 43 / 33, 49 planes 48 / 34, 512 109 / 69, 2048 366 / 262
//   FP64  1 plane 47 / 57, 49 planes 52 / 58, 512 118 / 111, 1100 235 / 273, 2048
//         399 / 418, 8192 2141 / 2278, 16384 3224 / 3039
// 65536 elements:
//   FP32  49 planes 50 / 53, 128 63 / 54, 384 122 / 115, 512 146 / 146, 1024 269 / 297
//   FP64  128 planes 68 / 98, 2048 624 / 847
// and 131072 elements: FP32 128 planes 86 / 102.  One block per plane for FP32 below
// 49152 elements, and up to 98304 for 65 to 511 planes; for FP64 below 49152 elements
// and more than 4096 planes (there it spares the workspace).
constexpr int SPLIT_N = 49152, SPLIT_PLANES = 4096;
template <bool FP32>
bool split_pays(int n, int nplanes) {
  if (n <= MCAP) return false;
  if (FP32) return n >= 2 * SPLIT_N || (n >= SPLIT_N && (nplanes <= 64 || nplanes >= 512));
  return n >= SPLIT_N || nplanes <= SPLIT_PLANES;
}

// VEC: float4 loads, for planes that all start on 16 bytes.
template <bool VEC, bool FP32>
void launch_mad(const float* planes, long long stride, int n, int nplanes, double* mad, void* work, hipStream_t s) {
  if (n <= MCAP) {
    hipLaunchKernelGGL((k_band_mad<VEC, FP32, 1>), dim3(nplanes), dim3(MT), 0, s, planes, stride, n, mad);
    return;
  }
  if (!work || !split_pays<FP32>(n, nplanes)) {
    hipLaunchKernelGGL((k_band_mad<VEC, FP32, 4>), dim3(nplanes), dim3(MT), 0, s, planes, stride, n, mad);
    return;
  }
  const MadBlocks mb(n);
  const int group = mad_group(nplanes);
  MadState* st = static_cast<MadState*>(work);
  float* cand = reinterpret_cast<float*>(st + 2 * (size_t)group);
  uint16_t* part = reinterpret_cast<uint16_t*>(cand + (size_t)group * MCAP);
  uint64_t* above = reinterpret_cast<uint64_t*>(part + (size_t)group * mb.gh * HBINS);
  for (int p0 = 0; p0 < nplanes; p0 += group) {
    const int k = min(group, nplanes - p0);
    const MadPlanes io{planes + (size_t)p0 * stride, stride, n, st, cand, part, above, mb.gh, mb.gg};
    launch_mad_stage<0, VEC, FP32>(io, k, mad + p0, s);
    launch_mad_stage<1, VEC, FP32>(io, k, mad + p0, s);
  }
}

}  // namespace
}  // namespace shx

extern "C" size_t shx_band_mad_workspace(long long plane_elems, int nplanes) {
  using namespace shx;
  if (plane_elems > 0x7fffffffLL || nplanes < 1) return 0;
  const int n = (int)plane_elems;
  if (!split_pays<false>(n, nplanes) && !split_pays<true>(n, nplanes)) return 0;
  return (size_t)mad_group(nplanes) * MadBlocks(plane_elems).bytes();
}

extern "C" int shx_band_mad_ws(const float* planes, long long plane_elems, long long plane_stride, int nplanes,
                               int arith, double* mad, void* work, size_t work_bytes, void* stream) {
  using namespace shx;
  if (!planes || !mad) return fail(SHX_ERR_ARG, "null pointer");
  if (plane_elems < 1 || plane_elems > 0x7fffffffLL) return fail(SHX_ERR_ARG, "plane size %lld outside [1, 2^31)", plane_elems);
  if (plane_stride < plane_elems) return fail(SHX_ERR_ARG, "plane stride %lld below the plane size %lld", plane_stride, plane_elems);
  if (nplanes < 0) return fail(SHX_ERR_ARG, "negative plane count");
  if (arith != SHX_MAD_FP64 && arith != SHX_MAD_FP32) return fail(SHX_ERR_ARG, "unknown arithmetic %d", arith);
  if (nplanes == 0) return SHX_OK;
  if (work && (work_bytes < shx_band_mad_workspace(plane_elems, nplanes) || (uintptr_t)work % 16))
    return fail(SHX_ERR_ARG, "workspace of %zu bytes (16-byte aligned, at least %zu)", work_bytes,
                shx_band_mad_workspace(plane_elems, nplanes));
  const int n = (int)plane_elems;
  const bool vec = ((uintptr_t)planes % 16 == 0) && (plane_stride % 4 == 0);
  hipStream_t s = (hipStream_t)stream;
  if (arith == SHX_MAD_FP32)
    vec ? launch_mad<true, true>(planes, plane_stride, n, nplanes, mad, work, s)
        : launch_mad<false, true>(planes, plane_stride, n, nplanes, mad, work, s);
  else
    vec ? launch_mad<true, false>(planes, plane_stride, n, nplanes, mad, work, s)
        : launch_mad<false, false>(planes, plane_stride, n, nplanes, mad, work, s);
  SHX_HIP(hipGetLastError());
  return SHX_OK;
}

extern "C" int shx_band_mad(const float* planes, long long plane_elems, long long plane_stride, int nplanes,
                            int arith, double* mad, void* stream) {
  return shx_band_mad_ws(planes, plane_elems, plane_stride, nplanes, arith, mad, nullptr, 0, stream);
}
