// 3D line FFT passes and band-pass mask kernels (gfx950).
//
// Replaces, for the 3D path, the reference's per-band cuFFT 3D plans at
// nextpow2(n + 23) with zeroPad / modulateAndNormalize3D / applyHardThreshold /
// addVector (shearcuda3d/3DShearTrans/src_cuda/ShDecThRec_cuda.cpp:228-325,
// shearcuda/shear_cuda.cu:143-195,2284-2386), and the CPU Fourier-domain
// band-pass of shearcuda3d/3DBP/PrySDdec_onestep.m:56-125 and
// PrySDrec_onestep.m:56-118.
//
// Each line transform of N = R1 * R2 points is the two-pass register FFT of
// fft_reg.h: pass A (global -> registers, DFT R2, twiddles), one LDS
// transpose, pass B (DFT R1 -> global).  Zero padding is applied on load and
// the output window on store, so padded forward transforms and cropped
// inverse transforms cost no extra passes.
#include "fft_reg.h"
#include "spectral3d.h"

namespace shx {

__device__ __forceinline__ bool in_window(int j, int n) { return (unsigned)j < (unsigned)n; }

// ---------------------------------------------------------------------------
// Rows (contiguous axis).  A block holds LPB lines and T = LPB * R2 threads;
// pass A uses LPB * R1 of them.
template <int N>
struct Rows3Cfg {
  static constexpr int R1 = Split<N>::R1, R2 = Split<N>::R2;
  static constexpr int LPB = 256 / R2;
  static constexpr int T = LPB * R2;
  static constexpr int LD = N + 1;
  static constexpr int LDS = LPB * LD;
};

template <int N, int DIR>
__global__ void __launch_bounds__(256) k3_rows(Rows3 io, const float2* __restrict__ tw) {
  using C = Rows3Cfg<N>;
  constexpr int R1 = C::R1, R2 = C::R2;
  __shared__ float2 buf[C::LDS];
  const int tid = threadIdx.x;
  const int line0 = blockIdx.x * C::LPB;
  const float2* in = io.in + (size_t)blockIdx.y * io.in_bs;
  float2* out = io.out + (size_t)blockIdx.y * io.out_bs;
  const int la = tid / R1, n1 = tid % R1;
  if (la < C::LPB && line0 + la < io.nlines) {
    const float2* src = in + (size_t)(line0 + la) * io.in_ld;
    float2 v[R2];
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) {
      const int j = n1 + R1 * n2 - io.o_in;
      v[n2] = in_window(j, io.n_in) ? src[j] : make_float2(0.f, 0.f);
    }
    passA<R1, R2, DIR, 1>(v, n1, tw);
#pragma unroll
    for (int k = 0; k < R2; ++k) buf[la * C::LD + n1 + R1 * k] = v[k];
  }
  __syncthreads();
  const int lb = tid / R2, k2 = tid % R2;
  if (line0 + lb < io.nlines) {
    float2 u[R1];
#pragma unroll
    for (int a = 0; a < R1; ++a) u[a] = buf[lb * C::LD + a + R1 * k2];
    dft<R1, DIR>(u);
    float2* dst = out + (size_t)(line0 + lb) * io.out_ld;
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) {
      const int j = k2 + R2 * k1 - io.o_out;
      if (in_window(j, io.n_out)) dst[j] = u[k1];
    }
  }
}

// Inverse rows of F_g . S for a group of bands; S is loaded once.
template <int N>
__global__ void __launch_bounds__(256) k3_rows_mul(Rows3Mul io, const float2* __restrict__ tw) {
  using C = Rows3Cfg<N>;
  constexpr int R1 = C::R1, R2 = C::R2;
  __shared__ float2 buf[C::LDS];
  const int tid = threadIdx.x;
  const int line0 = blockIdx.x * C::LPB;
  const int la = tid / R1, n1 = tid % R1;
  const bool vA = la < C::LPB && line0 + la < io.nlines;
  const int lb = tid / R2, k2 = tid % R2;
  const bool vB = line0 + lb < io.nlines;
  const size_t lineA = (size_t)(line0 + la) * N;
  float2 sv[R2];
  if (vA) {
    const float2* S = io.S + (size_t)blockIdx.y * io.s_bs + lineA;
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) sv[n2] = cscale(S[n1 + R1 * n2], io.scale);
  }
  float2* outb = io.out + (size_t)blockIdx.y * io.out_bs + (size_t)(line0 + lb) * io.out_ld;
  for (int g = 0; g < io.G; ++g) {
    if (vA) {
      const float2* F = io.F + (size_t)g * io.f_gs + lineA;
      float2 v[R2];
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) v[n2] = cmul(sv[n2], F[n1 + R1 * n2]);
      passA<R1, R2, +1, 1>(v, n1, tw);
#pragma unroll
      for (int k = 0; k < R2; ++k) buf[la * C::LD + n1 + R1 * k] = v[k];
    }
    __syncthreads();
    if (vB) {
      float2 u[R1];
#pragma unroll
      for (int a = 0; a < R1; ++a) u[a] = buf[lb * C::LD + a + R1 * k2];
      dft<R1, +1>(u);
      float2* dst = outb + (size_t)g * io.out_gs;
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) {
        const int j = k2 + R2 * k1 - io.o_out;
        if (in_window(j, io.n_out)) dst[j] = u[k1];
      }
    }
    __syncthreads();
  }
}

// Forward rows of G band inputs times conj(F_g), summed over the group.
template <int N>
__global__ void __launch_bounds__(256) k3_rows_cmac(Rows3Cmac io, const float2* __restrict__ tw) {
  using C = Rows3Cfg<N>;
  constexpr int R1 = C::R1, R2 = C::R2;
  __shared__ float2 buf[C::LDS];
  const int tid = threadIdx.x;
  const int line0 = blockIdx.x * C::LPB;
  const int la = tid / R1, n1 = tid % R1;
  const bool vA = la < C::LPB && line0 + la < io.nlines;
  const int lb = tid / R2, k2 = tid % R2;
  const bool vB = line0 + lb < io.nlines;
  float2 acc[R1];
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) acc[k1] = make_float2(0.f, 0.f);
  const size_t lineB = (size_t)(line0 + lb) * N;
  for (int g = 0; g < io.G; ++g) {
    if (vA) {
      const float2* src = io.in + (size_t)blockIdx.y * io.in_bs + (size_t)g * io.in_gs + (size_t)(line0 + la) * io.in_ld;
      float2 v[R2];
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) {
        const int j = n1 + R1 * n2 - io.o_in;
        v[n2] = in_window(j, io.n_in) ? src[j] : make_float2(0.f, 0.f);
      }
      passA<R1, R2, -1, 1>(v, n1, tw);
#pragma unroll
      for (int k = 0; k < R2; ++k) buf[la * C::LD + n1 + R1 * k] = v[k];
    }
    // band spectrum loads in flight across the barrier and the second pass
    float2 f[R1];
    const float2* F = io.F + (size_t)g * io.f_gs + lineB;
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) f[k1] = vB ? F[k2 + R2 * k1] : make_float2(0.f, 0.f);
    __syncthreads();
    if (vB) {
      float2 u[R1];
#pragma unroll
      for (int a = 0; a < R1; ++a) u[a] = buf[lb * C::LD + a + R1 * k2];
      dft<R1, -1>(u);
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) acc[k1] = cadd(acc[k1], cmulc(u[k1], f[k1]));
    }
    __syncthreads();
  }
  if (vB) {
    float2* dst = io.out + (size_t)blockIdx.y * io.out_bs + lineB;
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) acc[k1] = cscale(acc[k1], io.scale);
    if (io.accumulate) {  // every old value loaded before the first store
      float2 old[R1];
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) old[k1] = dst[k2 + R2 * k1];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) acc[k1] = cadd(old[k1], acc[k1]);
    }
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) dst[k2 + R2 * k1] = acc[k1];
  }
}

// ---------------------------------------------------------------------------
// Fused plane inverse: rows then cols of one k0 plane for a chunk of CW
// output columns, through an LDS tile of N rows x CW columns.  Blocks are
// ordered volume-fastest, then band, chunk, plane, so the blocks that share an
// S plane or an F plane run together, and each XCD (the low 3 bits of the
// dispatch order) takes a contiguous range of that order, so the sharing
// stays in one L2.
template <int N>
struct Plane3Cfg {
  static constexpr int R1 = Split<N>::R1, R2 = Split<N>::R2;
  static constexpr int T = N >= 80 ? 512 : 256;
  static constexpr int RC = T / R2;  // rows per row pass
  static constexpr int CC = T / R2;  // columns per column pass
};

template <int N, int CW>
__global__ void __launch_bounds__(Plane3Cfg<N>::T) k3_plane_inv(Plane3Inv io, int nchunk, int nblk, int nvol,
                                                                const float2* __restrict__ tw) {
  using C = Plane3Cfg<N>;
  constexpr int R1 = C::R1, R2 = C::R2, RC = C::RC, CC = C::CC, T = C::T;
  constexpr int CWP = CW + 1;
  constexpr int SCR = (RC * (N + 1) > N * CC) ? RC * (N + 1) : N * CC;
  __shared__ float2 tile[N * CWP];
  __shared__ float2 scr[SCR];
  // XCD-aware block order
  const int pid = blockIdx.x;
  const int per = nblk / 8;
  const int lid = (nblk % 8 == 0) ? (pid % 8) * per + pid / 8 : pid;
  int t = lid;
  const int v = t % nvol;
  t /= nvol;
  const int g = t % io.G;
  t /= io.G;
  const int ch = t % nchunk;
  const int k0 = t / nchunk;
  const int tid = threadIdx.x;
  const int col0 = ch * CW;
  const float2* Sp = io.S + (size_t)v * io.s_bs + (size_t)k0 * N * N;
  const float2* Fp = io.F + (size_t)g * io.f_gs + (size_t)k0 * N * N;
  // rows: inverse along axis 2, keep columns [o_out + col0, o_out + col0 + CW)
  for (int r0 = 0; r0 < N; r0 += RC) {
    const int ra = tid / R1, n1 = tid % R1;
    if (ra < RC && r0 + ra < N) {
      const float2* srow = Sp + (size_t)(r0 + ra) * N;
      const float2* frow = Fp + (size_t)(r0 + ra) * N;
      float2 vv[R2];
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) vv[n2] = cscale(cmul(srow[n1 + R1 * n2], frow[n1 + R1 * n2]), io.scale);
      passA<R1, R2, +1, 1>(vv, n1, tw);
#pragma unroll
      for (int k = 0; k < R2; ++k) scr[ra * (N + 1) + n1 + R1 * k] = vv[k];
    }
    __syncthreads();
    const int rb = tid / R2, k2 = tid % R2;
    if (r0 + rb < N) {
      float2 u[R1];
#pragma unroll
      for (int a = 0; a < R1; ++a) u[a] = scr[rb * (N + 1) + a + R1 * k2];
      dft<R1, +1>(u);
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) {
        const int j = k2 + R2 * k1 - io.o_out - col0;
        if (j >= 0 && j < CW) tile[(r0 + rb) * CWP + j] = u[k1];
      }
    }
    __syncthreads();
  }
  // cols: inverse along axis 1, keep rows [o_out, o_out + n_out)
  const int n = io.n_out;
  float2* op = io.out + (size_t)v * io.out_bs + (size_t)g * io.out_gs + (size_t)k0 * n * n + col0;
  for (int c0 = 0; c0 < CW; c0 += CC) {
    const int c = tid % CC, n1 = tid / CC;
    if (n1 < R1 && c0 + c < CW) {
      float2 vv[R2];
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) vv[n2] = tile[(n1 + R1 * n2) * CWP + c0 + c];
      passA<R1, R2, +1, 1>(vv, n1, tw);
#pragma unroll
      for (int k = 0; k < R2; ++k) scr[(n1 + R1 * k) * CC + c] = vv[k];
    }
    __syncthreads();
    const int k2 = tid / CC;
    if (c0 + c < CW && col0 + c0 + c < n) {
      float2 u[R1];
#pragma unroll
      for (int a = 0; a < R1; ++a) u[a] = scr[(a + R1 * k2) * CC + c];
      dft<R1, +1>(u);
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) {
        const int i1 = k2 + R2 * k1 - io.o_out;
        if (in_window(i1, n)) op[(size_t)i1 * n + c0 + c] = u[k1];
      }
    }
    __syncthreads();
  }
  (void)T;
}

// ---------------------------------------------------------------------------
// Cols (axis 1): a tile of CT adjacent columns, T = CT * R2 threads; element
// (m, c) of the tile at LDS slot m * CT + c.
template <int N, int CT>
struct Cols3Cfg {
  static constexpr int R1 = Split<N>::R1, R2 = Split<N>::R2;
  static constexpr int T = CT * R2;
  static constexpr int LDS = N * CT;
};

template <int N, int CT, int DIR>
__global__ void __launch_bounds__(CT * Split<N>::R2) k3_cols(Cols3 io, const float2* __restrict__ tw) {
  using C = Cols3Cfg<N, CT>;
  constexpr int R1 = C::R1, R2 = C::R2;
  __shared__ float2 buf[C::LDS];
  const int tid = threadIdx.x;
  const int c = tid % CT, n1 = tid / CT;
  const int c0 = blockIdx.x * CT;
  const size_t W = io.W;
  if (n1 < R1) {
    const float2* src = io.in + (size_t)blockIdx.z * io.in_bs + (size_t)blockIdx.y * io.in_ps + c0 + c;
    float2 v[R2];
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) {
      const int j = n1 + R1 * n2 - io.o_in;
      v[n2] = in_window(j, io.n_in) ? src[(size_t)j * W] : make_float2(0.f, 0.f);
    }
    passA<R1, R2, DIR, 1>(v, n1, tw);
#pragma unroll
    for (int k = 0; k < R2; ++k) buf[(n1 + R1 * k) * CT + c] = v[k];
  }
  __syncthreads();
  const int k2 = tid / CT;
  float2 u[R1];
#pragma unroll
  for (int a = 0; a < R1; ++a) u[a] = buf[(a + R1 * k2) * CT + c];
  dft<R1, DIR>(u);
  float2* dst = io.out + (size_t)blockIdx.z * io.out_bs + (size_t)blockIdx.y * io.out_ps + c0 + c;
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) {
    const int j = k2 + R2 * k1 - io.o_out;
    if (in_window(j, io.n_out)) dst[(size_t)j * W] = u[k1];
  }
}

// ---------------------------------------------------------------------------
// Pencils (axis 0): two real columns (2e, 2e+1) form one complex sequence
// z = a + i b; a tile holds CT such pairs.
template <int N, int CT>
__global__ void __launch_bounds__(CT * Split<N>::R2) k3_pencil_fwd(Pencil3Fwd io, const float2* __restrict__ tw) {
  using C = Cols3Cfg<N, CT>;
  constexpr int R1 = C::R1, R2 = C::R2;
  __shared__ float2 buf[C::LDS];
  const int tid = threadIdx.x;
  const int c = tid % CT, n1 = tid / CT;
  const int e = blockIdx.x * CT + c;  // pair index
  const size_t E = io.E;
  if (n1 < R1) {
    const float* src = io.in + (size_t)blockIdx.z * io.in_bs + (size_t)blockIdx.y * io.in_gs + 2 * (size_t)e;
    float2 v[R2];
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) {
      const int j = n1 + R1 * n2 - io.o_in;
      v[n2] = in_window(j, io.n_in) ? *reinterpret_cast<const float2*>(src + (size_t)j * E) : make_float2(0.f, 0.f);
    }
    passA<R1, R2, -1, 1>(v, n1, tw);
#pragma unroll
    for (int k = 0; k < R2; ++k) buf[(n1 + R1 * k) * CT + c] = v[k];
  }
  __syncthreads();
  const int k2 = tid / CT;
  float2 u[R1];
#pragma unroll
  for (int a = 0; a < R1; ++a) u[a] = buf[(a + R1 * k2) * CT + c];
  dft<R1, -1>(u);
  __syncthreads();
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) buf[(k2 + R2 * k1) * CT + c] = u[k1];
  __syncthreads();
  float2* dst = io.out + (size_t)blockIdx.z * io.out_bs + (size_t)blockIdx.y * io.out_gs + 2 * (size_t)e;
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) {
    const int k = k2 + R2 * k1;
    if (k <= N / 2) {
      const float2 z = u[k1];
      const float2 zm = cconj(buf[((N - k) % N) * CT + c]);
      const float2 s = cadd(z, zm), d = csub(z, zm);
      // A = (Z[k] + conj Z[N-k]) / 2, B = (Z[k] - conj Z[N-k]) / (2i)
      *reinterpret_cast<float4*>(dst + (size_t)k * E) = make_float4(0.5f * s.x, 0.5f * s.y, 0.5f * d.y, -0.5f * d.x);
    }
  }
}

template <int N, int CT>
__global__ void __launch_bounds__(CT * Split<N>::R2) k3_pencil_inv(Pencil3Inv io, const float2* __restrict__ tw) {
  using C = Cols3Cfg<N, CT>;
  constexpr int R1 = C::R1, R2 = C::R2;
  __shared__ float2 buf[C::LDS];
  const int tid = threadIdx.x;
  const int c = tid % CT, n1 = tid / CT, k2 = tid / CT;
  const int e = blockIdx.x * CT + c;
  const size_t E = io.E;
  const int b = blockIdx.z;
  // storing form: one band per block
  const int g0 = io.mode == 0 ? blockIdx.y : 0, g1 = io.mode == 0 ? g0 + 1 : io.G;
  float2 acc[R1];
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) acc[k1] = make_float2(0.f, 0.f);
  for (int g = g0; g < g1; ++g) {
    const float t = io.mode == 1 ? io.th[(size_t)b * io.th_bs + io.th0 + g] : 0.0f;
    if (n1 < R1) {
      const float2* src = io.in + (size_t)b * io.in_bs + (size_t)g * io.in_gs + 2 * (size_t)e;
      // data and twiddle loads all in flight before the arithmetic
      PassTw<R2> pt;
      float2 v[R2];
      float4 ab[R2];
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) {
        const int m = n1 + R1 * n2;
        const int km = m <= N / 2 ? m : N - m;
        ab[n2] = *reinterpret_cast<const float4*>(src + (size_t)km * E);
      }
      passA_tw<R2, +1, 1>(pt, n1, tw);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) {
        const int m = n1 + R1 * n2;
        // Z[m] = A[m] + i B[m]; Z[N-m] = conj(A[m]) + i conj(B[m]); the
        // imaginary parts at m = 0 and N/2 are dropped as in a real inverse.
        if (m == 0 || m == N / 2)
          v[n2] = make_float2(ab[n2].x, ab[n2].z);
        else if (m < N / 2)
          v[n2] = make_float2(ab[n2].x - ab[n2].w, ab[n2].y + ab[n2].z);
        else
          v[n2] = make_float2(ab[n2].x + ab[n2].w, ab[n2].z - ab[n2].y);
      }
      passA_apply<R2, +1>(v, pt);
#pragma unroll
      for (int k = 0; k < R2; ++k) buf[(n1 + R1 * k) * CT + c] = v[k];
    }
    __syncthreads();
    float2 u[R1];
#pragma unroll
    for (int a = 0; a < R1; ++a) u[a] = buf[(a + R1 * k2) * CT + c];
    dft<R1, +1>(u);
    if (io.mode == 0) {
      float* dst = io.out + (size_t)b * io.out_bs + (size_t)g * io.out_gs + 2 * (size_t)e;
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) {
        const int j = k2 + R2 * k1 - io.o_out;
        if (in_window(j, io.n_out)) *reinterpret_cast<float2*>(dst + (size_t)j * E) = u[k1];
      }
    } else if (io.mode == 1) {
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1)
        acc[k1] = cadd(acc[k1], make_float2(hard_keep(u[k1].x, t), hard_keep(u[k1].y, t)));
    } else {
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) acc[k1] = cadd(acc[k1], u[k1]);
    }
    __syncthreads();
  }
  if (io.mode != 0) {
    float* dst = io.out + (size_t)b * io.out_bs + 2 * (size_t)e;
    if (!io.first) {  // add to out: every old value loaded before the first store
      float2 old[R1];
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) {
        const int j = k2 + R2 * k1 - io.o_out;
        old[k1] = in_window(j, io.n_out) ? *reinterpret_cast<const float2*>(dst + (size_t)j * E)
                                         : make_float2(0.f, 0.f);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) acc[k1] = cadd(old[k1], acc[k1]);
    }
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) {
      const int j = k2 + R2 * k1 - io.o_out;
      if (in_window(j, io.n_out)) *reinterpret_cast<float2*>(dst + (size_t)j * E) = acc[k1];
    }
  }
}

// ---------------------------------------------------------------------------
// Slab form of the thresholded band loop.  After the inverse rows, the other
// two axes of one output index j2 ("slab") are a half spectrum of (N/2 + 1) x N
// values: 84 KB at N = 144, which fits a CU's LDS.  k3_rows_band writes the
// rows slab by slab, and one block of k3_slab inverse transforms a slab along
// axis 1 and axis 0, thresholds it and keeps the running sum of its bands in
// registers.  Against separate column and pencil passes, one write and one read
// of the band spectra (19 of 41 MB per band and volume at 128^3) stay on the
// chip.  Transforms are N = P * Q two-pass splits with P and Q close, so that
// (nearly) every lane works in both passes and a line's exchange stays inside
// one wave.
// 8 bands of two 128^3 volumes: rows 82 -> 62 us (290 MB: the copy rate), columns
// and pencils 67 + 50 -> 73 us (172 MB; the block's LDS and vector pipes are each
// busy half of the time, one after the other: one block per CU).
// The grid of 128 has no such split here: it belongs to levels of side 80 (or 64 with
// filters of 40 and more), which no dictionary of the workloads has, so its two row
// kernels and the separate passes serve it, as they do the grids of 8 and 16.
template <int N>
struct Split3;
template <> struct Split3<24> { static constexpr int P = 4, Q = 6, NP = 12; };
template <> struct Split3<32> { static constexpr int P = 4, Q = 8, NP = 16; };
template <> struct Split3<48> { static constexpr int P = 6, Q = 8, NP = 24; };
template <> struct Split3<64> { static constexpr int P = 8, Q = 8, NP = 32; };
template <> struct Split3<80> { static constexpr int P = 8, Q = 10, NP = 40; };
// NP: most axis-1 pairs of a slab.  Sides of at most 128 (64 pairs) leave both
// LDS tiles inside the CU.
template <> struct Split3<144> { static constexpr int P = 12, Q = 12, NP = 64; };

template <int N>
struct Slab3Cfg {
  static constexpr int P = Split3<N>::P, Q = Split3<N>::Q, NP = Split3<N>::NP;
  static constexpr int H = N / 2 + 1;
  static constexpr int LPW = 64 / Q;                       // lines per wave
  static constexpr int WL = (H + LPW - 1) / LPW, WP = (NP + LPW - 1) / LPW;
  static constexpr int T = 64 * (WL > WP ? WL : WP);
  // line stride in LDS: 2 LS mod 64 words is an odd multiple of 4, so the
  // 16-byte reads down the lines (phase 2) fall on distinct banks
  static constexpr int LS = N + 2;
  static_assert(T <= 1024 && P <= Q && Q % 2 == 0, "one round per phase");
};

// LDS accesses of one wave stay in order; this keeps the compiler from moving
// them across the exchange.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Place of (n1, k2) in a line's exchange.  The second pass reads it at a stride
// of P over the lanes; where that falls on few banks (multiples of 8 words at
// P = 12, of 16 at P = 8) a slot is skipped after every four k2.
template <int P, int Q>
__device__ __forceinline__ int xch(int n1, int k2) {
  if constexpr (P == 12 || P == 8)
    return n1 + P * k2 + k2 / 4;
  else
    return n1 + P * k2;
}
// First pass of a transform on x[n1 + P n2] (n2 < Q): DFT of length Q,
// twiddles w_N^(n1 k2) (tws[m] = exp(-2 pi i m / N)), to the exchange.
template <int P, int Q, int DIR>
__device__ __forceinline__ void two_first(float2 (&v)[Q], int n1, float2* line, const float2* tws) {
  dft<Q, DIR>(v);
  line[xch<P, Q>(n1, 0)] = v[0];
#pragma unroll
  for (int k = 1; k < Q; ++k)
    line[xch<P, Q>(n1, k)] = DIR > 0 ? cmulc(v[k], tws[n1 * k]) : cmul(v[k], tws[n1 * k]);
}
// Second pass: X[k2 + Q k1], k1 < P.
template <int P, int Q, int DIR>
__device__ __forceinline__ void two_second(float2 (&u)[P], int k2, const float2* line) {
#pragma unroll
  for (int a = 0; a < P; ++a) u[a] = line[xch<P, Q>(a, k2)];
  dft<P, DIR>(u);
}

// Inverse rows of F_g . S, 16 lines per block, bands [z, z + 1) * gper of the
// group.  The next band's F is loaded while this band is transformed.  SLAB:
// outputs leave line-fastest, 128 contiguous bytes per slab; else row by row.
constexpr int SLAB_LINES = 16;
template <int N, bool SLAB>
__global__ void __launch_bounds__(SLAB_LINES * Split3<N>::Q) k3_rows_band(Rows3Mul io, int gper,
                                                                          const float2* __restrict__ tw) {
  constexpr int P = Split3<N>::P, Q = Split3<N>::Q, LS = N + 5, T = SLAB_LINES * Q;
  __shared__ float2 buf[SLAB_LINES * LS];
  __shared__ float2 tws[N];
  const int tid = threadIdx.x;
  for (int i = tid; i < N; i += T) tws[i] = tw[i];
  // volumes fastest: those of one line block read the same F lines, and run on
  // one XCD (the low 3 bits of the dispatch order)
  const int nv = gridDim.y, total = gridDim.x * nv;
  int id = blockIdx.x + gridDim.x * blockIdx.y;
  if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
  const int b = id % nv, line0 = (id / nv) * SLAB_LINES;
  const int g0 = blockIdx.z * gper, g1 = min(io.G, g0 + gper);
  const int la = tid / P, n1 = tid % P;
  const bool vA = la < SLAB_LINES && line0 + la < io.nlines;
  const int lb = SLAB ? tid % SLAB_LINES : tid / Q, k2 = SLAB ? tid / SLAB_LINES : tid % Q;
  const bool vB = line0 + lb < io.nlines;
  float2 sv[Q], f[Q];
  const float2* F = io.F + (size_t)g0 * io.f_gs + (size_t)(line0 + la) * N + n1;
  if (vA) {
    const float2* S = io.S + (size_t)b * io.s_bs + (size_t)(line0 + la) * N + n1;
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) {
      sv[n2] = S[P * n2];
      f[n2] = F[P * n2];
    }
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) sv[n2] = cscale(sv[n2], io.scale);
  }
  float2* out = io.out + (size_t)b * io.out_bs + (SLAB ? (size_t)(line0 + lb) : (size_t)(line0 + lb) * io.out_ld);
  const size_t step = SLAB ? io.nlines : 1;
  __syncthreads();  // tws
  for (int g = g0; g < g1; ++g) {
    if (vA) {
      float2 v[Q];
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) v[n2] = cmul(sv[n2], f[n2]);
      if (g + 1 < g1) {
        F += io.f_gs;
#pragma unroll
        for (int n2 = 0; n2 < Q; ++n2) f[n2] = F[P * n2];
      }
      two_first<P, Q, +1>(v, n1, buf + la * LS, tws);
    }
    __syncthreads();
    if (vB) {
      float2 u[P];
      two_second<P, Q, +1>(u, k2, buf + lb * LS);
      float2* dst = out + (size_t)g * io.out_gs;
#pragma unroll
      for (int k1 = 0; k1 < P; ++k1) {
        const int j = k2 + Q * k1 - io.o_out;
        if (in_window(j, io.n_out)) dst[(size_t)j * step] = u[k1];
      }
    }
    __syncthreads();
  }
}

// Forward rows of G band inputs times conj(F_g), summed over the group, on the
// lane-filling split: CMAC_LINES lines per block, and the group's bands spread
// over CMAC_CH chunks of the block's threads (chunk c takes bands c, c + CMAC_CH,
// ...), whose sums are added through LDS in chunk order.  One chunk per block
// was a chain of 8 transforms in 400 small blocks on the 80^3 grid: 15.6 us per
// group of 8.
constexpr int CMAC_LINES = 8, CMAC_CH = 4;
template <int N>
__global__ void __launch_bounds__(CMAC_CH * CMAC_LINES * Split3<N>::Q) k3_rows_cmac2(Rows3Cmac io,
                                                                                     const float2* __restrict__ tw) {
  constexpr int P = Split3<N>::P, Q = Split3<N>::Q, LS = N + 5, TC = CMAC_LINES * Q, T = CMAC_CH * TC;
  __shared__ float2 buf[CMAC_CH][CMAC_LINES * LS];
  __shared__ float2 tws[N];
  const int tid = threadIdx.x % TC, ch = threadIdx.x / TC;
  for (int i = threadIdx.x; i < N; i += T) tws[i] = tw[i];
  const int line0 = blockIdx.x * CMAC_LINES;
  const int la = tid / P, n1 = tid % P;
  const bool vA = la < CMAC_LINES && line0 + la < io.nlines;
  const int lb = tid / Q, k2 = tid % Q;
  const bool vB = line0 + lb < io.nlines;
  const float2* in = io.in + (size_t)blockIdx.y * io.in_bs + (size_t)(line0 + la) * io.in_ld;
  const float2* Fl = io.F + (size_t)(line0 + lb) * N + k2;
  float2 v[Q], f[P], acc[P];
#pragma unroll
  for (int k = 0; k < P; ++k) acc[k] = make_float2(0.f, 0.f);
  const auto load = [&](int g) {
    if (vA && g < io.G) {
      const float2* src = in + (size_t)g * io.in_gs;
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) {
        const int j = n1 + P * n2 - io.o_in;
        v[n2] = in_window(j, io.n_in) ? src[j] : make_float2(0.f, 0.f);
      }
    }
  };
  load(ch);
  __syncthreads();  // tws
  for (int g0 = 0; g0 < io.G; g0 += CMAC_CH) {  // the same rounds for every chunk
    const int g = g0 + ch;
    const bool on = g < io.G;
    if (vB && on) {
#pragma unroll
      for (int k = 0; k < P; ++k) f[k] = Fl[(size_t)g * io.f_gs + Q * k];
    }
    if (vA && on) two_first<P, Q, -1>(v, n1, buf[ch] + la * LS, tws);
    load(g + CMAC_CH);
    __syncthreads();
    if (vB && on) {
      float2 u[P];
      two_second<P, Q, -1>(u, k2, buf[ch] + lb * LS);
#pragma unroll
      for (int k = 0; k < P; ++k) acc[k] = cadd(acc[k], cmulc(u[k], f[k]));
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < P; ++k) buf[ch][lb * LS + k2 + Q * k] = acc[k];
  __syncthreads();
  if (ch == 0 && vB) {
    float2* dst = io.out + (size_t)blockIdx.y * io.out_bs + (size_t)(line0 + lb) * N + k2;
#pragma unroll
    for (int c = 1; c < CMAC_CH; ++c)
#pragma unroll
      for (int k = 0; k < P; ++k) acc[k] = cadd(acc[k], buf[c][lb * LS + k2 + Q * k]);
#pragma unroll
    for (int k = 0; k < P; ++k) acc[k] = cscale(acc[k], io.scale);
    if (io.accumulate) {  // every old value loaded before the first store
      float2 old[P];
#pragma unroll
      for (int k = 0; k < P; ++k) old[k] = dst[Q * k];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < P; ++k) acc[k] = cadd(old[k], acc[k]);
    }
#pragma unroll
    for (int k = 0; k < P; ++k) dst[Q * k] = acc[k];
  }
}

// One block per (slab, split, volume); bands in turn.  Phase 1: line k0 along
// axis 1 (its exchange in its own LDS line).  Phase 2: pair e of axis-1 columns
// (2e, 2e+1) as one complex pencil along axis 0.  A block of 15 waves fills the
// CU at N = 144 (one block, 160 KB of LDS); the next band's lines are loaded
// before phase 2, so their latency hides behind it.
template <int N>
__global__ void __launch_bounds__(Slab3Cfg<N>::T) k3_slab(Slab3 io, const float2* __restrict__ tw) {
  using C = Slab3Cfg<N>;
  constexpr int P = C::P, Q = C::Q, H = C::H, LS = C::LS;
  __shared__ __align__(16) float2 U[H * LS];
  __shared__ float2 Z[C::NP * LS];
  __shared__ float2 tws[N];
  const int tid = threadIdx.x, lane = tid & 63, sub = lane / Q, i = lane % Q;
  const int line = (tid >> 6) * C::LPW + sub;  // k0 in phase 1, the pair in phase 2
  const int j2 = blockIdx.x, split = blockIdx.y, b = blockIdx.z, n = io.n, np = n / 2;
  const bool vl = sub < C::LPW && line < H, vp = sub < C::LPW && line < np;
  for (int k = tid; k < N; k += C::T) tws[k] = tw[k];
  const float2* src = io.in + (size_t)b * io.in_bs + (size_t)j2 * (H * N) + (size_t)line * N + i;
  float2 v[Q], acc[P];
#pragma unroll
  for (int k = 0; k < P; ++k) acc[k] = make_float2(0.f, 0.f);
  const auto load = [&](int g) {
    if (vl && i < P && g < io.G) {
      const float2* p = src + (size_t)g * io.in_gs;
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) v[n2] = p[P * n2];
    }
  };
  load(split);
  __syncthreads();  // tws
  float2* ul = U + line * LS;
  float2* zl = Z + line * LS;
  for (int g = split; g < io.G; g += io.nsplit) {
    if (vl && i < P) two_first<P, Q, +1>(v, i, ul, tws);
    wave_order();
    float2 u[P];
    if (vl) two_second<P, Q, +1>(u, i, ul);
    wave_order();
    if (vl) {
#pragma unroll
      for (int k1 = 0; k1 < P; ++k1) ul[i + Q * k1] = u[k1];  // the whole line: phase 2 reads its window
    }
    load(g + io.nsplit);
    const float t = io.th[(size_t)b * io.th_bs + io.th0 + g];
    __syncthreads();  // the slab's columns are complete
    float2 z[Q];
    if (vp && i < P) {
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) {
        // m = i + P n2 < N/2 exactly for n2 < Q/2
        const int km = n2 < Q / 2 ? i + P * n2 : N - P * n2 - i;
        const float4 ab = *reinterpret_cast<const float4*>(U + km * LS + io.o + 2 * line);
        // Z[m] = A[m] + i B[m]; Z[N-m] = conj(A[m]) + i conj(B[m]); the
        // imaginary parts at m = 0 and N/2 are dropped as in a real inverse.
        z[n2] = n2 < Q / 2 ? make_float2(ab.x - ab.w, ab.y + ab.z) : make_float2(ab.x + ab.w, ab.z - ab.y);
        if (n2 == 0 || n2 == Q / 2)
          if (i == 0) z[n2] = make_float2(ab.x, ab.z);
      }
    }
    __syncthreads();  // the next band may overwrite the columns
    if (vp && i < P) two_first<P, Q, +1>(z, i, zl, tws);
    wave_order();
    if (vp) {
      two_second<P, Q, +1>(u, i, zl);
#pragma unroll
      for (int k1 = 0; k1 < P; ++k1)
        acc[k1] = cadd(acc[k1], make_float2(hard_keep(u[k1].x, t), hard_keep(u[k1].y, t)));
    }
    wave_order();
  }
  if (vp) {
    float2* a = io.acc + (size_t)b * io.acc_bs + (size_t)split * io.acc_ss + ((size_t)j2 * np + line) * n;
    if (!io.first) {  // every old value loaded before the first store
      float2 old[P];
#pragma unroll
      for (int k1 = 0; k1 < P; ++k1) {
        const int j = i + Q * k1 - io.o;
        old[k1] = in_window(j, n) ? a[j] : make_float2(0.f, 0.f);
      }
#pragma unroll
      for (int k1 = 0; k1 < P; ++k1) acc[k1] = cadd(old[k1], acc[k1]);
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
      const int j = i + Q * k1 - io.o;
      if (in_window(j, n)) a[j] = acc[k1];
    }
  }
}

// Sum of the splits' accumulators, transposed to (i0, i1, j2): a block takes
// one pair of axis-1 columns and a tile of 32 x 32 (j2, i0).
__global__ void __launch_bounds__(256) k3_slab_out(const float2* __restrict__ acc, long long ss, long long bs, int nsplit,
                                                   float* __restrict__ out, long long obs, int n) {
  __shared__ float2 t[32][33];
  const int np = n / 2, e = blockIdx.y, b = blockIdx.z, nt = (n + 31) / 32;
  const int j0 = (blockIdx.x / nt) * 32, i0 = (blockIdx.x % nt) * 32;
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
  const float2* a = acc + (size_t)b * bs;
#pragma unroll
  for (int r = 0; r < 32; r += 8) {
    const int j = j0 + y + r, i = i0 + x;
    float2 s = make_float2(0.f, 0.f);
    if (j < n && i < n)
      for (int k = 0; k < nsplit; ++k) s = cadd(s, a[(size_t)k * ss + ((size_t)j * np + e) * n + i]);
    t[y + r][x] = s;
  }
  __syncthreads();
  float* o = out + (size_t)b * obs;
#pragma unroll
  for (int r = 0; r < 32; r += 8) {
    const int i = i0 + y + r, j = j0 + x;
    if (i < n && j < n) {
      const float2 s = t[x][y + r];
      o[((size_t)i * n + 2 * e) * n + j] = s.x;
      o[((size_t)i * n + 2 * e + 1) * n + j] = s.y;
    }
  }
}

// A block runs all bands of its lines (the spectrum S is then read once) unless
// that leaves fewer than 1024 blocks (4 per CU): the small levels' launches were
// chains of 8 transforms in 205 blocks (80^3 grid: 16.6 us per group of 8, split
// 11.3 us).
template <int N, bool SLAB>
static hipError_t rows_band_n(const Rows3Mul& io, int nb, const float2* tw, hipStream_t s) {
  const int nl = (io.nlines + SLAB_LINES - 1) / SLAB_LINES;
  int gper = io.G;
  while (gper > 1 && nl * nb * ((io.G + gper - 1) / gper) < 1024) gper = (gper + 1) / 2;
  hipLaunchKernelGGL((k3_rows_band<N, SLAB>), dim3(nl, nb, (io.G + gper - 1) / gper), dim3(SLAB_LINES * Split3<N>::Q), 0,
                     s, io, gper, tw);
  return hipGetLastError();
}
template <int N>
static hipError_t rows_cmac2_n(const Rows3Cmac& io, int nb, const float2* tw, hipStream_t s) {
  hipLaunchKernelGGL((k3_rows_cmac2<N>), dim3((io.nlines + CMAC_LINES - 1) / CMAC_LINES, nb),
                     dim3(CMAC_CH * CMAC_LINES * Split3<N>::Q), 0, s, io, tw);
  return hipGetLastError();
}
template <int N>
static hipError_t slab_n(const Slab3& io, int nb, const float2* tw, hipStream_t s) {
  hipLaunchKernelGGL((k3_slab<N>), dim3(io.n, io.nsplit, nb), dim3(Slab3Cfg<N>::T), 0, s, io, tw);
  return hipGetLastError();
}
#define SHX3_SLAB_BY_N(N, F)          \
  switch (N) {                        \
    case 24: return F(24);            \
    case 32: return F(32);            \
    case 48: return F(48);            \
    case 64: return F(64);            \
    case 80: return F(80);            \
    case 144: return F(144);          \
    default: return hipErrorInvalidValue; \
  }
bool slab3_supported(int N, int n, int o) {
  switch (N) {
    case 24: case 32: case 48: case 64: case 80: return n % 2 == 0 && n + o <= N && o % 2 == 0;
    case 144: return n % 2 == 0 && n <= 128 && n + o <= N && o % 2 == 0;
    default: return false;
  }
}
int slab3_splits(int n, int G) {
  int s = 1;  // 128: two splits, a block for every CU; small sides, whose blocks share a CU, up to 8
  while (s < 8 && 2 * s <= G && n * s < 256) s *= 2;
  return s;
}
hipError_t launch3_rows_slab(int N, const Rows3Mul& io, int nb, const float2* tw, hipStream_t s) {
#define F(M) rows_band_n<M, true>(io, nb, tw, s)
  SHX3_SLAB_BY_N(N, F)
#undef F
}
hipError_t launch3_slab(int N, const Slab3& io, int nb, const float2* tw, hipStream_t s) {
#define F(M) slab_n<M>(io, nb, tw, s)
  SHX3_SLAB_BY_N(N, F)
#undef F
}
hipError_t launch3_slab_out(const float2* acc, long long acc_ss, long long acc_bs, int nsplit, float* out,
                            long long out_bs, int n, int nb, hipStream_t s) {
  const int nt = (n + 31) / 32;
  hipLaunchKernelGGL(k3_slab_out, dim3(nt * nt, n / 2, nb), dim3(256), 0, s, acc, acc_ss, acc_bs, nsplit, out, out_bs, n);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Band-pass masks (half axis = memory axis 0).
__device__ __forceinline__ double lf_at(const BpMask& m, int n, int k0, int k1, int k2) {
  const int f1 = k1 <= n - k1 ? k1 : n - k1;
  const int f2 = k2 <= n - k2 ? k2 : n - k2;
  if (k0 > m.P || f1 > m.P || f2 > m.P) return 0.0;
  return m.v[k0] * m.v[f1] * m.v[f2];
}

__global__ void k3_bp_split(const float2* __restrict__ X, long long xs, float2* __restrict__ Hs, long long hs,
                            float2* __restrict__ Lp, long long ls, int n, int M, BpMask m, double hscale,
                            double lscale) {
  const long long HX = (long long)(n / 2 + 1) * n * n;
  const long long HL = (long long)(M / 2 + 1) * M * M;
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  X += (size_t)b * xs;
  if (e < HX) {
    const int k2 = (int)(e % n), k1 = (int)((e / n) % n), k0 = (int)(e / ((long long)n * n));
    const double lf = lf_at(m, n, k0, k1, k2);
    const double h = sqrt(1.0 - lf * lf) * hscale;
    const float2 x = X[e];
    Hs[(size_t)b * hs + e] = make_float2((float)(x.x * h), (float)(x.y * h));
  } else if (e < HX + HL) {
    const long long q = e - HX;
    const int q2 = (int)(q % M), q1 = (int)((q / M) % M), q0 = (int)(q / ((long long)M * M));
    const int f1 = q1 <= M / 2 ? q1 : q1 - M, f2 = q2 <= M / 2 ? q2 : q2 - M;
    const int a1 = f1 < 0 ? -f1 : f1, a2 = f2 < 0 ? -f2 : f2;
    float2 r = make_float2(0.f, 0.f);
    if (q0 <= m.P && a1 <= m.P && a2 <= m.P) {
      const double lf = m.v[q0] * m.v[a1] * m.v[a2] * lscale;
      const int s1 = f1 < 0 ? f1 + n : f1, s2 = f2 < 0 ? f2 + n : f2;
      const float2 x = X[((size_t)q0 * n + s1) * n + s2];
      r = make_float2((float)(x.x * lf), (float)(x.y * lf));
    }
    Lp[(size_t)b * ls + q] = r;
  }
}

__global__ void k3_bp_merge(const float2* __restrict__ H, long long hs, const float2* __restrict__ Lp, long long ls,
                            float2* __restrict__ out, long long os, int n, int M, BpMask m, double hscale,
                            double lscale) {
  const long long HX = (long long)(n / 2 + 1) * n * n;
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (e >= HX) return;
  const int k2 = (int)(e % n), k1 = (int)((e / n) % n), k0 = (int)(e / ((long long)n * n));
  const double lf = lf_at(m, n, k0, k1, k2);
  const float2 h = H[(size_t)b * hs + e];
  const double hf = sqrt(1.0 - lf * lf) * hscale;
  double re = h.x * hf, im = h.y * hf;
  if (lf != 0.0) {
    const int f1 = k1 <= n / 2 ? k1 : k1 - n, f2 = k2 <= n / 2 ? k2 : k2 - n;
    const int s1 = f1 < 0 ? f1 + M : f1, s2 = f2 < 0 ? f2 + M : f2;
    const float2 l = Lp[(size_t)b * ls + ((size_t)k0 * M + s1) * M + s2];
    const double g = lf * lscale;
    re += l.x * g;
    im += l.y * g;
  }
  out[(size_t)b * os + e] = make_float2((float)re, (float)im);
}

// ---------------------------------------------------------------------------
// Launchers.
template <int N>
struct Launch3 {
  using RC = Rows3Cfg<N>;
  static hipError_t rows(int dir, const Rows3& io, int nb, const float2* tw, hipStream_t s) {
    const dim3 grid((io.nlines + RC::LPB - 1) / RC::LPB, nb);
    if (dir < 0)
      hipLaunchKernelGGL((k3_rows<N, -1>), grid, dim3(RC::T), 0, s, io, tw);
    else
      hipLaunchKernelGGL((k3_rows<N, +1>), grid, dim3(RC::T), 0, s, io, tw);
    return hipGetLastError();
  }
  static hipError_t rows_mul(const Rows3Mul& io, int nb, const float2* tw, hipStream_t s) {
    const dim3 grid((io.nlines + RC::LPB - 1) / RC::LPB, nb);
    hipLaunchKernelGGL((k3_rows_mul<N>), grid, dim3(RC::T), 0, s, io, tw);
    return hipGetLastError();
  }
  template <int CW>
  static hipError_t plane_cw(const Plane3Inv& io, int nb, const float2* tw, hipStream_t s) {
    const int nchunk = (io.n_out + CW - 1) / CW;
    const int nblk = nchunk * io.H * io.G * nb;
    hipLaunchKernelGGL((k3_plane_inv<N, CW>), dim3(nblk), dim3(Plane3Cfg<N>::T), 0, s, io, nchunk, nblk, nb, tw);
    return hipGetLastError();
  }
  static hipError_t plane_inv(const Plane3Inv& io, int nb, int cw, const float2* tw, hipStream_t s) {
    if constexpr (N >= 24) {
      if (cw == 0) cw = io.n_out >= 64 ? 64 : 32;
      if (cw == 64) return plane_cw<64>(io, nb, tw, s);
      if (cw == 32) return plane_cw<32>(io, nb, tw, s);
    }
    return hipErrorInvalidValue;
  }
  static hipError_t rows_cmac(const Rows3Cmac& io, int nb, const float2* tw, hipStream_t s) {
    const dim3 grid((io.nlines + RC::LPB - 1) / RC::LPB, nb);
    hipLaunchKernelGGL((k3_rows_cmac<N>), grid, dim3(RC::T), 0, s, io, tw);
    return hipGetLastError();
  }
  template <int CT>
  static hipError_t cols_ct(int dir, const Cols3& io, int nb, const float2* tw, hipStream_t s) {
    const dim3 grid(io.W / CT, io.P, nb);
    if (dir < 0)
      hipLaunchKernelGGL((k3_cols<N, CT, -1>), grid, dim3(Cols3Cfg<N, CT>::T), 0, s, io, tw);
    else
      hipLaunchKernelGGL((k3_cols<N, CT, +1>), grid, dim3(Cols3Cfg<N, CT>::T), 0, s, io, tw);
    return hipGetLastError();
  }
  static hipError_t cols(int dir, const Cols3& io, int nb, const float2* tw, hipStream_t s) {
    if (io.W % 16 == 0) return cols_ct<16>(dir, io, nb, tw, s);
    if (io.W % 8 == 0) return cols_ct<8>(dir, io, nb, tw, s);
    return hipErrorInvalidValue;
  }
  template <int CT>
  static hipError_t pfwd_ct(const Pencil3Fwd& io, int G, int nb, const float2* tw, hipStream_t s) {
    const dim3 grid(io.E / 2 / CT, G, nb);
    hipLaunchKernelGGL((k3_pencil_fwd<N, CT>), grid, dim3(Cols3Cfg<N, CT>::T), 0, s, io, tw);
    return hipGetLastError();
  }
  static hipError_t pencil_fwd(const Pencil3Fwd& io, int G, int nb, const float2* tw, hipStream_t s) {
    if ((io.E / 2) % 16 == 0) return pfwd_ct<16>(io, G, nb, tw, s);
    if ((io.E / 2) % 8 == 0) return pfwd_ct<8>(io, G, nb, tw, s);
    return hipErrorInvalidValue;
  }
  template <int CT>
  static hipError_t pinv_ct(const Pencil3Inv& io, int nb, const float2* tw, hipStream_t s) {
    const dim3 grid(io.E / 2 / CT, io.mode == 0 ? io.G : 1, nb);
    hipLaunchKernelGGL((k3_pencil_inv<N, CT>), grid, dim3(Cols3Cfg<N, CT>::T), 0, s, io, tw);
    return hipGetLastError();
  }
  static hipError_t pencil_inv(const Pencil3Inv& io, int nb, const float2* tw, hipStream_t s) {
    if ((io.E / 2) % 16 == 0) return pinv_ct<16>(io, nb, tw, s);
    if ((io.E / 2) % 8 == 0) return pinv_ct<8>(io, nb, tw, s);
    return hipErrorInvalidValue;
  }
};

#define SHX3_BY_N(N, EXPR)                                   \
  switch (N) {                                               \
    case 8: { using LT = Launch3<8>; return EXPR; }          \
    case 16: { using LT = Launch3<16>; return EXPR; }        \
    case 24: { using LT = Launch3<24>; return EXPR; }        \
    case 32: { using LT = Launch3<32>; return EXPR; }        \
    case 48: { using LT = Launch3<48>; return EXPR; }        \
    case 64: { using LT = Launch3<64>; return EXPR; }        \
    case 80: { using LT = Launch3<80>; return EXPR; }        \
    case 128: { using LT = Launch3<128>; return EXPR; }      \
    case 144: { using LT = Launch3<144>; return EXPR; }      \
    default: return hipErrorInvalidValue;                    \
  }

bool fft3_supported(int N) {
  switch (N) {
    case 8: case 16: case 24: case 32: case 48: case 64: case 80: case 128: case 144: return true;
    default: return false;
  }
}

hipError_t launch3_rows(int N, int dir, const Rows3& io, int nb, const float2* tw, hipStream_t s) {
  SHX3_BY_N(N, LT::rows(dir, io, nb, tw, s))
}
hipError_t launch3_rows_mul(int N, const Rows3Mul& io, int nb, const float2* tw, hipStream_t s) {
  switch (N) {
    case 24: return rows_band_n<24, false>(io, nb, tw, s);
    case 32: return rows_band_n<32, false>(io, nb, tw, s);
    case 48: return rows_band_n<48, false>(io, nb, tw, s);
    case 64: return rows_band_n<64, false>(io, nb, tw, s);
    case 80: return rows_band_n<80, false>(io, nb, tw, s);
    case 144: return rows_band_n<144, false>(io, nb, tw, s);
    case 8: return Launch3<8>::rows_mul(io, nb, tw, s);
    case 16: return Launch3<16>::rows_mul(io, nb, tw, s);
    case 128: return Launch3<128>::rows_mul(io, nb, tw, s);
    default: return hipErrorInvalidValue;
  }
}
hipError_t launch3_rows_cmac(int N, const Rows3Cmac& io, int nb, const float2* tw, hipStream_t s) {
  switch (N) {
    case 24: return rows_cmac2_n<24>(io, nb, tw, s);
    case 32: return rows_cmac2_n<32>(io, nb, tw, s);
    case 48: return rows_cmac2_n<48>(io, nb, tw, s);
    case 64: return rows_cmac2_n<64>(io, nb, tw, s);
    case 80: return rows_cmac2_n<80>(io, nb, tw, s);
    case 144: return rows_cmac2_n<144>(io, nb, tw, s);
    case 8: return Launch3<8>::rows_cmac(io, nb, tw, s);
    case 16: return Launch3<16>::rows_cmac(io, nb, tw, s);
    case 128: return Launch3<128>::rows_cmac(io, nb, tw, s);
    default: return hipErrorInvalidValue;
  }
}
bool plane3_supported(int N, int n_out) { return N >= 24 && fft3_supported(N) && n_out >= 8; }

hipError_t launch3_plane_inv(int N, const Plane3Inv& io, int nb, int cw, const float2* tw, hipStream_t s) {
  SHX3_BY_N(N, LT::plane_inv(io, nb, cw, tw, s))
}

hipError_t launch3_cols(int N, int dir, const Cols3& io, int nb, const float2* tw, hipStream_t s) {
  SHX3_BY_N(N, LT::cols(dir, io, nb, tw, s))
}
hipError_t launch3_pencil_fwd(int N, const Pencil3Fwd& io, int G, int nb, const float2* tw, hipStream_t s) {
  SHX3_BY_N(N, LT::pencil_fwd(io, G, nb, tw, s))
}
hipError_t launch3_pencil_inv(int N, const Pencil3Inv& io, int nb, const float2* tw, hipStream_t s) {
  SHX3_BY_N(N, LT::pencil_inv(io, nb, tw, s))
}

hipError_t launch3_bp_split(const float2* X, long long xs, float2* Hs, long long hs, float2* Lp, long long ls, int n,
                            int M, const BpMask& m, double hscale, double lscale, int nb, hipStream_t s) {
  const long long tot = (long long)(n / 2 + 1) * n * n + (long long)(M / 2 + 1) * M * M;
  const dim3 grid((unsigned)((tot + 255) / 256), nb);
  hipLaunchKernelGGL(k3_bp_split, grid, dim3(256), 0, s, X, xs, Hs, hs, Lp, ls, n, M, m, hscale, lscale);
  return hipGetLastError();
}

hipError_t launch3_bp_merge(const float2* H, long long hs, const float2* Lp, long long ls, float2* out,
                            long long os, int n, int M, const BpMask& m, double hscale, double lscale, int nb,
                            hipStream_t s) {
  const long long tot = (long long)(n / 2 + 1) * n * n;
  const dim3 grid((unsigned)((tot + 255) / 256), nb);
  hipLaunchKernelGGL(k3_bp_merge, grid, dim3(256), 0, s, H, hs, Lp, ls, out, os, n, M, m, hscale, lscale);
  return hipGetLastError();
}

}  // namespace shx
