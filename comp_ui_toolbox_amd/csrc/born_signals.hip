// Time gain compensation and time-domain signals (gfx950).
#include "born_internal.h"

#include <algorithm>
#include <cmath>

namespace born {

// ------------------------------------------------------ time gain compensation
// One discrete convolution along the frequency coefficients of every mix,
// cut off to the mix's own length N (linear_transforms.convolutions.fft,
// fft.m:85-126 with cut_off; convolution.m:62-98).  Taps k[d], |d| <= M:
//   forward  y[i] = sum_d k[d] x[i - d]         (0 <= i - d < N)
//   adjoint  y[j] = sum_d conj(k[d]) x[j + d]   (0 <= j + d < N)
// A wave computes 64 R outputs of one (mix, right-hand side), R consecutive
// ones per lane: the inputs of TGC_TC taps pass through its own LDS and slide
// through registers, one read per tap for R outputs; the taps are uniform
// (scalar loads).  R is taken so that one wave holds the longest mix where it
// can: 257 rows take R = 5, one wave, instead of two tiles of 256 rows with
// two reads per product (76 us for 5632 rows of 257 with 133 taps; 45 us here).
__device__ __forceinline__ void cfma(float2& a, float2 k, float2 x) {
  a.x = fmaf(k.x, x.x, fmaf(-k.y, x.y, a.x));
  a.y = fmaf(k.x, x.y, fmaf(k.y, x.x, a.y));
}
__device__ __forceinline__ void cfma(double2& a, double2 k, double2 x) {
  a.x = fma(k.x, x.x, fma(-k.y, x.y, a.x));
  a.y = fma(k.x, x.y, fma(k.y, x.x, a.y));
}

constexpr int TGC_TC = 240;   // taps per stage: a multiple of every R below

template <typename T, bool ADJ, int R>
__global__ __launch_bounds__(256) void k_tgc(const T* __restrict__ x, T* __restrict__ y, const T* __restrict__ taps,
                                             const int2* __restrict__ tiles, int n_tiles, const int* __restrict__ half,
                                             const int64_t* __restrict__ tap_off, const int64_t* __restrict__ mk_off,
                                             const int* __restrict__ mk_meta, int64_t N_obs) {
  // entry t of the window (t = lane R + k + tap offset) at (t / R) RP + t % R:
  // an odd lane stride keeps the lanes on different banks
  constexpr int RP = R | 1, WIN = 64 * R + TGC_TC, LDS = WIN / R * RP;
  extern __shared__ __align__(16) unsigned char tgc_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int tile = blockIdx.x * 4 + wave;
  if (tile >= n_tiles) return;
  T* win = reinterpret_cast<T*>(tgc_lds) + (size_t)wave * LDS;
  const int2 tl = tiles[tile];
  const int mk = tl.x, i0 = tl.y;
  const int M = half[mk], N = mk_meta[mk * 4 + 1];
  const int64_t o0 = mk_off[mk * 4 + 0];
  const T* kt = taps + tap_off[mk] + M;   // kt[d], -M <= d <= M
  const T* xr = x + (size_t)blockIdx.y * N_obs + o0;
  const T* mine = win + lane * RP;
  T acc[R];
#pragma unroll
  for (int k = 0; k < R; ++k) acc[k].x = acc[k].y = 0;
  for (int d0 = -M; d0 <= M; d0 += TGC_TC) {
    const int nd = min(TGC_TC, M - d0 + 1);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // adjoint: window entry t is x[i0 + d0 + t]; forward: mirrored,
    // entry t is x[i0 + 64 R - 1 - d0 - t], and lane and k count from the end
    for (int t = lane; t < WIN; t += 64) {
      const int j = ADJ ? i0 + d0 + t : i0 + 64 * R - 1 - d0 - t;
      T v;
      v.x = v.y = 0;
      if (j >= 0 && j < N) v = xr[j];
      win[t / R * RP + t % R] = v;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    T r[R];   // entries t + lane R .. + R - 1, entry e at e % R
#pragma unroll
    for (int k = 0; k < R; ++k) r[k] = mine[k];
    const int nb = (nd + R - 1) / R;
    for (int b = 0; b < nb; ++b) {
#pragma unroll
      for (int s = 0; s < R; ++s) {
        const int d = b * R + s;
        if (d < nd) {
          T kv = kt[d0 + d];
          if (ADJ) kv.y = -kv.y;
#pragma unroll
          for (int k = 0; k < R; ++k) cfma(acc[k], kv, r[(k + s) % R]);
          r[s] = mine[(b + 1) * RP + s];
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = ADJ ? i0 + lane * R + k : i0 + 64 * R - 1 - (lane * R + k);
    if (i < N) y[(size_t)blockIdx.y * N_obs + o0 + i] = acc[k];
  }
}

// Outputs per lane of k_tgc for mixes of up to N rows: one wave per mix up to 512 rows.
int tgc_outputs(int N) {
  for (int R : {1, 2, 3, 4, 5, 6})
    if (N <= 64 * R) return R;
  return 8;
}

template <typename T, int R>
static void tgc_launch(const Plan& P, bool adjoint, const void* in, void* out, const T* taps, int N_rhs, hipStream_t s) {
  constexpr int RP = R | 1, WIN = 64 * R + TGC_TC;
  const dim3 grid((unsigned)((P.n_tgc_tiles + 3) / 4), (unsigned)N_rhs);
  const size_t lds = (size_t)4 * (WIN / R * RP) * sizeof(T);
#define BORN_TGC(A)                                                                                                     \
  do {                                                                                                                  \
    hipFuncSetAttribute((const void*)k_tgc<T, A, R>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);           \
    hipLaunchKernelGGL((k_tgc<T, A, R>), grid, dim3(256), lds, s, (const T*)in, (T*)out, taps, P.d_tgc_tiles,           \
                       P.n_tgc_tiles, P.d_tgc_half, P.d_tgc_off, P.d_mk_off, P.d_mk_meta, P.N_obs);                     \
  } while (0)
  if (adjoint) BORN_TGC(true);
  else BORN_TGC(false);
#undef BORN_TGC
}

template <typename T>
static void tgc_by_outputs(const Plan& P, bool adjoint, const void* in, void* out, const T* taps, int N_rhs, hipStream_t s) {
  switch (P.tgc_R) {
    case 1: return tgc_launch<T, 1>(P, adjoint, in, out, taps, N_rhs, s);
    case 2: return tgc_launch<T, 2>(P, adjoint, in, out, taps, N_rhs, s);
    case 3: return tgc_launch<T, 3>(P, adjoint, in, out, taps, N_rhs, s);
    case 4: return tgc_launch<T, 4>(P, adjoint, in, out, taps, N_rhs, s);
    case 5: return tgc_launch<T, 5>(P, adjoint, in, out, taps, N_rhs, s);
    case 6: return tgc_launch<T, 6>(P, adjoint, in, out, taps, N_rhs, s);
    default: return tgc_launch<T, 8>(P, adjoint, in, out, taps, N_rhs, s);
  }
}

void launch_tgc(const Plan& P, bool adjoint, bool f64, const void* in, void* out, int N_rhs, hipStream_t s) {
  if (f64) tgc_by_outputs<double2>(P, adjoint, in, out, P.d_tgc_k64, N_rhs, s);
  else tgc_by_outputs<float2>(P, adjoint, in, out, P.d_tgc_k32, N_rhs, s);
}

// ------------------------------------------------------ time-domain signals
// rf[r][mk][n] = sum over the frequencies f of mix mk of
//   w_q * Re(u[r][obs(mk, f)] * exp(+j 2 pi q n / N_t)),
// q = f / delta_f the integer frequency index, w_q = 1 for q = 0 and for the
// Nyquist index N_t / 2, else 2: N_t * ifft(X, N_t, 'symmetric') of the
// zero-padded spectrum (signal_matrix.m:379-391, lbs_q = 0).  The phase is
// reduced exactly in integers, (q n) mod N_t, before the FP32 sincos.  Any
// frequency lists; regular plans with evenly spaced q take k_time_regular.
__global__ __launch_bounds__(256) void k_time_signals(const float2* __restrict__ u, const int* __restrict__ q_obs,
                                                      const int64_t* __restrict__ mk_off,
                                                      const int* __restrict__ mk_meta, int N_mk, int64_t N_obs,
                                                      int N_rhs, int N_t, float* __restrict__ rf) {
  const size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (idx >= (size_t)N_rhs * N_mk * N_t) return;
  const int n = (int)(idx % N_t);
  const size_t rs = idx / N_t;
  const int mk = (int)(rs % N_mk);
  const int r = (int)(rs / N_mk);
  const int64_t o0 = mk_off[mk * 4 + 0];
  const int Nf = mk_meta[mk * 4 + 1];
  const float2* ur = u + (size_t)r * N_obs;
  const float w0 = 6.283185307179586f / (float)N_t;
  float acc = 0.f;
  for (int f = 0; f < Nf; ++f) {
    const int q = q_obs[o0 + f];
    const float2 x = ur[o0 + f];
    const int ph = (int)(((int64_t)q * n) % N_t);
    float sn, cs;
    __sincosf(w0 * (float)ph, &sn, &cs);
    const float wq = (q == 0 || 2 * q == N_t) ? 1.f : 2.f;
    acc += wq * (x.x * cs - x.y * sn);
  }
  rf[idx] = acc;
}

void launch_time_signals(const Plan& P, const float2* u, const int* q_obs, int N_rhs, int N_t, float* rf,
                         hipStream_t s) {
  const size_t total = (size_t)N_rhs * P.N_mk * N_t;
  hipLaunchKernelGGL(k_time_signals, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, u, q_obs, P.d_mk_off,
                     P.d_mk_meta, P.N_mk, P.N_obs, N_rhs, N_t, rf);
}

// cs[i] = exp(j 2 pi i / N_t), evaluated in FP64
__global__ __launch_bounds__(256) void k_time_table(int N_t, float2* __restrict__ cs) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= N_t) return;
  double s, c;
  sincospi(2.0 * (double)i / (double)N_t, &s, &c);
  cs[i] = make_float2((float)c, (float)s);
}

// Regular plans (row = signal of a right-hand side, rows of N_f coefficients
// one after the other) with q = q0 + dq f.  A wave takes 64 samples of RB rows:
// the phase factor of 8 frequencies is one table entry times the kept factors
// of 1 .. 7 steps, and serves RB rows, whose coefficients are uniform.  With C
// the sum of the cosine and S that of the sine products, sample n is C - S and
// sample N_t - n is C + S: half of the samples are summed, and the one at N_t / 2
// by a sum of alternating signs.  Bound: the vector ALU, 2 RB + 5 instructions
// per frequency and two samples in place of a sincos and a 64-bit remainder per
// product (5632 rows of 640 samples from 257 frequencies: 1150 us there, 88 us
// here sample by sample, 56 in pairs).
template <int RB>
__global__ __launch_bounds__(256) void k_time_regular(const float2* __restrict__ u, const float2* __restrict__ cs,
                                                      int64_t rows, int Nf, int N_t, int q0, int dq, int n_nb,
                                                      int64_t task0, float* __restrict__ rf) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t task = task0 + (int64_t)blockIdx.x * 4 + wave;
  const int64_t row0 = task / n_nb * RB;
  if (row0 >= rows) return;
  const int n = (int)(task % n_nb) * 64 + lane, n_half = (N_t + 1) / 2;   // samples 0 .. n_half - 1
  const int nn = min(n, n_half - 1);
  const int rb = (int)(rows - row0 < RB ? rows - row0 : RB);
  const float2* x[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) x[r] = u + (row0 + min(r, rb - 1)) * Nf;
  const int step = (int)((int64_t)dq * nn % N_t);
  int at = (int)((int64_t)q0 * nn % N_t);
  float2 pw[8];
  {
    int k = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      pw[i] = cs[k];
      k += step;
      if (k >= N_t) k -= N_t;
    }
  }
  const int step8 = (int)((int64_t)dq * 8 * nn % N_t);
  float C[RB], S[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) C[r] = S[r] = 0.f;
  int f = 0;
  for (; f + 8 <= Nf; f += 8) {
    const float2 w = cs[at];
    at += step8;
    if (at >= N_t) at -= N_t;
    float sc[RB], ss[RB];   // of 8 frequencies: shorter chains round less
#pragma unroll
    for (int r = 0; r < RB; ++r) sc[r] = ss[r] = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float c = i ? fmaf(w.x, pw[i].x, -(w.y * pw[i].y)) : w.x;
      const float s = i ? fmaf(w.x, pw[i].y, w.y * pw[i].x) : w.y;
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const float2 v = x[r][f + i];
        sc[r] = fmaf(v.x, c, sc[r]);
        ss[r] = fmaf(v.y, s, ss[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      C[r] += sc[r];
      S[r] += ss[r];
    }
  }
  for (; f < Nf; ++f) {
    const float2 w = cs[at];
    at += step;
    if (at >= N_t) at -= N_t;
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const float2 v = x[r][f];
      C[r] = fmaf(v.x, w.x, C[r]);
      S[r] = fmaf(v.y, w.y, S[r]);
    }
  }
  // the zero and Nyquist indices count once: take half of them back (an infinite
  // one stays what it is)
  auto half = [](float v) { return fabsf(v) <= 3.402823466e+38f ? 0.5f * v : 0.f; };
  const int fz = q0 == 0 ? 0 : -1, fn = 2 * (q0 + dq * (Nf - 1)) == N_t ? Nf - 1 : -1;
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    float c = C[r];
    if (fz >= 0) c -= half(x[r][0].x);
    if (fn >= 0) c -= half(nn & 1 ? -x[r][fn].x : x[r][fn].x);
    if (r < rb && n < n_half) {
      float* out = rf + (row0 + r) * N_t;
      out[n] = 2.f * (c - S[r]);
      if (n > 0) out[N_t - n] = 2.f * (c + S[r]);
    }
  }
  if ((N_t & 1) || n >= 64) return;
  // sample N_t / 2, by the wave of samples 0 .. 63
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    float c = 0.f;
    for (int k = lane; k < Nf; k += 64) {
      const float v = (k == fz || k == fn ? 0.5f : 1.f) * x[r][k].x;
      c += (q0 + dq * k) & 1 ? -v : v;
    }
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) c += __shfl_xor(c, m);
    if (lane == 0 && r < rb) rf[(row0 + r) * N_t + N_t / 2] = 2.f * c;
  }
}

void launch_time_table(int N_t, float2* cs, hipStream_t s) {
  hipLaunchKernelGGL(k_time_table, dim3((N_t + 255) / 256), dim3(256), 0, s, N_t, cs);
}

void launch_time_regular(const Plan& P, const float2* u, int N_rhs, int N_t, int q0, int dq, float* rf, hipStream_t s) {
  constexpr int RB = 4;   // 8: 6 us slower at 5632 rows; 12 and 16: the uniform coefficients no longer fit, 190 and 230 us
  const int64_t rows = (int64_t)P.N_mk * N_rhs;
  const int n_nb = ((N_t + 1) / 2 + 63) / 64;
  const int64_t tasks = (rows + RB - 1) / RB * n_nb, at_once = 4 * ((1ll << 24) - 1);   // (a launch holds less than 2^32 threads)
  for (int64_t t0 = 0; t0 < tasks; t0 += at_once)
    hipLaunchKernelGGL(k_time_regular<RB>, dim3((unsigned)((std::min(at_once, tasks - t0) + 3) / 4)), dim3(256), 0, s, u,
                       P.d_time_cs, rows, P.N_fu, N_t, q0, dq, n_nb, t0, rf);
}

}  // namespace born
