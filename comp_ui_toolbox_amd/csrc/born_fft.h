// Transforms of length 64, 128 and 256 inside a wave (gfx950 device code).
//
// A transform of length L = 16 * TL runs on TL lanes of a wave with 16
// entries each, n = j + TL * q (lane j, entry q): a DFT of 16 in registers,
// twiddles, an exchange through the wave's own LDS, and 16 / TL DFTs of TL in
// registers, whose outputs land in the same order.  A wave carries
// FPW = 64 / TL transforms, lane = j * FPW + g.
#pragma once
#include <hip/hip_runtime.h>

namespace born {

// Aligned as a whole: for the LDS that a launch sizes the compiler has no other
// word that an entry may be read and written in one access.
template <typename R>
struct alignas(2 * sizeof(R)) Cx {
  R x, y;
};
typedef Cx<float> cf;

template <typename R>
__device__ __forceinline__ Cx<R> cadd(Cx<R> a, Cx<R> b) { return {a.x + b.x, a.y + b.y}; }
template <typename R>
__device__ __forceinline__ Cx<R> csub(Cx<R> a, Cx<R> b) { return {a.x - b.x, a.y - b.y}; }
template <typename R>
__device__ __forceinline__ Cx<R> caddi(Cx<R> a, Cx<R> b) { return {a.x - b.y, a.y + b.x}; }   // a + i b
template <typename R>
__device__ __forceinline__ Cx<R> csubi(Cx<R> a, Cx<R> b) { return {a.x + b.y, a.y - b.x}; }   // a - i b
template <typename R>
__device__ __forceinline__ Cx<R> cmulc(Cx<R> a, R c, R s) {   // a * (c + i s)
  return {fma(a.x, c, -(a.y * s)), fma(a.x, s, a.y * c)};
}
template <typename R>
__device__ __forceinline__ void cmac(Cx<R>& acc, Cx<R> a, Cx<R> b) {
  acc.x = fma(a.x, b.x, fma(-a.y, b.y, acc.x));
  acc.y = fma(a.x, b.y, fma(a.y, b.x, acc.y));
}

// DFT of 4, exp(+2 pi i ab / 4), in place
template <typename R>
__device__ __forceinline__ void dft4(Cx<R>& a, Cx<R>& b, Cx<R>& c, Cx<R>& d) {
  const Cx<R> s = cadd(a, c), t = csub(a, c), u = cadd(b, d), v = csub(b, d);
  a = cadd(s, u);
  b = caddi(t, v);
  c = csub(s, u);
  d = csubi(t, v);
}

// Products with the constants of the DFTs of 16 and 8.  FP32 rounds cos(pi/8)
// and sqrt(1/2) down, which lowers the energy of every transform by 3e-8; with
// ACC the constants carry their remainders (one more multiply-add per
// product), for sums of squared outputs: 5e-9 is left.
template <typename R, bool ACC>
__device__ __forceinline__ R fft_r2(R a) {
  const double r2 = 0.70710678118654752440;
  if constexpr (ACC && sizeof(R) == 4) return fma(a, (R)r2, a * (R)(r2 - (double)(R)r2));
  return a * (R)r2;
}

constexpr double FFT_C1 = 0.92387953251128675613, FFT_S1 = 0.38268343236508977173;

// a * exp(i pi / 8) and a * exp(3 i pi / 8) with the remainder of cos(pi/8) within
// the products (added to a rounded product most of it would be lost again)
template <typename R>
__device__ __forceinline__ Cx<R> fft_p8(Cx<R> a) {
  const R c = (R)FFT_C1, l = (R)(FFT_C1 - (double)(R)FFT_C1), s = (R)FFT_S1;
  return {fma(a.x, c, fma(a.x, l, -(a.y * s))), fma(a.y, c, fma(a.y, l, a.x * s))};
}
template <typename R>
__device__ __forceinline__ Cx<R> fft_p38(Cx<R> a) {
  const R c = (R)FFT_C1, l = (R)(FFT_C1 - (double)(R)FFT_C1), s = (R)FFT_S1;
  return {fma(-a.y, c, fma(-a.y, l, a.x * s)), fma(a.x, c, fma(a.x, l, a.y * s))};
}

// DFT of 16, exp(+2 pi i q k / 16), in place and in order; the entries
// q >= NZ are taken as zero.
template <typename R, int NZ, bool ACC = false>
__device__ __forceinline__ void dft16(Cx<R> (&x)[16]) {
  const R c1 = (R)FFT_C1, s1 = (R)FFT_S1;
  Cx<R> t[4][4];   // t[b][c], q = 4 a + b, k = c + 4 d
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (4 + b >= NZ) {   // one entry
      t[b][0] = t[b][1] = t[b][2] = t[b][3] = x[b];
    } else if (8 + b >= NZ) {   // two
      t[b][0] = cadd(x[b], x[4 + b]);
      t[b][1] = caddi(x[b], x[4 + b]);
      t[b][2] = csub(x[b], x[4 + b]);
      t[b][3] = csubi(x[b], x[4 + b]);
    } else if (12 + b >= NZ) {   // three
      const Cx<R> s = cadd(x[b], x[8 + b]), d = csub(x[b], x[8 + b]);
      t[b][0] = cadd(s, x[4 + b]);
      t[b][1] = caddi(d, x[4 + b]);
      t[b][2] = csub(s, x[4 + b]);
      t[b][3] = csubi(d, x[4 + b]);
    } else {
      t[b][0] = x[b];
      t[b][1] = x[4 + b];
      t[b][2] = x[8 + b];
      t[b][3] = x[12 + b];
      dft4(t[b][0], t[b][1], t[b][2], t[b][3]);
    }
  }
  auto r8 = [&](Cx<R> a) -> Cx<R> { return {fft_r2<R, ACC>(a.x - a.y), fft_r2<R, ACC>(a.x + a.y)}; };      // * exp(i pi / 4)
  auto r38 = [&](Cx<R> a) -> Cx<R> { return {-fft_r2<R, ACC>(a.x + a.y), fft_r2<R, ACC>(a.x - a.y)}; };   // * exp(3 i pi / 4)
  if constexpr (ACC && sizeof(R) == 4) {
    t[1][1] = fft_p8(t[1][1]);
    t[1][3] = fft_p38(t[1][3]);
    t[3][1] = fft_p38(t[3][1]);
    t[3][3] = fft_p8<R>({-t[3][3].x, -t[3][3].y});
  } else {
    t[1][1] = cmulc(t[1][1], c1, s1);
    t[1][3] = cmulc(t[1][3], s1, c1);
    t[3][1] = cmulc(t[3][1], s1, c1);
    t[3][3] = cmulc(t[3][3], -c1, -s1);
  }
  t[1][2] = r8(t[1][2]);
  t[2][1] = r8(t[2][1]);
  t[2][2] = {-t[2][2].y, t[2][2].x};
  t[2][3] = r38(t[2][3]);
  t[3][2] = r38(t[3][2]);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    dft4(t[0][c], t[1][c], t[2][c], t[3][c]);
    x[c] = t[0][c];
    x[c + 4] = t[1][c];
    x[c + 8] = t[2][c];
    x[c + 12] = t[3][c];
  }
}

// DFT of 8, in order
template <typename R, bool ACC = false>
__device__ __forceinline__ void dft8(Cx<R> (&x)[8]) {
  Cx<R> e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
  dft4(e[0], e[1], e[2], e[3]);
  dft4(o[0], o[1], o[2], o[3]);
  o[1] = {fft_r2<R, ACC>(o[1].x - o[1].y), fft_r2<R, ACC>(o[1].x + o[1].y)};
  o[2] = {-o[2].y, o[2].x};
  o[3] = {-fft_r2<R, ACC>(o[3].x + o[3].y), fft_r2<R, ACC>(o[3].x - o[3].y)};
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    x[c] = cadd(e[c], o[c]);
    x[c + 4] = csub(e[c], o[c]);
  }
}

// LDS entries of one wave: 16 rows of 64 lanes, padded by FPW entries so that
// the reads of the exchange (rows j', lanes j * FPW + g) fall on all banks.
template <int TL>
struct FftShape {
  static constexpr int FPW = 64 / TL, ROW = 64 + FPW, LDS = 16 * ROW;
};

// Transform of the FPW length-16*TL sequences of a wave, exp(+2 pi i n k / L):
// x[q] holds entry j + TL * q on entry and on return, entries q >= NZ are
// taken as zero.  tw(k): the lane's twiddle exp(2 pi i j k / L); lds: the
// wave's own exchange buffer (the LDS operations of one wave complete in
// order, so no barrier is needed).
// mid: called between the exchange's writes and its reads (loads that the
// second half should cover).
template <typename R, int TL, int NZ, bool ACC, typename Tw, typename Mid>
__device__ __forceinline__ void fft_wave_t(Cx<R> (&x)[16], Tw&& tw, Cx<R>* lds, int lane, Mid&& mid) {
  constexpr int FPW = FftShape<TL>::FPW, ROW = FftShape<TL>::ROW;
  const int j = lane / FPW, g = lane % FPW;
  dft16<R, NZ, ACC>(x);
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    if (k > 0) {
      const Cx<R> w = tw(k);
      x[k] = cmulc(x[k], w.x, w.y);
    }
    lds[k * ROW + lane] = x[k];
  }
  mid();
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if constexpr (TL == 16) {
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = lds[j * ROW + i * FPW + g];
    dft16<R, 16, ACC>(x);
  } else if constexpr (TL == 8) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      Cx<R> y[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = lds[(j + 8 * m) * ROW + i * FPW + g];
      dft8<R, ACC>(y);
#pragma unroll
      for (int k = 0; k < 8; ++k) x[m + 2 * k] = y[k];
    }
  } else {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      Cx<R> y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = lds[(j + 4 * m) * ROW + i * FPW + g];
      dft4(y[0], y[1], y[2], y[3]);
#pragma unroll
      for (int k = 0; k < 4; ++k) x[m + 4 * k] = y[k];
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Twiddles in registers
template <typename R, int TL, bool HALF, bool ACC = false>
__device__ __forceinline__ void fft_wave(Cx<R> (&x)[16], const Cx<R> (&tw)[16], Cx<R>* lds, int lane) {
  fft_wave_t<R, TL, HALF ? 8 : 16, ACC>(x, [&](int k) { return tw[k]; }, lds, lane, [] {});
}

// Twiddles in LDS, [16][TL]: 30 registers fewer, a third wave per SIMD where
// these were what kept it out.
template <int TL, int NZ, typename Mid>
__device__ __forceinline__ void fft_wave_l(cf (&x)[16], const cf* twl, cf* lds, int lane, Mid&& mid) {
  const cf* mine = twl + lane / FftShape<TL>::FPW;
  cf tw[16];
#pragma unroll
  for (int k = 1; k < 16; ++k) tw[k] = mine[k * TL];
  __builtin_amdgcn_sched_barrier(0);   // in flight during the first DFT
  fft_wave_t<float, TL, NZ, false>(x, [&](int k) { return tw[k]; }, lds, lane, mid);
}
template <int TL, int NZ>
__device__ __forceinline__ void fft_wave_l(cf (&x)[16], const cf* twl, cf* lds, int lane) {
  fft_wave_l<TL, NZ>(x, twl, lds, lane, [] {});
}

// All threads of the workgroup.
template <int TL>
__device__ __forceinline__ void load_twiddles_lds(const float2* __restrict__ tw, cf* twl) {
  for (int i = threadIdx.x; i < 16 * TL; i += blockDim.x) {
    const float2 v = tw[(i % TL) * 16 + i / TL];
    twl[i] = {v.x, v.y};
  }
  __syncthreads();
}

template <int TL>
__device__ __forceinline__ void load_twiddles(const float2* __restrict__ tw, int j, cf (&t)[16]) {
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const float2 v = tw[j * 16 + k];
    t[k] = {v.x, v.y};
  }
}

}  // namespace born
