// Received energies of structured plans (gfx950), FP64.
//
//   E[p] = sum over the mixes k and frequencies f of a measurement of
//          |p_inc[f, p]|^2 |sum_a pref[k][f, a] h_ref[f, shift(p, e_a)]|^2
// (energy_rx_canonical, operator_born.m:718-859, identity TGC).  The lateral
// structure of the shift map turns the inner sums into correlations of one
// h_ref row: with point i = Np s + phi and t = N_ex - 1 - e_x, element e_x
// meets row entry Np (s + t) + phi.  A wave takes LPW R consecutive s of every
// phase of one row (lane = jl Np + phi holds s = R jl .. R jl + R - 1), keeps
// the row's window in its own LDS and slides it through registers: one LDS
// read serves R multiply-adds.  The waves of a workgroup share the row
// segment and split the measurement's frequencies.
//
// k_energy_single: mixes of one active element, where |sum|^2 is a real
// correlation of |h|^2 with the summed squared prefactors of each (pair,
// element) (k_energy_weights); k_energy_multi: all other mixes, KB
// observations at a time, complex.
//
// The map-driven kernel (k_energy_rx, one thread per point, one map read and
// one gather per element) stays for plans off the structured path: it waits
// on those reads.  128 elements, 384 x 384 points, 129 frequencies, identity
// mixes: 22.4 ms per measurement there, 0.18 ms here (FP64 rate: 0.06 ms).
#include "born_fft.h"
#include "born_internal.h"

#include <algorithm>
#include <type_traits>

namespace born {

// points of the window that the waves of one row segment keep per phase
__host__ __device__ constexpr int e_window(int LPW, int nb, int R) {
  const int w = (LPW + nb) * (R + 1);
  return w + (20 - w % 16) % 16;   // phases 4 entries apart modulo 16: lanes on all banks
}

__device__ __forceinline__ void e_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// ew[(pair * Ney + ey) * NeP + t], t = Nex - 1 - ex: sum of |prefactor|^2 over
// the observations of the pair whose mix has this element alone; zero padding.
__global__ __launch_bounds__(256) void k_energy_weights(const int64_t* __restrict__ pe_off, const int2* __restrict__ pe_ent,
                                                        const double2* __restrict__ pref, const int* __restrict__ obs_mk,
                                                        const int* __restrict__ mk_meta, int N_pairs, int Nex, int Ney,
                                                        int NeP, double* __restrict__ ew) {
  const size_t idx = blockIdx.x * (size_t)256 + threadIdx.x;
  if (idx >= (size_t)N_pairs * Ney * NeP) return;
  const int t = (int)(idx % NeP);
  const size_t py = idx / NeP;
  const int ey = (int)(py % Ney);
  const size_t pair = py / Ney;
  double s = 0.0;
  if (t < Nex) {
    const size_t pe = pair * ((size_t)Nex * Ney) + (Nex - 1 - t) + (size_t)Nex * ey;
    for (int64_t j = pe_off[pe]; j < pe_off[pe + 1]; ++j) {
      const int2 oe = pe_ent[j];
      if (mk_meta[obs_mk[oe.x] * 4 + 2] != 1) continue;
      const double2 c = pref[oe.y];
      s += c.x * c.x + c.y * c.y;
    }
  }
  ew[idx] = s;
}

struct EnergyArgs {
  const float2* h;
  const float2* P;
  const int* ext;
  const int* hrow;
  const int* pair_fg;
  int pair0, n_pairs;     // the measurement's pairs
  int Nx, n_rows, Np, Nex, Ney, N_ext, N_pts, HR, NeP;
  int64_t H_plane;
  int nseg, nb, LPW, WLp;
  const double* ew;
  // observations of mixes with several active elements, by pair
  const int64_t* row_off;
  const int2* rows;       // (mix, frequency of the mix)
  const int* mk_meta;
  const int64_t* mk_off;
  const int* act;
  const double2* pref;
  int add;                // k_energy_multi: add to E
};

// Fills the wave's window of row hr: entry x of phase phi at win[phi * WLp + x + x / R].
template <int R, int NP, typename T, typename F>
__device__ __forceinline__ void e_fill(const EnergyArgs& A, const float2* __restrict__ hr, int s0, int lane, T* win, F&& conv) {
  const int Np = NP > 0 ? NP : A.Np;
  const int n = Np * (A.LPW + A.nb) * R, t0 = Np * s0;
  for (int idx = lane; idx < n; idx += 64) {
    const int x = idx / Np, phi = idx - x * Np;
    float2 v = make_float2(0.f, 0.f);
    if (t0 + idx < A.N_ext) v = hr[A.ext[t0 + idx]];
    win[phi * A.WLp + x + x / R] = conv(v);
  }
}

// Entry N of the 16 that each row of 16 lanes holds, in all lanes.
template <int N>
__device__ __forceinline__ double e_bcast(double w) {
  return __builtin_amdgcn_update_dpp(w, w, 0x150 + N, 0xf, 0xf, true);
}

// S[k] += w[D .. D1 - 1] of the chunk times entries k + D .. of x (block 0 at
// x0, the next at x1).
template <int R, int D, int D1>
__device__ __forceinline__ void e_mac(double (&S)[R], double w, const double (&x0)[R], const double (&x1)[R]) {
  if constexpr (D < D1) {
    const double wv = e_bcast<D>(w);
#pragma unroll
    for (int k = 0; k < R; ++k) S[k] = fma(wv, k + D % R < R ? x0[(k + D) % R] : x1[(k + D) % R], S[k]);
    e_mac<R, D + 1, D1>(S, w, x0, x1);
  }
}

// The elements' weights are taken 2 R at a time: lane l holds number l % 16 of
// the chunk, and each is broadcast within the rows of 16 lanes (through the
// scalar cache, which they miss, a step of R elements took 750 cycles for 36
// multiply-adds).  MI > 0: a lane's MI entries of the window and its weights are
// loaded for the next pair during the multiply-adds of this one (positions in
// the row and in LDS are the same for all pairs); MI = 0, for more than 16
// entries: in between.
// 128 elements, 384 x 384 points, 129 frequencies: 354 us with scalar weights
// and windows filled in between, 268 with the windows loaded ahead, 182 with
// both (the FP64 multiply-adds alone: 62).  What is left: 384 workgroups on 256
// compute units (1.33), one broadcast and the window's LDS reads per R
// multiply-adds.  Positions packed in one register (three waves per SIMD
// instead of two) cost 14 % for the unpacking.
template <int R, int MI>
__global__ __launch_bounds__(512) void k_energy_single(EnergyArgs A, double* __restrict__ E) {
  extern __shared__ double e_lds[];
  const int Np = A.Np;
  const int W = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int row = blockIdx.x / A.nseg, seg = blockIdx.x - row * A.nseg;
  const int jl = lane / Np, phi = lane - jl * Np;
  const bool on = jl < A.LPW;
  const int s0 = seg * A.LPW * R;
  const int n_win = Np * A.WLp, n_w = A.nb * R;   // window, weights, then an entry for what lies past both
  const int per_wave = n_win + n_w + 1;
  double* win = e_lds + (size_t)wave * per_wave;
  const double* mine = win + phi * A.WLp + (on ? jl : 0) * (R + 1);
  const double* wl = win + n_win + min(lane & 15, 2 * R - 1);
  const int c0 = (int)((long)A.n_pairs * wave / W), c1 = (int)((long)A.n_pairs * (wave + 1) / W);
  int at[R];
  double acc[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = Np * (s0 + jl * R + k) + phi;
    at[k] = row * A.Nx + min(i, A.Nx - 1);
    acc[k] = 0.0;
  }
  constexpr int M = MI > 0 ? MI : 1;
  unsigned from[M];   // byte in the row; past its end where the window has no entry: reads 0
  int to[M];          // entry of the window
  float2 hv[M];
  double wv[3];
  if constexpr (MI > 0) {
    const int n = Np * (A.LPW + A.nb) * R, t0 = Np * s0;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int idx = lane + 64 * i, x = idx / Np;
      const unsigned at_x = 8u * (unsigned)A.ext[min(t0 + idx, A.N_ext - 1)];
      from[i] = idx < n && t0 + idx < A.N_ext ? at_x : 0x7ffffff0u;
      to[i] = idx < n ? (idx - x * Np) * A.WLp + x + x / R : per_wave - 1;
    }
  }
  auto row_of = [&](int fg, int ey) {
    return A.h + (size_t)fg * A.H_plane + (size_t)A.hrow[ey * A.n_rows + row] * A.HR;
  };
  auto load_w = [&](int c, int ey) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)(A.ew + ((size_t)(A.pair0 + c) * A.Ney + ey) * A.NeP), 0, A.NeP * 8, 0x27000);
#pragma unroll
    for (int i = 0; i < 3; ++i) {   // (at most 144)
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, 8 * (lane + 64 * i), 0, 0);
      wv[i] = __hiloint2double((int)v[1], (int)v[0]);
    }
  };
  auto load = [&](int c, int fg, int ey) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)row_of(fg, ey), 0, A.HR * 8, 0x27000);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, from[i], 0, 0);
      hv[i] = make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
    }
    load_w(c, ey);
  };
  int fg = 0;   // frequency of the pair, a pair ahead (MI > 0) of the loads that it is for
  if (c0 < c1) {
    fg = A.pair_fg[A.pair0 + c0];
    if constexpr (MI > 0) load(c0, fg, 0);
  }
  for (int c = c0; c < c1; ++c) {
    const int fg_next = A.pair_fg[A.pair0 + min(c + 1, c1 - 1)];
    const float2* P = A.P + (size_t)(A.pair0 + c) * A.N_pts;
    float2 pv[R];
#pragma unroll
    for (int k = 0; k < R; ++k) pv[k] = P[at[k]];
    double S[R];
#pragma unroll
    for (int k = 0; k < R; ++k) S[k] = 0.0;
    for (int ey = 0; ey < A.Ney; ++ey) {
      e_fence();
      auto square = [](float2 v) { return (double)v.x * v.x + (double)v.y * v.y; };
      if constexpr (MI > 0) {
#pragma unroll
        for (int i = 0; i < MI; ++i) win[to[i]] = square(hv[i]);
      } else {
        load_w(c, ey);
        e_fill<R, 0>(A, row_of(fg, ey), s0, lane, win, square);
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) win[n_win + min(lane + 64 * i, n_w)] = wv[i];
      if constexpr (MI > 0) {
        __builtin_amdgcn_sched_barrier(0);
        const bool last = ey + 1 == A.Ney;
        load(last ? min(c + 1, c1 - 1) : c, last ? fg_next : fg, last ? 0 : ey + 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      e_fence();
      double a[R], b[R];
#pragma unroll
      for (int i = 0; i < R; ++i) a[i] = mine[i];
      const double* x = mine + R + 1;
      for (int t = 0; t < A.nb; t += 2) {
        const double w = wl[t * R];
#pragma unroll
        for (int i = 0; i < R; ++i) b[i] = x[i];
        x += R + 1;
        e_mac<R, 0, R>(S, w, a, b);
#pragma unroll
        for (int i = 0; i < R; ++i) a[i] = x[i];
        x += R + 1;
        e_mac<R, R, 2 * R>(S, w, b, a);
      }
    }
#pragma unroll
    for (int k = 0; k < R; ++k) acc[k] = fma((double)pv[k].x * pv[k].x + (double)pv[k].y * pv[k].y, S[k], acc[k]);
    fg = fg_next;
  }
  e_fence();
#pragma unroll
  for (int k = 0; k < R; ++k) win[k * 64 + lane] = acc[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = Np * (s0 + jl * R + k) + phi;
    if (k % W == wave && on && i < A.Nx) {
      double s = 0.0;
      for (int v = 0; v < W; ++v) s += e_lds[(size_t)v * per_wave + k * 64 + lane];
      E[(size_t)row * A.Nx + i] = s;
    }
  }
}

// KB observations of one pair at a time, their prefactors over the elements
// of a slice in the wave's LDS.
template <int R, int NP, int KB>
__global__ __launch_bounds__(256) void k_energy_multi(EnergyArgs A, double* __restrict__ E) {
  extern __shared__ double e_lds[];
  const int Np = NP > 0 ? NP : A.Np;
  const int W = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int row = blockIdx.x / A.nseg, seg = blockIdx.x - row * A.nseg;
  const int jl = lane / Np, phi = lane - jl * Np;
  const bool on = jl < A.LPW;
  const int s0 = seg * A.LPW * R;
  const size_t per_wave = (size_t)Np * A.WLp + (size_t)A.nb * R * KB * 2;   // doubles
  float2* win = reinterpret_cast<float2*>(e_lds + wave * per_wave);
  double2* coef = reinterpret_cast<double2*>(e_lds + wave * per_wave + (size_t)Np * A.WLp);
  const float2* mine = win + phi * A.WLp + (on ? jl : 0) * (R + 1);
  const int c0 = (int)((long)A.n_pairs * wave / W), c1 = (int)((long)A.n_pairs * (wave + 1) / W);
  int at[R];
  double acc[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = Np * (s0 + jl * R + k) + phi;
    at[k] = row * A.Nx + min(i, A.Nx - 1);
    acc[k] = 0.0;
  }
  for (int c = c0; c < c1; ++c) {
    const int pair = A.pair0 + c;
    const float2* P = A.P + (size_t)pair * A.N_pts;
    const float2* h = A.h + (size_t)A.pair_fg[pair] * A.H_plane;
    float2 pv[R];
#pragma unroll
    for (int k = 0; k < R; ++k) pv[k] = P[at[k]];
    double q2[R];
#pragma unroll
    for (int k = 0; k < R; ++k) q2[k] = 0.0;
    const int64_t r0 = A.row_off[pair], r1 = A.row_off[pair + 1];
    for (int64_t rb = r0; rb < r1; rb += KB) {
      double qx[KB][R], qy[KB][R];
#pragma unroll
      for (int b = 0; b < KB; ++b)
#pragma unroll
        for (int k = 0; k < R; ++k) qx[b][k] = qy[b][k] = 0.0;
      for (int ey = 0; ey < A.Ney; ++ey) {
        e_fence();
        if (rb == r0 || A.Ney > 1)
          e_fill<R, NP>(A, h + (size_t)A.hrow[ey * A.n_rows + row] * A.HR, s0, lane, win, [](float2 v) { return v; });
        for (int i = lane; i < A.nb * R * KB; i += 64) coef[i] = make_double2(0.0, 0.0);
        e_fence();
        for (int b = 0; b < KB && rb + b < r1; ++b) {
          const int2 mf = A.rows[rb + b];
          const int Nf = A.mk_meta[mf.x * 4 + 1], Na = A.mk_meta[mf.x * 4 + 2];
          const int64_t a_off = A.mk_off[mf.x * 4 + 2], p_off = A.mk_off[mf.x * 4 + 3];
          for (int a = lane; a < Na; a += 64) {
            const int e = A.act[a_off + a];
            const int ex = e % A.Nex;
            if (e / A.Nex == ey) coef[(A.Nex - 1 - ex) * KB + b] = A.pref[p_off + (int64_t)a * Nf + mf.y];
          }
        }
        e_fence();
        double2 x[R];
#pragma unroll
        for (int i = 0; i < R; ++i) {
          const float2 v = mine[i];
          x[i] = make_double2(v.x, v.y);
        }
        for (int t = 0; t < A.nb; ++t) {
#pragma unroll
          for (int d = 0; d < R; ++d) {
            // x holds entries R t + d .. R t + d + R - 1, entry i at (i % R)
#pragma unroll
            for (int b = 0; b < KB; ++b) {
              const double2 w = coef[(t * R + d) * KB + b];
#pragma unroll
              for (int k = 0; k < R; ++k) {
                const double2 v = x[(k + d) % R];
                qx[b][k] = fma(w.x, v.x, fma(-w.y, v.y, qx[b][k]));
                qy[b][k] = fma(w.x, v.y, fma(w.y, v.x, qy[b][k]));
              }
            }
            const float2 v = mine[(t + 1) * (R + 1) + d];
            x[d] = make_double2(v.x, v.y);
          }
        }
      }
#pragma unroll
      for (int b = 0; b < KB; ++b)
#pragma unroll
        for (int k = 0; k < R; ++k) q2[k] += qx[b][k] * qx[b][k] + qy[b][k] * qy[b][k];
    }
#pragma unroll
    for (int k = 0; k < R; ++k) acc[k] = fma((double)pv[k].x * pv[k].x + (double)pv[k].y * pv[k].y, q2[k], acc[k]);
  }
  e_fence();
  double* red = e_lds + wave * per_wave;
#pragma unroll
  for (int k = 0; k < R; ++k) red[k * 64 + lane] = acc[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = Np * (s0 + jl * R + k) + phi;
    if (k % W == wave && on && i < A.Nx) {
      double s = A.add ? E[(size_t)row * A.Nx + i] : 0.0;
      for (int v = 0; v < W; ++v) s += e_lds[v * per_wave + k * 64 + lane];
      E[(size_t)row * A.Nx + i] = s;
    }
  }
}

// ------------------------------------------------------ energies under TGC
// E[p] = sum over the mixes and rows i of |sum_j k[i - j] Phi[j, p]|^2, Phi[j, p]
// = p_inc[j, p] sum_a pref[j, a] h_ref[j, shift(p, e_a)] (operator_born.m:830-848,
// convolution.m:62-98).  On regular plans the convolution along the N
// frequencies is a product of transforms of length L >= N + M (M the longest
// half length), or of length L = 2 (N - 1) with the one lag pair +-(N - 1),
// which would fall on one entry, taken separately.  A wave takes FPW
// neighbouring points and the mixes mk0 + wave, + 4, ...: Phi in FP64,
// rounded once, the transforms in FP32, the squares summed in FP64.
//
// Bound: the vector ALU, about 980 instructions per FPW points and mix in
// place of the N (2 M + 1) products of k_energy_rx_tgc, which stays for the
// other plans and longer mixes.  64 elements, 192 x 192 points, 65 frequencies,
// M = 64: 8.7 ms per measurement there, 0.54 ms here; relative L2 error against
// FP64 5.4e-8 there (the taps' rounding), 2.8e-8 here (1.1e-7 without the
// remainders of the transforms' constants and spectra, 4 % each, and twiddles of
// magnitude 1; another 96 x 12 points: 1.4e-8 with 65 and 1.3e-8 with 100 frequencies,
// 1.7e-8 and 2.3e-8 there).

// spec[mk][2][8][TL][2]: transform of the taps of mix mk (lags over L / 2 left
// out), divided by L, and what its rounding to FP32 leaves
template <int TL>
__global__ __launch_bounds__(64) void k_tgc_spectra(const double2* __restrict__ taps, const int* __restrict__ half,
                                                    const int64_t* __restrict__ tap_off, int N_mk,
                                                    float4* __restrict__ spec) {
  constexpr int FPW = FftShape<TL>::FPW, L = 16 * TL;
  __shared__ Cx<double> lds[FftShape<TL>::LDS];
  const int lane = threadIdx.x, j = lane / FPW, g = lane % FPW;
  const int mk = blockIdx.x * FPW + g;
  Cx<double> tw[16], x[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    double s, c;
    sincospi(2.0 * (double)(j * k) / L, &s, &c);
    tw[k] = {c, s};
  }
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    x[q] = {0.0, 0.0};
    const int n = j + TL * q, d = n < L / 2 ? n : n - L;
    if (mk < N_mk && n != L / 2 && d >= -half[mk] && d <= half[mk]) {
      const double2 k = taps[tap_off[mk] + half[mk] + d];
      x[q] = {k.x / L, k.y / L};
    }
  }
  fft_wave<double, TL, false>(x, tw, lds, lane);
  if (mk >= N_mk) return;
  float4* out = spec + (size_t)mk * L + j;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const float4 k = make_float4((float)x[2 * q].x, (float)x[2 * q].y, (float)x[2 * q + 1].x, (float)x[2 * q + 1].y);
    out[q * TL] = k;
    out[L / 2 + q * TL] = make_float4((float)(x[2 * q].x - k.x), (float)(x[2 * q].y - k.y), (float)(x[2 * q + 1].x - k.z),
                                      (float)(x[2 * q + 1].y - k.w));
  }
}

// NQ: entries of a lane that can hold frequencies (N <= NQ * TL)
template <int TL, int NQ>
__global__ __launch_bounds__(256, 2) void k_energy_tgc_fft(EnergyArgs A, const float4* __restrict__ spec,
                                                           const double2* __restrict__ taps, const int* __restrict__ half,
                                                           const int64_t* __restrict__ tap_off,
                                                           const float2* __restrict__ twid, int mk0, int mk1, int b0,
                                                           double* __restrict__ E) {
  constexpr int FPW = FftShape<TL>::FPW, L = 16 * TL;
  __shared__ cf lds_all[4 * FftShape<TL>::LDS];
  __shared__ double red[4][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int j = lane / FPW, g = lane % FPW;
  cf* lds = lds_all + wave * FftShape<TL>::LDS;
  const int N = A.n_pairs;
  const int p0 = (b0 + (int)blockIdx.x) * FPW + g, p = min(p0, A.N_pts - 1);
  const int row = p / A.Nx, ix = p - row * A.Nx;
  cf tw[16];
  load_twiddles<TL>(twid, j, tw);
  float2 pv[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int n = min(j + TL * q, N - 1);
    pv[q] = A.P[(size_t)(A.pair0 + n) * A.N_pts + p];
  }
  const bool edge = N == L / 2 + 1;   // lags +-(N - 1) separately
  double acc = 0.0;
  for (int mk = mk0 + wave; mk < mk1; mk += 4) {
    const int Na = A.mk_meta[mk * 4 + 2];
    const int* act = A.act + A.mk_off[mk * 4 + 2];
    const double2* pref = A.pref + A.mk_off[mk * 4 + 3];
    double qx[NQ], qy[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) qx[q] = qy[q] = 0.0;
    for (int a = 0; a < Na; ++a) {
      const int e = act[a], ey = e / A.Nex, ex = e - ey * A.Nex;
      const float2* h = A.h + (int64_t)A.hrow[ey * A.n_rows + row] * A.HR + A.ext[ix - ex * A.Np + (A.Nex - 1) * A.Np];
      const double2* c = pref + (int64_t)a * N;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int n = min(j + TL * q, N - 1);
        const float2 hv = h[(int64_t)n * A.H_plane];
        const double2 cv = c[n];
        qx[q] += cv.x * hv.x - cv.y * hv.y;
        qy[q] += cv.x * hv.y + cv.y * hv.x;
      }
    }
    cf x[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      x[q] = {0.f, 0.f};
      if (q < NQ && j + TL * q < N) {
        const int r = q < NQ ? q : 0;
        x[q] = {(float)(qx[r] * pv[r].x - qy[r] * pv[r].y), (float)(qx[r] * pv[r].y + qy[r] * pv[r].x)};
      }
    }
    // with N = L / 2 + 1, lane j = 0 holds the first (q = 0) and the last (q = 8) row
    const cf first = x[0], last = x[8];
    float4 kv[8], kl[8];
    const float4* ks = spec + (size_t)mk * L + j;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      kv[q] = ks[q * TL];
      kl[q] = ks[L / 2 + q * TL];
    }
    fft_wave<float, TL, (NQ <= 8), true>(x, tw, lds, lane);
#pragma unroll
    for (int q = 0; q < 8; ++q) {   // conjugated, for the exponent's sign
      const cf u = x[2 * q], v = x[2 * q + 1];
      x[2 * q] = {fmaf(kv[q].x, u.x, fmaf(kl[q].x, u.x, -fmaf(kv[q].y, u.y, kl[q].y * u.y))),
                  -fmaf(kv[q].x, u.y, fmaf(kl[q].x, u.y, fmaf(kv[q].y, u.x, kl[q].y * u.x)))};
      x[2 * q + 1] = {fmaf(kv[q].z, v.x, fmaf(kl[q].z, v.x, -fmaf(kv[q].w, v.y, kl[q].w * v.y))),
                      -fmaf(kv[q].z, v.y, fmaf(kl[q].z, v.y, fmaf(kv[q].w, v.x, kl[q].w * v.x)))};
    }
    fft_wave<float, TL, false, true>(x, tw, lds, lane);
    if (NQ > 8 && edge && half[mk] == N - 1 && j == 0) {
      const double2* k = taps + tap_off[mk];   // lags -(N - 1) .. N - 1
      const float2 kn = make_float2((float)k[0].x, (float)k[0].y);
      const float2 kp = make_float2((float)k[2 * (N - 1)].x, (float)k[2 * (N - 1)].y);
      cf y0 = {x[0].x, -x[0].y}, y8 = {x[8].x, -x[8].y};
      cmac(y0, cf{kn.x, kn.y}, last);
      cmac(y8, cf{kp.x, kp.y}, first);
      x[0] = y0;
      x[8] = y8;
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      if (j + TL * q < N) acc += (double)x[q].x * x[q].x + (double)x[q].y * x[q].y;
  }
  red[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && j == 0 && p0 < A.N_pts) {
    double s = 0.0;
    for (int w = 0; w < 4; ++w)
      for (int t = 0; t < TL; ++t) s += red[w][t * FPW + g];
    E[p] = s;
  }
}

// ------------------------------------------------------------------ host side
int energy_pad(int Nex) { return (Nex + 23) / 24 * 24; }   // a multiple of 4, 6 and 8

void launch_energy_weights(const Plan& P, double* ew, hipStream_t s) {
  const int Ney = P.nd == 3 ? P.Ney : 1, NeP = energy_pad(P.Nex);
  const size_t n = (size_t)P.N_pairs * Ney * NeP;
  hipLaunchKernelGGL(k_energy_weights, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, P.d_pe_off, P.d_pe_ent,
                     P.d_pref, P.d_obs_mk, P.d_mk_meta, P.N_pairs, P.Nex, Ney, NeP, ew);
}

static EnergyArgs energy_args(const Plan& P, int m, int R) {
  EnergyArgs A;
  A.h = P.d_h;
  A.P = P.d_p;
  A.ext = P.d_ext;
  A.hrow = P.d_hrow;
  A.pair_fg = P.d_pair_fg;
  A.pair0 = P.meas_pair_base[m];
  A.n_pairs = P.meas_Nfm[m];
  A.Nx = P.Nx;
  A.n_rows = P.n_rows;
  A.Np = P.Np;
  A.Nex = P.Nex;
  A.Ney = P.nd == 3 ? P.Ney : 1;
  A.N_ext = P.N_ext;
  A.N_pts = P.N_pts;
  A.HR = P.HR;
  A.NeP = energy_pad(P.Nex);
  A.H_plane = P.H_plane;
  A.LPW = 64 / P.Np;
  const int S = (P.Nx + P.Np - 1) / P.Np;
  A.nseg = (S + A.LPW * R - 1) / (A.LPW * R);
  A.nb = (P.Nex + R - 1) / R;
  A.WLp = e_window(A.LPW, A.nb, R);
  A.ew = P.d_ew;
  A.row_off = P.d_erow_off;
  A.rows = P.d_erows;
  A.mk_meta = P.d_mk_meta;
  A.mk_off = P.d_mk_off;
  A.act = P.d_act;
  A.pref = P.d_pref;
  A.add = 0;
  return A;
}

// Whether the fast kernels' lanes and windows cover the plan: up to 64 points
// per pitch, and a window of 4 points per lane within one wave's share of LDS.
// Their windows meet padding weights of 0 past the elements, which a table
// entry that is not finite would carry to points that do not see it.
bool energy_fast(const Plan& P) { return P.structured && P.Np <= 64 && !P.h_odd; }

// f(R, MI) of the single-element kernel that a plan takes.  R = 4, 6 or 8 points
// per lane: the fewest points computed past the row's end, then the largest (one
// LDS read per R multiply-adds).
template <int R, typename F>
static void with_single_entries(const EnergyArgs& A, F&& f) {
  const int mi = (A.Np * (A.LPW + A.nb) * R + 63) / 64;
  using I = std::integral_constant<int, R>;
  if (R < 8 && mi <= 8) f(I(), std::integral_constant<int, (R < 8 ? 8 : 12)>());   // (8 points per lane have more)
  else if (mi <= 12) f(I(), std::integral_constant<int, 12>());
  else if (mi <= 16) f(I(), std::integral_constant<int, 16>());
  else f(I(), std::integral_constant<int, 0>());
}
static EnergyArgs single_args(const Plan& P, int m, int R) {
  EnergyArgs A = energy_args(P, m, R);
  A.nb += A.nb & 1;
  A.WLp = e_window(A.LPW, A.nb, R);
  return A;
}
static size_t single_lds(const EnergyArgs& A, int R) { return ((size_t)A.Np * A.WLp + A.nb * R + 1) * sizeof(double); }
template <typename F>
static void with_single_kernel(const Plan& P, int m, F&& f) {
  const int LPW = 64 / P.Np, S = (P.Nx + P.Np - 1) / P.Np;
  auto pad = [&](int R) { return (S + LPW * R - 1) / (LPW * R) * LPW * R; };
  auto run = [&](auto R) {
    const EnergyArgs A = single_args(P, m, R());
    with_single_entries<R()>(A, [&](auto, auto MI) { f(A, R, MI); });
  };
  if (pad(8) <= pad(6) && pad(8) <= pad(4)) run(std::integral_constant<int, 8>());
  else if (pad(6) <= pad(4)) run(std::integral_constant<int, 6>());
  else run(std::integral_constant<int, 4>());
}

// Waves per workgroup of the single-element kernel: 8 while the compute units
// hold all workgroups at once (one each, two of the smallest kernels), else 4,
// of which two share a compute unit.  One measurement of 128 elements, rows of
// 384 points, 65 frequencies: 256 rows 61 us with 4 waves and 53 with 8, 272 rows
// 89 and 96, 384 rows 90 and 100; rows of 250 points (4 points per lane), 64
// elements, 300 rows: 43 and 38.
int energy_single_waves(const Plan& P) {
  int W = 4;
  with_single_kernel(P, 0, [&](const EnergyArgs& A, auto R, auto MI) {
    const size_t per_wave = single_lds(A, R());
    const void* fn = (const void*)k_energy_single<R(), MI()>;
    int at_once = 0;
    if (8 * per_wave <= 150 * 1024 &&
        hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess &&
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&at_once, fn, 512, 8 * per_wave) == hipSuccess &&
        (int64_t)A.n_rows * A.nseg <= (int64_t)at_once * P.n_cu)
      W = 8;
    while (W > 1 && W * per_wave > 150 * 1024) W /= 2;
  });
  return W;
}

void launch_energy_single(const Plan& P, int m, double* E, hipStream_t s) {
  with_single_kernel(P, m, [&](const EnergyArgs& A, auto R, auto MI) {
    hipFuncSetAttribute((const void*)k_energy_single<R(), MI()>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    hipLaunchKernelGGL((k_energy_single<R(), MI()>), dim3(A.n_rows * A.nseg), dim3(64 * P.e_waves),
                       P.e_waves * single_lds(A, R()), s, A, E);
  });
}

void launch_energy_multi(const Plan& P, int m, bool add, double* E, hipStream_t s) {
  constexpr int R = 4, KB = 4;
  EnergyArgs A = energy_args(P, m, R);
  A.add = add;
  const int wgs = A.n_rows * A.nseg;
  const size_t per_wave = ((size_t)A.Np * A.WLp + (size_t)A.nb * R * KB * 2) * sizeof(double);
  int W = 4;   // (the kernel's launch bound; fewer where LDS does not hold them)
  while (W > 1 && W * per_wave > 150 * 1024) W /= 2;
  const size_t lds = W * per_wave;
#define BORN_EM(NPv)                                                                                                      \
  do {                                                                                                                    \
    hipFuncSetAttribute((const void*)k_energy_multi<R, NPv, KB>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); \
    hipLaunchKernelGGL((k_energy_multi<R, NPv, KB>), dim3(wgs), dim3(64 * W), lds, s, A, E);                             \
  } while (0)
  if (P.Np == 4) BORN_EM(4);
  else if (P.Np == 2) BORN_EM(2);
  else BORN_EM(0);
#undef BORN_EM
}

// Transform length (as TL = L / 16) of the energies under TGC: the smallest
// that holds N rows and half lengths up to M; 0: none.
int energy_tgc_length(int N, int M) {
  for (int TL = 4; TL <= 16; TL *= 2) {
    const int L = 16 * TL;
    if (N + M <= L || (N == L / 2 + 1 && M == N - 1)) return TL;
  }
  return 0;
}

void launch_tgc_spectra(const Plan& P, int TL, float2* spec, hipStream_t s) {
  const int FPW = 64 / TL;
  const dim3 grid((P.N_mk + FPW - 1) / FPW);
#define BORN_TS(TLv)                                                                                                \
  hipLaunchKernelGGL(k_tgc_spectra<TLv>, grid, dim3(64), 0, s, P.d_tgc_k64, P.d_tgc_half, P.d_tgc_off, P.N_mk, \
                     (float4*)spec)
  if (TL == 16) BORN_TS(16);
  else if (TL == 8) BORN_TS(8);
  else BORN_TS(4);
#undef BORN_TS
}

void launch_energy_tgc_fft(const Plan& P, int m, double* E, hipStream_t s) {
  int mk0 = 0;
  while (mk0 < P.N_mk && P.mk_meas[mk0] != m) ++mk0;
  int mk1 = mk0;
  while (mk1 < P.N_mk && P.mk_meas[mk1] == m) ++mk1;
  const EnergyArgs A = energy_args(P, m, 4);
  const int TL = P.tgc_TL, FPW = 64 / TL, N = P.N_fu;
  const int blocks = (int)(((int64_t)P.N_pts + FPW - 1) / FPW), at_once = (1 << 24) - 1;   // (a launch holds less than 2^32 threads)
#define BORN_ET(TLv, NQv)                                                                                  \
  hipLaunchKernelGGL((k_energy_tgc_fft<TLv, NQv>), grid, dim3(256), 0, s, A, (const float4*)P.d_tgc_spec, \
                     P.d_tgc_k64, P.d_tgc_half, P.d_tgc_off, P.d_tgc_tw, mk0, mk1, b0, E)
#define BORN_ETN(TLv)                  \
  do {                                 \
    if (N <= 4 * TLv) BORN_ET(TLv, 4); \
    else if (N <= 8 * TLv) BORN_ET(TLv, 8); \
    else if (N <= 9 * TLv) BORN_ET(TLv, 9); \
    else BORN_ET(TLv, 16);             \
  } while (0)
  for (int b0 = 0; b0 < blocks; b0 += at_once) {
    const dim3 grid(std::min(at_once, blocks - b0));
    if (TL == 16) BORN_ETN(16);
    else if (TL == 8) BORN_ETN(8);
    else BORN_ETN(4);
  }
#undef BORN_ETN
#undef BORN_ET
}

}  // namespace born
