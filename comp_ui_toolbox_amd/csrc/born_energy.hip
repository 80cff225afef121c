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
// mixes: 22.4 ms per measurement there, 0.35 ms here (FP64 rate: 0.06 ms; the
// fill of the windows takes as long as the multiply-adds).
#include "born_internal.h"

#include <algorithm>

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

template <int R, int NP>
__global__ __launch_bounds__(1024) void k_energy_single(EnergyArgs A, double* __restrict__ E) {
  extern __shared__ double e_lds[];
  const int Np = NP > 0 ? NP : A.Np;
  const int W = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int row = blockIdx.x / A.nseg, seg = blockIdx.x - row * A.nseg;
  const int jl = lane / Np, phi = lane - jl * Np;
  const bool on = jl < A.LPW;
  const int s0 = seg * A.LPW * R;
  double* win = e_lds + (size_t)wave * Np * A.WLp;
  const double* mine = win + phi * A.WLp + (on ? jl : 0) * (R + 1);
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
    double S[R];
#pragma unroll
    for (int k = 0; k < R; ++k) S[k] = 0.0;
    for (int ey = 0; ey < A.Ney; ++ey) {
      e_fence();
      e_fill<R, NP>(A, h + (size_t)A.hrow[ey * A.n_rows + row] * A.HR, s0, lane, win,
                    [](float2 v) { return (double)v.x * v.x + (double)v.y * v.y; });
      e_fence();
      const double* w = A.ew + ((size_t)pair * A.Ney + ey) * A.NeP;
      double a[R], b[R];
#pragma unroll
      for (int i = 0; i < R; ++i) a[i] = mine[i];
      for (int t = 0; t < A.nb; ++t) {
#pragma unroll
        for (int i = 0; i < R; ++i) b[i] = mine[(t + 1) * (R + 1) + i];
#pragma unroll
        for (int d = 0; d < R; ++d) {
          const double wv = w[t * R + d];
#pragma unroll
          for (int k = 0; k < R; ++k) S[k] = fma(wv, k + d < R ? a[k + d] : b[k + d - R], S[k]);
        }
#pragma unroll
        for (int i = 0; i < R; ++i) a[i] = b[i];
      }
    }
#pragma unroll
    for (int k = 0; k < R; ++k) acc[k] = fma((double)pv[k].x * pv[k].x + (double)pv[k].y * pv[k].y, S[k], acc[k]);
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
      for (int v = 0; v < W; ++v) s += e_lds[(size_t)v * Np * A.WLp + k * 64 + lane];
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
bool energy_fast(const Plan& P) { return P.structured && P.Np <= 64; }

// Waves per workgroup: 4, up to 16 while the launch has fewer than 4096 waves.
static int energy_waves(int wgs, size_t lds_per_wave, int most) {
  int W = 4;
  while (W < most && wgs * W < 4096 && 2 * W * lds_per_wave <= 150 * 1024) W *= 2;
  while (W > 1 && W * lds_per_wave > 150 * 1024) W /= 2;
  return W;
}

template <int R>
static void energy_single(const Plan& P, int m, double* E, hipStream_t s) {
  const EnergyArgs A = energy_args(P, m, R);
  const int wgs = A.n_rows * A.nseg;
  const size_t per_wave = (size_t)A.Np * A.WLp * sizeof(double);
  const int W = energy_waves(wgs, per_wave, 16);
  const size_t lds = W * per_wave;
#define BORN_ES(NPv)                                                                                                   \
  do {                                                                                                                 \
    hipFuncSetAttribute((const void*)k_energy_single<R, NPv>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); \
    hipLaunchKernelGGL((k_energy_single<R, NPv>), dim3(wgs), dim3(64 * W), lds, s, A, E);                             \
  } while (0)
  if (P.Np == 4) BORN_ES(4);
  else if (P.Np == 2) BORN_ES(2);
  else BORN_ES(0);
#undef BORN_ES
}

// R = 4, 6 or 8 points per lane: the fewest points computed past the row's
// end, then the largest (one LDS read per R multiply-adds).
void launch_energy_single(const Plan& P, int m, double* E, hipStream_t s) {
  const int LPW = 64 / P.Np, S = (P.Nx + P.Np - 1) / P.Np;
  auto pad = [&](int R) { return (S + LPW * R - 1) / (LPW * R) * LPW * R; };
  if (pad(8) <= pad(6) && pad(8) <= pad(4)) energy_single<8>(P, m, E, s);
  else if (pad(6) <= pad(4)) energy_single<6>(P, m, E, s);
  else energy_single<4>(P, m, E, s);
}

void launch_energy_multi(const Plan& P, int m, bool add, double* E, hipStream_t s) {
  constexpr int R = 4, KB = 4;
  EnergyArgs A = energy_args(P, m, R);
  A.add = add;
  const int wgs = A.n_rows * A.nseg;
  const size_t per_wave = ((size_t)A.Np * A.WLp + (size_t)A.nb * R * KB * 2) * sizeof(double);
  const int W = energy_waves(wgs, per_wave, 4);
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

}  // namespace born
