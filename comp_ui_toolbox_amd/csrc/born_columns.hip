// Columns of A on structured plans (gfx950), FP64 sums.
//
//   u[j][mk, f] = p_inc[pair(m, f)][p_j] sum_a pref[mk][f, a] h_ref[f][entry(p_j, e_a)]
//
// h_ref and p_inc keep grid points fastest, so one point's values over the
// frequencies lie a table plane apart: read once per observation they cost a
// memory line for 8 bytes.  Both kernels here stage a point's values in LDS
// once and then run along the observations, frequency fastest, as they lie in
// the output.  They take regular plans, where every measurement and mix uses
// all frequencies in order (observation = mk * N_f + f).
#include "born_internal.h"

#include <algorithm>

namespace born {

constexpr int COL_NT = 512;   // threads of k_columns_single: 6 waves per SIMD in the LDS of 3 workgroups

struct ColArgs {
  const float2* h;
  const float2* P;
  const int* ext;
  const int* hrow;
  int Nx, n_rows, Np, Nex, N_e, HR, Nf, N_pts;
  int64_t H_plane, N_obs;
  const int* pts;
  int n;
};

__device__ __forceinline__ int64_t col_entry(const ColArgs& A, int p, int e) {
  const int row = p / A.Nx, ix = p - row * A.Nx;
  const int ey = e / A.Nex, ex = e - ey * A.Nex;
  return (int64_t)A.hrow[ey * A.n_rows + row] * A.HR + A.ext[ix - ex * A.Np + (A.Nex - 1) * A.Np];
}

template <typename OutT>
__device__ __forceinline__ OutT col_value(double qx, double qy, float2 p) {
  OutT o;
  o.x = qx * p.x - qy * p.y;
  o.y = qx * p.y + qy * p.x;
  return o;
}

// Mixes of one active element.  A workgroup takes one point, COL_EB elements
// and groups of up to COL_MG measurements: its observations are whole rows of
// N_f outputs, the rows of neighbouring elements adjacent.  Bound: the writes
// of the output and, per output, one prefactor from the L2; scattered points
// also wait on one page of the tables per (pair, point).  256 random points
// at 361,856 observations: 2.39 ms map-driven, 0.33 ms here (0.25 ms with all
// points alike; writing the output alone takes 0.12 ms).
template <typename OutT>
__global__ __launch_bounds__(COL_NT) void k_columns_single(ColArgs A, const int* __restrict__ ent_off,
                                                        const int2* __restrict__ ent, const int64_t* __restrict__ mk_off,
                                                        const double2* __restrict__ pref, int n_eb, int n_mg,
                                                        int n_part, int N_meas, OutT* __restrict__ u) {
  constexpr int COL_TILE = 128, UN = 4, UL = 4;
  extern __shared__ float2 col_lds[];
  __shared__ int4 el_lds[COL_TILE];
  const int Nf = A.Nf, NfP = Nf | 1;
  float2* hl = col_lds;                          // [COL_EB][NfP]
  float2* pl = col_lds + (size_t)COL_EB * NfP;   // [COL_MG][Nf]
  const int b = blockIdx.x;
  const int lb = (b % XCDS) * ((int)gridDim.x / XCDS) + b / XCDS;   // one point's blocks on one die
  if (lb >= n_eb * n_part * A.n) return;
  const int eb = lb % n_eb, t = lb / n_eb;
  const int part = t % n_part, j = t / n_part;
  const int p = A.pts[j];
  const int mg0 = n_mg * part / n_part, mg1 = n_mg * (part + 1) / n_part;
  const int el = threadIdx.x % COL_EB, e = eb * COL_EB + el;
  if (e < A.N_e) {
    const int64_t at = col_entry(A, p, e);
    for (int f = threadIdx.x / COL_EB; f < Nf; f += COL_NT / COL_EB * UL) {
      float2 v[UL];
#pragma unroll
      for (int k = 0; k < UL; ++k) v[k] = A.h[(int64_t)min(f + COL_NT / COL_EB * k, Nf - 1) * A.H_plane + at];
#pragma unroll
      for (int k = 0; k < UL; ++k)
        if (f + COL_NT / COL_EB * k < Nf) hl[el * NfP + f + COL_NT / COL_EB * k] = v[k];
    }
  }
  OutT* out = u + (int64_t)j * A.N_obs;
  for (int mg = mg0; mg < mg1; ++mg) {
    const int i0 = ent_off[eb * n_mg + mg], i1 = ent_off[eb * n_mg + mg + 1];
    const int m0 = mg * COL_MG, nm = min(COL_MG, N_meas - m0);
    __syncthreads();
    for (int i = threadIdx.x; i < nm * Nf; i += COL_NT * UL) {
      float2 v[UL];
#pragma unroll
      for (int k = 0; k < UL; ++k) v[k] = A.P[((size_t)m0 * Nf + min(i + COL_NT * k, nm * Nf - 1)) * A.N_pts + p];
#pragma unroll
      for (int k = 0; k < UL; ++k)
        if (i + COL_NT * k < nm * Nf) pl[i + COL_NT * k] = v[k];
    }
    for (int ib = i0; ib < i1; ib += COL_TILE) {
      const int ne = min(COL_TILE, i1 - ib);
      __syncthreads();
      if ((int)threadIdx.x < ne) {
        const int2 x = ent[ib + threadIdx.x];   // mix, element within the block | measurement within the group << 16
        el_lds[threadIdx.x] = make_int4(x.x, (x.y & 0xffff) * NfP, (x.y >> 16) * Nf, (int)mk_off[x.x * 4 + 3]);
      }
      __syncthreads();
      const int total = ne * Nf;
      const int sr = COL_NT / Nf, sf = COL_NT - sr * Nf;   // a step of COL_NT outputs in (row, frequency)
      int r = (int)threadIdx.x / Nf, fr = (int)threadIdx.x - r * Nf;
      for (int i = threadIdx.x; i < total; i += COL_NT * UN) {
        int4 x[UN];
        int f[UN];
        double2 c[UN];
#pragma unroll
        for (int k = 0; k < UN; ++k) {   // UN prefactors in flight
          f[k] = fr;
          x[k] = el_lds[min(r, ne - 1)];
          c[k] = pref[x[k].w + fr];
          r += sr;
          fr += sf;
          if (fr >= Nf) {
            fr -= Nf;
            ++r;
          }
        }
#pragma unroll
        for (int k = 0; k < UN; ++k) {
          if (i + COL_NT * k >= total) break;
          const float2 hv = hl[x[k].y + f[k]];
          out[(int64_t)x[k].x * Nf + f[k]] = col_value<OutT>(c[k].x * hv.x - c[k].y * hv.y,
                                                             c[k].x * hv.y + c[k].y * hv.x, pl[x[k].z + f[k]]);
        }
      }
    }
  }
}

// Mixes of several active elements.  A workgroup takes JB points, COL_FB
// frequencies and every n_part-th group of 16 mixes; each prefactor it reads
// serves JB points.
template <typename OutT, int JB>
__global__ __launch_bounds__(256) void k_columns_multi(ColArgs A, const int* __restrict__ mks, int n_mk,
                                                       const int* __restrict__ mk_meta, const int64_t* __restrict__ mk_off,
                                                       const int* __restrict__ act, const double2* __restrict__ pref,
                                                       int n_part, OutT* __restrict__ u) {
  extern __shared__ float2 col_lds[];   // [JB][N_e][COL_FB + 1]
  const int Nf = A.Nf;
  const int n_fb = (Nf + COL_FB - 1) / COL_FB;
  int t = blockIdx.x;
  const int part = t % n_part;
  t /= n_part;
  const int jb = t / n_fb, f0 = (t - jb * n_fb) * COL_FB;
  for (int i = threadIdx.x; i < JB * A.N_e; i += 256) {
    const int k = i / A.N_e, e = i - k * A.N_e;
    const int64_t at = col_entry(A, A.pts[min(jb * JB + k, A.n - 1)], e);
    for (int f = 0; f < COL_FB; ++f)
      if (f0 + f < Nf) col_lds[(size_t)i * (COL_FB + 1) + f] = A.h[(int64_t)(f0 + f) * A.H_plane + at];
  }
  __syncthreads();
  const int fl = threadIdx.x % COL_FB, f = f0 + fl;
  if (f >= Nf) return;
  for (int i = part * 16 + threadIdx.x / COL_FB; i < n_mk; i += n_part * 16) {
    const int mk = mks[i];
    const int m = mk_meta[mk * 4 + 0], Na = mk_meta[mk * 4 + 2];
    const int* ac = act + mk_off[mk * 4 + 2];
    const double2* pr = pref + mk_off[mk * 4 + 3] + f;
    double qx[JB], qy[JB];
#pragma unroll
    for (int k = 0; k < JB; ++k) qx[k] = qy[k] = 0.0;
    for (int a = 0; a < Na; ++a) {
      const double2 c = pr[(int64_t)a * Nf];
      const float2* hl = col_lds + (size_t)ac[a] * (COL_FB + 1) + fl;
#pragma unroll
      for (int k = 0; k < JB; ++k) {
        const float2 hv = hl[(size_t)k * A.N_e * (COL_FB + 1)];
        qx[k] += c.x * hv.x - c.y * hv.y;
        qy[k] += c.x * hv.y + c.y * hv.x;
      }
    }
#pragma unroll
    for (int k = 0; k < JB; ++k) {
      const int j = jb * JB + k;
      if (j < A.n)
        u[(int64_t)j * A.N_obs + (int64_t)mk * Nf + f] =
            col_value<OutT>(qx[k], qy[k], A.P[((size_t)m * Nf + f) * A.N_pts + A.pts[j]]);
    }
  }
}

// ------------------------------------------------------------------ host side
// LDS of the two kernels within a compute unit's 160 KB (the first keeps room
// for two workgroups where it can).
static size_t single_lds(int Nf) { return ((size_t)COL_EB * (Nf | 1) + (size_t)COL_MG * Nf) * sizeof(float2); }
static int multi_points(int N_e) {
  for (int JB : {4, 2, 1})
    if ((size_t)JB * N_e * (COL_FB + 1) * sizeof(float2) <= 150 * 1024) return JB;
  return 0;
}
bool columns_fast(const Plan& P) {
  return P.structured && P.regular && (P.col_n_single == 0 || single_lds(P.N_fu) <= 150 * 1024) &&
         (P.col_n_multi == 0 || multi_points(P.N_e) > 0);
}

// Points that one launch takes, in groups of JB with `blocks` workgroups of
// `threads` each: a launch holds less than 2^32 threads.
static int launch_points(int64_t blocks, int threads, int JB) {
  const int64_t groups = std::max<int64_t>(1, ((int64_t)0xffffffff / threads - XCDS) / blocks);
  return (int)std::min<int64_t>(groups, INT32_MAX / JB) * JB;
}

template <typename OutT>
static void launch_fast(const Plan& P, const int* pts, int n, OutT* u, hipStream_t s) {
  ColArgs A;
  A.h = P.d_h;
  A.P = P.d_p;
  A.ext = P.d_ext;
  A.hrow = P.d_hrow;
  A.Nx = P.Nx;
  A.n_rows = P.n_rows;
  A.Np = P.Np;
  A.Nex = P.Nex;
  A.N_e = P.N_e;
  A.HR = P.HR;
  A.Nf = P.N_fu;
  A.N_pts = P.N_pts;
  A.H_plane = P.H_plane;
  A.N_obs = P.N_obs;
  if (P.col_n_single > 0) {
    const int N_meas = (int)P.meas_Nfm.size();
    const int n_eb = (P.N_e + COL_EB - 1) / COL_EB, n_mg = (N_meas + COL_MG - 1) / COL_MG;
    const size_t lds = single_lds(P.N_fu);
    hipFuncSetAttribute((const void*)k_columns_single<OutT>, hipFuncAttributeMaxDynamicSharedMemorySize, 152 * 1024);
    // few points: the measurement groups of a block go to several workgroups
    const int n_part = std::max(1, (int)std::min<int64_t>(n_mg, 1024 / ((int64_t)n * n_eb)));
    const int at_once = launch_points((int64_t)n_eb * n_part, COL_NT, 1);
    for (int64_t j0 = 0; j0 < n; j0 += at_once) {
      A.pts = pts + j0;
      A.n = (int)std::min<int64_t>(at_once, n - j0);
      hipLaunchKernelGGL(k_columns_single<OutT>, dim3((unsigned)(((size_t)A.n * n_eb * n_part + XCDS - 1) / XCDS * XCDS)),
                         dim3(COL_NT), lds, s, A, P.d_col_off, P.d_col_ent, P.d_mk_off, P.d_pref, n_eb, n_mg, n_part,
                         N_meas, u + j0 * P.N_obs);
    }
  }
  if (P.col_n_multi > 0) {
    const int JB = multi_points(P.N_e);
    const int n_fb = (P.N_fu + COL_FB - 1) / COL_FB, n_jb = (n + JB - 1) / JB;
    // parts: enough workgroups for the chip, at least 16 mixes each
    const int n_part = std::max(1, (int)std::min<int64_t>((P.col_n_multi + 15) / 16, 1024 / std::max<int64_t>(1, (int64_t)n_fb * n_jb)));
    const size_t lds = (size_t)JB * P.N_e * (COL_FB + 1) * sizeof(float2);
    const int at_once = launch_points((int64_t)n_fb * n_part, 256, JB);
#define BORN_COL_M(JBv)                                                                                               \
  do {                                                                                                                \
    hipFuncSetAttribute((const void*)k_columns_multi<OutT, JBv>, hipFuncAttributeMaxDynamicSharedMemorySize,          \
                        160 * 1024);                                                                                  \
    hipLaunchKernelGGL((k_columns_multi<OutT, JBv>), grid, dim3(256), lds, s, A, P.d_col_multi, P.col_n_multi,       \
                       P.d_mk_meta, P.d_mk_off, P.d_act, P.d_pref, n_part, u + j0 * P.N_obs);               \
  } while (0)
    for (int64_t j0 = 0; j0 < n; j0 += at_once) {
      A.pts = pts + j0;
      A.n = (int)std::min<int64_t>(at_once, n - j0);
      const dim3 grid((unsigned)((size_t)((A.n + JB - 1) / JB) * n_fb * n_part));
      if (JB == 4) BORN_COL_M(4);
      else if (JB == 2) BORN_COL_M(2);
      else BORN_COL_M(1);
    }
#undef BORN_COL_M
  }
}

void launch_columns_fast(const Plan& P, const int* pts, int n, void* u, bool out_f64, hipStream_t s) {
  if (out_f64) launch_fast(P, pts, n, (double2*)u, s);
  else launch_fast(P, pts, n, (float2*)u, s);
}

}  // namespace born
