// 3-D contractions by fast lateral correlation in x and y (gfx950).
//
// As born_fft.hip, on planes: with grid point (i_x, i_y) = (Npx s_x + phi_x,
// Npy s_y + phi_y) and the depth plane of h_ref in its Npx Npy phases, element
// (e_x, e_y) meets point s of a phase at m = s + t, t = (N_ex - 1 - e_x,
// N_ey - 1 - e_y), and one (frequency, depth, phase) is a two-dimensional
// correlation: a product of transforms of length Lx x Ly with
// S_x + N_ex - 1 <= Lx, S_y + N_ey - 1 <= Ly (64 or 128 each).
//
// A workgroup of W waves transforms a plane in two steps, the x transforms of
// the rows (slot = (s_y, phi_x), phi_x fastest) and the y transforms of the
// columns k_x, through a plane [slot][Lx + 1] in LDS; px phases phi_x go
// through together, one phi_y at a time.  The y transforms of a phase leave
// entry (k_x, k_y) at the same lane and register for every phase,
// k_x = (pass W + wave) FPWY + g, k_y = j + TLY q, so that the forward sums
// its products over phases and depths in registers and transforms back once;
// the adjoint starts from there.
//
// Bound: the vector ALU, per plane of 64 x 64 points at 2 points per pitch
// 384 transforms of 64 points (about 7400 wave instructions) in place of
// 32 x 32 x 64 x 64 complex multiply-adds, at 60-65 % of its rate with two waves
// per SIMD (registers and LDS) and two barriers per tile.  32 x 32 elements,
// 64^3 points, 33 frequencies, 3 waves, 4 right-hand sides: forward 0.67 ms,
// adjoint 0.58 ms against 5.6 and 7.0 ms of the split BF16 products (128 x 128 x
// 192 points, 65 frequencies, 5 waves, one: 8.4 and 8.1 ms).  What the loads
// ahead, the twiddles in LDS and 64-bit LDS accesses gave: 0.72 and 0.62 ms
// before, 242 -> 180 and 231 -> 180 us at 20 x 8 elements, 33 x 70 x 60 points,
// 20 frequencies, 3 waves, and 12.9 -> 8.4 ms for the forward of the large one.
#include "born_fft.h"
#include "born_internal.h"

#include <algorithm>

namespace born {

template <int TLX, int TLY>
struct Fft3Shape {
  static constexpr int W = TLX == 4 && TLY == 4 ? 4 : 8;          // waves
  static constexpr int FPWX = 64 / TLX, FPWY = 64 / TLY;
  static constexpr int LX = 16 * TLX, LY = 16 * TLY;
  static constexpr int NBP = LX / (W * FPWY);                     // y passes per phase
  static constexpr int EX = FftShape<TLX>::LDS > FftShape<TLY>::LDS ? FftShape<TLX>::LDS : FftShape<TLY>::LDS;
  static constexpr int ROW = LX + 1;                              // odd: rows on all banks
};

// ------------------------------------------------------------------ spectra
// x transforms (FP64) of the rows m_y of every phase, divided by Lx Ly, one
// frequency: tmp[z][phi_y][phi_x][m_y][k_x].
template <int TLX>
__global__ __launch_bounds__(64) void k_fft3_table_x(const float2* __restrict__ h, const int* __restrict__ ext,
                                                     const int* __restrict__ exty, int HR, int HY, int N_ext, int N_exty,
                                                     int Npx, int Npy, int Ly, int64_t n_rows,
                                                     const float* __restrict__ delta, double2* __restrict__ tmp) {
  constexpr int FPW = FftShape<TLX>::FPW, L = 16 * TLX;
  __shared__ Cx<double> lds[FftShape<TLX>::LDS];
  const int lane = threadIdx.x, j = lane / FPW, g = lane % FPW;
  Cx<double> tw[16], x[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    double s, c;
    sincospi(2.0 * (double)(j * k) / L, &s, &c);
    tw[k] = {c, s};
  }
  const int64_t row = (int64_t)blockIdx.x * FPW + g;
  const bool on = row < n_rows;
  const int my = (int)(row % Ly);
  int64_t t = row / Ly;
  const int phx = (int)(t % Npx);
  t /= Npx;
  const int phy = (int)(t % Npy);
  const int64_t z = t / Npy;
  const int ty = Npy * my + phy;
  const bool have = on && ty < N_exty;
  const float2* src = h + (have ? ((int64_t)exty[ty] + HY * z) * HR : 0);
  const double scale = 1.0 / ((double)L * Ly);
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int tx = Npx * (j + TLX * q) + phx;
    x[q] = {0.0, 0.0};
    if (have && tx < N_ext) {
      const float2 v = src[ext[tx]];
      x[q] = {v.x * scale, -v.y * scale};   // conjugated twice for the exponent's sign
    }
  }
  fft_wave<double, TLX, false>(x, tw, lds, lane);
  if (!on) return;
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const double d = 1.0 + delta[j + TLX * q];
    tmp[row * L + j + TLX * q] = make_double2(x[q].x * d, x[q].y * d);
  }
}

// y transforms (FP64): H[(z, phi_y, phi_x)][k_x / FPWY][8][64 lanes][2]
template <int TLY>
__global__ __launch_bounds__(64) void k_fft3_table_y(const double2* __restrict__ tmp, int Lx, int64_t n_cols,
                                                     const float* __restrict__ delta, float2* __restrict__ H) {
  constexpr int FPW = FftShape<TLY>::FPW, L = 16 * TLY;
  __shared__ Cx<double> lds[FftShape<TLY>::LDS];
  const int lane = threadIdx.x, j = lane / FPW, g = lane % FPW;
  Cx<double> tw[16], x[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    double s, c;
    sincospi(2.0 * (double)(j * k) / L, &s, &c);
    tw[k] = {c, s};
  }
  const int64_t col = (int64_t)blockIdx.x * FPW + g;   // (z, phase, k_x); a multiple of FPW columns in all
  if (col >= n_cols) return;
  const int64_t zp = col / Lx, kx = col - zp * Lx;
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const double2 v = tmp[(zp * L + j + TLY * q) * Lx + kx];
    x[q] = {v.x, v.y};
  }
  fft_wave<double, TLY, false>(x, tw, lds, lane);
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const double d = 1.0 + delta[j + TLY * q];
    x[q] = {x[q].x * d, x[q].y * d};
  }
  float4* out = reinterpret_cast<float4*>(H) + (col / FPW) * 512 + lane;
#pragma unroll
  for (int q = 0; q < 8; ++q)
    out[q * 64] = make_float4((float)x[2 * q].x, -(float)x[2 * q].y, (float)x[2 * q + 1].x, -(float)x[2 * q + 1].y);
}

__device__ __forceinline__ int fft3_block(int per) { return (blockIdx.x % XCDS) * per + blockIdx.x / XCDS; }

// ------------------------------------------------------------------ forward
// One workgroup per (depth block, column, right-hand side).  p_inc and the
// input of the next tile's rows are loaded during the last column transforms of
// this one (behind the spectra of these, which return first).
template <int TLX, int TLY, bool HALF>
__global__ __launch_bounds__((64 * Fft3Shape<TLX, TLY>::W), 2) void k_fft3_fwd(Fft3Args A, int n_wg, int per) {
  using S = Fft3Shape<TLX, TLY>;
  constexpr int NQ = HALF ? 8 : 16;
  constexpr bool AHEAD = HALF && S::NBP == 1;   // (the others have no registers left for it)
  extern __shared__ cf f3_lds[];   // exchange buffers, plane, twiddles
  cf* twlx = f3_lds + A.tw_at;
  cf* twly = twlx + 16 * TLX;
  load_twiddles_lds<TLX>(A.twx, twlx);
  load_twiddles_lds<TLY>(A.twy, twly);
  const int wg = fft3_block(per);
  if (wg >= n_wg) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  cf* lds = f3_lds + wave * S::EX;
  cf* plane = f3_lds + S::W * S::EX;
  const int jx = lane / S::FPWX, gx = lane % S::FPWX, jy = lane / S::FPWY, gy = lane % S::FPWY;
  const int r = wg % A.N_rhs, cz = wg / A.N_rhs;
  const int c = cz % A.n_cols, zb = cz / A.n_cols;
  const int2 pf = A.col[c];
  const int z0 = zb * A.ZR, z1 = min(A.Nz, z0 + A.ZR);
  const float2* P = A.P + (size_t)pf.x * A.N_pts;
  const float2* gm = A.gm + (size_t)r * A.N_pts;
  cf G[S::NBP][16];
#pragma unroll
  for (int b = 0; b < S::NBP; ++b)
#pragma unroll
    for (int q = 0; q < 16; ++q) G[b][q] = {0.f, 0.f};
  const int n_tx = A.Npx / A.px, n_slot = A.px * A.Sy, n_tile = A.Npy * n_tx;
  // the rows of slots s0 .. of a tile: whether the lane has one, its first x,
  // and its entries' values (those past the grid read entry 0 of the row)
  struct Row {
    bool ok;
    int phx;
  };
  auto row_of = [&](int tile, int s0) {
    const int phy = tile / n_tx, slot = s0 + gx, sy = slot / A.px;
    return Row{slot < n_slot && A.Npy * sy + phy < A.Ny, (tile - phy * n_tx) * A.px + slot - sy * A.px};
  };
  float2 pv[NQ], gv[NQ];
  auto load = [&](int z, int tile, int s0) {
    const Row R = row_of(tile, s0);
    const int phy = tile / n_tx, sy = (s0 + gx) / A.px;
    const int base = (z * A.Ny + (R.ok ? A.Npy * sy + phy : 0)) * A.Nx;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int ix = A.Npx * (jx + TLX * q) + R.phx;
      const int at = base + (ix < A.Nx ? ix : 0);
      pv[q] = P[at];
      gv[q] = gm[at];
    }
  };
  const int first = wave * S::FPWX;
  if (AHEAD && z0 < z1 && first < n_slot) load(z0, 0, first);
  for (int z = z0; z < z1; ++z) {
    const float4* Hz = reinterpret_cast<const float4*>(A.H) +
                       ((size_t)pf.y * A.Nz + z) * A.Npy * A.Npx * (S::LX * S::LY / 2) + lane;
    for (int tile = 0; tile < n_tile; ++tile) {
      const int phy = tile / n_tx, phx0 = (tile - phy * n_tx) * A.px;
      for (int s0 = first; s0 < n_slot; s0 += S::W * S::FPWX) {
        if (!AHEAD || s0 != first) load(z, tile, s0);
        const Row R = row_of(tile, s0);
        cf x[16];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const bool ok = R.ok && A.Npx * (jx + TLX * q) + R.phx < A.Nx;
          const float2 g = ok ? gv[q] : make_float2(0.f, 0.f);
          x[q] = {fmaf(pv[q].x, g.x, -(pv[q].y * g.y)), fmaf(pv[q].x, g.y, pv[q].y * g.x)};
        }
        fft_wave_l<TLX, NQ>(x, twlx, lds, lane);
        if (s0 + gx < n_slot) {
          cf* row = plane + (s0 + gx) * S::ROW + jx;
#pragma unroll
          for (int q = 0; q < 16; ++q) row[TLX * q] = x[q];
        }
      }
      __syncthreads();
      for (int ph = 0; ph < A.px; ++ph) {
        const float4* Hp = Hz + (size_t)(phy * A.Npx + phx0 + ph) * (S::LX * S::LY / 2);
#pragma unroll
        for (int b = 0; b < S::NBP; ++b) {
          float4 hv[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) hv[q] = Hp[((b * S::W + wave) * 8 + q) * 64];
          __builtin_amdgcn_sched_barrier(0);
          if (AHEAD && ph == A.px - 1 && first < n_slot) {
            const bool last = tile + 1 == n_tile;
            load(last ? min(z + 1, z1 - 1) : z, last ? 0 : tile + 1, first);   // (the last tile loads one again)
          }
          __builtin_amdgcn_sched_barrier(0);
          const int kx = (b * S::W + wave) * S::FPWY + gy;
          cf x[16];
#pragma unroll
          for (int q = 0; q < NQ; ++q) {
            x[q] = {0.f, 0.f};
            const int sy = jy + TLY * q;
            if (sy < A.Sy) x[q] = plane[(sy * A.px + ph) * S::ROW + kx];
          }
          fft_wave_l<TLY, NQ>(x, twly, lds, lane);
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            cmac(G[b][2 * q], cf{hv[q].x, hv[q].y}, x[2 * q]);
            cmac(G[b][2 * q + 1], cf{hv[q].z, hv[q].w}, x[2 * q + 1]);
          }
        }
      }
      __syncthreads();
    }
  }
  // transform back: rows t_y < N_ey, then entries t_x < N_ex
#pragma unroll
  for (int b = 0; b < S::NBP; ++b) {
    fft_wave_l<TLY, 16>(G[b], twly, lds, lane);
    const int kx = (b * S::W + wave) * S::FPWY + gy;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int ty = jy + TLY * q;
      if (ty < A.Ney) plane[ty * S::ROW + kx] = G[b][q];
    }
  }
  __syncthreads();
  float2* out = A.vp + ((size_t)(zb * A.N_rhs + r) * A.n_cols + c) * A.N_e;
  for (int s0 = wave * S::FPWX; s0 < A.Ney; s0 += S::W * S::FPWX) {
    const int ty = s0 + gx;
    cf x[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      x[q] = {0.f, 0.f};
      if (ty < A.Ney) x[q] = plane[ty * S::ROW + jx + TLX * q];
    }
    fft_wave_l<TLX, 16>(x, twlx, lds, lane);
    if (ty < A.Ney) {
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int tx = jx + TLX * q;
        if (tx < A.Nex) out[(A.Ney - 1 - ty) * A.Nex + A.Nex - 1 - tx] = make_float2(x[q].x, x[q].y);
      }
    }
  }
}

// ------------------------------------------------------------------ adjoint
// Spectra of the un-mixed weights (d_W) of one (pair, right-hand side) per
// workgroup: conj(W) at t, wt[row][k_x / FPWY][8][64 lanes][2].
template <int TLX, int TLY>
__global__ __launch_bounds__((64 * Fft3Shape<TLX, TLY>::W)) void k_fft3_weights(Fft3Args A, const float2* __restrict__ Wt,
                                                                             float2* __restrict__ wt) {
  using S = Fft3Shape<TLX, TLY>;
  extern __shared__ cf f3_lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  cf* lds = f3_lds + wave * S::EX;
  cf* plane = f3_lds + S::W * S::EX;
  const int jx = lane / S::FPWX, gx = lane % S::FPWX, jy = lane / S::FPWY, gy = lane % S::FPWY;
  const size_t row = blockIdx.x;   // pair * N_rhs + r
  const size_t pair = row / A.N_rhs, r = row - pair * A.N_rhs;
  const float2* src = Wt + pair * A.N_e * A.N_rhs + r;
  cf tw[16];
  load_twiddles<TLX>(A.twx, jx, tw);
  for (int s0 = wave * S::FPWX; s0 < A.Ney; s0 += S::W * S::FPWX) {
    const int ty = s0 + gx;
    cf x[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int tx = jx + TLX * q;
      x[q] = {0.f, 0.f};
      if (ty < A.Ney && tx < A.Nex) {
        const float2 v = src[(size_t)((A.Ney - 1 - ty) * A.Nex + A.Nex - 1 - tx) * A.N_rhs];
        x[q] = {v.x, -v.y};
      }
    }
    fft_wave<float, TLX, false>(x, tw, lds, lane);
    if (ty < A.Ney) {
#pragma unroll
      for (int q = 0; q < 16; ++q) plane[ty * S::ROW + jx + TLX * q] = x[q];
    }
  }
  __syncthreads();
  load_twiddles<TLY>(A.twy, jy, tw);
  for (int b = 0; b < S::NBP; ++b) {
    const int kx = (b * S::W + wave) * S::FPWY + gy;
    cf x[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int ty = jy + TLY * q;
      x[q] = {0.f, 0.f};
      if (ty < A.Ney) x[q] = plane[ty * S::ROW + kx];
    }
    fft_wave<float, TLY, false>(x, tw, lds, lane);
    float4* out = reinterpret_cast<float4*>(wt) + row * (S::LX * S::LY / 2) + (size_t)(b * S::W + wave) * 512 + lane;
#pragma unroll
    for (int q = 0; q < 8; ++q) out[q * 64] = make_float4(x[2 * q].x, x[2 * q].y, x[2 * q + 1].x, x[2 * q + 1].y);
  }
}

// One workgroup per (column group, depth, phase tile, right-hand side); it
// sums its columns' products with p_inc in registers.
template <int TLX, int TLY, bool HALF>
__global__ __launch_bounds__((64 * Fft3Shape<TLX, TLY>::W), 2) void k_fft3_adj(Fft3Args A, float2* __restrict__ g_out,
                                                                            int n_wg, int per) {
  using S = Fft3Shape<TLX, TLY>;
  constexpr int NQ = HALF ? 8 : 16;
  constexpr bool AHEAD = HALF && S::NBP == 1;   // (the others have no registers left for it)
  extern __shared__ cf f3_lds[];   // exchange buffers, plane, twiddles
  cf* twlx = f3_lds + A.tw_at;
  cf* twly = twlx + 16 * TLX;
  load_twiddles_lds<TLX>(A.twx, twlx);
  load_twiddles_lds<TLY>(A.twy, twly);
  int t = fft3_block(per);
  if (t >= n_wg) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  cf* lds = f3_lds + wave * S::EX;
  cf* plane = f3_lds + S::W * S::EX;
  const int jx = lane / S::FPWX, gx = lane % S::FPWX, jy = lane / S::FPWY, gy = lane % S::FPWY;
  const int n_tx = A.Npx / A.px, n_tile = A.Npy * n_tx, n_slot = A.px * A.Sy;
  const int r = t % A.N_rhs;
  t /= A.N_rhs;
  const int tile = t % n_tile;
  t /= n_tile;
  const int z = t % A.Nz, fgr = t / A.Nz;
  const int c0 = (int)((long)A.n_cols * fgr / A.FG), c1 = (int)((long)A.n_cols * (fgr + 1) / A.FG);
  const int phy = tile / n_tx, phx0 = (tile - phy * n_tx) * A.px;
  const int Syp = (A.Ny - phy + A.Npy - 1) / A.Npy;
  cf acc[FFT3_PASSES][NQ];
#pragma unroll
  for (int a = 0; a < FFT3_PASSES; ++a)
#pragma unroll
    for (int q = 0; q < NQ; ++q) acc[a][q] = {0.f, 0.f};
  // Spectra of H and of the weights, [b][8]: with one pass per phase (AHEAD) those
  // of the next phase or column are loaded during this one's transforms.
  float4 hv[8], wv[8];
  auto load_h = [&](int2 pf, int ph, int b) {
    const float4* Hp = reinterpret_cast<const float4*>(A.H) + lane +
                       ((((size_t)pf.y * A.Nz + z) * A.Npy + phy) * A.Npx + phx0 + ph) * (S::LX * S::LY / 2);
#pragma unroll
    for (int q = 0; q < 8; ++q) hv[q] = Hp[((b * S::W + wave) * 8 + q) * 64];
  };
  auto load_w = [&](int2 pf, int b) {
    const float4* Wp = reinterpret_cast<const float4*>(A.wt) + ((size_t)pf.x * A.N_rhs + r) * (S::LX * S::LY / 2) + lane;
#pragma unroll
    for (int q = 0; q < 8; ++q) wv[q] = Wp[((b * S::W + wave) * 8 + q) * 64];
  };
  int2 pf_next = A.col[min(c0, A.n_cols - 1)];
  if (AHEAD && c0 < c1) {
    load_h(pf_next, 0, 0);
    load_w(pf_next, 0);
  }
  for (int c = c0; c < c1; ++c) {
    const int2 pf = pf_next;
    pf_next = A.col[min(c + 1, c1 - 1)];
    for (int ph = 0; ph < A.px; ++ph) {
#pragma unroll
      for (int b = 0; b < S::NBP; ++b) {
        const int kx = (b * S::W + wave) * S::FPWY + gy;
        if (!AHEAD) {
          load_h(pf, ph, b);
          load_w(pf, b);
        }
        cf x[16];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const float4 h = hv[q], w = wv[q];
          x[2 * q] = {fmaf(h.x, w.x, -(h.y * w.y)), fmaf(h.x, w.y, h.y * w.x)};
          x[2 * q + 1] = {fmaf(h.z, w.z, -(h.w * w.w)), fmaf(h.z, w.w, h.w * w.z)};
        }
        if (AHEAD) {
          __builtin_amdgcn_sched_barrier(0);
          if (ph + 1 < A.px) {
            load_h(pf, ph + 1, 0);
          } else {   // (the last column's again)
            load_h(pf_next, 0, 0);
            load_w(pf_next, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        fft_wave_l<TLY, 16>(x, twly, lds, lane);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const int sy = jy + TLY * q;
          if (sy < A.Sy) plane[(sy * A.px + ph) * S::ROW + kx] = x[q];
        }
      }
    }
    __syncthreads();
    const float2* P = A.P + (size_t)pf.x * A.N_pts;
#pragma unroll
    for (int a = 0; a < FFT3_PASSES; ++a) {
      const int slot = (a * S::W + wave) * S::FPWX + gx;
      if ((a * S::W + wave) * S::FPWX < n_slot) {
        const int sy = slot / A.px, phx = phx0 + slot - sy * A.px;
        const bool row_ok = slot < n_slot && sy < Syp;
        const int base = (z * A.Ny + (row_ok ? A.Npy * sy + phy : 0)) * A.Nx;
        float2 pv[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
          const int ix = A.Npx * (jx + TLX * q) + phx;
          pv[q] = P[base + (row_ok && ix < A.Nx ? ix : 0)];
        }
        cf x[16];
        const cf* src = plane + (slot < n_slot ? slot : 0) * S::ROW + jx;
#pragma unroll
        for (int q = 0; q < 16; ++q) x[q] = src[TLX * q];
        fft_wave_l<TLX, 16>(x, twlx, lds, lane);
#pragma unroll
        for (int q = 0; q < NQ; ++q) cmac(acc[a][q], cf{pv[q].x, pv[q].y}, x[q]);
      }
    }
    __syncthreads();
  }
  float2* out = (A.FG > 1 ? A.gp + (size_t)fgr * A.N_rhs * A.N_pts : g_out) + (size_t)r * A.N_pts;
#pragma unroll
  for (int a = 0; a < FFT3_PASSES; ++a) {
    const int slot = (a * S::W + wave) * S::FPWX + gx;
    const int sy = slot / A.px, phx = phx0 + slot - sy * A.px;
    if (slot < n_slot && sy < Syp) {
      float2* o = out + (size_t)(z * A.Ny + A.Npy * sy + phy) * A.Nx;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int ix = A.Npx * (jx + TLX * q) + phx;
        if (ix < A.Nx) o[ix] = make_float2(acc[a][q].x, -acc[a][q].y);
      }
    }
  }
}

// ------------------------------------------------------------------ host side
#define BORN_FFT3_SHAPE(F, ...)                                       \
  do {                                                                \
    if (F.TLX == 4 && F.TLY == 4) { __VA_ARGS__(4, 4) }               \
    else if (F.TLX == 8 && F.TLY == 4) { __VA_ARGS__(8, 4) }          \
    else if (F.TLX == 4 && F.TLY == 8) { __VA_ARGS__(4, 8) }          \
    else { __VA_ARGS__(8, 8) }                                        \
  } while (0)

// Lengths, phases per tile and LDS of a plan; TLX = 0 where the planes do not
// fit (a workgroup's plane and exchange buffers within 152 KB, FFT3_PASSES
// rounds of row transforms): those plans keep the direct kernels.
Fft3Choice fft3_shape(int Nx, int Ny, int Npx, int Npy, int Nex, int Ney) {
  Fft3Choice c;
  c.Sx = (Nx + Npx - 1) / Npx;
  c.Sy = (Ny + Npy - 1) / Npy;
  auto len = [](int n) { return n <= 64 ? 4 : (n <= 128 ? 8 : 0); };
  const int TLX = len(c.Sx + Nex - 1), TLY = len(c.Sy + Ney - 1);
  if (TLX == 0 || TLY == 0) return c;
  const int W = TLX == 4 && TLY == 4 ? 4 : 8, slots = W * (64 / TLX);
  const int ex = std::max(16 * (64 + 64 / TLX), 16 * (64 + 64 / TLY));
  c.half = c.Sx <= 8 * TLX && c.Sy <= 8 * TLY;
  for (int px = Npx; px >= 1; --px) {
    if (Npx % px != 0) continue;
    c.tw_at = W * ex + std::max(px * c.Sy, Ney) * (16 * TLX + 1);
    const size_t lds = ((size_t)c.tw_at + 16 * (TLX + TLY)) * sizeof(float2);
    // several phases at once only while they fill no more than one round of
    // row transforms (and two workgroups share a compute unit)
    if (px > 1 && (px * c.Sy > slots || lds > 80 * 1024)) continue;
    if (px * c.Sy > FFT3_PASSES * slots || lds > 152 * 1024) continue;
    c.TLX = TLX;
    c.TLY = TLY;
    c.px = px;
    c.lds = lds;
    return c;
  }
  return c;
}

static Fft3Args fft3_args(const Plan& P, int N_rhs) {
  const Plan::Fft& F = P.fft;
  Fft3Args A;
  A.H = F.d_H;
  A.P = P.d_p;
  A.gm = P.d_gm;
  A.col = F.d_col;
  A.wt = F.d_wt;
  A.vp = F.d_vp;
  A.gp = F.d_gp;
  A.twx = F.d_tw;
  A.twy = F.d_tw + F.s3.TLX * 16;
  A.Nx = P.Nx;
  A.Ny = P.Ny;
  A.Nz = P.Nz;
  A.Npx = P.Np;
  A.Npy = P.Npy;
  A.Nex = P.Nex;
  A.Ney = P.Ney;
  A.N_e = P.N_e;
  A.N_pts = P.N_pts;
  A.n_cols = P.N_pairs;
  A.N_rhs = N_rhs;
  A.Sy = F.s3.Sy;
  A.px = F.s3.px;
  A.tw_at = F.s3.tw_at;
  A.ZR = F.ZR;
  A.FG = F.FG;
  return A;
}

// Spectra of one frequency through `tmp` (fft3_tmp entries).
size_t fft3_plane(const Fft3Choice& c) { return (size_t)256 * c.TLX * c.TLY; }
size_t fft3_tmp(const Plan& P) { return (size_t)P.Nz * P.Npy * P.Np * fft3_plane(P.fft.s3); }
void launch_fft3_table(const Plan& P, int f, double2* tmp, hipStream_t s) {
  const Fft3Choice& c = P.fft.s3;
  const int Lx = 16 * c.TLX, Ly = 16 * c.TLY;
  const int64_t planes = (int64_t)P.Nz * P.Npy * P.Np;
  const float2* h = P.d_h + (size_t)f * P.H_plane;
  float2* H = P.fft.d_H + (size_t)f * planes * Lx * Ly;
  const int fx = 64 / c.TLX, fy = 64 / c.TLY;
  const float* delta = reinterpret_cast<const float*>(P.fft.d_tw + Lx + Ly);   // behind the twiddles of both axes
#define BORN_T3X(T)                                                                                                    \
  hipLaunchKernelGGL(k_fft3_table_x<T>, dim3((unsigned)(planes * Ly / fx)), dim3(64), 0, s, h, P.d_ext, P.d_exty, P.HR, \
                     P.HY, P.N_ext, (int)P.exty.size(), P.Np, P.Npy, Ly, planes* Ly, delta, tmp)
#define BORN_T3Y(T) \
  hipLaunchKernelGGL(k_fft3_table_y<T>, dim3((unsigned)(planes * Lx / fy)), dim3(64), 0, s, tmp, Lx, planes* Lx,   \
                     delta + Lx, H)
  if (c.TLX == 4) BORN_T3X(4);
  else BORN_T3X(8);
  if (c.TLY == 4) BORN_T3Y(4);
  else BORN_T3Y(8);
#undef BORN_T3X
#undef BORN_T3Y
}

void launch_fft3_fwd(const Plan& P, int N_rhs, hipStream_t s) {
  const Fft3Choice& c = P.fft.s3;
  const Fft3Args A = fft3_args(P, N_rhs);
  const int n_wg = P.N_pairs * N_rhs * P.fft.NZB, per = (n_wg + XCDS - 1) / XCDS;
#define BORN_F3H(X, Y, HF)                                                                                          \
  do {                                                                                                              \
    hipFuncSetAttribute((const void*)k_fft3_fwd<X, Y, HF>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); \
    hipLaunchKernelGGL((k_fft3_fwd<X, Y, HF>), dim3(per * XCDS), dim3(64 * Fft3Shape<X, Y>::W), c.lds, s, A, n_wg,  \
                       per);                                                                                        \
  } while (0);
#define BORN_F3(X, Y) if (c.half) BORN_F3H(X, Y, true) else BORN_F3H(X, Y, false)
  BORN_FFT3_SHAPE(c, BORN_F3);
#undef BORN_F3
#undef BORN_F3H
}

// d_W (un-mixed weights [pair][e][rhs]) -> spectra
void launch_fft3_weights(const Plan& P, int N_rhs, hipStream_t s) {
  const Fft3Choice& c = P.fft.s3;
  const Fft3Args A = fft3_args(P, N_rhs);
  const dim3 grid((unsigned)((size_t)P.N_pairs * N_rhs));
#define BORN_W3(X, Y)                                                                                               \
  hipFuncSetAttribute((const void*)k_fft3_weights<X, Y>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);   \
  hipLaunchKernelGGL((k_fft3_weights<X, Y>), grid, dim3(64 * Fft3Shape<X, Y>::W), c.lds, s, A, P.d_W, P.fft.d_wt);
  BORN_FFT3_SHAPE(c, BORN_W3);
#undef BORN_W3
}

void launch_fft3_adj(const Plan& P, int N_rhs, float2* g, hipStream_t s) {
  const Fft3Choice& c = P.fft.s3;
  const Fft3Args A = fft3_args(P, N_rhs);
  const int n_wg = P.fft.FG * P.Nz * P.Npy * (P.Np / c.px) * N_rhs, per = (n_wg + XCDS - 1) / XCDS;
#define BORN_A3H(X, Y, HF)                                                                                          \
  do {                                                                                                              \
    hipFuncSetAttribute((const void*)k_fft3_adj<X, Y, HF>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); \
    hipLaunchKernelGGL((k_fft3_adj<X, Y, HF>), dim3(per * XCDS), dim3(64 * Fft3Shape<X, Y>::W), c.lds, s, A, g,     \
                       n_wg, per);                                                                                  \
  } while (0);
#define BORN_A3(X, Y) if (c.half) BORN_A3H(X, Y, true) else BORN_A3H(X, Y, false)
  BORN_FFT3_SHAPE(c, BORN_A3);
#undef BORN_A3
#undef BORN_A3H
}

}  // namespace born
