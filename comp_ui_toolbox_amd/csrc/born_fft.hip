// 2-D contractions by fast lateral correlation (gfx950).
//
// With grid point i = Np*s + phi and the lateral row H of h_ref in its Np
// phases H_phi[m] = row[ext[Np*m + phi]], element e of the array meets point
// s of phase phi at m = s + t, t = N_e - 1 - e.  So for one (frequency, row,
// phase) both directions are the correlation y[t or s] = sum H[s + t] x[s or t]:
//   forward  V[e]  = sum over rows, phases and s of H[s + t] p_inc[s] gamma[s],
//   adjoint  Y*[s] = sum over t of H[s + t] conj(W[e]),
//            conj(gamma_hat[s]) = sum over frequencies and waves of p_inc[s] Y*[s].
// A correlation over S points and N_e elements with S + N_e - 1 <= L is a
// product of discrete Fourier transforms of length L; longer rows are cut
// into segments.  The spectra of H are kept in a table, the forward sums its
// products over rows and phases in the frequency domain and transforms back
// once, and the adjoint transforms the weights once per (wave, frequency).
// Each (row, wave, frequency) then costs one transform per phase instead of
// the N_e * S products of the direct form.  All arithmetic is FP32; the
// spectra of H are formed in FP64 and stored in FP32.
//
// A wave carries FPW = 64 / TL transforms of length L = 16 * TL (born_fft.h)
// for FPW consecutive slots; slots enumerate (row, segment, phase), phase
// fastest, so that with 4 points per pitch and L = 256 a wave reads 64
// consecutive grid points per load.
//
// Bound: the stream of the p_inc table (7.1 GB per direction at 128 elements,
// 512 x 512 points, 257 frequencies, 11 waves) close to the vector ALU.
// Measured there per call: forward kernel 1.77 ms, adjoint kernel 1.39 ms (5.2
// TB/s, what the memory gives), against 7.2 and 6.8 ms of the direct products
// on FP32 MFMA and 2.4 and 2.6 ms in split BF16; relative L2 error of
// the pair against FP64 2.3e-7 (3.3e-7 and 6.3e-6 there).  Entries of a lane come in counts of
// 4 to 16 (fft_entries), twiddles from LDS: with 8 or 16 entries, branches on
// the slot's length and twiddles in registers the two took 1.79 and 1.54 ms,
// and 264 and 232 instead of 223 and 202 us at 100 elements, 301 x 411 points,
// 2 points per pitch, 7 waves.
#include "born_fft.h"
#include "born_internal.h"

#include <algorithm>
#include <climits>
#include <cmath>

namespace born {

// ------------------------------------------------------------------ spectra
// H[f][slot] (FP64 transform of the FP32 row, conjugated twice for the
// exponent's sign, divided by L and by the transforms' mean gain (fft_gains):
// the inverse transforms of both directions need no other factor, and products
// and sums keep the range of the direct form's).  Layout, that of its readers:
// per group of FPW slots [8][64 lanes][2] entries, so that a lane reads two
// entries at once.
template <int TL>
__global__ __launch_bounds__(64) void k_fft_table(const float2* __restrict__ h, const int* __restrict__ ext,
                                                  const int* __restrict__ hrow, int H_plane, int HR, int N_ext, int Np,
                                                  int nseg, int Sv, int n_slots, int n_ws, const float* __restrict__ delta,
                                                  float2* __restrict__ H) {
  constexpr int FPW = FftShape<TL>::FPW, L = 16 * TL;
  __shared__ Cx<double> lds[FftShape<TL>::LDS];
  const int lane = threadIdx.x, j = lane / FPW, g = lane % FPW;
  const int ws = blockIdx.x, f = blockIdx.y;
  Cx<double> tw[16], x[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    double s, c;
    sincospi(2.0 * (double)(j * k) / L, &s, &c);
    tw[k] = {c, s};
  }
  const int slot = ws * FPW + g;
  const bool ok = slot < n_slots;
  const int phi = slot % Np, rs = slot / Np;
  const int seg = rs % nseg, row = rs / nseg;
  const float2* src = h + (size_t)f * H_plane + (ok ? (size_t)hrow[row] * HR : 0);
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int t = Np * (seg * Sv + j + TL * q) + phi;
    x[q] = {0.0, 0.0};
    if (ok && t < N_ext) {
      const float2 v = src[ext[t]];
      x[q] = {(double)v.x / L, -(double)v.y / L};
    }
  }
  fft_wave<double, TL, false>(x, tw, lds, lane);
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const double d = 1.0 + delta[j + TL * q];
    x[q] = {x[q].x * d, x[q].y * d};
  }
  float4* out = reinterpret_cast<float4*>(H + ((size_t)f * n_ws + ws) * 1024);
#pragma unroll
  for (int q = 0; q < 8; ++q)
    out[q * 64 + lane] = make_float4((float)x[2 * q].x, -(float)x[2 * q].y, (float)x[2 * q + 1].x, -(float)x[2 * q + 1].y);
}

// Whether the lateral rows (2-D) or planes (3-D) of h_ref may be transformed.
// A transform spreads the rounding of the whole sequence over all its outputs,
// where the direct products keep that of an entry to itself.  A field's row has
// its norm in a main lobe of many entries.  One that has it in one (a grid
// point next to an element, entries of another scale) would lose the others.
// *bad gets bit 0 for a row with an entry that is not finite, and bit 1 for one
//   - whose largest entry holds more than a quarter of the row's energy and
//     exceeds the geometric mean of the nonzero entries 16 times (rows of few
//     entries reach the first by themselves): in volumes the entry in front of
//     an element has 1/8 of its plane's energy at half a grid spacing and 1/4 at
//     a third of one, in 2-D it stays below;
//   - one of whose phases, the sequences that are transformed, has more than
//     1/16 of its energy in one entry and more than half of the nonzero ones, 8 at
//     least, 2^32 times below that (a lobe of a few entries in every phase, which
//     holds less of the row).  Sharper rules meet ordinary fields: a receive filter
//     leaves rows of three or four entries close to the array, and where its edge
//     falls on grazing angles (half a wavelength per pitch) all beyond 11 times the
//     depth is 2^32 times below the lobe, which has 1/32 in one entry at 2 mm and
//     1/16 at 1 mm;
//   - whose entries all lie below 2^-100 (spectra divided by the length would
//     become subnormal).
__global__ __launch_bounds__(256) void k_fft_range(const float2* __restrict__ h, const int* __restrict__ ext,
                                                   const int* __restrict__ exty, int N_ext, int ny, int H_plane, int HR,
                                                   int HY, int Nz, int Npx, int Npy, int64_t n_rows,
                                                   int* __restrict__ bad) {
  __shared__ float red[4][4];
  const int tid = threadIdx.x, wave = tid >> 6;
  auto reduce = [&](float& most, float& a, float& b, float& c) {   // a maximum and three sums over the block, in all threads
    __syncthreads();
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      most = fmaxf(most, __shfl_xor(most, m));
      a += __shfl_xor(a, m);
      b += __shfl_xor(b, m);
      c += __shfl_xor(c, m);
    }
    if ((tid & 63) == 0) {
      red[0][wave] = most;
      red[1][wave] = a;
      red[2][wave] = b;
      red[3][wave] = c;
    }
    __syncthreads();
    most = fmaxf(fmaxf(red[0][0], red[0][1]), fmaxf(red[0][2], red[0][3]));
    a = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    b = red[2][0] + red[2][1] + red[2][2] + red[2][3];
    c = red[3][0] + red[3][1] + red[3][2] + red[3][3];
  };
  for (int64_t row = blockIdx.x; row < n_rows; row += gridDim.x) {
    const float2* src = h + (size_t)(row / Nz) * H_plane + (size_t)(row % Nz) * HY * HR;
    auto entry = [&](int i, int n, int px, int py, int sx, int sy) {   // the i-th of a phase with n along x
      if (!exty) return src[ext[px + sx * i]];
      const int ty = i / n;
      return src[(size_t)exty[py + sy * ty] * HR + ext[px + sx * (i - ty * n)]];
    };
    float top = 0.f, odd = 0.f, n1 = 0.f, n2 = 0.f;   // (n1, n2: not used)
    for (int i = tid; i < N_ext * ny; i += 256) {
      const float2 v = entry(i, N_ext, 0, 0, 1, 1);
      if (!(fabsf(v.x) < 1e30f && fabsf(v.y) < 1e30f)) odd = 1.f;   // (NaN among them)
      else top = fmaxf(top, fmaxf(fabsf(v.x), fabsf(v.y)));
    }
    reduce(top, odd, n1, n2);
    if (odd > 0.f) {
      if (tid == 0) atomicOr(bad, 3);
      continue;
    }
    if (top == 0.f) continue;
    if (top < 0x1p-100f) {
      if (tid == 0) atomicOr(bad, 2);
      continue;
    }
    bool uneven = false;
    float peak = 0.f, energy = 0.f, logs = 0.f, count = 0.f;
    const float scale = 1.f / top;
    for (int ph = 0; ph < Npx * Npy; ++ph) {
      const int px = ph % Npx, py = ph / Npx, nx = (N_ext - px + Npx - 1) / Npx, m = nx * ((ny - py + Npy - 1) / Npy);
      float e = 0.f, l = 0.f, n = 0.f, first = 0.f;
      for (int i = tid; i < m; i += 256) {
        const float2 v = entry(i, nx, px, py, Npx, Npy);
        const float x = v.x * scale, y = v.y * scale, q = x * x + y * y;
        first = fmaxf(first, q);
        e += q;
        if (q > 0.f) {
          l += log2f(q);
          n += 1.f;
        }
      }
      reduce(first, e, l, n);
      peak = fmaxf(peak, first);
      if (16.f * first > e) {
        float low = 0.f;
        for (int i = tid; i < m; i += 256) {
          const float2 v = entry(i, nx, px, py, Npx, Npy);
          const float x = v.x * scale, y = v.y * scale, q = x * x + y * y;
          if (q > 0.f && q * 0x1p32f < first) low += 1.f;
        }
        reduce(n1, low, n1, n2);
        if (low >= 8.f && 2.f * low > n) uneven = true;
      }
      energy += e;
      logs += l;
      count += n;
    }
    if (peak > 0.25f * energy && log2f(peak) - logs / count > 8.f) uneven = true;   // (of squares)
    if (uneven && tid == 0) atomicOr(bad, 2);
  }
}

// ------------------------------------------------------------------ forward
// Blocks in logical order: blocks are dispatched round-robin over the XCDS
// dies, so block b takes logical block (b % XCDS) * per + b / XCDS and the
// columns of one frequency, which read the same spectra, run on one die.
__device__ __forceinline__ int logical_block(int per) { return (blockIdx.x % XCDS) * per + blockIdx.x / XCDS; }

__device__ __forceinline__ const FftInst& fft_instance(const FftInst* inst, int n_inst, int wg, bool fwd) {
  int i = 0;
  while (i + 1 < n_inst && wg >= (fwd ? inst[i + 1].wg_f : inst[i + 1].wg_a)) ++i;
  return inst[i];
}

// The masked input (occupancy, cu:466-488: a point takes part iff some
// right-hand side has |Re| or |Im| above DBL_EPSILON) in the order the forward
// reads it: gs[r][group of slots][NZ / 2][64 lanes][2], zero where a lane's
// entry lies past its slot, so that the forward needs no bounds on it.
template <int TL>
__global__ __launch_bounds__(256) void k_fft_gamma(const float2* __restrict__ gm, const int2* __restrict__ slot, int n_ws,
                                                   int NZ, int N_pts, int Np, int N_rhs, int mask,
                                                   float2* __restrict__ gs) {
  constexpr int FPW = FftShape<TL>::FPW;
  const size_t idx = blockIdx.x * (size_t)256 + threadIdx.x;
  if (idx >= (size_t)n_ws * NZ * 64) return;
  const int lane = (int)(idx >> 1) & 63;
  const size_t wq = idx >> 7;
  const int ws = (int)(wq / (NZ / 2)), q = (int)(wq - (size_t)ws * (NZ / 2)) * 2 + (int)(idx & 1);
  const int2 sl = slot[ws * FPW + lane % FPW];
  const int sp = lane / FPW + TL * q;
  bool occ = sp < sl.y;
  const int at = sl.x + (occ ? Np * sp : 0);
  if (occ && mask) {
    occ = false;
    for (int r = 0; r < N_rhs; ++r) {
      const float2 v = gm[(size_t)r * N_pts + at];
      occ |= fabsf(v.x) > 2.220446049250313e-16f || fabsf(v.y) > 2.220446049250313e-16f;
    }
  }
  for (int r = 0; r < N_rhs; ++r)
    gs[(size_t)r * n_ws * NZ * 64 + idx] = occ ? gm[(size_t)r * N_pts + at] : make_float2(0.f, 0.f);
}

// One wave per (slot block, column, right-hand side): column = pair in
// frequency order.  The products with the spectra of H add up in registers
// over the wave's slots; their transform back gives the slot block's partial
// sums of the elements.  NZ: entries of a lane that can hold points, NP:
// points per pitch (0: any).  Lanes read NZ entries of p_inc whether or not
// their slot holds as many (the others meet a zero of gs), with no branch on
// the slot's length: a branch around a load makes the compiler wait for the
// whole batch in front of the transform.  p_inc and the input of the next
// step are in flight during a step, the spectra of a step during the second
// half of its transform.
// Compute alone (p_inc not read) takes 1.22-1.31 ms of the 1.75 ms at the
// size above, the stream of p_inc alone 1.3 ms; measured and no faster: p_inc
// two steps ahead (1.77), two columns per wave (1.79), four waves of a block
// on one column's rows (1.94-2.26), three waves per SIMD with spills.
template <int TL, int NZ, int NP>
__global__ __launch_bounds__(256, 2) void k_fft_fwd(const FftInst* __restrict__ inst, int n_inst,
                                                    const float2* __restrict__ twid, int n_wg, int per) {
  constexpr int FPW = FftShape<TL>::FPW;
  __shared__ cf lds_all[4 * FftShape<TL>::LDS];
  __shared__ cf twl[16 * TL];
  load_twiddles_lds<TL>(twid, twl);
  const int wg = logical_block(per);
  if (wg >= n_wg) return;
  const FftInst& I = fft_instance(inst, n_inst, wg, true);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int task = (wg - I.wg_f) * 4 + wave;
  const int n_cols = I.n_cols, N_rhs = I.N_rhs;
  if (task >= n_cols * N_rhs * I.NZB) return;
  cf* lds = lds_all + wave * FftShape<TL>::LDS;
  const int j = lane / FPW, g = lane % FPW;
  const int r = task % N_rhs, cz = task / N_rhs;
  const int c = cz % n_cols, zb = cz / n_cols;
  const int2 pf = I.col[c];   // pair, frequency
  const int ws0 = zb * I.ZR, ws1 = min(I.n_ws, ws0 + I.ZR);
  const int Np = NP > 0 ? NP : I.Np;
  BORN_GLOBAL const float2* P = I.P + (size_t)pf.x * I.N_pts;
  BORN_GLOBAL const float4* gs = (BORN_GLOBAL const float4*)I.gs + ((size_t)r * I.n_ws + ws0) * (NZ * 32) + lane;
  BORN_GLOBAL const float4* H = (BORN_GLOBAL const float4*)(I.H + ((size_t)pf.y * I.n_ws + ws0) * 1024) + lane;
  BORN_GLOBAL const int2* slots = I.slot + g;
  cf G[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) G[q] = {0.f, 0.f};
  // p_inc of the pair through a buffer descriptor: reads past the grid give 0
  const auto pr = __builtin_amdgcn_make_buffer_rsrc((void*)P, 0, (int)((unsigned)I.N_pts * 8u), 0x27000);
  float2 pv[NZ];
  float4 gv[NZ / 2];
  auto load = [&](int ws, int base) {
    const int off = (base + Np * j) * 8;
#pragma unroll
    for (int q = 0; q < NZ; ++q) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(pr, off + Np * TL * 8 * q, 0, 0);
      pv[q] = make_float2(__uint_as_float(v[0]), __uint_as_float(v[1]));
    }
#pragma unroll
    for (int q = 0; q < NZ / 2; ++q) gv[q] = gs[(size_t)(ws - ws0) * (NZ * 32) + q * 64];
  };
  load(ws0, slots[ws0 * FPW].x);
  int next = slots[min(ws0 + 1, ws1 - 1) * FPW].x;
  for (int ws = ws0; ws < ws1; ++ws) {
    cf x[16];
#pragma unroll
    for (int q = 0; q < NZ; ++q) {
      const float gx = q & 1 ? gv[q / 2].z : gv[q / 2].x, gy = q & 1 ? gv[q / 2].w : gv[q / 2].y;
      x[q] = {fmaf(pv[q].x, gx, -(pv[q].y * gy)), fmaf(pv[q].x, gy, pv[q].y * gx)};
    }
    load(min(ws + 1, ws1 - 1), next);   // (the last step reads its own entries again)
    next = slots[min(ws + 2, ws1 - 1) * FPW].x;
    __builtin_amdgcn_sched_barrier(0);
    float4 hv[8];
    fft_wave_l<TL, NZ>(x, twl, lds, lane, [&] {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 8; ++q) hv[q] = H[q * 64];
      __builtin_amdgcn_sched_barrier(0);
    });
    H += 512;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      cmac(G[2 * q], cf{hv[q].x, hv[q].y}, x[2 * q]);
      cmac(G[2 * q + 1], cf{hv[q].z, hv[q].w}, x[2 * q + 1]);
    }
  }
  // sum over the wave's slots, transform back, store elements e = N_e - 1 - t
#pragma unroll
  for (int q = 0; q < 16; ++q)
#pragma unroll
    for (int m = 1; m < FPW; m <<= 1) {
      G[q].x += __shfl_xor(G[q].x, m);
      G[q].y += __shfl_xor(G[q].y, m);
    }
  fft_wave_l<TL, 16>(G, twl, lds, lane);
  if (g == 0) {
    BORN_GLOBAL float2* out = I.vp + ((size_t)(zb * N_rhs + r) * n_cols + c) * I.N_e;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int t = j + TL * q;
      if (t < I.N_e) out[I.N_e - 1 - t] = make_float2(G[q].x, G[q].y);
    }
  }
}

// Slot-block partials -> V[pair][e][r] (FP64 sums), NS threads per value.  MIX:
// plans whose mixes have one active element each: every observation is one
// value times its prefactor, written here (OutT) in place of V and a mixing
// kernel behind it (64 elements, 256 x 256 points, 65 frequencies, one wave:
// 3.9 and 4.1 us for the two kernels, 4.5 here).
template <int NS, bool MIX, typename OutT>
__global__ __launch_bounds__(256) void k_fft_reduce(const float2* __restrict__ vp, const int2* __restrict__ col, int n_cols,
                                                    int NZB, int N_e, int N_rhs, double2* __restrict__ V,
                                                    const int64_t* __restrict__ pe_off, const int2* __restrict__ pe_ent,
                                                    const double2* __restrict__ pref, int64_t N_obs, OutT* __restrict__ u) {
  constexpr int NV = 256 / NS;
  __shared__ double2 part[NS][NV];
  const int k = threadIdx.x % NV, slice = threadIdx.x / NV;
  const size_t idx = blockIdx.x * (size_t)NV + k;
  const size_t plane = (size_t)n_cols * N_e, total = plane * N_rhs;
  const size_t at = idx < total ? idx : total - 1;
  double sx = 0.0, sy = 0.0;
#pragma unroll 8
  for (int zb = slice; zb < NZB; zb += NS) {
    const float2 v = vp[(size_t)zb * total + at];
    sx += v.x;
    sy += v.y;
  }
  if constexpr (NS > 1) {
    part[slice][k] = make_double2(sx, sy);
    __syncthreads();
    if (slice != 0) return;
#pragma unroll
    for (int i = 1; i < NS; ++i) {
      sx += part[i][k].x;
      sy += part[i][k].y;
    }
  }
  if (idx >= total) return;
  const int r = (int)(idx / plane);
  const size_t ce = idx - (size_t)r * plane;
  const int c = (int)(ce / N_e), e = (int)(ce - (size_t)c * N_e);
  const size_t pe = (size_t)col[c].x * N_e + e;
  if constexpr (MIX) {
    const int64_t i1 = pe_off[pe + 1];
    for (int64_t i = pe_off[pe]; i < i1; ++i) {
      const int2 oe = pe_ent[i];
      const double2 w = pref[oe.y];
      OutT o;
      o.x = w.x * sx - w.y * sy;
      o.y = w.x * sy + w.y * sx;
      u[r * N_obs + oe.x] = o;
    }
  } else {
    V[pe * N_rhs + r] = make_double2(sx, sy);
  }
}

// ------------------------------------------------------------------ adjoint
struct alignas(8) Ent4 {
  int2 e[4];
};

// Un-mixing (as k_adj_unmix) and the spectra of the weights: a wave takes FPW
// (pair, right-hand side) rows, entry t = N_e - 1 - e holds conj(W[e]).
// wt[row][8][TL lanes][2].
template <int TL, bool LONG>
__global__ __launch_bounds__(256) void k_fft_weights(const float2* __restrict__ u, const int64_t* __restrict__ pe_off,
                                                     const int2* __restrict__ pe_ent, const double2* __restrict__ pref,
                                                     const float2* __restrict__ twid, int N_pairs, int N_e,
                                                     int N_rhs, int64_t N_obs, float4* __restrict__ wt) {
  constexpr int FPW = FftShape<TL>::FPW, L = 16 * TL;
  __shared__ cf lds_all[4 * FftShape<TL>::LDS];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int j = lane / FPW, g = lane % FPW;
  const int row = (blockIdx.x * 4 + wave) * FPW + g;
  const bool ok = row < N_pairs * N_rhs;
  const int pair = ok ? row / N_rhs : 0, r = ok ? row - pair * N_rhs : 0;
  const float2* ur = u + (int64_t)r * N_obs;
  // QB elements at a time: the offsets of their lists, then the loads of all of
  // them together (past the end of a list its first entry again; element by
  // element they took 10.6 us for one wave of 64 elements and 33 frequencies, now
  // 8.2).  LONG: 4 entries of each list at a time while all have 4 left: the lanes
  // read as many lists, a line of the L2 each, and one entry of 8 bytes per line
  // is what bounds it (32 waves x 16 mixes of 128 elements, 257 frequencies: 426
  // us by single entries, 215 by four; with lists of one entry 8 elements at a
  // time are 1 us faster).
  constexpr int QB = LONG ? 4 : 8;
  cf tw[16], x[16];
  load_twiddles<TL>(twid, j, tw);
#pragma unroll
  for (int h = 0; h < 16 / QB; ++h) {
    int64_t first[QB];
    int n[QB], most = 0, least = INT_MAX;
    double sx[QB], sy[QB];
#pragma unroll
    for (int q = 0; q < QB; ++q) {
      const int t = j + TL * (QB * h + q);
      const bool have = ok && t < N_e;
      const size_t pe = (size_t)pair * N_e + (have ? N_e - 1 - t : 0);
      first[q] = pe_off[pe];
      n[q] = have ? (int)(pe_off[pe + 1] - first[q]) : -1;
      sx[q] = sy[q] = 0.0;
    }
#pragma unroll
    for (int q = 0; q < QB; ++q) {
      if (n[q] <= 0) first[q] = 0;
      most = max(most, n[q]);
      if (n[q] >= 0) least = min(least, n[q]);
    }
    int i = 0;
    if constexpr (LONG)
      for (; most > 0 && i + 4 <= least; i += 4) {
        Ent4 oe[QB];
        double2 c[QB][4];
        float2 v[QB][4];
#pragma unroll
        for (int q = 0; q < QB; ++q) oe[q] = *reinterpret_cast<const Ent4*>(pe_ent + first[q] + (n[q] > 0 ? i : 0));
#pragma unroll
        for (int q = 0; q < QB; ++q)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            c[q][k] = pref[oe[q].e[k].y];
            v[q][k] = ur[oe[q].e[k].x];
          }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < QB; ++q)
          if (n[q] > 0)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              sx[q] += c[q][k].x * v[q][k].x + c[q][k].y * v[q][k].y;
              sy[q] += c[q][k].x * v[q][k].y - c[q][k].y * v[q][k].x;
            }
      }
    for (; i < most; ++i) {
      int2 oe[QB];
      double2 c[QB];
      float2 v[QB];
#pragma unroll
      for (int q = 0; q < QB; ++q) oe[q] = pe_ent[first[q] + (i < n[q] ? i : 0)];
#pragma unroll
      for (int q = 0; q < QB; ++q) {
        c[q] = pref[oe[q].y];
        v[q] = ur[oe[q].x];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < QB; ++q)
        if (i < n[q]) {
          sx[q] += c[q].x * v[q].x + c[q].y * v[q].y;
          sy[q] += c[q].x * v[q].y - c[q].y * v[q].x;
        }
    }
#pragma unroll
    for (int q = 0; q < QB; ++q) x[QB * h + q] = {(float)sx[q], -(float)sy[q]};
  }
  fft_wave<float, TL, false>(x, tw, lds_all + wave * FftShape<TL>::LDS, lane);
  if (!ok) return;
  float4* out = wt + (size_t)row * (L / 2) + j;
#pragma unroll
  for (int q = 0; q < 8; ++q) out[q * TL] = make_float4(x[2 * q].x, x[2 * q].y, x[2 * q + 1].x, x[2 * q + 1].y);
}

// One workgroup per (slot group, right-hand side, column group); its 4 waves
// share the group's columns and add up their sums through LDS.
template <int TL, int NZ>
__global__ __launch_bounds__(256, 2) void k_fft_adj(const FftInst* __restrict__ inst, int n_inst, OutPtrs outs,
                                                    const float2* __restrict__ twid, int n_wg, int per) {
  constexpr int FPW = FftShape<TL>::FPW;
  __shared__ cf lds_all[4 * FftShape<TL>::LDS];
  __shared__ cf twl[16 * TL];
  load_twiddles_lds<TL>(twid, twl);
  const int wg = logical_block(per);
  if (wg >= n_wg) return;
  const FftInst& I = fft_instance(inst, n_inst, wg, false);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int j = lane / FPW, g = lane % FPW;
  cf* lds = lds_all + wave * FftShape<TL>::LDS;
  const int N_rhs = I.N_rhs, n_cols = I.n_cols, FG = I.FG;
  int t = wg - I.wg_a;
  const int r = t % N_rhs;
  t /= N_rhs;
  const int ws = t % I.n_ws, fgr = t / I.n_ws;
  const int part = fgr * 4 + wave;   // of 4 FG contiguous column ranges
  const int c0 = (int)((long)n_cols * part / (4 * FG)), c1 = (int)((long)n_cols * (part + 1) / (4 * FG));
  const int2 sl = I.slot[ws * FPW + g];
  const int Np = I.Np;
  int at[NZ];
  bool ok[NZ];
#pragma unroll
  for (int q = 0; q < NZ; ++q) {
    const int s = j + TL * q;
    ok[q] = s < sl.y;
    at[q] = sl.x + (ok[q] ? Np * s : 0);
  }
  cf acc[NZ];
#pragma unroll
  for (int q = 0; q < NZ; ++q) acc[q] = {0.f, 0.f};
  float4 hv[8];
  int f_have = -1;
  for (int c = c0; c < c1; ++c) {
    const int2 pf = I.col[c];
    BORN_GLOBAL const float2* P = I.P + (size_t)pf.x * I.N_pts;
    if (pf.y != f_have) {
      f_have = pf.y;
      BORN_GLOBAL const float4* H = (BORN_GLOBAL const float4*)(I.H + ((size_t)pf.y * I.n_ws + ws) * 1024) + lane;
#pragma unroll
      for (int q = 0; q < 8; ++q) hv[q] = H[q * 64];
    }
    BORN_GLOBAL const float4* wt = (BORN_GLOBAL const float4*)I.wt + ((size_t)pf.x * N_rhs + r) * (8 * TL) + j;
    float4 wv[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) wv[q] = wt[q * TL];
    __builtin_amdgcn_sched_barrier(0);   // all loads in flight before the first is waited for,
    float2 pv[NZ];                       // p_inc last: it stays in flight during the transform
#pragma unroll
    for (int q = 0; q < NZ; ++q) pv[q] = P[at[q]];
    __builtin_amdgcn_sched_barrier(0);
    cf x[16];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      x[2 * q] = {fmaf(hv[q].x, wv[q].x, -(hv[q].y * wv[q].y)), fmaf(hv[q].x, wv[q].y, hv[q].y * wv[q].x)};
      x[2 * q + 1] = {fmaf(hv[q].z, wv[q].z, -(hv[q].w * wv[q].w)), fmaf(hv[q].z, wv[q].w, hv[q].w * wv[q].z)};
    }
    fft_wave_l<TL, 16>(x, twl, lds, lane);
#pragma unroll
    for (int q = 0; q < NZ; ++q) cmac(acc[q], cf{pv[q].x, pv[q].y}, x[q]);
  }
#pragma unroll
  for (int q = 0; q < NZ; ++q) lds[q * 64 + lane] = acc[q];
  __syncthreads();
  BORN_GLOBAL float2* out = FG > 1 ? I.gp + (size_t)fgr * N_rhs * I.N_pts : (BORN_GLOBAL float2*)outs.p[&I - inst];
  out += (size_t)r * I.N_pts;
#pragma unroll
  for (int q = 0; q < NZ; ++q)
    if ((q & 3) == wave && ok[q]) {
      cf s = {0.f, 0.f};
#pragma unroll
      for (int w = 0; w < 4; ++w) s = cadd(s, lds_all[w * FftShape<TL>::LDS + q * 64 + lane]);
      out[at[q]] = make_float2(s.x, -s.y);
    }
}

__global__ __launch_bounds__(256) void k_fft_adj_reduce(const float2* __restrict__ gp, int FG, size_t n,
                                                        float2* __restrict__ out) {
  const size_t i = blockIdx.x * (size_t)256 + threadIdx.x;
  if (i >= n) return;
  double x = 0.0, y = 0.0;
#pragma unroll 8
  for (int k = 0; k < FG; ++k) {
    const float2 v = gp[(size_t)k * n + i];
    x += v.x;
    y += v.y;
  }
  out[i] = make_float2((float)x, (float)y);
}

// ------------------------------------------------------------------ host side
// Entries of a lane that the kernels take, at least n: 4, 6, 8, 10, 12 or 16.
static int fft_entries(int n) { return n <= 4 ? 4 : n <= 12 ? (n + 1) / 2 * 2 : 16; }

// Transform length and segments of a row of S points per phase under N_e
// elements: the cheapest of the lengths (time grows with the entries
// transformed; sequences at most half full skip part of the first stage).
FftShapeChoice fft_shape(int Nx, int Np, int N_e) {
  FftShapeChoice best;
  const int S = (Nx + Np - 1) / Np;
  double cost_best = 1e300;
  for (int TL = 4; TL <= 16; TL *= 2) {
    const int L = 16 * TL;
    if (L < N_e) continue;
    const int room = L - N_e + 1;
    FftShapeChoice c;
    c.TL = TL;
    c.nseg = (S + room - 1) / room;
    c.Sv = (S + c.nseg - 1) / c.nseg;
    c.nz = fft_entries((c.Sv + TL - 1) / TL);
    const double cost = (double)c.nseg * L * (c.nz <= 8 ? 1.0 : 1.12);
    if (cost < cost_best) {
      cost_best = cost;
      best = c;
    }
  }
  return best;
}

// unit: of the values next to each twiddle the one of magnitude closest to 1,
// for sums of squared outputs (rounded to the nearest the twiddles of length
// 128 have the mean magnitude 1 - 5e-9, which two transforms make -2e-8 of the
// energy); their phases are off by up to 6e-8 in place of 3e-8.
void fft_twiddles(int TL, std::vector<float2>& tw, bool unit) {
  tw.resize((size_t)TL * 16);
  for (int j = 0; j < TL; ++j)
    for (int k = 0; k < 16; ++k) {
      const double a = 2.0 * M_PI * j * k / (16.0 * TL), c = std::cos(a), s = std::sin(a);
      const float cf = (float)c, sf = (float)s;
      float2 best = make_float2(cf, sf);
      double least = 1e300;
      for (int i = 0; unit && i < 9; ++i) {
        const float x = i % 3 == 0 ? cf : std::nextafterf(cf, i % 3 == 1 ? 2.f : -2.f);
        const float y = i / 3 == 0 ? sf : std::nextafterf(sf, i / 3 == 1 ? 2.f : -2.f);
        const double mag = c * (x - c) + s * (y - s), phase = c * (y - s) - s * (x - c);
        const double cost = 16.0 * mag * mag + phase * phase;
        if (cost < least) {
          least = cost;
          best = make_float2(x, y);
        }
      }
      tw[(size_t)j * 16 + k] = best;
    }
}

// What the spectra have to be multiplied with, minus 1, for transforms without a
// bias.  FP32 rounds sqrt(1/2) and cos(pi/8) down and the twiddles' magnitudes
// vary, so that a transform takes 2e-8 to 3e-8 off its outputs: no more than
// their rounding, but the same for all of them, where a sum of squares averages the rounding
// out.  Entry n of the input meets entry k = k1 + 16 k2 of the output, n = j + TL q,
// through the factors of (q, k1), of the twiddle (j, k1) and of (j, k2); entry m
// of a spectrum comes from the inputs of the first transform and goes to the
// outputs of the second (S points and N_e elements, or the other way round in
// the adjoint), and is divided by the mean of both.  Squared norms of forward and adjoint were
// 0.8 to 1.5e-7 low and are within 5e-9.
void fft_gains(int TL, const std::vector<float2>& tw, int S, int N_e, std::vector<float>& delta) {
  const double r2 = 0.70710678118654752440;
  const double e2 = (double)(float)r2 / r2 - 1.0;
  const double e1 = (double)(float)FFT_C1 * FFT_C1 + (double)(float)FFT_S1 * FFT_S1 - 1.0;
  auto of16 = [&](int a, int b) {   // dft16: products of entries a % 4 and b % 4
    const int p = (a % 4) * (b % 4);
    return p % 2 == 1 ? e1 : p == 2 || p == 6 ? e2 : 0.0;
  };
  auto of_last = [&](int j, int k2) { return TL == 16 ? of16(j, k2) : TL == 8 && j % 2 == 1 && k2 % 2 == 1 ? e2 : 0.0; };
  const int L = 16 * TL;
  std::vector<double> sum(L, 0.0), twist((size_t)TL * 16);
  for (int j = 0; j < TL; ++j)
    for (int k1 = 0; k1 < 16; ++k1) {
      const double a = 2.0 * M_PI * j * k1 / L;
      const float2 w = tw[(size_t)j * 16 + k1];
      twist[(size_t)j * 16 + k1] = w.x * std::cos(a) + w.y * std::sin(a) - 1.0;
    }
  for (int N : {S, N_e}) {
    std::vector<double> in_q(16, 0.0), in_j(TL, 0.0), out_k1(16, 0.0), out_k2(TL, 0.0);   // shares of the N entries
    for (int n = 0; n < N; ++n) {
      in_q[n / TL] += 0.5 / N;
      in_j[n % TL] += 0.5 / N;
      out_k1[n % 16] += 0.5 / N;
      out_k2[n / 16] += 0.5 / N;
    }
    for (int m = 0; m < L; ++m) {
      for (int i = 0; i < 16; ++i)
        sum[m] += in_q[i] * of16(i, m % 16) + out_k1[i] * (of16(m / TL, i) + twist[(size_t)(m % TL) * 16 + i]);
      for (int i = 0; i < TL; ++i)
        sum[m] += in_j[i] * (twist[(size_t)i * 16 + m % 16] + of_last(i, m / 16)) + out_k2[i] * of_last(m % TL, i);
    }
  }
  delta.resize(L);
  for (int m = 0; m < L; ++m) delta[m] = (float)-sum[m];
}

void launch_fft_table(const Plan& P, hipStream_t s) {
  const Plan::Fft& F = P.fft;
  const dim3 grid(F.n_ws, P.N_fu);
#define BORN_FFT_TABLE(TLv)                                                                                            \
  hipLaunchKernelGGL(k_fft_table<TLv>, grid, dim3(64), 0, s, P.d_h, P.d_ext, P.d_hrow, P.H_plane, P.HR, P.N_ext, P.Np, \
                     F.shape.nseg, F.shape.Sv, F.n_slots, F.n_ws, reinterpret_cast<const float*>(F.d_tw + 16 * TLv), F.d_H)
  if (F.shape.TL == 16) BORN_FFT_TABLE(16);
  else if (F.shape.TL == 8) BORN_FFT_TABLE(8);
  else BORN_FFT_TABLE(4);
#undef BORN_FFT_TABLE
}

#define BORN_FFT_NZ(F, TLv)         \
  do {                              \
    switch (S.nz) {                 \
      case 4: F(TLv, 4); break;     \
      case 6: F(TLv, 6); break;     \
      case 8: F(TLv, 8); break;     \
      case 10: F(TLv, 10); break;   \
      case 12: F(TLv, 12); break;   \
      default: F(TLv, 16); break;   \
    }                               \
  } while (0)
#define BORN_FFT_DISPATCH(F)               \
  do {                                     \
    if (S.TL == 16) BORN_FFT_NZ(F, 16);    \
    else if (S.TL == 8) BORN_FFT_NZ(F, 8); \
    else BORN_FFT_NZ(F, 4);                \
  } while (0)

void launch_fft_range(const Plan& P, int* bad, hipStream_t s) {
  const bool y = P.nd == 3;
  const int64_t rows = (int64_t)P.Nz * P.N_fu;
  hipLaunchKernelGGL(k_fft_range, dim3((unsigned)std::min<int64_t>(rows, 1 << 20)), dim3(256), 0, s, P.d_h, P.d_ext,
                     y ? P.d_exty : nullptr, P.N_ext, y ? P.Ny + (P.Ney - 1) * P.Npy : 1, P.H_plane, P.HR, P.HY, P.Nz,
                     P.Np, y ? P.Npy : 1, rows, bad);
}

void launch_fft_gamma(const Plan& P, const float2* gamma, int N_rhs, bool mask, hipStream_t s) {
  const Plan::Fft& F = P.fft;
  const dim3 grid((unsigned)(((size_t)F.n_ws * F.shape.nz * 64 + 255) / 256));
#define BORN_FFT_G(TLv)                                                                                               \
  hipLaunchKernelGGL(k_fft_gamma<TLv>, grid, dim3(256), 0, s, gamma, F.d_slot, F.n_ws, F.shape.nz, P.N_pts, P.Np, \
                     N_rhs, (int)mask, F.d_gs)
  if (F.shape.TL == 16) BORN_FFT_G(16);
  else if (F.shape.TL == 8) BORN_FFT_G(8);
  else BORN_FFT_G(4);
#undef BORN_FFT_G
}

void launch_fft_fwd(const FftSet& S, hipStream_t s) {
  if (S.inst.empty()) return;
  const int per = (S.n_wg_f + XCDS - 1) / XCDS;
  int Np = S.inst[0].Np;
  for (const FftInst& I : S.inst)
    if (I.Np != Np) Np = 0;
#define BORN_FFT_F(TLv, NZv, NPv)                                                                                   \
  hipLaunchKernelGGL((k_fft_fwd<TLv, NZv, NPv>), dim3(per * XCDS), dim3(256), 0, s, S.d_inst, (int)S.inst.size(), \
                     S.d_tw, S.n_wg_f, per)
#define BORN_FFT_FN(TLv, NZv)                  \
  do {                                         \
    if (Np == 4) BORN_FFT_F(TLv, NZv, 4);      \
    else if (Np == 2) BORN_FFT_F(TLv, NZv, 2); \
    else BORN_FFT_F(TLv, NZv, 0);              \
  } while (0)
  BORN_FFT_DISPATCH(BORN_FFT_FN);
#undef BORN_FFT_FN
#undef BORN_FFT_F
}

void launch_fft_adj(const FftSet& S, const OutPtrs& outs, hipStream_t s) {
  if (S.inst.empty()) return;
  const int per = (S.n_wg_a + XCDS - 1) / XCDS;
#define BORN_FFT_A(TLv, NZv)                                                                                          \
  hipLaunchKernelGGL((k_fft_adj<TLv, NZv>), dim3(per * XCDS), dim3(256), 0, s, S.d_inst, (int)S.inst.size(), outs, \
                     S.d_tw, S.n_wg_a, per)
  BORN_FFT_DISPATCH(BORN_FFT_A);
#undef BORN_FFT_A
}

// Threads per value: 8 where there are fewer values than threads the chip
// holds and more than 16 blocks to add (one thread takes them one after the
// other: 10 us for 32 blocks of 1400 values, 28 us for 64 of 10^4, with 8
// threads 4 and 6), else 1 (10^6 values of 8 blocks: 19 us, with 8 threads 31).
void launch_fft_reduce(const Plan& P, int N_rhs, void* u, bool out_f64, hipStream_t s) {
  const size_t total = (size_t)P.N_pairs * P.N_e * N_rhs;
  const bool many = total < ((size_t)1 << 19) && P.fft.NZB > 16;
  const dim3 grid((unsigned)(many ? (total + 31) / 32 : (total + 255) / 256));
#define BORN_FFT_R(NSv, MIXv, T)                                                                                        \
  hipLaunchKernelGGL((k_fft_reduce<NSv, MIXv, T>), grid, dim3(256), 0, s, P.fft.d_vp, P.fft.d_col, P.N_pairs, P.fft.NZB, \
                     P.N_e, N_rhs, P.d_V, P.d_pe_off, P.d_pe_ent, P.d_pref, P.N_obs, (T*)u)
#define BORN_FFT_RM(NSv)                                  \
  do {                                                    \
    if (!P.single_mixes) BORN_FFT_R(NSv, false, float2);  \
    else if (out_f64) BORN_FFT_R(NSv, true, double2);     \
    else BORN_FFT_R(NSv, true, float2);                   \
  } while (0)
  if (many) BORN_FFT_RM(8);
  else BORN_FFT_RM(1);
#undef BORN_FFT_RM
#undef BORN_FFT_R
  if (!P.single_mixes) launch_fwd_mix(P, N_rhs, u, out_f64, s);
}

void launch_fft_weights(const Plan& P, const float2* u, int N_rhs, hipStream_t s) {
  const int TL = P.fft.shape.TL, FPW = 64 / TL;
  const size_t rows = (size_t)P.N_pairs * N_rhs;
  const dim3 grid((unsigned)((rows + 4 * FPW - 1) / (4 * FPW)));
#define BORN_FFT_WL(TLv, LONGv)                                                                                      \
  hipLaunchKernelGGL((k_fft_weights<TLv, LONGv>), grid, dim3(256), 0, s, u, P.d_pe_off, P.d_pe_ent, P.d_pref,        \
                     P.fft.d_tw, P.N_pairs, P.N_e, N_rhs, P.N_obs, (float4*)P.fft.d_wt)
#define BORN_FFT_W(TLv)                                                          \
  do {                                                                           \
    if (P.n_pe_ent >= 4 * (int64_t)P.N_pairs * P.N_e) BORN_FFT_WL(TLv, true);    \
    else BORN_FFT_WL(TLv, false);                                                \
  } while (0)
  if (TL == 16) BORN_FFT_W(16);
  else if (TL == 8) BORN_FFT_W(8);
  else BORN_FFT_W(4);
#undef BORN_FFT_WL
#undef BORN_FFT_W
}

void launch_fft_adj_reduce(const Plan& P, int N_rhs, float2* out, hipStream_t s) {
  if (P.fft.FG <= 1) return;
  const size_t n = (size_t)P.N_pts * N_rhs;
  hipLaunchKernelGGL(k_fft_adj_reduce, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, P.fft.d_gp, P.fft.FG, n, out);
}

}  // namespace born
