// soi_filter_g.hpp -- Step 1 of the SOI FFT in complex128 on MFMA (parallel_filter_subsampling.cpp:
// 52-527): B-tap filter, subsampling and S-point DFT, stored segment-major.
//
// GEMM of lane i on v_mfma_f64_16x16x4_f64: rows are eight row groups m by real and imaginary
// part, columns the n_mu phases of ND consecutive row groups,
//   C[8 part + m][theta + n_mu D] = sum_k x_i[d J0 + ND d m + k].part * t_i[theta][k - d D],
// ND = 3, 15 columns for mu = 5/4 and ND = 2, 16 columns for mu = 8/7, K = 4 NK >= B + d (ND - 1).
// Lane layout (checked by soik_mfma64_layout_probe): A[row][k] in lane row + 16k, B[k][col] in lane
// col + 16k, D[row][col] in lane col + 16 (row % 4), register row / 4; so lane col + 16g holds m = g
// (registers 0 and 2: real and imaginary part) and m = 4 + g (registers 1 and 3).
// Real taps (exact windows: the factor e^{i pi t} splits into a phase per (theta, i), applied to the
// result, and (-1)^b) take one product; complex taps (the reference's window values: narrow
// windows, mu = 8/7) two, with Re t and Im t as the B operand and the same A operand, whose results
// combine within the lane.
//
// Wave w owns the lanes i = NW li + w, li < LPW.  The S-point DFT of each output row R splits as
// i = NW li + w, s = s1 + LPW s2:
//   X[s] = sum_w w_NW^{w s2} [ w_S^{w s1} sum_li gamma[NW li + w] w_LPW^{li s1} ],
// the LPW-point DFTs in the registers of the wave that holds the lanes, then one exchange through
// LDS and an NW-point DFT per (R, s1), whose NW results go straight to HBM.
//
// What bounds it and what the layout follows from.  FP64 MFMA and FP64 FMA have the same peak
// (78.6 TFLOP/s); the matrix form wins because one 8-byte LDS read per lane feeds one or two products
// of 1024 FMAs, where the VALU form (soi_filter.hip) reads 16 bytes for about nine FMAs.  The B
// operands of a wave's lanes (NK or 2 NK values per lane i) stay in registers where they take 160 or
// fewer (RES: complex taps S <= 16 with up to 20 K steps and S = 32 with 10; real taps S <= 16, and S = 32 with
// 20); elsewhere they stream from L2 a few K steps ahead; the rows of all lanes
// exceed LDS at S = 64, so lanes go through in groups of 16.  Two row buffers alternate, one filling
// (direct-to-LDS loads) while the other is multiplied; results of all groups stay in registers until
// the S-point DFT.  Long transforms of S = 32 with resident real taps have four
// buffers of eight lanes instead (QUAD): with two, the wait for a group's rows covers the stores of the
// tile before, which share their queue.  N = 2^27 1.34 -> 1.24 ms, 2^26 685 -> 632 us, 2^22 57.7 -> 54.9;
// it loses where one product chain a wave does not fill the matrix pipe or there is little to multiply
// (S = 16, N = 2^24 173 -> 187; B = 30, S = 32 157 -> 179).  Measured, VALU form -> here: S = 64, mu = 8/7, N = 7*2^23 1.91 -> 0.95 ms (the
// products alone: 0.55); S = 32, mu = 8/7, N = 7*2^20 190 -> 111 us; B = 44, N = 2^22, S = 16 88 ->
// 54; S = 64, N = 2^24 305 -> 230.  Against rows in a ring that only the new rows of a tile entered
// (real taps, S <= 32): N = 2^22, S = 4 59 -> 49 us, S = 8 56 -> 48, S = 16 56 -> 50, S = 32 58 -> 56;
// N = 2^27, S = 32 1.33 ms either way (products 0.73, memory 0.85; two buffers).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "soi_common.hpp"
#include "soi_kernels.h"

namespace soi {

typedef double gd4 __attribute__((ext_vector_type(4)));
typedef double gd2 __attribute__((ext_vector_type(2)));

template <int S_, int NMU_, int DMU_, int NK_, bool CT_, bool QUAD_ = false> struct FilterG {
  static constexpr int S = S_, NMU = NMU_, DMU = DMU_, NK = NK_;
  static constexpr bool CT = CT_;
  static constexpr int ND = NMU == 5 ? 3 : 2;    // row groups side by side in the columns
  static constexpr int NCOL = NMU * ND;          // columns used (15 or 16)
  static constexpr int TJ = 8 * ND;              // row groups per tile
  static constexpr int MS = ND * DMU;            // input rows from m to m + 1
  static constexpr int ROWS = 7 * MS + 4 * NK;   // input rows per tile
  static constexpr int NW = S < 16 ? S / 2 : 8;  // waves
  static constexpr int LPW = S / NW;             // lanes i = NW li + w of a wave, li < LPW
  // B operands resident in registers, or streamed
  static constexpr bool RES = LPW * NK * (CT ? 4 : 2) <= 160;
  static constexpr bool QUAD = QUAD_;            // four row buffers of eight lanes, not two
  static constexpr int NBUF = QUAD ? 4 : 2;
  static constexpr int GL = S < 16 ? S : QUAD ? 8 : 16;  // lanes per group: GL / NW a wave
  static constexpr int NGRP = S / GL;
  static constexpr int T = NW * 64;
  static constexpr int RPC = 64 / GL;            // rows per chunk (64 values, one wave-wide load)
  static constexpr int NCHK = (ROWS + RPC - 1) / RPC;
  static constexpr int NLD = (NCHK + NW - 1) / NW;   // loads per wave and buffer
  static constexpr int CP = 65;                  // chunk pitch: a 16-byte gap spreads the banks
  static constexpr int GR = TJ * NMU;            // output rows per tile
  static constexpr int NH = S == 64 ? 2 : 1;     // rounds of the exchange (its rows by halves of m)
  static constexpr int GRH = GR / NH;
  static constexpr int GP = S + 1;
  static constexpr int NTASK = GRH * LPW;
  static constexpr int NC = (NTASK + T - 1) / T;
  static constexpr int NB = 64 / (4 * GL);       // A address bases (K steps per chunk)
  static constexpr int LDS_BYTES = (NBUF * NCHK * CP + GRH * GP + S + (CT ? 1 : NMU * S)) * 16;
  static constexpr int MIN_M = NCHK * RPC;       // rows of a tile's loads wrap at most once
  static_assert(NK % 2 == 0 || CT, "real taps are loaded two K steps at a time");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS");
  static_assert(!QUAD || (RES && !CT && S == 32 && NC == 1), "four buffers");
};

// Products and an 8-point DFT with the fused operations spelled out: a tile's results are then the same bit
// for bit in every code copy that the compiler makes (batched launches split the tiles over blocks
// differently).
__device__ __forceinline__ double2 cmul_fma(double2 a, double2 b)
{
  return double2{__builtin_fma(a.x, b.x, -(a.y * b.y)), __builtin_fma(a.x, b.y, a.y * b.x)};
}
__device__ __forceinline__ void dft8_plain(double2 *a)
{
#pragma clang fp contract(off)
  const double r = 0.70710678118654752440084436210485;
  dft4(a[0], a[2], a[4], a[6]);
  dft4(a[1], a[3], a[5], a[7]);
  const double2 e0 = a[0], e1 = a[2], e2 = a[4], e3 = a[6], o2 = cmul_mi(a[5]);
  const double s1 = a[3].x + a[3].y, d1 = a[3].y - a[3].x, d3 = a[7].y - a[7].x, s3 = a[7].x + a[7].y;
  a[0] = double2{e0.x + a[1].x, e0.y + a[1].y};
  a[4] = double2{e0.x - a[1].x, e0.y - a[1].y};
  a[1] = double2{__builtin_fma(r, s1, e1.x), __builtin_fma(r, d1, e1.y)};
  a[5] = double2{__builtin_fma(-r, s1, e1.x), __builtin_fma(-r, d1, e1.y)};
  a[2] = double2{e2.x + o2.x, e2.y + o2.y};
  a[6] = double2{e2.x - o2.x, e2.y - o2.y};
  a[3] = double2{__builtin_fma(r, d3, e3.x), __builtin_fma(-r, s3, e3.y)};
  a[7] = double2{__builtin_fma(-r, d3, e3.x), __builtin_fma(r, s3, e3.y)};
}
template <int R> __device__ __forceinline__ void dft_plain(double2 *a)
{
  if constexpr (R == 8) dft8_plain(a);
  else dft_r<R>(a);
}

// Place q of n in the order from both ends inwards: 0, n - 1, 1, n - 2, ...
constexpr int inwards(int q, int n) { return q & 1 ? n - 1 - q / 2 : q / 2; }

// B operands of lane i: double2 {Re t, Im t} per K step (complex taps) or two K steps (real)
template <typename F>
__global__ __launch_bounds__(F::T, 2) void k_filter_g(const double2 *__restrict__ x,
                                                      double2 *__restrict__ at,
                                                      const double2 *__restrict__ wt,
                                                      const double2 *__restrict__ post,
                                                      const double2 *__restrict__ twS, long M,
                                                      long Mh, long nJ, int tiles_per_block,
                                                      SoiBatch b)
{
  constexpr int S = F::S, NK = F::NK, NW = F::NW, LPW = F::LPW, NGRP = F::NGRP, GP = F::GP;
  constexpr bool CT = F::CT;
  typedef __attribute__((address_space(3))) void lds_t;
  typedef __attribute__((address_space(1))) gd2 ggd2;
  x = batch_ptr(x, b.x);
  at = batch_ptr(at, b.at);
  ggd2 *const atg = (ggd2 *)at;
  // (buffers of their own names: the compiler then knows which loads an LDS read has to wait for)
  constexpr int BSZ = F::NCHK * F::CP;
  __shared__ __align__(16) double2 buf0[BSZ];
  __shared__ __align__(16) double2 buf1[BSZ];
  __shared__ __align__(16) double2 buf2[F::QUAD ? BSZ : 1];
  __shared__ __align__(16) double2 buf3[F::QUAD ? BSZ : 1];
  __shared__ __align__(16) double2 G[F::GRH * GP];
  __shared__ __align__(16) double2 tw[S];
  __shared__ __align__(16) double2 pfl[CT ? 1 : F::NMU * S];
  auto rows_buf = [&](int i) __attribute__((always_inline)) -> double2 * {
    return i == 0 ? buf0 : i == 1 ? buf1 : i == 2 ? buf2 : buf3;
  };
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;

  const long ntiles = (nJ + F::TJ - 1) / F::TJ;
  // tiles t0, t0 + step, ..., t1.  QUAD: the blocks go through the tiles side by side, so that what
  // they load and store at a time is adjacent
  const long step = F::QUAD ? gridDim.x : 1;
  const long t0 = F::QUAD ? xcd_remap(blockIdx.x, gridDim.x) : (long)blockIdx.x * tiles_per_block;
  if (t0 >= ntiles) return;
  const long t1 = F::QUAD ? t0 + (ntiles - 1 - t0) / step * step : min(ntiles, t0 + tiles_per_block) - 1;

  // rows of lane group gr of a tile into a buffer: element e of the tile's rows (row e / GL, place
  // e % GL) at LDS place e + e / 64.  With 16 lanes a row is all the banks of an 8-byte read, so odd
  // rows hold their lanes 8 places round.  Every wave issues NLD loads (the last ones of some waves
  // repeat the last chunk).
  auto dma = [&](double2 *dst, long tile, int gr) {
    const long row0 = tile * F::TJ * F::DMU;
#pragma unroll
    for (int q = 0; q < F::NLD; ++q) {
      const int c = min(wave + q * NW, F::NCHK - 1);
      const int e = c * 64 + lane, r = e / F::GL;
      int il = e % F::GL;
      if constexpr (F::GL == 16) il ^= 8 * (r & 1);
      long row = row0 + r;
      if (row >= M) row -= M;
      __builtin_amdgcn_global_load_lds((const void *)(x + row * S + gr * F::GL + il),
                                       (lds_t *)(dst + c * F::CP), 16, 0, 0);
    }
  };
  dma(buf0, t0, 0);
  if constexpr (F::QUAD) {
    dma(buf1, t0, 1);
    dma(buf2, t0, 2);
  }

  for (int e = tid; e < S; e += F::T) tw[e] = twS[e];
  if constexpr (!CT)
    for (int e = tid; e < F::NMU * S; e += F::T) pfl[e] = post[e];

  // B operand table: item it of lane i at wt[(i * NIT + it) * 64 + lane].  Items are multiplied from the
  // ends of the taps inwards (item(j) is the j-th; of its two K steps, real taps, the outer one
  // first): the taps peak in the middle, so a chain's sum stays small until its last steps.  In the
  // order of the taps every step after the peak rounds the whole sum: S = 16, error of the filter with
  // 72 real taps 3.8e-16 -> 2.9e-16, with 44 complex 2.5e-16 -> 1.8e-16 (the VALU form, which adds two
  // or four slices: 1.8e-16).  The time is the same.
  constexpr int NIT = CT ? NK : NK / 2;
  auto item = [](int j) { return inwards(j, NIT); };
  auto kstep = [&](int q) {
    if constexpr (CT) return item(q);
    else return 2 * item(q / 2) + ((q & 1) ^ (q / 2 & 1));
  };
  const unsigned lane16 = lane * 16u;
  typedef const __attribute__((address_space(1))) char gchar;
  typedef const __attribute__((address_space(1))) gd2 cgd2;
  gchar *wbase = (gchar *)(wt + (long)wave * NIT * 64);
  auto bload = [&](int li, int it) -> double2 {
    const gd2 w = *(cgd2 *)(wbase + (NW * li * NIT + it) * 1024 + lane16);
    return double2{w.x, w.y};
  };
  double2 wb[F::RES ? LPW : 1][F::RES ? NIT : 1];
  if constexpr (F::RES) {
#pragma unroll
    for (int li = 0; li < LPW; ++li)
#pragma unroll
      for (int it = 0; it < NIT; ++it) wb[li][it] = bload(li, it);
  }
  // streamed: complex taps run the two lanes of a group one after the other (SEQ = 2 NIT items),
  // real taps side by side (an item for each); PD items ahead, also into the next group
  constexpr int SEQ = CT ? 2 * NIT : NIT, WID = CT ? 1 : 2;
  constexpr int PD = SEQ % 10 == 0 ? (CT ? 10 : 5) : SEQ % 13 == 0 ? 13 : SEQ % 11 == 0 ? 11 : 8;
  static_assert(F::RES || SEQ % PD == 0, "prefetch ring");
  double2 bq[F::RES ? 1 : PD][WID];
  auto bnext = [&](int gr, int it) {  // item it (< SEQ) of group gr into its ring place
    if constexpr (CT) bq[it % PD][0] = bload(2 * gr + it / NIT, item(it % NIT));
    else {
      bq[it % PD][0] = bload(2 * gr, item(it));
      bq[it % PD][WID - 1] = bload(2 * gr + 1, item(it));
    }
  };
  if constexpr (!F::RES) {
#pragma unroll
    for (int it = 0; it < PD; ++it) bnext(0, it);
  }

  // A operand of lane (n, g): row m = n & 7, part n >> 3, k = g: row MS m + 4 ks + g, lane place il
  int ab[2][F::NB];
#pragma unroll
  for (int lh = 0; lh < 2; ++lh)
#pragma unroll
    for (int j = 0; j < F::NB; ++j) {
      const int r = F::MS * (n & 7) + g + 4 * j;
      int il = NW * lh + wave;
      if constexpr (F::GL == 16) il ^= 8 * (r & 1);
      const int e = r * F::GL + il;
      ab[lh][j] = (e + (e >> 6)) * 16 + (n >> 3) * 8;
    }
  auto aread = [&](const double2 *buf, int lh, int ks) -> double {
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(buf) +
                                             ab[lh][ks % F::NB] + ks / F::NB * (F::CP * 16));
  };

  double2 gam[LPW][2];  // [li][h]: row m = 4h + g, column n

  auto wait_loads = [&](auto n_tag) __attribute__((always_inline)) {  // all but the last n vector memory operations
    constexpr int N = decltype(n_tag)::value;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | (N >> 4 << 14));
  };
  // MFMA of lane group gr from buf
  auto mul = [&](const double2 *buf, auto gr_tag) __attribute__((always_inline)) {
    constexpr int gr = decltype(gr_tag)::value, ng = (gr + 1) % NGRP;
    if constexpr (F::QUAD) {
      gd4 cr = {0, 0, 0, 0};
      double a[3] = {aread(buf, 0, kstep(0)), aread(buf, 0, kstep(1))};
#pragma unroll
      for (int q = 0; q < NK; ++q) {
        const int ks = kstep(q);
        const double2 w = wb[gr][ks / 2];
        if (q + 2 < NK) a[(q + 2) % 3] = aread(buf, 0, kstep(q + 2));
        cr = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q % 3], ks & 1 ? w.y : w.x, cr, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) gam[gr][h] = double2{cr[h], cr[h + 2]};
    } else if constexpr (CT) {
#pragma unroll
      for (int lh = 0; lh < 2; ++lh) {
        gd4 cr = {0, 0, 0, 0}, ci = {0, 0, 0, 0};
        double a = aread(buf, lh, kstep(0));
#pragma unroll
        for (int q = 0; q < NK; ++q) {
          const int it = lh * NK + q;
          double2 w;
          if constexpr (F::RES) w = wb[2 * gr + lh][kstep(q)];
          else w = bq[it % PD][0];
          double an = 0;
          if (q + 1 < NK) an = aread(buf, lh, kstep(q + 1));
          cr = __builtin_amdgcn_mfma_f64_16x16x4f64(a, w.x, cr, 0, 0, 0);
          ci = __builtin_amdgcn_mfma_f64_16x16x4f64(a, w.y, ci, 0, 0, 0);
          if constexpr (!F::RES) {
            if (it + PD < SEQ) bnext(gr, it + PD);
            else bnext(ng, it + PD - SEQ);
          }
          a = an;
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) gam[2 * gr + lh][h] = double2{cr[h] - ci[h + 2], cr[h + 2] + ci[h]};
      }
    } else {
      gd4 c0 = {0, 0, 0, 0}, c1 = {0, 0, 0, 0};
      double a0 = aread(buf, 0, kstep(0)), a1 = aread(buf, 1, kstep(0));
#pragma unroll
      for (int q = 0; q < NK; ++q) {
        const int it = q / 2, ks = kstep(q);
        double2 w0, w1;
        if constexpr (F::RES) w0 = wb[2 * gr][ks / 2], w1 = wb[2 * gr + 1][ks / 2];
        else w0 = bq[it % PD][0], w1 = bq[it % PD][WID - 1];
        double n0 = 0, n1 = 0;
        if (q + 1 < NK) n0 = aread(buf, 0, kstep(q + 1)), n1 = aread(buf, 1, kstep(q + 1));
        c0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, ks & 1 ? w0.y : w0.x, c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, ks & 1 ? w1.y : w1.x, c1, 0, 0, 0);
        if constexpr (!F::RES) {
          if (q & 1) {
            if (it + PD < SEQ) bnext(gr, it + PD);
            else bnext(ng, it + PD - SEQ);
          }
        }
        a0 = n0, a1 = n1;
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        gam[2 * gr][h] = double2{c0[h], c0[h + 2]};
        gam[2 * gr + 1][h] = double2{c1[h], c1[h + 2]};
      }
    }
  };

  // S-point DFT of a tile, round rd of the exchange: LPW-point DFTs of the wave's lanes into G
  auto put = [&](int rd) __attribute__((always_inline)) {
    int tv = tid;
    asm volatile("" : "+v"(tv));  // keep the addresses below out of registers in the tile loop
    const int nv = tv & 15, gv = (tv >> 4) & 3;
#pragma unroll
    for (int hh = 0; hh < 2 / F::NH; ++hh) {
      const int h = F::NH == 2 ? rd : hh;
      double2 v[LPW];
#pragma unroll
      for (int li = 0; li < LPW; ++li) {
        v[li] = gam[li][h];
        if constexpr (!CT) v[li] = cmul_fma(v[li], pfl[nv % F::NMU * S + NW * li + wave]);
      }
      dft_plain<LPW>(v);
      if (F::NCOL == 16 || nv < F::NCOL) {
        double2 *gr = G + (F::NCOL * (F::NH == 2 ? gv : 4 * h + gv) + nv) * GP + wave;
        gr[0] = v[0];
#pragma unroll
        for (int s1 = 1; s1 < LPW; ++s1) gr[s1 * NW] = cmul_fma(v[s1], tw[(wave * s1) % S]);
      }
    }
  };
  // ... and NW-point DFTs out of G to HBM.  `wait` runs before the first stores.
  auto get = [&](int rd, long tile, auto wait) __attribute__((always_inline)) {
    const int jrem = (int)min((long)F::TJ, nJ - tile * F::TJ);  // the last tile may hold fewer row groups
    int tv = tid;
    asm volatile("" : "+v"(tv));
    const long R0 = tile * F::GR;
#pragma unroll
    for (int c = 0; c < F::NC; ++c) {
      const int e = tv + c * F::T;
      const int r = e % F::GRH, s1 = e / F::GRH;
      double2 u[NW];
      const bool on = (c + 1) * F::T <= F::NTASK || e < F::NTASK;
      if (on) {
#pragma unroll
        for (int w = 0; w < NW; ++w) u[w] = G[r * GP + s1 * NW + w];
        dft_plain<NW>(u);
      }
      if (c == 0) wait();
      if (on && (rd * F::GRH + r) / F::NMU < jrem) {
#pragma unroll
        for (int s2 = 0; s2 < NW; ++s2)
          __builtin_nontemporal_store(gd2{u[s2].x, u[s2].y},
                                      atg + (long)(s1 + LPW * s2) * Mh + R0 + rd * F::GRH + r);
      }
    }
  };
  typedef std::integral_constant<int, 0> zero;
  // The loads of the next tile's first group (issued before this tile's last product) are waited for
  // before the stores are issued, so that the wait does not cover them.
  auto epilogue = [&](long tile) __attribute__((always_inline)) {
#pragma unroll
    for (int rd = 0; rd < F::NH; ++rd) {
      put(rd);
      lds_barrier();
      get(rd, tile, [&]() __attribute__((always_inline)) { if (rd == 0) wait_loads(zero{}); });
      lds_barrier();  // G is free; after the last round the next tile's rows are complete too
    }
  };

  // One tile, its group 0 in buffer BUF.
  //
  // Two buffers: the next group's rows load while a group is multiplied.
  //
  // Four (QUAD): rows load three groups ahead, and a group's end waits for the next group's rows only:
  // the two groups loaded after them stay in flight, and so do the stores of a tile that were issued
  // since (the waves that store issue all NW of them, but for the last tile of all, which nothing
  // follows).  One barrier a group: the last one also covers G, which the next tile's put, a barrier
  // or more later, overwrites; a wave that has stored goes on to the next product by itself.
  constexpr int NL = F::NLD;
  const bool stores = wave * 64 < F::NTASK;
  auto body = [&](long tile, auto buf_tag) __attribute__((always_inline)) {
    constexpr int BUF = decltype(buf_tag)::value;
    // an opaque table address (in the global address space, or the loads would wait for LDS too):
    // the loads are the same in every tile, and hoisted out of the loop they would not fit the
    // registers
    asm volatile("" : "+s"(wbase));
    auto group = [&](auto gr_tag) __attribute__((always_inline)) {
      constexpr int gr = decltype(gr_tag)::value, cur = (BUF + gr) % F::NBUF;
      if constexpr (F::QUAD) {
        // past the block's last tile its rows again, so that the counts below hold
        dma(rows_buf((cur + 3) % 4), min(tile + (gr + 3) / NGRP * step, t1), (gr + 3) % NGRP);
        mul(rows_buf(cur), gr_tag);
        if constexpr (gr == NGRP - 1) put(0);
        // the stores of the tile before came after the next rows' loads in groups 0 and 1
        if (gr < 2 && stores && tile > t0) wait_loads(std::integral_constant<int, 2 * NL + F::NC * NW>{});
        else wait_loads(std::integral_constant<int, 2 * NL>{});
        lds_barrier();
        if constexpr (gr == NGRP - 1) get(0, tile, []() {});
      } else {
        if constexpr (gr + 1 < NGRP) dma(rows_buf(cur ^ 1), tile, gr + 1);
        else if (tile < t1) dma(rows_buf(cur ^ 1), tile + step, 0);
        mul(rows_buf(cur), gr_tag);
        if constexpr (gr + 1 < NGRP) {
          wait_loads(zero{});  // the next group's rows
          lds_barrier();
        }
      }
    };
    group(std::integral_constant<int, 0>{});
    if constexpr (NGRP > 1) group(std::integral_constant<int, 1>{});
    if constexpr (NGRP > 2) {
      group(std::integral_constant<int, 2>{});
      group(std::integral_constant<int, 3>{});
    }
    if constexpr (!F::QUAD) epilogue(tile);
  };

  wait_loads(zero{});
  lds_barrier();
  if constexpr (NGRP % F::NBUF == 0) {  // a tile ends in the buffer it began with
    for (long tile = t0; tile <= t1; tile += step) body(tile, zero{});
  } else {
    for (long tile = t0; tile <= t1; tile += 2 * step) {
      body(tile, zero{});
      if (tile < t1) body(tile + step, std::integral_constant<int, NGRP>{});
    }
  }
  if constexpr (F::QUAD) wait_loads(zero{});  // no load may outlive the block's LDS
}

// B operand table (see k_filter_g): column col = lane % 16 = theta + n_mu D, k = 4 ks + lane / 16,
// t = taps[(theta*S + i)*BPAD + k - d D], zero outside
template <typename F>
__global__ void k_filter_g_table(const double *__restrict__ taps, double2 *__restrict__ wt, int BPAD)
{
  constexpr int NIT = F::CT ? F::NK : F::NK / 2;
  const int total = F::S * NIT * 64;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < total; e += gridDim.x * blockDim.x) {
    const int lane = e % 64, it = e / 64 % NIT, i = e / (64 * NIT);
    const int col = lane % 16, theta = col % F::NMU, D = col / F::NMU;
    auto tap = [&](int ks, int im) -> double {
      const int bb = 4 * ks + lane / 16 - F::DMU * D;
      if (col >= F::NCOL || bb < 0 || bb >= BPAD) return 0.0;
      const long at = ((long)theta * F::S + i) * BPAD + bb;
      return F::CT ? taps[2 * at + im] : taps[at];
    };
    wt[e] = F::CT ? double2{tap(it, 0), tap(it, 1)} : double2{tap(2 * it, 0), tap(2 * it + 1, 0)};
  }
}

template <typename F> static int filter_g_launch(const SoiFilterArgs *a, hipStream_t st)
{
  if (F::MIN_M > a->M) return (int)hipErrorInvalidValue;
  const long ntiles = (a->nJ + F::TJ - 1) / F::TJ;
  // one round of blocks (eight waves a CU); a batch shares about two rounds over its members
  const long per_cu = 8 / F::NW;
  long nb = a->b.n > 1 ? (512 * per_cu + a->b.n - 1) / a->b.n : 256 * per_cu;
  if (nb > ntiles) nb = ntiles;
  const int tpb = (int)((ntiles + nb - 1) / nb);
  // four row buffers where blocks walk more than two tiles (S = 32, N = 2^21: 33.5 -> 32.8 us; two tiles,
  // N = 2^20: 24 with two buffers, 28 with four); the same bits either way
  if constexpr (!F::QUAD && F::RES && !F::CT && F::S == 32) {
    using Q = FilterG<F::S, F::NMU, F::DMU, F::NK, F::CT, true>;
    if (tpb > 2 && Q::MIN_M <= a->M) return filter_g_launch<Q>(a, st);
  }
  if (!F::QUAD) nb = (ntiles + tpb - 1) / tpb;
  hipLaunchKernelGGL(k_filter_g<F>, dim3((unsigned)nb, a->b.n > 0 ? a->b.n : 1), dim3(F::T), 0, st,
                     (const double2 *)a->x, (double2 *)a->at, (const double2 *)a->wt,
                     (const double2 *)a->post, (const double2 *)a->twS, a->M, a->Mh, a->nJ, tpb, a->b);
  return (int)hipGetLastError();
}

template <typename F> static int filter_g_table(const double *taps, void *wt, int BPAD, hipStream_t st)
{
  hipLaunchKernelGGL(k_filter_g_table<F>, dim3(64), dim3(256), 0, st, taps, (double2 *)wt, BPAD);
  return (int)hipGetLastError();
}

}  // namespace soi
