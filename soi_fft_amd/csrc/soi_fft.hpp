// soi_fft.hpp -- register-resident segment FFT passes of the SOI FFT on MI355X (reference: the
// DFTI transform pfft.c:227-228 runs at pfft.c:642, then the demodulation pfft.c:649-693).
//
// Four-step split M_hat = n1 * n2, R = n2*r1 + r2, m = m1 + n1*m2:
//   pass 1 (columns): for each column r2, Z[r2][m1] = sum_r1 x[n2 r1 + r2] w_n1^{r1 m1}, times the
//                     twiddle w_Mhat^{r2 m1};
//   pass 2 (rows):    y[m1 + n1 m2] = sum_r2 Z[r2][m1] w_n2^{r2 m2}, demodulated and stored as
//                     X[s*M + m] = W_inv[m] * y[m] for m < M.
// Short segments (k_fft_one) take one pass, one segment per block.
//
// What bounds the passes and what the layout follows from (copy kernels with the passes' access
// patterns, 2.68 GB in and out): columns of 64-byte runs reach 5.1 TB/s and 128-byte runs no
// more, 32-byte runs 3.8; row stores need 128-byte runs (5.2 TB/s; 64-byte runs 3.8).  A block
// holds its whole tile in LDS and registers, so what it does between its loads and its stores
// (LDS exchanges, butterflies) is time its CU does not load or store unless another block is
// resident.  Hence two or three stages of large radices per transform, each stage's butterflies
// spread over the threads as they come (the last round of a stage may leave threads idle):
// 2560 = 16.16.10 on 160 threads exchanges twice where 10.4.4.4.4 on 128 exchanged four times.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "soi_common.hpp"
#include "soi_kernels.h"

namespace soi {

// ---------------------------------------------------------------------------------------------
// forward DFTs in registers beyond those of soi_common.hpp
// ---------------------------------------------------------------------------------------------
template <typename C> __device__ __forceinline__ void dft16(C *a)
{
  typedef decltype(a[0].x) T;
  // 16 = 4 x 4: columns n = n1 + 4 n2, first DFT4 over n2, twiddle w16^{n1 k2}, DFT4 over n1
  C b[16];
#pragma unroll
  for (int n1 = 0; n1 < 4; ++n1) {
    C x0 = a[n1], x1 = a[n1 + 4], x2 = a[n1 + 8], x3 = a[n1 + 12];
    dft4(x0, x1, x2, x3);
    b[n1 * 4 + 0] = x0;
    b[n1 * 4 + 1] = x1;
    b[n1 * 4 + 2] = x2;
    b[n1 * 4 + 3] = x3;
  }
  const T c1 = (T)0.92387953251128675613, s1 = (T)0.38268343236508977173;
  const T r2 = (T)0.70710678118654752440;
  // twiddles w16^{n1 k2} = e^{-2 pi i n1 k2 / 16}
  // n1 = 1: k2 = 1,2,3 -> w^1, w^2, w^3 ; n1 = 2: w^2, w^4, w^6 ; n1 = 3: w^3, w^6, w^9
  const C w1 = C{c1, -s1}, w2 = C{r2, -r2}, w3 = C{s1, -c1};
  const C w6 = C{-r2, -r2}, w9 = C{-c1, s1};
  b[1 * 4 + 1] = cmul(b[5], w1);
  b[1 * 4 + 2] = cmul(b[6], w2);
  b[1 * 4 + 3] = cmul(b[7], w3);
  b[2 * 4 + 1] = cmul(b[9], w2);
  b[2 * 4 + 2] = cmul_mi(b[10]);
  b[2 * 4 + 3] = cmul(b[11], w6);
  b[3 * 4 + 1] = cmul(b[13], w3);
  b[3 * 4 + 2] = cmul(b[14], w6);
  b[3 * 4 + 3] = cmul(b[15], w9);
#pragma unroll
  for (int k2 = 0; k2 < 4; ++k2) {
    C x0 = b[0 * 4 + k2], x1 = b[1 * 4 + k2], x2 = b[2 * 4 + k2], x3 = b[3 * 4 + k2];
    dft4(x0, x1, x2, x3);
    // output k = k2 + 4 k1
    a[k2 + 0] = x0;
    a[k2 + 4] = x1;
    a[k2 + 8] = x2;
    a[k2 + 12] = x3;
  }
}

template <typename C> __device__ __forceinline__ void dft9(C *a)
{
  typedef decltype(a[0].x) T;
  // 9 = 3 x 3: n = n1 + 3 n2, DFT3 over n2, twiddle w9^{n1 k2}, DFT3 over n1; k = k2 + 3 k1
  const C w1 = C{(T)0.76604444311897803520, (T)-0.64278760968653932632};
  const C w2 = C{(T)0.17364817766693034885, (T)-0.98480775301220805937};
  const C w4 = C{(T)-0.93969262078590838405, (T)-0.34202014332566873304};
#pragma unroll
  for (int n1 = 0; n1 < 3; ++n1) dft3(a[n1], a[n1 + 3], a[n1 + 6]);
  a[4] = cmul(a[4], w1);
  a[7] = cmul(a[7], w2);
  a[5] = cmul(a[5], w2);
  a[8] = cmul(a[8], w4);
  // column k2 holds a[3 k2 + n1]; its outputs go to k2 + 3 k1
  C b[9];
#pragma unroll
  for (int k2 = 0; k2 < 3; ++k2) {
    C x0 = a[3 * k2], x1 = a[3 * k2 + 1], x2 = a[3 * k2 + 2];
    dft3(x0, x1, x2);
    b[k2] = x0, b[k2 + 3] = x1, b[k2 + 6] = x2;
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) a[k] = b[k];
}

template <int R, typename C> __device__ __forceinline__ void dft_any(C *a);

// inverse of x modulo m (coprime, small)
constexpr int inv_mod(int x, int m)
{
  for (int i = 1; i < m; ++i)
    if (x * i % m == 1) return i;
  return 1;
}

// N = A * B with A and B coprime: the Good-Thomas index maps n = B a + A b (mod N) and
// k = B (B^-1 mod A) ka + A (A^-1 mod B) kb (mod N) make the A- and B-point DFTs independent, with no
// twiddles between them.
template <int A, int B, typename C> __device__ __forceinline__ void dft_coprime(C *v)
{
  constexpr int N = A * B, KA = B * inv_mod(B % A, A) % N, KB = A * inv_mod(A % B, B) % N;
  C t[B][A];
#pragma unroll
  for (int b = 0; b < B; ++b) {
#pragma unroll
    for (int a = 0; a < A; ++a) t[b][a] = v[(B * a + A * b) % N];
    dft_any<A>(t[b]);
  }
#pragma unroll
  for (int a = 0; a < A; ++a) {
    C u[B];
#pragma unroll
    for (int b = 0; b < B; ++b) u[b] = t[b][a];
    dft_any<B>(u);
#pragma unroll
    for (int b = 0; b < B; ++b) v[(KA * a + KB * b) % N] = u[b];
  }
}

template <int R, typename C> __device__ __forceinline__ void dft_any(C *a)
{
  if constexpr (R == 6) dft_coprime<2, 3>(a);
  else if constexpr (R == 9) dft9(a);
  else if constexpr (R == 10) dft_coprime<2, 5>(a);
  else if constexpr (R == 12) dft_coprime<4, 3>(a);
  else if constexpr (R == 15) dft_coprime<3, 5>(a);
  else if constexpr (R == 16) dft16(a);
  else if constexpr (R == 18) dft_coprime<2, 9>(a);
  else if constexpr (R == 20) dft_coprime<4, 5>(a);
  else dft_r<R>(a);
}

// ---------------------------------------------------------------------------------------------
// The same operations with every fused multiply-add written out, the way the compiler contracts
// soi_common.hpp's forms in the LDS transform: for results that do not depend on what surrounds them.
// ---------------------------------------------------------------------------------------------
namespace pinned {
#pragma clang fp contract(off)
__device__ __forceinline__ float fm(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
  return float2{fm(a.x, b.x, -(a.y * b.y)), fm(a.y, b.x, a.x * b.y)};
}
// ... the pass-1 twiddle: the other product of the imaginary part is the rounded one
__device__ __forceinline__ float2 cmul_t(float2 a, float2 t)
{
  return float2{fm(a.x, t.x, -(a.y * t.y)), fm(a.x, t.y, a.y * t.x)};
}
__device__ __forceinline__ void dft3(float2 *a)
{
  const float h = 0.86602540378443864676f;
  const float2 t = cadd(a[1], a[2]), d = csub(a[1], a[2]);
  const float2 m = float2{fm(-0.5f, t.x, a[0].x), fm(-0.5f, t.y, a[0].y)};
  a[0] = cadd(a[0], t);
  a[1] = float2{fm(h, d.y, m.x), fm(-h, d.x, m.y)};
  a[2] = float2{fm(-h, d.y, m.x), fm(h, d.x, m.y)};
}
__device__ __forceinline__ void dft5(float2 *a)
{
  const float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;
  const float s1 = 0.95105651629515357212f, s2 = 0.58778525229247312917f;
  const float2 b1 = cadd(a[1], a[4]), b2 = cadd(a[2], a[3]);
  const float2 d1 = csub(a[1], a[4]), d2 = csub(a[2], a[3]), x0 = a[0];
  const float2 p1 = float2{fm(c2, b2.x, fm(c1, b1.x, x0.x)), fm(c2, b2.y, fm(c1, b1.y, x0.y))};
  const float2 p2 = float2{fm(c1, b2.x, fm(c2, b1.x, x0.x)), fm(c1, b2.y, fm(c2, b1.y, x0.y))};
  const float2 q1 = float2{fm(s2, d2.x, s1 * d1.x), fm(s2, d2.y, s1 * d1.y)};
  const float2 q2 = float2{fm(s2, d1.x, -(s1 * d2.x)), fm(s2, d1.y, -(s1 * d2.y))};
  a[0] = cadd(cadd(x0, b1), b2);
  a[1] = float2{p1.x + q1.y, p1.y - q1.x};
  a[4] = float2{p1.x - q1.y, p1.y + q1.x};
  a[2] = float2{p2.x + q2.y, p2.y - q2.x};
  a[3] = float2{p2.x - q2.y, p2.y + q2.x};
}
__device__ __forceinline__ void dft8(float2 *a)
{
  const float r = 0.70710678118654752440f;
  dft4(a[0], a[2], a[4], a[6]);
  dft4(a[1], a[3], a[5], a[7]);
  const float2 e0 = a[0], e1 = a[2], e2 = a[4], e3 = a[6], o0 = a[1], o2 = cmul_mi(a[5]);
  const float s1 = a[3].x + a[3].y, d1 = a[3].y - a[3].x, d3 = a[7].y - a[7].x, s3 = a[7].x + a[7].y;
  a[0] = cadd(e0, o0);
  a[4] = csub(e0, o0);
  a[1] = float2{fm(r, s1, e1.x), fm(r, d1, e1.y)};
  a[5] = float2{fm(-r, s1, e1.x), fm(-r, d1, e1.y)};
  a[2] = cadd(e2, o2);
  a[6] = csub(e2, o2);
  a[3] = float2{fm(r, d3, e3.x), fm(-r, s3, e3.y)};
  a[7] = float2{fm(-r, d3, e3.x), fm(r, s3, e3.y)};
}
template <int R> __device__ __forceinline__ void dft_any(float2 *a)
{
  if constexpr (R == 3) dft3(a);
  else if constexpr (R == 5) dft5(a);
  else if constexpr (R == 8) dft8(a);
  else dft_r<R>(a);  // 2, 4: additions only
}
}  // namespace pinned

// by FORM (see Sched): products and DFTs as the compiler fuses them, or pinned
template <int FORM, typename C> __device__ __forceinline__ C cmul_as(C a, C b)
{
  if constexpr (FORM == 0) return cmul(a, b);
  else return pinned::cmul(a, b);
}
template <int FORM, int R, typename C> __device__ __forceinline__ void dft_as(C *a)
{
  if constexpr (FORM == 0) dft_any<R>(a);
  else pinned::dft_any<R>(a);
}

// ---------------------------------------------------------------------------------------------
// compile-time schedule of one transform: L points, TS threads per sequence, radices in stage
// order.  Stage s has L/R butterflies; thread ts takes butterflies ts, ts + TS, ...
// ---------------------------------------------------------------------------------------------
//
// A stage may be a chain of radices that run one after the other in registers: two decimal digits
// for each, the first in front (20503 = radix 2, then 5, then 3: 30 values, all twiddles of the
// three stages from the table).  FORM says how twiddles are made and which DFTs are used:
//   0: see chain; products of coprime factors without twiddles;
//   2: every twiddle from the table, as soi_common.hpp's LDS transform does.
// ---------------------------------------------------------------------------------------------
constexpr int code_prod(int c) { return c < 100 ? c : c % 100 * code_prod(c / 100); }
constexpr int code_first(int c) { return c < 100 ? c : code_first(c / 100); }
constexpr int code_rest(int c) { return c < 100 ? 0 : c % 100 + 100 * code_rest(c / 100); }

template <int L_, int TS_, int... Rs> struct Sched {
  static constexpr int L = L_, TS = TS_, n = sizeof...(Rs), FORM = 0;
  static constexpr int r[n] = {Rs...};
  static constexpr int code(int s) { return r[s]; }
  static constexpr int at(int s) { return code_prod(r[s]); }
  static constexpr int span(int s)  // product of radices before stage s
  {
    int p = 1;
    for (int i = 0; i < s; ++i) p *= at(i);
    return p;
  }
  static constexpr int nb(int s) { return L / at(s); }                     // butterflies
  static constexpr int nc(int s) { return (nb(s) + TS - 1) / TS; }         // rounds per thread
  static constexpr int e()                                                 // values per thread
  {
    int m = 0;
    for (int s = 0; s < n; ++s)
      if (nc(s) * at(s) > m) m = nc(s) * at(s);
    return m;
  }
  static constexpr int E = e();
  static_assert(span(n) == L, "radices do not multiply to L");
  // the same transform on at most N threads
  template <int N> using Cap = Sched<L_, (TS_ < N ? TS_ : N), Rs...>;
};
template <int F, typename SC> struct WithForm : SC { static constexpr int FORM = F; };

// LDS position of element pos of a sequence.  The first stage's threads write R0 positions apart.
// When R0 is a power of two those fall on the same banks, unless a position covers all of them
// (T elements of `es` bytes, 256 bytes of banks): the low bits are XORed with the bits above the
// radix (a bijection within runs of R0, so the tile fills LDS exactly).  Positions base + k D
// with D a multiple of R0 then lie at one of MB swizzled bases plus k D, so that an access costs no
// address arithmetic: at(x, i) is the base of x for i = k D / R0 (mod MB).
constexpr int log2_of(int x) { return x <= 1 ? 0 : 1 + log2_of(x / 2); }
template <typename SC, int T, int es> struct Swz {
  static constexpr int R0 = SC::at(0);
  static constexpr bool ON = (R0 & (R0 - 1)) == 0 && R0 >= 4 && T * es < 256;
  static constexpr int MB = !ON ? 1 : T * es >= 128 ? 2 : 4;
  static constexpr int SH = log2_of(R0);
  static __device__ __forceinline__ int at(int x, int i)
  {
    if constexpr (ON) return x ^ (((x >> SH) + i) & (MB - 1));
    return x;
  }
};

// Exchange stage S0's outputs through LDS into stage S0 + 1's input order: outputs of butterfly j
// (radix R, span NS) land at (j - j%NS)*R + j%NS + k*NS; butterfly j2 of the next stage reads
// j2 + k*L/R2.  FULL: whole complex values in one round; otherwise the real and the imaginary
// halves in turn, in half the LDS.
template <typename SC, int T, int S0, bool FULL, typename C>
__device__ __forceinline__ void exchange(C (&v)[SC::E], unsigned char *lds, int q, int ts)
{
  constexpr int L = SC::L, TS = SC::TS;
  constexpr int R = SC::at(S0), NS = SC::span(S0), NB = SC::nb(S0), NC = SC::nc(S0);
  constexpr int R2 = SC::at(S0 + 1), NB2 = SC::nb(S0 + 1), NC2 = SC::nc(S0 + 1), D = L / R2;
  constexpr bool LAST = S0 + 2 == SC::n;  // nothing is written to LDS after the last exchange
  using E = typename std::conditional<FULL, C, real_t<C>>::type;
  using X = Swz<SC, T, (int)sizeof(E)>;
  constexpr int MB = X::MB;
  E *l = reinterpret_cast<E *>(lds) + q;
#pragma unroll
  for (int half = 0; half < (FULL ? 1 : 2); ++half) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int j = ts + TS * c;
      if ((c + 1) * TS <= NB || j < NB) {
        E *p[MB];
        if constexpr (NS == 1) {  // positions R j + k: k's low bits XOR j's
#pragma unroll
          for (int i = 0; i < MB; ++i) p[i] = l + (R * j + (i ^ (j & (MB - 1)))) * T;
        } else {
          const int jm = j % NS;
          const int base = (j - jm) * R + jm;
#pragma unroll
          for (int i = 0; i < MB; ++i) p[i] = l + X::at(base, i) * T;
        }
#pragma unroll
        for (int k = 0; k < R; ++k) {
          E *w = NS == 1 ? p[k & (MB - 1)] + (k & ~(MB - 1)) * T
                         : p[(k * NS >> X::SH) & (MB - 1)] + k * NS * T;
          if constexpr (FULL) *w = v[c * R + k];
          else *w = half ? v[c * R + k].y : v[c * R + k].x;
        }
      }
    }
    lds_barrier();
#pragma unroll
    for (int c = 0; c < NC2; ++c) {
      const int j = ts + TS * c;
      if ((c + 1) * TS <= NB2 || j < NB2) {
        const E *p[MB];
#pragma unroll
        for (int i = 0; i < MB; ++i) p[i] = l + X::at(j, i) * T;
#pragma unroll
        for (int k = 0; k < R2; ++k) {
          const E val = p[(k * D >> X::SH) & (MB - 1)][k * D * T];
          if constexpr (FULL) v[c * R2 + k] = val;
          else if (half) v[c * R2 + k].y = val;
          else v[c * R2 + k].x = val;
        }
      }
    }
    if (!LAST || (!FULL && half == 0)) lds_barrier();
  }
}

constexpr int odd_part(int x) { return x % 2 ? x : odd_part(x / 2); }

// The radices of CODE on the values v of one butterfly: input k is position j + k*L/R, output k goes to
// position k*NS of the butterfly's outputs, jm = j % NS.  The first radix R1 of the chain has R/R1
// butterflies with the same jm; its output k continues, by itself, with jm + k*NS at span NS*R1.
// Twiddles w^k: FORM 2 reads each from the table.  FORM 0 reads those with k < 4 or k % 4 == 0 and forms the
// others as one product of two of them (radix 16: six reads instead of 15).  Products of all of k's
// bits, up to three of them, cost 4 to 8% of a complex128 pass's error (512-point rows 1.98e-16 ->
// 2.14e-16, now 1.98e-16).  Complex128 of 2^a < 2048 points reads all up to radix 8 (512-point rows with products
// of two 2.08e-16); at 2048 those loads cost 6% of a whole transform (N = 2^27, S = 32; 8% at 2^24, S = 8), and
// other lengths are as close with products (3 to 6% of the time of N = 45*2^16 and 9*2^19).  Complex64 waits for
// loads more: reading all costs 0 to 8% of a transform (N = 2^23, S = 32 161 -> 167 us, 2^26 1309 -> 1491) for 1 to
// 4% of its error (3*2^22, S = 8 2.96e-7 -> 2.84e-7).
template <int FORM, int L, int NS, int CODE, typename C>
__device__ __forceinline__ void chain(C *v, int jm, const C *__restrict__ tw)
{
  constexpr int R1 = code_first(CODE), REST = code_rest(CODE), M = REST ? code_prod(REST) : 1;
  constexpr int step = L / (NS * R1);
  constexpr bool ALL = FORM == 2 || (sizeof(C) == 16 && R1 <= 8 && odd_part(L) == 1 && L < 2048);
  C w[R1];
  if constexpr (NS > 1) {
#pragma unroll
    for (int k = 1; k < R1; ++k) {
      if (ALL || k % 4 == 0 || k < 4) w[k] = tw[k * jm * step];
      else w[k] = cmul_as<FORM>(w[k & ~3], w[k & 3]);
    }
  }
  C u[R1][M];
#pragma unroll
  for (int i = 0; i < M; ++i) {
    C a[R1];
#pragma unroll
    for (int k = 0; k < R1; ++k) a[k] = v[i + k * M];
    if constexpr (NS > 1) {
#pragma unroll
      for (int k = 1; k < R1; ++k) a[k] = cmul_as<FORM>(a[k], w[k]);
    }
    dft_as<FORM, R1>(a);
#pragma unroll
    for (int k = 0; k < R1; ++k) u[k][i] = a[k];
  }
#pragma unroll
  for (int k = 0; k < R1; ++k) {
    if constexpr (REST != 0) chain<FORM, L, NS * R1, REST>(u[k], jm + k * NS, tw);
#pragma unroll
    for (int i = 0; i < M; ++i) v[k + R1 * i] = u[k][i];
  }
}

// twiddle + DFT of every butterfly of stage S0 held in registers
template <typename SC, int S0, typename C>
__device__ __forceinline__ void stage(C (&v)[SC::E], int ts, const C *__restrict__ tw)
{
  constexpr int TS = SC::TS, R = SC::at(S0), NS = SC::span(S0), NB = SC::nb(S0), NC = SC::nc(S0);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int j = ts + TS * c;
    if ((c + 1) * TS <= NB || j < NB)
      chain<SC::FORM, SC::L, NS, SC::code(S0)>(&v[c * R], NS > 1 ? j % NS : 0, tw);
  }
}

// Run stages S0 .. n-1 on register data already in stage S0's input order.
template <typename SC, int T, bool FULL, int S0, typename C>
__device__ __forceinline__ void run_stages(C (&v)[SC::E], unsigned char *lds, int q, int ts,
                                           const C *__restrict__ tw)
{
  stage<SC, S0, C>(v, ts, tw);
  if constexpr (S0 + 1 < SC::n) {
    exchange<SC, T, S0, FULL, C>(v, lds, q, ts);
    run_stages<SC, T, FULL, S0 + 1, C>(v, lds, q, ts, tw);
  }
}
// After the last stage (span L/R), value v[c*R + k] of butterfly j = ts + TS*c is output index
// j + k*L/R.

// ---------------------------------------------------------------------------------------------
// launch shapes
// ---------------------------------------------------------------------------------------------
template <typename SC, int T, bool FULL, typename C> constexpr size_t fft_lds()
{
  return SC::n > 1 ? (size_t)SC::L * T * (FULL ? sizeof(C) : sizeof(real_t<C>)) : 0;
}
// Waves per SIMD the register budget is sized for: as many blocks as LDS holds, unless their
// values do not fit that many times (512 registers a SIMD lane; about 72 beside the values)
template <typename SC, int T, bool FULL, typename C> constexpr int fft_minw()
{
  const int threads = T * SC::TS, waves = (threads + 63) / 64;
  const size_t lds = fft_lds<SC, T, FULL, C>();
  int blocks = lds ? (int)(160 * 1024 / lds) : 8;
  const int regs = SC::E * (int)(sizeof(C) / 4) + 72;
  while (blocks > 1 && (blocks * waves + 3) / 4 * regs > 512) --blocks;
  const int w = (blocks * waves + 3) / 4;
  return w > 8 ? 8 : w;
}

// Rows per tile of the complex64 pass-1 output: element (m1, r2) of a segment at
// ((m1/TR)*n2 + r2)*TR + m1%TR.  With eight, the eight m1 by eight r2 that a wave of the column
// pass stores are one run of 512 bytes, and a row block reads two tiles in runs of 64 bytes that
// are adjacent from lane group to lane group.
constexpr int TR = 8;

// Load / store at a uniform base plus 32-bit per-thread byte offset: one address register serves
// all accesses of a butterfly, whose bases differ by uniform strides
template <typename C> __device__ __forceinline__ C ld_at(const C *base, unsigned off)
{
  return *reinterpret_cast<const C *>(reinterpret_cast<const char *>(base) + off);
}
template <typename C> __device__ __forceinline__ void st_at(C *base, unsigned off, C v)
{
  *reinterpret_cast<C *>(reinterpret_cast<char *>(base) + off) = v;
}

// ---------------------------------------------------------------------------------------------
// Pass 1: T adjacent columns of L = n1 points (stride n2).  In place, or (TILED) into TR-row
// tiles of the tile buffer, whose segments are Mt values apart.  A tile past the last column (n2 % T != 0) loads column n2 - 1
// again and stores nothing there.
// ---------------------------------------------------------------------------------------------
template <typename SC, int T, bool FULL, typename C, bool TILED, int MW>
__global__ __launch_bounds__(T *SC::TS, MW) void k_fft_cols(
    C *__restrict__ data, const C *__restrict__ tw, const C *__restrict__ thi,
    const C *__restrict__ tlo, int n2, int lb1, long Mh, int S, C *__restrict__ tout, long Mt,
    SoiBatch b)
{
  constexpr int L = SC::L, TS = SC::TS;
  data = batch_ptr(data, b.at);
  if constexpr (TILED) tout = batch_ptr(tout, b.tb);
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int tid = threadIdx.x;
  const int q = tid % T, ts = tid / T;
  const int ncb = (n2 + T - 1) / T;
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int cb = bid % ncb, s = bid / ncb;
  if (s >= S) return;
  const int col = cb * T + q;
  const bool on = col < n2;
  const unsigned r2 = (unsigned)(on ? col : n2 - 1), n2s = (unsigned)n2;
  C *seg = data + (long)s * Mh;

  C v[SC::E];
  constexpr int R0 = SC::at(0);
#pragma unroll
  for (int c = 0; c < SC::nc(0); ++c) {
    const int j = ts + TS * c;
    if ((c + 1) * TS <= SC::nb(0) || j < SC::nb(0)) {
      const unsigned off = ((unsigned)j * n2s + r2) * (unsigned)sizeof(C);
#pragma unroll
      for (int k = 0; k < R0; ++k) v[c * R0 + k] = ld_at(seg + (size_t)(k * (L / R0)) * n2s, off);
    }
  }

  // FORM 2 reads a pair for each value, and the lanes' entries of the lower table lie all over it (up
  // to 64 cache lines an instruction, 60% of the L1's cycles): a copy in LDS (1440 points: 199 against
  // 226 us)
  [[maybe_unused]] C *llo = reinterpret_cast<C *>(lds_raw + fft_lds<SC, T, FULL, C>());
  if constexpr (SC::FORM == 2)
    for (int e = tid; e < 1 << lb1; e += T * TS) llo[e] = tlo[e];

  run_stages<SC, T, FULL, 0, C>(v, lds_raw, q, ts, tw);

  // twiddle w_Mhat^{r2 m1}, m1 = j + k*L/RL, from the two-level table (hi[e >> lb1] *
  // lo[e & mask], exponents below M_hat < 2^32), factored into w^{r2 j} w^{r2 k L/RL}: a thread
  // reads NC + RL - 1 table pairs instead of NC * RL (FORM 2: unfactored)
  constexpr int RL = SC::at(SC::n - 1), NC = SC::nc(SC::n - 1), NB = SC::nb(SC::n - 1);
  // Below 256 points the extra products would cost 5 to 8% of the pass's error (complex128, 64 points; unfactored
  // in as much time); above, 2 to 3% against 2 to 6% of a whole transform's time (N = 45*2^16, S = 8 89.5 us,
  // unfactored 95.0; 2^22, S = 16 126 and 131.5).  Complex64 of other odd parts than 1 and 5 stays
  // unfactored: N = 27*2^17 3.23e-7, unfactored 3.17e-7, in the same time.
  constexpr int ODD = odd_part(L);
  constexpr bool FACT = SC::FORM == 0 && L >= 256 && (sizeof(C) == 16 || ODD == 1 || ODD == 5);
  const unsigned lmask = (1u << lb1) - 1;
  if (!on) return;  // no barrier follows
  C tc[NC];
  if constexpr (FACT)
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int j = ts + TS * c;
    if ((c + 1) * TS <= NB || j < NB) {
      const unsigned ex = r2 * (unsigned)j;
      tc[c] = cmul_as<SC::FORM>(thi[ex >> lb1], tlo[ex & lmask]);
    }
  }
  C *tseg = TILED ? tout + (long)s * Mt : nullptr;
#pragma unroll
  for (int k = 0; k < RL; ++k) {
    C tk = C{1, 0};
    if (FACT && k) {
      const unsigned ex = r2 * (unsigned)(k * (L / RL));
      tk = cmul_as<SC::FORM>(thi[ex >> lb1], tlo[ex & lmask]);
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int j = ts + TS * c;
      if ((c + 1) * TS <= NB || j < NB) {
        C t;
        if constexpr (FACT) {
          t = k ? cmul_as<SC::FORM>(tc[c], tk) : tc[c];
        } else {
          const unsigned ex = r2 * (unsigned)(j + k * (L / RL));
          const C *lo = SC::FORM == 2 ? llo : tlo;
          t = cmul_as<SC::FORM>(thi[ex >> lb1], lo[ex & lmask]);
        }
        C y;
        if constexpr (SC::FORM == 2) y = pinned::cmul_t(v[c * RL + k], t);
        else y = cmul_as<SC::FORM>(v[c * RL + k], t);
        if constexpr (TILED && (L / RL) % TR == 0) {  // j + k*L/RL: k moves whole tiles
          const unsigned off = (((unsigned)j / TR * n2s + r2) * TR + (unsigned)j % TR) * (unsigned)sizeof(C);
          st_at(tseg + (size_t)(k * (L / RL)) * n2s, off, y);
        } else if constexpr (TILED) {
          const unsigned m1 = (unsigned)(j + k * (L / RL));
          tseg[(m1 / TR * n2s + r2) * TR + m1 % TR] = y;
        } else {
          const unsigned off = ((unsigned)j * n2s + r2) * (unsigned)sizeof(C);
          st_at(seg + (size_t)(k * (L / RL)) * n2s, off, y);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Pass 2: T adjacent rows of L = n2 points, demodulated.  Lanes run over the T rows first, so
// each store instruction writes runs of T consecutive m straight from registers (128 bytes at
// T = 8 complex128 and T = 16 complex64).  Rows come from the [n1][n2] layout (T runs of 128
// bytes per load instruction for complex128) or (TILED) from pass 1's tiles.
// ---------------------------------------------------------------------------------------------
template <typename SC, int T, bool FULL, typename C, bool TILED, int MW>
__global__ __launch_bounds__(T *SC::TS, MW) void k_fft_rows(
    const C *__restrict__ data, C *__restrict__ X, const C *__restrict__ tw,
    const double2 *__restrict__ winv, int n1, long Mh, long M, int S, int sg, SoiBatch b)
{
  constexpr int L = SC::L, TS = SC::TS;
  data = batch_ptr(data, TILED ? b.tb : b.at);
  X = batch_ptr(X, b.x);
  extern __shared__ __align__(16) unsigned char lds_raw[];
  const int tid = threadIdx.x;
  const int q = tid % T, ts = tid / T;
  const int nrb = (n1 + T - 1) / T;
  // order: sg segments of one row block together (they share its W_inv entries), then the next
  // row block, then the next sg segments
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int g = bid / (sg * nrb), sn = min(sg, S - g * sg), r = bid - g * sg * nrb;
  const int s = g * sg + r % sn, rb = r / sn;
  const int a = rb * T + q;
  const bool on = a < n1;
  const C *row = data + (long)s * Mh;
  const unsigned ra = (unsigned)(on ? a : n1 - 1);

  C v[SC::E];
  constexpr int R0 = SC::at(0);
#pragma unroll
  for (int c = 0; c < SC::nc(0); ++c) {
    const int j = ts + TS * c;
    if ((c + 1) * TS <= SC::nb(0) || j < SC::nb(0)) {
      const unsigned off = TILED ? ((ra / TR * L + (unsigned)j) * TR + ra % TR) * (unsigned)sizeof(C)
                                 : (ra * L + (unsigned)j) * (unsigned)sizeof(C);
#pragma unroll
      for (int k = 0; k < R0; ++k) v[c * R0 + k] = ld_at(row + k * (L / R0) * (TILED ? TR : 1), off);
    }
  }

  run_stages<SC, T, FULL, 0, C>(v, lds_raw, q, ts, tw);

  // W_inv in FP64, loaded a few at a time ahead of the stores that use them (index clamped, so
  // that the loads need no branch); more where the launch leaves each thread the registers
  // (complex64, 1536 points in blocks of 512 threads: 189 against 204 us; with less room they spill)
  constexpr int RL = SC::at(SC::n - 1), NC = SC::nc(SC::n - 1), NB = SC::nb(SC::n - 1);
  constexpr int GW = sizeof(C) == 8 && MW <= 3 ? 8 : 4;
  if (!on) return;  // no barrier follows
  C *out = X + (long)s * M;
  const unsigned Ml = (unsigned)M;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int j = ts + TS * c;
    if ((c + 1) * TS <= NB || j < NB) {
      const unsigned m0 = (unsigned)a + (unsigned)n1 * (unsigned)j;
#pragma unroll
      for (int k0 = 0; k0 < RL; k0 += GW) {
        double2 w[GW];
#pragma unroll
        for (int i = 0; i < GW && k0 + i < RL; ++i) {
          const unsigned m = m0 + (unsigned)n1 * (unsigned)((k0 + i) * (L / RL));
          w[i] = ld_at(winv, min(m, Ml - 1) * 16u);
        }
#pragma unroll
        for (int i = 0; i < GW && k0 + i < RL; ++i) {
          const unsigned m = m0 + (unsigned)n1 * (unsigned)((k0 + i) * (L / RL));
          if (m < Ml) st_at(out, m * (unsigned)sizeof(C), demod<C>(w[i], v[c * RL + k0 + i]));
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// One pass: a block transforms one segment of L = M_hat points and demodulates it.
// ---------------------------------------------------------------------------------------------
template <typename SC, typename C>
__global__ __launch_bounds__(SC::TS) void k_fft_one(const C *__restrict__ data, C *__restrict__ X,
                                                   const C *__restrict__ tw,
                                                   const double2 *__restrict__ winv, long M,
                                                   SoiBatch b)
{
  constexpr int L = SC::L, TS = SC::TS;
  data = batch_ptr(data, b.at);
  X = batch_ptr(X, b.x);
  __shared__ __align__(16) C lds[L];
  const int ts = threadIdx.x, s = blockIdx.x;
  const C *row = data + (long)s * L;
  C v[SC::E];
  constexpr int R0 = SC::at(0);
#pragma unroll
  for (int c = 0; c < SC::nc(0); ++c) {
    const int j = ts + TS * c;
    if ((c + 1) * TS <= SC::nb(0) || j < SC::nb(0)) {
#pragma unroll
      for (int k = 0; k < R0; ++k) v[c * R0 + k] = row[j + k * (L / R0)];
    }
  }
  run_stages<SC, 1, true, 0, C>(v, reinterpret_cast<unsigned char *>(lds), 0, ts, tw);
  constexpr int RL = SC::at(SC::n - 1), NC = SC::nc(SC::n - 1), NB = SC::nb(SC::n - 1);
  C *out = X + (long)s * M;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int j = ts + TS * c;
    if ((c + 1) * TS <= NB || j < NB) {
      double2 w[RL];  // W_inv, applied in FP64
#pragma unroll
      for (int k = 0; k < RL; ++k) w[k] = winv[min(j + k * (L / RL), (int)M - 1)];
#pragma unroll
      for (int k = 0; k < RL; ++k) {
        const int m = j + k * (L / RL);
        if (m < M) out[m] = demod<C>(w[k], v[c * RL + k]);
      }
    }
  }
}

}  // namespace soi

// ---------------------------------------------------------------------------------------------
// dispatch (instantiated once per precision and pass: soi_fft_{cols,rows}{64,32}.hip)
// ---------------------------------------------------------------------------------------------
#include "soi_fft_lengths.h"

namespace soi {

template <typename K> static void allow_lds(K kern, size_t lds)
{
  (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

template <typename SC, int T, bool FULL, typename C>
static int launch_cols(C *data, const C *tw, const C *thi, const C *tlo, int n2, int lb1, long Mh,
                       int S, C *tout, long Mt, SoiBatch b, hipStream_t st)
{
  constexpr bool TILED = sizeof(C) == 8;  // complex64: into the row pass's tiles
  auto kern = k_fft_cols<SC, T, FULL, C, TILED, fft_minw<SC, T, FULL, C>()>;
  constexpr size_t base = fft_lds<SC, T, FULL, C>();
  static_assert(base <= 160 * 1024 && T * SC::TS <= 1024, "tile");
  const size_t lds = base + (SC::FORM == 2 ? sizeof(C) << lb1 : 0);
  if (lds > 160 * 1024) return (int)hipErrorInvalidValue;
  static bool once = (allow_lds(kern, SC::FORM == 2 ? 160 * 1024 : base), true);
  (void)once;
  hipLaunchKernelGGL(kern, dim3((unsigned)((n2 + T - 1) / T * S), b.n > 0 ? b.n : 1),
                     dim3(T * SC::TS), lds, st, data, tw, thi, tlo, n2, lb1, Mh, S, tout, Mt, b);
  return (int)hipGetLastError();
}

template <typename SC, int T, bool FULL, typename C>
static int launch_rows(const C *data, C *X, const C *tw, const double2 *winv, int n1, long Mh,
                       long M, int S, SoiBatch b, hipStream_t st)
{
  constexpr bool TILED = sizeof(C) == 8;
  // segments of one row block that run together.  Sharing W_inv entries saves its traffic (16
  // bytes per output from the last-level cache), but segment strides that are multiples of a
  // large power of two put their stores on the same memory channels.  Measured (complex128): all
  // segments together 48 against 57 us one by one where the data stay in the last-level cache
  // (512 x 512, 32 segments); 0.58 against 0.64 ms where W_inv is 64 MB (2560 x 2048); elsewhere
  // one by one (1024 x 1024, 64 segments: 0.46 against 0.51 ms).
  // Whole transforms with up to 1, 4, 16 and 64 together, 65 shapes (N = 2^18 to 2^27, odd parts 1
  // and 3, 8 and 32 segments, one with 64, both precisions): no other number takes 3.5% less than
  // the rule's, but for four shapes below 2^20 points, where fewer together take up to 7.5% less
  // (complex64, N = 3*2^18, 8 segments: one by one 34.1 against 36.8 us).  One by one takes 3 to 4%
  // more at 2^27.
  const bool cached = (double)S * Mh * sizeof(C) <= 192e6;
  // (complex64 FORM 2, whose W_inv entries are twice its values: four together, 133 against 144 us
  // at 1024 x 960, 32 segments.)
  const int sg = SC::FORM == 2 ? (S < 4 ? S : 4)
                 : cached      ? S
                               : M >= (1L << 21) ? (S < 16 ? S : 16) : 1;
  auto kern = k_fft_rows<SC, T, FULL, C, TILED, fft_minw<SC, T, FULL, C>()>;
  constexpr size_t lds = fft_lds<SC, T, FULL, C>();
  static_assert(lds <= 160 * 1024 && T * SC::TS <= 1024, "tile");
  static bool once = (allow_lds(kern, lds), true);
  (void)once;
  hipLaunchKernelGGL(kern, dim3((unsigned)((n1 + T - 1) / T * S), b.n > 0 ? b.n : 1),
                     dim3(T * SC::TS), lds, st, data, X, tw, winv, n1, Mh, M, S, sg, b);
  return (int)hipGetLastError();
}

// Column tiles.  variant 0 is the default; 1 is an alternative that the autotuner times.
// Measured rates at 1.34 GB in, 1.34 GB out (a copy with the pattern: 5.1 - 5.7 TB/s):
//   complex128: 512 points 5.3 TB/s, 1280 points eight wide whole 4.9 (halves 4.7, four wide 3.9),
//     640 points halves 4.9 (whole 4.5: two blocks a CU instead of four), 2560 four wide whole 4.3
//     (halves 3.7; the former 10.4.4.4.4 schedule 3.8).
//   complex64 is bound by its FP32 arithmetic as much as by memory, so more, smaller blocks:
//     512 points halves 4.7 (whole 4.5), 1280 whole 4.1, 2048 halves on 64 threads 4.5 (whole 3.6),
//     2560 eight wide whole on 80 threads 3.5 (halves 3.3, four wide 3.4).
template <typename SC, typename C, typename... A> static int cols_len(int variant, A... a)
{
  constexpr int L = SC::L;
  if constexpr (sizeof(C) == 16) {
    if constexpr (L <= 200) {
      if (variant == 0) return launch_cols<SC, 16, true, C>(a...);
    } else if constexpr (L <= 640) {
      if (variant == 0) return launch_cols<SC, 8, (L <= 512), C>(a...);
    } else if constexpr (L <= 1280) {
      if (variant == 0) return launch_cols<SC, 8, true, C>(a...);
      if (variant == 1) return launch_cols<SC, 8, false, C>(a...);
    } else {
      if (variant == 0) return launch_cols<SC, 4, true, C>(a...);
      if (variant == 1) return launch_cols<SC, 4, false, C>(a...);
    }
  } else {
    if constexpr (L <= 240) {
      if (variant == 0) return launch_cols<SC, 16, true, C>(a...);
    } else if constexpr (L <= 640) {
      if (variant == 0) return launch_cols<SC, 8, false, C>(a...);
    } else if constexpr (L <= 1280) {
      if (variant == 0) return launch_cols<SC, 8, true, C>(a...);
      if (variant == 1) return launch_cols<SC, 8, false, C>(a...);
    } else {
      // 64 threads a column: two blocks of eight waves; 2560 points take 80 (40 values each)
      using SN = typename SC::template Cap<(L < 2560 ? 64 : 80)>;
      if (variant == 0) return launch_cols<SN, 8, (L == 2560), C>(a...);
      if (variant == 1) return launch_cols<SN, 8, (L < 2560), C>(a...);
    }
  }
  return (int)hipErrorInvalidValue;
}

// Row tiles: 128-byte store runs (8 rows complex128, 16 rows complex64).  Same measure:
//   complex128: 512 points 5.0 TB/s, 1024 whole 4.4 (halves 4.1: it spills), 1280 whole 4.4 (4.3),
//     2048 halves 4.1 (its whole tile does not fit);
//   complex64: 512 points halves 4.8 (whole 4.3), 1280 whole 3.2 (3.0), 2048 halves 3.5.
template <typename SC, typename C, typename... A> static int rows_len(int variant, A... a)
{
  constexpr int L = SC::L;
  if constexpr (sizeof(C) == 16) {
    if constexpr (L <= 200) {
      if (variant == 0) return launch_rows<SC, 16, true, C>(a...);
    } else if constexpr (L <= 640) {
      if (variant == 0) return launch_rows<SC, 8, (L <= 512), C>(a...);
    } else if constexpr (L <= 1280) {
      if (variant == 0) return launch_rows<SC, 8, true, C>(a...);
      if (variant == 1) return launch_rows<SC, 8, false, C>(a...);
    } else if constexpr (L <= 2048) {
      if (variant == 0) return launch_rows<SC, 8, false, C>(a...);
    } else {
      if (variant == 0) return launch_rows<SC, 4, true, C>(a...);
    }
  } else {
    using SN = typename SC::template Cap<64>;
    if constexpr (L <= 640) {
      if (variant == 0) return launch_rows<SN, 16, (L <= 240), C>(a...);
    } else if constexpr (L <= 1280) {
      if (variant == 0) return launch_rows<SN, 16, true, C>(a...);
      if (variant == 1) return launch_rows<SN, 16, false, C>(a...);
    } else if constexpr (L <= 2048) {
      if (variant == 0) return launch_rows<SN, 16, false, C>(a...);
    } else {
      if (variant == 0) return launch_rows<typename SC::template Cap<80>, 8, true, C>(a...);
    }
  }
  return (int)hipErrorInvalidValue;
}

#define SOI_X(L, ...) \
  case L: return cols_len<Sched<L, __VA_ARGS__>, C>(variant, a...);
template <typename C, typename... A> static int cols_any(int n1, int variant, A... a)
{
  switch (n1) {
    SOI_FFT_SHORT(SOI_X) SOI_FFT_LONG(SOI_X) SOI_FFT_LONGEST(SOI_X)
    default: return (int)hipErrorInvalidValue;
  }
}
#undef SOI_X
#define SOI_X(L, ...) \
  case L: return rows_len<Sched<L, __VA_ARGS__>, C>(variant, a...);
template <typename C, typename... A> static int rows_any(int n2, int variant, A... a)
{
  switch (n2) {
    SOI_FFT_SHORT(SOI_X) SOI_FFT_LONG(SOI_X) SOI_FFT_LONGEST(SOI_X)
    default: return (int)hipErrorInvalidValue;
  }
}
#undef SOI_X

}  // namespace soi
