// soi_kernels.hip -- MI355X (gfx950) kernels of the SOI FFT hot path and their C-ABI launchers.
//
// Data layout in HBM (one GPU, P virtual ranks, S = k*P segments):
//   input  alpha[q][i]            q < M rows, i < S lanes (the natural-order N-vector)
//   alpha_tilde[s][R]             s < S segments, R < M_hat (segment-major: the reference's
//                                 all-to-all, pfft.c:553-578, is the identity in this layout)
//   output X[s*M + m]             written over alpha (in place, as the reference does)
//
// Stages (reference -> here):
//   Step 1  parallel_filter_subsampling.cpp:134-524  -> k_filter_sdft   (conv + S-point DFT)
//   Step 2  exchange pfft.c:474-583                  -> identity (layout) / VLC codec kernels
//   Step 3  pfft.c:642 DFTI M_hat-point              -> k_fft_single or k_fft_col + k_fft_row
//           pfft.c:649-693 demodulation              -> fused into the last FFT pass's store
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <math.h>
#include "soi_common.hpp"
#include "soi_kernels.h"

using namespace soi;

// =============================================================================================
// Tables (init only; FP64 on the GPU)
// =============================================================================================

// sin and cos of pi num/den, the rounding of the quotient made good: a quotient near 1 is off by up to
// 5e-17, the angle by 1.7e-16, more than the rounding of the entry itself
__device__ __forceinline__ void sincospi_ratio(long num, long den, double *sn, double *cs)
{
  long r = num % (2 * den);
  if (r < -den) r += 2 * den;
  else if (r >= den) r -= 2 * den;
  const double hi = (double)r / (double)den;
  const double lo = M_PI * (fma(-hi, (double)den, (double)r) / (double)den);
  double s0, c0;
  sincospi(hi, &s0, &c0);
  *sn = fma(c0, lo, s0);
  *cs = fma(-s0, lo, c0);
}

// Filter taps and phase factors.  The reference window (pfft.c:42-66) is
//   w[theta][b][i] = e^{i pi t} y(t) / mu,  t = theta*d/n - b - i/S + kappa/2,
//   y(t) = sin(pi tau t)/(pi tau t) * exp(-pi^2 t^2 / sigma), y(0) = 1.
// ref = 1: t as the reference forms it in double, ((double)theta/M_hat - (double)j/N +
//          (double)kappa/(2M))*M with j = b*S + i (no contraction), so the table reproduces the
//          reference's window values; ref = 0: t from its exact rational numerator over 2nS.
// ct = 0 (real taps, exact t only): e^{i pi t} = e^{i pi (t+b)} (-1)^b, so
//          w = post[theta][i] * taps[theta][i][b], taps = (-1)^b y(t)/mu real,
//          post = e^{i pi (theta d/n + kappa/2 - i/S)}.
// ct = 1: taps[theta][i][b] = w (complex), post = 1.
// w_full receives w in the reference's logical layout [theta][b][i] (descriptor field w).

// y(t)/mu for t = num/den, rounded once but for sincospi and exp: the values between are sums hi + lo.
// With t and pi tau t rounded, a tap is off by up to 1e-16 of the largest one whatever its own size:
// that was over half of the filter's error (S = 4, B = 76: 2.7e-16, with these taps 2.1e-16).
__device__ __forceinline__ double window_y_mu(long num, long den, double tau, double sigma, double mu)
{
  if (num == 0) return __ddiv_rn(1.0, mu);
  const double PI_LO = 1.2246467991473532e-16;  // pi - M_PI
  const double t = (double)num / (double)den;
  const double tl = fma(-t, (double)den, (double)num) / (double)den;
  // a = tau t, d = pi a
  const double a = __dmul_rn(tau, t), al = fma(tau, t, -a) + tau * tl;
  const double d = __dmul_rn(M_PI, a), dl = fma(M_PI, a, -d) + (M_PI * al + PI_LO * a);
  double s0, c0;
  sincospi(a, &s0, &c0);
  const double q = __ddiv_rn(s0, d);  // sin(pi a)/(pi a)
  const double ql = (fma(-q, d, s0) + (c0 * (M_PI * al) - q * dl)) / d;
  // g = (pi t)^2 / sigma
  const double u = __dmul_rn(M_PI, t), ul = fma(M_PI, t, -u) + (M_PI * tl + PI_LO * t);
  const double v = __dmul_rn(u, u), vl = fma(u, u, -v) + 2 * u * ul;
  const double g = __ddiv_rn(v, sigma);
  if (g > 800) return 0.0;
  const double gl = g == 0 ? 0.0 : (fma(-g, sigma, v) + vl) / sigma;
  const double e = exp(-g);
  const double y = __dmul_rn(q, e), yl = fma(q, e, -y) + e * (ql - q * gl);
  const double r = __ddiv_rn(y, mu);
  return r + (fma(-r, mu, y) + yl) / mu;
}

// y(t) as the reference forms it, from a rounded t
__device__ __forceinline__ double window_y(double t, double tau, double sigma)
{
  if (t == 0.0) return 1.0;
  const double PI_D = 3.14159265358979323846;
  // sin(pi tau t) with the product tau*t carried to double-double
  double ph = __dmul_rn(tau, t);
  double pl = fma(tau, t, -ph);
  double sp, cp;
  sincospi(ph, &sp, &cp);
  double num = fma(M_PI * pl, cp, sp);
  double den = __dmul_rn(__dmul_rn(PI_D, tau), t);
  double e = exp(__ddiv_rn(__dmul_rn(__dmul_rn(__dmul_rn(-PI_D, PI_D), t), t), sigma));
  return __dmul_rn(__ddiv_rn(num, den), e);
}

__global__ void k_make_taps(void *taps, double2 *post, double2 *w_full, int S, int n_mu,
                            int d_mu, int B, int B_pad, double tau, double sigma, long N, long M,
                            long Mh, int ref, int ct)
{
  long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
  long total = (long)n_mu * S * B_pad;
  if (idx >= total) return;
  int b = (int)(idx % B_pad);
  long rest = idx / B_pad;
  int i = (int)(rest % S);
  int theta = (int)(rest / S);
  const long den = 2L * n_mu * S;
  const int kappa = B - d_mu;
  const double mu = (double)n_mu / (double)d_mu;
  long num0 = 2L * theta * d_mu * S + (long)kappa * n_mu * S - 2L * i * n_mu;  // (t + b) * den
  double sp0, cp0;
  sincospi_ratio(num0, den, &sp0, &cp0);  // post phase
  if (b == 0) post[theta * S + i] = ct ? double2{1.0, 0.0} : double2{cp0, sp0};
  double2 wv = double2{0.0, 0.0};
  if (b < B) {
    double sp, cp, ymu = 0;
    if (ref) {
      long j = (long)b * S + i;
      double a0 = __ddiv_rn((double)theta, (double)Mh);
      double a1 = __ddiv_rn((double)j, (double)N);
      double a2 = __ddiv_rn((double)kappa, (double)(2 * M));
      const double t = __dmul_rn(__dadd_rn(__dsub_rn(a0, a1), a2), (double)M);
      sincospi(t, &sp, &cp);
      const double y = window_y(t, tau, sigma);
      wv = double2{__ddiv_rn(__dmul_rn(cp, y), mu), __ddiv_rn(__dmul_rn(sp, y), mu)};
    } else {
      const long num = num0 - 2L * b * n_mu * S;
      sincospi_ratio(num, den, &sp, &cp);
      ymu = window_y_mu(num, den, tau, sigma, mu);
      wv = double2{__dmul_rn(cp, ymu), __dmul_rn(sp, ymu)};
    }
    if (w_full) w_full[((long)theta * B + b) * S + i] = wv;
    if (!ct) ((double *)taps)[idx] = (b & 1) ? -ymu : ymu;  // (exact t only)
  } else if (!ct) {
    ((double *)taps)[idx] = 0.0;
  }
  if (ct) ((double2 *)taps)[idx] = wv;
}

// W_inv[m] = e^{-2 pi i kappa m / (2M)} / w_hat(m/M - 1/2)   (pfft.c:68-82)
// w_hat(t) = [erfc(sqrt(sigma)(t - tau/2)) - erfc(sqrt(sigma)(t + tau/2))] / (2 tau)
__global__ void k_make_winv(double2 *winv, long M, int kappa, double tau, double sigma)
{
  long m = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (m >= M) return;
  double t = (double)m / (double)M - 0.5;
  double ss = sqrt(sigma);
  double y = 1.0 / (2.0 * tau) * (erfc(ss * (t - tau / 2)) - erfc(ss * (t + tau / 2)));
  double sp, cp;
  sincospi_ratio((long)kappa * m, M, &sp, &cp);
  winv[m] = double2{cp / y, -sp / y};
}

// tw[m] = e^{-2 pi i m mult / L} for m < n
__global__ void k_make_twiddles(double2 *tw, long n, long L, long mult)
{
  long m = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (m >= n) return;
  double sp, cp;
  sincospi_ratio(2 * (m * mult % L), L, &sp, &cp);
  tw[m] = double2{cp, -sp};
}

__global__ void k_f64_to_f32(const double2 *in, float2 *out, long n)
{
  long m = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (m < n) out[m] = float2{(float)in[m].x, (float)in[m].y};
}

// =============================================================================================
// Step 3: M_hat-point FFT per segment, demodulation fused into the last pass
// =============================================================================================
// Single pass: `count` whole segments per block (M_hat small enough for LDS).
template <typename C>
__global__ __launch_bounds__(256) void k_fft_single(const C *__restrict__ at, C *__restrict__ X,
                                                    const C *__restrict__ tw,
                                                    const double2 *__restrict__ winv, long L,
                                                    long M, int S, int count, SoiBatch b)
{
  at = batch_ptr(at, b.at);
  X = batch_ptr(X, b.x);
  extern __shared__ __align__(16) unsigned char lds_raw[];
  C *lds = reinterpret_cast<C *>(lds_raw);
  const int tid = threadIdx.x, nt = blockDim.x;
  const int s0 = blockIdx.x * count;
  const int nseq = min(count, S - s0);
  const int qs = (int)L + 1;
  for (int e = tid; e < nseq * L; e += nt) {
    int q = e / (int)L, j = e - q * (int)L;
    lds[q * qs + j] = at[(long)(s0 + q) * L + j];
  }
  __syncthreads();
  lds_fft<32>(lds, (int)L, nseq, qs, 1, tw);
  for (int e = tid; e < nseq * M; e += nt) {
    int q = e / (int)M, m = e - q * (int)M;
    X[(long)(s0 + q) * M + m] = demod<C>(winv[m], lds[q * qs + m]);
  }
}

// Pass 1 (column FFTs): segment viewed as n1 x n2 row-major (R = n2*r1 + r2).  A block takes
// Tc adjacent columns, runs n1-point FFTs down them, multiplies element m1 of column r2 by
// e^{-2 pi i r2 m1 / M_hat} (two-level table: hi[e / B1] * lo[e % B1]) and stores in place.
template <typename C>
__global__ __launch_bounds__(256) void k_fft_col(C *__restrict__ data, const C *__restrict__ tw1,
                                                 const C *__restrict__ thi,
                                                 const C *__restrict__ tlo, int n1, int n2,
                                                 int Tc, int B1, long Mh, int S, SoiBatch b)
{
  data = batch_ptr(data, b.at);
  extern __shared__ __align__(16) unsigned char lds_raw[];
  C *lds = reinterpret_cast<C *>(lds_raw);
  const int tid = threadIdx.x, nt = blockDim.x;
  const int ncb = n2 / Tc;
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int cb = bid % ncb;
  const int s = bid / ncb;
  if (s >= S) return;
  const int c0 = cb * Tc;
  C *seg = data + (long)s * Mh;
  for (int e = tid; e < n1 * Tc; e += nt) {
    int r1 = e / Tc, q = e - r1 * Tc;
    lds[e] = seg[(long)r1 * n2 + c0 + q];
  }
  __syncthreads();
  lds_fft<32>(lds, n1, Tc, 1, Tc, tw1);
  for (int e = tid; e < n1 * Tc; e += nt) {
    int m1 = e / Tc, q = e - m1 * Tc;
    long ex = (long)(c0 + q) * m1;  // < M_hat
    C t = cmul(thi[ex / B1], tlo[ex % B1]);
    seg[(long)m1 * n2 + c0 + q] = cmul(lds[e], t);
  }
}

// Pass 2 (row FFTs + demodulation): a block takes Tr adjacent rows m1, runs n2-point FFTs along
// them; element m2 of row m1 is y[m1 + n1*m2].  For m < M it stores W_inv[m] * y[m] to X[s*M+m]
// (pfft.c:649-693), Tr adjacent m per contiguous run.
template <typename C>
__global__ __launch_bounds__(256) void k_fft_row(const C *__restrict__ data, C *__restrict__ X,
                                                 const C *__restrict__ tw2,
                                                 const double2 *__restrict__ winv, int n1,
                                                 int n2, int Tr, long Mh, long M, int S,
                                                 SoiBatch b)
{
  data = batch_ptr(data, b.at);
  X = batch_ptr(X, b.x);
  extern __shared__ __align__(16) unsigned char lds_raw[];
  C *lds = reinterpret_cast<C *>(lds_raw);
  const int tid = threadIdx.x, nt = blockDim.x;
  const int nrb = n1 / Tr;
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int s = bid % S;          // segments of one row block are adjacent: W_inv rows shared
  const int rb = bid / S;
  if (rb >= nrb) return;
  const int a = rb * Tr;
  const C *seg = data + (long)s * Mh;
  for (int e = tid; e < n2 * Tr; e += nt) {
    int q = e / n2, r2 = e - q * n2;
    lds[r2 * Tr + q] = seg[(long)(a + q) * n2 + r2];
  }
  __syncthreads();
  lds_fft<32>(lds, n2, Tr, 1, Tr, tw2);
  C *out = X + (long)s * M;
  for (int e = tid; e < n2 * Tr; e += nt) {
    int m2 = e / Tr, q = e - m2 * Tr;
    long m = (long)(a + q) + (long)n1 * m2;
    if (m < M) out[m] = demod<C>(winv[m], lds[e]);
  }
}

// =============================================================================================
// VLC codec (compress.c).  Every 16-element chunk of a stream contributes one field per lane;
// field widths are fixed per stream, so each 32-bit word of lane j is computable directly.
// =============================================================================================
__device__ __forceinline__ int exp_field(double v)
{
  uint64_t u = (uint64_t)__double_as_longlong(v);
  return (int)((u >> 52) & 0x7FF);
}

// per-chunk max exponent (compress.c:46-93).  One block per chunk.
__global__ void k_max_exponent(const double *__restrict__ x, int len, int *__restrict__ out)
{
  __shared__ int red[1024];
  const double *c = x + (long)blockIdx.x * len;
  int m = INT_MIN;
  for (int e = threadIdx.x; e < len; e += blockDim.x) m = max(m, exp_field(c[e]));
  red[threadIdx.x] = m;
  __syncthreads();
  for (int h = blockDim.x / 2; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] = max(red[threadIdx.x], red[threadIdx.x + h]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = (int)((unsigned)red[0] - 1023u);
}

struct VlcParams {
  int i1Len, i2Len, fbits;  // field widths; fbits = bits per element in a lane
  double e1, e2, e3;        // 2^(21-e_max), 2^(52-e_max), 2^31
  double d1, d2;            // 2^(e_max-21), 2^(e_max-52)
};

__device__ __forceinline__ VlcParams vlc_params(int e_max, int e_max_i)
{
  VlcParams v;
  int dl = e_max - e_max_i;
  v.i1Len = 24 - dl;
  v.i2Len = min(32, 55 - dl);
  v.fbits = (v.i1Len > 0 ? v.i1Len : 0) + (v.i2Len > 0 ? v.i2Len : 0);
  v.e1 = ldexp(1.0, 21 - e_max);
  v.e2 = ldexp(1.0, 52 - e_max);
  v.e3 = ldexp(1.0, 31);
  v.d1 = ldexp(1.0, e_max - 21);
  v.d2 = ldexp(1.0, e_max - 52);
  return v;
}

// The two integers of one element, i1 and i2 (their low i1Len and i2Len bits are sent).
// vec=1: rint + fmsub (compress.c:230-280); vec=0: round() + unfused (compress.c:333-342).
__device__ __forceinline__ uint2 vlc_ints(double x, const VlcParams &v, bool vec)
{
  double d1, d2;
  if (vec) {
    d1 = rint(x * v.e1);
    d2 = rint(fma(x, v.e2, -(d1 * v.e3)));
  } else {
    d1 = round(x * v.e1);
    double pr = __dmul_rn(x, v.e2);
    d2 = round(__dsub_rn(pr, __dmul_rn(d1, v.e3)));
  }
  return uint2{(uint32_t)(int32_t)d1, (uint32_t)(int32_t)d2};
}

// The bit pattern of one element: i1Len bits of i1 (when i1Len > 0) followed by i2Len bits of
// i2, as a value of fbits <= 56 bits, MSB first.
__device__ __forceinline__ uint64_t vlc_encode(double x, const VlcParams &v, bool vec)
{
  const uint2 i = vlc_ints(x, v, vec);
  uint64_t f2 = v.i2Len >= 32 ? (uint64_t)i.y : ((uint64_t)i.y & ((1ull << v.i2Len) - 1));
  if (v.i1Len > 0) {
    uint64_t f1 = (uint64_t)i.x & ((1ull << v.i1Len) - 1);
    return (f1 << v.i2Len) | f2;
  }
  return f2;
}

// bits [pos, pos+32) of a lane stream made of consecutive fbits-wide fields (MSB first).
template <typename F>
__device__ __forceinline__ uint32_t vlc_word(long pos, int fbits, long nfields, F field)
{
  uint32_t word = 0;
  long f0, f1;
  if (pos + 31 <= (long)UINT32_MAX) {  // 32-bit divisions: a fraction of the 64-bit sequence
    f0 = (uint32_t)pos / (uint32_t)fbits;
    f1 = (uint32_t)(pos + 31) / (uint32_t)fbits;
  } else {
    f0 = pos / fbits;
    f1 = (pos + 31) / fbits;
  }
  for (long f = f0; f <= f1 && f < nfields; ++f) {
    uint64_t val = field(f);
    long fstart = f * fbits;
    // overlap of [fstart, fstart+fbits) with [pos, pos+32)
    long lo = max(fstart, pos), hi = min(fstart + fbits, pos + 32);
    if (lo >= hi) continue;
    int nb = (int)(hi - lo);
    int shift_out = (int)(fstart + fbits - hi);  // bits of the field after hi
    uint64_t part = (val >> shift_out) & ((1ull << nb) - 1);
    word |= (uint32_t)(part << (pos + 32 - hi));
  }
  return word;
}

// Word wi of a chunk's stream (compress.c:205-372): vector rows (16 lanes interleaved) then the
// scalar tail.
__device__ __forceinline__ uint32_t compress_word(const double *__restrict__ in, int len,
                                                  const VlcParams &v, long wi)
{
  const long nvf = len / 16;                 // fields per lane in the vector body
  const long vrows = (nvf * v.fbits + 31) / 32;
  if (wi < vrows * 16) {
    const long row = wi / 16;
    const int lane = (int)(wi % 16);
    return vlc_word(row * 32, v.fbits, nvf,
                    [&](long f) { return vlc_encode(in[f * 16 + lane], v, true); });
  }
  const long ntail = len - nvf * 16;
  const double *tin = in + nvf * 16;
  return vlc_word((wi - vrows * 16) * 32, v.fbits, ntail,
                  [&](long f) { return vlc_encode(tin[f], v, false); });
}

// Words of a chunk's stream (compress()'s return value)
__device__ __forceinline__ long compress_words(int len, const VlcParams &v)
{
  if (v.i2Len <= 0) return 0;
  const long nvf = len / 16;
  return (nvf * v.fbits + 31) / 32 * 16 + ((len - nvf * 16) * v.fbits + 31) / 32;
}

// compress: one thread per output word, blockIdx.y = chunk.  nwords[c] = compress()'s return
// value.
__global__ void k_compress(int *__restrict__ out, long stride, const double *__restrict__ x,
                           int len, int nchunk, int e_max, const int *__restrict__ emi,
                           int *__restrict__ nwords, const int *__restrict__ e_max_dev)
{
  const int c = blockIdx.y;
  if (c >= nchunk) return;
  VlcParams v = vlc_params(e_max_dev ? *e_max_dev : e_max, emi[c]);
  const double *in = x + (long)c * len;
  int *o = out + (long)c * stride;
  const long total = compress_words(len, v);
  if (blockIdx.x == 0 && threadIdx.x == 0) nwords[c] = (int)total;
  for (long wi = blockIdx.x * (long)blockDim.x + threadIdx.x; wi < total;
       wi += (long)gridDim.x * blockDim.x)
    o[wi] = (int)compress_word(in, len, v, wi);
}

// extract the fbits-wide field f of a lane stream whose word w is at base[w*wstride]
__device__ __forceinline__ uint64_t vlc_field(const int *base, long wstride, long f, int fbits)
{
  long pos = f * fbits;
  long w0 = pos / 32;
  int off = (int)(pos - w0 * 32);
  uint64_t hi = (uint32_t)base[w0 * wstride];
  uint64_t lo = (off + fbits > 32) ? (uint32_t)base[(w0 + 1) * wstride] : 0u;
  uint64_t bits = (hi << 32) | lo;  // 64-bit window starting at word w0
  int sh = 64 - off - fbits;
  if (off + fbits > 64) {
    // field spans three words (fbits <= 56 and off <= 31 can reach 87 bits)
    uint64_t lo2 = (uint32_t)base[(w0 + 2) * wstride];
    int extra = off + fbits - 64;
    uint64_t top = bits & ((fbits - extra >= 64) ? ~0ull : ((1ull << (64 - off)) - 1));
    return (top << extra) | (lo2 >> (32 - extra));
  }
  return (bits >> sh) & ((fbits >= 64) ? ~0ull : ((1ull << fbits) - 1));
}

// the element that the two (sign-extended) integers stand for
__device__ __forceinline__ double vlc_value(int32_t i1, int32_t i2, const VlcParams &v, bool vec)
{
  if (vec) return fma((double)i1, v.d1, (double)i2 * v.d2);       // compress.c:472-483
  return __dadd_rn(__dmul_rn((double)i1, v.d1), __dmul_rn((double)i2, v.d2));  // :529-531
}

__device__ __forceinline__ double vlc_decode(uint64_t fv, const VlcParams &v, bool vec)
{
  int32_t i1 = 0, i2;
  uint64_t f2 = v.i2Len >= 32 ? (fv & 0xFFFFFFFFull) : (fv & ((1ull << v.i2Len) - 1));
  // sign-extend i2Len bits
  i2 = (int32_t)((int64_t)(f2 << (64 - v.i2Len)) >> (64 - v.i2Len));
  if (v.i1Len > 0) {
    uint64_t f1 = (fv >> v.i2Len) & ((1ull << v.i1Len) - 1);
    i1 = (int32_t)((int64_t)(f1 << (64 - v.i1Len)) >> (64 - v.i1Len));
  }
  return vlc_value(i1, i2, v, vec);
}

// Element e of a chunk decoded from its stream w (compress.c:428-544)
__device__ __forceinline__ double decompress_elem(const int *__restrict__ w, int len,
                                                  const VlcParams &v, long e)
{
  if (v.i2Len <= 0) return 0.0;
  const long nvf = len / 16;
  if (e < nvf * 16)
    return vlc_decode(vlc_field(w + e % 16, 16, e / 16, v.fbits), v, true);
  const long vrows = (nvf * v.fbits + 31) / 32;
  return vlc_decode(vlc_field(w + vrows * 16, 1, e - nvf * 16, v.fbits), v, false);
}

__global__ void k_decompress(double *__restrict__ out, const int *__restrict__ in, long stride,
                             int len, int nchunk, int e_max, const int *__restrict__ emi,
                             const int *__restrict__ e_max_dev)
{
  const int c = blockIdx.y;
  if (c >= nchunk) return;
  VlcParams v = vlc_params(e_max_dev ? *e_max_dev : e_max, emi[c]);
  double *o = out + (long)c * len;
  const int *w = in + (long)c * stride;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < len;
       e += (long)gridDim.x * blockDim.x)
    o[e] = decompress_elem(w, len, v, e);
}

// ---------------------------------------------------------------------------------------------
// The exchange of one device: compress every chunk and (DECODE) decode it in place, in one pass.
// 32 consecutive fields of a lane fill exactly fbits words, so a thread takes 32 fields of one
// lane: no field is in two threads' words, each is encoded once, and its decoded value goes back over
// the element that it came from.  All threads have the same work whatever the chunks' field
// widths, and the 16 lanes of a vector row are adjacent threads (128-byte runs of elements, 64-byte
// runs of words).  The scalar tail of a chunk (fewer than 16 elements) is one thread's.
// Bound by memory: elements read once, words and elements written once.  N = 7*2^23 (1.07 GB of
// elements, about 0.7 GB of words): 609 us, 4.7 TB/s; compressing and decompressing in two passes
// over runs of words took 690 + 541 us.
// ---------------------------------------------------------------------------------------------
constexpr int VLC_FIELDS = 32;

// One lane's bit stream, MSB first: word r goes to o[r * pitch]; cur holds the last nacc (< 32)
// bits that are not in a word yet, below anything.  A field comes left-aligned, so that the
// bits above it fall out of the shifts; the widths are the same in all lanes of a wave.
struct VlcPack {
  int *o;
  int pitch;
  uint32_t cur;
  int nacc;
  __device__ __forceinline__ void put(uint32_t left, int n)  // 1 <= n <= 32
  {
    if (nacc + n >= 32) {
      *o = (int)__builtin_amdgcn_alignbit(cur, left, (uint32_t)nacc);
      o += pitch;
      nacc -= 32;
    }
    cur = __builtin_amdgcn_alignbit(cur, left, (uint32_t)(32 - n));
    nacc += n;
  }
  __device__ __forceinline__ void flush()
  {
    if (nacc > 0) *o = (int)(cur << (32 - nacc));
  }
};

// One element into the stream; returns the value that decoding it gives
__device__ __forceinline__ double vlc_put(double x, const VlcParams &v, bool vec, VlcPack &w)
{
  const uint2 i = vlc_ints(x, v, vec);
  int32_t i1 = 0;
  if (v.i1Len > 0) {
    const uint32_t left = i.x << (32 - v.i1Len);
    w.put(left, v.i1Len);
    i1 = (int32_t)left >> (32 - v.i1Len);
  }
  const uint32_t left = i.y << (32 - v.i2Len);
  w.put(left, v.i2Len);
  return vlc_value(i1, (int32_t)left >> (32 - v.i2Len), v, vec);
}

template <bool DECODE>
__global__ __launch_bounds__(256) void k_vlc_exchange(int *__restrict__ out, long stride,
                                                      double *__restrict__ x, int len, int nchunk,
                                                      const int *__restrict__ e_max_dev,
                                                      const int *__restrict__ emi)
{
  const int nvf = len / 16, ntail = len - nvf * 16;
  const int nu = (nvf + VLC_FIELDS - 1) / VLC_FIELDS;
  // a wave takes 4 neighbouring units of one chunk: the chunk and its widths are scalars
  const int per = (nu + 3) / 4 + (ntail ? 1 : 0);
  const long wv = (long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int c = (int)(wv / per), g = (int)(wv - (long)c * per);
  if (c >= nchunk) return;
  const int lane = threadIdx.x & 15, u = g * 4 + (((int)threadIdx.x >> 4) & 3);
  const VlcParams v = vlc_params(*e_max_dev, emi[c]);
  const bool coded = v.i2Len > 0;
  double *xc = x + (long)c * len;
  int *oc = out + (long)c * stride;
  constexpr int G = 8;  // fields loaded together
  if ((g + 1) * 4 * VLC_FIELDS <= nvf) {
    double *p = xc + (long)u * (VLC_FIELDS * 16) + lane;
    if (coded) {
      VlcPack w = {oc + ((long)u * v.fbits) * 16 + lane, 16, 0, 0};
      double a[G], b[G];
#pragma unroll
      for (int i = 0; i < G; ++i) a[i] = p[i * 16];
#pragma unroll
      for (int f = 0; f < VLC_FIELDS; f += G) {
#pragma unroll
        for (int i = 0; i < G; ++i) b[i] = a[i];
        if (f + G < VLC_FIELDS) {
#pragma unroll
          for (int i = 0; i < G; ++i) a[i] = p[(f + G + i) * 16];
        }
#pragma unroll
        for (int i = 0; i < G; ++i) {
          const double y = vlc_put(b[i], v, true, w);
          if constexpr (DECODE) p[(f + i) * 16] = y;
        }
      }
    } else if constexpr (DECODE) {
#pragma unroll
      for (int f = 0; f < VLC_FIELDS; ++f) p[f * 16] = 0.0;
    }
  } else if (g * 4 < nu) {  // the last units of the chunk
    if (u >= nu) return;
    double *p = xc + (long)u * (VLC_FIELDS * 16) + lane;
    VlcPack w = {oc + ((long)u * v.fbits) * 16 + lane, 16, 0, 0};
    const int nf = min(VLC_FIELDS, nvf - u * VLC_FIELDS);
    for (int f = 0; f < nf; ++f) {
      const double y = coded ? vlc_put(p[f * 16], v, true, w) : 0.0;
      if constexpr (DECODE) p[f * 16] = y;
    }
    w.flush();
  } else if ((threadIdx.x & 63) == 0) {  // the scalar tail
    double *p = xc + (long)nvf * 16;
    VlcPack w = {oc + ((long)nvf * v.fbits + 31) / 32 * 16, 1, 0, 0};
    for (int f = 0; f < ntail; ++f) {
      const double y = coded ? vlc_put(p[f], v, false, w) : 0.0;
      if constexpr (DECODE) p[f] = y;
    }
    w.flush();
  }
}

// Copy between device and pinned host memory, 16-byte units.  A kernel follows the kernels before it in
// the stream directly, where a DMA engine's copy waits for a signal between queues.
__global__ __launch_bounds__(256) void k_copy(double2 *__restrict__ dst,
                                              const double2 *__restrict__ src, long n)
{
  const long nt = (long)gridDim.x * blockDim.x;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += nt) dst[e] = src[e];
}

// =============================================================================================
// Synthetic inputs (seeded, counter based) for tests and the benchmark
// =============================================================================================
__device__ __forceinline__ uint64_t splitmix64(uint64_t z)
{
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ double u01(uint64_t seed, uint64_t n)
{
  return (double)(splitmix64(seed ^ (n * 0xD1B54A32D192ED03ull)) >> 11) * 0x1.0p-53;
}

// uniform[-1,1] re/im (identical to the oracle's orc_uniform_input)
__global__ void k_gen_uniform(double2 *x, long N, uint64_t seed)
{
  long n = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (n >= N) return;
  x[n] = double2{2.0 * u01(seed, 2 * n) - 1.0, 2.0 * u01(seed, 2 * n + 1) - 1.0};
}

// sum of tones a_j e^{2 pi i f_j n / N + i phi_j} plus complex Gaussian noise (Box-Muller)
__global__ void k_gen_tones(double2 *x, long N, const double *__restrict__ tf,
                            const double *__restrict__ tph, int ntones, double amp,
                            double noise_sigma, uint64_t seed)
{
  long n = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (n >= N) return;
  double re = 0, im = 0;
  for (int j = 0; j < ntones; ++j) {
    // phase in turns: f*n/N exactly reduced using the integer part of f
    double f = tf[j];
    double fi = floor(f), ff = f - fi;
    long fn = ((long)fi % N) * (n % N) % N;  // (fi*n) mod N, exact for N < 2^31
    double turns = (double)fn / (double)N + ff * ((double)n / (double)N) + tph[j];
    turns -= floor(turns);
    double sp, cp;
    sincospi(2.0 * turns, &sp, &cp);
    re += amp * cp;
    im += amp * sp;
  }
  if (noise_sigma > 0) {
    double u1 = u01(seed, 2 * n), u2 = u01(seed, 2 * n + 1);
    double rr = sqrt(-2.0 * log(1.0 - u1)) * noise_sigma;
    double sp, cp;
    sincospi(2.0 * u2, &sp, &cp);
    re += rr * cp;
    im += rr * sp;
  }
  x[n] = double2{re, im};
}

// =============================================================================================
// C-ABI launchers
// =============================================================================================
static inline unsigned nblk(long n, int t) { return (unsigned)((n + t - 1) / t); }

extern "C" int soik_make_tables(void *taps, double2 *post, double2 *w_full, double2 *winv,
                                int S, int n_mu, int d_mu, int B, int B_pad, double tau,
                                double sigma, long N, long M, long Mh, int ref, int ct,
                                hipStream_t st)
{
  long nt = (long)n_mu * S * B_pad;
  hipLaunchKernelGGL(k_make_taps, dim3(nblk(nt, 256)), dim3(256), 0, st, taps, post, w_full, S,
                     n_mu, d_mu, B, B_pad, tau, sigma, N, M, Mh, ref, ct);
  hipLaunchKernelGGL(k_make_winv, dim3(nblk(M, 256)), dim3(256), 0, st, winv, M, B - d_mu, tau,
                     sigma);
  return (int)hipGetLastError();
}

extern "C" int soik_make_twiddles(double2 *tw, long n, long L, long mult, hipStream_t st)
{
  hipLaunchKernelGGL(k_make_twiddles, dim3(nblk(n, 256)), dim3(256), 0, st, tw, n, L, mult);
  return (int)hipGetLastError();
}

static void set_lds_attr(const void *f)
{
  (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
}

template <typename C>
static int fft_single(const C *at, C *X, const C *tw, const double2 *winv, long L, long M, int S,
                      int count, SoiBatch b, hipStream_t st)
{
  static bool once = false;
  if (!once) { set_lds_attr((const void *)k_fft_single<C>); once = true; }
  size_t lds = (size_t)count * (L + 1) * sizeof(C);
  hipLaunchKernelGGL(k_fft_single<C>, dim3((S + count - 1) / count, b.n > 0 ? b.n : 1), dim3(256),
                     lds, st, at, X, tw, winv, L, M, S, count, b);
  return (int)hipGetLastError();
}

template <typename C>
static int fft_col(C *data, const C *tw1, const C *thi, const C *tlo, int n1, int n2, int Tc,
                   int B1, long Mh, int S, SoiBatch b, hipStream_t st)
{
  static bool once = false;
  if (!once) { set_lds_attr((const void *)k_fft_col<C>); once = true; }
  size_t lds = (size_t)n1 * Tc * sizeof(C);
  unsigned grid = (unsigned)((n2 / Tc) * S);
  hipLaunchKernelGGL(k_fft_col<C>, dim3(grid, b.n > 0 ? b.n : 1), dim3(256), lds, st, data, tw1,
                     thi, tlo, n1, n2, Tc, B1, Mh, S, b);
  return (int)hipGetLastError();
}

template <typename C>
static int fft_row(const C *data, C *X, const C *tw2, const double2 *winv, int n1, int n2,
                   int Tr, long Mh, long M, int S, SoiBatch b, hipStream_t st)
{
  static bool once = false;
  if (!once) { set_lds_attr((const void *)k_fft_row<C>); once = true; }
  size_t lds = (size_t)n2 * Tr * sizeof(C);
  unsigned grid = (unsigned)((n1 / Tr) * S);
  hipLaunchKernelGGL(k_fft_row<C>, dim3(grid, b.n > 0 ? b.n : 1), dim3(256), lds, st, data, X,
                     tw2, winv, n1, n2, Tr, Mh, M, S, b);
  return (int)hipGetLastError();
}

extern "C" int soik_fft_single(const double2 *at, double2 *X, const double2 *tw,
                               const double2 *winv, long L, long M, int S, int count,
                               SoiBatch b, hipStream_t st)
{
  return fft_single<double2>(at, X, tw, winv, L, M, S, count, b, st);
}

extern "C" int soik_fft_col(double2 *data, const double2 *tw1, const double2 *thi,
                            const double2 *tlo, int n1, int n2, int Tc, int B1, long Mh, int S,
                            SoiBatch b, hipStream_t st)
{
  return fft_col<double2>(data, tw1, thi, tlo, n1, n2, Tc, B1, Mh, S, b, st);
}

extern "C" int soik_fft_row(const double2 *data, double2 *X, const double2 *tw2,
                            const double2 *winv, int n1, int n2, int Tr, long Mh, long M, int S,
                            SoiBatch b, hipStream_t st)
{
  return fft_row<double2>(data, X, tw2, winv, n1, n2, Tr, Mh, M, S, b, st);
}

// FP32 form: complex64 data and tables; W_inv stays FP64
extern "C" int soik_fft_single_f32(const float2 *at, float2 *X, const float2 *tw,
                                   const double2 *winv, long L, long M, int S, int count,
                                   SoiBatch b, hipStream_t st)
{
  return fft_single<float2>(at, X, tw, winv, L, M, S, count, b, st);
}

extern "C" int soik_fft_col_f32(float2 *data, const float2 *tw1, const float2 *thi,
                                const float2 *tlo, int n1, int n2, int Tc, int B1, long Mh,
                                int S, SoiBatch b, hipStream_t st)
{
  return fft_col<float2>(data, tw1, thi, tlo, n1, n2, Tc, B1, Mh, S, b, st);
}

extern "C" int soik_fft_row_f32(const float2 *data, float2 *X, const float2 *tw2,
                                const double2 *winv, int n1, int n2, int Tr, long Mh, long M,
                                int S, SoiBatch b, hipStream_t st)
{
  return fft_row<float2>(data, X, tw2, winv, n1, n2, Tr, Mh, M, S, b, st);
}

extern "C" int soik_max_exponent(const double *x, int len, int nchunk, int *out, hipStream_t st)
{
  if (nchunk <= 0) return 0;
  hipLaunchKernelGGL(k_max_exponent, dim3(nchunk), dim3(256), 0, st, x, len, out);
  return (int)hipGetLastError();
}

extern "C" int soik_compress(int *out, long stride, const double *x, int len, int nchunk,
                             int e_max, const int *emi, int *nwords, const int *e_max_dev,
                             hipStream_t st)
{
  if (nchunk <= 0) return 0;
  long maxw = (long)len * 56 / 32 / 1 + 64;
  // blocks per chunk: enough for about 2048 blocks in all (the kernel strides over the chunk's
  // words), not one thread per possible word: a chunk of short fields has few words, and a
  // grid sized for 55-bit fields would be mostly idle blocks
  unsigned gx = nblk(maxw, 256);
  const unsigned cap = (unsigned)((2048 + nchunk - 1) / nchunk);
  if (gx > cap) gx = cap;
  hipLaunchKernelGGL(k_compress, dim3(gx, nchunk), dim3(256), 0, st, out, stride, x, len, nchunk,
                     e_max, emi, nwords, e_max_dev);
  return (int)hipGetLastError();
}

extern "C" int soik_decompress(double *out, const int *in, long stride, int len, int nchunk,
                               int e_max, const int *emi, const int *e_max_dev, hipStream_t st)
{
  if (nchunk <= 0) return 0;
  unsigned gx = nblk(len, 256);
  const unsigned cap = (unsigned)((2048 + nchunk - 1) / nchunk);  // about 2048 blocks in all
  if (gx > cap) gx = cap;
  hipLaunchKernelGGL(k_decompress, dim3(gx, nchunk), dim3(256), 0, st, out, in, stride, len,
                     nchunk, e_max, emi, e_max_dev);
  return (int)hipGetLastError();
}

// VLC planning on the device (pfft.c:316-343, 390-440): from the per-chunk exponents of the
// S x P chunks (chunk (s, p) = s*P + p), the per-segment maximum (the reference's
// MPI_Allreduce(MAX) over ranks), the global maximum, every chunk's segment exponent, the
// per-segment send counts in doubles and the cost-balanced segment boundaries.  One block; only
// the prefix sum of the costs is serial (the reference's double arithmetic, unfused and in its
// order, so that the boundaries are bit-identical to the host restatement); its terms and the
// boundary searches run on all threads (S = P = 64: 13 us, 56 us with the walk
// and the terms serial).
// out: [0] global maximum, [1 .. S] segment maxima, [1+S .. 2S] send counts,
//      [1+2S .. 1+2S+P] segment boundaries; pcs: S + 1 doubles of scratch.
__global__ void k_vlc_plan(const int *__restrict__ exps, int S, int P, int k, long l, long Mh,
                           double ratio, int *__restrict__ emi, int *__restrict__ out,
                           double *__restrict__ pcs_g, int *__restrict__ nwords)
{
#pragma clang fp contract(off)
  // segment maxima and prefix costs in LDS when S is small enough (the serial sum below then
  // reads no global memory), else in the caller's scratch
  constexpr int SMAX = 2048;
  __shared__ int smax, segs[SMAX];
  __shared__ double pcs_s[SMAX + 1];
  const bool inl = S <= SMAX;
  double *pcs = inl ? pcs_s : pcs_g;
  const int tid = threadIdx.x, nt = blockDim.x;
  if (tid == 0) smax = INT_MIN;
  if (inl)
    for (int s = tid; s < S; s += nt) segs[s] = INT_MIN;
  __syncthreads();
  if (inl) {
    // the chunks of a segment over the threads: consecutive threads on consecutive chunks
    for (int c = tid; c < S * P; c += nt) atomicMax(&segs[c / P], exps[c]);
    __syncthreads();
    for (int s = tid; s < S; s += nt) {
      out[1 + s] = segs[s];
      atomicMax(&smax, segs[s]);
    }
  } else {
    for (int s = tid; s < S; s += nt) {
      int m = INT_MIN;
      for (int p = 0; p < P; ++p) m = max(m, exps[s * P + p]);
      out[1 + s] = m;
      atomicMax(&smax, m);
    }
  }
  __syncthreads();
  const int total = smax;
  // per segment: send count and cost (the term that the prefix sum adds), then per chunk
  for (int s = tid; s < S; s += nt) {
    int bits = 52 + 3 - (total - (inl ? segs[s] : out[1 + s]));
    if (bits > 31) ++bits;
    const int lenPerSimdLane = (int)((l * 2 / 16 * bits + 31) / 32);
    const int remainder = (int)((l * 2 % 16 * bits + 31) / 32);
    int sendLen = lenPerSimdLane * 16 + remainder;
    if (bits <= 0) sendLen = 0;
    const int cnt = (sendLen + 1) / 2;
    out[1 + S + s] = cnt;
    pcs[s + 1] = ratio * cnt / 2 / Mh;
  }
  const int len = (int)(2 * l);
  for (int c = tid; c < S * P; c += nt) {
    const int seg = inl ? segs[c / P] : out[1 + c / P];
    emi[c] = seg;
    nwords[c] = (int)compress_words(len, vlc_params(total, seg));
  }
  __syncthreads();
  if (tid == 0) {
    out[0] = total;
    double acc = 0;
    pcs[0] = 0;
    for (int s = 0; s < S; ++s) {
      acc = acc + pcs[s + 1] + 1;
      pcs[s + 1] = acc;
    }
  }
  __syncthreads();
  int *bd = out + 1 + 2 * S;
  const double costPerRank = pcs[S] / P;
  if (tid == 0) bd[0] = 0, bd[P] = S;
  if (ratio >= 0) {
    // increasing costs: every boundary by itself, the first s >= 1 with pcs[s] >= target
    for (int p = 1 + tid; p < P; p += nt) {
      const double target = p * costPerRank;
      int lo = 1, hi = S;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (pcs[mid] >= target) hi = mid;
        else lo = mid + 1;
      }
      bd[p] = (pcs[lo] - target > target - pcs[lo - 1]) ? lo - 1 : lo;
    }
  } else if (tid == 0) {  // the reference's walk, ended at the last segment (ratio negative or NaN)
    int s = 1;
    for (int p = 1; p < P;) {
      const double target = p * costPerRank;
      if (pcs[s] >= target) {
        bd[p] = (pcs[s] - target > target - pcs[s - 1]) ? s - 1 : s;
        ++p;
      } else if (s < S) {
        ++s;
      } else {
        bd[p] = S;
        ++p;
      }
    }
  }
}

extern "C" int soik_vlc_plan(const int *exps, int S, int P, int k, long l, long Mh, double ratio,
                             int *emi, int *out, double *pcs, long *, int *nwords, hipStream_t st)
{
  hipLaunchKernelGGL(k_vlc_plan, dim3(1), dim3(1024), 0, st, exps, S, P, k, l, Mh, ratio, emi, out,
                     pcs, nwords);
  return (int)hipGetLastError();
}

template <bool DECODE>
static int vlc_exchange(int *out, long stride, double *x, int len, int nchunk, const int *e_max_dev,
                        const int *emi, hipStream_t st)
{
  if (nchunk <= 0 || len <= 0) return 0;
  const int nvf = len / 16, nu = (nvf + VLC_FIELDS - 1) / VLC_FIELDS;
  const long waves = (long)nchunk * ((nu + 3) / 4 + (len % 16 ? 1 : 0));
  hipLaunchKernelGGL(k_vlc_exchange<DECODE>, dim3(nblk(waves, 4)), dim3(256), 0, st, out, stride,
                     x, len, nchunk, e_max_dev, emi);
  return (int)hipGetLastError();
}

// Words of all chunks, and the chunks decoded from them in place (after soik_vlc_plan)
extern "C" int soik_vlc_exchange(int *out, long stride, double *x, int len, int nchunk,
                                 const int *e_max_dev, const int *emi, hipStream_t st)
{
  return vlc_exchange<true>(out, stride, x, len, nchunk, e_max_dev, emi, st);
}

// The two halves by themselves, for the tests: the words (x stays), and decoding them
extern "C" int soik_compress_flat(int *out, long stride, const double *x, int len, int nchunk,
                                  const int *e_max_dev, const int *emi, const long *,
                                  hipStream_t st)
{
  return vlc_exchange<false>(out, stride, const_cast<double *>(x), len, nchunk, e_max_dev, emi, st);
}

extern "C" int soik_decompress_flat(double *out, const int *in, long stride, int len, int nchunk,
                                    const int *e_max_dev, const int *emi, hipStream_t st)
{
  return soik_decompress(out, in, stride, len, nchunk, 0, emi, e_max_dev, st);
}

extern "C" int soik_copy(void *dst, const void *src, size_t bytes, hipStream_t st)
{
  if (bytes % 16) return (int)hipErrorInvalidValue;
  const unsigned nb = nblk((long)(bytes / 16), 256);
  hipLaunchKernelGGL(k_copy, dim3(nb < 1024 ? nb : 1024), dim3(256), 0, st, (double2 *)dst,
                     (const double2 *)src, (long)(bytes / 16));
  return (int)hipGetLastError();
}

extern "C" int soik_gen_uniform(double2 *x, long N, uint64_t seed, hipStream_t st)
{
  hipLaunchKernelGGL(k_gen_uniform, dim3(nblk(N, 256)), dim3(256), 0, st, x, N, seed);
  return (int)hipGetLastError();
}

extern "C" int soik_gen_tones(double2 *x, long N, const double *tf, const double *tph, int ntones,
                              double amp, double noise_sigma, uint64_t seed, hipStream_t st)
{
  hipLaunchKernelGGL(k_gen_tones, dim3(nblk(N, 256)), dim3(256), 0, st, x, N, tf, tph, ntones,
                     amp, noise_sigma, seed);
  return (int)hipGetLastError();
}

extern "C" int soik_f64_to_f32(const double2 *in, float2 *out, long n, hipStream_t st)
{
  hipLaunchKernelGGL(k_f64_to_f32, dim3(nblk(n, 256)), dim3(256), 0, st, in, out, n);
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Allocation-free compress (soi_compress_noalloc in compress.h): the per-chunk segment exponents
// and word counts that compress() stages through hipMalloc'ed buffers live in a file-scope
// device array instead.  Its device address comes from hipGetSymbolAddress, once per device on
// the first call there (the array's name is a host-side stand-in in host code and is never
// passed to a kernel or a copy).  Every call on a device shares that device's array: calls
// that overlap on one device race.  The kernel writes every word count it reports, and the
// exponents are copied in before the kernel runs, so nothing needs clearing between calls.
// ---------------------------------------------------------------------------------------------
#include <mutex>

#define SOI_NOALLOC_MAX_CHUNKS 4096
#define SOI_NOALLOC_MAX_DEVICES 64
static __device__ __align__(256) int scratch[2 * SOI_NOALLOC_MAX_CHUNKS];
static int *g_scratch_ptr[SOI_NOALLOC_MAX_DEVICES];
static std::mutex g_scratch_mu;

extern "C" void soi_internal_set_error(int status, const char *msg);

static int *scratch_for_current_device(void)
{
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SOI_NOALLOC_MAX_DEVICES) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
      (void)hipGetLastError();
      return nullptr;
    }
    g_scratch_ptr[dev] = static_cast<int *>(p);
  }
  return g_scratch_ptr[dev];
}

extern "C" int soi_compress_noalloc(int *out, long stride_words, const double *x, int len,
                                    int nchunk, int e_max, const int *e_max_i, int *nwords,
                                    void *stream)
{
  if (!out || !x || !e_max_i || !nwords || len < 0 || nchunk < 1 ||
      stride_words < (long)len * 56 / 32 + 32) {
    soi_internal_set_error(1, "soi_compress_noalloc: needs device out and x, host e_max_i and "
                              "nwords, nchunk >= 1, stride_words >= len*56/32 + 32");
    return 1;
  }
  if (nchunk > SOI_NOALLOC_MAX_CHUNKS) {
    soi_internal_set_error(1, "soi_compress_noalloc: nchunk exceeds the scratch maximum of 4096 "
                              "chunks");
    return 1;
  }
  int *ptr = scratch_for_current_device();
  if (!ptr) {
    soi_internal_set_error(5, "soi_compress_noalloc: hipGetSymbolAddress of the scratch failed");
    return 5;
  }
  hipStream_t st = (hipStream_t)stream;
  int *emi = ptr, *nw = ptr + SOI_NOALLOC_MAX_CHUNKS;
  int e = (int)hipMemcpyAsync(emi, e_max_i, sizeof(int) * nchunk, hipMemcpyHostToDevice, st);
  if (!e) e = soik_compress(out, stride_words, x, len, nchunk, e_max, emi, nw, nullptr, st);
  if (!e) e = (int)hipMemcpyAsync(nwords, nw, sizeof(int) * nchunk, hipMemcpyDeviceToHost, st);
  if (!e) e = (int)hipStreamSynchronize(st);
  if (e) {
    soi_internal_set_error(5, hipGetErrorString((hipError_t)e));
    return 5;
  }
  soi_internal_set_error(0, "");
  return 0;
}
