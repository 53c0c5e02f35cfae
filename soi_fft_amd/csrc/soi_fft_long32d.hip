// soi_fft_long32d.hip -- complex64 segment FFT passes in chains of small radices, on the stages of soi_fft.hpp,
// for lengths whose odd part is not 1, 5 or 25 (the planner's choice: plan_fft in pfft.c).
//
// The results are those of the LDS kernels (k_fft_col, k_fft_row), bit for bit: the same radices in the same
// order (eights, then 4 or 2, then fives, then threes), each twiddle from the table.  What differs is where
// they run: chains of radices in registers, two exchanges instead of four or five passes over LDS.
#include "soi_fft.hpp"

using namespace soi;

// X(L, threads per sequence, chains)
#define SOI_FFT_LONGD(X) \
  X(576, 72, 8, 8, 303) X(600, 75, 8, 5, 503) X(640, 80, 8, 8, 205) X(720, 90, 8, 205, 303) \
  X(768, 96, 8, 8, 403) X(800, 80, 8, 405, 5) X(960, 64, 8, 8, 503) X(1000, 100, 8, 5, 505) \
  X(1024, 64, 8, 8, 802) X(1080, 72, 8, 503, 303) X(1152, 72, 8, 802, 303) \
  X(1200, 80, 8, 205, 503) X(1280, 80, 8, 8, 405) X(1440, 80, 8, 405, 303) \
  X(1536, 64, 8, 8, 803) X(1600, 100, 8, 8, 505) X(1920, 128, 8, 802, 503) \
  X(2000, 100, 8, 205, 505) X(2048, 64, 8, 8, 804) X(2160, 90, 8, 205, 30303) \
  X(2304, 96, 8, 804, 303) X(2400, 120, 8, 405, 503) X(2560, 80, 8, 8, 805)

// rows only: beside long columns
#define SOI_FFT_LONGD_ROWS(X) \
  X(2880, 72, 8, 8, 50303) X(3072, 64, 8, 8, 80203) X(3200, 80, 8, 8, 20505) \
  X(3456, 72, 8, 8, 2030303) X(3840, 80, 8, 8, 40503)

// Columns in halves, two or three blocks a CU beside the lower twiddle table (up to 32 KiB); rows eight
// to a block, whole.  Measured with the passes they replace (tile: 64-byte runs; N = 27*2^20, 16 segments of
// 1440 x 1536): 677 -> 199 us and 626 -> 189; N = 3*2^24, 32 of 1280 x 1536: 1000 MB in and out, 284 and 325;
// whole columns are 345 there, rows sixteen to a block 350.  Bound by latency and L1 gathers of twiddles
// (five reads a value), not by memory (half the rate of the factored forms').
template <typename S, typename... A> static int colsd(A... a)
{
  using SC = typename S::template Cap<(S::L <= 640 ? 64 : 1024)>;
  return launch_cols<WithForm<2, SC>, 8, false, float2>(a...);
}
template <typename S, typename... A> static int rowsd(A... a)
{
  return launch_rows<WithForm<2, S>, 8, (S::L <= 2560), float2>(a...);
}

extern "C" int soik_fft_longd_supported(int L, int rows)
{
#define SOI_X(N, ...) case N:
  switch (L) {
    SOI_FFT_LONGD(SOI_X)
      return 1;
    SOI_FFT_LONGD_ROWS(SOI_X)
      return rows;
    default: return 0;
  }
#undef SOI_X
}

extern "C" int soik_fft_longd_cols(float2 *data, const float2 *tw1, const float2 *thi,
                                   const float2 *tlo, int n1, int n2, int lb1, long Mh, int S,
                                   float2 *tout, long Mt, SoiBatch b, hipStream_t st)
{
  switch (n1) {
#define SOI_X(L, ...) \
    case L: return colsd<Sched<L, __VA_ARGS__>>(data, tw1, thi, tlo, n2, lb1, Mh, S, tout, Mt, b, st);
    SOI_FFT_LONGD(SOI_X)
#undef SOI_X
    default: return (int)hipErrorInvalidValue;
  }
}

extern "C" int soik_fft_longd_rows(const float2 *data, float2 *X, const float2 *tw2,
                                   const double2 *winv, int n1, int n2, long Mt, long M, int S,
                                   SoiBatch b, hipStream_t st)
{
  switch (n2) {
#define SOI_X(L, ...) \
    case L: return rowsd<Sched<L, __VA_ARGS__>>(data, X, tw2, winv, n1, Mt, M, S, b, st);
    SOI_FFT_LONGD(SOI_X) SOI_FFT_LONGD_ROWS(SOI_X)
#undef SOI_X
    default: return (int)hipErrorInvalidValue;
  }
}
