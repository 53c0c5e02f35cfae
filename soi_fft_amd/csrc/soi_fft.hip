// soi_fft.hip -- one-pass segment FFTs and what the planner asks about the register FFT lengths
// (see soi_fft.hpp).
#include "soi_fft.hpp"

using namespace soi;

namespace {

template <typename SC, typename C>
int launch_one(const C *at, C *X, const C *tw, const double2 *winv, long M, int S, SoiBatch b,
               hipStream_t st)
{
  hipLaunchKernelGGL((k_fft_one<SC, C>), dim3(S, b.n > 0 ? b.n : 1), dim3(SC::TS), 0, st, at, X, tw,
                     winv, M, b);
  return (int)hipGetLastError();
}

template <typename C, typename... A> int one_any(int L, A... a)
{
  switch (L) {
#define SOI_X(L, ...) \
  case L: return launch_one<Sched<L, __VA_ARGS__>, C>(a...);
    SOI_FFT_ONE(SOI_X)
#undef SOI_X
    default: return (int)hipErrorInvalidValue;
  }
}

}  // namespace

extern "C" int soik_fft_one(const double2 *at, double2 *X, const double2 *tw, const double2 *winv,
                            int L, long M, int S, SoiBatch b, hipStream_t st)
{
  return one_any<double2>(L, at, X, tw, winv, M, S, b, st);
}

extern "C" int soik_fft_one_f32(const float2 *at, float2 *X, const float2 *tw, const double2 *winv,
                                int L, long M, int S, SoiBatch b, hipStream_t st)
{
  return one_any<float2>(L, at, X, tw, winv, M, S, b, st);
}

// lengths the passes take: as columns (rows = 0), rows (1) or a whole segment (2)
extern "C" int soik_fft_reg_supported(int L, int rows)
{
#define SOI_X(N, ...) case N:
  switch (L) {
    SOI_FFT_SHORT(SOI_X) SOI_FFT_LONG(SOI_X) SOI_FFT_LONGEST(SOI_X)
      if (rows < 2) return 1;
  }
  switch (L) {
    SOI_FFT_ONE(SOI_X)
      if (rows == 2) return 1;
  }
#undef SOI_X
  return 0;
}

// alternative tiles of a length (variants 0 .. n - 1 of the launchers)
extern "C" int soik_fft_reg_variants(int L, int rows)
{
  if (L > 640 && L <= 1280) return 2;
  return L > 1280 && !rows ? 2 : 1;
}
