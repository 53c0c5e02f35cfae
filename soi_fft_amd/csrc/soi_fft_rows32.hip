// soi_fft_rows32.hip -- pass 2 of the register FFT (see soi_fft.hpp), complex64.
#include "soi_fft.hpp"

extern "C" int soik_fft_rows_f32(const float2 *data, float2 *X, const float2 *tw2, const double2 *winv, int n1,
                             int n2, long Mh, long M, int S, int variant, SoiBatch b,
                             hipStream_t st)
{
  return soi::rows_any<float2>(n2, variant, data, X, tw2, winv, n1, Mh, M, S, b, st);
}
