// soi_fft_cols32.hip -- pass 1 of the register FFT (see soi_fft.hpp), complex64.
#include "soi_fft.hpp"

extern "C" int soik_fft_cols_f32(float2 *data, const float2 *tw1, const float2 *thi, const float2 *tlo, int n1,
                             int n2, int lb1, long Mh, int S, int variant, float2 *tout, long Mt,
                             SoiBatch b, hipStream_t st)
{
  return soi::cols_any<float2>(n1, variant, data, tw1, thi, tlo, n2, lb1, Mh, S, tout, Mt, b, st);
}
