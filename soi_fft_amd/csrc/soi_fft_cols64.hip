// soi_fft_cols64.hip -- pass 1 of the register FFT (see soi_fft.hpp), complex128.
#include "soi_fft.hpp"

extern "C" int soik_fft_cols(double2 *data, const double2 *tw1, const double2 *thi, const double2 *tlo, int n1,
                             int n2, int lb1, long Mh, int S, int variant, double2 *tout, long Mt,
                             SoiBatch b, hipStream_t st)
{
  return soi::cols_any<double2>(n1, variant, data, tw1, thi, tlo, n2, lb1, Mh, S, tout, Mt, b, st);
}
