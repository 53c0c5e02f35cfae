// soi_fft_rows64.hip -- pass 2 of the register FFT (see soi_fft.hpp), complex128.
#include "soi_fft.hpp"

extern "C" int soik_fft_rows(const double2 *data, double2 *X, const double2 *tw2, const double2 *winv, int n1,
                             int n2, long Mh, long M, int S, int variant, SoiBatch b,
                             hipStream_t st)
{
  return soi::rows_any<double2>(n2, variant, data, X, tw2, winv, n1, Mh, M, S, b, st);
}
