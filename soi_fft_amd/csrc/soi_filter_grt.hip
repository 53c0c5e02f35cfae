// soi_filter_grt.hip -- the shapes of k_filter_g (soi_filter_g.hpp) with real taps, mu = 5/4.
#include "soi_filter_g.hpp"

using namespace soi;

#define SHAPES(X) \
  X(4, 20) X(4, 22) \
  X(8, 20) X(8, 22) \
  X(16, 20) X(16, 22) \
  X(32, 20) X(32, 22) \
  X(64, 20) X(64, 22)

// kind 0: launch; 1: B operand table
extern "C" int soik_filter_grt(const SoiFilterArgs *a, int kind, const double *taps, void *wt,
                              hipStream_t st)
{
#define X(S_, NK_) \
  if (a->S == S_ && a->nk == NK_) \
    return kind ? filter_g_table<FilterG<S_, 5, 4, NK_, false>>(taps, wt, a->NP * a->BP, st) \
                : filter_g_launch<FilterG<S_, 5, 4, NK_, false>>(a, st);
  SHAPES(X)
#undef X
  return (int)hipErrorInvalidValue;
}
