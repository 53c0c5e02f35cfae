// soi_filter_g87.hip -- the shapes of k_filter_g (soi_filter_g.hpp) with complex taps, mu = 8/7.
#include "soi_filter_g.hpp"

using namespace soi;

#define SHAPES(X) \
  X(4, 16) X(4, 20) X(4, 22) \
  X(8, 16) X(8, 20) X(8, 22) \
  X(16, 16) X(16, 20) X(16, 22) \
  X(32, 16) X(32, 20) \
  X(64, 16) X(64, 20)

// kind 0: launch; 1: B operand table
extern "C" int soik_filter_g87(const SoiFilterArgs *a, int kind, const double *taps, void *wt,
                              hipStream_t st)
{
#define X(S_, NK_) \
  if (a->S == S_ && a->nk == NK_) \
    return kind ? filter_g_table<FilterG<S_, 8, 7, NK_, true>>(taps, wt, a->NP * a->BP, st) \
                : filter_g_launch<FilterG<S_, 8, 7, NK_, true>>(a, st);
  SHAPES(X)
#undef X
  return (int)hipErrorInvalidValue;
}
