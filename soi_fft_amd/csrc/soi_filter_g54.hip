// soi_filter_g54.hip -- the shapes of k_filter_g (soi_filter_g.hpp) with complex taps, mu = 5/4.
#include "soi_filter_g.hpp"

using namespace soi;

#define SHAPES(X) \
  X(4, 10) X(4, 13) X(4, 16) X(4, 20) X(4, 22) \
  X(8, 10) X(8, 13) X(8, 16) X(8, 20) X(8, 22) \
  X(16, 10) X(16, 13) X(16, 16) X(16, 20) X(16, 22) \
  X(32, 10) X(32, 13) X(32, 16) X(32, 20) X(32, 22) \
  X(64, 10) X(64, 13) X(64, 16) X(64, 20) X(64, 22)

// kind 0: launch; 1: B operand table
extern "C" int soik_filter_g54(const SoiFilterArgs *a, int kind, const double *taps, void *wt,
                              hipStream_t st)
{
#define X(S_, NK_) \
  if (a->S == S_ && a->nk == NK_) \
    return kind ? filter_g_table<FilterG<S_, 5, 4, NK_, true>>(taps, wt, a->NP * a->BP, st) \
                : filter_g_launch<FilterG<S_, 5, 4, NK_, true>>(a, st);
  SHAPES(X)
#undef X
  return (int)hipErrorInvalidValue;
}
