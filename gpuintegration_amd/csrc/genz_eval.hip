// genz_eval.hip -- precompiled evaluation kernels for the Genz descriptor
// path: 6 families x ndim 2..10 x {FP64, FP32 integrand}.
#include <hip/hip_runtime.h>

#include <cmath>

#include "pagani/eval_kernel.hpp"
#include "pagani/genz.hpp"
#include "genz_visit.hpp"
#include "pagani_ext.h"

// Each part of the source (PAGANI_PART, see build.py) holds the kernels of
// some dimensions at one precision; the part with dimension 2 at FP64 also
// dispatches.
namespace pagani {
namespace internal {

template <class Real, int D>
int genz_launch(const pagani_genz* g, const pagani_eval_args* a)
{
  return visit_genz<Real, D>(g, [&](const auto& f) {
    return pagani::eval_regions<D, std::decay_t<decltype(f)>, Real>(f, a);
  });
}

#define PAGANI_GENZ(Real, D) \
  template int genz_launch<Real, D>(const pagani_genz*, const pagani_eval_args*);
#if PAGANI_PART == 0
PAGANI_GENZ(double, 2)
PAGANI_GENZ(double, 3)
PAGANI_GENZ(double, 4)
PAGANI_GENZ(double, 5)
#elif PAGANI_PART == 1
PAGANI_GENZ(double, 6)
PAGANI_GENZ(double, 7)
#elif PAGANI_PART == 2
PAGANI_GENZ(double, 8)
PAGANI_GENZ(double, 9)
#elif PAGANI_PART == 3
PAGANI_GENZ(double, 10)
PAGANI_GENZ(float, 10)
PAGANI_GENZ(float, 2)
#elif PAGANI_PART == 4
PAGANI_GENZ(float, 3)
PAGANI_GENZ(float, 4)
PAGANI_GENZ(float, 5)
PAGANI_GENZ(float, 6)
#else
PAGANI_GENZ(float, 7)
PAGANI_GENZ(float, 8)
PAGANI_GENZ(float, 9)
#endif

#if PAGANI_PART == 0
#define PAGANI_GENZ_ELSEWHERE(Real, D) \
  extern template int genz_launch<Real, D>(const pagani_genz*, const pagani_eval_args*);
PAGANI_GENZ_ELSEWHERE(double, 6)
PAGANI_GENZ_ELSEWHERE(double, 7)
PAGANI_GENZ_ELSEWHERE(double, 8)
PAGANI_GENZ_ELSEWHERE(double, 9)
PAGANI_GENZ_ELSEWHERE(double, 10)
PAGANI_GENZ_ELSEWHERE(float, 2)
PAGANI_GENZ_ELSEWHERE(float, 3)
PAGANI_GENZ_ELSEWHERE(float, 4)
PAGANI_GENZ_ELSEWHERE(float, 5)
PAGANI_GENZ_ELSEWHERE(float, 6)
PAGANI_GENZ_ELSEWHERE(float, 7)
PAGANI_GENZ_ELSEWHERE(float, 8)
PAGANI_GENZ_ELSEWHERE(float, 9)
PAGANI_GENZ_ELSEWHERE(float, 10)

template <class Real>
int launch_dim(const pagani_genz* g, const pagani_eval_args* a)
{
  switch (g->ndim) {
  case 2: return genz_launch<Real, 2>(g, a);
  case 3: return genz_launch<Real, 3>(g, a);
  case 4: return genz_launch<Real, 4>(g, a);
  case 5: return genz_launch<Real, 5>(g, a);
  case 6: return genz_launch<Real, 6>(g, a);
  case 7: return genz_launch<Real, 7>(g, a);
  case 8: return genz_launch<Real, 8>(g, a);
  case 9: return genz_launch<Real, 9>(g, a);
  case 10: return genz_launch<Real, 10>(g, a);
  default: return PAGANI_EUNSUPPORTED;
  }
}
#endif

}  // namespace internal
}  // namespace pagani

#if PAGANI_PART == 0
extern "C" int pagani_genz_eval_launch(const pagani_genz* g, int precision,
                                       const pagani_eval_args* a)
{
  if (!g || !a) return PAGANI_EBADARG;
  if (precision == PAGANI_FP64) return pagani::internal::launch_dim<double>(g, a);
  if (precision == PAGANI_FP32) return pagani::internal::launch_dim<float>(g, a);
  return PAGANI_EBADARG;
}
#endif
