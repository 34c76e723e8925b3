// mcubes_edge.hpp -- where the refined grid's edge lies (rebin,
// vegasT.cuh:617-637), for the device's refinement (mcubes.hip) and its test
// on the host.
#pragma once

namespace pagani {
namespace mc {

// The point where the weights r[1..bins], linear inside the bins with right
// edges x[1..bins], sum to th + tl (two doubles, above zero and below the
// whole sum).  C[i] is r's prefix sum to twice the working precision, each
// entry added in an order of its own: over a run of bins of weight zero the
// entries are equal to rounding only and need not ascend, so the search may
// end in such a run when the sum falls on it.  A bin without weight holds no
// edge: the next one with weight takes it.
template <class DD>
__host__ __device__ inline double rebin_edge(const DD* C, const double* r, const double* x,
                                             int bins, double th, double tl)
{
#pragma clang fp contract(off)
  int k = 1;  // the first bin whose prefix sum is not below th + tl
  for (int end = bins; k < end;) {
    const int mid = (k + end) / 2;
    const DD m = C[mid];
    if (m.hi < th || (m.hi == th && m.lo < tl))
      k = mid + 1;
    else
      end = mid;
  }
  while (k < bins && r[k] == 0.0) ++k;
  if (r[k] == 0.0) return x[k];
  const double dr = (C[k].hi - th) + (C[k].lo - tl);
  return x[k] - (x[k] - x[k - 1]) * dr / r[k];
}

}  // namespace mc
}  // namespace pagani
