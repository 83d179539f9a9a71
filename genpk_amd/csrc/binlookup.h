// Bin lookup of an integer |k|^2 = q from thresholds staged in LDS, shared
// by the fused binning and the adjoint's fused weight.
#pragma once
#include <hip/hip_runtime.h>

namespace genpk {

// LDS thresholds that bin_lds reads.
__host__ __device__ inline int bin_lds_slots(int nrbins) { return nrbins > 2 ? nrbins : 2; }

// Bin of q >= 1 from LDS copies of the thresholds (thr32[b] = smallest q whose
// bin is >= b, b < bin_lds_slots).  The estimate lq * log2(q) of the exact bin
// coordinate is off by less than a few parts in 10^7 of it, below 0.01 bins
// for the 8192 bins that are allowed, so it names the bin or a neighbour and
// two thresholds settle which: no branch, and the lookups of a run of modes
// overlap.  (Tracking the bin along a run and searching when it ends made
// nearly every wave take the search at every mode, some lane always crossing
// an edge: the x pass + bin took 0.120 ms so and 0.106 this way at 360^3 FP32,
// 0.079 and 0.070 at 320^3.)
__device__ __forceinline__ int bin_lds(int q, const int *thr32, int nrbins, float lq) {
  const int b = min((int)(lq * __log2f((float)q)), max(nrbins - 2, 0));
  return b + (q >= thr32[b + 1] ? 1 : 0) - (q < thr32[b] ? 1 : 0);
}

}  // namespace genpk
