// bisect.h -- bisection of a descending sequence, for device code and the host's check of it.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#define PICARD_HD __host__ __device__ __forceinline__
#else
#define PICARD_HD inline
#endif

namespace picard {

// Entries of d[lo .. hi), descending, greater than q.  lo + hi may be beyond 2^31
// (positions among more than 2^30 particles), so the middle is taken from the difference.
template <typename D>
PICARD_HD int greater_in(const D &d, int lo, int hi, int32_t q) {
  const int first = lo;
  while (lo < hi) {
    const int mid = lo + ((hi - lo) >> 1);
    if (d[mid] > q) lo = mid + 1;
    else hi = mid;
  }
  return lo - first;
}

}  // namespace picard
