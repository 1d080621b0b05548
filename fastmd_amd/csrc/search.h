// Search of sorted keys, shared by the kernels and a host test.
#pragma once

#include <stdint.h>

// The first of `rows` sorted keys that is not below s (rows if none). The midpoint from the distance: for more
// than 2^30 rows lo + hi passes the 32-bit range, and half of the wrapped sum lies before the keys.
template <typename Keys>
__host__ __device__ __forceinline__ int32_t lower_bound(const Keys& key, int32_t rows, uint32_t s) {
  int32_t lo = 0, hi = rows;
  while (lo < hi) {
    const int32_t mid = lo + ((hi - lo) >> 1);
    if (key[mid] < s)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}
