// Row pointer of a CRS matrix, looked over on the host.
#pragma once

#include <algorithm>
#include <cstdint>

namespace cghip {

// First row i with ptr[i + 1] < ptr[i], or -1 if there is none; then *longest
// is the number of entries of the longest row.  One pass without branches.
// The pointers themselves are compared: a difference of 32 bits wraps to a
// positive length where the pointer falls by more than 2^31, and from
// ptr[0] = 0 it can be back at any end after a few such rows.  Lengths are
// exact where nothing decreases (0 = ptr[0] <= ... <= ptr[n]).
inline int crs_rows(int n, const int *ptr, int *longest) {
  int most = 0;
  unsigned decreases = 0;
  for (int i = 0; i < n; i++) {
    decreases |= ptr[i + 1] < ptr[i];
    most = std::max(most, (int)((uint32_t)ptr[i + 1] - (uint32_t)ptr[i]));
  }
  *longest = most;
  if (decreases)
    for (int i = 0; i < n; i++)
      if (ptr[i + 1] < ptr[i]) return i;
  return -1;
}

}  // namespace cghip
