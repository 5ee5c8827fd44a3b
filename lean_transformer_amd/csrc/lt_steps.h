// Which k-steps of a reduction in one or two segments are whole.  Plain C++, so that it can be tested on the host.
#pragma once
#include <cstdint>

#ifdef __HIP__
#define LT_HOST_DEVICE __host__ __device__
#else
#define LT_HOST_DEVICE
#endif

// Each segment takes ceil(k / step) k-steps of its own, the second's after the first's; the last of a segment is ragged where step
// does not divide its length.  Number of leading steps that are whole (k1 == 0: one segment).
LT_HOST_DEVICE inline int lt_leading_whole_steps(int64_t k0, int64_t k1, int step) {
  const int first = (int)((k0 + step - 1) / step);
  if (k0 % step != 0) return first - 1;
  return first + (int)(k1 / step);
}
