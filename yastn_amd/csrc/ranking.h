// The order of column norms and singular values: descending, ties by index, NaN together with infinity.  A total order, so
// that the ranks of any values are a permutation: the kernels read columns through its inverse, and a rank that no value
// has would leave an index unset (plain comparisons give every NaN the rank 0).
#pragma once

#include <math.h>
#include <stdint.h>

__host__ __device__ inline bool ranks_before(double x, int64_t i, double y, int64_t j) {
  const double a = x == x ? x : HUGE_VAL, b = y == y ? y : HUGE_VAL;
  return a > b || (a == b && i < j);
}
