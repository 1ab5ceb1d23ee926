// pair_order.h -- order of a shell pair's primitive records.
#pragma once

namespace oqph {

// Decreasing |K|, NaN (a NaN coefficient) last: a comparison that is false both ways for
// a NaN is no order, and std::sort may then read and write outside its range.
inline bool larger_k(double x, double y) {
  x = __builtin_fabs(x);
  y = __builtin_fabs(y);
  return x > y || (x == x && y != y);
}

}  // namespace oqph
