// Bound of log2 of a state's two-norm after amplitudes were written into it.
// Host C++ only (no HIP), so tests can run it on the CPU.
#pragma once

#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstring>

namespace qcs {

// the bits of n values, or-ed
inline uint64_t or_bits(const double *x, long n) {
  uint64_t r = 0;
  for (long i = 0; i < n; ++i) {
    uint64_t b;
    std::memcpy(&b, x + i, 8);
    r |= b;
  }
  return r;
}

// log2 of a bound of the two-norm of `count` written amplitudes, infinite
// where one of their values is infinite or NaN; `bits` are or_bits of the
// 2 * count values
inline double written_bound(const double *in, long count, uint64_t bits) {
  // |x| < 2 for every value unless some exponent says otherwise
  double top = 2.0;
  if (((bits >> 52) & 0x7ff) >= 0x400) {
    top = 0.0;
    for (long i = 0; i < 2 * count; ++i) {
      const double x = std::fabs(in[i]);
      if (!(x <= DBL_MAX)) return INFINITY;  // (as a maximum, NaN gives way to the next value)
      if (x > top) top = x;
    }
  }
  return std::log2(top) + 0.5 * std::log2(2.0 * double(count));
}

// The bound after such a write: `old` is the bound before it, which the
// amplitudes left as they were keep unless the `whole` state was written.  A
// NaN (a matrix with one was applied) bounds nothing, before and after.
inline double bound_after_write(double old, double written, bool whole) {
  if (whole) old = written;
  if (!(written < 1e300)) return written;  // infinite
  return (old <= written ? written : old) + 0.5;
}

}  // namespace qcs
