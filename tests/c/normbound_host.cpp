// The bound of a state's two-norm after a write (qcs_amd/csrc/normbound.h):
// never below the norm, and not finite where a value is not.
#include <cstdio>
#include <vector>

#include "../../qcs_amd/csrc/normbound.h"

static int bad = 0;
static void check(bool ok, const char *what) {
  if (ok) return;
  std::printf("FAIL %s\n", what);
  ++bad;
}
static double bound(const std::vector<double> &v) {
  const long count = long(v.size()) / 2;
  return qcs::written_bound(v.data(), count, qcs::or_bits(v.data(), long(v.size())));
}

int main() {
  const double inf = INFINITY, nan = NAN;
  // a value that is not finite, at every place among ordinary and large ones
  for (double x : {inf, -inf, nan, -nan})
    for (double other : {0.0, 0.5, 1.9, 3.0, 1e300})
      for (size_t at = 0; at < 6; ++at) {
        std::vector<double> v(6, other);
        v[at] = x;
        check(!(bound(v) < 1e300), "a value that is not finite bounds nothing");
        v[(at + 1) % 6] = nan;
        check(!(bound(v) < 1e300), "two such values");
      }
  // the largest value wherever it stands
  for (double x : {1.5, 2.0, 8.0, 1e200, 1.7e308})
    for (size_t at = 0; at < 6; ++at) {
      std::vector<double> v(6, 0.25);
      v[at] = -x;
      check(bound(v) < 1e300 && bound(v) >= std::log2(x), "finite, and at least the largest value");
    }
  check(bound({1e300, nan, 1.0, 1.0}) > 900.0, "a large value before NaN");
  // a part of the state written: what was unbounded stays so, what was bounded
  // keeps the larger bound; the whole state written: the new values' bound
  for (double old : {nan, -nan, inf}) {
    check(!(qcs::bound_after_write(old, 3.0, false) < 1e300), "an unbounded rest");
    check(qcs::bound_after_write(old, 3.0, true) < 1e300, "all of it replaced");
  }
  for (double old : {-20.0, 0.0, 700.0})
    for (double w : {-20.0, 0.0, 700.0}) {
      const double want = 0.5 * std::log2(std::exp2(2 * old) + std::exp2(2 * w));
      const double b = qcs::bound_after_write(old, w, false);
      check(b < 1e300 && (want > 1e300 || b >= want - 1e-12), "both parts together");
      check(!(qcs::bound_after_write(old, inf, false) < 1e300), "an unbounded part");
    }
  if (!bad) std::printf("ok\n");
  return bad != 0;
}
