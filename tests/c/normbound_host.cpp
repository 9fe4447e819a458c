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
  if (!bad) std::printf("ok\n");
  return bad != 0;
}
