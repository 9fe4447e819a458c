// The queue of plain gates: gates are pushed and the planner's passes taken
// from its head at the sizes queue_next_look names, as the backend does, and
// the queue never holds more than kQueueMax gates.
#include <cstdio>

#include "../../qcs_amd/csrc/gateplan.h"

using namespace qcs;

// `count` gates on n qubits: CNOTs alone (they take no room in a program, so
// the pass of a state of one tile never closes), or H gates with CNOTs between
static size_t longest(int n, int tb, int rb, int count, bool maps) {
  const double r = std::sqrt(0.5);
  const double x[8] = {0, 0, 1, 0, 1, 0, 0, 0}, h[8] = {r, 0, r, 0, r, 0, -r, 0};
  std::vector<PlanGate> q;
  std::vector<PassGroup> groups;
  PassPick pick;
  size_t look = kQueueLow, most = 0;
  for (int i = 0; i < count; ++i) {
    const int t = i % n, c = (t + 1 + i / n % (n - 1)) % n;
    q.push_back(maps || i % 3 ? plan_gate(QCS_HIP_G_CU, t, c, x)
                              : plan_gate(QCS_HIP_G_1Q, t, -1, h));
    most = std::max(most, q.size());
    if (q.size() < look) continue;
    bool open = false;
    while (q.size() >= kQueueLow) {
      plan_pick(q, n, tb, 4, 2, 64, &pick, &groups, n > tb, rb);
      if (!pick.full && q.size() < kQueueMax) {
        open = true;
        break;
      }
      std::vector<char> gone(q.size(), 0);
      for (int k : pick.gates) gone[size_t(k)] = 1;
      for (int k : pick.swaps) gone[size_t(k)] = 1;
      if (pick.gates.empty() && pick.swaps.empty()) gone[0] = 1;
      std::vector<PlanGate> rest;
      for (size_t k = 0; k < q.size(); ++k)
        if (!gone[k]) rest.push_back(q[k]);
      q.swap(rest);
    }
    look = queue_next_look(q.size(), open);
    if (look <= q.size()) {
      std::printf("FAIL: the next look at %zu of %zu gates\n", look, q.size());
      return size_t(-1);
    }
  }
  return most;
}

int main() {
  int bad = 0;
  for (bool maps : {true, false})
    for (int n : {7, 10, 12, 14, 20}) {
      const int tb = n <= 12 ? n : n < 20 ? 10 : 12;
      const size_t most = longest(n, tb, tb <= 11 ? 2 : 4, 4000, maps);
      if (most > kQueueMax) {
        std::printf("FAIL: %d qubits, %s: %zu gates queued\n", n, maps ? "CNOT" : "H, CNOT", most);
        bad = 1;
      }
    }
  if (!bad) std::printf("ok\n");
  return bad;
}
