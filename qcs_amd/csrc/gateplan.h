// Host planner of the gate passes (gatepass.hip): cuts a list of plain gates
// into passes over HBM and writes the program each pass runs.  Host C++ only
// (no HIP), so tests can run the plans on the CPU.
//
// A pass holds a tile of 2^tb amplitudes in the registers of a work-group,
// 16 to a thread (rb = 4, fewer for small tiles): rb of the tile's index bits select the register
// ("register bits"), the others the thread.  A gate that mixes amplitudes
// needs its target among the register bits; a diagonal gate, and a control,
// may sit anywhere, since an amplitude's index bits are known.  Between two
// choices of register bits (layouts) the tile is exchanged through LDS.
//
// Order.  The amplitudes have to equal those of the gates applied one after
// another, bit for bit, so two gates change places only where that is exact:
// on different qubits, and one of them only moves amplitudes or multiplies
// them by +-1 or +-i.  CNOTs and SWAPs are maps of the tile's index, linear
// over GF(2): they run as address maps of an exchange or of the final store
// and cost no arithmetic.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <vector>

#include "../../include/qcs_hip.h"

namespace qcs {

constexpr int kPRegBits = 4;               // register bits of a layout, at most
constexpr int kPMaxTile = 12;              // tile bits, at most
constexpr int kPThrBits = 9;               // thread bits, at most
constexpr int kPLineBits = 3;              // 8 amplitudes: a 128-byte line (complex128)
constexpr int kPMaxSwaps = 16;             // SWAPs of two bits outside the tile per pass
constexpr int kPMaxTerms = 6;              // controls outside the tile per exchange
constexpr int kPWords = 848;               // program words of a pass
constexpr int kPPad = 17;                  // words read past the last op

// The queue of gates that are not launched yet.
constexpr size_t kQueueLow = 96;     // gates kept back to plan the next pass
constexpr size_t kQueueStep = 64;    // gates to the next look at a queue whose pass is still open,
constexpr size_t kQueueNext = 8;     // and after one that launched what it could (64: the device
                                     // waited for the next pass, 17 qubits 283 -> 270 us)
constexpr size_t kQueueMax = 1024;   // a queue of this size is launched from, open or not
// The size at which a queue is next looked at: now it holds `size` gates, and
// `open` if its next pass would take more of them.
inline size_t queue_next_look(size_t size, bool open) {
  return std::min(kQueueMax, std::max(kQueueLow, size + (open ? kQueueStep : kQueueNext)));
}

// A gate as the planner sees it.  kGCuDense (a controlled matrix that is
// neither X nor a phase; no qc_* gate makes one) is not planned: it runs by
// itself.
enum : uint8_t {
  kGDense, kGReal, kGAnti, kGDiag, kGPhase, kGCuDense, kGCPhase, kGCnot, kGSwap
};
struct PlanGate {
  uint8_t cls;
  uint8_t exact;  // a permutation times +-1 or +-i
  int8_t t, c;
  uint64_t qubits;  // every qubit it acts on
  uint64_t need;    // qubits that have to be tile bits
  double m[8];
};

// Program of a pass: layout records, each followed by its ops.
// Op word: kind | words of the op << 5 | u1 << 10 | u2 << 16 | l1 << 22 |
// l2 << 25, then the parameters in the state's precision.  Conditions: bits
// u1, u2 of the wave's uniform word (pass_uniform) and lane bits l1, l2 have to
// be set.
enum : uint8_t {
  kPDense = 0,     // + register bit: m[0..7]
  kPReal = 4,      // m00, m01, m10, m11 (real parts)
  kPAnti = 8,      // m01, m10
  kPDiag = 12,     // m00, m11
  kPPhase = 16,    // m11; under conditions
  kPEuler = 20,    // diag(a, conj a), [[c, s], [-s, c]], diag(b, conj b)
  kPCPhase = 24,   // + pair index of two register bits: m11
  kPScale = 30,    // every amplitude, under conditions: m11
  kPSelect = 31    // every amplitude: conditions ? m11 : m00
};
// What a whole wave shares: the index bits outside the tile, above them the
// thread bits past the lane's, and a bit that is always set.
constexpr int kPLaneBits = 6, kPWaveBit = 40, kPAlways = 63;
constexpr int kPNoLane = 7;
constexpr uint64_t pass_uniform(uint64_t base, unsigned wave) {
  return base | uint64_t(wave) << kPWaveBit | uint64_t(1) << kPAlways;
}
// condition: lane bit b, or 64 + a bit of the uniform word
constexpr int kPNoCond = 255;

// Layout record, in whole words (scalar loads are 32 bits and up).  A pair
// belongs to the exchange that follows the layout: in the upper half the LDS
// byte offset a thread or register bit of this layout is written to, in the
// lower half the one it reads as a bit of the next layout.
struct PassLayout {
  uint32_t thr[kPThrBits], reg[kPRegBits];
  // words that follow the record: ops, then terms of the exchange (index bit |
  // offset << 16: written offsets change where the bit is set)
  uint32_t nterm, opwords;
};
constexpr int kPLayoutWords = int(sizeof(PassLayout) / 4);

struct PassProgram {
  uint32_t tb;
  uint32_t nlayouts;
  // Tiles: number t has its bits at the set bits of `outer` (ascending) and on
  // the bits of `swaps`, and `fixed` elsewhere outside the tile (pass_tile).
  uint64_t outer, fixed;
  // Amplitudes of the tile that are zero without being so in memory: where
  // the index differs from `basis` in a bit of skip_t (thread bits) or skip_r
  // (register bits).
  uint64_t skip_t, skip_r, basis;
  uint64_t load_t[kPThrBits], load_r[kPRegBits];    // index masks of the first layout
  uint64_t store_t[kPThrBits], store_r[kPRegBits];  // index masks (XOR) of the last layout
  uint64_t store_term[kPMaxTerms];                  // XOR where index bit store_q is set
  uint32_t store_q[kPMaxTerms];
  // SWAPs of two index bits outside the tile (pairs of tiles change places)
  uint32_t nswaps, swaps[kPMaxSwaps];  // low bit | high bit << 8
  uint32_t rb;                         // register bits
  uint32_t store_nterm;
  uint32_t store_add;  // the registers' masks share no bit with others: XOR is addition
  uint32_t words[kPWords + kPPad];
};
static_assert(sizeof(PassProgram) <= 4096 - 16, "a pass program travels as a kernel argument");

// Work-groups of a pass.  Without SWAPs outside the tile each takes a tile.
// With p of them it takes a tile and the one it changes places with, and there
// is one for each such pair: numbered, above the bits of `outer`, by the first
// SWAP whose two bits differ (of the pair, the tile with its low bit set is
// the work-group's first), the equal bits of the SWAPs before it and any bits
// of those after it; last come the tiles that stay where they are.
// (constexpr: host and device code)
template <typename P>
constexpr uint64_t pass_work_groups(const P prog, int outer_bits) {
  const int p = int(prog->nswaps);
  uint64_t g = uint64_t(1) << p;
  for (int k = 0; k < p; ++k) g += uint64_t(1) << (2 * p - 2 - k);
  return g << outer_bits;
}
template <typename P>
constexpr uint64_t pass_tile(const P prog, uint64_t t) {
  uint64_t base = prog->fixed;
  for (uint64_t o = prog->outer; o; o &= o - 1, t >>= 1)
    if (t & 1) base |= o & (~o + 1);
  const int p = int(prog->nswaps);
  int first = 0;
  for (; first < p; ++first) {
    const uint64_t count = uint64_t(1) << (2 * p - 2 - first);
    if (t < count) break;
    t -= count;
  }
  for (int k = 0; k < p; ++k) {
    const uint32_t lo = prog->swaps[k] & 255, hi = prog->swaps[k] >> 8;
    uint64_t bits = 1;  // low bit, then high bit
    if (k < first) bits = (t & 1) * 3, t >>= 1;
    else if (k > first) bits = t & 3, t >>= 2;
    base |= (bits & 1) << lo | bits >> 1 << hi;
  }
  return base;
}
// where the tile is stored
template <typename P>
constexpr uint64_t pass_home(const P prog, uint64_t base) {
  for (uint32_t k = 0; k < prog->nswaps; ++k) {
    const uint32_t lo = prog->swaps[k] & 255, hi = prog->swaps[k] >> 8;
    const uint64_t d = (base >> lo ^ base >> hi) & 1;
    base ^= d << lo | d << hi;
  }
  return base;
}

// XOR swizzle of an LDS slot (8 bytes): bits 5.. fold onto the low five, so
// that 32 lanes whose positions have independent vectors use 32 slots that
// differ modulo 32.
inline int pass_bank(int p) {
  static const int v[kPMaxTile] = {1, 2, 4, 8, 16, 1, 2, 4, 8, 16, 9, 18};
  return v[p];
}
inline int pass_slot(int e) {
  int s = e;
  for (e >>= 5; e; e &= e - 1) s ^= pass_bank(5 + __builtin_ctz(unsigned(e)));
  return s;
}

inline bool plan_unit(double re, double im) {  // +-1 or +-i
  return (im == 0.0 && (re == 1.0 || re == -1.0)) || (re == 0.0 && (im == 1.0 || im == -1.0));
}

inline PlanGate plan_gate(int kind, int target, int control, const double *m) {
  PlanGate g;
  std::memset(&g, 0, sizeof(g));
  g.t = int8_t(target);
  g.c = int8_t(kind == QCS_HIP_G_1Q ? -1 : control);
  g.qubits = uint64_t(1) << target;
  if (kind != QCS_HIP_G_1Q) g.qubits |= uint64_t(1) << control;
  g.need = uint64_t(1) << target;
  if (kind == QCS_HIP_G_SWAP) {
    g.cls = kGSwap;
    g.exact = 1;
    g.need = g.qubits;
    return g;
  }
  std::memcpy(g.m, m, sizeof(g.m));
  const bool z01 = m[2] == 0.0 && m[3] == 0.0, z10 = m[4] == 0.0 && m[5] == 0.0;
  const bool z00 = m[0] == 0.0 && m[1] == 0.0, z11 = m[6] == 0.0 && m[7] == 0.0;
  g.exact = (z01 && z10 && plan_unit(m[0], m[1]) && plan_unit(m[6], m[7])) ||
            (z00 && z11 && plan_unit(m[2], m[3]) && plan_unit(m[4], m[5]));
  // diag(1, x) and X are told apart as the per-gate kernels do
  const bool phase = m[0] == 1.0 && m[1] == 0.0 && z01 && z10;
  if (kind == QCS_HIP_G_CU) {
    const bool x = z00 && m[2] == 1.0 && m[3] == 0.0 && m[4] == 1.0 && m[5] == 0.0 && z11;
    g.cls = x ? kGCnot : phase ? kGCPhase : kGCuDense;
    if (phase) g.need = 0;
    return g;
  }
  if (phase) g.cls = kGPhase;
  else if (z01 && z10) g.cls = kGDiag;
  else if (m[1] == 0.0 && m[3] == 0.0 && m[5] == 0.0 && m[7] == 0.0) g.cls = kGReal;
  else if (z00 && z11) g.cls = kGAnti;
  else g.cls = kGDense;
  if (g.cls == kGPhase || g.cls == kGDiag) g.need = 0;
  return g;
}

// Fraction of the state's bytes (read + write = 2) the per-gate kernels move
// for a gate: what a pass has to beat.
inline double plan_gate_traffic(const PlanGate &g) {
  switch (g.cls) {
    case kGPhase: case kGCnot: case kGSwap: return 1.0;
    case kGCPhase: return 0.5;
    default: return 2.0;
  }
}

inline bool plan_same_bits(double a, double b) { return std::memcmp(&a, &b, sizeof(a)) == 0; }
// the repeated entries of an RZ and of an RY
inline bool plan_z_like(const PlanGate &g) {
  return g.cls == kGDiag && plan_same_bits(g.m[6], g.m[0]) && plan_same_bits(g.m[7], -g.m[1]);
}
inline bool plan_y_like(const PlanGate &g) {
  return g.cls == kGReal && plan_same_bits(g.m[6], g.m[0]) && plan_same_bits(g.m[4], -g.m[2]);
}

inline int plan_op_words(const PlanGate &g, int param_words) {  // an upper bound
  switch (g.cls) {
    case kGDense: return 1 + 8 * param_words;
    case kGReal: case kGAnti: case kGDiag: return 1 + 4 * param_words;
    case kGPhase: case kGCPhase: return 1 + 2 * param_words;
    default: return 0;
  }
}

// Qubits along which a gate can move weight to amplitudes that were zero.
inline uint64_t plan_spread(const PlanGate &g) {
  return g.cls == kGSwap ? g.qubits : g.cls == kGCuDense ? uint64_t(1) << g.t : g.need;
}

// What a pass takes from the head of a gate list.
struct PassPick {
  std::vector<int> gates;  // indices, in the order they run
  uint64_t bits;           // tile bits
  bool full;               // the next gate does not fit: more gates would not change the pick
  std::vector<int> swaps;  // SWAPs of two qubits outside the tile, after the others
  uint64_t swapped;        // their qubits
  int rb;                  // register bits of the layouts
};

// One group: ops on at most rb register qubits, then index maps.
struct PassGroup {
  std::vector<int> ops;   // indices into the gate list
  std::vector<int> maps;  // CNOTs and SWAPs, applied after the ops
  uint64_t regs = 0, mapped = 0;
};

// Appends gate g to the groups (opening a new one where it has to); returns
// false when it cannot, because of the exchange's limit of outside terms.
inline bool plan_add(std::vector<PassGroup> &gs, const std::vector<PlanGate> &gates, int i,
                     uint64_t tile, int words_left, int rb) {
  const PlanGate &g = gates[size_t(i)];
  if (gs.empty()) gs.emplace_back();
  PassGroup *cur = &gs.back();
  if (g.cls == kGCnot || g.cls == kGSwap) {
    if (g.cls == kGCnot && !((tile >> g.c) & 1)) {
      // distinct outside controls of the maps pending here
      uint64_t outs = uint64_t(1) << g.c;
      for (int k : cur->maps)
        if (gates[size_t(k)].cls == kGCnot && !((tile >> gates[size_t(k)].c) & 1))
          outs |= uint64_t(1) << gates[size_t(k)].c;
      if (__builtin_popcountll(outs) > kPMaxTerms) {
        if (words_left < 2 * kPLayoutWords) return false;
        gs.emplace_back();
        cur = &gs.back();
      }
    }
    cur->maps.push_back(i);
    cur->mapped |= g.qubits;
    return true;
  }
  const uint64_t reg = g.need;  // the target of a gate that mixes amplitudes
  const bool fits = !(g.qubits & cur->mapped) &&
                    __builtin_popcountll(cur->regs | reg) <= rb;
  if (!fits) {
    if (words_left < 2 * kPLayoutWords) return false;
    gs.emplace_back();
    cur = &gs.back();
  }
  cur->ops.push_back(i);
  cur->regs |= reg;
  return true;
}

// The gates of the next pass: in order, each that fits the tile and may run
// before the ones left behind.  `scan` bounds how far past the first gate
// left behind the list is searched for gates that may overtake it.  With
// `pairs`, a SWAP of two qubits outside the tile needs no tile bits: the pass
// stores the tiles it relates in each other's place, and leaves later gates on
// its qubits behind.
inline void plan_pick(const std::vector<PlanGate> &gates, int n, int tb, int low,
                      int param_words, int scan, PassPick *out, std::vector<PassGroup> *groups,
                      bool pairs = false, int rb = kPRegBits) {
  uint64_t tile = (uint64_t(1) << (low < n ? low : n)) - 1;
  if (tb >= n) tile = (uint64_t(1) << n) - 1;
  uint64_t left = 0;  // qubits of the gates left behind
  bool left_inexact = false;
  int words = 0, past = 0;
  out->gates.clear();
  out->full = false;
  out->swaps.clear();
  out->swapped = 0;
  out->rb = rb;
  groups->clear();
  // the layouts of the load and the store besides the groups'
  const int budget = kPWords - 2 * kPLayoutWords;
  for (size_t i = 0; i < gates.size(); ++i) {
    const PlanGate &g = gates[i];
    bool take = !(g.qubits & (left | out->swapped)) && (g.exact || !left_inexact);
    if (take && pairs && g.cls == kGSwap && !(g.qubits & tile) &&
        int(out->swaps.size()) < kPMaxSwaps) {
      out->swaps.push_back(int(i));
      out->swapped |= g.qubits;
      continue;
    }
    if (take) {
      const int w = words + plan_op_words(g, param_words);
      const int room = budget - w - int(groups->size()) * kPLayoutWords;
      if (__builtin_popcountll(tile | g.need) > tb || room < kPLayoutWords) take = false;
      // a control outside the tile now must not become a tile bit later: the
      // maps read it as one or the other, so the final tile decides (below)
      if (take) {
        tile |= g.need;
        words = w;
        out->gates.push_back(int(i));
      }
    }
    if (!take) {
      left |= g.qubits;
      left_inexact = left_inexact || !g.exact;
    }
    if (left_inexact && ++past > scan) break;
  }
  out->full = left_inexact;
  // fill the tile with the lowest unused bits (longer runs)
  for (int q = 0; q < n && __builtin_popcountll(tile) < tb; ++q)
    tile |= (uint64_t(1) << q) & ~out->swapped;
  if (__builtin_popcountll(tile) < (tb < n ? tb : n)) {  // the swapped qubits have to fill it
    plan_pick(gates, n, tb, low, param_words, scan, out, groups, false, rb);
    return;
  }
  out->bits = tile;
  // groups, with the final tile
  size_t used = 0;
  words = 0;
  for (; used < out->gates.size(); ++used) {
    const int i = out->gates[used];
    const PlanGate &g = gates[size_t(i)];
    words += plan_op_words(g, param_words);
    if (g.cls == kGCnot && !((tile >> g.c) & 1)) ++words;  // a term, at most
    const int room = budget - words - int(groups->size()) * kPLayoutWords;
    if (room < kPLayoutWords || !plan_add(*groups, gates, i, tile, room, rb)) {
      out->full = true;
      break;
    }
  }
  // gates that no longer fit: only the ones before them in the run order go.
  // The rest stay in the list in their order; what was taken ran before them
  // legally, since it ran before them in `gates` order of the pick as well.
  // A SWAP set aside may have followed one of them.
  while (used < out->gates.size() && !out->swaps.empty() &&
         out->swaps.back() > out->gates[used]) {
    out->swapped &= ~gates[size_t(out->swaps.back())].qubits;
    out->swaps.pop_back();
  }
  out->gates.resize(used);
  if (groups->empty()) groups->emplace_back();
}

// ---- writing the program ---------------------------------------------------

struct LayoutMap {
  int reg[kPRegBits];  // tile positions of the register bits, ascending
  int thr[kPThrBits];  // tile positions of the thread bits
  int nthr, nreg;
  int thread_bit(int pos) const {
    for (int b = 0; b < nthr; ++b)
      if (thr[b] == pos) return b;
    return -1;
  }
  int reg_bit(int pos) const {
    for (int b = 0; b < nreg; ++b)
      if (reg[b] == pos) return b;
    return -1;
  }
  bool io() const { return reg[0] >= kPLineBits; }  // threads 0..7 cover a line
};

// `need`: tile positions.  Free register bits go to the highest positions,
// which keeps the low ones for the lanes.
inline LayoutMap make_layout(unsigned need, int tb, int rb) {
  LayoutMap m;
  unsigned regs = need;
  for (int p = tb - 1; p >= 0 && __builtin_popcount(regs) < rb; --p)
    regs |= 1u << p;
  int r = 0, rest[kPMaxTile], nrest = 0;
  for (int p = 0; p < tb; ++p) {
    if ((regs >> p) & 1) m.reg[r++] = p;
    else rest[nrest++] = p;
  }
  m.nthr = nrest;
  m.nreg = r;
  // lanes: the first four positions' bank vectors independent modulo 16,
  // five modulo 32, taking the lowest positions that are
  int norder = 0;  // m.thr
  bool used[kPMaxTile] = {false};
  int basis[5] = {0, 0, 0, 0, 0};
  for (int want = 0, mask = 15; want < 5; ++want) {
    if (want == 4) {
      mask = 31;  // redo the basis in the larger space
      for (int &b : basis) b = 0;
      for (int b = 0; b < norder; ++b) {
        int v = pass_bank(m.thr[b]);
        for (int k = 4; k >= 0; --k)
          if ((v >> k) & 1) {
            if (!basis[k]) { basis[k] = v; break; }
            v ^= basis[k];
          }
      }
    }
    for (int x = 0; x < nrest; ++x) {
      if (used[x]) continue;
      int v = pass_bank(rest[x]) & mask;
      for (int k = 4; k >= 0; --k)
        if (((v >> k) & 1) && basis[k]) v ^= basis[k] & mask;
      if (!v) continue;
      for (int k = 4; k >= 0; --k)
        if ((v >> k) & 1) { basis[k] = v; break; }
      used[x] = 1;
      m.thr[norder++] = rest[x];
      break;
    }
  }
  for (int x = 0; x < nrest; ++x)
    if (!used[x]) m.thr[norder++] = rest[x];
  return m;
}

// Index map of the pending CNOTs and SWAPs over the tile's positions.
struct IndexMap {
  int col[kPMaxTile];
  int nterm;
  uint8_t termq[kPMaxTerms];
  int termv[kPMaxTerms];
};

inline IndexMap make_map(const std::vector<PlanGate> &gates, const std::vector<int> &maps,
                         const int *pos, uint64_t tile) {
  IndexMap a;
  for (int p = 0; p < kPMaxTile; ++p) a.col[p] = 1 << p;
  a.nterm = 0;
  for (int i : maps) {
    const PlanGate &g = gates[size_t(i)];
    const int t = pos[int(g.t)];
    if (g.cls == kGCnot && !((tile >> g.c) & 1)) {
      int k = 0;
      while (k < a.nterm && a.termq[k] != uint8_t(g.c)) ++k;
      if (k == a.nterm) {
        a.termq[k] = uint8_t(g.c);
        a.termv[k] = 0;
        ++a.nterm;
      }
      a.termv[k] ^= 1 << t;
      continue;
    }
    const int c = pos[int(g.c)];
    auto apply = [&](int &v) {
      const int bc = (v >> c) & 1, bt = (v >> t) & 1;
      if (g.cls == kGCnot) v ^= bc << t;
      else if (bc != bt) v ^= (1 << c) | (1 << t);
    };
    for (int p = 0; p < kPMaxTile; ++p) apply(a.col[p]);
    for (int k = 0; k < a.nterm; ++k) apply(a.termv[k]);
  }
  return a;
}

template <typename T>
inline void put_op(uint32_t *&w, int kind, int c1, int c2, const T *par, int npar) {
  const int words = 1 + npar * int(sizeof(T) / 4);
  int u[2] = {kPAlways, kPAlways}, l[2] = {kPNoLane, kPNoLane}, nu = 0, nl = 0;
  for (int c : {c1, c2}) {
    if (c == kPNoCond) continue;
    if (c < 64) l[nl++] = c;
    else u[nu++] = c - 64;
  }
  *w++ = uint32_t(kind | words << 5 | u[0] << 10 | u[1] << 16 | l[0] << 22 | l[1] << 25);
  std::memcpy(w, par, size_t(npar) * sizeof(T));
  w += words - 1;
}

// Ops of one group in layout m.
template <typename T>
inline void write_ops(const std::vector<PlanGate> &gates, const std::vector<int> &ops,
                      const LayoutMap &m, const int *pos, uint64_t tile, uint32_t *&w) {
  auto cond = [&](int q) {
    if (!((tile >> q) & 1)) return 64 + q;
    const int b = m.thread_bit(pos[q]);
    return b < kPLaneBits ? b : 64 + kPWaveBit + b - kPLaneBits;
  };
  auto reg = [&](int q) { return ((tile >> q) & 1) ? m.reg_bit(pos[q]) : -1; };
  for (size_t x = 0; x < ops.size(); ++x) {
    const PlanGate &g = gates[size_t(ops[x])];
    T v[8];
    for (int k = 0; k < 8; ++k) v[k] = T(g.m[k]);
    const int t = g.t, rt = reg(t);
    if (x + 2 < ops.size() && rt >= 0) {
      const PlanGate &y = gates[size_t(ops[x + 1])], &z = gates[size_t(ops[x + 2])];
      if (y.t == g.t && z.t == g.t && plan_z_like(g) && plan_y_like(y) && plan_z_like(z)) {
        const T e[6] = {T(g.m[0]), T(g.m[1]), T(y.m[0]), T(y.m[2]), T(z.m[0]), T(z.m[1])};
        put_op(w, kPEuler + rt, kPNoCond, kPNoCond, e, 6);
        x += 2;
        continue;
      }
    }
    const T diag[4] = {v[0], v[1], v[6], v[7]};
    switch (g.cls) {
      case kGDense: put_op(w, kPDense + rt, kPNoCond, kPNoCond, v, 8); break;
      case kGReal: {
        const T r[4] = {v[0], v[2], v[4], v[6]};
        put_op(w, kPReal + rt, kPNoCond, kPNoCond, r, 4);
        break;
      }
      case kGAnti: put_op(w, kPAnti + rt, kPNoCond, kPNoCond, v + 2, 4); break;
      case kGDiag:
        if (rt >= 0) put_op(w, kPDiag + rt, kPNoCond, kPNoCond, diag, 4);
        else put_op(w, kPSelect, cond(t), kPNoCond, diag, 4);
        break;
      case kGPhase:
        if (rt >= 0) put_op(w, kPPhase + rt, kPNoCond, kPNoCond, v + 6, 2);
        else put_op(w, kPScale, cond(t), kPNoCond, v + 6, 2);
        break;
      default: {  // kGCPhase: symmetric in its two qubits
        const int rc = reg(g.c);
        if (rt >= 0 && rc >= 0) {
          static const int pair[4][4] = {{0, 0, 1, 2}, {0, 0, 3, 4}, {1, 3, 0, 5}, {2, 4, 5, 0}};
          put_op(w, kPCPhase + pair[rc][rt], kPNoCond, kPNoCond, v + 6, 2);
        } else if (rt >= 0) {
          put_op(w, kPPhase + rt, cond(g.c), kPNoCond, v + 6, 2);
        } else if (rc >= 0) {
          put_op(w, kPPhase + rc, cond(t), kPNoCond, v + 6, 2);
        } else {
          put_op(w, kPScale, cond(g.c), cond(t), v + 6, 2);
        }
      }
    }
  }
}

// The program of a pass.  Amplitudes whose index differs from `basis` in a bit
// outside `support` are zero (and stay so): the pass runs the other tiles.
// Where `filled` is not all ones, memory holds only the amplitudes that agree
// with `basis` outside `filled` (which includes `support`): the pass runs
// their tiles and reads nothing else; afterwards the tile bits are filled too.
template <typename T>
inline void write_pass(const std::vector<PlanGate> &gates, const PassPick &pick,
                       const std::vector<PassGroup> &groups, int n, int tb, uint64_t support,
                       uint64_t basis, PassProgram *pp, uint64_t filled = ~uint64_t(0)) {
  std::memset(pp, 0, offsetof(PassProgram, words));
  pp->tb = uint32_t(tb);
  pp->rb = uint32_t(pick.rb);
  const uint64_t all = n < 64 ? (uint64_t(1) << n) - 1 : ~uint64_t(0);
  if (~filled & all) support = filled;
  support |= pick.swapped;
  pp->nswaps = uint32_t(pick.swaps.size());
  for (size_t k = 0; k < pick.swaps.size(); ++k) {
    const PlanGate &g = gates[size_t(pick.swaps[k])];
    pp->swaps[k] = uint32_t(g.t) | uint32_t(g.c) << 8;
  }
  pp->outer = support & all & ~(pick.bits | pick.swapped);
  pp->fixed = basis & all & ~(support | pick.bits);
  int pos[64], bits[kPMaxTile];
  for (int &p : pos) p = -1;
  int np = 0;
  for (int q = 0; q < 64; ++q)
    if ((pick.bits >> q) & 1) {
      pos[q] = np;
      bits[np++] = q;
    }
  auto positions = [&](uint64_t qubits) {
    unsigned r = 0;
    for (qubits &= pick.bits; qubits; qubits &= qubits - 1) r |= 1u << pos[__builtin_ctzll(qubits)];
    return r;
  };
  // the layouts: the groups', with one of the load and one of the store
  // added where a group's does not read or write whole lines
  struct Step {
    LayoutMap m;
    const PassGroup *g;
    IndexMap a;
  };
  std::vector<Step> steps;
  steps.reserve(groups.size() + 2);
  const std::vector<int> none;
  const IndexMap ident = make_map(gates, none, pos, pick.bits);
  const LayoutMap io = make_layout(0, tb, pick.rb);
  for (const PassGroup &g : groups)
    steps.push_back(Step{make_layout(positions(g.regs), tb, pick.rb), &g,
                         make_map(gates, g.maps, pos, pick.bits)});
  if (!steps.front().m.io()) steps.insert(steps.begin(), Step{io, nullptr, ident});
  {
    const Step &s = steps.back();
    // maps that move part of a line elsewhere go through an exchange
    bool lines = s.m.io();
    for (int p = 0; p < kPLineBits; ++p) lines = lines && (s.a.col[p] >> kPLineBits) == 0;
    if (!lines) steps.push_back(Step{io, nullptr, ident});
  }
  pp->nlayouts = uint32_t(steps.size());
  auto index_mask = [&](int e) {
    uint64_t r = 0;
    for (; e; e &= e - 1) r |= uint64_t(1) << bits[__builtin_ctz(unsigned(e))];
    return r;
  };
  const Step &first = steps.front(), &last = steps.back();
  for (int b = 0; b < first.m.nthr; ++b) pp->load_t[b] = index_mask(1 << first.m.thr[b]);
  for (int b = 0; b < pick.rb; ++b) pp->load_r[b] = index_mask(1 << first.m.reg[b]);
  for (uint64_t m : pp->load_t) pp->skip_t |= m & ~filled;
  pp->skip_t |= pick.swapped & ~filled;  // (whole tiles)
  for (uint64_t m : pp->load_r) pp->skip_r |= m & ~filled;
  pp->basis = basis;
  for (int b = 0; b < last.m.nthr; ++b) pp->store_t[b] = index_mask(last.a.col[last.m.thr[b]]);
  for (int b = 0; b < pick.rb; ++b) pp->store_r[b] = index_mask(last.a.col[last.m.reg[b]]);
  pp->store_nterm = uint32_t(last.a.nterm);
  for (int k = 0; k < last.a.nterm; ++k) {
    pp->store_q[k] = last.a.termq[k];
    pp->store_term[k] = index_mask(last.a.termv[k]);
  }
  uint64_t seen = 0;
  for (uint64_t m : pp->store_t) seen |= m;
  for (uint64_t m : pp->store_term) seen |= m;
  pp->store_add = 1;
  for (uint64_t m : pp->store_r) {
    if (seen & m) pp->store_add = 0;
    seen |= m;
  }
  uint32_t *w = pp->words;
  for (size_t x = 0; x < steps.size(); ++x) {
    const Step &s = steps[x], &next = steps[x + 1 < steps.size() ? x + 1 : x];
    PassLayout l;
    std::memset(&l, 0, sizeof(l));
    auto pair = [&](int from, int to) {
      return uint32_t(8 * pass_slot(1 << to)) | uint32_t(8 * pass_slot(s.a.col[from])) << 16;
    };
    for (int b = 0; b < s.m.nthr; ++b) l.thr[b] = pair(s.m.thr[b], next.m.thr[b]);
    for (int b = 0; b < pick.rb; ++b) l.reg[b] = pair(s.m.reg[b], next.m.reg[b]);
    // (the last layout's map is the store's)
    l.nterm = x + 1 < steps.size() ? uint32_t(s.a.nterm) : 0;
    uint32_t *rec = w;
    w += kPLayoutWords;
    if (s.g) write_ops<T>(gates, s.g->ops, s.m, pos, pick.bits, w);
    l.opwords = uint32_t(w - rec - kPLayoutWords);
    for (uint32_t k = 0; k < l.nterm; ++k)
      *w++ = uint32_t(s.a.termq[k]) | uint32_t(8 * pass_slot(s.a.termv[k])) << 16;
    std::memcpy(rec, &l, sizeof(l));
  }
}

}  // namespace qcs
