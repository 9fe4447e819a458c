// Gate-pass plans run on the CPU.
//
// Random gate lists are planned pass by pass (gateplan.h), each pass's
// program is interpreted the way k_gate_pass runs it -- threads, register
// amplitudes, LDS slots, conditions, index maps -- and the state is compared,
// value for value, with the same gates applied one after another by the
// per-gate arithmetic.  Every LDS slot and every amplitude index is checked
// for range, and every exchange and every pass for being a permutation.
#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "../../qcs_amd/csrc/gateplan.h"

using namespace qcs;

static uint64_t rng_state;
static uint64_t rnd() {
  uint64_t z = (rng_state += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
static double uni() { return double(rnd() >> 11) / 9007199254740992.0; }

static long swaps_set_aside;

static void fail(const char *what) {
  std::printf("FAIL: %s\n", what);
  std::exit(1);
}

struct Gate {
  int kind, t, c;
  double m[8];
};

template <typename T>
struct Vec {
  std::vector<T> r, i;
};

template <typename T>
static void cmul(T ar, T ai, T br, T bi, T &rr, T &ri) {
  const T a = ar * br, b = ai * bi, c = ar * bi, d = ai * br;
  rr = a - b;
  ri = c + d;
}

template <typename T>
static void apply(Vec<T> &v, int n, const Gate &g) {
  const uint64_t N = uint64_t(1) << n, tb = uint64_t(1) << g.t;
  T m[8];
  for (int k = 0; k < 8; ++k) m[k] = T(g.m[k]);
  for (uint64_t i0 = 0; i0 < N; ++i0) {
    if (g.kind == QCS_HIP_G_SWAP) {
      const uint64_t cb = uint64_t(1) << g.c;
      if ((i0 & tb) && !(i0 & cb)) {
        std::swap(v.r[i0], v.r[(i0 ^ tb) | cb]);
        std::swap(v.i[i0], v.i[(i0 ^ tb) | cb]);
      }
      continue;
    }
    if (i0 & tb) continue;
    if (g.kind == QCS_HIP_G_CU && !((i0 >> g.c) & 1)) continue;
    const uint64_t i1 = i0 | tb;
    T a, b, c, d, e, f, p, q;
    cmul(m[0], m[1], v.r[i0], v.i[i0], a, b);
    cmul(m[2], m[3], v.r[i1], v.i[i1], c, d);
    cmul(m[4], m[5], v.r[i0], v.i[i0], e, f);
    cmul(m[6], m[7], v.r[i1], v.i[i1], p, q);
    v.r[i0] = a + c;
    v.i[i0] = b + d;
    v.r[i1] = e + p;
    v.i[i1] = f + q;
  }
}

template <typename V>
static V xor_bits(uint32_t x, const V *e, int n) {
  V r = 0;
  for (int b = 0; b < n; ++b)
    if ((x >> b) & 1) r ^= e[b];
  return r;
}

template <typename T>
static T par(const uint32_t *w, int i) {
  T x;
  std::memcpy(&x, reinterpret_cast<const char *>(w) + size_t(i) * sizeof(T), sizeof(T));
  return x;
}

template <typename T>
static void op1(int cls, T *vr, T *vi, int amps, int q, const uint32_t *w, bool on) {
  for (int j = 0; j < amps; ++j) {
    if ((j >> q) & 1) continue;
    const int k = j | (1 << q);
    T x0 = vr[j], y0 = vi[j], x1 = vr[k], y1 = vi[k];
    T p[8];
    for (int z = 0; z < 8; ++z) p[z] = z < (cls == kPDense ? 8 : cls == kPEuler ? 6 : cls == kPPhase ? 2 : 4) ? par<T>(w, z) : T(0);
    switch (cls) {
      case kPDense: {
        T a, b, c, d;
        cmul(p[0], p[1], x0, y0, a, b);
        cmul(p[2], p[3], x1, y1, c, d);
        vr[j] = a + c;
        vi[j] = b + d;
        cmul(p[4], p[5], x0, y0, a, b);
        cmul(p[6], p[7], x1, y1, c, d);
        vr[k] = a + c;
        vi[k] = b + d;
        break;
      }
      case kPReal:
        vr[j] = p[0] * x0 + p[1] * x1;
        vi[j] = p[0] * y0 + p[1] * y1;
        vr[k] = p[2] * x0 + p[3] * x1;
        vi[k] = p[2] * y0 + p[3] * y1;
        break;
      case kPAnti:
        cmul(p[0], p[1], x1, y1, vr[j], vi[j]);
        cmul(p[2], p[3], x0, y0, vr[k], vi[k]);
        break;
      case kPDiag:
        cmul(p[0], p[1], x0, y0, vr[j], vi[j]);
        cmul(p[2], p[3], x1, y1, vr[k], vi[k]);
        break;
      case kPPhase:
        cmul(on ? p[0] : T(1), on ? p[1] : T(0), x1, y1, vr[k], vi[k]);
        break;
      case kPEuler: {
        cmul(p[0], p[1], x0, y0, x0, y0);
        cmul(p[0], -p[1], x1, y1, x1, y1);
        const T u0 = p[2] * x0 + p[3] * x1, v0 = p[2] * y0 + p[3] * y1;
        const T u1 = -p[3] * x0 + p[2] * x1, v1 = -p[3] * y0 + p[2] * y1;
        cmul(p[4], p[5], u0, v0, vr[j], vi[j]);
        cmul(p[4], -p[5], u1, v1, vr[k], vi[k]);
        break;
      }
      default: fail("unknown op");
    }
  }
}

// One pass over the state, as k_gate_pass runs it.
template <typename T>
static void run_pass(Vec<T> &v, int n, const PassProgram &pp, uint64_t filled) {
  const int tb = int(pp.tb), kPRegBits = int(pp.rb), kPAmps = 1 << kPRegBits;
  const int nthr = 1 << (tb - kPRegBits);
  if (tb - kPRegBits > kPThrBits) fail("thread bits");
  const uint64_t N = uint64_t(1) << n;
  // the work-groups' tiles: with SWAPs outside the tile, pairs that change
  // places and tiles that stay
  std::vector<uint64_t> tiles;
  const uint64_t work_groups = pass_work_groups(&pp, __builtin_popcountll(pp.outer));
  for (uint64_t g = 0; g < work_groups; ++g) {
    const uint64_t first = pass_tile(&pp, g), other = pass_home(&pp, first);
    if (pass_home(&pp, other) != first) fail("a pair of tiles");
    tiles.push_back(first);
    if (other != first) tiles.push_back(other);
  }
  std::vector<char> touched(N, 0), stored(N, 0);
  Vec<T> out = v;
  for (const uint64_t base : tiles) {
    std::vector<T> vr(size_t(nthr) * kPAmps), vi(vr.size());
    for (int t = 0; t < nthr; ++t)
      for (int j = 0; j < kPAmps; ++j) {
        const uint64_t i = base | xor_bits<uint64_t>(uint32_t(t), pp.load_t, kPThrBits) |
                           xor_bits<uint64_t>(uint32_t(j), pp.load_r, kPRegBits);
        if (i >= N || touched[i]) fail("load index");
        touched[i] = 1;
        const bool skip = ((i ^ pp.basis) & (pp.skip_t | pp.skip_r)) != 0;
        vr[size_t(t) * kPAmps + j] = skip ? T(0) : v.r[i];
        vi[size_t(t) * kPAmps + j] = skip ? T(0) : v.i[i];
      }
    // whole lines: threads 0..7 on 8 consecutive amplitudes
    for (int t = 0; t < 8; ++t)
      if (xor_bits<uint64_t>(uint32_t(t), pp.load_t, kPThrBits) != uint64_t(t)) fail("load line");
    const uint32_t *w = pp.words;
    for (uint32_t l = 0;;) {
      PassLayout lay;
      std::memcpy(&lay, w, sizeof(lay));
      w += kPLayoutWords;
      const uint32_t *end = w + lay.opwords;
      while (w < end) {
        const uint32_t h = w[0];
        const uint32_t *pw = w + 1;
        w += (h >> 5) & 31;
        const int kind = int(h & 31);
        if (((h >> 5) & 31) == 0 || w > end) fail("op length");
        for (int t = 0; t < nthr; ++t) {
          T *r = &vr[size_t(t) * kPAmps], *s = &vi[size_t(t) * kPAmps];
          const uint64_t uni = pass_uniform(base, unsigned(t >> kPLaneBits));
          bool on = true;
          for (int c : {int(h >> 10) & 63, int(h >> 16) & 63}) {
            const bool wave = c >= kPWaveBit && c - kPWaveBit < tb - kPRegBits - kPLaneBits;
            if (c != kPAlways && c >= n && !wave) fail("condition");
            on = on && ((uni >> c) & 1);
          }
          for (int c : {int(h >> 22) & 7, int(h >> 25) & 7}) {
            if (c == kPNoLane) continue;
            if (c >= kPLaneBits || c >= tb - kPRegBits) fail("condition");
            on = on && ((t >> c) & 1);
          }
          if (kind < kPCPhase) {
            if ((1 << (kind & 3)) >= kPAmps) fail("register bit");
            op1<T>(kind & ~3, r, s, kPAmps, kind & 3, pw, on);
            continue;
          }
          static const int sets[6] = {3, 5, 9, 6, 10, 12};
          const int set = kind < kPScale ? sets[kind - kPCPhase] : 0;
          if (set >= kPAmps) fail("register bits");
          T ar = par<T>(pw, 0), ai = par<T>(pw, 1);
          if (kind == kPScale && !on) ar = T(1), ai = T(0);
          if (kind == kPSelect && on) ar = par<T>(pw, 2), ai = par<T>(pw, 3);
          if (kind > kPSelect) fail("unknown kind");
          for (int j = 0; j < kPAmps; ++j)
            if ((j & set) == set) cmul(ar, ai, r[j], s[j], r[j], s[j]);
        }
      }
      const uint32_t *terms = w;
      w += lay.nterm;
      if (++l == pp.nlayouts) break;
      std::vector<T> lr(size_t(1) << tb), li(lr.size());
      std::vector<char> full(lr.size(), 0);
      for (int t = 0; t < nthr; ++t) {
        uint32_t ws = xor_bits<uint32_t>(uint32_t(t), lay.thr, kPThrBits) >> 16;
        for (uint32_t k = 0; k < lay.nterm; ++k)
          if ((base >> (terms[k] & 63)) & 1) ws ^= terms[k] >> 16;
        for (int j = 0; j < kPAmps; ++j) {
          uint32_t x = ws ^ (xor_bits<uint32_t>(uint32_t(j), lay.reg, kPRegBits) >> 16);
          if (x & 7) fail("write offset");
          x /= 8;
          if (x >= full.size() || full[x]) fail("write slot");
          full[x] = 1;
          lr[x] = vr[size_t(t) * kPAmps + j];
          li[x] = vi[size_t(t) * kPAmps + j];
        }
      }
      for (int t = 0; t < nthr; ++t) {
        const uint32_t rs = xor_bits<uint32_t>(uint32_t(t), lay.thr, kPThrBits) & 0xffffu;
        for (int j = 0; j < kPAmps; ++j) {
          uint32_t x = rs ^ (xor_bits<uint32_t>(uint32_t(j), lay.reg, kPRegBits) & 0xffffu);
          if (x & 7) fail("read offset");
          x /= 8;
          if (x >= full.size() || full[x] != 1) fail("read slot");
          full[x] = 2;
          vr[size_t(t) * kPAmps + j] = lr[x];
          vi[size_t(t) * kPAmps + j] = li[x];
        }
      }
    }
    if (w - pp.words > kPWords) fail("program length");
    uint64_t b2 = base, used = 0;
    for (uint32_t k = 0; k < pp.nswaps; ++k) {
      // distinct bits outside the tile: the tiles change places in pairs
      const uint32_t lo = pp.swaps[k] & 255, hi = pp.swaps[k] >> 8;
      const uint64_t both = uint64_t(1) << lo | uint64_t(1) << hi;
      if (lo == hi || (both & used) || (both & pp.outer) || (base >> lo ^ b2 >> lo) & 1)
        fail("swapped bits");
      used |= both;
      const uint64_t d = (b2 >> lo ^ b2 >> hi) & 1;
      b2 ^= d << lo | d << hi;
    }
    for (uint32_t k = 0; k < pp.store_nterm; ++k)
      if ((base >> pp.store_q[k]) & 1) b2 ^= pp.store_term[k];
    for (int t = 0; t < nthr; ++t)
      for (int j = 0; j < kPAmps; ++j) {
        const uint64_t i0 = b2 ^ xor_bits<uint64_t>(uint32_t(t), pp.store_t, kPThrBits);
        const uint64_t i = i0 ^ xor_bits<uint64_t>(uint32_t(j), pp.store_r, kPRegBits);
        if (pp.store_add && i != i0 + xor_bits<uint64_t>(uint32_t(j), pp.store_r, kPRegBits))
          fail("store sum");
        if (i >= N || stored[i]) fail("store index");
        stored[i] = 1;
        out.r[i] = vr[size_t(t) * kPAmps + j];
        out.i[i] = vi[size_t(t) * kPAmps + j];
      }
  }
  for (uint64_t i = 0; i < N; ++i)
    if (touched[i] != stored[i] || (!touched[i] && ((i ^ pp.basis) & ~filled) == 0 &&
                                    (v.r[i] != T(0) || v.i[i] != T(0))))
      fail("an amplitude was left out");
  v = out;
}

template <typename T>
static int check(int n, int tb, int low, int count, int style, bool basis_state, bool unfilled, bool pairs, int rb) {
  const uint64_t N = uint64_t(1) << n;
  std::vector<Gate> gates;
  std::vector<PlanGate> q;
  for (int x = 0; x < count; ++x) {
    Gate g;
    std::memset(&g, 0, sizeof(g));
    g.t = int(rnd() % uint64_t(n));
    g.c = int(rnd() % uint64_t(n - 1));
    if (g.c >= g.t) ++g.c;
    const double a = 6.283185307179586 * uni(), c = std::cos(a / 2), s = std::sin(a / 2);
    // style 0: every kind; 1: rotations and CNOTs; 2: H and controlled phases;
    // 3: mostly SWAPs
    int k = int(rnd() % 13);
    if (style == 1) k = k < 8 ? 6 + k % 2 : 9;
    if (style == 2) k = k < 3 ? 0 : k < 11 ? 10 : 11;
    if (style == 3) k = k < 2 ? 0 : k < 4 ? 9 : k < 6 ? 10 : 11;
    if (style == 1 && k == 7 && x + 3 <= count) {  // RZ RY RZ
      for (int y = 0; y < 3; ++y) {
        Gate z;
        std::memset(&z, 0, sizeof(z));
        const double b = 6.283185307179586 * uni(), cb = std::cos(b / 2), sb = std::sin(b / 2);
        z.kind = QCS_HIP_G_1Q;
        z.t = g.t;
        const double rz[8] = {cb, -sb, 0, 0, 0, 0, cb, sb}, ry[8] = {cb, 0, -sb, 0, sb, 0, cb, 0};
        std::memcpy(z.m, y == 1 ? ry : rz, sizeof(z.m));
        gates.push_back(z);
      }
      x += 2;
      continue;
    }
    const double r = 1.0 / std::sqrt(2.0);
    const double mats[9][8] = {{r, 0, r, 0, r, 0, -r, 0}, {0, 0, 1, 0, 1, 0, 0, 0},
                               {0, 0, 0, -1, 0, 1, 0, 0}, {1, 0, 0, 0, 0, 0, -1, 0},
                               {1, 0, 0, 0, 0, 0, c, s},  {c, 0, 0, -s, 0, -s, c, 0},
                               {c, 0, -s, 0, s, 0, c, 0}, {c, -s, 0, 0, 0, 0, c, s},
                               {c, s, 0, 0, 0, 0, s, -c}};
    g.kind = QCS_HIP_G_1Q;
    if (k < 9) {
      std::memcpy(g.m, mats[k], sizeof(g.m));
    } else if (k == 11) {
      g.kind = QCS_HIP_G_SWAP;
    } else {
      g.kind = QCS_HIP_G_CU;
      std::memcpy(g.m, k == 9 ? mats[1] : k == 10 ? mats[4] : mats[3], sizeof(g.m));
    }
    if (g.kind == QCS_HIP_G_1Q && k == 5 && rnd() % 2) {  // a dense matrix
      for (double &z : g.m) z = 0.5 * (uni() - 0.5);
    }
    gates.push_back(g);
  }
  Vec<T> a;
  a.r.resize(N);
  a.i.resize(N);
  for (uint64_t i = 0; i < N; ++i) {
    a.r[i] = T(uni() - 0.5);
    a.i[i] = T(uni() - 0.5);
  }
  // a basis state (`unfilled`: only its one amplitude in memory), or any state
  const uint64_t basis = rnd() & (N - 1);
  uint64_t support = basis_state ? 0 : ~uint64_t(0);
  for (uint64_t i = 0; basis_state && i < N; ++i) {
    a.r[i] = T(i == basis ? 1 : 0);
    a.i[i] = T(0);
  }
  Vec<T> b = a;
  for (const Gate &g : gates) apply(a, n, g);
  for (const Gate &g : gates) q.push_back(plan_gate(g.kind, g.t, g.c, g.m));
  uint64_t filled = unfilled ? 0 : ~uint64_t(0);
  for (uint64_t i = 0; unfilled && i < N; ++i)
    if (i != basis) b.r[i] = b.i[i] = T(NAN);
  int passes = 0;
  PassPick pick;
  std::vector<PassGroup> groups;
  static PassProgram pp;
  while (!q.empty()) {
    plan_pick(q, n, tb, low, int(sizeof(T) / 4), 64, &pick, &groups, pairs, rb);
    if (!pairs && !pick.swaps.empty()) fail("swaps");
    std::vector<int> taken = pick.gates;
    taken.insert(taken.end(), pick.swaps.begin(), pick.swaps.end());
    std::sort(taken.begin(), taken.end());
    if (taken.empty()) fail("a pass without gates");
    if (__builtin_popcountll(pick.bits) != tb) fail("tile bits");
    write_pass<T>(q, pick, groups, n, tb, support, basis, &pp, filled);
    run_pass<T>(b, n, pp, filled);
    filled |= pick.bits | pick.swapped;
    swaps_set_aside += long(pick.swaps.size());
    for (int i : taken) support |= plan_spread(q[size_t(i)]);
    std::vector<PlanGate> rest;
    size_t x = 0;
    for (size_t i = 0; i < q.size(); ++i) {
      if (x < taken.size() && size_t(taken[x]) == i) ++x;
      else rest.push_back(q[i]);
    }
    q.swap(rest);
    ++passes;
  }
  for (uint64_t i = 0; i < N; ++i)
    if ((i ^ basis) & ~filled) {
      if (unfilled && !(b.r[i] != b.r[i])) fail("an amplitude outside the filled ones was written");
      b.r[i] = b.i[i] = T(0);
    }
  for (uint64_t i = 0; i < N; ++i)
    if (!(a.r[i] == b.r[i] && a.i[i] == b.i[i])) fail("amplitudes differ");
  return passes;
}

int main() {
  rng_state = 12345;
  long total = 0;
  for (int n = 7; n <= 13; ++n)
    for (int style = 0; style < 4; ++style)
      for (int rep = 0; rep < 6; ++rep) {
        // the whole state in a tile, then tiles smaller than it
        for (int tb = n < kPMaxTile ? n : kPMaxTile; tb >= 7 && tb >= n - 5; tb -= 2)
          for (int low = 3; low <= 4; ++low) {
            if (tb < n && tb < low + 4) continue;
            const int count = 20 + int(rnd() % 200);
            for (int rb = 4; rb >= (low == 4 ? 2 : 4) && tb - rb <= kPThrBits; --rb) {
              total += check<double>(n, tb, low, count, style, rep % 3 > 0, rep % 3 > 1, rep > 2, rb);
              total += check<float>(n, tb, low, count, style, rep % 3 > 0, rep % 3 > 1, rep > 2, rb);
            }
          }
      }
  if (swaps_set_aside < 100) fail("no pass moved its tiles");
  std::printf("ok %ld passes\n", total);
  return 0;
}
