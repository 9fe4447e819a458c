// Gate passes: many plain gates in one sweep over HBM.
//
// A gate by itself reads and writes the state once (gates.hip: bound by HBM,
// 5.8 TB/s in place).  A pass reads it once, runs the gates of gateplan.h's
// program on it and writes it once, so the cost of a gate becomes its
// arithmetic: a pass of the 28-qubit layered circuit (694 gates in 22 passes)
// takes 1.5-2.4 ms, where each gate by itself took 1.2 ms.  The passes are
// bound by FP64 multiplies and adds (VALU 88-93 % busy at the 1.9 GHz the card
// holds under them; 288 of about 330 instructions per RZ RY RZ), HBM below it
// at 3.6-5.6 TB/s.  The circuit went from 863 to 36 ms, the 28-qubit QFT of any
// state (476 gates with its preparation) from 269 to 14 ms.
//
// k_gate_pass.  One work-group per tile of 2^tb amplitudes; thread t holds 16
// (small states: 4) of them in registers, those that differ in the layout's
// register bits.  A layout change exchanges the tile through LDS, complex128 as
// two planes (all real parts, then all imaginary parts), so a 12-bit tile takes
// 32 KiB: five work-groups of 256 threads fit a CU (96 registers a thread), and
// one computes while another waits for HBM.  The arithmetic is that of
// gates.hip without the products by exact-zero entries, which add only signed
// zeros; the amplitudes compare equal to the per-gate kernels' (bound_gate
// keeps states whose amplitudes could overflow out).
//
// A state that starts as a basis state is zero wherever an index bit no gate
// has mixed yet differs from the basis index; tiles of zeros are left alone
// (28 qubits, H on every qubit and three layers: 21.5 -> 18.4 ms, with cheaper
// addresses; the QFT of a basis state 15.4 -> 5.0 ms), and those that no pass
// has written yet are not read (launch_basis_start): 1.4 ms for that QFT.
//
// A SWAP of two bits outside the tile moves whole tiles: a work-group of two
// halves reads a tile and the one it changes places with and stores each in
// the other's place, so a bit reversal, which took four passes, takes one (28
// qubits: the QFT's last gates and its 14 SWAPs 6.3 -> 3.7 ms).  Every pair has
// one work-group: with one per tile and half of them leaving, the XCDs' shares
// differed by 1.5 to 2 times (5.4 ms).
#include <algorithm>
#include <cmath>
#include <exception>
#include <iterator>
#include <mutex>
#include <vector>

#include "device.h"
#include "gateplan.h"
#include "internal.h"

namespace qcs {

// ---- ops on the register group -----------------------------------------------
//
// vr[j], vi[j]: the amplitude whose register bits are the bits of j.  Every
// index is a compile-time constant.

// Every product of a pair is formed before any sum: each result is then
// defined after the last use of the inputs and takes an input's register, so
// every op leaves each amplitude in the register it came in and the joins
// after the dispatch need no copies.  pair_end keeps the scheduler from
// interleaving the pairs, which would need more registers than the four
// waves a SIMD holds leave.
__device__ __forceinline__ void pair_end() { __builtin_amdgcn_sched_barrier(0); }

template <int Q, typename T, int N>
__device__ __forceinline__ void p_dense(T (&vr)[N], T (&vi)[N], const T (&m)[8]) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (j & (1 << Q)) continue;
    const int k = j | (1 << Q);
    const T x0 = vr[j], y0 = vi[j], x1 = vr[k], y1 = vi[k];
    const T a0 = m[0] * x0, a1 = m[1] * y0, a2 = m[0] * y0, a3 = m[1] * x0;
    const T c0 = m[2] * x1, c1 = m[3] * y1, c2 = m[2] * y1, c3 = m[3] * x1;
    const T b0 = m[4] * x0, b1 = m[5] * y0, b2 = m[4] * y0, b3 = m[5] * x0;
    const T d0 = m[6] * x1, d1 = m[7] * y1, d2 = m[6] * y1, d3 = m[7] * x1;
    vr[j] = (a0 - a1) + (c0 - c1);
    vi[j] = (a2 + a3) + (c2 + c3);
    vr[k] = (b0 - b1) + (d0 - d1);
    vi[k] = (b2 + b3) + (d2 + d3);
    pair_end();
  }
}

// every imaginary part 0: {m00, m01, m10, m11}
template <int Q, typename T, int N>
__device__ __forceinline__ void p_real(T (&vr)[N], T (&vi)[N], T m00, T m01, T m10, T m11) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (j & (1 << Q)) continue;
    const int k = j | (1 << Q);
    const T x0 = vr[j], y0 = vi[j], x1 = vr[k], y1 = vi[k];
    const T a0 = m00 * x0, a1 = m00 * y0, b0 = m10 * x0, b1 = m10 * y0;
    const T c0 = m01 * x1, c1 = m01 * y1, d0 = m11 * x1, d1 = m11 * y1;
    vr[j] = a0 + c0;
    vi[j] = a1 + c1;
    vr[k] = b0 + d0;
    vi[k] = b1 + d1;
    pair_end();
  }
}

// zero diagonal: out0 = (ar, ai) v1, out1 = (br, bi) v0
template <int Q, typename T, int N>
__device__ __forceinline__ void p_anti(T (&vr)[N], T (&vi)[N], T ar, T ai, T br, T bi) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (j & (1 << Q)) continue;
    const int k = j | (1 << Q);
    const T x0 = vr[j], y0 = vi[j], x1 = vr[k], y1 = vi[k];
    const T c0 = ar * x1, c1 = ai * y1, c2 = ar * y1, c3 = ai * x1;
    const T b0 = br * x0, b1 = bi * y0, b2 = br * y0, b3 = bi * x0;
    vr[j] = c0 - c1;
    vi[j] = c2 + c3;
    vr[k] = b0 - b1;
    vi[k] = b2 + b3;
    pair_end();
  }
}

template <typename T>
__device__ __forceinline__ void p_scale(T &vr, T &vi, T ar, T ai) {
  const T a0 = ar * vr, a1 = ai * vi, a2 = ar * vi, a3 = ai * vr;
  vr = a0 - a1;
  vi = a2 + a3;
}

// the amplitudes whose register bits include those of SET, times (ar, ai)
template <int SET, typename T, int N>
__device__ __forceinline__ void p_phase(T (&vr)[N], T (&vi)[N], T ar, T ai) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if ((j & SET) == SET) {
      p_scale(vr[j], vi[j], ar, ai);
      if (j & 1) pair_end();
    } else {
      // tied to its register as if it changed: left alone, the amplitudes an
      // op does not touch were copied at the join (42 moves beside 48
      // arithmetic instructions)
      asm volatile("" : "+v"(vr[j]), "+v"(vi[j]));
    }
  }
}

template <int Q, typename T, int N>
__device__ __forceinline__ void p_diag(T (&vr)[N], T (&vi)[N], T ar, T ai, T br, T bi) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (j & (1 << Q)) continue;
    const int k = j | (1 << Q);
    p_scale(vr[j], vi[j], ar, ai);
    p_scale(vr[k], vi[k], br, bi);
    pair_end();
  }
}

// diag(ar + i ai, conj), [[c, s], [-s, c]], diag(br + i bi, conj), one after
// the other: the products of the three gates, whose other entries are copies
// and negations of these
template <int Q, typename T, int N>
__device__ __forceinline__ void p_euler(T (&vr)[N], T (&vi)[N], T ar, T ai, T c, T s, T br,
                                        T bi) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (j & (1 << Q)) continue;
    const int k = j | (1 << Q);
    p_scale(vr[j], vi[j], ar, ai);
    p_scale(vr[k], vi[k], ar, -ai);
    const T x0 = vr[j], y0 = vi[j], x1 = vr[k], y1 = vi[k];
    const T a0 = c * x0, a1 = c * y0, b0 = -s * x0, b1 = -s * y0;
    const T c0 = s * x1, c1 = s * y1, d0 = c * x1, d1 = c * y1;
    vr[j] = a0 + c0;
    vi[j] = a1 + c1;
    vr[k] = b0 + d0;
    vi[k] = b1 + d1;
    p_scale(vr[j], vi[j], br, bi);
    p_scale(vr[k], vi[k], br, -bi);
    pair_end();
  }
}

// The program is read where the launch put it, by scalar loads: as a plain
// by-value parameter indexed at run time it would be copied to scratch.
#define QCS_KERNARG __attribute__((address_space(4)))
typedef const QCS_KERNARG uint32_t *Words;
typedef const QCS_KERNARG PassLayout *LayoutPtr;
typedef const QCS_KERNARG PassProgram *ProgramPtr;

// An op's word and the 16 words behind it (its parameters, at most), in
// scalar registers.  The next op's are loaded before this one runs, so the
// two waits of a dispatch (the op word, then its parameters) are covered by
// arithmetic (28 qubits, complex64: 1.10 -> 0.87 ms a pass; 16 qubits,
// complex128: 21 -> 19 us).
typedef uint32_t Par __attribute__((ext_vector_type(16), aligned(4)));
struct Op {
  uint32_t h;
  Par p;
};
__device__ __forceinline__ Op load_op(Words w) {
  return Op{w[0], *(const QCS_KERNARG Par *)(w + 1)};
}

// parameter i of an op
template <typename T>
__device__ __forceinline__ T par(const Par &w, int i) {
  if constexpr (sizeof(T) == 8) {
    return __builtin_bit_cast(T, uint64_t(w[2 * i]) | uint64_t(w[2 * i + 1]) << 32);
  } else {
    const uint32_t x = w[i];  // (a bit cast of the element itself takes element 0)
    return __builtin_bit_cast(T, x);
  }
}

// XOR of the entries whose bit is set in x (a lane's value): two or three
// instructions a bit
template <int N>
__device__ __forceinline__ uint32_t xor_lanes(uint32_t x, const QCS_KERNARG uint32_t *e) {
  uint32_t r = 0;
#pragma unroll
  for (int b = 0; b < N; ++b) r ^= e[b] & uint32_t(__builtin_amdgcn_sbfe(int(x), b, 1));
  return r;
}
template <int N>
__device__ __forceinline__ uint64_t xor_lanes(uint32_t x, const QCS_KERNARG uint64_t *e) {
  uint32_t lo = 0, hi = 0;
#pragma unroll
  for (int b = 0; b < N; ++b) {
    const uint32_t m = uint32_t(__builtin_amdgcn_sbfe(int(x), b, 1));
    lo ^= uint32_t(e[b]) & m;
    hi ^= uint32_t(e[b] >> 32) & m;
  }
  return uint64_t(hi) << 32 | lo;
}
// the same of a compile-time index (scalar arithmetic)
template <int N, typename V>
__device__ __forceinline__ V xor_const(int x, const QCS_KERNARG V *e) {
  V r = 0;
#pragma unroll
  for (int b = 0; b < N; ++b)
    if ((x >> b) & 1) r ^= e[b];
  return r;
}

// the same value, but not for the compiler: what is computed from it is not
// kept in registers from an earlier use (here the thread-bit masks, which
// cost 17 spilled registers across the ops)
__device__ __forceinline__ uint32_t fresh(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

// a where mask is all ones, b where it is 0: by bits, since a select between
// a loaded value and another becomes a branch around the load
__device__ __forceinline__ double blend(uint32_t mask, double a, double b) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
  const uint64_t m = uint64_t(mask) << 32 | mask;
  return __builtin_bit_cast(double, (x & m) | (y & ~m));
}
__device__ __forceinline__ float blend(uint32_t mask, float a, float b) {
  const uint32_t x = __builtin_bit_cast(uint32_t, a), y = __builtin_bit_cast(uint32_t, b);
  return __builtin_bit_cast(float, (x & mask) | (y & ~mask));
}

// Conditions of an op (its word h).  The wave's: bits of a scalar, so an op
// that no amplitude of the wave meets is skipped by a scalar branch and one
// that all meet takes its factor from scalar registers.  The lane's: all ones
// in the lanes that meet them.  A controlled phase is 48 multiplies and adds;
// with every condition a lane's mask its test and its blended factor were 14
// instructions more (28-qubit QFT: passes of 113, 143 and 131 gates 4.4, 4.0,
// 3.4 -> 4.1, 3.5, 3.1 ms).
__device__ __forceinline__ bool wave_meets(uint32_t h, uint64_t uni) {
  return ((uni >> ((h >> 10) & 63)) & (uni >> ((h >> 16) & 63)) & 1) != 0;
}
__device__ __forceinline__ bool any_lane(uint32_t h) { return ((h >> 22) & 63) == 63; }
__device__ __forceinline__ uint32_t lanes_meet(uint32_t h, int tid) {
  const int t = int(fresh(uint32_t(tid))) | 1 << kPNoLane;
  return uint32_t(__builtin_amdgcn_sbfe(t, (h >> 22) & 7, 1)) &
         uint32_t(__builtin_amdgcn_sbfe(t, (h >> 25) & 7, 1));
}

// A scalar parameter of one op only: without it the products that several ops
// share are formed before the dispatch, 22 registers of them spilled.
template <typename T>
__device__ __forceinline__ T own(T x) {
  asm volatile("" : "+s"(x));
  return x;
}

// m11 on the amplitudes of SET in the lanes that meet the conditions: in the
// others the factor is 1 (x * 1 - y * 0 is x)
template <int SET, typename T, int N>
__device__ __forceinline__ void p_phase_if(uint32_t h, int tid, T (&vr)[N], T (&vi)[N], T ar,
                                           T ai) {
  if (any_lane(h)) {
    p_phase<SET, T>(vr, vi, own(ar), own(ai));
  } else {
    const uint32_t on = lanes_meet(h, tid);
    p_phase<SET, T>(vr, vi, blend(on, ar, T(1)), blend(on, ai, T(0)));
  }
}

// one-qubit gates on register bit Q
template <int Q, typename T, int N>
__device__ __forceinline__ void p_op(int cls, T (&vr)[N], T (&vi)[N], const Par &w) {
  switch (cls) {
    case kPDense: {
      const T m[8] = {par<T>(w, 0), par<T>(w, 1), par<T>(w, 2), par<T>(w, 3),
                      par<T>(w, 4), par<T>(w, 5), par<T>(w, 6), par<T>(w, 7)};
      p_dense<Q, T>(vr, vi, m);
      break;
    }
    case kPReal:
      p_real<Q, T>(vr, vi, par<T>(w, 0), par<T>(w, 1), par<T>(w, 2), par<T>(w, 3));
      break;
    case kPAnti:
      p_anti<Q, T>(vr, vi, par<T>(w, 0), par<T>(w, 1), par<T>(w, 2), par<T>(w, 3));
      break;
    case kPDiag:
      p_diag<Q, T>(vr, vi, own(par<T>(w, 0)), own(par<T>(w, 1)), own(par<T>(w, 2)),
                   own(par<T>(w, 3)));
      break;
    default:  // kPEuler
      p_euler<Q, T>(vr, vi, par<T>(w, 0), par<T>(w, 1), par<T>(w, 2), par<T>(w, 3), par<T>(w, 4),
                    par<T>(w, 5));
      break;
  }
}

// The op under way and the next one.
struct Feed {
  Words w, end;  // w: the next op
  Op cur, next;
  __device__ __forceinline__ void start(Words first, Words last) {
    w = first;
    end = last;
    next = load_op(w);
  }
  __device__ __forceinline__ bool more() const { return w < end; }
  __device__ __forceinline__ void advance() {
    cur = next;
    w += (cur.h >> 5) & 31;
    next = load_op(w);
  }
};

// Brings the program's lines into the scalar cache while the tile's own loads
// are under way, all of them before one wait: a launch finds none there, and
// read as the program gets to them each is a trip to L2 in a chain that a small
// grid does not hide (8 and 10 qubits 89 -> 81 and 116 -> 105 us, 17 qubits 255 ->
// 244).  With 4 amplitudes a thread a grid has 512 work-groups at most (19
// qubits); the ops of 16 amplitudes a thread are long enough to hide the trips
// (12 qubits 162 -> 169, a 20-qubit circuit with its histogram 630 -> 657).
__device__ __forceinline__ void warm_program(Words w) {
  static_assert(52 * 64 + 4 <= kPWords * 4, "inside the program");
  uint32_t x;
  asm volatile(
      "s_load_dword %0, %1, 0x0\ns_load_dword %0, %1, 0x40\n"
      "s_load_dword %0, %1, 0x80\ns_load_dword %0, %1, 0xc0\n"
      "s_load_dword %0, %1, 0x100\ns_load_dword %0, %1, 0x140\n"
      "s_load_dword %0, %1, 0x180\ns_load_dword %0, %1, 0x1c0\n"
      "s_load_dword %0, %1, 0x200\ns_load_dword %0, %1, 0x240\n"
      "s_load_dword %0, %1, 0x280\ns_load_dword %0, %1, 0x2c0\n"
      "s_load_dword %0, %1, 0x300\ns_load_dword %0, %1, 0x340\n"
      "s_load_dword %0, %1, 0x380\ns_load_dword %0, %1, 0x3c0\n"
      "s_load_dword %0, %1, 0x400\ns_load_dword %0, %1, 0x440\n"
      "s_load_dword %0, %1, 0x480\ns_load_dword %0, %1, 0x4c0\n"
      "s_load_dword %0, %1, 0x500\ns_load_dword %0, %1, 0x540\n"
      "s_load_dword %0, %1, 0x580\ns_load_dword %0, %1, 0x5c0\n"
      "s_load_dword %0, %1, 0x600\ns_load_dword %0, %1, 0x640\n"
      "s_load_dword %0, %1, 0x680\ns_load_dword %0, %1, 0x6c0\n"
      "s_load_dword %0, %1, 0x700\ns_load_dword %0, %1, 0x740\n"
      "s_load_dword %0, %1, 0x780\ns_load_dword %0, %1, 0x7c0\n"
      "s_load_dword %0, %1, 0x800\ns_load_dword %0, %1, 0x840\n"
      "s_load_dword %0, %1, 0x880\ns_load_dword %0, %1, 0x8c0\n"
      "s_load_dword %0, %1, 0x900\ns_load_dword %0, %1, 0x940\n"
      "s_load_dword %0, %1, 0x980\ns_load_dword %0, %1, 0x9c0\n"
      "s_load_dword %0, %1, 0xa00\ns_load_dword %0, %1, 0xa40\n"
      "s_load_dword %0, %1, 0xa80\ns_load_dword %0, %1, 0xac0\n"
      "s_load_dword %0, %1, 0xb00\ns_load_dword %0, %1, 0xb40\n"
      "s_load_dword %0, %1, 0xb80\ns_load_dword %0, %1, 0xbc0\n"
      "s_load_dword %0, %1, 0xc00\ns_load_dword %0, %1, 0xc40\n"
      "s_load_dword %0, %1, 0xc80\ns_load_dword %0, %1, 0xcc0\n"
      "s_load_dword %0, %1, 0xd00\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&s"(x)
      : "s"(w));
  asm volatile("" ::"s"(x));
}

template <typename T, int RB>
__global__ __launch_bounds__(1 << kPThrBits, 5) void k_gate_pass(
    const PassProgram by_value, typename Amp<T>::type *a) {
  typedef typename Amp<T>::type A;
  constexpr int N = 1 << RB;
  constexpr int TH = RB < kPRegBits ? kPThrBits : kPMaxTile - RB;  // thread bits
  // the first argument starts the kernel-argument segment
  const ProgramPtr prog = (ProgramPtr)__builtin_amdgcn_kernarg_segment_ptr();
  const int tb = int(prog->tb);
  // With SWAPs of bits outside the tile a work-group takes a tile in its lower
  // half and the one it changes places with in its upper: both are read before
  // either is stored, in the other's place.  (A tile that stays where it is is
  // taken by both halves, which store the same.)
  const int half = prog->nswaps == 0
                       ? 0
                       : __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> (tb - RB));
  const int tid = int(threadIdx.x) - (half << (tb - RB));
  // a tile of fewer than 64 threads (7 qubits, 4 amplitudes a thread) still
  // takes a whole wave, whose lanes past the tile compute on copies and store
  // nothing
  const bool in = tid < (1 << (tb - RB));
  // amplitude index of the tile, and of the place it is stored in
  uint64_t base = pass_tile(prog, xcd_order(blockIdx.x, gridDim.x)), home = base;
  if (prog->nswaps != 0) {
    const uint64_t other = pass_home(prog, base);
    (half != 0 ? base : home) = other;
  }
  T vr[N], vi[N];
  {
    // one thread address, plus a scalar offset per register (the masks of a
    // load share no bit); lanes past the tile read its first amplitudes,
    // their masks being zero
    const uint64_t i0 = base | xor_lanes<TH>(uint32_t(tid), prog->load_t);
    const char *p = reinterpret_cast<const char *>(a + i0);
    A v[N];
    if ((prog->skip_t | prog->skip_r) == 0) {
#pragma unroll
      for (int j = 0; j < N; ++j)
        v[j] = ld_stream(reinterpret_cast<const A *>(
            p + xor_const<RB>(j, prog->load_r) * sizeof(A)));
    } else {
      const bool lane = ((i0 ^ prog->basis) & prog->skip_t) == 0;
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const uint64_t off = xor_const<RB>(j, prog->load_r);
        v[j].x = v[j].y = T(0);
        if (((off ^ prog->basis) & prog->skip_r) == 0 && lane)
          v[j] = ld_stream(reinterpret_cast<const A *>(p + off * sizeof(A)));
      }
    }
    if constexpr (RB < kPRegBits) warm_program(prog->words);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      vr[j] = v[j].x;
      vi[j] = v[j].y;
    }
  }
  const uint64_t uni = pass_uniform(
      base, unsigned(__builtin_amdgcn_readfirstlane(tid >> kPLaneBits)));
  Words w = prog->words;
  for (int l = 0;;) {
    const LayoutPtr lay = (LayoutPtr)w;
    w += kPLayoutWords;
    Feed f;
    f.start(w, w + lay->opwords);
    while (f.more()) {
      f.advance();
      const int kind = int(f.cur.h & 31);
      const Par pw = f.cur.p;
      if ((kind & ~3) == kPPhase) {
        if (!wave_meets(f.cur.h, uni)) continue;
        const T ar = par<T>(pw, 0), ai = par<T>(pw, 1);
        switch (kind & (RB == 4 ? 3 : 1)) {
          case 0: p_phase_if<1, T>(f.cur.h, tid, vr, vi, ar, ai); break;
          case 1: p_phase_if<2, T>(f.cur.h, tid, vr, vi, ar, ai); break;
          case 2: p_phase_if<4, T>(f.cur.h, tid, vr, vi, ar, ai); break;
          default: p_phase_if<8, T>(f.cur.h, tid, vr, vi, ar, ai); break;
        }
        continue;
      }
      if (kind < kPCPhase) {
        switch (kind & (RB == 4 ? 3 : 1)) {
          case 0: p_op<0, T>(kind & ~3, vr, vi, pw); break;
          case 1: p_op<1, T>(kind & ~3, vr, vi, pw); break;
          case 2:
            if constexpr (RB > 2) p_op<2, T>(kind & ~3, vr, vi, pw);
            break;
          default:
            if constexpr (RB > 2) p_op<3, T>(kind & ~3, vr, vi, pw);
        }
        continue;
      }
      const T ar = par<T>(pw, 0), ai = par<T>(pw, 1);
      switch (kind) {
        case kPCPhase + 0: p_phase<3, T>(vr, vi, own(ar), own(ai)); break;
        case kPCPhase + 1: p_phase<5, T>(vr, vi, own(ar), own(ai)); break;
        case kPCPhase + 2: p_phase<9, T>(vr, vi, own(ar), own(ai)); break;
        case kPCPhase + 3: p_phase<6, T>(vr, vi, own(ar), own(ai)); break;
        case kPCPhase + 4: p_phase<10, T>(vr, vi, own(ar), own(ai)); break;
        case kPCPhase + 5: p_phase<12, T>(vr, vi, own(ar), own(ai)); break;
        case kPSelect: {
          const uint32_t on = wave_meets(f.cur.h, uni) ? lanes_meet(f.cur.h, tid) : 0u;
          p_phase<0, T>(vr, vi, blend(on, par<T>(pw, 2), ar), blend(on, par<T>(pw, 3), ai));
          break;
        }
        default:  // kPScale
          if (wave_meets(f.cur.h, uni)) p_phase_if<0, T>(f.cur.h, tid, vr, vi, ar, ai);
      }
    }
    const Words terms = f.end;
    w = terms + lay->nterm;
    if (++l == int(prog->nlayouts)) break;
    // exchange: written in this layout, through its index map, and read in
    // the next one
    const uint32_t both = xor_lanes<TH>(fresh(uint32_t(tid)), lay->thr);
    const uint32_t lds0 = uint32_t(half) << (tb + 3);
    uint32_t ws = both >> 16 | lds0;
    uint32_t rs = (both & 0xffffu) | lds0;
    for (uint32_t k = 0; k < lay->nterm; ++k) {
      const uint32_t t = terms[k];
      if ((base >> (t & 63)) & 1) ws ^= t >> 16;
    }
    // byte offsets from the start of LDS, which is all dynamic here
    typedef __attribute__((address_space(3))) double *LdsDouble;
    typedef __attribute__((address_space(3))) f2v *LdsFloat2;
    typedef __attribute__((address_space(3))) d2v *LdsDouble2;
    auto wslot = [&](int j) { return ws ^ (xor_const<RB>(j, lay->reg) >> 16); };
    auto rslot = [&](int j) { return rs ^ (xor_const<RB>(j, lay->reg) & 0xffffu); };
    __syncthreads();  // the reads of the exchange before
    if constexpr (sizeof(T) == 8 && RB < kPRegBits) {
      // a small tile fits LDS with both parts side by side
      if (in) {
#pragma unroll
        for (int j = 0; j < N; ++j) *(LdsDouble2)uintptr_t(2 * wslot(j)) = d2v{vr[j], vi[j]};
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const d2v x = *(LdsDouble2)uintptr_t(2 * rslot(j));
        vr[j] = x.x;
        vi[j] = x.y;
      }
    } else if constexpr (sizeof(T) == 8) {
      if (in) {
#pragma unroll
        for (int j = 0; j < N; ++j) *(LdsDouble)uintptr_t(wslot(j)) = vr[j];
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < N; ++j)
        vr[j] = *(LdsDouble)uintptr_t(rslot(j));
      __syncthreads();
      if (in) {
#pragma unroll
        for (int j = 0; j < N; ++j) *(LdsDouble)uintptr_t(wslot(j)) = vi[j];
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < N; ++j)
        vi[j] = *(LdsDouble)uintptr_t(rslot(j));
    } else {
      if (in) {
#pragma unroll
        for (int j = 0; j < N; ++j) *(LdsFloat2)uintptr_t(wslot(j)) = f2v{vr[j], vi[j]};
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const f2v x = *(LdsFloat2)uintptr_t(rslot(j));
        vr[j] = x.x;
        vi[j] = x.y;
      }
    }
  }
  if (prog->nlayouts == 1) {
    // no exchange has held the waves together, and the store's index map may
    // hit amplitudes that another wave loads: every load first
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
  if (!in) return;
  uint64_t i0 = home ^ xor_lanes<TH>(fresh(uint32_t(tid)), prog->store_t);
  for (uint32_t k = 0; k < prog->store_nterm; ++k)
    if ((base >> prog->store_q[k]) & 1) i0 ^= prog->store_term[k];
  auto amp = [&](int j) {
    A o;
    o.x = vr[j];
    o.y = vi[j];
    return o;
  };
  if (prog->store_add) {
    char *p = reinterpret_cast<char *>(a + i0);
#pragma unroll
    for (int j = 0; j < N; ++j)
      st_stream(reinterpret_cast<A *>(p + xor_const<RB>(j, prog->store_r) * sizeof(A)),
                amp(j));
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j)
      st_stream(a + (i0 ^ xor_const<RB>(j, prog->store_r)), amp(j));
  }
}

// ---- the queue of plain gates --------------------------------------------------

// Tile of a pass over an n-qubit state, and register bits of its layouts.
//
// Large states: 12 bits with 16 amplitudes a thread, 256 threads, five
// work-groups to a CU, which overlap their HBM and arithmetic phases
// (complex128 layered circuit, 24 and 28 qubits, 13-bit tiles 1.73 and 24.5
// ms, 12 bits 1.80 and 21.8, 11 bits 25.7 at 28).
//
// Up to 19 qubits such tiles leave most SIMDs idle and each wave is a long
// chain: 10 bits with 4 amplitudes a thread spread the arithmetic 16 times as
// wide, at the price of more exchanges and of more passes (layered circuits, 12
// bits and 16 amplitudes / 10 and 4, complex128, 13 qubits: 358 / 266 us, 14:
// 314 / 281, 16: 358 / 321, 17: 396 / 368, 19: 425 / 404, 20: equal, 21: 519 /
// 567; complex64 13: 278 / 262, 14: 293 / 278, 19: 363 / 354, 20: 420 / 433).
// A state of up to 12 qubits is one tile, so a pass ends only where its program
// is full, with 4 amplitudes a thread while 512 threads hold it (10 qubits 16 /
// 4 amplitudes 142 / 124 us, 8 qubits 111 / 99).
static int pass_tile_bits(int n) { return n <= kPMaxTile ? n : n < 20 ? 10 : kPMaxTile; }
static int pass_reg_bits(int tb) { return tb <= kPThrBits + 2 ? 2 : kPRegBits; }

// Two-norm bounds (log2) under which no amplitude can overflow: beyond them
// the products by exact zeros are no longer zeros and the gates run one by
// one.
static double bound_limit(const qcs_hip_state *s) {
  return s->precision == QCS_HIP_C128 ? 900.0 : 100.0;
}

bool bounded(const qcs_hip_state *s) { return s->log2_bound < bound_limit(s); }

void bound_reset(qcs_hip_state *s, double log2_norm) { s->log2_bound = log2_norm; }

void bound_normalized(qcs_hip_state *s) {
  if (bounded(s)) s->log2_bound = 1.0;
}

// growth of the two-norm by a matrix of `count` complex entries: its
// Frobenius norm
void bound_matrix(qcs_hip_state *s, const double *m, long count) {
  double f = 0.0;
  for (long i = 0; i < 2 * count; ++i) f += m[i] * m[i];
  f = 0.5 * std::log2(f);
  s->log2_bound += f > 0.0 || f != f ? f : 0.0;
}

void bound_gate(qcs_hip_state *s, const double m[8]) {
  const double a = m[0] * m[0] + m[1] * m[1] + m[4] * m[4] + m[5] * m[5];
  const double b = m[2] * m[2] + m[3] * m[3] + m[6] * m[6] + m[7] * m[7];
  const double re = m[0] * m[2] + m[1] * m[3] + m[4] * m[6] + m[5] * m[7];
  const double im = m[0] * m[3] - m[1] * m[2] + m[4] * m[7] - m[5] * m[6];
  const double e = 1e-9;
  if (std::fabs(a - 1.0) < e && std::fabs(b - 1.0) < e && std::fabs(re) < e && std::fabs(im) < e)
    s->log2_bound += 1e-8;
  else
    bound_matrix(s, m, 4);  // never less than before: a controlled gate keeps a half
}

static int launch_gate(qcs_hip_state *s, int kind, int target, int control, const double *m) {
  if (kind == QCS_HIP_G_1Q) return launch_1q(s, target, m);
  if (kind == QCS_HIP_G_CU) return launch_cu(s, control, target, m);
  return launch_swap(s, target, control);
}

template <typename T>
static int launch_pass(qcs_hip_state *s, const PassPick &pick,
                       const std::vector<PassGroup> &groups, int tb) {
  typedef typename Amp<T>::type A;
  PassProgram prog;
  write_pass<T>(s->queue, pick, groups, s->n, tb, s->support, s->basis, &prog, s->filled);
  const int outer_bits = __builtin_popcountll(prog.outer);
  const int halves = prog.nswaps > 0 ? 2 : 1;
  const int threads = std::max(64, halves << (tb - pick.rb));
  const size_t slot = pick.rb < kPRegBits ? sizeof(A) : 8;
  const size_t lds = prog.nlayouts > 1 ? (slot * size_t(halves)) << tb : 0;
  TimedLaunch tl;
  const double amps = double(uint64_t(1) << (outer_bits + 2 * int(prog.nswaps) + tb));
  const double read = amps / double(uint64_t(1) << __builtin_popcountll(prog.skip_t | prog.skip_r));
  timing_begin(s, QCS_HIP_K_FUSED, (amps + read) * sizeof(A),
               6.0 * amps * double(pick.gates.size()), &tl);
  const dim3 grid(unsigned(pass_work_groups(&prog, outer_bits))), block{unsigned(threads)};
  A *a = static_cast<A *>(s->vec);
  if (pick.rb == 2)
    hipLaunchKernelGGL((k_gate_pass<T, 2>), grid, block, lds, s->stream, prog, a);
  else
    hipLaunchKernelGGL((k_gate_pass<T, 4>), grid, block, lds, s->stream, prog, a);
  int rc = launch_check("k_gate_pass");
  if (rc) return rc;
  if (s->filled != ~uint64_t(0)) {
    s->filled |= pick.bits | pick.swapped;
    if ((~s->filled & (s->size - 1)) == 0) s->filled = ~uint64_t(0);
  }
  return timing_end(s, &tl);
}

// Launches passes from the head of the queue: all of it, or only those that
// further gates would not change, while enough is left to plan the next.  A
// launch that fails loses its own gates, as a gate's own launch would; those
// behind it still run, and the first failure is the result.
static int run_queue(qcs_hip_state *s, bool all) {
  std::vector<PlanGate> &q = s->queue;
  PassPick pick;
  std::vector<PassGroup> groups;
  std::vector<int> taken;  // the pick's gates and SWAPs
  bool open = false;  // the last pick would take more gates
  int first_rc = 0;
  const int tb = pass_tile_bits(s->n);
  const int words = s->precision == QCS_HIP_C128 ? 2 : 1;
  while (!q.empty() && (all || q.size() >= kQueueLow)) {
    plan_pick(q, s->n, tb, kPassLowBits, words, 64, &pick, &groups, s->n > tb,
              pass_reg_bits(tb));
    if (!all && !pick.full && q.size() < kQueueMax) {
      open = true;
      break;
    }
    taken.clear();
    std::merge(pick.gates.begin(), pick.gates.end(), pick.swaps.begin(), pick.swaps.end(),
               std::back_inserter(taken));
    int rc;
    double traffic = 0.0;
    for (int i : taken) traffic += plan_gate_traffic(q[size_t(i)]);
    if (taken.size() <= 1 || (s->n >= kPassBigState && traffic <= 2.0)) {
      // the per-gate kernels move no more than the pass would
      if (taken.empty()) taken.push_back(0);
      const int fill_rc = rc = launch_fill_rest(s);
      for (int i : taken) {
        if (fill_rc) break;  // memory is not the state yet
        const PlanGate &g = q[size_t(i)];
        const int kind = g.cls == kGSwap ? QCS_HIP_G_SWAP : g.c >= 0 ? QCS_HIP_G_CU : QCS_HIP_G_1Q;
        const int gate_rc = launch_gate(s, kind, g.t, g.c, g.m);
        if (gate_rc && !rc) rc = gate_rc;
      }
    } else {
      rc = s->precision == QCS_HIP_C128 ? launch_pass<double>(s, pick, groups, tb)
                                        : launch_pass<float>(s, pick, groups, tb);
    }
    if (rc && !first_rc) first_rc = rc;
    if (rc) s->support = ~uint64_t(0);
    for (int i : taken) s->support |= plan_spread(q[size_t(i)]);
    size_t keep = 0, x = 0;
    for (size_t i = 0; i < q.size(); ++i) {
      if (x < taken.size() && size_t(taken[x]) == i) ++x;
      else q[keep++] = q[i];
    }
    q.resize(keep);
  }
  s->queue_mark = queue_next_look(q.size(), open);
  return first_rc;
}

// (the planner's vectors may throw; the queue is whole either way)
int queue_flush(qcs_hip_state *s, bool fill) try {
  if (!s->queued) return 0;
  std::lock_guard<std::mutex> lock(s->queue_mu);
  const int rc = s->queue.empty() ? 0 : run_queue(s, true);
  const int fill_rc = fill ? launch_fill_rest(s) : 0;
  return rc ? rc : fill_rc;
} catch (const std::exception &) {
  return fail(QCS_HIP_ENOMEM, "planning the queued gates: out of host memory");
}

// what could not be launched, given up
void queue_drop(qcs_hip_state *s) {
  std::lock_guard<std::mutex> lock(s->queue_mu);
  s->queue.clear();
}

int queue_gate(qcs_hip_state *s, int kind, int target, int control, const double *m) try {
  if (!s->queued) return launch_gate(s, kind, target, control, m);
  std::lock_guard<std::mutex> lock(s->queue_mu);
  if (kind != QCS_HIP_G_SWAP) bound_gate(s, m);
  const PlanGate g = plan_gate(kind, target, control, m);
  if (g.cls == kGCuDense || !bounded(s)) {
    const int earlier = s->queue.empty() ? 0 : run_queue(s, true);
    int rc = launch_fill_rest(s);
    s->support = ~uint64_t(0);  // 0 times infinity
    if (!rc) rc = launch_gate(s, kind, target, control, m);
    return earlier ? earlier : rc;
  }
  s->queue.push_back(g);
  return s->queue.size() >= s->queue_mark ? run_queue(s, false) : 0;
} catch (const std::exception &) {
  return fail(QCS_HIP_ENOMEM, "queueing a gate: out of host memory");
}

}  // namespace qcs
