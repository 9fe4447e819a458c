// FP64 reductions and the observation path: norm / renormalise, qubit
// probabilities + collapse (measurement), argmax, shot sampling, Grover's
// oracle and diffusion, and the state comparison (1 - F, max-abs).
//
// Every reduction runs on a fixed grid of <= kRedBlocks work-groups that
// write per-block partials; one work-group then folds the partials in a fixed
// order, so results are bit-reproducible run to run.
#include <algorithm>
#include <cmath>
#include <mutex>

#include "device.h"
#include "internal.h"

namespace qcs {

static unsigned red_blocks(uint64_t n) {
  const uint64_t b = ceil_div(n, uint64_t(kThreads) * 4);
  return unsigned(b < uint64_t(kRedBlocks) ? (b ? b : 1) : kRedBlocks);
}

// ---- generic partial + final ---------------------------------------------------

// Sum |a|^2, split by bit q of the index when q >= 0 (slot 0: bit = 0,
// slot 1: bit = 1); q < 0 puts everything in slot 0.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_norm_partial(
    const typename Amp<T>::type *a, uint64_t n, int q, double *partial) {
  __shared__ double lds[kThreads / 64];
  double s0 = 0.0, s1 = 0.0;
  const uint64_t qb = q >= 0 ? (uint64_t(1) << q) : 0;
  // XCD-ordered virtual blocks (each XCD reads one contiguous range), four
  // loads in flight per thread
  const uint64_t nvb = ceil_div(n, uint64_t(kThreads)), G = gridDim.x;
  auto at = [&](uint64_t vb) { return xcd_order(vb, nvb) * kThreads + threadIdx.x; };
  uint64_t vb = blockIdx.x;
  for (; vb + 3 * G < nvb; vb += 4 * G) {
    const uint64_t i0 = at(vb), i1 = at(vb + G), i2 = at(vb + 2 * G), i3 = at(vb + 3 * G);
    // xcd_order can put the grid's one partial virtual block at any of the
    // four slots, so each load is guarded (a skipped term adds 0.0: the
    // association of the sum is unchanged)
    const double p0 = i0 < n ? norm2(ld_stream(a + i0)) : 0.0;
    const double p1 = i1 < n ? norm2(ld_stream(a + i1)) : 0.0;
    const double p2 = i2 < n ? norm2(ld_stream(a + i2)) : 0.0;
    const double p3 = i3 < n ? norm2(ld_stream(a + i3)) : 0.0;
    if (i0 & qb) s1 += p0; else s0 += p0;
    if (i1 & qb) s1 += p1; else s0 += p1;
    if (i2 & qb) s1 += p2; else s0 += p2;
    if (i3 & qb) s1 += p3; else s0 += p3;
  }
  for (; vb < nvb; vb += G) {
    const uint64_t i = at(vb);
    if (i >= n) continue;
    const double p = norm2(ld_stream(a + i));
    if (i & qb) s1 += p; else s0 += p;
  }
  s0 = block_sum(s0, lds);
  s1 = block_sum(s1, lds);
  if (threadIdx.x == 0) {
    partial[blockIdx.x * kRedSlots + 0] = s0;
    partial[blockIdx.x * kRedSlots + 1] = s1;
  }
}

// Sum |a|^2 over the half of the state whose bit q is set (bq = 2^q) or
// clear (bq = 0): half-index j is amplitude insert0(j, q) | bq, so the half
// is read in runs of 2^q amplitudes (the caller uses it where a run is at
// least a 128-byte line).  Same loop shape as k_norm_partial; slot 0 only.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_half_norm_partial(
    const typename Amp<T>::type *a, uint64_t nh, int q, uint64_t bq, double *partial) {
  __shared__ double lds[kThreads / 64];
  double s0 = 0.0;
  const uint64_t nvb = ceil_div(nh, uint64_t(kThreads)), G = gridDim.x;
  auto at = [&](uint64_t vb) {
    return insert0(xcd_order(vb, nvb) * kThreads + threadIdx.x, q) | bq;
  };
  auto inside = [&](uint64_t vb) { return xcd_order(vb, nvb) * kThreads + threadIdx.x < nh; };
  uint64_t vb = blockIdx.x;
  for (; vb + 3 * G < nvb; vb += 4 * G) {
    // each of the four may be the partial virtual block (see k_norm_partial)
    const double p0 = inside(vb) ? norm2(ld_stream(a + at(vb))) : 0.0;
    const double p1 = inside(vb + G) ? norm2(ld_stream(a + at(vb + G))) : 0.0;
    const double p2 = inside(vb + 2 * G) ? norm2(ld_stream(a + at(vb + 2 * G))) : 0.0;
    const double p3 = inside(vb + 3 * G) ? norm2(ld_stream(a + at(vb + 3 * G))) : 0.0;
    s0 += p0;
    s0 += p1;
    s0 += p2;
    s0 += p3;
  }
  for (; vb < nvb; vb += G)
    if (inside(vb)) s0 += norm2(ld_stream(a + at(vb)));
  s0 = block_sum(s0, lds);
  if (threadIdx.x == 0) partial[blockIdx.x * kRedSlots + 0] = s0;
}

// Fold `nb` partials of `nslots` slots: slots in max_mask take the maximum,
// the others the sum.  Results go to out[0..nslots).
__global__ __launch_bounds__(kThreads) void k_final(const double *partial,
                                                    int nb, int nslots,
                                                    unsigned max_mask,
                                                    double *out) {
  __shared__ double lds[kThreads];
  for (int slot = 0; slot < nslots; ++slot) {
    const bool is_max = (max_mask >> slot) & 1u;
    double v = 0.0;
    for (int b = threadIdx.x; b < nb; b += kThreads) {
      const double x = partial[b * kRedSlots + slot];
      v = is_max ? fmax(v, x) : v + x;
    }
    lds[threadIdx.x] = v;
    __syncthreads();
    for (int w = kThreads / 2; w > 0; w >>= 1) {
      if (threadIdx.x < w) {
        const double y = lds[threadIdx.x + w];
        lds[threadIdx.x] = is_max ? fmax(lds[threadIdx.x], y)
                                  : lds[threadIdx.x] + y;
      }
      __syncthreads();
    }
    if (threadIdx.x == 0) out[slot] = lds[0];
    __syncthreads();
  }
}

// a *= factor
template <typename T>
__global__ __launch_bounds__(kThreads) void k_scale(typename Amp<T>::type *a,
                                                    uint64_t n, double f) {
  const uint64_t nvb = ceil_div(n, uint64_t(kThreads));
  for (uint64_t vb = blockIdx.x; vb < nvb; vb += gridDim.x) {
    const uint64_t i = xcd_order(vb, nvb) * kThreads + threadIdx.x;
    if (i >= n) continue;
    typename Amp<T>::type v = ld_stream(a + i);
    v.x = T(double(v.x) * f);
    v.y = T(double(v.y) * f);
    st_stream(a + i, v);
  }
}

// a *= 1/sqrt(ns) when ns > 1e-12 and ns != 1 (q_state_normalize's guard,
// src/q_utils.c:112-118), with ns read from device memory.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_scale_dev(
    typename Amp<T>::type *a, uint64_t n, const double *ns) {
  const double v = *ns;
  if (!(v > 1e-12 && v != 1.0)) return;
  const double f = 1.0 / sqrt(v);
  const uint64_t nvb = ceil_div(n, uint64_t(kThreads));
  for (uint64_t vb = blockIdx.x; vb < nvb; vb += gridDim.x) {
    const uint64_t i = xcd_order(vb, nvb) * kThreads + threadIdx.x;
    if (i >= n) continue;
    typename Amp<T>::type x = ld_stream(a + i);
    x.x = T(double(x.x) * f);
    x.y = T(double(x.y) * f);
    st_stream(a + i, x);
  }
}

// qc_measure's collapse: zero the amplitudes whose bit q differs from
// `outcome`, scale the others by f when do_scale.
template <typename T>
__device__ __forceinline__ void collapse_body(typename Amp<T>::type *a, uint64_t n, int q,
                                              int outcome, double f, int do_scale);

template <typename T>
__global__ __launch_bounds__(kThreads) void k_collapse(
    typename Amp<T>::type *a, uint64_t n, int q, int outcome, double f,
    int do_scale) {
  collapse_body<T>(a, n, q, outcome, f, do_scale);
}

// qc_measure's decision on the device (src/qcs.c:261-283): m[0], m[1] hold
// p0 and p1; outcome = (u <= p0) ? 0 : 1, and the kept half, whose norm is
// p0 or p1, is rescaled by 1/sqrt of it when that is > 1e-12 and != 1 (the
// rule of q_state_normalize).  m[2..4] = outcome, factor, rescale flag; the
// outcome also goes to *record.
__global__ void k_measure_decide(double *m, double u, double *record) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const double p0 = m[0], p1 = m[1];
  const int o = (u <= p0) ? 0 : 1;
  const double ns = o == 0 ? p0 : p1;
  const int sc = (ns > 1e-12 && ns != 1.0) ? 1 : 0;
  m[2] = double(o);
  m[3] = sc ? 1.0 / sqrt(ns) : 1.0;
  m[4] = double(sc);
  *record = double(o);
}

// k_collapse with the outcome, factor and flag k_measure_decide wrote
template <typename T>
__global__ __launch_bounds__(kThreads) void k_collapse_dev(typename Amp<T>::type *a,
                                                           uint64_t n, int q,
                                                           const double *m) {
  collapse_body<T>(a, n, q, int(m[2]), m[3], int(m[4]));
}

template <typename T>
__device__ __forceinline__ void collapse_body(typename Amp<T>::type *a, uint64_t n, int q,
                                              int outcome, double f, int do_scale) {
  const uint64_t nvb = ceil_div(n, uint64_t(kThreads));
  for (uint64_t vb = blockIdx.x; vb < nvb; vb += gridDim.x) {
    const uint64_t i = xcd_order(vb, nvb) * kThreads + threadIdx.x;
    if (i >= n) continue;
    const int bit = int((i >> q) & 1);
    typename Amp<T>::type v;
    if (bit != outcome) {
      v.x = T(0);
      v.y = T(0);
      st_stream(a + i, v);
    } else if (do_scale) {
      v = ld_stream(a + i);
      v.x = T(double(v.x) * f);
      v.y = T(double(v.y) * f);
      st_stream(a + i, v);
    }
  }
}

// ---- measurement of qubits 0, 1, ... in order ------------------------------------
//
// qc_measure_all measures every qubit in turn; one after another each costs
// two reads of half the state and a rewrite of all of it.  But the outcome of
// the lowest kMargBits qubits only needs their joint weights, which one read
// gives: W[x] = sum of |a_i|^2 over the i whose low bits are x.  The sums over
// fewer of the bits follow by halving W, so k_marg_decide walks the qubits
// with the probabilities (p0, p1) the collapsed state would have.  The
// survivors, one amplitude in 2^kMargBits, give the next qubits' weights the
// same way, and one write collapses the state at the end.  26 qubits,
// complex128: read 1 GiB and write 1 GiB instead of moving 2.5 GiB 26 times;
// 13.1 -> 0.44 ms.
constexpr int kMargBits = 10;
constexpr int kMargSize = 1 << kMargBits;
constexpr int kMargBlocks = 1024;  // work-groups of the first read, at most

struct MargUniforms {
  double u[kMargBits];
};
// device side, after the partials: the folded weights, then
struct MargState {
  double scale;         // product of the factors so far
  uint64_t pattern;     // outcomes so far: bit q = outcome of qubit q
  double factor[kMaxQubits];
  double outcome[kMaxQubits];
};

// Weights of the `lb` index bits from `shift` up, over the amplitudes whose
// lower bits are the outcomes so far.  A thread keeps the sums of the
// patterns threadIdx.x + k * 256, so the state is read in whole lines.
__global__ __launch_bounds__(kThreads) void k_marg_partial(
    const double2 *a, uint64_t rows, int lb, int shift, const MargState *ms,
    double *partial) {
  constexpr int P = kMargSize / kThreads;
  const uint64_t pat = shift ? ms->pattern : 0;
  double s[P];
#pragma unroll
  for (int k = 0; k < P; ++k) s[k] = 0.0;
  auto at = [&](uint64_t r, int k) {
    return a + ((((r << lb) | (threadIdx.x + unsigned(k) * kThreads)) << shift) | pat);
  };
  if (lb == kMargBits) {
    uint64_t vr = blockIdx.x;
    const uint64_t G = gridDim.x;
    for (; vr + G < rows; vr += 2 * G) {  // eight loads in flight per thread
      const uint64_t r0 = xcd_order(vr, rows), r1 = xcd_order(vr + G, rows);
      double p[2 * P];
#pragma unroll
      for (int k = 0; k < P; ++k) {
        p[k] = norm2(ld_stream(at(r0, k)));
        p[P + k] = norm2(ld_stream(at(r1, k)));
      }
#pragma unroll
      for (int k = 0; k < P; ++k) s[k] += p[k] + p[P + k];
    }
    for (; vr < rows; vr += G) {
      const uint64_t r = xcd_order(vr, rows);
#pragma unroll
      for (int k = 0; k < P; ++k) s[k] += norm2(ld_stream(at(r, k)));
    }
  } else {  // the last qubits: one row of fewer patterns
#pragma unroll
    for (int k = 0; k < P; ++k)
      if (int(threadIdx.x) + k * kThreads < (1 << lb)) s[k] = norm2(ld_stream(at(0, k)));
  }
#pragma unroll
  for (int k = 0; k < P; ++k)
    partial[uint64_t(blockIdx.x) * kMargSize + threadIdx.x + unsigned(k) * kThreads] = s[k];
}

// w[x] = sum of the nb partials of pattern x; 64 patterns per work-group, four
// slices of the partials summed side by side
__global__ __launch_bounds__(kThreads) void k_marg_fold(const double *partial, int nb,
                                                        double *w) {
  __shared__ double lds[kThreads];
  const int x = int(blockIdx.x) * 64 + (threadIdx.x & 63), slice = threadIdx.x >> 6;
  // sixteen loads ahead of their additions (26 qubits 78 -> 19 us)
  constexpr int U = 16, S = kThreads / 64;
  double s = 0.0;
  for (int b = slice; b < nb; b += U * S) {
    double v[U];
#pragma unroll
    for (int k = 0; k < U; ++k)
      v[k] = b + k * S < nb ? partial[uint64_t(b + k * S) * kMargSize + x] : 0.0;
#pragma unroll
    for (int k = 0; k < U; ++k) s += v[k];
  }
  lds[threadIdx.x] = s;
  __syncthreads();
  if (slice == 0)
    w[x] = (lds[threadIdx.x] + lds[threadIdx.x + 64]) +
           (lds[threadIdx.x + 128] + lds[threadIdx.x + 192]);
}

// qc_measure's decision for `count` qubits from qubit `shift` on (the first
// `count` of the lb bits that w covers): outcome = (u <= p0) ? 0 : 1, rescale
// factor 1/sqrt(p) of the kept half when that is > 1e-12 and != 1
__global__ __launch_bounds__(kThreads) void k_marg_decide(const double *w, int lb, int shift,
                                                          int count, MargUniforms un,
                                                          MargState *ms) {
  // level b at offset 2^(b+1) - 2: the weights of patterns of bits 0..b
  __shared__ double tree[2 * kMargSize];
  const int top = 1 << lb;
  for (int x = threadIdx.x; x < top; x += kThreads) tree[top - 2 + x] = w[x];
  __syncthreads();
  for (int size = top >> 1; size >= 2; size >>= 1) {
    for (int x = threadIdx.x; x < size; x += kThreads)
      tree[size - 2 + x] = tree[2 * size - 2 + x] + tree[2 * size - 2 + size + x];
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  double f = shift ? ms->scale : 1.0;
  uint64_t pat = 0;
  for (int b = 0; b < count; ++b) {
    const double *t = tree + ((2 << b) - 2);
    const double p0 = t[pat] * (f * f), p1 = t[pat | (uint64_t(1) << b)] * (f * f);
    const int o = (un.u[b] <= p0) ? 0 : 1;
    const double ns = o == 0 ? p0 : p1;
    const double g = (ns > 1e-12 && ns != 1.0) ? 1.0 / sqrt(ns) : 1.0;
    if (o) pat |= uint64_t(1) << b;
    f *= g;
    ms->factor[shift + b] = g;
    ms->outcome[shift + b] = double(o);
  }
  ms->scale = f;
  ms->pattern = (shift ? ms->pattern : 0) | (pat << shift);
}

// the measurements' collapses at once: zero where one of the `count` low bits
// differs from its outcome, the factors one after another elsewhere
__global__ __launch_bounds__(kThreads) void k_marg_collapse(double2 *a, uint64_t n, int count,
                                                            const MargState *ms) {
  const uint64_t mask = (uint64_t(1) << count) - 1, pat = ms->pattern;
  const uint64_t nvb = ceil_div(n, uint64_t(kThreads));
  for (uint64_t vb = blockIdx.x; vb < nvb; vb += gridDim.x) {
    const uint64_t i = xcd_order(vb, nvb) * kThreads + threadIdx.x;
    if (i >= n) continue;
    double2 v = make_double2(0.0, 0.0);
    if ((i & mask) == pat) {
      v = a[i];
      for (int q = 0; q < count; ++q)
        if (ms->factor[q] != 1.0) {
          v.x *= ms->factor[q];
          v.y *= ms->factor[q];
        }
    }
    st_stream(a + i, v);
  }
}

// ---- argmax -------------------------------------------------------------------

__device__ __forceinline__ bool better(double p, uint64_t i, double bp,
                                       uint64_t bi) {
  return p > bp || (p == bp && i < bi);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_argmax_partial(
    const typename Amp<T>::type *a, uint64_t n, double *partial) {
  __shared__ double lp[kThreads];
  __shared__ uint64_t li[kThreads];
  double bp = -1.0;
  uint64_t bi = ~uint64_t(0);
  // XCD-ordered virtual blocks, four loads in flight; a thread does not
  // visit its indices in increasing order, so ties go to the smaller index
  // explicitly (the first maximum in index order wins; NaN is skipped)
  const uint64_t nvb = ceil_div(n, uint64_t(kThreads)), G = gridDim.x;
  auto at = [&](uint64_t vb) { return xcd_order(vb, nvb) * kThreads + threadIdx.x; };
  auto take = [&](double p, uint64_t i) {
    if (better(p, i, bp, bi)) {
      bp = p;
      bi = i;
    }
  };
  uint64_t vb = blockIdx.x;
  for (; vb + 3 * G < nvb; vb += 4 * G) {
    const uint64_t i0 = at(vb), i1 = at(vb + G), i2 = at(vb + 2 * G), i3 = at(vb + 3 * G);
    // any of the four may be the partial virtual block (see k_norm_partial)
    const double p0 = i0 < n ? norm2(ld_stream(a + i0)) : -1.0;
    const double p1 = i1 < n ? norm2(ld_stream(a + i1)) : -1.0;
    const double p2 = i2 < n ? norm2(ld_stream(a + i2)) : -1.0;
    const double p3 = i3 < n ? norm2(ld_stream(a + i3)) : -1.0;
    if (i0 < n) take(p0, i0);
    if (i1 < n) take(p1, i1);
    if (i2 < n) take(p2, i2);
    if (i3 < n) take(p3, i3);
  }
  for (; vb < nvb; vb += G) {
    const uint64_t i = at(vb);
    if (i < n) take(norm2(ld_stream(a + i)), i);
  }
  lp[threadIdx.x] = bp;
  li[threadIdx.x] = bi;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      const double p = lp[threadIdx.x + w];
      const uint64_t i = li[threadIdx.x + w];
      if (better(p, i, lp[threadIdx.x], li[threadIdx.x])) {
        lp[threadIdx.x] = p;
        li[threadIdx.x] = i;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    partial[blockIdx.x * kRedSlots + 0] = lp[0];
    partial[blockIdx.x * kRedSlots + 1] = __longlong_as_double((long long)li[0]);
  }
}

__global__ __launch_bounds__(kThreads) void k_argmax_final(
    const double *partial, int nb, double *out) {
  __shared__ double lp[kThreads];
  __shared__ uint64_t li[kThreads];
  double bp = -1.0;
  uint64_t bi = ~uint64_t(0);
  for (int b = threadIdx.x; b < nb; b += kThreads) {
    const double p = partial[b * kRedSlots + 0];
    const uint64_t i = uint64_t(__double_as_longlong(partial[b * kRedSlots + 1]));
    if (better(p, i, bp, bi)) {
      bp = p;
      bi = i;
    }
  }
  lp[threadIdx.x] = bp;
  li[threadIdx.x] = bi;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) {
      const double p = lp[threadIdx.x + w];
      const uint64_t i = li[threadIdx.x + w];
      if (better(p, i, lp[threadIdx.x], li[threadIdx.x])) {
        lp[threadIdx.x] = p;
        li[threadIdx.x] = i;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = lp[0];
    out[1] = __longlong_as_double((long long)li[0]);
  }
}

// ---- sampling -------------------------------------------------------------------
//
// The CDF of qc_run_shots (src/qcs.c:597-604) is defined blockwise:
//   chunk c covers indices [c*L, (c+1)*L), L = min(kChunk, N), read as rows of
//   64; inside a row the 64 lanes take an inclusive wave scan; rows are
//   chained by a sequential running sum.  chunk_tot[c] is the final running
//   sum.  E[c] (exclusive) and P[c] = E[c] + chunk_tot[c] come from a
//   sequential chain per scan thread.  cdf(i) = E[c] + local(i).
// The sampling kernel recomputes local(i) with the same operations, so
// cdf(last of chunk c) == P[c] bit for bit.

//
// The rows' totals do not depend on one another, only their chain does: a
// work-group takes a chunk, its waves the rows, and one lane runs the chain.
// (A wave per chunk, row after row, waited for memory and for the scan's
// lane crossings 64 times over: at 20 qubits 43 -> 6 us; at 28 qubits, bound by
// HBM either way, 0.73 -> 0.71 ms.)
constexpr int kRowWaves = kThreads / 64;
constexpr int kRowsMax = int(kChunk / 64);

// totals of the chunk's rows (as wave_incl_scan's last lane) into rows[]
template <typename A>
__device__ __forceinline__ void chunk_rows(const A *p, uint64_t len, double *rows) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int U = kRowsMax / kRowWaves;
  A v[U];
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const uint64_t i = uint64_t(k * kRowWaves + wave) * 64 + lane;
    v[k].x = v[k].y = 0;
    if (i < len) v[k] = p[i];
  }
#pragma unroll
  for (int k = 0; k < U; ++k) {
    const double t = wave_scan_total(norm2(v[k]));
    if (lane == 0) rows[k * kRowWaves + wave] = t;
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_chunk_tot(const typename Amp<T>::type *a,
                                                        uint64_t len, double *tot) {
  __shared__ double rows[kRowsMax];
  const uint64_t c = blockIdx.x;
  chunk_rows(a + c * len, len, rows);
  __syncthreads();
  if (threadIdx.x != 0) return;
  double running = 0.0;
#pragma unroll 16
  for (int r = 0; r < kRowsMax; ++r) running = running + rows[r];
  tot[c] = running;
}

// One work-group: excl[c] (in place over tot) and inc[c] = excl[c] + tot[c].
// The additions run in a fixed order (each thread's segment left to right,
// then the segment sums left to right), which the batch kernel's sampling
// shares; the loads are issued 16 at a time ahead of the additions, so the
// sequential chains wait on arithmetic rather than on memory.
__global__ __launch_bounds__(1024) void k_chunk_scan(double *tot, double *inc,
                                                     uint64_t nchunks) {
  constexpr int U = 16;
  __shared__ double base[1024];
  const uint64_t per = ceil_div(nchunks, 1024);
  const uint64_t b = uint64_t(threadIdx.x) * per;
  const uint64_t e = b + per < nchunks ? b + per : nchunks;
  double s = 0.0;
  uint64_t c = b;
  // A thread's segment is contiguous, so a wave's load touches 64 lines: in
  // pairs, where the segments are even, it does so half as often (64 Ki chunks
  // 112 -> 77 us).
  typedef double Pair __attribute__((ext_vector_type(2)));
  const bool pairs = per % 2 == 0;
  auto load = [&](uint64_t at, double (&v)[U]) {
    if (pairs) {
#pragma unroll
      for (int j = 0; j < U; j += 2) {
        const Pair p = *reinterpret_cast<const Pair *>(tot + at + j);
        v[j] = p.x;
        v[j + 1] = p.y;
      }
    } else {
#pragma unroll
      for (int j = 0; j < U; ++j) v[j] = tot[at + j];
    }
  };
  auto store = [&](double *to, const double (&v)[U]) {
    if (pairs) {
#pragma unroll
      for (int j = 0; j < U; j += 2) *reinterpret_cast<Pair *>(to + j) = Pair{v[j], v[j + 1]};
    } else {
#pragma unroll
      for (int j = 0; j < U; ++j) to[j] = v[j];
    }
  };
  for (; c + U <= e; c += U) {
    double v[U];
    load(c, v);
#pragma unroll
    for (int j = 0; j < U; ++j) s = s + v[j];
  }
  for (; c < e; ++c) s = s + tot[c];
  base[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double run = 0.0;
    // (the threads past the last chunk hold zeros)
    const int used = int(ceil_div(nchunks, per));
    for (int t0 = 0; t0 < used; t0 += U) {
      double v[U];
#pragma unroll
      for (int j = 0; j < U; ++j) v[j] = base[t0 + j];
#pragma unroll
      for (int j = 0; j < U; ++j) {
        base[t0 + j] = run;
        run = run + v[j];
      }
    }
  }
  __syncthreads();
  double run = base[threadIdx.x];
  c = b;
  for (; c + U <= e; c += U) {
    double v[U], w[U];
    load(c, v);
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const double t = v[j];
      v[j] = run;
      run = run + t;
      w[j] = run;
    }
    store(tot + c, v);
    store(inc + c, w);
  }
  for (; c < e; ++c) {
    const double t = tot[c];
    tot[c] = run;
    run = run + t;
    inc[c] = run;
  }
}

// first chunk whose inclusive prefix exceeds u (inc is non-decreasing)
__device__ __forceinline__ uint64_t find_chunk(const double *inc, uint64_t nchunks, double u) {
  uint64_t lo = 0, hi = nchunks;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if (inc[mid] > u) hi = mid; else lo = mid + 1;
  }
  return lo;
}

// A wave per shot, its chunk row by row.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_sample(
    const typename Amp<T>::type *a, uint64_t nchunks, uint64_t len,
    const double *excl, const double *inc, const double *u, uint64_t shots,
    long *out) {
  const int lane = threadIdx.x & 63;
  const uint64_t s = uint64_t(blockIdx.x) * (kThreads / 64) + (threadIdx.x >> 6);
  if (s >= shots) return;
  const double us = u[s];
  const uint64_t c = find_chunk(inc, nchunks, us);
  if (c >= nchunks) {  // u not below the total: dropped, as the reference
    if (lane == 0) out[s] = -1;
    return;
  }
  const double e = excl[c];
  const typename Amp<T>::type *p = a + c * len;
  double running = 0.0;
  long found = -1, last_nz = -1;
  for (uint64_t r = 0; r < len; r += 64) {
    const double x = (r + lane < len) ? norm2(p[r + lane]) : 0.0;
    const double sc = wave_incl_scan(x, lane);
    const double local = running + sc;
    const double cdf = e + local;
    const unsigned long long hit = __ballot(cdf > us && x > 0.0);
    const unsigned long long nz = __ballot(x > 0.0);
    if (nz) last_nz = long(c * len + r) + 63 - __clzll(nz);
    if (hit) {
      found = long(c * len + r) + __ffsll(hit) - 1;
      break;
    }
    running = running + __shfl(sc, 63, 64);
  }
  // only reachable at an ulp-level seam of the chunk scan: take the last
  // non-zero amplitude seen in the chunk
  if (found < 0) found = last_nz;
  if (lane == 0) out[s] = found;
}

// A work-group per shot, while there are few: the chunk's rows are summed at
// once and only those that may hold the shot are scanned, by one wave.  It
// reads all of the chunk, which a wave per shot leaves half-way on average: at
// 20 qubits 14 us for 1024 shots and 44 for 8192 where a wave per shot takes
// 45 and 69, but at 28 qubits, from HBM, 20 and 86 against 23 and 78.
constexpr long kWideShots = 4096;

template <typename T>
__global__ __launch_bounds__(kThreads) void k_sample_wide(
    const typename Amp<T>::type *a, uint64_t nchunks, uint64_t len, const double *excl,
    const double *inc, const double *u, long *out) {
  constexpr int kHeld = 1024;
  __shared__ double held[kHeld], rows[kRowsMax];
  const int lane = threadIdx.x & 63;
  const double us = u[blockIdx.x];
  uint64_t c;
  if (nchunks <= kHeld) {  // the search's dependent reads from LDS
    for (uint64_t k = threadIdx.x; k < nchunks; k += kThreads) held[k] = inc[k];
    __syncthreads();
    c = find_chunk(held, nchunks, us);
  } else {
    c = find_chunk(inc, nchunks, us);
  }
  if (c >= nchunks) {
    if (threadIdx.x == 0) out[blockIdx.x] = -1;
    return;
  }
  const typename Amp<T>::type *p = a + c * len;
  chunk_rows(p, len, rows);
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const double e = excl[c];
  double running = 0.0, mine = 0.0;  // lane r: the sum of the rows before r
#pragma unroll 16
  for (int r = 0; r < kRowsMax; ++r) {
    if (r == lane) mine = running;
    running = running + rows[r];
  }
  const uint64_t nrows = ceil_div(len, 64);
  long found = -1;
  unsigned long long may =
      __ballot(uint64_t(lane) < nrows && row_may_hit(rows[lane], e, mine, us));
  for (; may && found < 0; may &= may - 1) {
    const int r = __ffsll(may) - 1;
    const uint64_t i = uint64_t(r) * 64 + lane;
    const double x = i < len ? norm2(p[i]) : 0.0;
    const unsigned long long hit = row_hits(x, lane, e, read_lane(mine, r), us);
    if (hit) found = long(c * len + uint64_t(r) * 64) + __ffsll(hit) - 1;
  }
  // (as in k_sample)
  for (uint64_t r = nrows; r-- > 0 && found < 0;) {
    const uint64_t i = r * 64 + lane;
    const unsigned long long nz = __ballot((i < len ? norm2(p[i]) : 0.0) > 0.0);
    if (nz) found = long(c * len + r * 64) + 63 - __clzll(nz);
  }
  if (lane == 0) out[blockIdx.x] = found;
}

// ---- Grover (textbook) ----------------------------------------------------
//
// One round: a[m] = -a[m]; mu = sum(a)/N; a = 2*mu - a.  Every amplitude but
// the marked one goes through the same map, so after k rounds
//   a_i = (-1)^k a_i(0) + c_k   (i != m)
// with one c_k for all, and the sums the rounds need follow from A = sum of
// a_i(0) over i != m, c_k and a_m(k) alone:
//   2 mu_k = 2 ((-1)^k A + (N - 1) c_k - a_m(k)) / N
//   c_k+1 = 2 mu_k - c_k,  a_m(k+1) = 2 mu_k + a_m(k).
// So any number of rounds reads the state once for A, runs the recurrence on
// two lanes (real and imaginary part) and rewrites the state once, where a
// sweep per round moved 2 N s each time.  Any starting state is allowed.  The
// recurrence runs on pairs of doubles, so it adds no error of its own and an
// amplitude is rounded once instead of every round: from random states of 8 to
// 16 qubits the amplitudes are 1.8e-17 off the exact rounds on average and
// 1.8e-16 at most, with a sweep per round 1.1e-16 and 3.1e-15 (emulated; with
// A, which is summed in plain doubles, in pairs too 1.0e-17 and 5.5e-17).  From
// the H layer the layer's own error stays: 4 to 19 qubits and up to 571 rounds,
// the marked probability is 7.0e-16 off the closed form on average and 3.0e-15
// at most, with a sweep per round 8.9e-16 and 1.7e-14.  At some sizes the
// sweeps' roundings happened to offset the layer's (14 qubits, 100 rounds:
// 9.0e-16, now 1.13e-15, which an exact A leaves as it is; in plain doubles the
// recurrence gave 2.0e-15).  27 qubits, 16 rounds: 11.7 -> 0.98 ms; 14 qubits,
// 100 rounds: 0.70 -> 0.032 ms, 0.26 us of it a round.

// partial sums of the amplitudes other than m
template <typename T>
__global__ __launch_bounds__(kThreads) void k_gsum_partial(
    const typename Amp<T>::type *a, uint64_t n, uint64_t m, double *partial) {
  __shared__ double lds[kThreads / 64];
  double sr = 0.0, si = 0.0;
  const uint64_t nvb = ceil_div(n, uint64_t(kThreads)), G = gridDim.x;
  auto at = [&](uint64_t vb) { return xcd_order(vb, nvb) * kThreads + threadIdx.x; };
  auto take = [&](uint64_t i, const typename Amp<T>::type &v) {
    sr += i == m ? 0.0 : double(v.x);
    si += i == m ? 0.0 : double(v.y);
  };
  uint64_t vb = blockIdx.x;
  if (n % kThreads == 0) {
    for (; vb + 3 * G < nvb; vb += 4 * G) {  // four loads in flight per thread
      const uint64_t i0 = at(vb), i1 = at(vb + G), i2 = at(vb + 2 * G), i3 = at(vb + 3 * G);
      const typename Amp<T>::type v0 = ld_stream(a + i0), v1 = ld_stream(a + i1),
                                  v2 = ld_stream(a + i2), v3 = ld_stream(a + i3);
      take(i0, v0);
      take(i1, v1);
      take(i2, v2);
      take(i3, v3);
    }
  }
  for (; vb < nvb; vb += G) {
    const uint64_t i = at(vb);
    if (i < n) take(i, ld_stream(a + i));
  }
  sr = block_sum(sr, lds);
  si = block_sum(si, lds);
  if (threadIdx.x == 0) {
    partial[blockIdx.x * kRedSlots + 0] = sr;
    partial[blockIdx.x * kRedSlots + 1] = si;
  }
}

// A sum of two doubles and its rounding error (Knuth); pairs added with
// about 100 significant bits (Joldes, Muller, Popescu 2017, algorithm 6).
struct Pair {
  double h, l;
};
__device__ __forceinline__ Pair two_sum(double a, double b) {
  const double s = a + b, t = s - a;
  return Pair{s, (a - (s - t)) + (b - t)};
}
__device__ __forceinline__ Pair pair_add(Pair a, Pair b) {
  Pair s = two_sum(a.h, b.h);
  const Pair t = two_sum(a.l, b.l);
  const double v = s.h + (s.l + t.h);
  const double w = ((s.l + t.h) - (v - s.h)) + t.l;
  return Pair{v + w, w - ((v + w) - v)};
}
__device__ __forceinline__ Pair pair_scale(Pair a, double f) { return Pair{a.h * f, a.l * f}; }

// the recurrence: out = {c re, c im, a_m re, a_m im, (-1)^iters}
template <typename T>
__global__ __launch_bounds__(kThreads) void k_grounds(const typename Amp<T>::type *a, uint64_t n,
                                                      uint64_t m, const double *partial, int nb,
                                                      long iters, double *out) {
  __shared__ double lds[kThreads / 64], sum[2];
  double sr = 0.0, si = 0.0;
  for (int b = threadIdx.x; b < nb; b += kThreads) {
    sr += partial[b * kRedSlots + 0];
    si += partial[b * kRedSlots + 1];
  }
  sr = block_sum(sr, lds);
  si = block_sum(si, lds);
  if (threadIdx.x == 0) {
    sum[0] = sr;
    sum[1] = si;
  }
  __syncthreads();
  if (threadIdx.x >= 2) return;
  // 2 / N is a power of two, so with N - 1 = N (1 - 1 / N) the map is
  //   c <- c + (+-2 A / N) - (2 / N) (c + a_m),  a_m <- a_m + c_old + c_new
  // in additions and exact scalings; without a marked amplitude the count is
  // N, and the last term of c falls away.
  const bool marked = m < n;
  const double f = 2.0 / double(n);
  const double s = sum[threadIdx.x];
  double am = 0.0;
  if (marked) am = threadIdx.x ? double(a[m].y) : double(a[m].x);
  Pair C = {0.0, 0.0}, M = {am, 0.0};
  double sg = 1.0;
  for (long k = 0; k < iters; ++k) {
    Pair next = pair_add(C, Pair{sg * s * f, 0.0});
    if (marked) {
      next = pair_add(next, pair_scale(pair_add(C, M), -f));
      M = pair_add(M, pair_add(C, next));
    }
    C = next;
    sg = -sg;
  }
  double c = C.h;
  if (marked) am = M.h;
  if (!(fabs(c) < 1e300 && fabs(am) < 1e300)) {
    // infinite or NaN: the error terms turn infinities into NaN, so the
    // rounds as they are
    const double count = marked ? double(n - 1) : double(n);
    double t = s;
    c = 0.0;
    if (marked) am = threadIdx.x ? double(a[m].y) : double(a[m].x);
    for (long k = 0; k < iters; ++k) {
      const double mu2 = ((t + count * c) - am) * f;
      c = mu2 - c;
      if (marked) am = mu2 + am;
      t = -t;
    }
  }
  out[threadIdx.x] = c;
  out[2 + threadIdx.x] = am;
  if (threadIdx.x == 0) out[4] = (iters & 1) ? -1.0 : 1.0;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_gapply(typename Amp<T>::type *a, uint64_t n,
                                                     uint64_t m, const double *r) {
  const double cr = r[0], ci = r[1], sg = r[4];
  const uint64_t nvb = ceil_div(n, uint64_t(kThreads));
  for (uint64_t vb = blockIdx.x; vb < nvb; vb += gridDim.x) {
    const uint64_t i = xcd_order(vb, nvb) * kThreads + threadIdx.x;
    if (i >= n) continue;
    typename Amp<T>::type v = ld_stream(a + i);
    v.x = T(i == m ? r[2] : cr + sg * double(v.x));
    v.y = T(i == m ? r[3] : ci + sg * double(v.y));
    st_stream(a + i, v);
  }
}

// ---- Grover (compat, as written in src/q_gates.c:305-356) -----------------

// after the host swapped the buffers: vector[m] = -scratch[m]
template <typename T>
__global__ void k_flip_compat(typename Amp<T>::type *vec,
                              const typename Amp<T>::type *old, uint64_t m) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    typename Amp<T>::type v = old[m];
    v.x = -v.x;
    v.y = -v.y;
    vec[m] = v;
  }
}

// mean = sum a; if |mean| > 1e-10 then mean /= |mean|; out = 2*mean
__global__ __launch_bounds__(kThreads) void k_cfinal(const double *partial,
                                                     int nb, double *out) {
  __shared__ double lds[kThreads / 64];
  double sr = 0.0, si = 0.0;
  for (int b = threadIdx.x; b < nb; b += kThreads) {
    sr += partial[b * kRedSlots + 0];
    si += partial[b * kRedSlots + 1];
  }
  sr = block_sum(sr, lds);
  si = block_sum(si, lds);
  if (threadIdx.x == 0) {
    const double mag = sqrt(sr * sr + si * si);
    if (mag > 1e-10) {
      sr /= mag;
      si /= mag;
    }
    out[0] = 2.0 * sr;
    out[1] = 2.0 * si;
  }
}

// vector[i] = two_mean - scratch[i]
template <typename T>
__global__ __launch_bounds__(kThreads) void k_cdiff(
    const typename Amp<T>::type *old, typename Amp<T>::type *vec, uint64_t n,
    const double *two_mean) {
  const double tr = two_mean[0], ti = two_mean[1];
  const uint64_t stride = uint64_t(gridDim.x) * kThreads;
  for (uint64_t i = uint64_t(blockIdx.x) * kThreads + threadIdx.x; i < n;
       i += stride) {
    const typename Amp<T>::type v = old[i];
    typename Amp<T>::type o;
    o.x = T(tr - double(v.x));
    o.y = T(ti - double(v.y));
    vec[i] = o;
  }
}

// a[m] = -a[m]  (textbook oracle, one amplitude)
template <typename T>
__global__ void k_negate(typename Amp<T>::type *a, uint64_t m) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    typename Amp<T>::type v = a[m];
    v.x = -v.x;
    v.y = -v.y;
    a[m] = v;
  }
}

// ---- comparison --------------------------------------------------------------

template <typename TA, typename TB>
__global__ __launch_bounds__(kThreads) void k_cmp_partial(
    const typename Amp<TA>::type *a, const typename Amp<TB>::type *b,
    uint64_t n, double *partial) {
  __shared__ double lds[kThreads / 64];
  __shared__ double lmax[kThreads];
  const uint64_t stride = uint64_t(gridDim.x) * kThreads;
  double dr = 0.0, di = 0.0, na = 0.0, nb = 0.0, mx = 0.0;
  for (uint64_t i = uint64_t(blockIdx.x) * kThreads + threadIdx.x; i < n;
       i += stride) {
    const double ar = a[i].x, ai = a[i].y, br = b[i].x, bi = b[i].y;
    dr += ar * br + ai * bi;  // conj(a) * b
    di += ar * bi - ai * br;
    na += ar * ar + ai * ai;
    nb += br * br + bi * bi;
    const double ex = ar - br, ey = ai - bi;
    const double e = sqrt(ex * ex + ey * ey);
    mx = e > mx ? e : mx;
  }
  dr = block_sum(dr, lds);
  di = block_sum(di, lds);
  na = block_sum(na, lds);
  nb = block_sum(nb, lds);
  lmax[threadIdx.x] = mx;
  __syncthreads();
  for (int w = kThreads / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) lmax[threadIdx.x] = fmax(lmax[threadIdx.x], lmax[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    double *o = partial + blockIdx.x * kRedSlots;
    o[0] = dr;
    o[1] = di;
    o[2] = na;
    o[3] = nb;
    o[4] = lmax[0];
  }
}

// ---- host launchers ----------------------------------------------------------------

static double *result_slot(qcs_hip_state *s) {
  return s->red + size_t(kRedBlocks) * kRedSlots;
}

// copy `count` doubles from the device result slots to the pinned buffer and
// wait for the stream
static int fetch_results(qcs_hip_state *s, int count) {
  QCS_HIP_TRY(hipMemcpyAsync(s->host, result_slot(s), sizeof(double) * count,
                             hipMemcpyDeviceToHost, s->stream));
  QCS_HIP_TRY(hipStreamSynchronize(s->stream));
  return 0;
}

static unsigned stream_grid(uint64_t n) {
  const uint64_t b = ceil_div(n, kThreads);
  return unsigned(b < 8192 ? b : 8192);
}

// element-wise sweeps: one amplitude per thread over XCD-ordered virtual
// blocks, up to 2^20 work-groups (the gate kernels' launch shape)
static unsigned elem_grid(uint64_t n) {
  const uint64_t b = ceil_div(n, kThreads), cap = uint64_t(1) << 20;
  return unsigned(b < cap ? b : cap);
}

template <typename T>
static int norm_partials(qcs_hip_state *s, int q, unsigned nb) {
  typedef typename Amp<T>::type A;
  TimedLaunch tl;
  timing_begin(s, QCS_HIP_K_REDUCE, double(s->size) * sizeof(A), 3.0 * s->size,
               &tl);
  hipLaunchKernelGGL(k_norm_partial<T>, dim3(nb), dim3(kThreads), 0, s->stream,
                     static_cast<const A *>(s->vec), s->size, q, s->red);
  int rc = launch_check("k_norm_partial");
  if (rc) return rc;
  return timing_end(s, &tl);
}

static int fold(qcs_hip_state *s, unsigned nb, int nslots, unsigned max_mask) {
  hipLaunchKernelGGL(k_final, dim3(1), dim3(kThreads), 0, s->stream, s->red,
                     int(nb), nslots, max_mask, result_slot(s));
  return launch_check("k_final");
}

int reduce_norm(qcs_hip_state *s, double *out_host) {
  const unsigned nb = red_blocks(s->size);
  int rc = s->precision == QCS_HIP_C128 ? norm_partials<double>(s, -1, nb)
                                        : norm_partials<float>(s, -1, nb);
  if (rc) return rc;
  if ((rc = fold(s, nb, 1, 0u))) return rc;
  if ((rc = fetch_results(s, 1))) return rc;
  *out_host = s->host[0];
  return 0;
}

template <typename T>
static int scale_impl(qcs_hip_state *s, double f, const double *dev_ns) {
  typedef typename Amp<T>::type A;
  TimedLaunch tl;
  timing_begin(s, QCS_HIP_K_OTHER, 2.0 * double(s->size) * sizeof(A),
               2.0 * s->size, &tl);
  if (dev_ns)
    hipLaunchKernelGGL(k_scale_dev<T>, dim3(elem_grid(s->size)),
                       dim3(kThreads), 0, s->stream, static_cast<A *>(s->vec),
                       s->size, dev_ns);
  else
    hipLaunchKernelGGL(k_scale<T>, dim3(elem_grid(s->size)), dim3(kThreads),
                       0, s->stream, static_cast<A *>(s->vec), s->size, f);
  int rc = launch_check("k_scale");
  if (rc) return rc;
  return timing_end(s, &tl);
}

int scale_state(qcs_hip_state *s, double f) {
  return s->precision == QCS_HIP_C128 ? scale_impl<double>(s, f, nullptr)
                                      : scale_impl<float>(s, f, nullptr);
}

int normalize_device(qcs_hip_state *s) {
  const unsigned nb = red_blocks(s->size);
  int rc = s->precision == QCS_HIP_C128 ? norm_partials<double>(s, -1, nb)
                                        : norm_partials<float>(s, -1, nb);
  if (rc) return rc;
  if ((rc = fold(s, nb, 1, 0u))) return rc;
  return s->precision == QCS_HIP_C128
             ? scale_impl<double>(s, 1.0, result_slot(s))
             : scale_impl<float>(s, 1.0, result_slot(s));
}

int fold_norm_partials(qcs_hip_state *s, int nb, const double **ns_dev) {
  *ns_dev = result_slot(s);
  return fold(s, unsigned(nb), 1, 0u);
}

int normalize_from_partials(qcs_hip_state *s, int nb) {
  int rc;
  if ((rc = fold(s, unsigned(nb), 1, 0u))) return rc;
  return s->precision == QCS_HIP_C128
             ? scale_impl<double>(s, 1.0, result_slot(s))
             : scale_impl<float>(s, 1.0, result_slot(s));
}

int qubit_probs(qcs_hip_state *s, int q, double *p0, double *p1) {
  const unsigned nb = red_blocks(s->size);
  int rc = s->precision == QCS_HIP_C128 ? norm_partials<double>(s, q, nb)
                                        : norm_partials<float>(s, q, nb);
  if (rc) return rc;
  if ((rc = fold(s, nb, 2, 0u))) return rc;
  if ((rc = fetch_results(s, 2))) return rc;
  *p0 = s->host[0];
  *p1 = s->host[1];
  return 0;
}

template <typename T>
static int half_partials(qcs_hip_state *s, int q, int bit, unsigned nb) {
  typedef typename Amp<T>::type A;
  const uint64_t nh = s->size / 2;
  TimedLaunch tl;
  timing_begin(s, QCS_HIP_K_REDUCE, double(nh) * sizeof(A), 3.0 * double(nh), &tl);
  hipLaunchKernelGGL(k_half_norm_partial<T>, dim3(nb), dim3(kThreads), 0, s->stream,
                     static_cast<const A *>(s->vec), nh, q,
                     bit ? (uint64_t(1) << q) : uint64_t(0), s->red);
  int rc = launch_check("k_half_norm_partial");
  if (rc) return rc;
  return timing_end(s, &tl);
}

bool half_prob_pays(const qcs_hip_state *s, int q) {
  return (size_t(1) << q) * size_t(s->amp_bytes) >= 128;
}

int half_prob(qcs_hip_state *s, int q, int bit, double *p) {
  const unsigned nb = red_blocks(s->size / 2);
  int rc = s->precision == QCS_HIP_C128 ? half_partials<double>(s, q, bit, nb)
                                        : half_partials<float>(s, q, bit, nb);
  if (rc) return rc;
  if ((rc = fold(s, nb, 1, 0u))) return rc;
  if ((rc = fetch_results(s, 1))) return rc;
  *p = s->host[0];
  return 0;
}

template <typename T>
static int collapse_impl(qcs_hip_state *s, int q, int outcome, double f,
                         int do_scale) {
  typedef typename Amp<T>::type A;
  TimedLaunch tl;
  timing_begin(s, QCS_HIP_K_OTHER, 1.5 * double(s->size) * sizeof(A), 0.0, &tl);
  hipLaunchKernelGGL(k_collapse<T>, dim3(elem_grid(s->size)), dim3(kThreads),
                     0, s->stream, static_cast<A *>(s->vec), s->size, q,
                     outcome, f, do_scale);
  int rc = launch_check("k_collapse");
  if (rc) return rc;
  return timing_end(s, &tl);
}

int collapse(qcs_hip_state *s, int q, int outcome, double f, int do_scale) {
  return s->precision == QCS_HIP_C128
             ? collapse_impl<double>(s, q, outcome, f, do_scale)
             : collapse_impl<float>(s, q, outcome, f, do_scale);
}

// Measurements of `count` qubits in order, with no host round trip between
// them: per qubit the p0 / p1 reductions qcs_hip_measure uses (the half
// passes, or one pass for both where the halves' runs are shorter than a
// line; here p1 is always formed, as the device decides the outcome),
// k_measure_decide, and the collapse reading its decision.  Result slots:
// 8..12 the current measurement, 16.. the outcomes.
template <typename T>
static int measure_seq_impl(qcs_hip_state *s, int count, const int *qubits,
                            const double *u, int *outcomes) {
  typedef typename Amp<T>::type A;
  double *m = result_slot(s) + 8, *rec = result_slot(s) + 16;
  constexpr int kMaxRec = 48;
  int rc;
  for (int i0 = 0; i0 < count; i0 += kMaxRec) {
    const int c = std::min(kMaxRec, count - i0);
    for (int i = 0; i < c; ++i) {
      const int q = qubits[i0 + i];
      if (half_prob_pays(s, q)) {
        const unsigned nb = red_blocks(s->size / 2);
        for (int bit = 0; bit < 2; ++bit) {
          if ((rc = half_partials<T>(s, q, bit, nb))) return rc;
          hipLaunchKernelGGL(k_final, dim3(1), dim3(kThreads), 0, s->stream, s->red,
                             int(nb), 1, 0u, m + bit);
          if ((rc = launch_check("k_final"))) return rc;
        }
      } else {
        const unsigned nb = red_blocks(s->size);
        if ((rc = norm_partials<T>(s, q, nb))) return rc;
        hipLaunchKernelGGL(k_final, dim3(1), dim3(kThreads), 0, s->stream, s->red,
                           int(nb), 2, 0u, m);
        if ((rc = launch_check("k_final"))) return rc;
      }
      hipLaunchKernelGGL(k_measure_decide, dim3(1), dim3(64), 0, s->stream, m,
                         u[i0 + i], rec + i);
      if ((rc = launch_check("k_measure_decide"))) return rc;
      TimedLaunch tl;
      timing_begin(s, QCS_HIP_K_OTHER, 1.5 * double(s->size) * sizeof(A), 0.0, &tl);
      hipLaunchKernelGGL(k_collapse_dev<T>, dim3(elem_grid(s->size)), dim3(kThreads), 0,
                         s->stream, static_cast<A *>(s->vec), s->size, q, m);
      if ((rc = launch_check("k_collapse_dev"))) return rc;
      if ((rc = timing_end(s, &tl))) return rc;
    }
    QCS_HIP_TRY(hipMemcpyAsync(s->host, rec, sizeof(double) * size_t(c),
                               hipMemcpyDeviceToHost, s->stream));
    QCS_HIP_TRY(hipStreamSynchronize(s->stream));
    for (int i = 0; i < c; ++i) outcomes[i0 + i] = int(s->host[i]);
  }
  return 0;
}

// Qubits 0 .. count - 1 in order.  *done = 0 when the workspace cannot be
// had; nothing has been launched then.
static int measure_low(qcs_hip_state *s, int count, const double *u, int *outcomes, bool *done) {
  double2 *a = static_cast<double2 *>(s->vec);
  // four rows a work-group at least, so that the partials stay a small part
  // of what is read
  auto blocks = [](uint64_t rows) {
    const uint64_t b = rows / 4;
    return unsigned(b < 1 ? 1 : b < uint64_t(kMargBlocks) ? b : kMargBlocks);
  };
  const uint64_t rows0 = s->n > kMargBits ? s->size >> kMargBits : 1;
  const size_t nparts = size_t(blocks(rows0)) * kMargSize;
  *done = false;
  if (!s->marg) {
    const size_t bytes = (nparts + kMargSize) * sizeof(double) + sizeof(MargState);
    if (hipMalloc(&s->marg, bytes) != hipSuccess) {
      (void)hipGetLastError();  // not an error of a later launch
      s->marg = nullptr;
      return 0;
    }
  }
  int rc;
  if ((rc = ensure_pinned(s, 4096))) return rc;
  *done = true;
  double *partial = s->marg, *w = partial + nparts;
  MargState *ms = reinterpret_cast<MargState *>(w + kMargSize);
  TimedLaunch tl;
  for (int shift = 0; shift < count; shift += kMargBits) {
    const int lb = std::min(kMargBits, s->n - shift);
    const uint64_t rows = lb == kMargBits ? s->size >> (shift + lb) : 1;
    const unsigned nb = blocks(rows);
    const double amps = double(s->size >> shift);
    timing_begin(s, QCS_HIP_K_REDUCE, amps * sizeof(double2), 3.0 * amps, &tl);
    hipLaunchKernelGGL(k_marg_partial, dim3(nb), dim3(kThreads), 0, s->stream, a, rows, lb,
                       shift, ms, partial);
    if ((rc = launch_check("k_marg_partial")) || (rc = timing_end(s, &tl))) return rc;
    if (nb > 1) {
      hipLaunchKernelGGL(k_marg_fold, dim3(kMargSize / 64), dim3(kThreads), 0, s->stream,
                         partial, int(nb), w);
      if ((rc = launch_check("k_marg_fold"))) return rc;
    }
    MargUniforms un;
    const int c = std::min(count - shift, lb);
    for (int b = 0; b < kMargBits; ++b) un.u[b] = b < c ? u[shift + b] : 0.0;
    hipLaunchKernelGGL(k_marg_decide, dim3(1), dim3(kThreads), 0, s->stream,
                       nb > 1 ? w : partial, lb, shift, c, un, ms);
    if ((rc = launch_check("k_marg_decide"))) return rc;
  }
  timing_begin(s, QCS_HIP_K_OTHER, double(s->size) * sizeof(double2), 0.0, &tl);
  hipLaunchKernelGGL(k_marg_collapse, dim3(elem_grid(s->size)), dim3(kThreads), 0, s->stream,
                     a, s->size, count, ms);
  if ((rc = launch_check("k_marg_collapse")) || (rc = timing_end(s, &tl))) return rc;
  QCS_HIP_TRY(hipMemcpyAsync(s->host, ms->outcome, sizeof(double) * size_t(count),
                             hipMemcpyDeviceToHost, s->stream));
  QCS_HIP_TRY(hipStreamSynchronize(s->stream));
  for (int i = 0; i < count; ++i) outcomes[i] = int(s->host[i]);
  return 0;
}

int measure_seq(qcs_hip_state *s, int count, const int *qubits, const double *u,
                int *outcomes) {
  // qubits 0, 1, ... (qc_measure_all): weights instead of a sweep per qubit.
  // Other lists, and a single qubit, are measured one by one; so are
  // complex64 states, where each collapse rounds the amplitudes that the next
  // probability is a sum of.
  bool low = s->precision == QCS_HIP_C128 && count >= 2 && count <= s->n;
  for (int i = 0; low && i < count; ++i) low = qubits[i] == i;
  if (low) {
    bool done = false;
    const int rc = measure_low(s, count, u, outcomes, &done);
    if (rc || done) return rc;
  }
  return s->precision == QCS_HIP_C128
             ? measure_seq_impl<double>(s, count, qubits, u, outcomes)
             : measure_seq_impl<float>(s, count, qubits, u, outcomes);
}

template <typename T>
static int argmax_impl(qcs_hip_state *s, long *idx) {
  typedef typename Amp<T>::type A;
  const unsigned nb = red_blocks(s->size);
  TimedLaunch tl;
  timing_begin(s, QCS_HIP_K_REDUCE, double(s->size) * sizeof(A), 3.0 * s->size,
               &tl);
  hipLaunchKernelGGL(k_argmax_partial<T>, dim3(nb), dim3(kThreads), 0,
                     s->stream, static_cast<const A *>(s->vec), s->size, s->red);
  int rc = launch_check("k_argmax_partial");
  if (rc) return rc;
  if ((rc = timing_end(s, &tl))) return rc;
  hipLaunchKernelGGL(k_argmax_final, dim3(1), dim3(kThreads), 0, s->stream,
                     s->red, int(nb), result_slot(s));
  if ((rc = launch_check("k_argmax_final"))) return rc;
  if ((rc = fetch_results(s, 2))) return rc;
  long long bits;
  static_assert(sizeof(bits) == sizeof(double), "double is 64-bit");
  __builtin_memcpy(&bits, &s->host[1], sizeof(bits));
  *idx = (s->host[0] > 0.0) ? long(bits) : 0;
  return 0;
}

int argmax(qcs_hip_state *s, long *idx) {
  return s->precision == QCS_HIP_C128 ? argmax_impl<double>(s, idx)
                                      : argmax_impl<float>(s, idx);
}

template <typename T>
static int launch_sample(qcs_hip_state *s, uint64_t nchunks, uint64_t len, const double *excl,
                         const double *inc, long shots, const double *u, long *out) {
  const auto *a = static_cast<const typename Amp<T>::type *>(s->vec);
  if (shots <= 0) return 0;
  if (shots <= kWideShots) {
    hipLaunchKernelGGL(k_sample_wide<T>, dim3(unsigned(shots)), dim3(kThreads), 0, s->stream, a,
                       nchunks, len, excl, inc, u, out);
    return launch_check("k_sample_wide");
  }
  // one wave per shot; at most 2^24 shots per dispatch keeps the
  // work-item count below 2^32
  for (uint64_t s0 = 0; s0 < uint64_t(shots); s0 += uint64_t(1) << 24) {
    const uint64_t ns = std::min<uint64_t>(uint64_t(shots) - s0, uint64_t(1) << 24);
    hipLaunchKernelGGL(k_sample<T>, dim3(unsigned(ceil_div(ns, kThreads / 64))),
                       dim3(kThreads), 0, s->stream, a, nchunks, len, excl, inc, u + s0, ns,
                       out + s0);
    const int rc = launch_check("k_sample");
    if (rc) return rc;
  }
  return 0;
}

template <typename T>
static int sample_impl(qcs_hip_state *s, long shots, const double *u,
                       long *out) {
  typedef typename Amp<T>::type A;
  const uint64_t len = s->size < uint64_t(kChunk) ? s->size : uint64_t(kChunk);
  const uint64_t nchunks = s->size / len;
  if (s->chunk_cap < nchunks) {
    if (s->chunk_tot) (void)hipFree(s->chunk_tot);
    if (s->chunk_inc) (void)hipFree(s->chunk_inc);
    s->chunk_tot = s->chunk_inc = nullptr;
    s->chunk_cap = 0;
    QCS_HIP_TRY(hipMalloc(&s->chunk_tot, nchunks * sizeof(double)));
    QCS_HIP_TRY(hipMalloc(&s->chunk_inc, nchunks * sizeof(double)));
    s->chunk_cap = nchunks;
  }
  if (s->shots_cap < size_t(shots)) {
    if (s->u_dev) (void)hipFree(s->u_dev);
    if (s->idx_dev) (void)hipFree(s->idx_dev);
    s->u_dev = nullptr;
    s->idx_dev = nullptr;
    s->shots_cap = 0;
    QCS_HIP_TRY(hipMalloc(&s->u_dev, size_t(shots) * sizeof(double)));
    QCS_HIP_TRY(hipMalloc(&s->idx_dev, size_t(shots) * sizeof(long)));
    s->shots_cap = size_t(shots);
  }
  QCS_HIP_TRY(hipMemcpyAsync(s->u_dev, u, size_t(shots) * sizeof(double),
                             hipMemcpyHostToDevice, s->stream));
  const A *a = static_cast<const A *>(s->vec);
  TimedLaunch tl;
  timing_begin(s, QCS_HIP_K_REDUCE, double(s->size) * sizeof(A), 3.0 * s->size,
               &tl);
  hipLaunchKernelGGL(k_chunk_tot<T>, dim3(unsigned(nchunks)), dim3(kThreads), 0, s->stream, a,
                     len, s->chunk_tot);
  int rc = launch_check("k_chunk_tot");
  if (rc) return rc;
  if ((rc = timing_end(s, &tl))) return rc;
  hipLaunchKernelGGL(k_chunk_scan, dim3(1), dim3(1024), 0, s->stream,
                     s->chunk_tot, s->chunk_inc, nchunks);
  if ((rc = launch_check("k_chunk_scan"))) return rc;
  timing_begin(s, QCS_HIP_K_OTHER, double(shots) * len * sizeof(A), 0.0, &tl);
  if ((rc = launch_sample<T>(s, nchunks, len, s->chunk_tot, s->chunk_inc, shots, s->u_dev,
                             s->idx_dev)))
    return rc;
  if ((rc = timing_end(s, &tl))) return rc;
  QCS_HIP_TRY(hipMemcpyAsync(out, s->idx_dev, size_t(shots) * sizeof(long),
                             hipMemcpyDeviceToHost, s->stream));
  QCS_HIP_TRY(hipStreamSynchronize(s->stream));
  return 0;
}

int sample(qcs_hip_state *s, long shots, const double *u, long *out) {
  return s->precision == QCS_HIP_C128 ? sample_impl<double>(s, shots, u, out)
                                      : sample_impl<float>(s, shots, u, out);
}

// ---- sampling with no allocation ---------------------------------------------
//
// qcs_hip_sample_noalloc keeps the chunk totals (tot) and inclusive prefixes
// (inc) in one file-scope device array per GPU instead of buffers grown per
// state.  Its device address is looked up once per device with that device
// current; host code passes that address to the kernels, never the array's
// name (in host code the name is a host-side stand-in).  Every entry
// [0, nchunks) of both halves is written by k_chunk_tot / k_chunk_scan before
// any kernel reads it, so nothing needs clearing between calls.
constexpr uint64_t kNoAllocChunks = uint64_t(1) << (QCS_HIP_NOALLOC_MAX_QUBITS - 12);
static_assert(kChunk == 4096, "kNoAllocChunks assumes 4096-amplitude chunks");
static __device__ __align__(256) double scratch[2 * kNoAllocChunks];

constexpr int kMaxDevices = 64;
static std::once_flag g_scratch_once[kMaxDevices];
static double *g_scratch_ptr[kMaxDevices];
static hipError_t g_scratch_err[kMaxDevices];

static int noalloc_scratch(int device, double **out) {
  if (device < 0 || device >= kMaxDevices)
    return fail(QCS_HIP_EUNSUP, "sample_noalloc: device %d beyond %d", device, kMaxDevices);
  std::call_once(g_scratch_once[device], [device] {
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e == hipSuccess && cur != device) e = hipSetDevice(device);
    void *p = nullptr;
    if (e == hipSuccess) e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != device) (void)hipSetDevice(cur);
    g_scratch_err[device] = e;
    g_scratch_ptr[device] = e == hipSuccess ? static_cast<double *>(p) : nullptr;
  });
  if (g_scratch_err[device] != hipSuccess)
    return check_hip(g_scratch_err[device], "hipGetSymbolAddress(scratch)");
  *out = g_scratch_ptr[device];
  return 0;
}

template <typename T>
static int sample_noalloc_impl(qcs_hip_state *s, double *scr, long shots,
                               const double *u_dev, long *idx_dev) {
  typedef typename Amp<T>::type A;
  const uint64_t len = s->size < uint64_t(kChunk) ? s->size : uint64_t(kChunk);
  const uint64_t nchunks = s->size / len;
  double *tot = scr, *inc = scr + kNoAllocChunks;
  const A *a = static_cast<const A *>(s->vec);
  hipLaunchKernelGGL(k_chunk_tot<T>, dim3(unsigned(nchunks)), dim3(kThreads), 0, s->stream, a,
                     len, tot);
  int rc = launch_check("k_chunk_tot");
  if (rc) return rc;
  hipLaunchKernelGGL(k_chunk_scan, dim3(1), dim3(1024), 0, s->stream, tot, inc, nchunks);
  if ((rc = launch_check("k_chunk_scan"))) return rc;
  return launch_sample<T>(s, nchunks, len, tot, inc, shots, u_dev, idx_dev);
}

int sample_noalloc(qcs_hip_state *s, long shots, const double *u_dev, long *idx_dev) {
  if (s->n > QCS_HIP_NOALLOC_MAX_QUBITS)
    return fail(QCS_HIP_EINVAL,
                "sample_noalloc: %d qubits exceed the scratch array's %d (%llu chunk sums)",
                s->n, QCS_HIP_NOALLOC_MAX_QUBITS, (unsigned long long)kNoAllocChunks);
  double *scr = nullptr;
  int rc = noalloc_scratch(s->device, &scr);
  if (rc) return rc;
  return s->precision == QCS_HIP_C128
             ? sample_noalloc_impl<double>(s, scr, shots, u_dev, idx_dev)
             : sample_noalloc_impl<float>(s, scr, shots, u_dev, idx_dev);
}

template <typename T>
static int grover_impl(qcs_hip_state *s, long marked, long iters) {
  typedef typename Amp<T>::type A;
  A *a = static_cast<A *>(s->vec);
  const unsigned nb = red_blocks(s->size);
  const uint64_t m = marked < 0 ? ~uint64_t(0) : uint64_t(marked);
  TimedLaunch tl;
  timing_begin(s, QCS_HIP_K_REDUCE, double(s->size) * sizeof(A), 2.0 * s->size,
               &tl);
  hipLaunchKernelGGL(k_gsum_partial<T>, dim3(nb), dim3(kThreads), 0, s->stream,
                     a, s->size, m, s->red);
  int rc = launch_check("k_gsum_partial");
  if (rc) return rc;
  if ((rc = timing_end(s, &tl))) return rc;
  hipLaunchKernelGGL(k_grounds<T>, dim3(1), dim3(kThreads), 0, s->stream, a, s->size, m, s->red,
                     int(nb), iters, result_slot(s));
  if ((rc = launch_check("k_grounds"))) return rc;
  timing_begin(s, QCS_HIP_K_OTHER, 2.0 * double(s->size) * sizeof(A), 2.0 * s->size, &tl);
  hipLaunchKernelGGL(k_gapply<T>, dim3(elem_grid(s->size)), dim3(kThreads), 0, s->stream, a,
                     s->size, m, result_slot(s));
  if ((rc = launch_check("k_gapply"))) return rc;
  return timing_end(s, &tl);
}

int grover_textbook(qcs_hip_state *s, long marked, long iters) {
  return s->precision == QCS_HIP_C128 ? grover_impl<double>(s, marked, iters)
                                      : grover_impl<float>(s, marked, iters);
}

template <typename T>
static int flip_compat_impl(qcs_hip_state *s, long index) {
  typedef typename Amp<T>::type A;
  void *t = s->vec;  // src/q_gates.c:311-316
  s->vec = s->scratch;
  s->scratch = t;
  hipLaunchKernelGGL(k_flip_compat<T>, dim3(1), dim3(64), 0, s->stream,
                     static_cast<A *>(s->vec), static_cast<const A *>(s->scratch),
                     uint64_t(index));
  return launch_check("k_flip_compat");
}

int phase_flip_compat(qcs_hip_state *s, long index) {
  return s->precision == QCS_HIP_C128 ? flip_compat_impl<double>(s, index)
                                      : flip_compat_impl<float>(s, index);
}

template <typename T>
static int diffusion_compat_impl(qcs_hip_state *s) {
  typedef typename Amp<T>::type A;
  const unsigned nb = red_blocks(s->size);
  hipLaunchKernelGGL(k_gsum_partial<T>, dim3(nb), dim3(kThreads), 0, s->stream,
                     static_cast<const A *>(s->vec), s->size, ~uint64_t(0),
                     s->red);
  int rc = launch_check("k_gsum_partial");
  if (rc) return rc;
  double *two_mean = result_slot(s);
  hipLaunchKernelGGL(k_cfinal, dim3(1), dim3(kThreads), 0, s->stream, s->red,
                     int(nb), two_mean);
  if ((rc = launch_check("k_cfinal"))) return rc;
  void *t = s->vec;  // src/q_gates.c:346-348
  s->vec = s->scratch;
  s->scratch = t;
  hipLaunchKernelGGL(k_cdiff<T>, dim3(stream_grid(s->size)), dim3(kThreads), 0,
                     s->stream, static_cast<const A *>(s->scratch),
                     static_cast<A *>(s->vec), s->size, two_mean);
  return launch_check("k_cdiff");
}

int diffusion_compat(qcs_hip_state *s) {
  return s->precision == QCS_HIP_C128 ? diffusion_compat_impl<double>(s)
                                      : diffusion_compat_impl<float>(s);
}

int negate_one(qcs_hip_state *s, long index) {
  if (s->precision == QCS_HIP_C128)
    hipLaunchKernelGGL(k_negate<double>, dim3(1), dim3(64), 0, s->stream,
                       static_cast<double2 *>(s->vec), uint64_t(index));
  else
    hipLaunchKernelGGL(k_negate<float>, dim3(1), dim3(64), 0, s->stream,
                       static_cast<float2 *>(s->vec), uint64_t(index));
  return launch_check("k_negate");
}

template <typename TA, typename TB>
static int cmp_impl(qcs_hip_state *a, qcs_hip_state *b, unsigned nb) {
  typedef typename Amp<TA>::type AA;
  typedef typename Amp<TB>::type AB;
  hipLaunchKernelGGL((k_cmp_partial<TA, TB>), dim3(nb), dim3(kThreads), 0,
                     a->stream, static_cast<const AA *>(a->vec),
                     static_cast<const AB *>(b->vec), a->size, a->red);
  return launch_check("k_cmp_partial");
}

int compare(qcs_hip_state *a, qcs_hip_state *b, double *omf, double *maxabs) {
  // order b's pending work before a's stream reads it
  QCS_HIP_TRY(hipStreamSynchronize(b->stream));
  const unsigned nb = red_blocks(a->size);
  int rc;
  const bool a64 = a->precision == QCS_HIP_C128, b64 = b->precision == QCS_HIP_C128;
  if (a64 && b64) rc = cmp_impl<double, double>(a, b, nb);
  else if (a64) rc = cmp_impl<double, float>(a, b, nb);
  else if (b64) rc = cmp_impl<float, double>(a, b, nb);
  else rc = cmp_impl<float, float>(a, b, nb);
  if (rc) return rc;
  if ((rc = fold(a, nb, 5, 1u << 4))) return rc;
  if ((rc = fetch_results(a, 5))) return rc;
  const double dr = a->host[0], di = a->host[1], na = a->host[2],
               nbv = a->host[3];
  if (omf) *omf = (na > 0.0 && nbv > 0.0) ? 1.0 - (dr * dr + di * di) / (na * nbv) : 1.0;
  if (maxabs) *maxabs = a->host[4];
  return 0;
}

}  // namespace qcs
