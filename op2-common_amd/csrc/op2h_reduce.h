// Finishing a gbl reduction from per-workgroup partials, shared by the eager
// finish kernels and the graph's history kernel so that both produce the same
// bits.  One group of kRedThreads (4 waves) reduces one gbl:
//   thread t combines partials t, t + 256, t + 512, ... in that order, then a wave tree by xor shuffles,
//   then thread 0 of the group combines its 4 waves in order.
// Kinds: 1 sum of doubles; 2 max and 3 min of (value, loc) pairs, equal
// values keeping the lower loc (the first element reaching the extremum);
// 4 sum of Sum2 pairs.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

namespace op2h_red {

constexpr int kRedThreads = 256;
constexpr int kRedMaxLoads = 16;  // partials per thread (4096 per gbl)

// A sum kept as the unevaluated pair hi + lo: each addition to hi is an
// error-free two-sum (Knuth), its rounding error gathered in lo, so the pair
// holds the sum to about 2^-100 and its rounded value is the same whatever the
// order of the terms (the chance that 2^-85 of it straddles a rounding
// boundary aside).  Loops may therefore cut a reduction into any partials:
// eager chunks, fused patches and ensemble tiles give one result.
struct Sum2 {
  double hi, lo;
};

__device__ __forceinline__ void sum2_add(Sum2 &s, double v) {
  const double t = s.hi + v, z = t - s.hi;
  s.lo += (s.hi - (t - z)) + (v - z);
  s.hi = t;
}

__device__ __forceinline__ Sum2 sum2_join(Sum2 a, Sum2 b) {
  sum2_add(a, b.hi);
  a.lo += b.lo;
  return a;
}

// The rounded sum; an infinite or NaN hi stands (its lo is then NaN).
__device__ __forceinline__ double sum2_value(Sum2 s) {
  return isfinite(s.hi) ? s.hi + s.lo : s.hi;
}

struct ValLoc {
  double v;
  int loc;
  double lo;  // kind 4
};

__device__ __forceinline__ ValLoc combine(ValLoc a, ValLoc b, int kind) {
  if (kind == 1) return ValLoc{a.v + b.v, 0, 0.0};
  if (kind == 4) {
    const Sum2 s = sum2_join(Sum2{a.v, a.lo}, Sum2{b.v, b.lo});
    return ValLoc{s.hi, 0, s.lo};
  }
  const bool better = kind == 2 ? b.v > a.v : b.v < a.v;
  if (better || (b.v == a.v && b.loc < a.loc)) return b;
  return a;
}

__device__ __forceinline__ ValLoc identity(int kind) {
  return ValLoc{kind == 2 ? -INFINITY : kind == 3 ? INFINITY : 0.0, 0x7fffffff, 0.0};
}

// This thread's partials t, t + 256, ... (at most LOADS of them), all loads
// issued before the first is combined.
template <int LOADS>
__device__ __forceinline__ ValLoc thread_reduce(const double *vals, const int *locs,
                                                const double *lows, int n, int kind, int t) {
  ValLoc m = identity(kind);
  double v[LOADS], lo[LOADS];
  int l[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int p = t + i * kRedThreads;
    v[i] = p < n ? vals[p] : identity(kind).v;
    l[i] = (locs && p < n) ? locs[p] : 0x7fffffff;
    lo[i] = (lows && p < n) ? lows[p] : 0.0;
  }
#pragma unroll
  for (int i = 0; i < LOADS; ++i) m = combine(m, ValLoc{v[i], l[i], lo[i]}, kind);
  return m;
}

// Reduces `n` partials (vals; locs for kinds 2/3, lows for kind 4) with the
// group whose threads have local index `t` (0..kRedThreads-1) and wave slots
// s_v/s_l/s_lo [4] in LDS.  All threads of the group must call it; the result
// is returned to t == 0 (kind 4: the rounded sum in v).  The caller
// synchronises the workgroup between uses of the slots.  Up to 1024 partials
// (the eager update's 938 at 720,000 cells) go by the chain of 4 combines per
// thread that they need: the one of 16 took the finish 0.7 us longer.
__device__ __forceinline__ ValLoc group_reduce(const double *vals, const int *locs,
                                               const double *lows, int n, int kind, int t,
                                               double *s_v, int *s_l, double *s_lo) {
  ValLoc m = n <= 4 * kRedThreads ? thread_reduce<4>(vals, locs, lows, n, kind, t)
                                  : thread_reduce<kRedMaxLoads>(vals, locs, lows, n, kind, t);
  for (int o = 32; o > 0; o >>= 1) {
    ValLoc x{__shfl_xor(m.v, o, 64), __shfl_xor(m.loc, o, 64), __shfl_xor(m.lo, o, 64)};
    m = combine(m, x, kind);
  }
  const int lane = t & 63, wave = t >> 6;
  if (lane == 0) {
    s_v[wave] = m.v;
    s_l[wave] = m.loc;
    s_lo[wave] = m.lo;
  }
  __syncthreads();
  ValLoc r = identity(kind);
  if (t == 0) {
    for (int w = 0; w < kRedThreads / 64; ++w)
      r = combine(r, ValLoc{s_v[w], s_l[w], s_lo[w]}, kind);
    if (kind == 4) r.v = sum2_value(Sum2{r.v, r.lo});
  }
  return r;
}

// ---- the update's reductions, rms (INC) and maxerr (MAX) with errloc ----
struct MaxLoc {
  double v;
  int loc;
};

__device__ __forceinline__ MaxLoc maxloc_combine(MaxLoc a, MaxLoc b) {
  // larger value wins; equal values keep the lower element index, so the
  // result is the first element in set order reaching the maximum
  if (b.v > a.v || (b.v == a.v && b.loc < a.loc)) return b;
  return a;
}

// A thread's, wave's or workgroup's share: each cell's own sum (its four
// squares in component order) added to the pair.
struct UpdateAcc {
  Sum2 rms{0.0, 0.0};
  MaxLoc ml{-INFINITY, 0x7fffffff};
};

// One cell's share, its sum and its own maximum `mx` (-infinity where it has
// none, every change being NaN): joined as any other maximum, because the cells
// a thread takes need not come in index order (a thread's running maximum would
// keep the first it visits of two equal ones).
__device__ __forceinline__ void add_cell(UpdateAcc &a, double sum, double mx, int idx) {
  sum2_add(a.rms, sum);
  a.ml = maxloc_combine(a.ml, MaxLoc{mx, mx > -INFINITY ? idx : 0x7fffffff});
}

__device__ __forceinline__ void wave_join(UpdateAcc &a) {
  for (int o = 32; o > 0; o >>= 1) {
    a.rms = sum2_join(a.rms, Sum2{__shfl_xor(a.rms.hi, o, 64), __shfl_xor(a.rms.lo, o, 64)});
    a.ml = maxloc_combine(a.ml, MaxLoc{__shfl_xor(a.ml.v, o, 64), __shfl_xor(a.ml.loc, o, 64)});
  }
}

// Where the workgroups' partials go: one {hi, lo, max, loc} per workgroup.
struct UpdateParts {
  double *hi, *lo, *mx;
  int *loc;
};

// The workgroup's partial from its threads' shares, written at `L` by thread
// 0.  Every thread of the workgroup (at most 16 waves) calls it.
__device__ __forceinline__ void write_partial(UpdateAcc a, const UpdateParts &P, int L) {
  __shared__ double s_hi[16], s_lo[16], s_mx[16];
  __shared__ int s_loc[16];
  wave_join(a);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    s_hi[wave] = a.rms.hi;
    s_lo[wave] = a.rms.lo;
    s_mx[wave] = a.ml.v;
    s_loc[wave] = a.ml.loc;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    UpdateAcc b;
    const int nw = (blockDim.x + 63) >> 6;
    for (int w = 0; w < nw; ++w) {
      b.rms = sum2_join(b.rms, Sum2{s_hi[w], s_lo[w]});
      b.ml = maxloc_combine(b.ml, MaxLoc{s_mx[w], s_loc[w]});
    }
    P.hi[L] = b.rms.hi;
    P.lo[L] = b.rms.lo;
    P.mx[L] = b.ml.v;
    P.loc[L] = b.ml.loc;
  }
}

}  // namespace op2h_red
