// f3d_ringsum.h -- the sequential FP64 sum of a ring, in index order, by one
// wave (all 64 lanes taking part).
//
// The order of the additions fixes the rounding of every ring mean
// (src/reduction_generic.c:15-21), and taken literally it is one chain of
// dependent additions: 4.5 ns each on MI355X with both operands in registers,
// 6 ns per term with the hand-over from lane to lane (literal() below).  Most
// of that chain need not be walked.  While the running sum stays inside one
// binade [2^e, 2^(e+1)) every addition rounds to the same quantum u = 2^(e-52),
// so a run of terms adds a whole number of quanta, which depends on the sum it
// starts from only through that sum's parity (a term that lies halfway between
// two multiples of u goes to the even one).  So, for a chunk of 64 S terms, S
// consecutive ones per lane (chain() below):
//   - a plain prefix sum of the lanes' totals estimates where each lane's sum
//     starts.  The estimate and the literal chain differ by less than 2^-40 of
//     the largest sum in the chunk; a lane is accepted if its start is at least
//     2^-10 of that largest one and if, with a margin of 2^-30, the sum cannot
//     leave the start's binade inside the lane (S times its largest term).
//     Every other lane holds a passage from one binade to the next, or a zero,
//     tiny, infinite or NaN sum, and is added literally;
//   - an accepted lane adds its terms to two stand-ins of its binade, 1.5 2^e
//     and 1.5 2^e + u (one even, one odd), which gives its increment for either
//     parity.  The two differ only if the lane holds a halfway case, and then
//     both end on the same parity, so the parity that enters each lane of a run
//     of accepted lanes of one binade follows from two ballots and the parity
//     that enters the run;
//   - a run's increments are multiples of u below 2^(e+1): exact in any order.
//     One segmented prefix sum gives every run's total for an even sum
//     entering; an odd one changes it only at the run's first halfway case.
// What is left in order is one addition per run and the literal lanes.  The
// sum equals the literal chain bit for bit for any terms.
//
// Measured (one wave per ring, microseconds, literal -> chain): 1024 rings of
// 4096 cells 36.9 -> 11.6 (the loads alone take 8.1), 437 of 1250 10.1 -> 6.6,
// 7150 of 500 16.6 -> 10.3, 128 of 384 4.0 -> 3.7; on 3168 rings of 256 cells
// 6.6 -> 6.4 and on 48 of 96 2.9 -> 3.1, so rings of up to kLiteral terms keep
// the literal chain.  The terms reach the lanes through LDS: loads of S
// consecutive doubles per lane touch 64 cache lines each (37 -> 33 us on 4096
// cells for the literal chain alone).
#pragma once

#include <hip/hip_runtime.h>

namespace f3d_ring {

constexpr int kLiteral = 256;
// doubles of LDS that ordered_sum<S> stages a chunk's terms through: S per
// lane and one of padding, so that the lanes' reads fall into different banks
constexpr int lds_doubles(int S) { return 64 * (S + 1); }

// the value of the lane a DPP control names, +0.0 where there is none
template <int CTRL, int ROWS>
__device__ __forceinline__ double lane_move(double p) {
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(p), CTRL, ROWS, 0xF, false);
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(p), CTRL, ROWS, 0xF, false);
  return __hiloint2double(hi, lo);
}
// inclusive prefix sum over the wave: rows of 16 lanes (row_shr:1, 2, 4, 8),
// row_bcast:15 into rows 1 and 3, row_bcast:31 into rows 2 and 3
__device__ __forceinline__ double wave_prefix(double p) {
  p = p + lane_move<0x111, 0xF>(p);
  p = p + lane_move<0x112, 0xF>(p);
  p = p + lane_move<0x114, 0xF>(p);
  p = p + lane_move<0x118, 0xF>(p);
  p = p + lane_move<0x142, 0xA>(p);
  return p + lane_move<0x143, 0xC>(p);
}
// the same within segments: lane's segment starts at lane `head`
__device__ __forceinline__ double wave_prefix_from(double p, int lane, int head) {
  const int d = lane - head;
  double q = lane_move<0x111, 0xF>(p);
  p = d >= 1 ? p + q : p;
  q = lane_move<0x112, 0xF>(p);
  p = d >= 2 ? p + q : p;
  q = lane_move<0x114, 0xF>(p);
  p = d >= 4 ? p + q : p;
  q = lane_move<0x118, 0xF>(p);
  p = d >= 8 ? p + q : p;
  q = lane_move<0x142, 0xA>(p);
  p = head < (lane & 48) ? p + q : p;
  q = lane_move<0x143, 0xC>(p);
  return head < 32 && lane >= 32 ? p + q : p;
}
template <int CTRL, int ROWS>
__device__ __forceinline__ int lane_max(int v) {
  return max(v, __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false));
}
// the largest v >= 0 of the wave
__device__ __forceinline__ int wave_max_int(int v) {
  v = lane_max<0x111, 0xF>(v);
  v = lane_max<0x112, 0xF>(v);
  v = lane_max<0x114, 0xF>(v);
  v = lane_max<0x118, 0xF>(v);
  v = lane_max<0x142, 0xA>(v);
  v = lane_max<0x143, 0xC>(v);
  return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ double lane_value(double x, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}

// acc + the terms of lanes first .. last-1 in order, one after the other, lane
// L holding terms w[0..S) that follow those of lane L-1: every lane adds its
// own terms to the sum so far, and lane L's result is read out as the start of
// lane L+1's chain; the other lanes' results are discarded.
template <int S>
__device__ __forceinline__ double literal(const double (&w)[S], double acc, int first, int last) {
#pragma clang fp contract(off)
  for (int L = first; L < last; L++) {
    double t = acc;
#pragma unroll
    for (int s = 0; s < S; s++) t = t + w[s];
    acc = lane_value(t, L);
  }
  return acc;
}

// The same over lanes 0 .. lanes-1 (+0.0 in the lanes past them).
template <int S>
__device__ __forceinline__ double chain(const double (&w)[S], double acc, int lanes) {
#pragma clang fp contract(off)
  constexpr int kExp = 0x7ff00000, kSignExp = (int)0xfff00000u;
  const int lane = (int)threadIdx.x & 63;
  double tot = w[0], mx = fabs(w[0]);
#pragma unroll
  for (int s = 1; s < S; s++) {
    tot = tot + w[s];
    mx = fmax(mx, fabs(w[s]));
  }
  mx = S * mx;
  const double pre = wave_prefix(tot), st = acc + (pre - tot), a = fabs(st);
  const int se = __double2hiint(st) & kSignExp, ex = se & kExp;
  const int top = wave_max_int(max(ex, max(__double2hiint(pre) & kExp, __double2hiint(mx) & kExp)));
  const double b0 = __hiloint2double(ex, 0);
  const bool ok = ex >= 0x04000000 && ex <= 0x7b000000 && ex >= top - (10 << 20) && a - mx >= b0 * (1.0 + 0x1p-30) &&
                  a + mx <= b0 * (2.0 - 0x1p-30) && mx <= 0.49 * b0;
  const double s0 = __hiloint2double(se | 0x80000, 0), s1 = __hiloint2double(se | 0x80000, 1);
  double t0 = s0, t1 = s1;
#pragma unroll
  for (int s = 0; s < S; s++) {
    t0 = t0 + w[s];
    t1 = t1 + w[s];
  }
  const double c0 = t0 - s0, c1 = t1 - s1;
  const unsigned long long all = lanes >= 64 ? ~0ull : (1ull << lanes) - 1;
  const unsigned long long lit = __ballot(!ok) & all;
  const unsigned long long odd = __ballot(ok && (__double2loint(t0) & 1));
  const unsigned long long ties = __ballot(ok && c0 != c1);
  const int se_below = __builtin_amdgcn_update_dpp(0, se, 0x138, 0xF, 0xF, false);  // wave_shr:1
  // the lanes at which a run (or a literal lane) starts
  const unsigned long long heads = (lit << 1) | lit | __ballot(ok && se_below != se) | 1ull;
  const unsigned long long below = (1ull << lane) - 1;
  const int head = 63 - __clzll((long long)(heads & (below | (1ull << lane))));
  // the parity that enters this lane if an even sum enters its run: of the odd
  // increments since the run's start, or since the last lane with a halfway case
  unsigned long long from = below & (~0ull << head);
  if (ties & from) from &= ~0ull << (63 - __clzll((long long)(ties & from)));
  const bool par = __popcll(odd & from) & 1;
  const double run = wave_prefix_from(ok && lane < lanes ? (par ? c1 : c0) : 0.0, lane, head);
  const double flip = par ? c0 - c1 : c1 - c0;
  for (int L = 0; L < lanes;) {
    int end = L + 1;
    if (!((lit >> L) & 1)) {
      const unsigned long long next = L < 63 ? (heads & all) >> (L + 1) : 0;
      end = next ? L + __ffsll((long long)next) : lanes;
      if ((__builtin_amdgcn_readfirstlane(__double2hiint(acc)) & kSignExp) == __builtin_amdgcn_readlane(se, L)) {
        double add = lane_value(run, end - 1);
        const unsigned long long tie = (ties >> L) & (~0ull >> (64 - (end - L)));
        if (tie && (__builtin_amdgcn_readfirstlane(__double2loint(acc)) & 1))
          add = add + lane_value(flip, L + __ffsll((long long)tie) - 1);
        acc = acc + add;
        L = end;
        continue;
      }
    }
    acc = literal<S>(w, acc, L, end);
    L = end;
  }
  return acc;
}

// The sum of the terms v[at(i)] (W = 0) or v[at(i)] (x[at(i) + 1] - x[at(i)])
// (W = 1), i in [0, n), in order, in chunks of 64*S terms with the next chunk's loads in
// flight; sh: lds_doubles(S) doubles of LDS of this wave's own.  Every lane
// returns it.  Terms past the end are +0.0, which leaves a sum started at +0.0
// unchanged (in round-to-nearest such a sum is never -0.0).
template <int S, int W, class T, class At>
__device__ __forceinline__ double ordered_sum(const T* __restrict__ v, const double* __restrict__ x, const At& at,
                                              int n, double* sh) {
#pragma clang fp contract(off)
  const int lane = (int)threadIdx.x & 63;
  T a[S];
  double x0[S], x1[S];
  auto load = [&](int c) {
#pragma unroll
    for (int s = 0; s < S; s++) {
      const int i = at(min(c + s * 64 + lane, n - 1));
      a[s] = v[i];
      if (W) {
        x0[s] = x[i];
        x1[s] = x[i + 1];
      }
    }
  };
  if (n > 0) load(0);
  double acc = 0.0;
  for (int c = 0; c < n; c += 64 * S) {
    double w[S];
#pragma unroll
    for (int s = 0; s < S; s++) {
      const int q = s * 64 + lane;
      sh[q + q / S] = (c + q < n) ? (W ? (double)a[s] * (x1[s] - x0[s]) : (double)a[s]) : 0.0;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s = 0; s < S; s++) w[s] = sh[lane * (S + 1) + s];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (c + 64 * S < n) load(c + 64 * S);
    const int lanes = min(64, (n - c + S - 1) / S);
    acc = n <= kLiteral ? literal<S>(w, acc, 0, lanes) : chain<S>(w, acc, lanes);
  }
  return acc;
}
struct Straight {
  __device__ __forceinline__ int operator()(int i) const { return i; }
};

}  // namespace f3d_ring
