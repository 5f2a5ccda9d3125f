/*
 * hcs_reduce.h -- the per-pair reduction's device code, shared by the batched
 * and the per-call steps.
 */
#pragma once
#include "hcs_query.h"

namespace hcs {

/* Slice j of K of one pair's results, summed by one wave: the contributions
 * cb[lo..hi) lane-strided in slot order, then a fixed butterfly, and the
 * candidate counts of items i0..i1.  Every lane returns the sums. */
__device__ inline RedPart reduce_slice(const Contrib* __restrict__ cb, unsigned lo, unsigned hi, int j, int K,
                                       const int* __restrict__ item_ncand, int first, int cnt) {
  const int lane = threadIdx.x & 63;
  const uint64_t len = hi - lo;
  const unsigned s0 = lo + (unsigned)(len * j / K), s1 = lo + (unsigned)(len * (j + 1) / K);
  const int i0 = first + (int)((int64_t)cnt * j / K), i1 = first + (int)((int64_t)cnt * (j + 1) / K);
  double F[3] = {0, 0, 0}, tA[3] = {0, 0, 0}, tB[3] = {0, 0, 0};
  int64_t np = 0, nf = 0, nc = 0;
  auto add = [&](const Contrib& q) {
#pragma unroll
    for (int c = 0; c < 3; ++c) F[c] = F[c] + q.F[c], tA[c] = tA[c] + q.tA[c], tB[c] = tB[c] + q.tB[c];
    np += q.np, nf += q.nf;
  };
  /* four slots loaded before they are added, so four loads are in flight per
   * lane */
  unsigned i = s0 + lane;
  for (; i < s1 && s1 - i > 192; i += 256) {
    const Contrib q0 = cb[i], q1 = cb[i + 64], q2 = cb[i + 128], q3 = cb[i + 192];
    add(q0), add(q1), add(q2), add(q3);
  }
  for (; i < s1; i += 64) add(cb[i]);
  for (int k = i0 + lane; k < i1; k += 64) nc += item_ncand[k];
  RedPart r;
#pragma unroll
  for (int c = 0; c < 3; ++c)
    r.F[c] = wave_sum<double>(F[c]), r.tA[c] = wave_sum<double>(tA[c]), r.tB[c] = wave_sum<double>(tB[c]);
  r.np = wave_sum_i(np), r.nf = wave_sum_i(nf), r.nc = wave_sum_i(nc);
  return r;
}

}  // namespace hcs
