/*
 * hcs_samples.h -- sample counts of the taxel sensor's samplers.
 */
#pragma once
#include "hcs_device.h"

#pragma clang fp contract(off)

namespace hcs {

/* Samples are numbered by 32-bit offsets: a sampler that asks for more is
 * refused before anything is sized by its count. */
#define HCS_TS_MAX 0xffffffffull

/* All samples of a sensor, counted in 64 bits (a sum of 32-bit counts may
 * pass 2^32), and whether a sampler stopped at HCS_TS_MAX. */
struct TsTotal {
  unsigned long long n;
  int too_many, pad;
};

__device__ inline double edge_length(const double* a, const double* b) {
  const double d[3] = {a[0] - b[0], a[1] - b[1], a[2] - b[2]};
  return sqrt(dot3(d, d));
}

/* The reference's loop counts of one triangle (v0, v1, v2) under DEFAULT
 * sampling; false where they pass an int (more than HCS_TS_MAX samples, since
 * the inner loop takes two or more). */
__device__ inline bool grid_steps(const double* T, double res, int& st, int& st2) {
  const double n0 = edge_length(T + 3, T) / res, n1 = edge_length(T + 6, T) / res;
  if (n0 >= 2147483646.0 || n1 >= 2147483646.0) return false;
  const int st0 = (int)n0 + 1, st1 = (int)n1 + 1;
  st2 = st1;
  st = st0 > st1 ? st0 : st1;
  return true;
}

/* The samples of one triangle under DEFAULT sampling: the passes of the loops
 * a, b = 0, 1 / st, ... (rounded additions) while <= 1.  More than HCS_TS_MAX
 * for any number beyond it. */
__device__ inline unsigned long long grid_samples(const double* T, double res) {
  int st, st2;
  if (!grid_steps(T, res, st, st2) || (double)st * (double)st2 > 4.3e9) return HCS_TS_MAX + 1;
  unsigned long long na = 0, nb = 0;
  for (double a = 0; a <= 1; a += 1. / st) ++na;
  for (double b = 0; b <= 1; b += 1. / st2) ++nb;
  const unsigned long long n = na * nb;
  return n > HCS_TS_MAX ? HCS_TS_MAX + 1 : n;
}

/* The samples of one surface under AREA_IMPORTANCE: one for every sum acc =
 * 0, step, 2 step, ... (rounded additions) below top; each(k, acc) is called
 * with every one, and their number returned.  Where they pass HCS_TS_MAX (or,
 * with a step below the rounding of top, never end) nothing is called: the
 * quotient tells, since the rounding of 2^32 additions moves it by less than
 * 1e-6. */
template <class F>
__device__ inline unsigned area_chain(double top, double step, bool& too_many, F each) {
  unsigned n = 0;
  too_many = top > 4.3e9 * step;
  if (too_many) return 0;
  for (double acc = 0.0; acc < top; acc = acc + step, ++n) {
    too_many = n == HCS_TS_MAX;
    if (too_many) break;
    each(n, acc);
  }
  return n;
}

}  // namespace hcs
