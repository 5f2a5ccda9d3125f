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
