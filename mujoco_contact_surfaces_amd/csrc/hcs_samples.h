/*
 * hcs_samples.h -- sample counts of the taxel sensor's samplers, and the ray
 * cull of the curved sensor.
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

/* Whether a ray's line can be accepted by the hit test of a triangle: not when
 * it misses the triangle's bounding sphere (centre C, radius r), widened.  The
 * computed barycentrics err by at most 16 eps |D| (|s| + L) L^2 / |det| in
 * position, s the vector from the triangle to the ray's origin, D its
 * direction, L <= 2r the longest edge, and the hit test rejects |det| < 1e-10,
 * so an accepted hit lies within 3.6e-5 |D| (|s| + L) L^2 of the triangle; the
 * sphere is widened by more than four times that (|s| bounded through the
 * largest coordinates, |D| by dmax >= 1), by 1e-9 of the ray's largest
 * coordinate, and the comparison by 1e-14 |s|^2 for the cancellation in
 * |s|^2 - (s.D)^2 / |D|^2.  A NaN or infinity fails the comparison, so nothing
 * is skipped on it. */
#define HCS_SPHERE 5 /* C, r with its part of the widening, factor of the ray's part */
__device__ inline void fan_sphere(const double* T, double dmax, double* b) {
  double C[3], tm = 0.0, r2 = 0.0;
#pragma unroll
  for (int c = 0; c < 3; ++c)
    C[c] = ((T[c] + T[3 + c]) + T[6 + c]) * (1.0 / 3.0),
    tm = fmax(tm, fmax(fabs(T[c]), fmax(fabs(T[3 + c]), fabs(T[6 + c]))));
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    const double d[3] = {T[3 * v] - C[0], T[3 * v + 1] - C[1], T[3 * v + 2] - C[2]};
    r2 = fmax(r2, dot3(d, d));
  }
  const double r = sqrt(r2), k = 1.2e-3 * r2 * dmax;
  b[0] = C[0], b[1] = C[1], b[2] = C[2], b[3] = r + k * (tm + r), b[4] = k;
}
/* sc: the ray's largest coordinate, sl = 1e-9 sc + 1e-300, iD2 = 1 / |D|^2 */
__device__ inline bool line_misses(const double* b, const double* O, const double* D, double iD2, double sc,
                                   double sl) {
  const double s[3] = {b[0] - O[0], b[1] - O[1], b[2] - O[2]};
  const double ss = dot3(s, s), sd = dot3(s, D), re = (b[3] + b[4] * sc) + sl;
  return ss - (sd * sd) * iD2 > re * re + 1e-14 * ss;
}

}  // namespace hcs
