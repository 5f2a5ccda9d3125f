// CPU build of the taxel sensor's sample counts and the curved sensor's ray
// cull (hcs_samples.h), test infrastructure only.
#include <hip/hip_runtime.h>

#include "hcs_samples.h"

thread_local Dim3 threadIdx;
thread_local int g_lane;
WaveEmu* g_wave;

using namespace hcs;

extern "C" {

/* The samples of one surface (AREA_IMPORTANCE), or -1 where they are refused;
 * the first cap sums in acc. */
int64_t emu_area_chain(double top, double step, double* acc, int64_t cap) {
  bool too_many;
  const unsigned n = area_chain(top, step, too_many, [&](unsigned k, double a) {
    if ((int64_t)k < cap) acc[k] = a;
  });
  return too_many ? -1 : (int64_t)n;
}

/* The samples of one triangle (9 coordinates, DEFAULT), or -1. */
int64_t emu_grid_samples(const double* tri, double res) {
  const unsigned long long n = grid_samples(tri, res);
  return n > HCS_TS_MAX ? -1 : (int64_t)n;
}

/* skip[i]: the line of ray i (origin O, direction D) is skipped for triangle
 * i. */
void emu_lines_miss(const double* T, const double* O, const double* D, int64_t n, unsigned char* skip) {
  for (int64_t i = 0; i < n; ++i) {
    const double *o = O + 3 * i, *d = D + 3 * i;
    double b[HCS_SPHERE], sc = 0.0;
    for (int c = 0; c < 3; ++c) sc = fmax(sc, fabs(o[c]));
    const double D2 = dot3(d, d);
    fan_sphere(T + 9 * i, fmax(1.0, sqrt(D2)), b);
    skip[i] = line_misses(b, o, d, 1.0 / D2, sc, 1e-9 * sc + 1e-300);
  }
}

}  // extern "C"
