// CPU build of the taxel sensor's sample counts (hcs_samples.h), test
// infrastructure only.
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

}  // extern "C"
