/*
 * hcs_taxel_sensor.hip -- the taxel sensor on the GPU, FP64.
 *
 * Restates TaxelSensor::internal_update
 * (mujoco_contact_surface_sensors/src/taxel_sensor.cpp:158-478) over the
 * contact polygons kept by the last contact step:
 *   1. the polygons of the pairs touching the sensor geometry, in key order
 *      (pair, element of A, element of B) -- by rank, or radix passes over the
 *      packed key -- and their kTriangle fans (v_k, v_{k+1}, C), the surface's
 *      triangles;
 *   2. samples on every triangle: DEFAULT (:174-203), the reference's loops
 *      a, b += 1/st from 0 while <= 1 with st from |v1 - v0| and |v2 - v0|
 *      (both st1 and st2 from v2 - v0), one thread per triangle after a
 *      count and a scan; or AREA_IMPORTANCE (:205-246), a single sequential
 *      stream of libstdc++'s default_random_engine through
 *      uniform_real_distribution<double>(0, 1), its running sums in
 *      order and its samples in parallel;
 *   3. taxels against samples: dist = (-2 t.p + |t|^2) + |p|^2 to every
 *      sample; CLOSEST (:285-319) takes the first nearest sample, and within
 *      the margin writes its pressure when visualize is set and |p| > 1e-6,
 *      else 0; WEIGHTED and MEAN fall through to SQUARED (:320-457, no
 *      break): sum of max(0, margin - sqrt(dist))^2 |p| over the samples in
 *      the margin, times sample_resolution.  A taxel no sample reaches keeps
 *      its value; with no sample at all every taxel is 0 (:458-477).
 * Sums over samples run lane-strided within fixed slices of the samples, then
 * in a fixed butterfly and over the slices, so results are deterministic.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "hcs_device.h"
#include "hcs_internal.h"
#include "hcs_prim.h"
#include "hcs_query.h"
#include "hcs_samples.h"

#pragma clang fp contract(off)

using namespace hcs;

namespace hcs {

#define HCS_TS_TRI 12 /* fan triangle: v0, v1, v2 (W), e0, e1, e2 */

/* Sort keys of the kept polygons: (pair, element of A, element of B) packed
 * into the bits the pairs and meshes need when those fit 64 (ba, bb >= 0:
 * bits of the elements), else (element of A, element of B) with the pair in
 * kp.  Unselected polygons sort last.  For the rank sort, its counters are
 * cleared here and every place is empty (-1) until a polygon takes it.  The
 * sampler's total is cleared too. */
__global__ void k_ts_keys(const int64_t* __restrict__ key, int64_t np, const unsigned char* __restrict__ mask, int ba,
                          int bb, unsigned long long* __restrict__ k64, unsigned* __restrict__ kp,
                          int* __restrict__ idx, unsigned* __restrict__ rank, TsTotal* __restrict__ total) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= np) return;
  if (i == 0) *total = TsTotal{};
  const unsigned long long pair = key[3 * i], a = key[3 * i + 1], b = key[3 * i + 2];
  const bool on = mask[pair] != 0;
  if (ba >= 0) {
    k64[i] = on ? (((pair << ba) | a) << bb) | b : ~0ull;
  } else {
    k64[i] = (a << 32) | b;
    kp[i] = on ? (unsigned)pair : 0xffffffffu;
  }
  idx[i] = rank ? -1 : (int)i;
  if (rank) rank[i] = 0;
}

__global__ void k_ts_gather_u32(const unsigned* __restrict__ src, const int* __restrict__ idx, int64_t n,
                                unsigned* __restrict__ dst) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}

/* Rank sort, for up to HCS_TS_RANK polygons: the keys are distinct (one
 * polygon per element pair; the unselected share the largest key and need no
 * order), so a polygon's place is the number of smaller keys.  One thread
 * per polygon, blockIdx.y a slice of the keys it is compared with, staged in
 * LDS.  n^2 compares are cheaper than the radix sort's launches at these
 * sizes: 6.8k polygons 60 launches, about 300 us (12 passes of 5) -> 2
 * launches, 12 us; at 16k the compares take about 30 us, as much as the
 * radix sort on packed keys. */
#define HCS_TS_RANK 16384
__global__ __launch_bounds__(256) void k_ts_rank(const unsigned long long* __restrict__ k64, int n, int per,
                                                 unsigned* __restrict__ rank) {
  __shared__ unsigned long long tile[256];
  const int t = threadIdx.x, i = blockIdx.x * 256 + t;
  const unsigned long long k = i < n ? k64[i] : 0ull;
  const int j1 = min(n, (int)(blockIdx.y + 1) * per);
  unsigned less = 0;
  for (int j0 = blockIdx.y * per; j0 < j1; j0 += 256) {
    __syncthreads();
    tile[t] = j0 + t < j1 ? k64[j0 + t] : ~0ull;
    __syncthreads();
#pragma unroll 8
    for (int u = 0; u < 256; ++u) less += tile[u] < k;
  }
  if (i < n && less && k != ~0ull) atomicAdd(rank + i, less);
}

/* order by rank; the places after the last selected polygon stay -1 */
__global__ void k_ts_order(const unsigned long long* __restrict__ k64, const unsigned* __restrict__ rank, int n,
                           int* __restrict__ order) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && k64[i] != ~0ull) order[rank[i]] = i;
}

/* fans of the i-th polygon in order: 0 for an unselected one */
__global__ void k_ts_nfan(const double* __restrict__ poly, const int64_t* __restrict__ key,
                          const unsigned char* __restrict__ mask, const int* __restrict__ order, int n,
                          unsigned* __restrict__ nt) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i > n) return;
  const int q = i < n ? order[i] : -1;
  nt[i] = q >= 0 && mask[key[3 * (size_t)q]] ? (unsigned)poly[HCS_PREC * (size_t)q] : 0u;
}

__global__ void k_ts_fans(const double* __restrict__ poly, const int64_t* __restrict__ key,
                          const int* __restrict__ order, int n, const unsigned* __restrict__ off,
                          double* __restrict__ tris, int* __restrict__ surf, unsigned* __restrict__ cnt_end) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) *cnt_end = 0; /* (of k_ts_count) */
  if (i >= n || off[i] == off[i + 1]) return;
  const double* P = poly + HCS_PREC * (size_t)order[i];
  const int nv = (int)P[0];
  for (int k = 0; k < nv; ++k) {
    const int k2 = k + 1 < nv ? k + 1 : 0;
    double* T = tris + HCS_TS_TRI * (size_t)(off[i] + k);
#pragma unroll
    for (int c = 0; c < 3; ++c) T[c] = P[1 + 3 * k + c], T[3 + c] = P[1 + 3 * k2 + c], T[6 + c] = P[33 + c];
    T[9] = P[25 + k], T[10] = P[25 + k2], T[11] = P[36];
    surf[off[i] + k] = (int)key[3 * (size_t)order[i]];
  }
}

__device__ inline void ts_sample(const double* T, double b0, double b1, double b2, double* p, double* e) {
#pragma unroll
  for (int c = 0; c < 3; ++c) p[c] = (b0 * T[c] + b1 * T[3 + c]) + b2 * T[6 + c];
  *e = (b0 * T[9] + b1 * T[10]) + b2 * T[11];
}

/* Samples per triangle.  Their sum is at most HCS_TS_MAX when each is at most
 * an nt-th of it; one that is more raises cnt[nt] (cleared before), and the sum
 * is then made in 64 bits (k_ts_sum).  (Summing in 64 bits every time, one
 * atomic per wave, took 7.1 us for 3.5.) */
__global__ void k_ts_count(const double* __restrict__ tris, int64_t nt, double res, unsigned long long each,
                           unsigned* __restrict__ cnt) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= nt) return;
  const unsigned long long n = grid_samples(tris + HCS_TS_TRI * t, res);
  cnt[t] = (unsigned)n;
  if (n > each) cnt[nt] = 1;
}

__global__ __launch_bounds__(256) void k_ts_sum(const double* __restrict__ tris, int64_t nt, double res,
                                                TsTotal* __restrict__ total) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const unsigned long long n = t < nt ? grid_samples(tris + HCS_TS_TRI * t, res) : 0ull;
  if (n > HCS_TS_MAX) total->too_many = 1;
  const int64_t sum = wave_sum_i((int64_t)n);
  if ((threadIdx.x & 63) == 0) atomicAdd(&total->n, (unsigned long long)sum);
}

__global__ void k_ts_gen(const double* __restrict__ tris, int64_t nt, double res, const unsigned* __restrict__ off,
                         double* __restrict__ P, double* __restrict__ E) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= nt) return;
  const double* T = tris + HCS_TS_TRI * t;
  int st, st2;
  if (!grid_steps(T, res, st, st2)) return;
  size_t j = off[t];
  for (double a = 0; a <= 1; a += 1. / st)
    for (double b = 0; b <= 1; b += 1. / st2) {
      ts_sample(T, a, (1 - a) * (1 - b), (1 - a) * b, P + 3 * j, E + j);
      ++j;
    }
}

/* libstdc++ default_random_engine (minstd_rand0, seed 1) through
 * generate_canonical<double, 53>: two draws, sum = (g1 - 1) + (g2 - 1) r,
 * r = 2^31 - 2, over r^2; a result >= 1 becomes the largest double below 1.
 * The long double products of the library are exact here, so double
 * arithmetic gives the same bits. */
struct TsRng {
  unsigned long long x = 1;
  __device__ double next() {
    const double r = 2147483646.0;
    double sum = 0.0, tmp = 1.0;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      x = (x * 16807ull) % 2147483647ull;
      sum += (double)(x - 1) * tmp;
      tmp = tmp * r;
    }
    const double u = sum / tmp;
    return u >= 1.0 ? 0x1.fffffffffffffp-1 : u;
  }
};

/* AREA_IMPORTANCE (:205-246).  Per surface the reference walks the triangles
 * adding areas (at) and, while a running sum acc of resolution * total area is
 * below at, draws a sample on the current triangle, all from one random
 * stream.  The running sums are chains of rounded additions that decide which
 * triangle a sample falls on and how many there are, so they are added in
 * that order; everything else is parallel:
 *   k_ts_areas  the triangles' areas;
 *   k_ts_chain  one wave per surface: the prefix sums of its areas (the last
 *               is the total), then the chain of acc below the total, counted
 *               (write = false) or stored (write = true);
 *   k_ts_draw   one thread per sample: its triangle is the first whose prefix
 *               sum exceeds its acc, its random numbers come from jumping the
 *               generator ahead to its place in the stream.
 * One thread doing all of it, twice, took 28 ms for 25k triangles and 500
 * samples; the chain kernel's two passes take 0.5 ms (FP64 add latency). */
__global__ void k_ts_areas(const double* __restrict__ tris, const int* __restrict__ surf, int64_t nt,
                           double* __restrict__ area, int* __restrict__ surf0, unsigned* __restrict__ nsurf) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (t >= nt) return;
  const double* T = tris + HCS_TS_TRI * t;
  double e1[3] = {T[3] - T[0], T[4] - T[1], T[5] - T[2]}, e2[3] = {T[6] - T[0], T[7] - T[1], T[8] - T[2]}, cr[3];
  cross3(e1, e2, cr);
  area[t] = 0.5 * sqrt(dot3(cr, cr));
  /* the first triangle of every surface (in no order) */
  if (t == 0 || surf[t] != surf[t - 1]) surf0[atomicAdd(nsurf, 1u)] = (int)t;
}

#define HCS_TS_CHAIN 1024
__global__ __launch_bounds__(64) void k_ts_chain(const int* __restrict__ surf, int64_t nt,
                                                 const int* __restrict__ surf0, const unsigned* __restrict__ nsurf,
                                                 double res, bool write, double* __restrict__ at,
                                                 unsigned* __restrict__ count, TsTotal* __restrict__ total,
                                                 const unsigned* __restrict__ off, double* __restrict__ acc_out,
                                                 int2* __restrict__ tri_out) {
  __shared__ double L[HCS_TS_CHAIN];
  const int lane = threadIdx.x;
  if (blockIdx.x >= *nsurf) return;
  const int64_t t0 = surf0[blockIdx.x];
  const int id = surf[t0];
  /* the surface's end (the triangles are ordered by surface) */
  int64_t t1 = t0 + 1;
  for (int64_t hi = nt; t1 < hi;) {
    const int64_t mid = (t1 + hi) >> 1;
    if (surf[mid] == id) t1 = mid + 1;
    else hi = mid;
  }
  if (!write) {
    /* prefix sums in place of the areas, a tile of LDS at a time (padded with
     * zeros, which leave the sum as it is): every lane adds the same chain
     * (broadcast reads), lane 0 stores it */
    double total = 0.0;
    for (int64_t c0 = t0; c0 < t1; c0 += HCS_TS_CHAIN) {
      const int cn = (int)(t1 - c0 < HCS_TS_CHAIN ? t1 - c0 : HCS_TS_CHAIN);
      __syncthreads();
      for (int k = lane; k < HCS_TS_CHAIN; k += 64) L[k] = k < cn ? at[c0 + k] : 0.0;
      __syncthreads();
      for (int k = 0; k < cn; k += 16) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = L[k + u];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = total = total + v[u];
        if (lane == 0) {
#pragma unroll
          for (int u = 0; u < 16; ++u) L[k + u] = v[u];
        }
      }
      __syncthreads();
      for (int k = lane; k < cn; k += 64) at[c0 + k] = L[k];
    }
    __syncthreads();
  }
  /* a sample is drawn while acc is below some prefix sum: the total, or the
   * last that is a number (fmax passes over a NaN area and what follows it) */
  double top = 0.0;
#pragma unroll 8
  for (int64_t t = t0 + lane; t < t1; t += 64) top = fmax(top, at[t]);
  top = wave_max(top);
  const double step = res * at[t1 - 1];
  const unsigned base = write ? off[id] : 0u;
  bool too_many;
  const unsigned n = area_chain(top, step, too_many, [&](unsigned k, double acc) {
    if (write && lane == 0) acc_out[base + k] = acc, tri_out[base + k] = make_int2((int)t0, (int)t1 - 1);
  });
  if (write || lane != 0) return;
  count[id] = n;
  atomicAdd(&total->n, (unsigned long long)n);
  if (too_many) total->too_many = 1;
}

/* x * 16807^e modulo 2^31 - 1 */
__device__ inline unsigned long long minstd_jump(unsigned long long x, unsigned long long e) {
  for (unsigned long long g = 16807ull; e; e >>= 1, g = (g * g) % 2147483647ull)
    if (e & 1) x = (x * g) % 2147483647ull;
  return x;
}

__global__ void k_ts_draw(const double* __restrict__ tris, const double* __restrict__ at,
                          const double* __restrict__ acc, const int2* __restrict__ range, int64_t m,
                          double* __restrict__ P, double* __restrict__ E) {
  const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (j >= m) return;
  /* prefix sums do not decrease (a NaN counts as exceeding) */
  const double a0 = acc[j];
  int64_t lo = range[j].x, hi = range[j].y;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (at[mid] <= a0) lo = mid + 1;
    else hi = mid;
  }
  TsRng gen;
  gen.x = minstd_jump(gen.x, 4ull * (unsigned long long)j);
  const double u0 = gen.next(), u1 = gen.next();
  const double a = 1.0 - sqrt(u0);
  const double b = (1.0 - a) * u1;
  ts_sample(tris + HCS_TS_TRI * lo, a, (1 - a) * (1 - b), (1 - a) * b, P + 3 * j, E + j);
}

struct CsArgs {
  double X[12];
  double margin;
};

struct TsTaxelArgs {
  double X[12];
  double margin, res;
  int method, visualize;
};

/* One wave's result for a taxel over its slice of the samples: squared: the
 * weighted sum and the samples in the margin; closest: the least distance
 * and its first sample (n < 0: none). */
struct TsPart {
  double v;
  long long n;
};

/* Taxels against samples.  A wave takes HCS_TS_TX taxels and a slice of the
 * samples (blockIdx.y), a lane every 64th sample of it: a sample is loaded
 * once for the wave's taxels, and the slices fill the chip whatever the
 * number of taxels (one wave per taxel over all samples was 256 waves, each
 * a chain of 1600 loads of its own: 501 us for 256 taxels and 104k samples,
 * -> 27 us).  What bounds it is the latency of its loads and FP64 chains: 28%
 * of the issue slots, the waves waiting 58% of the time. */
#define HCS_TS_TX 8
template <bool CLOSEST>
__global__ __launch_bounds__(64) void k_ts_taxel(const double* __restrict__ P, const double* __restrict__ E,
                                                 int64_t m, TsTaxelArgs a, const double* __restrict__ taxels, int nx,
                                                 TsPart* __restrict__ part) {
  const int i0 = blockIdx.x * HCS_TS_TX, lane = threadIdx.x;
  double tw[HCS_TS_TX][3], tt[HCS_TS_TX], v[HCS_TS_TX];
  int64_t n[HCS_TS_TX];
#pragma unroll
  for (int k = 0; k < HCS_TS_TX; ++k) {
    const int i = i0 + k < nx ? i0 + k : nx - 1;
    xform(a.X, taxels + 3 * (size_t)i, tw[k]);
    tt[k] = dot3(tw[k], tw[k]);
    v[k] = CLOSEST ? __builtin_inf() : 0.0;
    n[k] = CLOSEST ? 0x7fffffffffffffffll : 0;
  }
  const double msq = a.margin * a.margin;
  const int64_t s0 = m * blockIdx.y / gridDim.y, s1 = m * (blockIdx.y + 1) / gridDim.y;
  for (int64_t j = s0 + lane; j < s1; j += 64) {
    const double p[3] = {P[3 * j], P[3 * j + 1], P[3 * j + 2]};
    const double e = CLOSEST ? 0.0 : fabs(E[j]);
    const double pp = dot3(p, p);
#pragma unroll
    for (int k = 0; k < HCS_TS_TX; ++k) {
      const double d = ((-2.0 * dot3(tw[k], p)) + tt[k]) + pp;
      if (CLOSEST) {
        if (d < v[k]) v[k] = d, n[k] = j;
      } else if (d < msq) {
        const double w0 = fmax(0.0, a.margin - sqrt(d));
        v[k] += (w0 * w0) * e;
        ++n[k];
      }
    }
  }
#pragma unroll
  for (int k = 0; k < HCS_TS_TX; ++k) {
    if (CLOSEST) {
      /* first nearest sample: (distance, index) lexicographic minimum */
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) {
        const double od = __shfl_xor(v[k], o, 64);
        const int64_t oj = __shfl_xor((long long)n[k], o, 64);
        if (od < v[k] || (od == v[k] && oj < n[k])) v[k] = od, n[k] = oj;
      }
    } else {
      v[k] = wave_sum<double>(v[k]);
      n[k] = wave_sum_i(n[k]);
    }
    if (lane == 0 && i0 + k < nx) part[(size_t)blockIdx.y * nx + i0 + k] = TsPart{v[k], (long long)n[k]};
  }
}

/* Per taxel, the slices' results in order, four lanes per taxel and then a
 * fixed butterfly; a taxel no sample reaches keeps its value. */
template <bool CLOSEST>
__global__ __launch_bounds__(64) void k_ts_combine(const TsPart* __restrict__ part, int nslice, int nx, TsTaxelArgs a,
                                                   const double* __restrict__ E, double* __restrict__ values) {
  const int i = blockIdx.x * 16 + (threadIdx.x & 15);
  TsPart b{CLOSEST ? __builtin_inf() : 0.0, CLOSEST ? 0x7fffffffffffffffll : 0};
  auto add = [&](const TsPart& q) {
    if (!CLOSEST) b.v += q.v, b.n += q.n;
    else if (q.v < b.v || (q.v == b.v && q.n < b.n)) b = q;
  };
  if (i < nx)
    for (int s = threadIdx.x >> 4; s < nslice; s += 4) add(part[(size_t)s * nx + i]);
#pragma unroll
  for (int o = 16; o <= 32; o <<= 1) add(TsPart{__shfl_xor(b.v, o, 64), __shfl_xor(b.n, o, 64)});
  if (i >= nx || threadIdx.x >= 16) return;
  if (CLOSEST) {
    if (b.v < a.margin * a.margin) values[i] = (a.visualize && fabs(E[b.n]) > 1e-6) ? E[b.n] : 0.0;
  } else if (b.n > 0) {
    values[i] = b.v * a.res;
  }
}

/* Sample slices of the taxel kernel: enough for about 2048 waves, at least
 * 256 samples each. */
static int ts_slices(int nx, int64_t m) {
  const int64_t groups = (nx + HCS_TS_TX - 1) / HCS_TS_TX;
  return (int)std::max<int64_t>(1, std::min<int64_t>(2048 / groups, m / 256));
}

/* The nearest hit of a ray in one slice of the triangles. */
struct CsHit {
  double t, u, v; /* t = 1e30: none */
  long long tri;
};

/* CurvedSensor rays: the sample moved by X (normal rotated, not
 * renormalised), ray from p + n 1e-8 along -n, Moeller-Trumbore
 * (S/src/bvh.cpp:49-74) in FP64 over the fan triangles, nearest t (first
 * triangle in order on ties).
 *
 * Triangles that the ray's line misses by more than the rounding of the hit
 * test are skipped (line_misses); the spheres are widened for the longest of
 * the wave's directions.
 *
 * One lane per ray, one wave per (64 rays, slice of the triangles): with a
 * thread walking every triangle, 2601 rays were 41 waves on 256 CUs, each a
 * chain of 11k triangle loads (5522 us); blockIdx.y cuts the chain so that
 * about 4096 waves run (see cs_slices).  The wave stages 64 triangles'
 * spheres in LDS (one per lane), so the inner loop is a broadcast read and
 * 16 FP64 operations, which bound it; each lane then hit-tests the triangles
 * of its own mask, so a round serves one triangle of every lane.  (The box of the ray segment
 * against the triangle's box, the test before, let a fifth of the triangles
 * through for rays oblique to the axes, so most triangles were hit-tested
 * for some lane: 67 us.)  2601 rays on 11.5k triangles: 5522 -> 45 us. */
__global__ __launch_bounds__(64) void k_cs_rays(const double* __restrict__ tris, int64_t nt, CsArgs a,
                                                const double* __restrict__ pts, const double* __restrict__ nrms, int m,
                                                CsHit* __restrict__ part) {
  __shared__ double sph[64][6]; /* (HCS_SPHERE, padded) */
  const int lane = threadIdx.x, j = blockIdx.x * 64 + lane, jr = j < m ? j : m - 1;
  double pw[3], nw[3], O[3], D[3], sc = 0.0;
  xform(a.X, pts + 3 * (size_t)jr, pw);
  rot(a.X, nrms + 3 * (size_t)jr, nw);
#pragma unroll
  for (int c = 0; c < 3; ++c) O[c] = pw[c] + nw[c] * 1e-8, D[c] = -nw[c], sc = fmax(sc, fabs(O[c]));
  const double D2 = dot3(D, D), iD2 = 1.0 / D2, sl = 1e-9 * sc + 1e-300;
  const double dmax = wave_max(fmax(1.0, sqrt(D2)));
  double best = 1e30, bu = 0.0, bv = 0.0;
  int64_t bt = -1;
  const int64_t t0 = nt * blockIdx.y / gridDim.y, t1 = nt * (blockIdx.y + 1) / gridDim.y;
  for (int64_t c0 = t0; c0 < t1; c0 += 64) {
    const int cn = (int)(t1 - c0 < 64 ? t1 - c0 : 64);
    __syncthreads();
    if (lane < cn) fan_sphere(tris + HCS_TS_TRI * (c0 + lane), dmax, sph[lane]);
    __syncthreads();
    /* the lane's triangles of the tile, then their hit tests in order */
    unsigned long long todo = 0;
#pragma unroll 8
    for (int k = 0; k < 64; ++k) todo |= line_misses(sph[k], O, D, iD2, sc, sl) ? 0ull : 1ull << k;
    todo &= ~0ull >> (64 - cn);
    while (todo) {
      const int64_t t = c0 + __builtin_ctzll(todo);
      todo &= todo - 1;
      const double* T = tris + HCS_TS_TRI * t;
      const double e1[3] = {T[3] - T[0], T[4] - T[1], T[5] - T[2]}, e2[3] = {T[6] - T[0], T[7] - T[1], T[8] - T[2]};
      double h[3];
      cross3(D, e2, h);
      const double det = dot3(e1, h);
      if (fabs(det) < 1e-10) continue;
      const double f = 1.0 / det;
      const double sv[3] = {O[0] - T[0], O[1] - T[1], O[2] - T[2]};
      const double u = f * dot3(sv, h);
      if (u < 0.0 || u > 1.0) continue;
      double qv[3];
      cross3(sv, e1, qv);
      const double v = f * dot3(D, qv);
      if (v < 0.0 || u + v > 1.0) continue;
      const double tt = f * dot3(e2, qv);
      if (tt > 0.0 && tt < best) best = tt, bu = u, bv = v, bt = t;
    }
  }
  if (j < m) part[(size_t)blockIdx.y * m + j] = CsHit{best, bu, bv, bt};
}

/* Per ray, the nearest of its slices' hits, the first triangle on ties; raw
 * pressure when 0 < t < margin.  16 rays per wave, the slices shared by four
 * lanes each (one lane per ray left 41 waves with 50 dependent loads). */
__global__ __launch_bounds__(64) void k_cs_hits(const double* __restrict__ tris, const CsHit* __restrict__ part,
                                                int nslice, double margin, int m, double* __restrict__ raw,
                                                unsigned char* __restrict__ hit) {
  const int j = blockIdx.x * 16 + (threadIdx.x & 15);
  CsHit b{1e30, 0.0, 0.0, 0x7fffffffffffffffll};
  if (j < m)
    for (int s = threadIdx.x >> 4; s < nslice; s += 4) {
      const CsHit h = part[(size_t)s * m + j];
      if (h.tri >= 0 && h.t < b.t) b = h;
    }
#pragma unroll
  for (int o = 16; o <= 32; o <<= 1) {
    const CsHit h{__shfl_xor(b.t, o, 64), __shfl_xor(b.u, o, 64), __shfl_xor(b.v, o, 64), __shfl_xor(b.tri, o, 64)};
    if (h.t < b.t || (h.t == b.t && h.tri < b.tri)) b = h;
  }
  if (j >= m || threadIdx.x >= 16) return;
  const bool ok = b.t < 1e30 && b.t < margin && b.t > 0.0;
  double r = 0.0;
  if (ok) {
    const double* T = tris + HCS_TS_TRI * b.tri;
    const double b0 = 1 - b.u - b.v;
    r = (b0 * T[9] + b.u * T[10]) + b.v * T[11];
  }
  raw[j] = r;
  hit[j] = ok ? 1 : 0;
}

/* Triangle slices of the ray kernel: enough for about 4096 waves (four per
 * SIMD), at least 64 triangles (one staged tile) each. */
static int cs_slices(int m, int64_t nt) {
  const int64_t groups = (m + 63) / 64;
  return (int)std::max<int64_t>(1, std::min<int64_t>(4096 / std::max<int64_t>(1, groups), nt / 64));
}

/* taxel i: sum over its samples of weight * raw, in list order; four entries
 * are loaded before they are added, so the chain of dependent loads (entry,
 * sample) is a quarter as long */
__global__ void k_cs_taxels(const int* __restrict__ ptr, const int* __restrict__ idx, const double* __restrict__ w,
                            int n, const double* __restrict__ raw, const unsigned char* __restrict__ hit,
                            double* __restrict__ values) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int k1 = ptr[i + 1];
  double pr = 0.0;
  for (int k = ptr[i]; k < k1; k += 4) {
    double term[4];
    bool on[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = k + u < k1 ? k + u : k;
      const int j = idx[q];
      on[u] = k + u < k1 && hit[j];
      term[u] = w[q] * raw[j];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (on[u]) pr += term[u];
  }
  values[i] = pr;
}

}  // namespace hcs

extern "C" {

/* Bits that hold the values 0 .. n. */
static int key_bits(int64_t n) {
  int b = 1;
  while (b < 62 && (n >> b) != 0) ++b;
  return b;
}

/* The kTriangle fan triangles of the kept polygons of the pairs touching
 * geometry geom, in key order, into c->ts.tris / c->ts.surf. */
static int sensor_fans(Ctx* c, int32_t geom, unsigned& ntri) {
  int rc;
  hipStream_t s = c->stream;
  const int npairs = (int)c->last_pairs.size();
  const int64_t np = c->last_npoly;
  std::vector<unsigned char> mask(std::max(1, npairs), 0);
  for (int e = 0; e < npairs; ++e)
    mask[e] = (c->last_geoms[2 * e] == geom || c->last_geoms[2 * e + 1] == geom) ? 1 : 0;
  TaxelSensorBufs& B = c->ts;
  const size_t n1 = (size_t)std::max<int64_t>(1, np);
  if ((rc = ensure(c, B.mask, mask.size())) || (rc = ensure(c, B.k64, 2 * sizeof(unsigned long long) * n1)) ||
      (rc = ensure(c, B.kp, 2 * sizeof(unsigned) * n1)) || (rc = ensure(c, B.idx, 2 * sizeof(int) * n1)) ||
      (rc = ensure(c, B.cnt, 64)) || (rc = ensure(c, B.nfan, sizeof(unsigned) * (n1 + 1))) ||
      (rc = ensure(c, B.fan_off, sizeof(unsigned) * (n1 + 1))))
    return rc;
  rc = hip_check(c, hipMemcpyAsync(B.mask.ptr, mask.data(), mask.size(), hipMemcpyHostToDevice, s), "upload mask");
  if (rc) return rc;
  unsigned long long* k64 = (unsigned long long*)B.k64.ptr;
  unsigned* kp = (unsigned*)B.kp.ptr;
  int *idx = (int*)B.idx.ptr, *order = idx + n1;
  const unsigned char* dmask = (const unsigned char*)B.mask.ptr;
  ntri = 0;
  if (np > 0) {
    /* bits of the packed key: pair numbers, and the element counts of the
     * pairs' meshes */
    int64_t ma = 1, mb = 1;
    for (int e = 0; e < npairs; ++e) {
      ma = std::max<int64_t>(ma, c->meshes[c->last_geoms[2 * e]].nelem);
      mb = std::max<int64_t>(mb, c->meshes[c->last_geoms[2 * e + 1]].nelem);
    }
    const int bp = key_bits(npairs), ba = key_bits(ma), bb = key_bits(mb);
    const bool packed = bp + ba + bb < 64;
    const bool rank = packed && np <= HCS_TS_RANK;
    const unsigned nb = (unsigned)((np + 255) / 256);
    hipLaunchKernelGGL(k_ts_keys, dim3(nb), dim3(256), 0, s, (const int64_t*)c->d_poly_key.ptr, np, dmask,
                       packed ? ba : -1, bb, k64, kp, rank ? order : idx, rank ? kp : nullptr, (TsTotal*)B.cnt.ptr);
    if (rank) {
      const int slices = (int)std::max<int64_t>(1, std::min<int64_t>(nb, 512 / nb));
      const int per = (int)((np + slices - 1) / slices);
      hipLaunchKernelGGL(k_ts_rank, dim3(nb, slices), dim3(256), 0, s, k64, (int)np, per, kp);
      hipLaunchKernelGGL(k_ts_order, dim3(nb), dim3(256), 0, s, k64, kp, (int)np, order);
    } else if (packed) {
      const size_t b = sort_temp_bytes(np, 8);
      if ((rc = ensure(c, B.tmp, std::max<size_t>(8, b)))) return rc;
      /* one bit more than the keys need: the unselected polygons' */
      if (radix_sort_pairs_u64(s, k64, k64 + n1, idx, order, np, 0, bp + ba + bb + 1, B.tmp.ptr, B.tmp.bytes) != 0)
        return set_err(c, HCS_ERR_LIMIT, "sensor: too many polygons to sort");
    } else {
      /* stable LSD passes: (element of A, element of B), then pair */
      const size_t b1 = sort_temp_bytes(np, 8), b2 = sort_temp_bytes(np, 4);
      if ((rc = ensure(c, B.tmp, std::max<size_t>(8, std::max(b1, b2))))) return rc;
      if (radix_sort_pairs_u64(s, k64, k64 + n1, idx, order, np, 0, 64, B.tmp.ptr, B.tmp.bytes) != 0)
        return set_err(c, HCS_ERR_LIMIT, "sensor: too many polygons to sort");
      hipLaunchKernelGGL(k_ts_gather_u32, dim3(nb), dim3(256), 0, s, kp, order, np, kp + n1);
      if (radix_sort_pairs_u32(s, kp + n1, kp, order, idx, np, 0, 32, B.tmp.ptr, B.tmp.bytes) != 0)
        return set_err(c, HCS_ERR_LIMIT, "sensor: too many polygons to sort");
      order = idx;
    }
    /* fan triangles of the selected polygons, in order */
    hipLaunchKernelGGL(k_ts_nfan, dim3((unsigned)((np + 1 + 255) / 256)), dim3(256), 0, s,
                       (const double*)c->d_poly_rec.ptr, (const int64_t*)c->d_poly_key.ptr, dmask, order, (int)np,
                       (unsigned*)B.nfan.ptr);
    if ((rc = ensure(c, B.tmp, std::max<size_t>(scan_temp_bytes((long long)np + 1), 8)))) return rc;
    if (exclusive_scan_u32(s, (const unsigned*)B.nfan.ptr, (unsigned*)B.fan_off.ptr, (long long)np + 1, B.tmp.ptr,
                           B.tmp.bytes) != 0)
      return set_err(c, HCS_ERR_LIMIT, "sensor: too many polygons to scan");
    rc = hip_check(c, hipMemcpyAsync(&ntri, (unsigned*)B.fan_off.ptr + np, sizeof(unsigned), hipMemcpyDeviceToHost, s),
                   "dl");
    if (!rc) rc = hip_check(c, hipStreamSynchronize(s), "sync");
    if (rc) return rc;
  }
  const size_t nt1 = std::max<size_t>(1, ntri);
  if ((rc = ensure(c, B.tris, sizeof(double) * HCS_TS_TRI * nt1)) || (rc = ensure(c, B.surf, sizeof(int) * nt1)) ||
      (rc = ensure(c, B.scnt, sizeof(unsigned) * (nt1 + 2))) || (rc = ensure(c, B.soff, sizeof(unsigned) * (nt1 + 2))))
    return rc;
  if (ntri > 0)
    hipLaunchKernelGGL(k_ts_fans, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, s,
                       (const double*)c->d_poly_rec.ptr, (const int64_t*)c->d_poly_key.ptr, order, (int)np,
                       (const unsigned*)B.fan_off.ptr, (double*)B.tris.ptr, (int*)B.surf.ptr,
                       (unsigned*)B.scnt.ptr + ntri);
  return hip_check(c, hipGetLastError(), "sensor triangles");
}

/* The sampler's count, when it is not refused. */
static int sample_total(Ctx* c, unsigned long long& m) {
  TsTotal t{};
  int rc = hip_check(c, hipMemcpyAsync(&t, c->ts.cnt.ptr, sizeof t, hipMemcpyDeviceToHost, c->stream), "dl");
  if (!rc) rc = hip_check(c, hipStreamSynchronize(c->stream), "sync");
  if (rc) return rc;
  if (t.too_many || t.n > HCS_TS_MAX)
    return set_err(c, HCS_ERR_LIMIT, "sensor: sample_resolution asks for more than 2^32 - 1 samples");
  m = t.n;
  return HCS_OK;
}

int hcs_taxel_sensor_update(hcs_ctx* h, const hcs_taxel_sensor* S, double* values, int64_t* nsamples) {
  if (!h || !S || !values || S->ntaxels < 0 || (S->ntaxels > 0 && !S->taxels) || S->method < 0 || S->method > 3 ||
      S->sample_method < 0 || S->sample_method > 1 || !(S->sample_resolution > 0) || !(S->include_margin >= 0))
    return HCS_ERR_ARG;
  Ctx* c = &h->c;
  if (!c->last_valid)
    return set_err(c, HCS_ERR_STATE, "hcs_taxel_sensor_update needs a contact step run with keep_polygons = 1");
  int rc = hip_check(c, hipSetDevice(c->device), "hipSetDevice");
  if (rc) return rc;
  hipStream_t s = c->stream;
  TaxelSensorBufs& B = c->ts;
  unsigned ntri = 0;
  if ((rc = sensor_fans(c, S->geom, ntri))) return rc;
  /* samples */
  unsigned long long m = 0;
  unsigned *nsurf = nullptr, *soff = nullptr;
  int* surf0 = nullptr;
  if (ntri > 0 && S->sample_method == 0) {
    const dim3 g((ntri + 255) / 256);
    const unsigned* soff32 = (const unsigned*)B.soff.ptr;
    hipLaunchKernelGGL(k_ts_count, g, dim3(256), 0, s, (const double*)B.tris.ptr, (int64_t)ntri, S->sample_resolution,
                       HCS_TS_MAX / ntri, (unsigned*)B.scnt.ptr);
    if ((rc = ensure(c, B.tmp, std::max<size_t>(scan_temp_bytes((long long)ntri + 2), 8)))) return rc;
    /* offsets, their end, and the end plus cnt[ntri] */
    if (exclusive_scan_u32(s, (const unsigned*)B.scnt.ptr, (unsigned*)B.soff.ptr, (long long)ntri + 2, B.tmp.ptr,
                           B.tmp.bytes) != 0)
      return set_err(c, HCS_ERR_LIMIT, "sensor: too many triangles to scan");
    unsigned end[2] = {0, 0};
    rc = hip_check(c, hipMemcpyAsync(end, soff32 + ntri, sizeof end, hipMemcpyDeviceToHost, s), "dl");
    if (!rc) rc = hip_check(c, hipStreamSynchronize(s), "sync");
    if (rc) return rc;
    m = end[0];
    if (end[1] != end[0]) {
      hipLaunchKernelGGL(k_ts_sum, g, dim3(256), 0, s, (const double*)B.tris.ptr, (int64_t)ntri, S->sample_resolution,
                         (TsTotal*)B.cnt.ptr);
      if ((rc = sample_total(c, m))) return rc;
    }
  } else if (ntri > 0) {
    /* areas and prefix sums; per pair the first triangle (in no order), the
     * sample count and its scan; the surfaces */
    const size_t np1 = c->last_pairs.size() + 1;
    if ((rc = ensure(c, B.area, sizeof(double) * ntri)) || (rc = ensure(c, B.pair_u, sizeof(unsigned) * (3 * np1 + 1))) ||
        (rc = ensure(c, B.tmp, std::max<size_t>(scan_temp_bytes((long long)np1), 8))))
      return rc;
    unsigned* cnt = (unsigned*)B.pair_u.ptr;
    nsurf = cnt + np1, soff = nsurf + 1, surf0 = (int*)(soff + np1);
    launch_fill_u32(s, cnt, 0u, (int)np1 + 1);
    hipLaunchKernelGGL(k_ts_areas, dim3((ntri + 255) / 256), dim3(256), 0, s, (const double*)B.tris.ptr,
                       (const int*)B.surf.ptr, (int64_t)ntri, (double*)B.area.ptr, surf0, nsurf);
    hipLaunchKernelGGL(k_ts_chain, dim3((unsigned)c->last_pairs.size()), dim3(64), 0, s, (const int*)B.surf.ptr,
                       (int64_t)ntri, surf0, nsurf, S->sample_resolution, false, (double*)B.area.ptr, cnt,
                       (TsTotal*)B.cnt.ptr, (const unsigned*)soff, (double*)nullptr, (int2*)nullptr);
    if (exclusive_scan_u32(s, cnt, soff, (long long)np1, B.tmp.ptr, B.tmp.bytes) != 0)
      return set_err(c, HCS_ERR_LIMIT, "sensor: too many pairs to scan");
    if ((rc = sample_total(c, m))) return rc;
  }
  if (nsamples) *nsamples = (int64_t)m;
  if (m == 0) {
    for (int i = 0; i < S->ntaxels; ++i) values[i] = 0.0;
    return HCS_OK;
  }
  if ((rc = ensure(c, B.P, sizeof(double) * 3 * m)) || (rc = ensure(c, B.E, sizeof(double) * m)) ||
      (rc = ensure(c, B.taxel, sizeof(double) * 3 * std::max(1, S->ntaxels))) ||
      (rc = ensure(c, B.val, sizeof(double) * std::max(1, S->ntaxels))))
    return rc;
  if (S->sample_method == 0)
    hipLaunchKernelGGL(k_ts_gen, dim3((ntri + 255) / 256), dim3(256), 0, s, (const double*)B.tris.ptr, (int64_t)ntri,
                       S->sample_resolution, (const unsigned*)B.soff.ptr, (double*)B.P.ptr, (double*)B.E.ptr);
  else {
    if ((rc = ensure(c, B.acc, (sizeof(double) + sizeof(int2)) * m))) return rc;
    double* acc = (double*)B.acc.ptr;
    int2* range = (int2*)(acc + m);
    hipLaunchKernelGGL(k_ts_chain, dim3((unsigned)c->last_pairs.size()), dim3(64), 0, s, (const int*)B.surf.ptr,
                       (int64_t)ntri, surf0, nsurf, S->sample_resolution, true, (double*)B.area.ptr,
                       (unsigned*)nullptr, (TsTotal*)nullptr, (const unsigned*)soff, acc, range);
    hipLaunchKernelGGL(k_ts_draw, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, (const double*)B.tris.ptr,
                       (const double*)B.area.ptr, (const double*)acc, (const int2*)range, (int64_t)m,
                       (double*)B.P.ptr, (double*)B.E.ptr);
  }
  if (S->ntaxels == 0) return hip_check(c, hipGetLastError(), "samples");
  TsTaxelArgs a;
  std::memcpy(a.X, S->X_W_sensor, sizeof a.X);
  a.margin = S->include_margin, a.res = S->sample_resolution, a.method = S->method, a.visualize = S->visualize != 0;
  rc = hip_check(c, hipMemcpyAsync(B.taxel.ptr, S->taxels, sizeof(double) * 3 * S->ntaxels, hipMemcpyHostToDevice, s),
                 "upload taxels");
  if (!rc)
    rc = hip_check(c, hipMemcpyAsync(B.val.ptr, values, sizeof(double) * S->ntaxels, hipMemcpyHostToDevice, s),
                   "upload values");
  if (rc) return rc;
  const int nx = S->ntaxels, nslice = ts_slices(nx, (int64_t)m);
  if ((rc = ensure(c, B.hits, sizeof(TsPart) * (size_t)nx * nslice))) return rc;
  TsPart* part = (TsPart*)B.hits.ptr;
  const dim3 grid((nx + HCS_TS_TX - 1) / HCS_TS_TX, nslice), cgrid((nx + 15) / 16);
  const double *P = (const double*)B.P.ptr, *E = (const double*)B.E.ptr;
  if (a.method == 0) {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_ts_taxel<true>), grid, dim3(64), 0, s, P, E, (int64_t)m, a,
                       (const double*)B.taxel.ptr, nx, part);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_ts_combine<true>), cgrid, dim3(64), 0, s, (const TsPart*)part, nslice, nx, a,
                       E, (double*)B.val.ptr);
  } else {
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_ts_taxel<false>), grid, dim3(64), 0, s, P, E, (int64_t)m, a,
                       (const double*)B.taxel.ptr, nx, part);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_ts_combine<false>), cgrid, dim3(64), 0, s, (const TsPart*)part, nslice, nx, a,
                       E, (double*)B.val.ptr);
  }
  rc = hip_check(c, hipGetLastError(), "taxel sensor");
  if (!rc)
    rc = hip_check(c, hipMemcpyAsync(values, B.val.ptr, sizeof(double) * S->ntaxels, hipMemcpyDeviceToHost, s), "dl");
  if (!rc) rc = hip_check(c, hipStreamSynchronize(s), "sync");
  return rc;
}

int hcs_curved_sensor_update(hcs_ctx* h, const hcs_curved_sensor* S, double* values) {
  if (!h || !S || !values || S->ntaxels < 0 || S->nsamples < 0 || !(S->include_margin >= 0) ||
      (S->ntaxels > 0 && !S->taxel_ptr) || (S->nsamples > 0 && (!S->points || !S->normals)))
    return HCS_ERR_ARG;
  Ctx* c = &h->c;
  if (S->ntaxels == 0) return HCS_OK;
  const int nnz = S->taxel_ptr[S->ntaxels];
  if (S->taxel_ptr[0] != 0 || nnz < 0 || (nnz > 0 && (!S->sample_idx || !S->weights)))
    return set_err(c, HCS_ERR_ARG, "invalid taxel sample lists");
  for (int i = 0; i < S->ntaxels; ++i)
    if (S->taxel_ptr[i + 1] < S->taxel_ptr[i]) return set_err(c, HCS_ERR_ARG, "taxel_ptr must be non-decreasing");
  for (int k = 0; k < nnz; ++k)
    if (S->sample_idx[k] < 0 || S->sample_idx[k] >= S->nsamples)
      return set_err(c, HCS_ERR_ARG, "sample index out of range");
  if (!c->last_valid)
    return set_err(c, HCS_ERR_STATE, "hcs_curved_sensor_update needs a contact step run with keep_polygons = 1");
  int rc = hip_check(c, hipSetDevice(c->device), "hipSetDevice");
  if (rc) return rc;
  hipStream_t s = c->stream;
  TaxelSensorBufs& B = c->ts;
  unsigned ntri = 0;
  if ((rc = sensor_fans(c, S->geom, ntri))) return rc;
  if (ntri == 0) {
    /* no contact surface touches the sensor (curved_sensor.cpp:434-438) */
    for (int i = 0; i < S->ntaxels; ++i) values[i] = 0.0;
    return HCS_OK;
  }
  const int m = S->nsamples;
  const size_t m1 = (size_t)std::max(1, m), n1 = (size_t)S->ntaxels, z1 = (size_t)std::max(1, nnz);
  const int nslice = cs_slices(m, ntri);
  if ((rc = ensure(c, B.P, sizeof(double) * 6 * m1)) || (rc = ensure(c, B.E, sizeof(double) * m1)) ||
      (rc = ensure(c, B.mask, m1)) || (rc = ensure(c, B.taxel, sizeof(double) * z1)) ||
      (rc = ensure(c, B.val, sizeof(double) * n1)) || (rc = ensure(c, B.scnt, sizeof(int) * (n1 + 1))) ||
      (rc = ensure(c, B.soff, sizeof(int) * z1)) || (rc = ensure(c, B.hits, sizeof(CsHit) * m1 * nslice)))
    return rc;
  double* pts = (double*)B.P.ptr;
  rc = hip_check(c, hipMemcpyAsync(pts, S->points, sizeof(double) * 3 * m, hipMemcpyHostToDevice, s), "ul");
  if (!rc)
    rc = hip_check(c, hipMemcpyAsync(pts + 3 * m1, S->normals, sizeof(double) * 3 * m, hipMemcpyHostToDevice, s), "ul");
  if (!rc)
    rc = hip_check(c, hipMemcpyAsync(B.scnt.ptr, S->taxel_ptr, sizeof(int) * (n1 + 1), hipMemcpyHostToDevice, s), "ul");
  if (!rc && nnz > 0)
    rc = hip_check(c, hipMemcpyAsync(B.soff.ptr, S->sample_idx, sizeof(int) * nnz, hipMemcpyHostToDevice, s), "ul");
  if (!rc && nnz > 0)
    rc = hip_check(c, hipMemcpyAsync(B.taxel.ptr, S->weights, sizeof(double) * nnz, hipMemcpyHostToDevice, s), "ul");
  if (rc) return rc;
  CsArgs a;
  std::memcpy(a.X, S->X_W_sensor, sizeof a.X);
  a.margin = S->include_margin;
  if (m > 0) {
    hipLaunchKernelGGL(k_cs_rays, dim3((m + 63) / 64, nslice), dim3(64), 0, s, (const double*)B.tris.ptr, (int64_t)ntri,
                       a, pts, pts + 3 * m1, m, (CsHit*)B.hits.ptr);
    hipLaunchKernelGGL(k_cs_hits, dim3((m + 15) / 16), dim3(64), 0, s, (const double*)B.tris.ptr,
                       (const CsHit*)B.hits.ptr, nslice, a.margin, m, (double*)B.E.ptr, (unsigned char*)B.mask.ptr);
  }
  hipLaunchKernelGGL(k_cs_taxels, dim3((S->ntaxels + 63) / 64), dim3(64), 0, s, (const int*)B.scnt.ptr,
                     (const int*)B.soff.ptr, (const double*)B.taxel.ptr, S->ntaxels, (const double*)B.E.ptr,
                     (const unsigned char*)B.mask.ptr, (double*)B.val.ptr);
  rc = hip_check(c, hipGetLastError(), "curved sensor");
  if (!rc)
    rc = hip_check(c, hipMemcpyAsync(values, B.val.ptr, sizeof(double) * n1, hipMemcpyDeviceToHost, s), "dl");
  if (!rc) rc = hip_check(c, hipStreamSynchronize(s), "sync");
  return rc;
}

}  // extern "C"
