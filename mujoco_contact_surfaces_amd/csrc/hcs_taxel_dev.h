/*
 * hcs_taxel_dev.h -- device code of the flat tactile sensor sampling
 * (FlatTactileSensor::bvh_update,
 * mujoco_contact_surface_sensors/src/flat_tactile_sensor.cpp:262-402): the
 * per-taxel samplers shared by the plain and batched kernels of
 * hcs_taxels.hip, in a header so the CPU tests can build them too.
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hcs_device.h"
#include "hcs_kernels.h"

#pragma clang fp contract(off)

namespace hcs {

/* The taxels that polygon P's vertices span.  All eight vertex slots are read
 * at once (a record holds them all): a loop to n waited for memory at every
 * vertex. */
__device__ inline void footprint(const double* P, const TaxelGridDev& g, int& x0, int& x1, int& y0, int& y1) {
  const int n = (int)P[0];
  double v[24];
#pragma unroll
  for (int i = 0; i < 24; ++i) v[i] = P[1 + i];
  double lo[2] = {1e300, 1e300}, hi[2] = {-1e300, -1e300};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const double d[3] = {v[3 * i] - g.X[9], v[3 * i + 1] - g.X[10], v[3 * i + 2] - g.X[11]};
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const double l = (g.X[c] * d[0] + g.X[3 + c] * d[1]) + g.X[6 + c] * d[2];
      lo[c] = i < n ? fmin(lo[c], l) : lo[c], hi[c] = i < n ? fmax(hi[c], l) : hi[c];
    }
  }
  const double m = 1e-9;
  x0 = (int)floor((lo[0] - m + g.xs) / g.res);
  x1 = (int)floor((hi[0] + m + g.xs) / g.res);
  y0 = (int)floor((lo[1] - m + g.ys) / g.res);
  y1 = (int)floor((hi[1] + m + g.ys) / g.res);
  x0 = max(x0, 0), y0 = max(y0, 0), x1 = min(x1, g.cx - 1), y1 = min(y1, g.cy - 1);
}

__device__ inline int64_t pkey(const int64_t* key, int q) {
  return (key[3 * q] << 42) | (key[3 * q + 1] << 21) | key[3 * q + 2];
}

/* One workgroup per taxel; samples strided over the threads, each thread
 * sums its samples in index order, then a fixed tree reduction.  T = Dual
 * carries one tangent direction: polygon tangents in ptan, sensor pose
 * tangent in Xd (the hit triangle is chosen on primal values). */
template <class T>
__device__ inline T ld(const double* v, const double* d, size_t i);
template <>
__device__ inline double ld<double>(const double* v, const double*, size_t i) {
  return v[i];
}
template <>
__device__ inline Dual ld<Dual>(const double* v, const double* d, size_t i) {
  return Dual(v[i], d[i]);
}

/* Polygons of one chunk of a taxel's list, staged in LDS for its rays: the
 * vertices (v[8] = the centroid C) and, per fan triangle (v_k, v_k+1, C),
 * the sample-index ranges [i0, i1] x [j0, j1] (i0 / j0 in the low, i1 / j1
 * in the high 16 bits) outside of which no ray of the taxel can hit it, so a
 * ray runs the Moeller-Trumbore test only on the fans whose range holds it,
 * on vertices read from LDS. */
#define HCS_TX_CHUNK 64
struct TxStage {
  double v[HCS_TX_CHUNK][9][3];
  uint2 rng[HCS_TX_CHUNK][8];
  int q[HCS_TX_CHUNK], nv[HCS_TX_CHUNK];
  int64_t kq[HCS_TX_CHUNK];
};

/* The sample-index ranges of the fans of polygon P for taxel (x, y).
 *  - |a| < 1e-10 (a = e1 . (D x e2), the same expression the hit test
 *    rejects on): no ray can hit; empty range.
 *  - |a| < 1e-3 max(|e1|, |e2|)^2 (nearly edge-on to the rays): every ray.
 *  - otherwise the rays whose sensor-plane position lies within m of the
 *    fan's projected box, m = 1e-9 (1 + extent + height gap).  For such a
 *    triangle the computed barycentrics err by less than ~7e-13 (L + |s|) / L
 *    (L the longest edge, s = origin - v0), so an accepted ray lies within
 *    ~7e-13 (L + |s|) of the projected triangle: m is three orders wider, and
 *    the floor / ceil below add up to one more sample on each side. */
__device__ inline void stage_fans(const double (*vv)[3], int nv, const TaxelGridDev& g, int x, int y, uint2* rng) {
  const int S = g.S;
  const double rSR = g.res / S;
  const double Dv[3] = {-g.X[2], -g.X[5], -g.X[8]};
  const double ox = -g.xs + x * g.res + 0.5 * rSR, oy = -g.ys + y * g.res + 0.5 * rSR, oz = 1.5 * g.zs;
  for (int k = 0; k < nv; ++k) {
    const int k1 = (k + 1 == nv) ? 0 : k + 1;
    const double* v0 = vv[k];
    const double* v1 = vv[k1];
    const double* v2 = vv[8];
    double e1[3] = {v1[0] - v0[0], v1[1] - v0[1], v1[2] - v0[2]};
    double e2[3] = {v2[0] - v0[0], v2[1] - v0[1], v2[2] - v0[2]};
    double h[3];
    cross3(Dv, e2, h);
    const double a = dot3(e1, h);
    const double L2 = fmax(dot3(e1, e1), dot3(e2, e2));
    uint2 r;
    if (fabs(a) < 1e-10) {
      r = make_uint2(1u, 1u); /* i0 = 1 > i1 = 0: empty */
    } else if (fabs(a) < 1e-3 * L2) {
      r = make_uint2((unsigned)(S - 1) << 16, (unsigned)(S - 1) << 16);
    } else {
      /* the fan's box in the sensor frame (x, y), and its height gap */
      double lx = 1e300, hx = -1e300, ly = 1e300, hy = -1e300, gap = 0.0;
      for (int t = 0; t < 3; ++t) {
        const double* w = t == 0 ? v0 : (t == 1 ? v1 : v2);
        const double d[3] = {w[0] - g.X[9], w[1] - g.X[10], w[2] - g.X[11]};
        const double px = (g.X[0] * d[0] + g.X[3] * d[1]) + g.X[6] * d[2];
        const double py = (g.X[1] * d[0] + g.X[4] * d[1]) + g.X[7] * d[2];
        const double pz = (g.X[2] * d[0] + g.X[5] * d[1]) + g.X[8] * d[2];
        lx = fmin(lx, px), hx = fmax(hx, px), ly = fmin(ly, py), hy = fmax(hy, py);
        gap = fmax(gap, fabs(oz - pz));
      }
      const double m = 1e-9 * (1.0 + fmax(hx - lx, hy - ly) + gap);
      /* clamp in double before the conversions */
      const double fi0 = fmax(floor((lx - m - ox) / rSR), 0.0), fi1 = fmin(ceil((hx + m - ox) / rSR), S - 1.0);
      const double fj0 = fmax(floor((ly - m - oy) / rSR), 0.0), fj1 = fmin(ceil((hy + m - oy) / rSR), S - 1.0);
      if (!(fi0 <= fi1) || !(fj0 <= fj1)) {
        r = make_uint2(1u, 1u);
      } else {
        r = make_uint2((unsigned)fi0 | ((unsigned)fi1 << 16), (unsigned)fj0 | ((unsigned)fj1 << 16));
      }
    }
    rng[k] = r;
  }
}

/* The value of taxel (x, y): one wave samples it, each lane the rays
 * lane, lane + 64, ... in order, then a fixed butterfly adds the lanes'
 * sums.  The taxel's candidate polygons are list[base .. base + n); when
 * they fit one chunk they are staged once for all rays. */
template <class T>
__device__ inline double sample_cell(const double* __restrict__ poly, const double* __restrict__ ptan,
                                     const int64_t* __restrict__ key, const TaxelGridDev& g,
                                     const double* __restrict__ Xd, unsigned base, unsigned n,
                                     const int* __restrict__ list, int x, int y) {
  __shared__ TxStage L;
  const int S = g.S;
  const double rSR = g.res / S;
  const double rmean = 1. / (S * S);
  const double di_factor = g.res / S;
  const double sub_halfwidth = di_factor / 2.0 - g.res / 2.0;
  const double max_dist = 1.41421356237 * g.res / 2.0;
  T X[12];
#pragma unroll
  for (int i = 0; i < 12; ++i) X[i] = ld<T>(g.X, Xd, i);
  const T nrm[3] = {X[2], X[5], X[8]};
  double rsigma_squared = 0, rtukey = 0;
  if (g.window == 1) rsigma_squared = 0.5 / (g.sigma * g.sigma);
  if (g.window == 2) rtukey = 1. / g.sigma * S * S;
  const double PI = 3.14159265358979323846;
  T acc = T(0.0);
  const int lane = threadIdx.x & 63;
  const bool one_chunk = n <= HCS_TX_CHUNK;
  auto stage = [&](unsigned c0, unsigned cn) {
    for (unsigned l = lane; l < cn; l += 64) {
      const int q = list[base + c0 + l];
      const double* P = poly + (size_t)q * HCS_PREC;
      L.q[l] = q;
      L.nv[l] = min((int)P[0], 8);
      L.kq[l] = pkey(key, q);
      for (int k = 0; k < 27; ++k) L.v[l][k / 3][k % 3] = k < 24 ? P[1 + k] : P[33 + k - 24];
      stage_fans(L.v[l], L.nv[l], g, x, y, L.rng[l]);
    }
  };
  if (one_chunk) {
    stage(0, n);
    __syncthreads();
  }
  /* rays in rounds of 64 (every lane runs every round, so the staging
   * barriers are reached by all) */
  for (int s0 = 0; s0 < S * S; s0 += 64) {
    const int s = s0 + lane;
    const bool active = s < S * S;
    const int i = active ? s / S : 0, j = active ? s % S : 0;
    T loc[3] = {T(-g.xs + x * g.res + i * rSR + 0.5 * rSR), T(-g.ys + y * g.res + j * rSR + 0.5 * rSR),
                T(1.5 * g.zs)};
    T pt[3];
    xform(X, loc, pt);
    T O[3], D[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) O[c] = pt[c] + nrm[c] * 1e-8, D[c] = -nrm[c];
    double best_t = 1e30;
    int64_t bkey = INT64_MAX;
    int bk = 0, bq = -1;
    const double Ov[3] = {val(O[0]), val(O[1]), val(O[2])}, Dv[3] = {val(D[0]), val(D[1]), val(D[2])};
    for (unsigned c0 = 0; c0 < n; c0 += HCS_TX_CHUNK) {
      const unsigned cn = (n - c0) < HCS_TX_CHUNK ? (n - c0) : HCS_TX_CHUNK;
      if (!one_chunk) {
        __syncthreads();
        stage(c0, cn);
        __syncthreads();
      }
      if (!active) continue;
      for (unsigned l = 0; l < cn; ++l) {
        const int nv = L.nv[l];
        const int q = L.q[l];
        const int64_t kq = L.kq[l];
        for (int k = 0; k < nv; ++k) {
          const uint2 r = L.rng[l][k];
          if (i < (int)(r.x & 0xffffu) || i > (int)(r.x >> 16) || j < (int)(r.y & 0xffffu) || j > (int)(r.y >> 16))
            continue;
          const int k1 = (k + 1 == nv) ? 0 : k + 1;
          const double* v0 = L.v[l][k];
          const double* v1 = L.v[l][k1];
          const double* v2 = L.v[l][8];
          double e1[3] = {v1[0] - v0[0], v1[1] - v0[1], v1[2] - v0[2]};
          double e2[3] = {v2[0] - v0[0], v2[1] - v0[1], v2[2] - v0[2]};
          double h[3];
          cross3(Dv, e2, h);
          const double a = dot3(e1, h);
          if (fabs(a) < 1e-10) continue;
          const double f = 1.0 / a;
          double sv[3] = {Ov[0] - v0[0], Ov[1] - v0[1], Ov[2] - v0[2]};
          const double u = f * dot3(sv, h);
          if (u < 0.0 || u > 1.0) continue;
          double qv[3];
          cross3(sv, e1, qv);
          const double v = f * dot3(Dv, qv);
          if (v < 0.0 || u + v > 1.0) continue;
          const double t = f * dot3(e2, qv);
          if (!(t > 0.0)) continue;
          const bool better = t < best_t || (t == best_t && (kq < bkey || (kq == bkey && k < bk)));
          if (better) best_t = t, bkey = kq, bk = k, bq = q;
        }
      }
    }
    if (!active) continue;
    if (bq >= 0 && best_t < 1.5 * g.zs && best_t > 0.0) {
      /* Moeller-Trumbore on the chosen triangle, in T arithmetic */
      const size_t pb = (size_t)bq * HCS_PREC;
      const int nv = (int)poly[pb];
      const int k1 = (bk + 1 == nv) ? 0 : bk + 1;
      T v0[3], v1[3], v2[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        v0[c] = ld<T>(poly, ptan, pb + 1 + 3 * bk + c);
        v1[c] = ld<T>(poly, ptan, pb + 1 + 3 * k1 + c);
        v2[c] = ld<T>(poly, ptan, pb + 33 + c);
      }
      T e1[3] = {v1[0] - v0[0], v1[1] - v0[1], v1[2] - v0[2]};
      T e2[3] = {v2[0] - v0[0], v2[1] - v0[1], v2[2] - v0[2]};
      T h[3];
      cross3(D, e2, h);
      const T f = T(1.0) / dot3(e1, h);
      T sv[3] = {O[0] - v0[0], O[1] - v0[1], O[2] - v0[2]};
      const T u = f * dot3(sv, h);
      T qv[3];
      cross3(sv, e1, qv);
      const T v = f * dot3(D, qv);
      const T pa = ld<T>(poly, ptan, pb + 25 + bk), pbb = ld<T>(poly, ptan, pb + 25 + k1),
              pc = ld<T>(poly, ptan, pb + 36);
      const T b0 = T(1.0) - u - v;
      const T raw = ((b0 * pa + u * pbb) + v * pc) * rmean;
      double weight = 1.0;
      if (g.window == 1) {
        const double dist = hypot(di_factor * i + sub_halfwidth, di_factor * j + sub_halfwidth) / max_dist;
        weight = exp(-(dist * dist) * rsigma_squared);
      } else if (g.window == 2) {
        const int ni = S / 2 - abs(S / 2 - i), nj = S / 2 - abs(S / 2 - j);
        if (ni <= g.sigma * S / 2) weight *= 0.5 * (1. - cos(2. * PI * ni * rtukey));
        if (nj <= g.sigma * S / 2) weight *= 0.5 * (1. - cos(2. * PI * nj * rtukey));
      } else if (g.window == 3) {
        const double inv = 1 - hypot(di_factor * i + sub_halfwidth, di_factor * j + sub_halfwidth) / max_dist;
        weight = inv * inv;
      }
      acc = acc + weight * raw;
    }
  }
  double v = ptan ? tangent(acc) : val(acc);
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = v + __shfl_xor(v, o, 64);
  return __shfl(v, 0, 64);
}

/* ---- fan-major sampling (double, S^2 <= HCS_TX_RAYS): a lane takes a fan
 * triangle and runs the hit test on the rays of its sample range only; the
 * nearest hit per ray is found with LDS atomics: the least t (its IEEE bits
 * order like t, t > 0), then among hits at that t the least (polygon key,
 * fan index), the tie rule of the ray-major loop above.
 *
 * The first pass also records, per ray, the fan whose atomic lowered t
 * (the owner) and flags a ray when a hit matched the t already there (a
 * tie).  The sum over the rays then evaluates each ray's owner; a ray whose
 * owner's t is its least t and that has no tie is settled.  Only if some ray
 * is not (rare), a second pass finds the least key among the hits at its
 * least t, and the sum is made again.  Every hit test is the ray-major loop's
 * arithmetic on the same values, so the chosen triangle, and the taxel, are
 * the same.
 *
 * Bound by FP64 instructions and the latency of their chains at 2 waves per
 * SIMD (207 VGPRs; held to 168 it spills and is no faster): 45% of the issue
 * slots with 76% of the lanes active, the waves waiting half of the time; so by
 * the hit tests and ranges a fan takes and by how evenly they fill the lanes.  A
 * fan covers 2 to 4 rays: sample ranges that end at the last ray inside (they
 * were rounded outward by up to a sample on each side), one evaluation per ray
 * (there were two) and row cuts without divisions by the spacing took 1024
 * pads of 16 x 16 taxels from 1.90 to 1.17 ms, and sharing out the rays of the
 * small fans to 0.85 ms; one pad went from 132 to 52 us, and with four waves a
 * taxel to 22 us. */
#define HCS_TX_RAYS 576
/* A fan whose range holds at most this many rays has them all tested; a larger
 * one has each row cut to the fan first, at the price of its setup again for
 * each row.  (24: 0.98 ms on the 1024 pads, 40: 0.93, 64: 0.86, 128: 0.86; on
 * a coarse surface, fans of 100 rays and more, 37, 36 and 39 us for 32, 64 and
 * 128.) */
#define HCS_TX_SMALL 64
static_assert(HCS_TX_RAYS == 24 * 24 && 64 * HCS_TX_SMALL < 65536, "codes of the fan-major sampler");
/* A fan's id: its polygon's position in the taxel's list * 16 + its vertex k * 2
 * + whether the next vertex is the first.  In a list of up to HCS_TX_POLYS no id
 * is HCS_TX_NONE; the callers take the ray-major sampler where a list could be
 * longer (as many kept polygons are 86 GB). */
#define HCS_TX_POLYS ((1ll << 28) - 1)
#define HCS_TX_NONE 0xffffffffu
__device__ inline unsigned fan_id(unsigned pos, int k, int k1) {
  return pos << 4 | (unsigned)k << 1 | (k1 == 0 ? 1u : 0u);
}
__device__ inline unsigned fan_pos(unsigned id) { return id >> 4; }
__device__ inline int fan_k(unsigned id) { return (int)(id >> 1 & 7); }
__device__ inline int fan_k1(unsigned id) { return id & 1 ? 0 : fan_k(id) + 1; }

/* A taxel's rays (7.5 KB) and each wave's fans (6 KB). */
struct TxHits {
  unsigned long long tmin[HCS_TX_RAYS];
  /* first pass: the fan of the hit that lowered t last; second pass: of the
   * least (key, fan) among the hits at tmin, HCS_TX_NONE before the first */
  unsigned own[HCS_TX_RAYS];
  unsigned char flag[HCS_TX_RAYS]; /* the ray needs the second pass */
  int again;
};
struct TxScatter {
  int q[HCS_TX_CHUNK];
  unsigned short fan0[HCS_TX_CHUNK + 1];
  /* the round's fans, one per lane: v0, e1, e2, f; id within the chunk; first
   * row, first column and width of the range (5 bits each); rays of the small
   * fans before it, and rows of the large ones (16 bits each) */
  double fan[10][64];
  unsigned short id[64], box[64];
  unsigned pre[64];
};

/* Orders the LDS accesses of one wave's lanes (the LDS serves a wave in
 * order): waves of a taxel take different numbers of rounds. */
__device__ inline void wave_sync() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#else
  __syncthreads();
#endif
}

/* One taxel's ray grid: ray (i, j) starts at (bx + i step + step / 2,
 * by + j step + step / 2, oz) of the sensor frame; inv = 1 / step for the
 * ranges, and the rounding of world coordinates at the sensor. */
struct TxRays {
  double step, inv, bx, by, oz, far;
};
__device__ inline TxRays taxel_rays(const TaxelGridDev& g, int x, int y) {
  TxRays r;
  r.step = g.res / g.S;
  r.inv = 1.0 / r.step;
  r.bx = -g.xs + x * g.res, r.by = -g.ys + y * g.res, r.oz = 1.5 * g.zs;
  r.far = 1e-14 * (fabs(g.X[9]) + fabs(g.X[10]) + fabs(g.X[11]));
  return r;
}

/* Hit-test constants of the fan (v_k, v_k1, C) of polygon P (the ray-major loop's e1, e2,
 * f = 1 / a with a = e1 . (D x e2)) and its sample range; false when no ray can hit it
 * (|a| < 1e-10, which the hit test rejects, or an empty range). */
struct TxFan {
  double v0[3], e1[3], e2[3], f;
  double px[3], py[3], m; /* the fan in the sensor's (x, y), the range margin */
  int i0, i1, j0, j1;
  bool rows; /* per-row ranges apply (false: the fan gets every ray) */
};
__device__ inline bool fan_setup(const double* P, int k, int k1, const TaxelGridDev& g, const TxRays& R, TxFan& c) {
  const int S = g.S;
  const double Dv[3] = {-g.X[2], -g.X[5], -g.X[8]};
  const double* v0 = P + 1 + 3 * k;
  const double* v1 = P + 1 + 3 * k1;
  const double* v2 = P + 33;
  double w[3][3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    w[0][d] = v0[d], w[1][d] = v1[d], w[2][d] = v2[d];
    c.v0[d] = w[0][d], c.e1[d] = w[1][d] - w[0][d], c.e2[d] = w[2][d] - w[0][d];
  }
  double h[3];
  cross3(Dv, c.e2, h);
  const double a = dot3(c.e1, h);
  if (fabs(a) < 1e-10) return false;
  c.f = 1.0 / a;
  const double L2 = fmax(dot3(c.e1, c.e1), dot3(c.e2, c.e2));
  c.rows = false;
  if (fabs(a) < 1e-3 * L2) {
    c.i0 = c.j0 = 0, c.i1 = c.j1 = S - 1;
    return true;
  }
  /* the rays within m of the fan's box, m the margin of stage_fans (and of
   * world coordinates far from the origin): three orders above the rounding
   * of an accepted hit, so also far above that of these indexes, and no
   * sample is added for it.  (A grid spacing at which it were not keeps a
   * sample on each side.) */
  double lx = 1e300, hx = -1e300, ly = 1e300, hy = -1e300, gap = 0.0;
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const double d[3] = {w[t][0] - g.X[9], w[t][1] - g.X[10], w[t][2] - g.X[11]};
    const double px = (g.X[0] * d[0] + g.X[3] * d[1]) + g.X[6] * d[2];
    const double py = (g.X[1] * d[0] + g.X[4] * d[1]) + g.X[7] * d[2];
    const double pz = (g.X[2] * d[0] + g.X[5] * d[1]) + g.X[8] * d[2];
    c.px[t] = px, c.py[t] = py;
    lx = fmin(lx, px), hx = fmax(hx, px), ly = fmin(ly, py), hy = fmax(hy, py);
    gap = fmax(gap, fabs(R.oz - pz));
  }
  const double m = 1e-9 * (1.0 + fmax(hx - lx, hy - ly) + gap) + R.far;
  c.m = m;
  c.rows = true;
  const double ox = R.bx + 0.5 * R.step, oy = R.by + 0.5 * R.step;
  const double slack = m * R.inv > 1e-12 * S ? 0.0 : 1.0;
  const double fi0 = fmax(ceil((lx - m - ox) * R.inv) - slack, 0.0);
  const double fi1 = fmin(floor((hx + m - ox) * R.inv) + slack, S - 1.0);
  const double fj0 = fmax(ceil((ly - m - oy) * R.inv) - slack, 0.0);
  const double fj1 = fmin(floor((hy + m - oy) * R.inv) + slack, S - 1.0);
  if (!(fi0 <= fi1) || !(fj0 <= fj1)) return false;
  c.i0 = (int)fi0, c.i1 = (int)fi1, c.j0 = (int)fj0, c.j1 = (int)fj1;
  return true;
}

/* The rays of row i (ray x index) that fan c can hold: the fan's y extent
 * over the slab of x within 2m of the row's x (each edge cut to the slab),
 * widened by 2m, within the fan's range [j0, j1]; empty when ja > jb.  The
 * margin m is the fan's range margin, so a row range holds every ray the
 * range holds that the hit test can accept.  (The products with 1 / dx and
 * 1 / step move a bound by a few ulps, against a margin of 1e-9.) */
__device__ inline void fan_row(const TxFan& c, const TaxelGridDev& g, const TxRays& R, int i, int& ja, int& jb) {
  ja = c.j0, jb = c.j1;
  if (!c.rows) return;
  const double ox = R.bx + 0.5 * R.step, oy = R.by + 0.5 * R.step;
  const double xi = ox + i * R.step, xa = xi - 2.0 * c.m, xb = xi + 2.0 * c.m;
  double lo = 1e300, hi = -1e300;
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    const int e1 = e == 2 ? 0 : e + 1;
    const double x0 = c.px[e], y0 = c.py[e], x1 = c.px[e1], y1 = c.py[e1];
    const bool in = !(fmax(x0, x1) < xa || fmin(x0, x1) > xb);
    const double dx = x1 - x0, ix = 1.0 / dx, ta = (xa - x0) * ix, tb = (xb - x0) * ix;
    const bool cut = fabs(dx) > 1e-30;
    const double t0 = cut ? fmin(fmax(fmin(ta, tb), 0.0), 1.0) : 0.0;
    const double t1 = cut ? fmin(fmax(fmax(ta, tb), 0.0), 1.0) : 1.0;
    const double ya = y0 + t0 * (y1 - y0), yb = y0 + t1 * (y1 - y0);
    lo = in ? fmin(lo, fmin(ya, yb)) : lo, hi = in ? fmax(hi, fmax(ya, yb)) : hi;
  }
  if (!(lo <= hi)) {
    ja = 1, jb = 0;
    return;
  }
  const double slack = c.m * R.inv > 1e-12 * g.S ? 0.0 : 1.0;
  const double fa = ceil((lo - 2.0 * c.m - oy) * R.inv) - slack, fb = floor((hi + 2.0 * c.m - oy) * R.inv) + slack;
  ja = fa > (double)ja ? (int)fmin(fa, (double)c.j1 + 1.0) : ja;
  jb = fb < (double)jb ? (int)fmax(fb, (double)c.j0 - 1.0) : jb;
}

/* The origin of ray (i, j) as the ray-major loop computes it: R loc + p +
 * 1e-8 n. */
__device__ inline void ray_origin(const TaxelGridDev& g, const TxRays& R, int i, int j, double* O) {
  const double loc[3] = {R.bx + i * R.step + 0.5 * R.step, R.by + j * R.step + 0.5 * R.step, R.oz};
  double pt[3];
  xform(g.X, loc, pt);
  const double nrm[3] = {g.X[2], g.X[5], g.X[8]};
#pragma unroll
  for (int d = 0; d < 3; ++d) O[d] = pt[d] + nrm[d] * 1e-8;
}

/* The hit of ray (i, j) with a fan (fan_setup's v0, e1, e2, f), as the
 * ray-major loop computes it (direction -n): t > 0, or a negative value. */
__device__ inline double fan_hit(const double* v0, const double* e1, const double* e2, double f,
                                 const TaxelGridDev& g, const TxRays& R, int i, int j) {
  double O[3], h[3];
  ray_origin(g, R, i, j, O);
  const double Dv[3] = {-g.X[2], -g.X[5], -g.X[8]};
  cross3(Dv, e2, h);
  double sv[3] = {O[0] - v0[0], O[1] - v0[1], O[2] - v0[2]};
  const double u = f * dot3(sv, h);
  if (u < 0.0 || u > 1.0) return -1.0;
  double qv[3];
  cross3(sv, e1, qv);
  const double v = f * dot3(Dv, qv);
  if (v < 0.0 || u + v > 1.0) return -1.0;
  const double t = f * dot3(e2, qv);
  return t > 0.0 ? t : -1.0;
}

/* The pressure where ray (i, j) meets the fan (v_k, v_k1, C) of polygon P,
 * which it hits, as the ray-major loop evaluates the chosen triangle; t: the
 * hit's t. */
__device__ inline double fan_pressure(const double* P, int k, int k1, const TaxelGridDev& g, const TxRays& R, int i, int j,
                                      double& t) {
  const double* v0 = P + 1 + 3 * k;
  const double* v1 = P + 1 + 3 * k1;
  const double* v2 = P + 33;
  double O[3];
  ray_origin(g, R, i, j, O);
  const double D[3] = {-g.X[2], -g.X[5], -g.X[8]};
  double e1[3] = {v1[0] - v0[0], v1[1] - v0[1], v1[2] - v0[2]};
  double e2[3] = {v2[0] - v0[0], v2[1] - v0[1], v2[2] - v0[2]};
  double h[3];
  cross3(D, e2, h);
  const double f = 1.0 / dot3(e1, h);
  double sv[3] = {O[0] - v0[0], O[1] - v0[1], O[2] - v0[2]};
  const double u = f * dot3(sv, h);
  double qv[3];
  cross3(sv, e1, qv);
  const double v = f * dot3(D, qv);
  t = f * dot3(e2, qv);
  const double b0 = 1.0 - u - v;
  return (b0 * P[25 + k] + u * P[25 + k1]) + v * P[36];
}

/* The entry of fan f of the staged chunk: the last entry whose first fan
 * is at most f (binary search; every entry has at least one fan). */
__device__ inline int fan_entry(const TxScatter& L, unsigned cn, int f) {
  int l = 0;
  for (int hi = (int)cn - 1; l < hi;) {
    const int mid = (l + hi + 1) >> 1;
    if (L.fan0[mid] <= f) l = mid;
    else hi = mid - 1;
  }
  return l;
}

/* The lane of the round whose rays (shift 0) or rows (shift 16) hold number t:
 * the last one with at most t before it. */
__device__ inline int round_lane(const TxScatter& L, int t, int shift) {
  int l = 0;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) l += (int)(L.pre[l + d] >> shift & 0xffffu) <= t ? d : 0;
  return l;
}

/* Whether fan a comes before fan b (the least key, then the least fan). */
__device__ inline bool fan_before(const int64_t* __restrict__ key, const int* __restrict__ list, unsigned a,
                                  unsigned b) {
  const int64_t ka = pkey(key, list[fan_pos(a)]), kb = pkey(key, list[fan_pos(b)]);
  return ka < kb || (ka == kb && fan_k(a) < fan_k(b));
}

/* A hit of ray s at t by fan id: PASS 0 keeps the least t per ray, PASS 1 the
 * least (key, fan) among hits at that t. */
template <int PASS>
__device__ inline void keep_hit(TxHits& H, const int64_t* __restrict__ key, const int* __restrict__ list, int s,
                                double t, unsigned id) {
  const unsigned long long tb = (unsigned long long)__double_as_longlong(t);
  if (PASS == 0) {
    const unsigned long long old = atomicMin(&H.tmin[s], tb);
    if (tb < old) H.own[s] = id;
    else if (tb == old) H.flag[s] = 1;
  } else if (tb == H.tmin[s]) {
    unsigned cur = __atomic_load_n(&H.own[s], __ATOMIC_RELAXED);
    while ((cur == HCS_TX_NONE || fan_before(key, list, id, cur)) &&
           !__atomic_compare_exchange_n(&H.own[s], &cur, id, false, __ATOMIC_RELAXED, __ATOMIC_RELAXED)) {
    }
  }
}

/* One pass over the fans of list[base + c0 ..] for the wave, 64 fans a round:
 * each lane sets up one fan, then the wave shares the rays of the small fans
 * and the rows of the large ones out evenly.  (A lane that tested its own
 * fan's rays waited for the largest fan of the wave: 29% of the lanes were
 * active.)  The minima do not depend on the order of the hits. */
template <int PASS>
__device__ inline void scatter_chunk(TxHits& H, TxScatter& L, const double* __restrict__ poly,
                                     const int64_t* __restrict__ key, const int* __restrict__ list,
                                     const TaxelGridDev& g, const TxRays& R, unsigned cn, unsigned c0) {
  const int lane = threadIdx.x & 63;
  const int nf = L.fan0[cn];
  for (int f0 = 0; f0 < nf; f0 += 64) {
    const int f = f0 + lane;
    unsigned work = 0;
    if (f < nf) {
      const int l = fan_entry(L, cn, f);
      const int k = f - L.fan0[l];
      const double* P = poly + (size_t)L.q[l] * HCS_PREC;
      const int nv = (int)L.fan0[l + 1] - (int)L.fan0[l], k1 = k + 1 == nv ? 0 : k + 1;
      TxFan c;
      if (fan_setup(P, k, k1, g, R, c)) {
        const int w = c.j1 - c.j0 + 1, h = c.i1 - c.i0 + 1;
        L.id[lane] = (unsigned short)fan_id((unsigned)l, k, k1);
        L.box[lane] = (unsigned short)(c.i0 | c.j0 << 5 | w << 10);
        work = w * h <= HCS_TX_SMALL ? (unsigned)(w * h) : (unsigned)h << 16;
#pragma unroll
        for (int d = 0; d < 3; ++d) L.fan[d][lane] = c.v0[d], L.fan[3 + d][lane] = c.e1[d], L.fan[6 + d][lane] = c.e2[d];
        L.fan[9][lane] = c.f;
      }
    }
    unsigned incl = work;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned t = __shfl(incl, lane >= o ? lane - o : lane, 64);
      if (lane >= o) incl += t;
    }
    const unsigned tot = __shfl(incl, 63, 64);
    L.pre[lane] = incl - work;
    wave_sync();
    for (int t = lane; t < (int)(tot & 0xffffu); t += 64) {
      const int w = round_lane(L, t, 0), box = L.box[w], n = t - (int)(L.pre[w] & 0xffffu);
      const int width = box >> 10, di = (int)(((float)n + 0.5f) / (float)width);
      const int i = (box & 31) + di, j = (box >> 5 & 31) + (n - di * width), s = i * g.S + j;
      if (PASS == 1 && !H.flag[s]) continue;
      const double v0[3] = {L.fan[0][w], L.fan[1][w], L.fan[2][w]};
      const double e1[3] = {L.fan[3][w], L.fan[4][w], L.fan[5][w]};
      const double e2[3] = {L.fan[6][w], L.fan[7][w], L.fan[8][w]};
      const double th = fan_hit(v0, e1, e2, L.fan[9][w], g, R, i, j);
      if (th > 0.0) keep_hit<PASS>(H, key, list, s, th, (c0 << 4) + L.id[w]);
    }
    for (int t = lane; t < (int)(tot >> 16); t += 64) {
      const int w = round_lane(L, t, 16);
      const unsigned id = L.id[w];
      const double* P = poly + (size_t)L.q[fan_pos(id)] * HCS_PREC;
      TxFan c;
      if (!fan_setup(P, fan_k(id), fan_k1(id), g, R, c)) continue;
      const int i = c.i0 + t - (int)(L.pre[w] >> 16);
      int ja, jb;
      fan_row(c, g, R, i, ja, jb);
      for (int j = ja; j <= jb; ++j) {
        const int s = i * g.S + j;
        if (PASS == 1 && !H.flag[s]) continue;
        const double th = fan_hit(c.v0, c.e1, c.e2, c.f, g, R, i, j);
        if (th > 0.0) keep_hit<PASS>(H, key, list, s, th, (c0 << 4) + id);
      }
    }
    wave_sync();
  }
}

/* The taxel's value by W waves: each takes equal shares of the list's
 * polygons (a taxel of a plain call has the chip nearly to itself), and the
 * rays' values are summed in the same order for any W. */
template <int W = 1>
__device__ inline double sample_cell_scatter(const double* __restrict__ poly, const int64_t* __restrict__ key,
                                             const TaxelGridDev& g, unsigned base, unsigned n,
                                             const int* __restrict__ list, int x, int y) {
  __shared__ TxHits H;
  __shared__ TxScatter LW[W];
  const int tid = threadIdx.x, lane = tid & 63, wave = W > 1 ? tid >> 6 : 0;
  TxScatter& L = LW[wave];
  const int S = g.S, nr = S * S;
  const TxRays R = taxel_rays(g, x, y);
  for (int s = tid; s < nr; s += 64 * W) H.tmin[s] = 0x7ff0000000000000ull, H.flag[s] = 0;
  if (tid == 0) H.again = 0;
  __syncthreads();
  list += base;
  auto stage = [&](unsigned c0, unsigned cn) {
    wave_sync();
    /* one entry per lane (cn <= 64): its polygon and fan count, and
     * the first fan of each entry by a prefix sum over the wave */
    unsigned nf = 0;
    if ((unsigned)lane < cn) {
      const int q = list[c0 + lane];
      L.q[lane] = q;
      nf = (unsigned)min((int)poly[(size_t)q * HCS_PREC], 8);
    }
    unsigned incl = nf;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned t = __shfl(incl, lane >= o ? lane - o : lane, 64);
      if (lane >= o) incl += t;
    }
    if ((unsigned)lane < cn) L.fan0[lane] = (unsigned short)(incl - nf);
    if ((unsigned)lane == cn - 1) L.fan0[cn] = (unsigned short)incl;
    wave_sync();
  };
  const unsigned share = (n + W - 1) / W, n0 = min(n, wave * share), n1 = min(n, n0 + share);
  const bool one_chunk = W == 1 && n <= HCS_TX_CHUNK;
  for (unsigned c0 = n0; c0 < n1; c0 += HCS_TX_CHUNK) {
    const unsigned cn = (n1 - c0) < HCS_TX_CHUNK ? (n1 - c0) : HCS_TX_CHUNK;
    stage(c0, cn);
    scatter_chunk<0>(H, L, poly, key, list, g, R, cn, c0);
  }
  __syncthreads();
  /* the weighted pressure of ray s on fan id; t: the hit's */
  const double rmean = 1. / (S * S);
  const double di_factor = g.res / S;
  const double sub_halfwidth = di_factor / 2.0 - g.res / 2.0;
  const double max_dist = 1.41421356237 * g.res / 2.0;
  double rsigma_squared = 0, rtukey = 0;
  if (g.window == 1) rsigma_squared = 0.5 / (g.sigma * g.sigma);
  if (g.window == 2) rtukey = 1. / g.sigma * S * S;
  const double PI = 3.14159265358979323846;
  auto value = [&](int s, unsigned id, double& t) {
    const int i = s / S, j = s % S, q = one_chunk ? L.q[fan_pos(id)] : list[fan_pos(id)];
    const double raw = fan_pressure(poly + (size_t)q * HCS_PREC, fan_k(id), fan_k1(id), g, R, i, j, t) * rmean;
    double weight = 1.0;
    if (g.window == 1) {
      const double dist = hypot(di_factor * i + sub_halfwidth, di_factor * j + sub_halfwidth) / max_dist;
      weight = exp(-(dist * dist) * rsigma_squared);
    } else if (g.window == 2) {
      const int ni = S / 2 - abs(S / 2 - i), nj = S / 2 - abs(S / 2 - j);
      if (ni <= g.sigma * S / 2) weight *= 0.5 * (1. - cos(2. * PI * ni * rtukey));
      if (nj <= g.sigma * S / 2) weight *= 0.5 * (1. - cos(2. * PI * nj * rtukey));
    } else if (g.window == 3) {
      const double inv = 1 - hypot(di_factor * i + sub_halfwidth, di_factor * j + sub_halfwidth) / max_dist;
      weight = inv * inv;
    }
    return weight * raw;
  };
  /* every settled ray's value in place of its t */
  for (int s = tid; s < nr; s += 64 * W) {
    const unsigned long long tb = H.tmin[s];
    double t = -1.0, w = 0.0;
    bool settled = true;
    if (tb != 0x7ff0000000000000ull) {
      if (!H.flag[s]) w = value(s, H.own[s], t);
      settled = t > 0.0 && (unsigned long long)__double_as_longlong(t) == tb;
      if (!(t < 1.5 * g.zs)) w = 0.0;
    }
    if (settled) H.tmin[s] = (unsigned long long)__double_as_longlong(w);
    else H.flag[s] = 1, H.own[s] = HCS_TX_NONE, H.again = 1;
  }
  __syncthreads();
  if (H.again) {
    for (unsigned c0 = n0; c0 < n1; c0 += HCS_TX_CHUNK) {
      const unsigned cn = (n1 - c0) < HCS_TX_CHUNK ? (n1 - c0) : HCS_TX_CHUNK;
      if (!one_chunk) stage(c0, cn);
      scatter_chunk<1>(H, L, poly, key, list, g, R, cn, c0);
    }
    __syncthreads();
    for (int s = tid; s < nr; s += 64 * W)
      if (H.flag[s]) {
        double t, w = 0.0;
        if (__longlong_as_double((long long)H.tmin[s]) < 1.5 * g.zs && H.own[s] != HCS_TX_NONE) w = value(s, H.own[s], t);
        H.tmin[s] = (unsigned long long)__double_as_longlong(w);
      }
    __syncthreads();
  }
  /* the sum, each lane of the first wave its rays in order */
  double acc = 0.0;
  if (W == 1 || wave == 0)
    for (int s = lane; s < nr; s += 64) acc = acc + __longlong_as_double((long long)H.tmin[s]);
  double v = acc;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = v + __shfl_xor(v, o, 64);
  return __shfl(v, 0, 64);
}

}  // namespace hcs
