/*
 * hcs_taxels.hip -- flat tactile sensor sampling on the GPU, FP64.
 *
 * Restates FlatTactileSensor::bvh_update
 * (mujoco_contact_surface_sensors/src/flat_tactile_sensor.cpp:262-402): per
 * taxel (x, y) and sub-sample (i, j) a ray from
 *   R (-xs + x res + (i+1/2) res/S, -ys + y res + (j+1/2) res/S, 1.5 zs) + t
 * offset by 1e-8 along the sensor normal n, direction -n, nearest hit over
 * the kTriangle fans of every contact polygon of the pairs touching the
 * sensor geometry (Moeller-Trumbore as in
 * mujoco_contact_surface_sensors/src/bvh.cpp:49-74, |det| < 1e-10 rejected),
 * accepted when 0 < t < 1.5 zs; value Evaluate(tri, (1-u-v, u, v)) / S^2
 * times the window weight, summed per taxel.
 *
 * Instead of the reference's per-update float32 BVH + TLAS over the contact
 * triangles, all rays are parallel, so the polygons are binned once into the
 * taxel grid by their footprint in the sensor plane; one workgroup per taxel
 * then tests only its bin.  Ties in t are broken by (polygon key, fan index),
 * the canonical polygon order.
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
#include "hcs_taxel_dev.h"

#pragma clang fp contract(off)

using namespace hcs;

namespace hcs {

/* Pairs whose polygons a sensor sees: bits for up to 256 pairs (they travel
 * with the launch), a byte per pair in device memory beyond. */
struct TxPairs {
  unsigned long long bits[4];
  const unsigned char* mask;
  __device__ bool has(int64_t e) const { return mask ? mask[e] != 0 : (bits[e >> 6] >> (e & 63) & 1) != 0; }
};

/* Adds one to counter[cell] for every lane with on set and returns the lane's
 * place; lanes of one cell share an atomic, for the first HCS_TX_SHARE cells
 * (the rest go by themselves).  Neighbouring small polygons lie in few taxels,
 * whose counters share cache lines, and atomics on one line complete one after
 * another; large polygons have their taxels to themselves, and looking for
 * company costs (none / 6 / 10 / 16 / all cells: a pad of 6.8k polygons 46, 17,
 * 13, 13 and 12 us; one of 3 mm polygons under 100 x 100 taxels 12, 21, 25, 30
 * and 38 us).  Called by whole
 * waves. */
#define HCS_TX_SHARE 10
__device__ inline unsigned count_cell(unsigned* __restrict__ counter, int cell, bool on) {
  const int lane = threadIdx.x & 63;
  int lead = lane;
  unsigned rank = 0, n = 1;
  unsigned long long todo = __ballot(on);
  for (int r = 0; r < HCS_TX_SHARE && todo != 0; ++r) {
    const int l = __builtin_ctzll(todo);
    const bool same = on && cell == __shfl(cell, l, 64);
    const unsigned long long m = __ballot(same);
    if (same) lead = l, rank = lane_prefix(m), n = (unsigned)__popcll(m);
    todo &= ~m;
  }
  unsigned base = 0;
  if (on && lane == lead) base = atomicAdd(counter + cell, n);
  return __shfl(base, lead, 64) + rank;
}

/* The taxels of footprint f, numbered base + x + cx y, counted (FILL = 0) or
 * given polygon q (FILL = 1).  Called by whole waves (an empty footprint: no
 * polygon). */
template <int FILL>
__device__ inline void bin_polygon(int q, const int4& f, int cx, int base, unsigned* __restrict__ counter,
                                   const unsigned* __restrict__ off, int* __restrict__ list, int64_t list_cap) {
  int x = f.x, y = f.z;
  bool on = f.x <= f.y && f.z <= f.w;
  while (__any(on)) {
    const int cell = on ? base + x + cx * y : -1;
    const unsigned k = count_cell(counter, cell, on);
    if (FILL && on && (int64_t)off[cell] + k < list_cap) list[off[cell] + k] = q;
    if (++x > f.y) x = f.x, ++y;
    on = on && y <= f.w;
  }
}

/* Binning, one polygon per thread.  FILL = 0 notes the taxels its footprint
 * covers and counts it there; FILL = 1 writes it into their lists.  Bound by
 * the latency of one polygon (a few thousand): 64 threads a block, the record
 * read at once and only in the first pass and shared atomics (count_cell) took
 * the pair of launches from 50 to 13 us (6.8k polygons). */
template <int FILL>
__global__ __launch_bounds__(64) void k_tx_bin(const double* __restrict__ poly, const int64_t* __restrict__ key,
                                               int64_t np, TxPairs pairs, TaxelGridDev g, int4* __restrict__ foot,
                                               unsigned* __restrict__ cnt, const unsigned* __restrict__ off,
                                               int* __restrict__ list, int64_t list_cap) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  int4 f = make_int4(0, -1, 0, -1);
  if (q < np) {
    if (FILL) {
      f = foot[q];
    } else {
      if (pairs.has(key[3 * q])) footprint(poly + q * HCS_PREC, g, f.x, f.y, f.z, f.w);
      foot[q] = f;
    }
  }
  bin_polygon<FILL>((int)q, f, g.cx, 0, cnt, off, list, list_cap);
}

/* Entries of all lists, in 64 bits: their offsets are 32-bit, and a sum beyond
 * that is refused.  Only made where the number of polygons and taxels does not
 * exclude it. */
__device__ inline void add_entries(const int4& f, bool on, unsigned long long* __restrict__ total) {
  const int64_t n = on && f.x <= f.y && f.z <= f.w ? (int64_t)(f.y - f.x + 1) * (f.w - f.z + 1) : 0;
  const int64_t sum = wave_sum_i(n);
  if ((threadIdx.x & 63) == 0 && sum > 0) atomicAdd(total, (unsigned long long)sum);
}
__global__ __launch_bounds__(64) void k_tx_total(const int4* __restrict__ foot, int64_t np,
                                                 unsigned long long* __restrict__ total) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  add_entries(q < np ? foot[q] : make_int4(0, -1, 0, -1), q < np, total);
}
constexpr unsigned long long kMaxEntries = 0xffffffffull;
/* The sum of a k_tx_total / k_txb_total launch made by enqueue(total). */
template <class F>
static int check_entries(Ctx* c, F enqueue) {
  int rc = ensure(c, c->d_tx_total, 8);
  if (rc) return rc;
  unsigned long long* total = (unsigned long long*)c->d_tx_total.ptr;
  launch_fill_u32(c->stream, (unsigned*)total, 0u, 2);
  enqueue(total);
  unsigned long long n = 0;
  rc = hip_check(c, hipMemcpyAsync(&n, total, 8, hipMemcpyDeviceToHost, c->stream), "dl");
  if (!rc) rc = hip_check(c, hipStreamSynchronize(c->stream), "sync");
  if (rc) return rc;
  if (n > kMaxEntries) return set_err(c, HCS_ERR_CAPACITY, "taxel polygon lists exceed 2^32 entries");
  return HCS_OK;
}

/* A taxel's list: off[cell] .. off[cell + 1], or none of it when it does not
 * fit the list buffer (the caller sees the total and runs again). */
__device__ inline unsigned tx_count(const unsigned* __restrict__ off, int cell, int64_t list_cap) {
  const unsigned a = off[cell], b = off[cell + 1];
  return a <= b && (int64_t)b <= list_cap ? b - a : 0u;
}

template <class T>
__global__ __launch_bounds__(64) void k_tx_sample(const double* __restrict__ poly, const double* __restrict__ ptan,
                                                   const int64_t* __restrict__ key, TaxelGridDev g,
                                                   const double* __restrict__ Xd, const unsigned* __restrict__ off,
                                                   const int* __restrict__ list, int64_t list_cap,
                                                   double* __restrict__ out) {
  const int cell = blockIdx.x;
  const int x = cell % g.cx, y = cell / g.cx;
  if (cell == 0 && threadIdx.x == 0) out[gridDim.x] = (double)off[gridDim.x];
  const double v = sample_cell<T>(poly, ptan, key, g, Xd, off[cell], tx_count(off, cell, list_cap), list, x, y);
  if (threadIdx.x == 0) out[x + g.cx * y] = v;
}

/* The same, fan-major (double, S^2 <= HCS_TX_RAYS, np <= HCS_TX_POLYS), W
 * waves per taxel. */
template <int W>
__global__ __launch_bounds__(64 * W) void k_tx_sample_fan(const double* __restrict__ poly, const int64_t* __restrict__ key,
                                                      TaxelGridDev g, const unsigned* __restrict__ off,
                                                      const int* __restrict__ list, int64_t list_cap,
                                                      double* __restrict__ out) {
  const int cell = blockIdx.x;
  const int x = cell % g.cx, y = cell / g.cx;
  if (cell == 0 && threadIdx.x == 0) out[gridDim.x] = (double)off[gridDim.x];
  const double v = sample_cell_scatter<W>(poly, key, g, off[cell], tx_count(off, cell, list_cap), list, x, y);
  if (threadIdx.x == 0) out[x + g.cx * y] = v;
}

/* Bins the polygons of the pairs with seen[e] != 0 into the taxel grid,
 * samples it and returns the taxels in out (host).  ptan/Xd select the tangent
 * pass (nullptr: values).  The counts are scanned on the device and the last
 * kernel writes to pinned memory, so a call waits once; a list buffer that was
 * too small shows in the total that comes with the taxels, and the lists are
 * made again. */
int run_taxels(Ctx* c, const TaxelGridDev& g, const std::vector<unsigned char>& seen, const double* poly,
               const double* ptan, const int64_t* key, int64_t np, const double* Xd, double* out) {
  /* taxels that the kernel writes to pinned memory itself, and that go there
   * by a copy; beyond, straight to the caller */
  constexpr int kDirect = 8192, kPinned = 1 << 20;
  const int ncell = g.cx * g.cy;
  const size_t scan_bytes = scan_temp_bytes((long long)ncell + 1);
  int rc;
  if ((rc = ensure(c, c->d_tx_cnt, sizeof(unsigned) * ((size_t)ncell + 1))) ||
      (rc = ensure(c, c->d_tx_off, sizeof(unsigned) * ((size_t)ncell + 1) + scan_bytes + 8)) ||
      (rc = ensure(c, c->d_tx_foot, sizeof(int4) * (size_t)std::max<int64_t>(1, np))) ||
      (rc = ensure(c, c->d_tx_list, sizeof(int) * (size_t)std::max<int64_t>(4096, 4 * np))) ||
      (rc = pinned(c, c->pin_down, c->pin_down_bytes, sizeof(double) * (std::min<size_t>(ncell, kPinned) + 1))))
    return rc;
  TxPairs pairs{};
  if (seen.size() > 256) {
    if ((rc = ensure(c, c->d_tx_grid, seen.size())) ||
        (rc = hip_check(c, hipMemcpyAsync(c->d_tx_grid.ptr, seen.data(), seen.size(), hipMemcpyHostToDevice, c->stream),
                        "upload mask")))
      return rc;
    pairs.mask = (const unsigned char*)c->d_tx_grid.ptr;
  } else {
    for (size_t e = 0; e < seen.size(); ++e)
      if (seen[e]) pairs.bits[e >> 6] |= 1ull << (e & 63);
  }
  double* got = (double*)c->pin_down;
  double* d_out = got;
  const double* total = got + (ncell > kPinned ? 0 : ncell);
  if (ncell > kDirect) {
    if ((rc = ensure(c, c->d_tx_out, sizeof(double) * ((size_t)ncell + 1)))) return rc;
    d_out = (double*)c->d_tx_out.ptr;
  }
  unsigned* cnt = (unsigned*)c->d_tx_cnt.ptr;
  unsigned* off = (unsigned*)c->d_tx_off.ptr;
  void* scan_tmp = (char*)off + (sizeof(unsigned) * ((size_t)ncell + 1) + 7) / 8 * 8;
  const dim3 nb((unsigned)((np + 63) / 64));
  launch_fill_u32(c->stream, cnt, 0u, ncell + 1);
  if (np > 0)
    hipLaunchKernelGGL(k_tx_bin<0>, nb, dim3(64), 0, c->stream, poly, key, np, pairs, g, (int4*)c->d_tx_foot.ptr, cnt,
                       (const unsigned*)nullptr, (int*)nullptr, (int64_t)0);
  if ((unsigned long long)np > kMaxEntries / (unsigned)ncell) {
    rc = check_entries(c, [&](unsigned long long* t) {
      hipLaunchKernelGGL(k_tx_total, nb, dim3(64), 0, c->stream, (const int4*)c->d_tx_foot.ptr, np, t);
    });
    if (rc) return rc;
  }
  if (exclusive_scan_u32(c->stream, cnt, off, (long long)ncell + 1, scan_tmp, scan_bytes) != 0)
    return set_err(c, HCS_ERR_LIMIT, "taxel grid too large");
  for (;;) {
    const int64_t list_cap = (int64_t)(c->d_tx_list.bytes / sizeof(int));
    int* list = (int*)c->d_tx_list.ptr;
    launch_fill_u32(c->stream, cnt, 0u, ncell + 1);
    if (np > 0)
      hipLaunchKernelGGL(k_tx_bin<1>, nb, dim3(64), 0, c->stream, poly, key, np, pairs, g, (int4*)c->d_tx_foot.ptr, cnt,
                         (const unsigned*)off, list, list_cap);
    if (ptan) {
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_tx_sample<Dual>), dim3(ncell), dim3(64), 0, c->stream, poly, ptan, key, g,
                         Xd, (const unsigned*)off, (const int*)list, list_cap, d_out);
    } else if (g.S * g.S <= HCS_TX_RAYS && np <= HCS_TX_POLYS) {
      /* up to eight taxels a CU, four waves share a taxel: 256 taxels 52 -> 22
       * us, 1600 taxels 21 -> 14 us; with 3600 taxels 14 -> 16 us */
      auto run = [&](auto kernel, int waves) {
        hipLaunchKernelGGL(kernel, dim3(ncell), dim3(64 * waves), 0, c->stream, poly, key, g, (const unsigned*)off,
                           (const int*)list, list_cap, d_out);
      };
      if (ncell <= 8 * c->num_cu) run(k_tx_sample_fan<4>, 4);
      else run(k_tx_sample_fan<1>, 1);
    } else {
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_tx_sample<double>), dim3(ncell), dim3(64), 0, c->stream, poly,
                         (const double*)nullptr, key, g, (const double*)nullptr, (const unsigned*)off,
                         (const int*)list, list_cap, d_out);
    }
    rc = hip_check(c, hipGetLastError(), "taxel kernels");
    if (!rc && ncell > kPinned) {
      rc = hip_check(c, hipMemcpyAsync(out, d_out, sizeof(double) * (size_t)ncell, hipMemcpyDeviceToHost, c->stream),
                     "download taxels");
      if (!rc)
        rc = hip_check(c, hipMemcpyAsync(got, d_out + ncell, sizeof(double), hipMemcpyDeviceToHost, c->stream), "download");
    } else if (!rc && d_out != got) {
      rc = hip_check(c, hipMemcpyAsync(got, d_out, sizeof(double) * ((size_t)ncell + 1), hipMemcpyDeviceToHost, c->stream),
                     "download taxels");
    }
    if (!rc) rc = hip_check(c, hipStreamSynchronize(c->stream), "sync");
    if (rc) return rc;
    if ((int64_t)*total <= list_cap) break;
    if ((rc = ensure(c, c->d_tx_list, sizeof(int) * (size_t)*total))) return rc;
  }
  if (ncell <= kPinned) std::memcpy(out, got, sizeof(double) * (size_t)ncell);
  return HCS_OK;
}

int taxel_grid_dev(const hcs_taxel_grid& G, TaxelGridDev& g) {
  int32_t cx, cy;
  if (hcs_taxel_dims(&G, &cx, &cy) != HCS_OK || G.sampling_resolution <= 0 || G.window < 0 || G.window > 3)
    return HCS_ERR_ARG;
  std::memcpy(g.X, G.X_W_sensor, sizeof g.X);
  g.xs = G.half_size[0], g.ys = G.half_size[1], g.zs = G.half_size[2], g.res = G.resolution, g.sigma = G.sigma;
  g.S = G.sampling_resolution, g.window = G.window, g.cx = cx, g.cy = cy;
  return HCS_OK;
}

/* ===================================================================
 * Batched sensors: every sensor of a batch in one pass per stage, inside
 * the step's graph (no host round trip; list sizes are checked after the
 * step, which is re-run when a buffer overflowed).
 * =================================================================== */

/* Sensor poses, the 12 doubles (rotation, position) at src[s] in the state,
 * and the step's counters cleared. */
__global__ __launch_bounds__(256) void k_txb_begin(TaxelGridDev* __restrict__ g, const int* __restrict__ src,
                                                   const double* __restrict__ state, int n, unsigned* __restrict__ cnt,
                                                   unsigned* __restrict__ cursor, int ncell,
                                                   unsigned* __restrict__ nlive) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < 12 * n) g[t / 12].X[t % 12] = state[src[t / 12] + t % 12];
  if (t <= ncell) cnt[t] = 0;
  if (t < ncell) cursor[t] = 0;
  if (t == 0) *nlive = 0;
}

/* Polygons strided over the grid; each polygon goes to every sensor of its
 * pair, into the taxels its footprint covers.  FILL = 0 counts per taxel and
 * keeps the footprint on the pair's first sensor; FILL = 1 writes the polygon
 * into the taxel's list slice.  Bound by reading the records (320 B a polygon,
 * 64-byte pieces of it), which the second pass now mostly leaves out: 1024
 * pads 131 + 185 us -> 153 + 67 us, with shared atomics. */
template <int FILL>
__global__ __launch_bounds__(256) void k_txb_bin(const double* __restrict__ poly, const int64_t* __restrict__ key,
                                                 const unsigned long long* __restrict__ poly_cnt, int64_t poly_cap,
                                                 const int* __restrict__ psoff, const int* __restrict__ psens,
                                                 const TaxelGridDev* __restrict__ grids,
                                                 const int* __restrict__ cell_base, int4* __restrict__ foot,
                                                 unsigned* __restrict__ cnt, const unsigned* __restrict__ off,
                                                 unsigned* __restrict__ cursor, int* __restrict__ list,
                                                 int64_t list_cap) {
  const int64_t np = min((int64_t)*poly_cnt, poly_cap);
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t q0 = blockIdx.x * (int64_t)blockDim.x; q0 < np; q0 += step) {
    const int64_t q = q0 + threadIdx.x;
    int k = 0, k1 = 0;
    bool first = true;
    if (q < np) {
      const int e = (int)key[3 * q];
      k = psoff[e], k1 = psoff[e + 1];
    }
    while (__any(k < k1)) {
      int4 f = make_int4(0, -1, 0, -1);
      int cx = 1, base = 0;
      if (k < k1) {
        const int s = psens[k];
        cx = grids[s].cx, base = cell_base[s];
        if (FILL && first) f = foot[q];
        else footprint(poly + q * HCS_PREC, grids[s], f.x, f.y, f.z, f.w);
        if (!FILL && first) foot[q] = f;
      }
      bin_polygon<FILL>((int)q, f, cx, base, FILL ? cursor : cnt, off, list, list_cap);
      first = false, ++k;
    }
  }
}

/* The entries that k_txb_bin counts, in 64 bits. */
__global__ __launch_bounds__(256) void k_txb_total(const double* __restrict__ poly, const int64_t* __restrict__ key,
                                                   int64_t np, const int* __restrict__ psoff,
                                                   const int* __restrict__ psens, const TaxelGridDev* __restrict__ grids,
                                                   unsigned long long* __restrict__ total) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t q0 = blockIdx.x * (int64_t)blockDim.x; q0 < np; q0 += step) {
    const int64_t q = q0 + threadIdx.x;
    int k = 0, k1 = 0;
    if (q < np) {
      const int e = (int)key[3 * q];
      k = psoff[e], k1 = psoff[e + 1];
    }
    for (; __any(k < k1); ++k) {
      int4 f = make_int4(0, -1, 0, -1);
      if (k < k1) footprint(poly + q * HCS_PREC, grids[psens[k]], f.x, f.y, f.z, f.w);
      add_entries(f, k < k1, total);
    }
  }
}

/* The taxels that have candidate polygons (and whose list fits the list
 * buffer; an overflowed list is re-run after the step with a larger one),
 * appended to live[] with one atomic per block of HCS_TXB_LIVE threads
 * (atomics on the one counter complete one after another, so one per wave
 * would queue thousands); every other taxel is 0. */
#define HCS_TXB_LIVE 1024
__global__ __launch_bounds__(HCS_TXB_LIVE) void k_txb_live(const unsigned* __restrict__ cnt,
                                                           const unsigned* __restrict__ off, int ncell,
                                                           int64_t list_cap, int* __restrict__ live,
                                                           unsigned* __restrict__ nlive,
                                                           double* __restrict__ out) {
  __shared__ unsigned s_off[HCS_TXB_LIVE / 64 + 1];
  const int cell = blockIdx.x * blockDim.x + threadIdx.x;
  if (cell < ncell) out[cell] = 0.0;
  const bool on = cell < ncell && cnt[cell] > 0 && (int64_t)off[cell] + cnt[cell] <= list_cap;
  const unsigned long long m = __ballot(on);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) s_off[w] = (unsigned)__popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned tot = 0;
    for (int x = 0; x < (int)(blockDim.x >> 6); ++x) {
      const unsigned n = s_off[x];
      s_off[x] = tot;
      tot += n;
    }
    s_off[HCS_TXB_LIVE / 64] = tot ? atomicAdd(nlive, tot) : 0u;
  }
  __syncthreads();
  if (on)
    live[s_off[HCS_TXB_LIVE / 64] + s_off[w] +
         __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] = cell;
}

/* One wave per live taxel of any sensor, strided over the grid; FAN: the
 * fan-major sampler (every sensor has S^2 <= HCS_TX_RAYS, and there is room for
 * at most HCS_TX_POLYS polygons). */
template <bool FAN>
__global__ __launch_bounds__(64) void k_txb_sample(const double* __restrict__ poly, const int64_t* __restrict__ key,
                                                   const TaxelGridDev* __restrict__ grids,
                                                   const int* __restrict__ cell_base, const int* __restrict__ cell_sensor,
                                                   const unsigned* __restrict__ off, const unsigned* __restrict__ cnt,
                                                   const int* __restrict__ list, const int* __restrict__ live,
                                                   const unsigned* __restrict__ nlive, double* __restrict__ out) {
  const unsigned nl = *nlive;
  for (unsigned k = blockIdx.x; k < nl; k += gridDim.x) {
    const int cell = live[k];
    const int s = cell_sensor[cell];
    const TaxelGridDev g = grids[s];
    const int local = cell - cell_base[s];
    const double v =
        FAN ? sample_cell_scatter(poly, key, g, off[cell], cnt[cell], list, local % g.cx, local / g.cx)
            : sample_cell<double>(poly, nullptr, key, g, nullptr, off[cell], cnt[cell], list, local % g.cx,
                                  local / g.cx);
    if (threadIdx.x == 0) out[cell] = v;
  }
}

int batch_taxels_setup(Ctx* c, BatchTaxels& t, int npairs, const int32_t* geoms, int n, const int32_t* pair,
                       const hcs_taxel_grid* grids) {
  std::vector<TaxelGridDev> g(std::max(1, n));
  std::vector<int> src(std::max(1, n)), base(n + 1, 0), psoff(npairs + 1, 0), psens(std::max(1, n));
  std::vector<unsigned char> mask(std::max(1, npairs), 0);
  for (int s = 0; s < n; ++s) {
    const int e = pair[s];
    if (e < 0 || e >= npairs) return set_err(c, HCS_ERR_ARG, "sensor " + std::to_string(s) + ": pair out of range");
    if (taxel_grid_dev(grids[s], g[s]) != HCS_OK)
      return set_err(c, HCS_ERR_ARG, "sensor " + std::to_string(s) + ": invalid taxel grid");
    /* the pose of the pair's geometry with the sensor's mesh handle (B when
     * both are) */
    int side;
    if (geoms[2 * e + 1] == grids[s].geom) side = 1;
    else if (geoms[2 * e] == grids[s].geom) side = 0;
    else return set_err(c, HCS_ERR_ARG, "sensor " + std::to_string(s) + ": its geom is not in its pair");
    src[s] = HCS_STATE * e + 12 * side;
    if ((int64_t)base[s] + (int64_t)g[s].cx * g[s].cy > (1 << 30))
      return set_err(c, HCS_ERR_ARG, "too many taxels in the batch's sensors");
    base[s + 1] = base[s] + g[s].cx * g[s].cy;
    ++psoff[e + 1];
    mask[e] = 1;
  }
  for (int e = 0; e < npairs; ++e) psoff[e + 1] += psoff[e];
  {
    std::vector<int> fill(psoff.begin(), psoff.end() - 1);
    for (int s = 0; s < n; ++s) psens[fill[pair[s]]++] = s;
  }
  const int ncell = base[n];
  std::vector<int> cs(std::max(1, ncell));
  for (int s = 0; s < n; ++s)
    for (int k = base[s]; k < base[s + 1]; ++k) cs[k] = s;
  int rc;
  if ((rc = ensure(c, t.grid, sizeof(TaxelGridDev) * g.size())) || (rc = ensure(c, t.src, sizeof(int) * src.size())) ||
      (rc = ensure(c, t.cell_base, sizeof(int) * base.size())) ||
      (rc = ensure(c, t.cell_sensor, sizeof(int) * cs.size())) || (rc = ensure(c, t.psoff, sizeof(int) * psoff.size())) ||
      (rc = ensure(c, t.psens, sizeof(int) * psens.size())) || (rc = ensure(c, t.mask, mask.size())) ||
      (rc = ensure(c, t.poly_cnt, 64)) || (rc = ensure(c, t.cnt, sizeof(unsigned) * (ncell + 1))) ||
      (rc = ensure(c, t.cursor, sizeof(unsigned) * std::max(1, ncell))) ||
      (rc = ensure(c, t.off, sizeof(unsigned) * (ncell + 1))) || (rc = ensure(c, t.out, sizeof(double) * std::max(1, ncell))) ||
      (rc = ensure(c, t.live, sizeof(int) * std::max(1, ncell))))
    return rc;
  const size_t sb = scan_temp_bytes((long long)ncell + 1);
  if ((rc = ensure(c, t.scan_tmp, std::max<size_t>(sb, 8)))) return rc;
  t.scan_bytes = sb;
  struct Up {
    DBuf& d;
    const void* h;
    size_t bytes;
  } ups[] = {{t.grid, g.data(), sizeof(TaxelGridDev) * g.size()}, {t.src, src.data(), sizeof(int) * src.size()},
             {t.cell_base, base.data(), sizeof(int) * base.size()}, {t.cell_sensor, cs.data(), sizeof(int) * cs.size()},
             {t.psoff, psoff.data(), sizeof(int) * psoff.size()}, {t.psens, psens.data(), sizeof(int) * psens.size()},
             {t.mask, mask.data(), mask.size()}};
  for (const Up& u : ups)
    if ((rc = hip_check(c, hipMemcpyAsync(u.d.ptr, u.h, u.bytes, hipMemcpyHostToDevice, c->stream), "upload sensors")))
      return rc;
  t.n = n, t.ncell = ncell;
  t.max_rays = 0;
  for (int k = 0; k < n; ++k) t.max_rays = std::max(t.max_rays, g[k].S * g[k].S);
  std::vector<int64_t> cells(npairs, 0);
  for (int k = 0; k < n; ++k) cells[pair[k]] += (int64_t)g[k].cx * g[k].cy;
  t.pair_cells = *std::max_element(cells.begin(), cells.end());
  t.bin_grid = std::max(1, c->num_cu * 4);
  return hip_check(c, hipStreamSynchronize(c->stream), "sync");
}

int batch_taxels_reserve(Ctx* c, BatchTaxels& t, int64_t poly_cap, int64_t list_cap) {
  poly_cap = std::max<int64_t>(poly_cap, 4096);
  list_cap = std::max<int64_t>(list_cap, 4096);
  /* list offsets are 32-bit */
  if (list_cap > 0xffffffffLL) return set_err(c, HCS_ERR_CAPACITY, "taxel polygon lists exceed 2^32 entries");
  int rc;
  if ((rc = ensure(c, t.poly_rec, sizeof(double) * HCS_PREC * poly_cap)) ||
      (rc = ensure(c, t.poly_key, sizeof(int64_t) * 3 * poly_cap)) ||
      (rc = ensure(c, t.foot, sizeof(int4) * poly_cap)) || (rc = ensure(c, t.list, sizeof(int) * list_cap)))
    return rc;
  t.poly_cap = poly_cap, t.list_cap = list_cap;
  return HCS_OK;
}

void batch_taxels_enqueue(Ctx* c, BatchTaxels& t, const double* state) {
  if (t.n == 0) return;
  hipStream_t s = c->stream;
  TaxelGridDev* g = (TaxelGridDev*)t.grid.ptr;
  unsigned* nlive = (unsigned*)t.poly_cnt.ptr + 2;
  hipLaunchKernelGGL(k_txb_begin, dim3((std::max(12 * t.n, t.ncell + 1) + 255) / 256), dim3(256), 0, s, g,
                     (const int*)t.src.ptr, state, t.n, (unsigned*)t.cnt.ptr, (unsigned*)t.cursor.ptr, t.ncell, nlive);
  const unsigned long long* pc = (const unsigned long long*)t.poly_cnt.ptr;
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_txb_bin<0>), dim3(t.bin_grid), dim3(256), 0, s, (const double*)t.poly_rec.ptr,
                     (const int64_t*)t.poly_key.ptr, pc, t.poly_cap, (const int*)t.psoff.ptr, (const int*)t.psens.ptr,
                     (const TaxelGridDev*)g, (const int*)t.cell_base.ptr, (int4*)t.foot.ptr, (unsigned*)t.cnt.ptr,
                     (const unsigned*)nullptr, (unsigned*)nullptr, (int*)nullptr, (int64_t)0);
  (void)exclusive_scan_u32(s, (const unsigned*)t.cnt.ptr, (unsigned*)t.off.ptr, (long long)t.ncell + 1,
                           t.scan_tmp.ptr, t.scan_bytes);
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_txb_bin<1>), dim3(t.bin_grid), dim3(256), 0, s, (const double*)t.poly_rec.ptr,
                     (const int64_t*)t.poly_key.ptr, pc, t.poly_cap, (const int*)t.psoff.ptr, (const int*)t.psens.ptr,
                     (const TaxelGridDev*)g, (const int*)t.cell_base.ptr, (int4*)t.foot.ptr, (unsigned*)t.cnt.ptr,
                     (const unsigned*)t.off.ptr, (unsigned*)t.cursor.ptr, (int*)t.list.ptr, t.list_cap);
  hipLaunchKernelGGL(k_txb_live, dim3((t.ncell + HCS_TXB_LIVE - 1) / HCS_TXB_LIVE), dim3(HCS_TXB_LIVE), 0, s,
                     (const unsigned*)t.cnt.ptr,
                     (const unsigned*)t.off.ptr, t.ncell, t.list_cap, (int*)t.live.ptr, nlive, (double*)t.out.ptr);
  const dim3 grid(std::max(1, std::min(t.ncell, c->num_cu * 16)));
  if (t.max_rays <= HCS_TX_RAYS && t.poly_cap <= HCS_TX_POLYS)
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_txb_sample<true>), grid, dim3(64), 0, s, (const double*)t.poly_rec.ptr,
                       (const int64_t*)t.poly_key.ptr, (const TaxelGridDev*)g, (const int*)t.cell_base.ptr,
                       (const int*)t.cell_sensor.ptr, (const unsigned*)t.off.ptr, (const unsigned*)t.cnt.ptr,
                       (const int*)t.list.ptr, (const int*)t.live.ptr, (const unsigned*)nlive, (double*)t.out.ptr);
  else
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_txb_sample<false>), grid, dim3(64), 0, s, (const double*)t.poly_rec.ptr,
                       (const int64_t*)t.poly_key.ptr, (const TaxelGridDev*)g, (const int*)t.cell_base.ptr,
                       (const int*)t.cell_sensor.ptr, (const unsigned*)t.off.ptr, (const unsigned*)t.cnt.ptr,
                       (const int*)t.list.ptr, (const int*)t.live.ptr, (const unsigned*)nlive, (double*)t.out.ptr);
}

int batch_taxels_demand(Ctx* c, BatchTaxels& t, int64_t& npoly, int64_t& nlist) {
  npoly = nlist = 0;
  if (t.n == 0) return HCS_OK;
  unsigned long long np = 0;
  unsigned nl = 0;
  int rc = hip_check(c, hipMemcpyAsync(&np, t.poly_cnt.ptr, 8, hipMemcpyDeviceToHost, c->stream), "dl");
  if (!rc)
    rc = hip_check(c, hipMemcpyAsync(&nl, (const unsigned*)t.off.ptr + t.ncell, 4, hipMemcpyDeviceToHost, c->stream),
                   "dl");
  if (!rc) rc = hip_check(c, hipStreamSynchronize(c->stream), "sync");
  npoly = (int64_t)np, nlist = (int64_t)nl;
  /* (polygons beyond the record buffer are counted when it has grown) */
  if (rc || npoly > t.poly_cap || np <= kMaxEntries / (unsigned long long)t.pair_cells) return rc;
  return check_entries(c, [&](unsigned long long* total) {
    hipLaunchKernelGGL(k_txb_total, dim3(t.bin_grid), dim3(256), 0, c->stream, (const double*)t.poly_rec.ptr,
                       (const int64_t*)t.poly_key.ptr, npoly, (const int*)t.psoff.ptr, (const int*)t.psens.ptr,
                       (const TaxelGridDev*)t.grid.ptr, total);
  });
}

void batch_taxels_free(BatchTaxels& t) {
  for (DBuf* b : {&t.grid, &t.src, &t.cell_base, &t.cell_sensor, &t.psoff, &t.psens, &t.mask, &t.poly_rec, &t.poly_key, &t.foot,
                  &t.poly_cnt, &t.cnt, &t.cursor, &t.off, &t.scan_tmp, &t.list, &t.out, &t.live})
    if (b->ptr) (void)hipFree(b->ptr), b->ptr = nullptr, b->bytes = 0;
  t = BatchTaxels();
}

}  // namespace hcs

extern "C" {

int hcs_taxel_dims(const hcs_taxel_grid* g, int32_t* cx, int32_t* cy) {
  if (!g || !cx || !cy || !(g->resolution > 0)) return HCS_ERR_ARG;
  /* ::floorl(2 * xs / resolution + 0.1), flat_tactile_sensor.cpp:196-197 */
  *cx = (int32_t)std::floor(2 * (long double)g->half_size[0] / g->resolution + 0.1L);
  *cy = (int32_t)std::floor(2 * (long double)g->half_size[1] / g->resolution + 0.1L);
  if (*cx <= 0 || *cy <= 0) return HCS_ERR_ARG;
  return HCS_OK;
}

int hcs_taxels(hcs_ctx* h, int32_t nsensors, const hcs_taxel_grid* grids, double* out) {
  if (!h || nsensors < 0 || (nsensors > 0 && (!grids || !out))) return HCS_ERR_ARG;
  Ctx* c = &h->c;
  if (!c->last_valid) return set_err(c, HCS_ERR_STATE, "hcs_taxels needs a contact step run with keep_polygons = 1");
  int rc = hip_check(c, hipSetDevice(c->device), "hipSetDevice");
  if (rc) return rc;
  const int npairs = (int)c->last_pairs.size();
  size_t off_out = 0;
  for (int s = 0; s < nsensors; ++s) {
    const hcs_taxel_grid& G = grids[s];
    TaxelGridDev g;
    if (taxel_grid_dev(G, g) != HCS_OK) return set_err(c, HCS_ERR_ARG, "invalid taxel grid");
    const int ncell = g.cx * g.cy;
    std::vector<unsigned char> seen(npairs, 0);
    for (int e = 0; e < npairs; ++e)
      seen[e] = (c->last_geoms[2 * e] == G.geom || c->last_geoms[2 * e + 1] == G.geom) ? 1 : 0;
    rc = run_taxels(c, g, seen, (const double*)c->d_poly_rec.ptr, nullptr, (const int64_t*)c->d_poly_key.ptr,
                    c->last_npoly, nullptr, out + off_out);
    if (rc) return rc;
    off_out += ncell;
  }
  return HCS_OK;
}

}  // extern "C"
