/*
 * hcs_call.hip -- the per-call contact step (hcs_contact_step, hcs_candidates
 * and hcs_contact_step_noalloc): a synchronous step of a few pairs whose
 * poses, and possibly pairs, are new in every call.
 *
 * Such a step is short (tens of microseconds on the device), so what it costs
 * is launches, copies and waves that run alone:
 *   - one upload: descriptors, state and tables are one blob in pinned host
 *     memory, which the first kernel copies to the device (and with it clears
 *     the counters and composes the pair poses); results are written to
 *     pinned host memory by the last kernel.  Six copies in, five out and
 *     three clears were 14 blit launches of 2.7 us and as many API calls.
 *   - the work items are enumerated on the device from the pairs' tables
 *     (chunks of 64 queries x the subtrees of an LBVH frontier), culled by
 *     their boxes and kept in order, so nothing is planned, uploaded or
 *     bounded per item on the host.
 *   - items are cut over frontiers deep enough to fill the chip: with one
 *     item per chunk over the whole tree, a pad of 8192 triangles ran on 110
 *     waves of up to 2300 candidates each.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "hcs_internal.h"
#include "hcs_items.h"
#include "hcs_prim.h"
#include "hcs_reduce.h"

#pragma clang fp contract(off)

namespace hcs {

namespace {

constexpr int kMaxCounters = 8;

struct FrontArgs {
  const uint4* src;
  uint4* dst;
  int64_t n16;
  const double* state; /* in src */
  double* xf;
  int npairs, ncounters;
  unsigned* counters[kMaxCounters]; /* 64 bytes each */
};

/* Copies the blob (unless it is in place), clears the counters and composes
 * X_AB = X_WA^-1 X_WB of every pair. */
__global__ __launch_bounds__(256) void k_call_front(FrontArgs f) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, n = (int64_t)gridDim.x * blockDim.x;
  if (t < 16 * f.ncounters) f.counters[t / 16][t % 16] = 0u;
  for (int64_t e = t; e < f.npairs; e += n) {
    double st[24], X[12];
#pragma unroll
    for (int k = 0; k < 24; ++k) st[k] = f.state[HCS_STATE * e + k];
    compose_SR(st, st + 12, X);
#pragma unroll
    for (int k = 0; k < 12; ++k) f.xf[12 * e + k] = X[k];
  }
  if ((const uint4*)f.dst != f.src)
    for (int64_t i = t; i < f.n16; i += n) f.dst[i] = f.src[i];
}

constexpr int kGenWaves = HCS_GEN_THREADS / 64;

/* A block's kept lanes: the waves' masks, and their number. */
__device__ inline void block_counts(bool keep, unsigned* __restrict__ cnt, unsigned long long* __restrict__ mask) {
  __shared__ unsigned n[kGenWaves];
  const int w = threadIdx.x >> 6;
  const unsigned long long m = __ballot(keep);
  if ((threadIdx.x & 63) == 0) mask[(size_t)blockIdx.x * kGenWaves + w] = m, n[w] = (unsigned)__popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned all = 0;
#pragma unroll
    for (int k = 0; k < kGenWaves; ++k) all += n[k];
    cnt[blockIdx.x] = all;
  }
}

/* Kept lanes before this thread (and through its block): a block adds up the
 * counts of the blocks before it (or reads their scan, when one was made), so
 * no pass is needed between counting and placing. */
__device__ inline unsigned kept_before(const unsigned* __restrict__ cnt, bool scanned,
                                       const unsigned long long* __restrict__ mask, bool& keep, unsigned& through) {
  __shared__ unsigned part[kGenWaves];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  unsigned before = 0;
  if (scanned) {
    before = cnt[blockIdx.x];
  } else {
    for (unsigned k = threadIdx.x; k < blockIdx.x; k += HCS_GEN_THREADS) before += cnt[k];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) before += __shfl_xor(before, o, 64);
    if (lane == 0) part[w] = before;
    __syncthreads();
    before = 0;
#pragma unroll
    for (int k = 0; k < kGenWaves; ++k) before += part[k];
  }
  const unsigned long long* mb = mask + (size_t)blockIdx.x * kGenWaves;
  unsigned pos = before;
  through = before;
#pragma unroll
  for (int k = 0; k < kGenWaves; ++k) {
    const unsigned n = (unsigned)__popcll(mb[k]);
    pos += k < w ? n : 0u;
    through += n;
  }
  const unsigned long long m = mb[w];
  keep = m >> lane & 1;
  return pos + lane_prefix(m);
}

/* Adds the block's expected candidates to *sum (whole numbers, so the sum and
 * with it the cut do not depend on the order). */
__device__ inline void add_expected(unsigned word, unsigned long long* __restrict__ sum) {
  __shared__ unsigned long long part[kGenWaves];
  const unsigned long long v = (unsigned long long)wave_sum_i((int64_t)(word & kEstMask));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long all = 0;
#pragma unroll
    for (int k = 0; k < kGenWaves; ++k) all += part[k];
    if (all) atomicAdd(sum, all);
  }
}

/* First cull: one block per HCS_GEN_THREADS items of one pair. */
__global__ __launch_bounds__(HCS_GEN_THREADS) void k_call_cull1(const EnvDesc* __restrict__ envs,
                                                                const int2* __restrict__ blocks,
                                                                const double* __restrict__ xf,
                                                                unsigned* __restrict__ cnt,
                                                                unsigned long long* __restrict__ mask) {
  const int2 b = blocks[blockIdx.x];
  const EnvDesc& E = envs[b.x];
  const int i = b.y + threadIdx.x;
  int chunk, node;
  block_counts(i < E.item_count && first_item(E, xf + 12 * (size_t)b.x, i, chunk, node), cnt, mask);
}

/* The items it keeps, in item order: (pair, chunk, place of the root).
 * Blocks past the items move the triangles of one tet-query pair each. */
__global__ __launch_bounds__(HCS_GEN_THREADS) void k_call_place1(const EnvDesc* __restrict__ envs,
                                                                 const int2* __restrict__ blocks, int nblk,
                                                                 const unsigned* __restrict__ cnt, bool scanned,
                                                                 const unsigned long long* __restrict__ mask,
                                                                 const int* __restrict__ xenv,
                                                                 const double* __restrict__ xf,
                                                                 double* __restrict__ xtri, int4* __restrict__ item,
                                                                 unsigned* __restrict__ cut,
                                                                 unsigned long long* __restrict__ cut_sum,
                                                                 unsigned* __restrict__ n1) {
  if ((int)blockIdx.x >= nblk) {
    const int e = xenv[blockIdx.x - nblk];
    move_triangles(envs[e], xf + 12 * (size_t)e, xtri, HCS_GEN_THREADS);
    return;
  }
  bool keep;
  unsigned through;
  const unsigned pos = kept_before(cnt, scanned, mask, keep, through);
  if (threadIdx.x == 0 && (int)blockIdx.x == nblk - 1) *n1 = through;
  const int2 b = blocks[blockIdx.x];
  const EnvDesc& E = envs[b.x];
  const int depth = is_tree(E) ? E.depth : 0, i = b.y + threadIdx.x;
  const int chunk = i >> depth, node = (1 << depth) + (i & ((1 << depth) - 1));
  if (!cut) {
    if (keep) item[pos] = make_int4(b.x, chunk, node, 0);
    return;
  }
  unsigned word = 0;
  if (keep) {
    const int root = is_tree(E) ? E.rootsA[node] : 0;
    word = cut_word(E, xf + 12 * (size_t)b.x, chunk, root);
    item[pos] = make_int4(b.x, chunk, root, 0);
    cut[pos] = word;
  }
  add_expected(word, cut_sum);
}

/* Second cull: the kept items cut e levels deeper, e the same for the launch
 * (2^e n1 items within the budget).  The contact lies in a few of the
 * first frontier's subtrees: a pad's 33k candidates came from 110 chunks and
 * 4 to 8 subtrees, 1000 and more per item; cut again where the boxes meet, the
 * longest item falls to a tenth and about a thousand waves share the work. */
__global__ __launch_bounds__(HCS_GEN_THREADS) void k_call_cull2(const EnvDesc* __restrict__ envs,
                                                                const double* __restrict__ xf,
                                                                const int4* __restrict__ item,
                                                                const unsigned* __restrict__ n1, unsigned budget,
                                                                unsigned* __restrict__ cnt,
                                                                unsigned long long* __restrict__ mask) {
  int i, sub, node;
  bool keep = second_item(envs, item, *n1, budget, blockIdx.x * HCS_GEN_THREADS + threadIdx.x, i, sub, node);
  if (keep) {
    const int4 it = item[i];
    const EnvDesc& E = envs[it.x];
    if (node != it.z) { /* a deeper subtree than the first cull tested */
      double Q[6];
      chunk_box(E, it.y, Q);
      keep = may_meet_subtree(E, xf + 12 * (size_t)it.x, Q, E.rootsA[node]);
    }
  }
  block_counts(keep, cnt, mask);
}

/* The pairs' first live items: a pair's from its first item (sub 0, placed
 * at pos), also for the pairs without items before it. */
__device__ inline void first_of_pair(const int4* __restrict__ item, int i, int pos, int* __restrict__ pair_lo) {
  for (int q = i > 0 ? item[i - 1].x + 1 : 0; q <= item[i].x; ++q) pair_lo[q] = pos;
}
__device__ inline void after_last_pair(const int4* __restrict__ item, unsigned n1, int npairs, int total,
                                       int* __restrict__ pair_lo) {
  for (int e = n1 ? item[n1 - 1].x + 1 : 0; e <= npairs; ++e) pair_lo[e] = total;
}

/* The live items in order, and each pair's first. */
__global__ __launch_bounds__(HCS_GEN_THREADS) void k_call_place2(const EnvDesc* __restrict__ envs,
                                                                 const int4* __restrict__ item,
                                                                 const unsigned* __restrict__ n1p, unsigned budget,
                                                                 const unsigned* __restrict__ cnt, bool scanned,
                                                                 const unsigned long long* __restrict__ mask,
                                                                 int npairs, int4* __restrict__ live_item,
                                                                 unsigned* __restrict__ live_cnt,
                                                                 int* __restrict__ pair_lo) {
  bool keep;
  unsigned through;
  const unsigned pos = kept_before(cnt, scanned, mask, keep, through);
  const unsigned n1 = *n1p, t = blockIdx.x * HCS_GEN_THREADS + threadIdx.x;
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
    *live_cnt = through;
    after_last_pair(item, n1, npairs, (int)through, pair_lo);
  }
  int i, sub, node;
  const bool on = second_item(envs, item, n1, budget, t, i, sub, node);
  if (on && sub == 0) first_of_pair(item, i, (int)pos, pair_lo);
  if (!keep) return;
  const int4 it = item[i];
  const EnvDesc& E = envs[it.x];
  live_item[pos] = live_record(E, it, is_tree(E) ? E.rootsA[node] : 0);
}

/* ---- spread plans: batches of many pairs, whose items differ too much for
 * one number of levels (some chunks are a few large triangles that meet a
 * whole mesh: 147k candidates in one item of 2048 objects, where a wave's
 * share was 4k).  The items that the first cull keeps are cut by their
 * expected candidates and culled again.  2048 objects, k_cand:
 * 3.28 -> 0.90 ms; 400 objects 746 -> 370 us, 64 objects 325 -> 145 us, 200
 * soft pairs 1.83 -> 1.36 ms.  (A second round of cuts with expectations for
 * the smaller boxes found little more to cut and cost its launches.) */

__device__ inline unsigned block_exclusive(unsigned v, unsigned& total) {
  __shared__ unsigned part[kGenWaves];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  unsigned inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
  }
  if (lane == 63) part[w] = inc;
  __syncthreads();
  unsigned before = inc - v;
  total = 0;
#pragma unroll
  for (int k = 0; k < kGenWaves; ++k) before += k < w ? part[k] : 0u, total += part[k];
  return before;
}
/* Pieces per block of items. */
__global__ __launch_bounds__(HCS_GEN_THREADS) void k_cut_count(CutArgs c, const unsigned* __restrict__ word,
                                                               unsigned* __restrict__ cnt) {
  const unsigned n = *c.n, i = blockIdx.x * HCS_GEN_THREADS + threadIdx.x;
  unsigned total;
  (void)block_exclusive(i < n ? cut_slots(word[i], cut_target(c)) : 0u, total);
  if (threadIdx.x == 0) cnt[blockIdx.x] = total;
}
/* First piece of every item, off[n] their number; in place of the words. */
__global__ __launch_bounds__(HCS_GEN_THREADS) void k_cut_place(CutArgs c, const unsigned* __restrict__ cnt,
                                                               unsigned* __restrict__ off) {
  const unsigned n = *c.n, i = blockIdx.x * HCS_GEN_THREADS + threadIdx.x;
  if (blockIdx.x * HCS_GEN_THREADS > n) return;
  unsigned v = 0, before, all;
  for (unsigned k = threadIdx.x; k < blockIdx.x; k += HCS_GEN_THREADS) v += cnt[k];
  (void)block_exclusive(v, before);
  __syncthreads();
  v = i < n ? cut_slots(off[i], cut_target(c)) : 0u;
  before += block_exclusive(v, all);
  if (i <= n) off[i] = before;
}
__global__ __launch_bounds__(HCS_GEN_THREADS) void k_cut_cull(const EnvDesc* __restrict__ envs,
                                                              const double* __restrict__ xf,
                                                              const int4* __restrict__ item,
                                                              const unsigned* __restrict__ n,
                                                              const unsigned* __restrict__ off,
                                                              unsigned* __restrict__ cnt,
                                                              unsigned long long* __restrict__ mask) {
  int i, sub, levels;
  bool keep = piece(off, *n, blockIdx.x * HCS_GEN_THREADS + threadIdx.x, i, sub, levels);
  if (keep && levels > 0) {
    const int4 it = item[i];
    const EnvDesc& E = envs[it.x];
    double Q[6];
    chunk_box(E, it.y, Q);
    keep = may_meet_subtree(E, xf + 12 * (size_t)it.x, Q, cut_root(E, it.z, levels, sub));
  }
  block_counts(keep, cnt, mask);
}
/* The kept pieces are the live items; and each pair's first. */
__global__ __launch_bounds__(HCS_GEN_THREADS) void k_cut_keep(const EnvDesc* __restrict__ envs,
                                                              const int4* __restrict__ item,
                                                              const unsigned* __restrict__ np,
                                                              const unsigned* __restrict__ off,
                                                              const unsigned* __restrict__ cnt,
                                                              const unsigned long long* __restrict__ mask, int npairs,
                                                              int4* __restrict__ live_item,
                                                              unsigned* __restrict__ live_cnt,
                                                              int* __restrict__ pair_lo) {
  bool keep;
  unsigned through;
  const unsigned pos = kept_before(cnt, false, mask, keep, through);
  const unsigned n = *np;
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
    *live_cnt = through;
    after_last_pair(item, n, npairs, (int)through, pair_lo);
  }
  int i, sub, levels;
  const bool on = piece(off, n, blockIdx.x * HCS_GEN_THREADS + threadIdx.x, i, sub, levels);
  if (on && sub == 0) first_of_pair(item, i, (int)pos, pair_lo);
  if (!keep) return;
  const int4 it = item[i];
  const EnvDesc& E = envs[it.x];
  live_item[pos] = live_record(E, it, cut_root(E, it.z, levels, sub));
}

/* Exclusive scan of the live items' survivor counts (off[n] = total), one
 * block: 3 to 9 us for up to 8192 live items and as much again for every 8192
 * more, where a scan of all places takes 9 us in three launches.  A small part
 * of the places is live: with up to kScanPlaces of them this is 5 us less for
 * 12 mixed pairs and 120 bodies on the ground, 3 for 250 and the same for 500
 * bodies, whose places just fit. */
constexpr int kScanThreads = 1024, kScanPer = 8, kScanPlaces = 65536;
__global__ __launch_bounds__(kScanThreads) void k_call_scan(const unsigned* __restrict__ in,
                                                            const unsigned* __restrict__ live_cnt,
                                                            unsigned* __restrict__ off) {
  __shared__ unsigned lds[kScanThreads / 64];
  const int n = (int)*live_cnt, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  unsigned carry = 0;
  for (int t0 = 0; t0 <= n; t0 += kScanThreads * kScanPer) {
    const int base = t0 + threadIdx.x * kScanPer;
    unsigned v[kScanPer], s = 0;
#pragma unroll
    for (int j = 0; j < kScanPer; ++j) v[j] = base + j < n ? in[base + j] : 0u, s += v[j];
    unsigned inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned u = __shfl_up(inc, o, 64);
      if (lane >= o) inc += u;
    }
    __syncthreads();
    if (lane == 63) lds[w] = inc;
    __syncthreads();
    unsigned run = carry + inc - s, all = 0;
#pragma unroll
    for (int k = 0; k < kScanThreads / 64; ++k) run += k < w ? lds[k] : 0u, all += lds[k];
#pragma unroll
    for (int j = 0; j < kScanPer; ++j) {
      if (base + j <= n) off[base + j] = run;
      run += v[j];
    }
    carry += all;
  }
}

/* Wave w: slice w % K of pair w / K. */
__global__ __launch_bounds__(64) void k_call_reduce(const int* __restrict__ pair_lo, int K,
                                                    const unsigned* __restrict__ off,
                                                    const int* __restrict__ item_ncand,
                                                    const unsigned long long* __restrict__ surv_cnt, int64_t surv_cap,
                                                    const Contrib* __restrict__ contrib, RedPart* __restrict__ part) {
  const int e = blockIdx.x / K, j = blockIdx.x % K;
  const int first = pair_lo[e], cnt = pair_lo[e + 1] - first;
  /* on survivor-list overflow the offsets run past the contribution slots:
   * sum nothing, the status reports the overflow */
  const bool over = (int64_t)*surv_cnt > surv_cap;
  const unsigned capu = (unsigned)(surv_cap < 0xffffffffLL ? surv_cap : 0xffffffffLL);
  const unsigned lo = min(off[first], capu), hi = over ? lo : max(lo, min(off[first + cnt], capu));
  const RedPart r = reduce_slice(contrib, lo, hi, j, K, item_ncand, first, cnt);
  if (threadIdx.x == 0) part[blockIdx.x] = r;
}

struct CombineArgs {
  const RedPart* part;
  int K;
  const unsigned long long *surv_cnt, *poly_cnt, *face_cnt, *cand_cnt;
  int64_t surv_cap;
  const int* err;
  PairOut* out;
  CallTail* tail;
};

/* One wave per pair: its K <= 64 slices, one per lane, by a fixed butterfly
 * (one thread adding 64 slices took 14 us); the record is written in one
 * burst, since out is host memory.  The step's counters with the first. */
__global__ __launch_bounds__(64) void k_call_combine(CombineArgs a) {
  __shared__ unsigned long long rec[16];
  const int e = blockIdx.x, lane = threadIdx.x;
  RedPart q{};
  if (lane < a.K) q = a.part[(size_t)e * a.K + lane];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    q.F[c] = wave_sum<double>(q.F[c]), q.tA[c] = wave_sum<double>(q.tA[c]), q.tB[c] = wave_sum<double>(q.tB[c]);
  q.np = wave_sum_i(q.np), q.nf = wave_sum_i(q.nf), q.nc = wave_sum_i(q.nc);
  const unsigned long long nsurv = *a.surv_cnt;
  const int err = *a.err;
  if (lane == 0) {
    PairOut* r = (PairOut*)rec;
#pragma unroll
    for (int c = 0; c < 3; ++c) r->F_A[c] = q.F[c], r->tau_A[c] = q.tA[c], r->F_B[c] = -q.F[c], r->tau_B[c] = q.tB[c];
    r->n_candidates = q.nc, r->n_polygons = q.np, r->n_faces = q.nf;
    r->status = err ? HCS_ERR_LIMIT : ((int64_t)nsurv > a.surv_cap ? HCS_ERR_CAPACITY : 0);
    if (e == 0) {
      CallTail t{};
      t.nsurv = nsurv, t.npoly = *a.poly_cnt, t.nface = *a.face_cnt, t.ncand = *a.cand_cnt, t.err = err;
      *a.tail = t;
    }
  }
  __syncthreads();
  if (lane < 16) ((unsigned long long*)(a.out + e))[lane] = rec[lane];
}

size_t align16(size_t n) { return (n + 15) & ~(size_t)15; }

}  // namespace

CallSizes call_sizes(const Plan& plan) {
  CallSizes z;
  z.blocks1 = plan.blocks.size();
  z.items = (size_t)std::max(1, plan.nitems);
  z.expand = plan.spread ? HCS_SPREAD_BUDGET : HCS_EXPAND_BUDGET;
  z.live = plan.spread ? z.items + z.expand : std::max<size_t>(z.items, z.expand);
  z.blocks2 = (z.live + HCS_GEN_THREADS - 1) / HCS_GEN_THREADS;
  /* slices of a pair's contributions: about 1024 waves in all, at most 64 per
   * pair */
  z.slices = std::max(1, std::min(64, 1024 / std::max(1, (int)plan.envs.size())));
  return z;
}

size_t call_blob_bytes(const Plan& plan, CallBlob& b) {
  b.state = align16(sizeof(EnvDesc) * plan.envs.size());
  b.blocks = align16(b.state + sizeof(double) * HCS_STATE * plan.envs.size());
  b.xenv = align16(b.blocks + sizeof(int2) * plan.blocks.size());
  b.bytes = align16(b.xenv + sizeof(int) * plan.xenv.size());
  return b.bytes;
}

void call_blob_fill(const Plan& plan, const hcs_pair_in* in, const CallBlob& b, char* dst) {
  std::memcpy(dst, plan.envs.data(), sizeof(EnvDesc) * plan.envs.size());
  for (size_t e = 0; in && e < plan.envs.size(); ++e) {
    double* st = (double*)(dst + b.state) + HCS_STATE * e;
    std::memcpy(st, in[e].X_WA, 12 * sizeof(double));
    std::memcpy(st + 12, in[e].X_WB, 12 * sizeof(double));
    std::memcpy(st + 24, in[e].V_WA, 6 * sizeof(double));
    std::memcpy(st + 30, in[e].V_WB, 6 * sizeof(double));
  }
  if (!plan.blocks.empty()) std::memcpy(dst + b.blocks, plan.blocks.data(), sizeof(int2) * plan.blocks.size());
  if (!plan.xenv.empty()) std::memcpy(dst + b.xenv, plan.xenv.data(), sizeof(int) * plan.xenv.size());
}

/* Device buffers of the step (a fixed slice is checked, not grown). */
int call_reserve(Ctx* c, Pipe& p, const Plan& plan, const CallBlob& b, int64_t cap) {
  const CallSizes z = call_sizes(plan);
  const size_t np = plan.envs.size(), nb = z.blocks1 + z.blocks2;
  int rc;
  if ((rc = ensure(c, p.blob, b.bytes)) || (rc = ensure(c, p.counter, 64)) || (rc = ensure(c, p.surv_cnt, 64)) ||
      (rc = ensure(c, p.err, 64)) || (rc = ensure(c, p.xf, sizeof(double) * 12 * np)) ||
      (rc = ensure(c, p.xtri, sizeof(double) * HCS_XTRI * std::max<int64_t>(1, plan.ntx))) ||
      (rc = ensure(c, p.gen_cnt, sizeof(unsigned) * (nb + 1))) ||
      (rc = ensure(c, p.gen_mask, sizeof(unsigned long long) * nb * kGenWaves)) ||
      (rc = ensure(c, p.gen_item, sizeof(int4) * z.items)) ||
      (plan.spread && (rc = ensure(c, p.gen_off, sizeof(unsigned) * (z.items + 1)))) || (rc = ensure(c, p.pair_lo, sizeof(int) * (np + 1))) ||
      (rc = ensure(c, p.live_item, sizeof(int4) * z.live)) || (rc = ensure(c, p.ncand, sizeof(int) * z.live)) ||
      (rc = ensure(c, p.nsurv, sizeof(unsigned) * (z.live + 1))) ||
      (rc = ensure(c, p.off, sizeof(unsigned) * (z.live + 1))) ||
      (rc = ensure(c, p.scan_tmp, scan_temp_bytes((long long)z.live + 1))) ||
      (rc = ensure(c, p.part, sizeof(RedPart) * np * z.slices)))
    return rc;
  cap = std::max<int64_t>(cap, 4096);
  if ((rc = ensure(c, p.surv, sizeof(int4) * cap)) || (rc = ensure(c, p.contrib, sizeof(Contrib) * cap))) return rc;
  p.cap = cap;
  p.scan_bytes = p.scan_tmp.bytes;
  return HCS_OK;
}

QueryArgs call_args(const Pipe& p, const Plan& plan, const CallBlob& b) {
  QueryArgs a{};
  const char* blob = (const char*)p.blob.ptr;
  a.envs = (const EnvDesc*)blob;
  a.state = (const double*)(blob + b.state);
  a.xf = (const double*)p.xf.ptr;
  a.items = (const Item*)p.live_item.ptr;
  a.live_item = (const int4*)p.live_item.ptr;
  a.nitems = (int)call_sizes(plan).live;
  a.queries_per_lane = 1;
  a.counter = (unsigned*)p.counter.ptr;
  a.live_cnt = (const unsigned*)p.counter.ptr + HCS_QUEUES;
  a.nqueues = 1;
  a.exact_slots = 1;
  a.error = (int*)p.err.ptr;
  a.surv = (int4*)p.surv.ptr;
  a.surv_cnt = (unsigned long long*)p.surv_cnt.ptr;
  a.surv_cap = p.cap;
  a.item_ncand = (int*)p.ncand.ptr;
  a.item_nsurv = (unsigned*)p.nsurv.ptr;
  a.xtri = (const double*)p.xtri.ptr;
  for (const EnvDesc& E : plan.envs) a.kinds |= 1 << E.kind;
  return a;
}

/* Clears, pose composition (with the blob's upload when it has a source) and
 * the two culls. */
int call_front(Ctx* c, Pipe& p, const QueryArgs& a, const Plan& plan, const CallBlob& b, unsigned* const* counters,
               int ncounters) {
  hipStream_t s = c->stream;
  const int np = (int)plan.envs.size(), nblk = (int)plan.blocks.size();
  FrontArgs f{};
  if (b.src) {
    f.src = (const uint4*)b.src, f.dst = (uint4*)p.blob.ptr, f.n16 = (int64_t)(b.bytes / 16);
    f.state = (const double*)((const char*)b.src + b.state);
  } else {
    f.state = a.state;
  }
  f.xf = (double*)p.xf.ptr, f.npairs = np;
  for (DBuf* d : {&p.counter, &p.surv_cnt, &p.err}) f.counters[f.ncounters++] = (unsigned*)d->ptr;
  for (int k = 0; k < ncounters && f.ncounters < kMaxCounters; ++k) f.counters[f.ncounters++] = counters[k];
  const int64_t want = std::max<int64_t>(std::max<int64_t>(f.n16, np), 16 * kMaxCounters);
  hipLaunchKernelGGL(k_call_front, dim3((unsigned)std::min<int64_t>((want + 255) / 256, 1024)), dim3(256), 0, s, f);
  const CallSizes z = call_sizes(plan);
  const char* blob = (const char*)p.blob.ptr;
  const int2* blocks = (const int2*)(blob + b.blocks);
  unsigned *cnt1 = (unsigned*)p.gen_cnt.ptr, *cnt2 = cnt1 + nblk;
  unsigned long long *mask1 = (unsigned long long*)p.gen_mask.ptr, *mask2 = mask1 + (size_t)kGenWaves * nblk;
  int4* item = (int4*)p.gen_item.ptr;
  unsigned *n1 = (unsigned*)p.err.ptr + 4, *live_cnt = (unsigned*)p.counter.ptr + HCS_QUEUES;
  /* beyond a few thousand blocks the sums of the counts before each block
   * would cost more than a scan */
  /* (the error block's words past the error and the zero counter) */
  unsigned* off = plan.spread ? (unsigned*)p.gen_off.ptr : nullptr;
  unsigned long long* sum = (unsigned long long*)((char*)p.err.ptr + 24);
  const bool scan1 = z.blocks1 > 4096, scan2 = z.blocks2 > 4096;
  int rc = 0;
  hipLaunchKernelGGL(k_call_cull1, dim3(nblk), dim3(HCS_GEN_THREADS), 0, s, a.envs, blocks, a.xf, cnt1, mask1);
  if (scan1) rc = exclusive_scan_u32(s, cnt1, cnt1, nblk, p.scan_tmp.ptr, p.scan_bytes);
  hipLaunchKernelGGL(k_call_place1, dim3(nblk + (unsigned)plan.xenv.size()), dim3(HCS_GEN_THREADS), 0, s, a.envs,
                     blocks, nblk, (const unsigned*)cnt1, scan1, (const unsigned long long*)mask1,
                     (const int*)(blob + b.xenv), a.xf, (double*)p.xtri.ptr, item, off, sum, n1);
  const dim3 g2((unsigned)z.blocks2);
  if (rc) return set_err(c, HCS_ERR_LIMIT, "too many work items to scan");
  if (off) {
    const CutArgs cut{n1, sum, (unsigned)c->num_cu * HCS_CUT_SHARES, (unsigned)z.live};
    const dim3 t(HCS_GEN_THREADS), g1((unsigned)(z.items / HCS_GEN_THREADS + 1));
    hipLaunchKernelGGL(k_cut_count, g1, t, 0, s, cut, (const unsigned*)off, cnt2);
    hipLaunchKernelGGL(k_cut_place, g1, t, 0, s, cut, (const unsigned*)cnt2, off);
    hipLaunchKernelGGL(k_cut_cull, g2, t, 0, s, a.envs, a.xf, (const int4*)item, (const unsigned*)n1,
                       (const unsigned*)off, cnt2, mask2);
    hipLaunchKernelGGL(k_cut_keep, g2, t, 0, s, a.envs, (const int4*)item, (const unsigned*)n1, (const unsigned*)off,
                       (const unsigned*)cnt2, (const unsigned long long*)mask2, np, (int4*)p.live_item.ptr, live_cnt,
                       (int*)p.pair_lo.ptr);
    return HCS_OK;
  }
  const unsigned budget = (unsigned)z.expand;
  hipLaunchKernelGGL(k_call_cull2, g2, dim3(HCS_GEN_THREADS), 0, s, a.envs, a.xf, (const int4*)item,
                     (const unsigned*)n1, budget, cnt2, mask2);
  if (scan2) rc |= exclusive_scan_u32(s, cnt2, cnt2, (long long)z.blocks2, p.scan_tmp.ptr, p.scan_bytes);
  if (rc) return set_err(c, HCS_ERR_LIMIT, "too many work items to scan");
  hipLaunchKernelGGL(k_call_place2, g2, dim3(HCS_GEN_THREADS), 0, s, a.envs, (const int4*)item, (const unsigned*)n1,
                     budget, (const unsigned*)cnt2, scan2, (const unsigned long long*)mask2, np,
                     (int4*)p.live_item.ptr, live_cnt, (int*)p.pair_lo.ptr);
  return HCS_OK;
}

/* Scan of the live items' survivor counts, [event e_clip], clip, [event
 * e_reduce], per-pair reduction into out[0..npairs) and *tail (device or
 * mapped host memory). */
int call_back(Ctx* c, Pipe& p, const QueryArgs& a, const Plan& plan, PairOut* out, CallTail* tail, hipEvent_t e_clip,
              hipEvent_t e_reduce) {
  hipStream_t s = c->stream;
  const CallSizes z = call_sizes(plan);
  const int np = (int)plan.envs.size();
  unsigned* off = (unsigned*)p.off.ptr;
  if (z.live <= (size_t)kScanPlaces) {
    hipLaunchKernelGGL(k_call_scan, dim3(1), dim3(kScanThreads), 0, s, (const unsigned*)a.item_nsurv,
                       (const unsigned*)a.live_cnt, off);
  } else if (exclusive_scan_u32(s, a.item_nsurv, off, (long long)z.live + 1, p.scan_tmp.ptr, p.scan_bytes) != 0) {
    /* (entries past the live items are not read) */
    return set_err(c, HCS_ERR_LIMIT, "too many work items to scan");
  }
  if (e_clip) (void)hipEventRecord(e_clip, s);
  launch_clip(c, p, a, clip_grid_for(c, p.cap));
  if (e_reduce) (void)hipEventRecord(e_reduce, s);
  const int K = z.slices;
  hipLaunchKernelGGL(k_call_reduce, dim3(np * K), dim3(64), 0, s, (const int*)p.pair_lo.ptr, K, (const unsigned*)off,
                     (const int*)a.item_ncand, (const unsigned long long*)a.surv_cnt, p.cap,
                     (const Contrib*)p.contrib.ptr, (RedPart*)p.part.ptr);
  CombineArgs q{};
  q.part = (const RedPart*)p.part.ptr, q.K = K;
  q.surv_cnt = a.surv_cnt, q.surv_cap = p.cap, q.err = a.error, q.out = out, q.tail = tail;
  /* a counter the step does not have reads as cleared words of the error
   * block */
  unsigned long long* zero = (unsigned long long*)((char*)p.err.ptr + 8);
  q.poly_cnt = a.poly_cnt ? a.poly_cnt : zero, q.face_cnt = a.face_cnt ? a.face_cnt : zero;
  q.cand_cnt = a.cand_cnt ? a.cand_cnt : zero;
  hipLaunchKernelGGL(k_call_combine, dim3(np), dim3(64), 0, s, q);
  return HCS_OK;
}

int call_enqueue(Ctx* c, Pipe& p, const QueryArgs& a, const Plan& plan, const CallBlob& b, unsigned* const* counters,
                 int ncounters, bool keys, int cand_grid, PairOut* out, CallTail* tail) {
  int rc = call_front(c, p, a, plan, b, counters, ncounters);
  if (rc) return rc;
  launch_cand(c, a, std::min(a.nitems, cand_grid), keys ? CAND_KEYS : CAND_STEP);
  return keys ? HCS_OK : call_back(c, p, a, plan, out, tail, nullptr, nullptr);
}

}  // namespace hcs
