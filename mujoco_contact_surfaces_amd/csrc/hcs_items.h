/*
 * hcs_items.h -- the work items of per-call steps and unconfigured batches, as
 * they are enumerated, culled and cut on the device.
 */
#pragma once
#include "hcs_query.h"

#pragma clang fp contract(off)

namespace hcs {

/* The candidates a spread plan's items are cut to: 1 / (32 num_cu) of the
 * expected total, within these.  (256 .. 1024 cut more items that turn out
 * nearly empty: 2048 objects 1.06 ms for 0.90; 1024 .. 4096: 400 objects 397
 * us for 370.) */
#define HCS_CUT_MIN 512
#define HCS_CUT_MAX 2048
#define HCS_CUT_SHARES 32

/* The box of the subtree `root` of A. */
__device__ inline void subtree_box(const EnvDesc& E, int root, double* T) {
  if (E.ntA == 1 || root < 0) {
    const HCS_GPTR double* b = E.boxA + 6 * (size_t)(E.ntA == 1 ? 0 : ~root);
#pragma unroll
    for (int c = 0; c < 6; ++c) T[c] = b[c];
  } else {
    const HCS_GPTR Node& N = E.nodesA[root];
#pragma unroll
    for (int c = 0; c < 3; ++c) T[c] = fmin(N.b[c], N.b[6 + c]), T[3 + c] = fmax(N.b[3 + c], N.b[9 + c]);
  }
}

/* Whether a chunk's box Q can meet the subtree `root` of A under pose X (the
 * test of the batched cull). */
__device__ inline bool may_meet_subtree(const EnvDesc& E, const double* X, const double* Q, int root) {
  if (root == HCS_WNONE) return false;
  double T[6];
  subtree_box(E, root, T);
  return boxes_may_overlap(X, Q, T);
}

/* About how many of a chunk's queries x a subtree's tets are candidates: the
 * queries spread evenly over the chunk's box (in A's frame) with their mean
 * extents, the tets over the subtree's with those of a filled box, each axis
 * by itself.  Only the cut of the items depends on it. */
__device__ inline unsigned expected_candidates(const EnvDesc& E, const double* X, int chunk, int root, int leaves) {
  double Q[6], T[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) Q[c] = E.cboxQ[6 * (size_t)chunk + c];
  subtree_box(E, root, T);
  const float nt = (float)leaves, nq = (float)min(64, E.nB - 64 * chunk);
  float lt[3], vol = 1.f;
#pragma unroll
  for (int c = 0; c < 3; ++c) lt[c] = fmaxf((float)(T[3 + c] - T[c]), 1e-30f), vol *= lt[c];
  const float s = 1.8f * cbrtf(vol / nt);
  float p = nt * nq;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    float c1 = (float)X[9 + i], h1 = 1e-30f, hq = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float r = (float)X[3 * i + k];
      c1 += r * (float)(0.5 * (Q[k] + Q[3 + k])), h1 += fabsf(r) * (float)(0.5 * (Q[3 + k] - Q[k]));
      hq += fabsf(r) * (float)E.csizeQ[3 * (size_t)chunk + k];
    }
    const float in = fminf(c1 + h1, (float)T[3 + i]) - fmaxf(c1 - h1, (float)T[i]);
    p *= fminf(1.f, (fmaxf(in, 0.f) + s) / lt[i]) * fminf(1.f, (2.f * hq + s) / (2.f * h1));
  }
  return (unsigned)fminf(fmaxf(p, 0.f), 1e9f);
}

__device__ inline void chunk_box(const EnvDesc& E, int chunk, double* Q) {
#pragma unroll
  for (int c = 0; c < 6; ++c) Q[c] = E.cboxQ[6 * (size_t)chunk + c];
}

__device__ inline bool is_tree(const EnvDesc& E) { return E.kind == KIND_TRI || E.kind == KIND_SOFT; }

/* Item i of the first cull of a pair: a chunk of 64 queries against one
 * subtree of the pair's frontier (against everything for tet and half-space
 * items). */
__device__ inline bool first_item(const EnvDesc& E, const double* X, int i, int& chunk, int& node) {
  const int depth = is_tree(E) ? E.depth : 0;
  chunk = i >> depth;
  node = (1 << depth) + (i & ((1 << depth) - 1)); /* its place in rootsA */
  double Q[6];
  chunk_box(E, chunk, Q);
  if (E.kind == KIND_PLANE) return box_may_meet_plane(X, Q);
  if (E.kind == KIND_TET) return boxes_may_overlap(X, hcs_plain(E.boxB), Q);
  return may_meet_subtree(E, X, Q, E.rootsA[node]);
}

/* The second cull's levels below an item of the first, of the e the launch
 * has room for: within the frontiers kept, down to subtrees of about 32 tets. */
__device__ inline int levels_below(const EnvDesc& E, int e) {
  if (!is_tree(E)) return 0;
  int n = 0;
  while (n < e && E.depth + n < HCS_ROOT_DEPTH && (E.ntA >> (E.depth + n)) > 32) ++n;
  return n;
}
__device__ inline int expand_levels(unsigned n1, unsigned budget) {
  int e = 0;
  while (e < HCS_ROOT_DEPTH && ((unsigned long long)n1 << (e + 1)) <= budget) ++e;
  return e;
}

/* An item's expected candidates, and the levels it can be cut (to about 16
 * tets), in one word.  A soft query's candidate costs about four of a
 * triangle's. */
constexpr unsigned kEstMask = (1u << 28) - 1;
__device__ inline unsigned cut_word(const EnvDesc& E, const double* X, int chunk, int root) {
  if (!is_tree(E)) return 0u;
  const int leaves = root < 0 || E.ntA == 1 ? 1 : E.nodesA[root].leaves;
  unsigned n = 0;
  while (n < 15 && (leaves >> n) > 16) ++n;
  const unsigned est = min(expected_candidates(E, X, chunk, root, leaves), 1u << 25);
  return (E.kind == KIND_SOFT ? 4 * est : est) | n << 28;
}
/* The pieces an item is cut into: halved until at most the target is left. */
__device__ inline unsigned cut_slots(unsigned word, unsigned target) {
  const unsigned q = (word & kEstMask) / target;
  return 1u << min(q > 0 ? 32u - (unsigned)__builtin_clz(q) : 0u, word >> 28);
}
/* Subtree number sub of the 2^n below root; a leaf reached earlier is its
 * first subtree only. */
__device__ inline int cut_root(const EnvDesc& E, int root, int n, int sub) {
  for (int b = n - 1; b >= 0; --b) {
    if (root < 0) return (sub & ((2 << b) - 1)) == 0 ? root : HCS_WNONE;
    root = E.nodesA[root].c[sub >> b & 1];
  }
  return root;
}

/* ---- the second cull: the kept items cut e levels deeper, the same e for the
 * launch */

/* Piece t: its item, its number in it and the place of its root. */
__device__ inline bool second_item(const EnvDesc* __restrict__ envs, const int4* __restrict__ item, unsigned n1,
                                   unsigned budget, unsigned t, int& i, int& sub, int& node) {
  const int e = expand_levels(n1, budget);
  i = (int)(t >> e), sub = (int)(t & ((1u << e) - 1));
  if ((unsigned)i >= n1) return false;
  const int4 it = item[i];
  const int n = levels_below(envs[it.x], e);
  node = (it.z << n) + sub;
  return sub < (1 << n);
}

__device__ inline int4 live_record(const EnvDesc& E, const int4& it, int root) {
  const int nq = is_tree(E) ? E.nB : E.ntA;
  return make_int4(it.x, 64 * it.y, min(64, nq - 64 * it.y), is_tree(E) ? root : 0);
}

/* ---- spread plans: each item cut by its expected candidates */

/* The candidates an item is cut to: a share of the total that gives every
 * wave several items, and few enough pieces for the room (an item of est
 * candidates has fewer than 1 + 2 est / target pieces). */
struct CutArgs {
  const unsigned* n;             /* items */
  const unsigned long long* sum; /* of their expected candidates */
  unsigned shares, room;
};
__device__ inline unsigned cut_target(const CutArgs& c) {
  const unsigned long long sum = *c.sum, room = c.room - min(c.room, *c.n);
  unsigned long long t = min(max(sum / c.shares, (unsigned long long)HCS_CUT_MIN), (unsigned long long)HCS_CUT_MAX);
  t = max(t, 2 * sum / max(1ull, room) + 1);
  return (unsigned)min(t, (unsigned long long)kEstMask);
}

/* The item that piece t belongs to. */
__device__ inline bool piece(const unsigned* __restrict__ off, unsigned n, unsigned t, int& i, int& sub, int& levels) {
  if (n == 0 || t >= off[n]) return false;
  unsigned lo = 0, hi = n;
  while (hi - lo > 1) {
    const unsigned mid = (lo + hi) / 2;
    if (off[mid] <= t) lo = mid;
    else hi = mid;
  }
  const unsigned first = off[lo];
  i = (int)lo, sub = (int)(t - first), levels = __builtin_ctz(off[lo + 1] - first);
  return true;
}

}  // namespace hcs
