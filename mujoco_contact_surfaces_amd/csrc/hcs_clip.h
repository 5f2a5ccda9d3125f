/*
 * hcs_clip.h -- the forward clip stage of launches that mix pair kinds, a wave
 * of 64 survivors at a time: clip or slice, faces, force law, one contribution
 * per survivor.  The arithmetic is process_candidate's (hcs_query.h), value
 * for value; what differs is how the work lies on the lanes.
 *
 * The register build for all kinds needs private memory and issues each kind's
 * polygon and up to eight faces for all lanes.  Here
 *   - polygons live in LDS, one column per lane, and a clipping plane computes
 *     its two crossings (read back by index) instead of one per possible edge;
 *   - the faces of all 64 polygons are dealt out to the lanes, 64 at a time,
 *     and each polygon's lane adds its faces' results in order;
 *   - divisions by 3 and by a face's slip speed are done with fused
 *     multiply-adds from one reciprocal and rounded as a division would be.
 * Against the register build for all kinds: 12 pairs of a scene 42 -> 25 us, a
 * batch of tet-query and triangle pairs 26 -> 20 us (16 pairs, 3.6k polygons),
 * 150 -> 115 (512, 169k) and 685 -> 512 (4096, 1.35M).  Launches of one kind
 * keep their own register builds: with millions of survivors the LDS round
 * trips of every plane and face cost more there than the instructions saved
 * (2.6M: 0.70 against 0.72 ms).
 */
#pragma once
#include "hcs_query.h"

#pragma clang fp contract(off)

namespace hcs {

#define HCS_CLIP_ST 64 /* column stride: one column per lane */

struct ClipLds {
  double v[3 * HCS_MAXV * HCS_CLIP_ST]; /* coordinate c of vertex k of lane l at (3 k + c) * 64 + l */
  unsigned short face[HCS_MAXV * 64];   /* all faces: lane * 8 + first vertex */
};

/* x / 3, correctly rounded: with y the rounded reciprocal and q = x y within
 * one ulp, q + (x - 3 q) y rounds to the quotient (Markstein; the remainder is
 * exact).  Infinities and NaN pass through q. */
__device__ inline double div3(double x) {
  const double y = 1.0 / 3.0, q = x * y;
  const double r = __builtin_fma(-3.0, q, x);
  return fabs(q) < __builtin_inf() ? __builtin_fma(r, y, q) : q;
}
/* x / b for y = the rounded 1 / b: q may be two ulps off, so the correction
 * is made twice.  For b of moderate size (the caller checks). */
__device__ inline double div_by(double x, double b, double y) {
  double q = x * y;
  q = __builtin_fma(__builtin_fma(-b, q, x), y, q);
  return __builtin_fma(__builtin_fma(-b, q, x), y, q);
}

/* The lane's polygon (at most NIN vertices) cut to nh.x + off <= 0, as
 * clip_halfspace cuts it.  A convex polygon crosses a plane at two edges or
 * none; rounding noise on a nearly coplanar one can give more, which takes the
 * general walk. */
template <int NIN>
__device__ inline void clip_plane(double* col, int& n, const double* nh, double off) {
  double x[NIN], y[NIN], z[NIN];
  unsigned in = 0;
#pragma unroll
  for (int i = 0; i < NIN; ++i) {
    x[i] = col[(3 * i) * HCS_CLIP_ST], y[i] = col[(3 * i + 1) * HCS_CLIP_ST], z[i] = col[(3 * i + 2) * HCS_CLIP_ST];
    const double s = ((nh[0] * x[i] + nh[1] * y[i]) + nh[2] * z[i]) + off;
    in |= (i < n && s <= 0) ? 1u << i : 0u;
  }
  const unsigned all = (1u << n) - 1u;
  if (in == all) return;
  if (in == 0) {
    n = 0;
    return;
  }
  const unsigned cross = in ^ (((in << 1) | (in >> (n - 1))) & all);
  if (__builtin_popcount(cross) != 2) {
    ColPoly P{col, HCS_CLIP_ST, n};
    clip_halfspace_col<NIN>(P, nh, off);
    n = P.n;
    return;
  }
  /* the crossings on the edges that end at vertices e[0] < e[1] */
  const int e[2] = {__builtin_ctz(cross), 31 - __builtin_clz(cross)};
  double q[2][3];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int i = e[k], j = i == 0 ? n - 1 : i - 1;
    const double* c = col + (3 * i) * HCS_CLIP_ST;
    const double* p = col + (3 * j) * HCS_CLIP_ST;
    const double cx = c[0], cy = c[HCS_CLIP_ST], cz = c[2 * HCS_CLIP_ST];
    const double px = p[0], py = p[HCS_CLIP_ST], pz = p[2 * HCS_CLIP_ST];
    const double sc = ((nh[0] * cx + nh[1] * cy) + nh[2] * cz) + off;
    const double sp = ((nh[0] * px + nh[1] * py) + nh[2] * pz) + off;
    const double wa = sp / (sp - sc);
    const double wb = 1.0 - wa;
    q[k][0] = wa * cx + wb * px, q[k][1] = wa * cy + wb * py, q[k][2] = wa * cz + wb * pz;
  }
  /* kept vertices and crossings in walk order */
#pragma unroll
  for (int i = 0; i < NIN; ++i) {
    const int pos = __builtin_popcount(in & ((1u << i) - 1u)) + __builtin_popcount(cross & ((2u << i) - 1u));
    if ((in >> i & 1u) && pos != i) {
      double* d = col + (3 * pos) * HCS_CLIP_ST;
      d[0] = x[i], d[HCS_CLIP_ST] = y[i], d[2 * HCS_CLIP_ST] = z[i];
    }
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    double* d = col + 3 * (__builtin_popcount(in & ((1u << e[k]) - 1u)) + k) * HCS_CLIP_ST;
    d[0] = q[k][0], d[HCS_CLIP_ST] = q[k][1], d[2 * HCS_CLIP_ST] = q[k][2];
  }
  n = __builtin_popcount(in) + 2;
}

/* dedupe_col where something is to be dropped; most polygons have no two
 * neighbouring vertices within 1e-14. */
template <int NMAX>
__device__ inline void drop_duplicates(double* col, int& n) {
  if (n < 3) {
    n = 0;
    return;
  }
  double lx = col[(3 * (n - 1)) * HCS_CLIP_ST], ly = col[(3 * (n - 1) + 1) * HCS_CLIP_ST],
         lz = col[(3 * (n - 1) + 2) * HCS_CLIP_ST];
  bool any = false;
  for (int i = 0; i < n; ++i) {
    const double* v = col + (3 * i) * HCS_CLIP_ST;
    const double x = v[0], y = v[HCS_CLIP_ST], z = v[2 * HCS_CLIP_ST];
    const double dx = lx - x, dy = ly - y, dz = lz - z;
    any = any || ((dx * dx + dy * dy) + dz * dz) < HCS_EPS2;
    lx = x, ly = y, lz = z;
  }
  if (!any) return;
  ColPoly P{col, HCS_CLIP_ST, n};
  dedupe_col<NMAX>(P);
  n = P.n;
}

/* polygon_centroid on a column polygon: the weight sum, and the centroid C. */
__device__ inline double column_centroid(const double* col, int n, const double* nrm, double* C) {
  auto at = [&](int k, double* v) {
    v[0] = col[(3 * k) * HCS_CLIP_ST], v[1] = col[(3 * k + 1) * HCS_CLIP_ST], v[2] = col[(3 * k + 2) * HCS_CLIP_ST];
  };
  double v0[3], a[3], b[3], e1[3], e2[3], cr[3];
  at(0, v0), at(1, a);
  double W = 0.0, S[3] = {0.0, 0.0, 0.0};
  for (int i = 1; i + 1 < n; ++i) {
    at(i + 1, b);
#pragma unroll
    for (int c = 0; c < 3; ++c) e1[c] = a[c] - v0[c], e2[c] = b[c] - v0[c];
    cross3(e1, e2, cr);
    const double w = dot3(cr, nrm);
    if (n == 3) {
#pragma unroll
      for (int c = 0; c < 3; ++c) C[c] = div3((v0[c] + a[c]) + b[c]);
      return w;
    }
    W = W + w;
#pragma unroll
    for (int c = 0; c < 3; ++c) S[c] = S[c] + w * ((v0[c] + a[c]) + b[c]), a[c] = b[c];
  }
  if (W == 0) {
    double m[3] = {0.0, 0.0, 0.0};
    for (int i = 0; i < n; ++i) {
      at(i, a);
#pragma unroll
      for (int c = 0; c < 3; ++c) m[c] = m[c] + a[c];
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) C[c] = m[c] / (double)n;
  } else {
    const double W3 = 3.0 * W;
#pragma unroll
    for (int c = 0; c < 3; ++c) C[c] = S[c] / W3;
  }
  return W;
}

/* Has the values loaded here, where nothing else waits, and not where each is
 * first used. */
template <int N>
__device__ inline void loaded(double* v) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
}

/* One survivor's polygon in the lane's column: n vertices (0: none), the
 * normal nS, the field (gA, cA) of A's tet, and the constants of its faces. */
struct LanePoly {
  int n;
  double nS[3], gA[3], cA, C[3], W2;
  FaceConst<double> fc;
};

__device__ inline void lane_polygon(const EnvDesc& E, const double* st, const double* X, int a, int b, double* col,
                                    LanePoly& p) {
  const int kind = E.kind;
  p.n = 0;
  const HCS_GPTR double* rr = E.recA + (size_t)HCS_TREC * a;
  p.gA[0] = rr[16], p.gA[1] = rr[17], p.gA[2] = rr[18], p.cA = rr[19];
  const double gh[3] = {rr[20], rr[21], rr[22]};
  double gBW[3] = {0.0, 0.0, 0.0};
  if (kind == KIND_SOFT) {
    /* soft-soft: equal-pressure plane of tets a (A) and b (B) */
    const HCS_GPTR double* rb = E.recB + (size_t)HCS_TREC * b;
    const double gbB[3] = {rb[16], rb[17], rb[18]}, ghB[3] = {rb[20], rb[21], rb[22]};
    double pl[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) pl[i] = rb[i];
    double gb[3], gbh[3];
    rot(X, gbB, gb);
    rot(X, ghB, gbh);
    const double cb = rb[19] - dot3(gb, X + 9);
    const double nn[3] = {p.gA[0] - gb[0], p.gA[1] - gb[1], p.gA[2] - gb[2]};
    const double mag = sqrt(dot3(nn, nn));
    if (!(mag > 0.0)) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) p.nS[c] = nn[c] / mag;
    const double off = -((cb - p.cA) / mag);
    if (!(((p.nS[0] * gh[0] + p.nS[1] * gh[1]) + p.nS[2] * gh[2]) > HCS_COS_ALPHA)) return;
    if (!(((-p.nS[0] * gbh[0] + -p.nS[1] * gbh[1]) + -p.nS[2] * gbh[2]) > HCS_COS_ALPHA)) return;
    Poly<double> q;
    if (!slice_tet<double>(E, a, p.nS, off, q)) return;
    loaded<16>(pl);
    p.n = q.n;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      col[(3 * i) * HCS_CLIP_ST] = q.x[i], col[(3 * i + 1) * HCS_CLIP_ST] = q.y[i], col[(3 * i + 2) * HCS_CLIP_ST] = q.z[i];
    /* tet b's half-spaces in A's frame */
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      double pn[3];
      rot(X, pl + 3 * k, pn);
      const double po = pl[12 + k] - dot3(pn, X + 9);
      if (p.n > 0) {
        if (k == 0) clip_plane<4>(col, p.n, pn, po);
        if (k == 1) clip_plane<5>(col, p.n, pn, po);
        if (k == 2) clip_plane<6>(col, p.n, pn, po);
        if (k == 3) clip_plane<7>(col, p.n, pn, po);
      }
    }
    drop_duplicates<8>(col, p.n);
    rot(st + 12, gbB, gBW);
  } else if (kind == KIND_PLANE) {
    /* soft-half-space: B's plane z = 0 (normal +z, out of the rigid side) */
    const double ez[3] = {0.0, 0.0, 1.0};
    rot(X, ez, p.nS);
    if (!(((gh[0] * p.nS[0] + gh[1] * p.nS[1]) + gh[2] * p.nS[2]) > HCS_COS_ALPHA)) return;
    const double off = -dot3(p.nS, X + 9);
    Poly<double> q;
    if (!slice_tet<double>(E, a, p.nS, off, q)) return;
    p.n = q.n;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      col[(3 * i) * HCS_CLIP_ST] = q.x[i], col[(3 * i + 1) * HCS_CLIP_ST] = q.y[i], col[(3 * i + 2) * HCS_CLIP_ST] = q.z[i];
  } else {
    /* soft-rigid: triangle b of the rigid mesh moved into A's frame */
    const HCS_GPTR int32_t* f = E.FB + 3 * (size_t)b;
    const double nR[3] = {E.nrmB[3 * (size_t)b], E.nrmB[3 * (size_t)b + 1], E.nrmB[3 * (size_t)b + 2]};
    double pl[16], y[9];
#pragma unroll
    for (int i = 0; i < 16; ++i) pl[i] = rr[i];
#pragma unroll
    for (int i = 0; i < 3; ++i) xform(X, hcs_plain(E.VB + 3 * (size_t)f[i]), y + 3 * i);
    loaded<9>(y);
    rot(X, nR, p.nS);
    if (!(((gh[0] * p.nS[0] + gh[1] * p.nS[1]) + gh[2] * p.nS[2]) > HCS_COS_ALPHA)) return;
    loaded<16>(pl);
#pragma unroll
    for (int i = 0; i < 9; ++i) col[i * HCS_CLIP_ST] = y[i];
    p.n = 3;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double* nh = pl + 3 * k;
      const double off = pl[12 + k];
      if (p.n > 0) {
        if (k == 0) clip_plane<3>(col, p.n, nh, off);
        if (k == 1) clip_plane<4>(col, p.n, nh, off);
        if (k == 2) clip_plane<5>(col, p.n, nh, off);
        if (k == 3) clip_plane<6>(col, p.n, nh, off);
      }
    }
    drop_duplicates<7>(col, p.n);
  }
  if (p.n < 3) {
    p.n = 0;
    return;
  }
  p.W2 = column_centroid(col, p.n, p.nS, p.C);
  double nW[3], gAW[3];
  rot(st, p.nS, nW);
  rot(st, p.gA, gAW);
  PairW<double> pw;
  pw.a_is_M = E.a_is_M, pw.b_soft = E.b_soft;
  face_const(pw, nW, gAW, gBW, p.fc);
}

/* A record slot for each active lane: one atomic on the counter. */
__device__ inline int64_t reserve(unsigned long long* cnt) {
  const unsigned long long m = __ballot(1);
  const int lead = __builtin_ctzll(m);
  unsigned long long base = 0;
  if ((int)(threadIdx.x & 63) == lead) base = atomicAdd(cnt, (unsigned long long)__popcll(m));
  return (int64_t)(__shfl(base, lead, 64) + lane_prefix(m));
}

/* The lane's polygon kept for the sensors (the record of emit_polygon). */
__device__ inline void keep_polygon(const OutPtrs& o, const double* st, const double* col, const LanePoly& p, int env,
                                    int ea, int eb) {
  const int64_t slot = reserve(o.poly_cnt);
  if (slot >= o.poly_cap) return;
  double* P = o.poly_rec + slot * HCS_PREC;
  P[0] = p.n;
  for (int i = 0; i < 8; ++i) {
    double y[3] = {0.0, 0.0, 0.0}, f = 0.0;
    if (i < p.n) {
      const double* v = col + (3 * i) * HCS_CLIP_ST;
      const double x[3] = {v[0], v[HCS_CLIP_ST], v[2 * HCS_CLIP_ST]};
      xform(st, x, y);
      f = p.cA + dot3(p.gA, x);
    }
    P[1 + 3 * i] = y[0], P[2 + 3 * i] = y[1], P[3 + 3 * i] = y[2];
    P[25 + i] = f;
  }
  double y[3], nW[3];
  xform(st, p.C, y);
  rot(st, p.nS, nW);
  P[33] = y[0], P[34] = y[1], P[35] = y[2], P[36] = p.cA + dot3(p.gA, p.C);
  P[37] = nW[0], P[38] = nW[1], P[39] = nW[2];
  o.poly_key[3 * slot] = env, o.poly_key[3 * slot + 1] = ea, o.poly_key[3 * slot + 2] = eb;
}

/* One face: eval_face's arithmetic on pair constants read where they lie (the
 * lanes of a round mostly share a pair, so the reads are broadcasts).  f:
 * force on A, torques about A's and B's origins. */
__device__ inline void face_force(const EnvDesc& E, const double* st, const double* n, double fn0,
                                  double k, const double* cW, double* f) {
  const bool aM = E.a_is_M;
  const double oA[3] = {st[9], st[10], st[11]}, oB[3] = {st[21], st[22], st[23]};
  double rA[3], rB[3], wA[3], wB[3], v[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) rA[c] = cW[c] - oA[c], rB[c] = cW[c] - oB[c];
  cross3(st + 24, rA, wA);
  cross3(st + 30, rB, wB);
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double vA = st[27 + c] + wA[c], vB = st[33 + c] + wB[c];
    v[c] = aM ? vA - vB : vB - vA;
  }
  const double vn = dot3(v, n);
  /* plugin.cpp:458 */
  const double fn = dmax0(1. - E.dstar * vn) * (fn0 - E.dt * k * vn);
  double fM[3] = {0.0, 0.0, 0.0};
  if (E.apply) {
    /* plugin.cpp:462-475 */
    const double stiction_tolerance = 1.0e-4;
    const double relative_tolerance = 1.0e-2;
    double vt[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) vt[c] = v[c] - n[c] * vn;
    double eps = stiction_tolerance * relative_tolerance;
    eps = eps * eps;
    const double v_slip = sqrt(dot3(vt, vt) + eps); /* at least 1e-6 */
    double mu_reg = E.mu, that[3];
    if (v_slip < 1e100) {
      const double s = div_by(v_slip, stiction_tolerance, 1.0 / stiction_tolerance);
      if (s < 1) mu_reg = E.mu * s * (2.0 - s);
      const double y = 1.0 / v_slip;
#pragma unroll
      for (int c = 0; c < 3; ++c) that[c] = div_by(vt[c], v_slip, y);
    } else {
#pragma unroll
      for (int c = 0; c < 3; ++c) that[c] = vt[c] / v_slip;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double f_slip = -mu_reg * that[c] * fn;
      fM[c] = f_slip + fn * n[c];
    }
  }
  /* +f on M, -f on N; reported on A (about o_A) and B (about o_B). */
  double fB[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    f[c] = aM ? fM[c] : -fM[c];
    fB[c] = -f[c];
  }
  cross3(rA, f, f + 3);
  cross3(rB, fB, f + 6);
}

/* One lane's survivor: elements a, b of pair env (-1: none), and the slot of
 * its contribution. */
struct LaneWork {
  int a, b, env;
  int64_t slot;
};
__device__ inline LaneWork lane_work(const QueryArgs& A, const ClipArgs& C, const int4& s) {
  /* (x -1: an unused slot of a wave's reserved chunk) */
  LaneWork w{s.x, s.y, -1, 0};
  if (s.x >= 0) {
    w.slot = (int64_t)C.item_off[s.z] + (unsigned)s.w;
    if (w.slot < C.cap) w.env = A.items[s.z].env;
  }
  return w;
}

/* The survivors i0, i0 + step, ... of one wave, 64 at a time; the next 64 are
 * fetched while these are worked on. */
__device__ inline void clip_wave(ClipLds& L, const QueryArgs& A, const ClipArgs& C, int64_t i0, int64_t step,
                                 int64_t n, const OutPtrs& o, Contrib* out) {
  const int lane = threadIdx.x & 63;
  double* col = L.v + lane;
  const int4 none = make_int4(-1, -1, -1, -1);
  LaneWork s = lane_work(A, C, i0 + lane < n ? A.surv[i0 + lane] : none);
  for (; i0 < n; i0 += step) {
    const int64_t in = i0 + step + lane;
    const int4 next = in < n ? A.surv[in] : none;
    const bool on = s.env >= 0;
    const int env = on ? s.env : 0;
    LanePoly p;
    p.n = 0;
    if (on) {
      const EnvDesc& E = A.envs[env];
      const double* st = A.state + (size_t)HCS_STATE * env;
      double X[12];
#pragma unroll
      for (int k = 0; k < 12; ++k) X[k] = A.xf[12 * (size_t)env + k];
      lane_polygon(E, st, X, s.a, s.b, col, p);
      if (p.n > 0 && o.poly_rec && (!o.poly_env || o.poly_env[env]))
        keep_polygon(o, st, col, p, env, s.a, s.b);
    }
    /* the polygons' faces (one of the whole polygon in the kPolygon
     * representation), numbered lane after lane */
    const bool whole = on && A.envs[env].repr != 0;
    const int nf = p.n > 0 ? (whole ? 1 : p.n) : 0;
    int first = nf;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int u = (int)__shfl((unsigned)first, lane >= d ? lane - d : lane, 64);
      if (lane >= d) first += u;
    }
    const int total = (int)__shfl((unsigned)first, 63, 64);
    first -= nf;
    for (int k = 0; k < nf; ++k) L.face[first + k] = (unsigned short)(lane * 8 + k);
    __syncthreads();
    const LaneWork sn = lane_work(A, C, next);
    double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    int faces = 0;
    for (int r0 = 0; r0 < total; r0 += 64) {
      const bool have = r0 + lane < total;
      const int fk = have ? L.face[r0 + lane] : lane * 8;
      const int w = fk >> 3, k = fk & 7;
      /* the owner's polygon */
      const int ow_n = (int)__shfl((unsigned)p.n, w, 64), ow_env = (int)__shfl((unsigned)env, w, 64);
      const bool ow_ok = __shfl((unsigned)(p.n > 0 && p.fc.ok), w, 64) != 0;
      const bool ow_whole = __shfl((unsigned)whole, w, 64) != 0;
      double Cc[3], gA[3], nW[3];
#pragma unroll
      for (int c = 0; c < 3; ++c)
        Cc[c] = __shfl(p.C[c], w, 64), gA[c] = __shfl(p.gA[c], w, 64), nW[c] = __shfl(p.fc.n[c], w, 64);
      const double cA = __shfl(p.cA, w, 64), g = __shfl(p.fc.g, w, 64), W2 = __shfl(p.W2, w, 64);
      bool hit = false;
      double f[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
      int ow_a = 0, ow_b = 0;
      if (o.face_rec) ow_a = (int)__shfl((unsigned)s.a, w, 64), ow_b = (int)__shfl((unsigned)s.b, w, 64);
      if (have) {
        const EnvDesc& E = A.envs[ow_env];
        const double* st = A.state + (size_t)HCS_STATE * ow_env;
        const double pC = cA + dot3(gA, Cc);
        double area, cS[3], p0;
        if (!ow_whole) {
          const int k1 = (k + 1 == ow_n) ? 0 : k + 1;
          const double* va = L.v + w + (3 * k) * HCS_CLIP_ST;
          const double* vb = L.v + w + (3 * k1) * HCS_CLIP_ST;
          const double a[3] = {va[0], va[HCS_CLIP_ST], va[2 * HCS_CLIP_ST]};
          const double b[3] = {vb[0], vb[HCS_CLIP_ST], vb[2 * HCS_CLIP_ST]};
          const double e1[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]};
          const double e2[3] = {Cc[0] - a[0], Cc[1] - a[1], Cc[2] - a[2]};
          double cr[3];
          cross3(e1, e2, cr);
          area = 0.5 * sqrt(dot3(cr, cr));
#pragma unroll
          for (int c = 0; c < 3; ++c) cS[c] = div3((a[c] + b[c]) + Cc[c]);
          const double third = 1.0 / 3.0, pa = cA + dot3(gA, a), pb = cA + dot3(gA, b);
          p0 = (third * pa + third * pb) + third * pC;
        } else {
          area = 0.5 * W2;
          cS[0] = Cc[0], cS[1] = Cc[1], cS[2] = Cc[2];
          p0 = pC;
        }
        /* (computed for a face that is none too: no branch before its loads) */
        double cW[3];
        xform(st, cS, cW);
        const double fn0 = area * p0, ka = area * g;
        face_force(E, st, nW, fn0, ka, cW, f);
        hit = area > 1.0e-14 && ow_ok;
        if (o.face_rec && hit) {
          const int64_t slot = reserve(o.face_cnt);
          if (slot < o.face_cap) {
            double* r = o.face_rec + slot * HCS_FREC;
#pragma unroll
            for (int c = 0; c < 3; ++c) r[c] = cW[c], r[3 + c] = nW[c];
            r[6] = fn0, r[7] = ka, r[8] = E.dstar, r[9] = area, r[10] = p0, r[11] = g;
            int64_t* key = o.face_key + 4 * slot;
            key[0] = ow_env, key[1] = ow_a, key[2] = ow_b, key[3] = k;
          }
        }
      }
      const unsigned long long m = __ballot(hit);
      /* each polygon's lane adds its faces of this round, in order */
      const int b0 = max(first, r0), nb = min(first + nf, r0 + 64) - b0;
      for (int t = 0; __ballot(t < nb) != 0; ++t) {
        const int q = (b0 - r0 + t) & 63;
        const bool add = t < nb && (m >> q & 1);
#pragma unroll
        for (int c = 0; c < 9; ++c) {
          const double x = __shfl(f[c], q, 64);
          acc[c] = add ? acc[c] + x : acc[c];
        }
        faces += add;
      }
    }
    if (on) {
      Contrib r;
#pragma unroll
      for (int c = 0; c < 3; ++c) r.F[c] = acc[c], r.tA[c] = acc[3 + c], r.tB[c] = acc[6 + c];
      r.np = p.n > 0 ? 1 : 0, r.nf = faces;
      out[s.slot] = r;
    }
    s = sn;
    __syncthreads(); /* the columns and the face list are written anew */
  }
}

}  // namespace hcs
