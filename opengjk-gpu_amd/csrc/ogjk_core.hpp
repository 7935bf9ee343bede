// opengjk-amd device core: mixed-precision support sweep, GJK and EPA for one
// pair on a group of LPP lanes.
//
// Precision design
//   * Vertices are stored as FP32.  The O(n) support sweep runs in FP32
//     (explicit FMAs) over an exactly power-of-two-scaled copy of the
//     direction, tracking each lane's best and second-best value.
//   * A rigorous bound on |FP32 dot - FP64 dot| (16 ulp of the direction's
//     max-norm times the body's max L1 vertex norm) defines a candidate
//     window below the FP32 maximum.  Only candidates are re-evaluated in
//     FP64 with the reference's association, so the selected vertex is exactly
//     the one the FP64 reference support selects, ties included.
//   * Everything that is O(1) per iteration (simplex, sub-distance regions,
//     termination, witnesses, EPA faces and horizon) runs in FP64 in the
//     reference's operation order, without FMA contraction.
//   Result: outputs match the FP64 CPU reference bit for bit before the final
//   rounding to the gkFloat ABI.
#pragma once

#include <type_traits>

#include "ogjk_math.hpp"

namespace ogjk {

// ------------------------------------------------------------------ bodies

// Vertex i of a body lives at x[i*STRIDE], y[i*STRIDE], z[i*STRIDE]:
// STRIDE 1 is the SoA scene, STRIDE 3 reads caller AoS coordinates in place.
// T is the storage type: float (the product path) or double (plain FP64).
template <class T, int STRIDE>
struct Body {
  using Elem = T;
  const T* x;
  const T* y;
  const T* z;
  int n;
  float r1;  // >= max_i |x_i|+|y_i|+|z_i| (used by the float sweep only)
  OGJK_DEV T rx(int i) const { return x[(int64_t)i * STRIDE]; }
  OGJK_DEV T ry(int i) const { return y[(int64_t)i * STRIDE]; }
  OGJK_DEV T rz(int i) const { return z[(int64_t)i * STRIDE]; }
  OGJK_DEV double c(int i, int k) const { return (double)(k == 0 ? rx(i) : (k == 1 ? ry(i) : rz(i))); }
  OGJK_DEV D3 d(int i) const { return D3{(double)rx(i), (double)ry(i), (double)rz(i)}; }
};

// Max L1 vertex norm over the group (FP32, rounded up by a relative 2^-22).
template <int LPP, class T, int STRIDE>
OGJK_DEV float body_r1(const Body<T, STRIDE>& b, int lane) {
  float m = 0.0f;
  for (int i = lane; i < b.n; i += LPP) {
    const float s = fabsf((float)b.rx(i)) + fabsf((float)b.ry(i)) + fabsf((float)b.rz(i));
    m = fmaxf(m, s);
  }
  m = group_max_f<LPP>(m);
  return m * (1.0f + 0x1.0p-22f);
}

// --------------------------------------------------------------- support

// Result of a support query: the selected vertex index and its coordinates
// (exact FP64 conversion of the stored values).
struct Sup {
  int i;
  D3 p;
};

// One support query.  has_inc selects the reference's rule:
//   has_inc: GJK (GJK/cpu/openGJK.c:615-639): the incumbent support point
//            keeps its place unless some vertex is strictly better; then the
//            lowest index attaining the maximum wins.
//   !has_inc: EPA (GJK/cpu/EPA.c:310-335): running max starts at -1e10, the
//            lowest index attaining the maximum wins; index -1 if none beats
//            -1e10.
struct Query {
  D3 dir;
  bool has_inc;
  int inc_idx;
  D3 inc_pt;
  bool unit = false;  // |dir| = 1 up to rounding: no scaling needed
};

// A lane's FP64-exact candidate after the sweep: value, index, point.
struct Cand {
  double v;
  int i;
  D3 p;
};

// FP32 sweep state of one lane.
struct Sweep32 {
  float dx, dy, dz;
  float best, second, bx, by, bz;
  int bi;
};

// Scale the direction by an exact power of two so its max-norm is in
// [0.5, 1): the FP32 copy then carries a relative error <= 2^-24 per
// component whatever the magnitude of dir (tiny GJK directions included).
// A unit direction is taken as it is (max-norm in [0.57, 1 + 2^-50]).
OGJK_DEV Sweep32 sweep32_begin(D3 dir, bool unit = false) {
  Sweep32 s;
  if (unit) {
    s.dx = (float)dir.x;
    s.dy = (float)dir.y;
    s.dz = (float)dir.z;
  } else {
    const double mx = fmax(fabs(dir.x), fmax(fabs(dir.y), fabs(dir.z)));
    int e = 0;
    (void)frexp(mx, &e);
    const double sc = ldexp(1.0, -e);
    s.dx = (float)(dir.x * sc);
    s.dy = (float)(dir.y * sc);
    s.dz = (float)(dir.z * sc);
  }
  s.best = s.second = -INFINITY;
  s.bx = s.by = s.bz = 0.0f;
  s.bi = -1;
  return s;
}

// The sweep's update for one vertex (d = -inf leaves the state as it is).
// Selects, not a branch: the update costs less than the jump round it.
OGJK_DEV void sweep32_take(Sweep32& s, float px, float py, float pz, float d, int i) {
  s.second = fmaxf(s.second, fminf(s.best, d));
  const bool better = d > s.best;
  s.best = better ? d : s.best;
  s.bi = better ? i : s.bi;
  s.bx = better ? px : s.bx;
  s.by = better ? py : s.by;
  s.bz = better ? pz : s.bz;
}

// U vertices of the sweep in flight: base + lane, base + LPP + lane, ...
template <int LPP, int U, int STRIDE>
OGJK_DEV void sweep32_batch(const Body<float, STRIDE>& b, int base, int lane, Sweep32& s) {
  float px[U], py[U], pz[U];
#pragma unroll
  for (int k = 0; k < U; k++) {
    const int i = min(base + k * LPP + lane, b.n - 1);
    px[k] = b.rx(i);
    py[k] = b.ry(i);
    pz[k] = b.rz(i);
  }
#pragma unroll
  for (int k = 0; k < U; k++) {
    const int i = base + k * LPP + lane;
    const float d = fmaf(px[k], s.dx, fmaf(py[k], s.dy, pz[k] * s.dz));
    sweep32_take(s, px[k], py[k], pz[k], i < b.n ? d : -INFINITY, i);
  }
}

// One lane's share of the FP32 sweep: vertices lane, lane + LPP, ...  Up to
// four of them are loaded at a time: with one per trip the loop waits out a
// memory round trip for every LPP vertices, and a sweep is little else.
template <int LPP, int STRIDE>
OGJK_DEV void sweep32(const Body<float, STRIDE>& b, int lane, Sweep32& s) {
  int base = 0;
#pragma clang loop unroll(disable)
  for (; base + 2 * LPP < b.n; base += 4 * LPP) sweep32_batch<LPP, 4>(b, base, lane, s);
  if (base + LPP < b.n) {
    sweep32_batch<LPP, 2>(b, base, lane, s);
  } else if (base < b.n) {
    sweep32_batch<LPP, 1>(b, base, lane, s);
  }
}

// Candidates within T of the FP32 maximum, re-ranked in FP64 with the
// reference's association.  `multi`: some lane of the group has more than one
// candidate, so every lane rescans its vertices inside the window.
template <int LPP, int STRIDE>
OGJK_DEV Cand candidates32(const Body<float, STRIDE>& b, const Sweep32& s, float T, bool multi,
                           D3 dir, int lane) {
  Cand c{-INFINITY, 0x7fffffff, D3{0.0, 0.0, 0.0}};
  if (!multi) {
    if (s.bi >= 0 && s.best >= T) {
      c.p = D3{(double)s.bx, (double)s.by, (double)s.bz};
      c.v = dot(c.p, dir);
      c.i = s.bi;
    }
  } else {
    for (int i = lane; i < b.n; i += LPP) {
      const float px = b.rx(i), py = b.ry(i), pz = b.rz(i);
      const float d = fmaf(px, s.dx, fmaf(py, s.dy, pz * s.dz));
      if (d >= T) {
        const D3 p{(double)px, (double)py, (double)pz};
        const double v = dot(p, dir);
        if (v > c.v) {  // ascending i within the lane keeps the lowest index
          c.v = v;
          c.i = i;
          c.p = p;
        }
      }
    }
  }
  if (!(c.v == c.v)) c.v = -INFINITY;
  return c;
}

// Group argmax of the lanes' candidates (lowest index on ties), then the
// acceptance rule of the query and the winner's point.  Usual case: one lane
// holds the only candidate and a single parallel shuffle fetches it.
// STRIDED: lane l swept indices l, l+LPP, ..., so the winner's index names
// its lane; otherwise the lane holding the winning index is found by ballot.
template <int LPP, bool STRIDED = true>
OGJK_DEV Sup finish1(Cand c, const Query& q) {
  const uint64_t holders = group_ballot<LPP>(c.v > -INFINITY);
  int src;
  if (__popcll(holders) == 1) {
    src = (int)__builtin_ctzll(holders);
    c.v = shfl_d<LPP>(c.v, src);
    c.i = shfl_i<LPP>(c.i, src);
  } else {
    const int mine = c.i;
    group_argmax_d<LPP>(c.v, c.i);
    if constexpr (STRIDED) {
      src = c.i & (LPP - 1);
    } else {
      src = (int)__builtin_ctzll(group_ballot<LPP>(mine == c.i) | (1ull << 63));
    }
  }
  if (q.has_inc && !(c.v > dot(q.inc_pt, q.dir))) return Sup{q.inc_idx, q.inc_pt};
  if (!q.has_inc && !(c.v > -1e10)) return Sup{-1, D3{0.0, 0.0, 0.0}};
  return Sup{c.i, D3{shfl_d<LPP>(c.p.x, src), shfl_d<LPP>(c.p.y, src), shfl_d<LPP>(c.p.z, src)}};
}

// The support point of a float body with its coordinates as stored (they are
// exact in FP32, so a group exchanges half the words).
struct SupF {
  int i;
  float x, y, z;
};
OGJK_DEV Sup widen(const SupF& s) { return Sup{s.i, D3{(double)s.x, (double)s.y, (double)s.z}}; }

// The acceptance rule for the only vertex r in the window of a float body's
// query, t the window's lower end.  FP32 settles it nearly always: r is the
// incumbent, or beats it by more than the window, or (EPA, unit direction: sweep
// values are not scaled) the window lies far above -1e10.
OGJK_DEV SupF accept(const SupF& r, const Query& q, const Sweep32& sw, float t) {
  const D3 p{(double)r.x, (double)r.y, (double)r.z};
  if (q.has_inc) {
    const float ix = (float)q.inc_pt.x, iy = (float)q.inc_pt.y, iz = (float)q.inc_pt.z;
    const float di = fmaf(ix, sw.dx, fmaf(iy, sw.dy, iz * sw.dz));
    if (r.i != q.inc_idx && !(t > di) && !(dot(p, q.dir) > dot(q.inc_pt, q.dir)))
      return SupF{q.inc_idx, ix, iy, iz};
  } else if (!(q.unit && t > -1e9f) && !(dot(p, q.dir) > -1e10)) {
    return SupF{-1, 0.0f, 0.0f, 0.0f};
  }
  return r;
}

// Support point of one body (FP32 sweep, FP64 re-rank of the window).  Nearly
// always a single vertex lies in the window: its lane is known from one
// ballot, and its index and FP32 point are fetched.
template <int LPP, int STRIDE>
OGJK_DEV SupF support_f(const Body<float, STRIDE>& A, const Query& q, int lane) {
  Sweep32 sw = sweep32_begin(q.dir, q.unit);
  sweep32<LPP>(A, lane, sw);
  const float m = group_max_f<LPP>(sw.best);
  // |D32 - scale*D64| <= 16u * r1 (u = 2^-24): candidates lie within 2x that.
  const float t = m - 0x1.0p-19f * A.r1;
  const bool multi = group_any<LPP>(sw.second >= t);
  const auto holders = lanes_where<LPP>(sw.bi >= 0 && sw.best >= t);
  if (!multi && count_lanes<LPP>(holders) == 1) {
    const int src = first_lane<LPP>(holders);
    return accept(SupF{shfl_i<LPP>(sw.bi, src), shfl_f<LPP>(sw.bx, src),
                       shfl_f<LPP>(sw.by, src), shfl_f<LPP>(sw.bz, src)},
                  q, sw, t);
  }
  const Sup r = finish1<LPP>(candidates32<LPP>(A, sw, t, multi, q.dir, lane), q);
  return SupF{r.i, (float)r.p.x, (float)r.p.y, (float)r.p.z};
}
template <int LPP, int STRIDE>
OGJK_DEV Sup support(const Body<float, STRIDE>& A, const Query& q, int lane) {
  return widen(support_f<LPP>(A, q, lane));
}

// ------------------------------------------------ clustered support sweep
//
// A scene body may carry a second copy of its vertices ordered by direction
// from the body's centre (Hilbert order of the octahedral map), cut into
// clusters of kCluster slots, each with a bounding sphere (float centre c,
// radius r >= max |x - c|) and box (half extents h about c).  A support
// query then
//   1. bounds every cluster: ub = c.d + min(r|d|, h.|d|) >= max of x.d,
//   2. sweeps the cluster with the largest ub: m0 = its FP32 maximum,
//   3. sweeps only the clusters with ub >= m0 - 2^-15 r1.
// Rounding: |fl(ub) - ub| <= 2^-17 r1 and |D32 - D| <= 2^-20 r1 (d scaled to
// max-norm in [0.5,1), |c|_1 <= 3 r1, |h|_1 <= 3 r1, r <= 2 r1), so every skipped vertex
// lies more than 2^-16 r1 below the maximum: it can neither be the FP64
// argmax nor tie with it, and the selection is the full sweep's.  Indices
// reported are the body-local input indices (the copy stores them).
//
// Bodies of more than kSuper clusters also carry superclusters (kSuper
// consecutive clusters, bounded the same way from their vertices): the query
// bounds the superclusters first and only opens those whose bound reaches
// the threshold, so a 100,000-vertex body reads ~100 supercluster bounds per
// query instead of ~3,000 cluster bounds.  A supercluster's bound covers
// every vertex of its clusters, so skipping it is exact by the same argument.
constexpr int kCluster = 32;
constexpr int kSuper = 32;
constexpr int kSuperMinClusters = 4 * kSuper;  // superclusters above 4,096 vertices

// Bounds of one cluster: centre c and radius r (c.w) of a sphere, and half
// extents h of the box around c, all rounded outwards.
struct ClusterBound {
  float4 c;
  float4 h;
};

struct ClusterView {
  const float* x;  // cluster-ordered vertices of every body
  const float* y;
  const float* z;
  const int32_t* orig;          // body-local input index of each slot
  const ClusterBound* bounds;   // per cluster
  const ClusterBound* sbounds;  // per supercluster
};

struct CBody : Body<float, 1> {
  ClusterView cv;
  int64_t slot;  // first slot of the body (a multiple of kCluster); < 0: no culling
};

// A clustered body of a scene that has superclusters (two-level queries).
struct CBody2 : CBody {};

// The body's first supercluster (< 0: none) is kept in the spare word of its
// first cluster's bound, so a body carries no extra field through GJK.
OGJK_DEV int first_super(const ClusterBound* body_bounds) {
  return __builtin_bit_cast(int, body_bounds[0].h.w);
}

// c.d + min(r |d|, h.|d|) >= max over the cluster of x.d
OGJK_DEV float cluster_ub(const ClusterBound& b, float dx, float dy, float dz, float dn) {
  const float cd = fmaf(b.c.x, dx, fmaf(b.c.y, dy, b.c.z * dz));
  const float box = fmaf(b.h.x, fabsf(dx), fmaf(b.h.y, fabsf(dy), b.h.z * fabsf(dz)));
  return cd + fminf(b.c.w * dn, box);
}

// Calls f(k) for every body-local slot k of the clusters c0 <= c < c0 + ncl
// whose bound reaches L (cb: the body's cluster bounds), each slot on exactly
// one lane, in the same order on every call.
template <int LPP, class F>
OGJK_DEV void visit_range(const CBody& A, const ClusterBound* cb, int c0, int ncl, float dx,
                          float dy, float dz, float dn, float L, int lane, F&& f) {
  for (int base = 0; base < ncl; base += LPP) {
    const int c = base + lane;
    const bool live = c < ncl && !(cluster_ub(cb[c0 + c], dx, dy, dz, dn) < L);
    uint64_t m = group_ballot<LPP>(live);
    while (m != 0) {
      if constexpr (LPP >= kCluster) {
        // LPP/kCluster clusters per round, one per kCluster-lane slice
        constexpr int PER = LPP / kCluster;
        int cid = -1;
#pragma unroll
        for (int j = 0; j < PER; j++) {
          if (m != 0) {
            if (j == lane / kCluster) cid = (int)__builtin_ctzll(m);
            m &= m - 1;
          }
        }
        if (cid >= 0) {
          const int k = (c0 + base + cid) * kCluster + (lane & (kCluster - 1));
          if (k < A.n) f(k);
        }
      } else {
        const int cid = (int)__builtin_ctzll(m);
        m &= m - 1;
#pragma unroll
        for (int t = lane; t < kCluster; t += LPP) {
          const int k = (c0 + base + cid) * kCluster + t;
          if (k < A.n) f(k);
        }
      }
    }
  }
}

// All surviving clusters of the body: through its superclusters when it has
// them (sb non-null), in supercluster then cluster order; without, the body
// is a single unit of nc clusters.  One loop for both keeps one copy of the
// cluster visit per call site.
template <int LPP, bool TWO, class F>
OGJK_DEV void visit_clusters(const CBody& A, const ClusterBound* cb, int nc,
                             const ClusterBound* sb, float dx, float dy, float dz, float dn,
                             float L, int lane, F&& f) {
  if constexpr (!TWO) {
    visit_range<LPP>(A, cb, 0, nc, dx, dy, dz, dn, L, lane, f);
    return;
  }
  const int nunits = sb != nullptr ? (nc + kSuper - 1) / kSuper : 1;
  for (int base = 0; base < nunits; base += LPP) {
    const int u = base + lane;
    const bool live = u < nunits && (sb == nullptr || !(cluster_ub(sb[u], dx, dy, dz, dn) < L));
    uint64_t m = group_ballot<LPP>(live);
    while (m != 0) {
      const int u0 = base + (int)__builtin_ctzll(m);
      m &= m - 1;
      const int c0 = sb != nullptr ? u0 * kSuper : 0;
      const int ncl = sb != nullptr ? min(kSuper, nc - c0) : nc;
      visit_range<LPP>(A, cb, c0, ncl, dx, dy, dz, dn, L, lane, f);
    }
  }
}

// Index (within [0, n)) of the entry of b with the largest bound.
template <int LPP>
OGJK_DEV int best_bound(const ClusterBound* b, int n, float dx, float dy, float dz, float dn,
                        int lane) {
  float bub = -INFINITY;
  int bi = 0;
  for (int c = lane; c < n; c += LPP) {
    const float ub = cluster_ub(b[c], dx, dy, dz, dn);
    if (ub > bub) {
      bub = ub;
      bi = c;
    }
  }
  const float gub = group_max_f<LPP>(bub);
  return shfl_i<LPP>(bi, (int)__builtin_ctzll(group_ballot<LPP>(bub == gub) | (1ull << 63)));
}

// The clustered query through superclusters (TWO) or, without TWO, as one
// level (used by groups of fewer than 64 lanes; see support(CBody) below).
template <int LPP, bool TWO>
OGJK_DEV Sup support_clustered(const CBody& A, const Query& q, int lane) {
  if (A.slot < 0) return support<LPP>(static_cast<const Body<float, 1>&>(A), q, lane);
  Sweep32 sw = sweep32_begin(q.dir);
  const float dx = sw.dx, dy = sw.dy, dz = sw.dz;
  const float dn = sqrtf(fmaf(dx, dx, fmaf(dy, dy, dz * dz))) * (1.0f + 0x1.0p-20f);
  const int nc = (A.n + kCluster - 1) / kCluster;
  const ClusterBound* cb = A.cv.bounds + A.slot / kCluster;
  const float* sx = A.cv.x + A.slot;
  const float* sy = A.cv.y + A.slot;
  const float* sz = A.cv.z + A.slot;

  const ClusterBound* sb = nullptr;
  if constexpr (TWO) {
    const int sup = first_super(cb);
    if (sup >= 0) sb = A.cv.sbounds + sup;
  }

  // 1-2: the cluster with the largest bound (inside the supercluster with the
  // largest bound, when there are superclusters) gives a lower bound of the max
  int c0 = 0, ncl = nc;
  if (TWO && sb != nullptr) {
    c0 = best_bound<LPP>(sb, (nc + kSuper - 1) / kSuper, dx, dy, dz, dn, lane) * kSuper;
    ncl = min(kSuper, nc - c0);
  }
  const int bc = c0 + best_bound<LPP>(cb + c0, ncl, dx, dy, dz, dn, lane);
  float m0 = -INFINITY;
#pragma unroll
  for (int t = lane; t < kCluster; t += LPP) {
    const int k = bc * kCluster + t;
    if (k < A.n) m0 = fmaxf(m0, fmaf(sx[k], dx, fmaf(sy[k], dy, sz[k] * dz)));
  }
  const float L = group_max_f<LPP>(m0) - 0x1.0p-15f * A.r1;

  // 3: sweep the surviving clusters
  visit_clusters<LPP, TWO>(A, cb, nc, sb, dx, dy, dz, dn, L, lane, [&](int k) {
    const float px = sx[k], py = sy[k], pz = sz[k];
    const float d = fmaf(px, dx, fmaf(py, dy, pz * dz));
    sw.second = fmaxf(sw.second, fminf(sw.best, d));
    if (d > sw.best) {
      sw.best = d;
      sw.bi = k;
      sw.bx = px;
      sw.by = py;
      sw.bz = pz;
    }
  });
  const float M = group_max_f<LPP>(sw.best);
  const float T = M - 0x1.0p-19f * A.r1;
  const bool multi = group_any<LPP>(sw.second >= T);

  // FP64 re-rank of the window; ties go to the lowest input index
  const int32_t* orig = A.cv.orig + A.slot;
  Cand c{-INFINITY, 0x7fffffff, D3{0.0, 0.0, 0.0}};
  if (!multi) {
    if (sw.bi >= 0 && sw.best >= T) {
      c.p = D3{(double)sw.bx, (double)sw.by, (double)sw.bz};
      c.v = dot(c.p, q.dir);
      c.i = orig[sw.bi];
    }
  } else {
    visit_clusters<LPP, TWO>(A, cb, nc, sb, dx, dy, dz, dn, L, lane, [&](int k) {
      const float px = sx[k], py = sy[k], pz = sz[k];
      const float d = fmaf(px, dx, fmaf(py, dy, pz * dz));
      if (d >= T) {
        const D3 p{(double)px, (double)py, (double)pz};
        const double v = dot(p, q.dir);
        const int oi = orig[k];
        if (v > c.v || (v == c.v && oi < c.i)) {
          c.v = v;
          c.i = oi;
          c.p = p;
        }
      }
    });
  }
  if (!(c.v == c.v)) c.v = -INFINITY;
  return finish1<LPP, false>(c, q);
}

// Whole-wave form.  A query is a chain of dependent memory round trips, and a
// wave has little else to do meanwhile, so what can be in flight together is:
// bounds stay in registers from the pass that finds the best cluster, the two
// best clusters are swept at once (one per half of the wave: the threshold is
// then the larger maximum of two, and there are fewer others to visit), and the
// clusters that reach the threshold are swept kBatch pairs at a time.

constexpr int kBatch = 4;

// Calls f(k, x, y, z, in range) for the slots k of the clusters that the lanes
// with `live` name, kCluster lanes to a cluster and kBatch pairs of clusters in
// flight.  One permute packs the names into the lowest lanes; taking them from
// the ballot bit by bit made the scalar unit the slowest part of a query.
template <class F>
OGJK_DEV void visit_live(bool live, int c, int n, const float* sx, const float* sy,
                         const float* sz, int lane, F&& f) {
  const uint64_t m = __ballot(live);
  const int cnt = (int)__popcll(m);
  if (cnt == 0) return;
  const int below = lanes_below<64>(m, lane);
  const int list = __builtin_amdgcn_ds_permute((live ? below : cnt + lane - below) << 2, c);
  const int half = lane >> 5, in = lane & (kCluster - 1);
  for (int at = 0; at < cnt; at += 2 * kBatch) {
    int k[kBatch];
    float px[kBatch], py[kBatch], pz[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; u++) {
      const int e = at + 2 * u + half;
      const int slot = __builtin_amdgcn_ds_bpermute(e << 2, list) * kCluster + in;
      k[u] = e < cnt && slot < n ? slot : -1;
    }
#pragma unroll
    for (int u = 0; u < kBatch; u++) {
      if (at + 2 * u < cnt) {
        const int slot = max(k[u], 0);
        px[u] = sx[slot];
        py[u] = sy[slot];
        pz[u] = sz[slot];
      }
    }
#pragma unroll
    for (int u = 0; u < kBatch; u++)
      if (at + 2 * u < cnt) f(k[u], px[u], py[u], pz[u], k[u] >= 0);
  }
}

// The entry with the largest of the lanes' values (the lowest lane's on ties),
// with its value.
OGJK_DEV int wave_best(float v, int i, float& top) {
  top = group_max_f<64>(v);
  return lane_value(i, (int)__builtin_ctzll(__ballot(v == top) | (1ull << 63)));
}

// The two entries with the largest bounds of b[0, n): ub[j] keeps the bound of
// entry lane + 64 j, later entries are bounded again.  second < 0: none.
OGJK_DEV void two_best(const ClusterBound* b, int n, float dx, float dy, float dz, float dn,
                       int lane, float (&ub)[2], int& first, int& second) {
  float v = -INFINITY;
  int i = 0;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int c = lane + 64 * j;
    ub[j] = c < n ? cluster_ub(b[c], dx, dy, dz, dn) : -INFINITY;
    if (ub[j] > v) {
      v = ub[j];
      i = c;
    }
  }
  for (int c = lane + 128; c < n; c += 64) {
    const float u = cluster_ub(b[c], dx, dy, dz, dn);
    if (u > v) {
      v = u;
      i = c;
    }
  }
  float top;
  first = wave_best(v, i, top);
  v = -INFINITY;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int c = lane + 64 * j;
    if (c != first && ub[j] > v) {
      v = ub[j];
      i = c;
    }
  }
  for (int c = lane + 128; c < n; c += 64) {
    const float u = c != first ? cluster_ub(b[c], dx, dy, dz, dn) : -INFINITY;
    if (u > v) {
      v = u;
      i = c;
    }
  }
  second = wave_best(v, i, top);
  if (!(top > -INFINITY)) second = -1;
}

template <bool TWO>
OGJK_DEV Sup support_clustered64(const CBody& A, const Query& q, int lane) {
  if (A.slot < 0) return support<64>(static_cast<const Body<float, 1>&>(A), q, lane);
  Sweep32 sw = sweep32_begin(q.dir, q.unit);
  const float dx = sw.dx, dy = sw.dy, dz = sw.dz;
  const float dn = sqrtf(fmaf(dx, dx, fmaf(dy, dy, dz * dz))) * (1.0f + 0x1.0p-20f);
  const int nc = (A.n + kCluster - 1) / kCluster;
  const ClusterBound* cb = A.cv.bounds + A.slot / kCluster;
  const float* sx = A.cv.x + A.slot;
  const float* sy = A.cv.y + A.slot;
  const float* sz = A.cv.z + A.slot;
  const ClusterBound* sb = nullptr;
  if constexpr (TWO) {
    const int sup = first_super(cb);
    if (sup >= 0) sb = A.cv.sbounds + sup;
  }
  // the build gives superclusters to every body of more clusters than this
  if (sb == nullptr && nc > kSuperMinClusters)
    return support_clustered<64, false>(A, q, lane);

  // 1: the two clusters with the largest bounds (of all, or of the two
  // superclusters with the largest)
  float ub[2], sub[2];
  int bc, bc2;
  const int half = lane >> 5, in = lane & (kCluster - 1);
  const int ns = (nc + kSuper - 1) / kSuper;
  if (!TWO || sb == nullptr) {
    two_best(cb, nc, dx, dy, dz, dn, lane, ub, bc, bc2);
  } else {
    int s1, s2;
    two_best(sb, ns, dx, dy, dz, dn, lane, sub, s1, s2);
    const int s = half ? s2 : s1;
    const int c = s * kSuper + in;
    const float v = s >= 0 && c < nc ? cluster_ub(cb[c], dx, dy, dz, dn) : -INFINITY;
    float top;
    bc = wave_best(v, c, top);
    bc2 = wave_best(c == bc ? -INFINITY : v, c, top);
    if (!(top > -INFINITY)) bc2 = -1;
  }

  auto sweep = [&](int k, float px, float py, float pz, bool ok) {
    const float d = fmaf(px, dx, fmaf(py, dy, pz * dz));
    sweep32_take(sw, px, py, pz, ok ? d : -INFINITY, k);
  };
  // 2: sweep both; the FP32 maximum of what was swept gives the threshold L
  {
    const int c = half ? bc2 : bc;
    const int k = c * kCluster + in;
    const bool ok = c >= 0 && k < A.n;
    const int at = ok ? k : 0;
    sweep(k, sx[at], sy[at], sz[at], ok);
  }
  const float L = group_max_f<64>(sw.best) - 0x1.0p-15f * A.r1;

  // 3: the other clusters whose bound reaches L (the visit order does not
  // change the selection: ties are broken by input index below)
  if (!TWO || sb == nullptr) {
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int c = lane + 64 * j;
      visit_live(c < nc && c != bc && c != bc2 && !(ub[j] < L), c, A.n, sx, sy, sz, lane, sweep);
    }
  } else {
    for (int base = 0; base < ns; base += 64) {
      const int s = base + lane;
      float u = base == 0 ? sub[0] : sub[1];
      if (base >= 128 && s < ns) u = cluster_ub(sb[s], dx, dy, dz, dn);
      uint64_t live = __ballot(s < ns && !(u < L));
      while (live != 0) {
        // the clusters of up to 2 kBatch superclusters, one per half and step
        int c[kBatch];
        ClusterBound b[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; j++) {
          c[j] = -1;
          if (live != 0) {
            int s0 = base + (int)__builtin_ctzll(live), s1 = -1;
            live &= live - 1;
            if (live != 0) {
              s1 = base + (int)__builtin_ctzll(live);
              live &= live - 1;
            }
            const int mine = half ? s1 : s0;
            c[j] = mine >= 0 && mine * kSuper + in < nc ? mine * kSuper + in : -1;
            b[j] = cb[max(c[j], 0)];
          }
        }
#pragma unroll
        for (int j = 0; j < kBatch; j++) {
          if (__ballot(c[j] >= 0) != 0)
            visit_live(c[j] >= 0 && c[j] != bc && c[j] != bc2 &&
                           !(cluster_ub(b[j], dx, dy, dz, dn) < L),
                       c[j], A.n, sx, sy, sz, lane, sweep);
        }
      }
    }
  }

  const int32_t* orig = A.cv.orig + A.slot;
  const int oi = sw.bi >= 0 ? orig[sw.bi] : 0x7fffffff;
  const float M = group_max_f<64>(sw.best);
  const float T = M - 0x1.0p-19f * A.r1;
  const bool multi = group_any<64>(sw.second >= T);
  const uint64_t holders = __ballot(sw.bi >= 0 && sw.best >= T);
  if (!multi && __popcll(holders) == 1) {  // as in support_f
    const int src = (int)__builtin_ctzll(holders);
    return widen(accept(SupF{lane_value(oi, src), lane_value(sw.bx, src),
                             lane_value(sw.by, src), lane_value(sw.bz, src)},
                        q, sw, T));
  }

  // FP64 re-rank of the window; ties go to the lowest input index
  Cand c{-INFINITY, 0x7fffffff, D3{0.0, 0.0, 0.0}};
  if (!multi) {
    if (sw.bi >= 0 && sw.best >= T) {
      c.p = D3{(double)sw.bx, (double)sw.by, (double)sw.bz};
      c.v = dot(c.p, q.dir);
      c.i = oi;
    }
  } else {
    // every cluster that may hold a vertex of the window reaches L
    visit_clusters<64, TWO>(A, cb, nc, sb, dx, dy, dz, dn, L, lane, [&](int k) {
      const float px = sx[k], py = sy[k], pz = sz[k];
      const float d = fmaf(px, dx, fmaf(py, dy, pz * dz));
      if (d >= T) {
        const D3 p{(double)px, (double)py, (double)pz};
        const double v = dot(p, q.dir);
        const int o = orig[k];
        if (v > c.v || (v == c.v && o < c.i)) {
          c.v = v;
          c.i = o;
          c.p = p;
        }
      }
    });
  }
  if (!(c.v == c.v)) c.v = -INFINITY;
  return finish1<64, false>(c, q);
}

// Whole-wave groups take the form above; narrower groups would keep 128 / LPP
// bounds per lane, which costs the small-hull kernels of the same scene more
// in spills than it saves.
template <int LPP>
OGJK_DEV Sup support(const CBody& A, const Query& q, int lane) {
  if constexpr (LPP >= 64) {
    return support_clustered64<false>(A, q, lane);
  } else {
    return support_clustered<LPP, false>(A, q, lane);
  }
}
template <int LPP>
OGJK_DEV Sup support(const CBody2& A, const Query& q, int lane) {
  if constexpr (LPP >= 64) {
    return support_clustered64<true>(A, q, lane);
  } else {
    return support_clustered<LPP, true>(A, q, lane);
  }
}

// ------------------------------------------------------------ posed bodies
//
// A body placed by a rigid pose: world vertex = R x + t, R from a unit
// quaternion (w, x, y, z) and t stored as 7 floats.  World coordinates are
// computed in FP64, each component as ((R0 x + R1 y) + R2 z) + t, the same
// arithmetic the checker uses to build its world vertices.  A support query
// sweeps the FP32 local vertices along R^T d and re-ranks its candidates on
// their FP64 world coordinates, so the selection is that of a sweep over the
// FP64 world vertices.

// A pose as the kernels hold it, in LDS: one lane per body makes the rotation
// matrix once per pair (it was made again for every query, some 45 FP64
// operations and the quaternion's loads).
struct Pose {
  double r[9];
  double t[3];
};
using LdsPose = const __attribute__((address_space(3))) Pose*;

OGJK_DEV void make_pose(const float* p, Pose* P) {
  const double w = p[0], x = p[1], y = p[2], z = p[3];
  P->r[0] = 1.0 - 2.0 * (y * y + z * z);
  P->r[1] = 2.0 * (x * y - w * z);
  P->r[2] = 2.0 * (x * z + w * y);
  P->r[3] = 2.0 * (x * y + w * z);
  P->r[4] = 1.0 - 2.0 * (x * x + z * z);
  P->r[5] = 2.0 * (y * z - w * x);
  P->r[6] = 2.0 * (x * z - w * y);
  P->r[7] = 2.0 * (y * z + w * x);
  P->r[8] = 1.0 - 2.0 * (x * x + y * y);
  P->t[0] = p[4];
  P->t[1] = p[5];
  P->t[2] = p[6];
}

struct PBody : Body<float, 1> {
  LdsPose P;
  OGJK_DEV D3 world(double x, double y, double z) const {
    return D3{((P->r[0] * x + P->r[1] * y) + P->r[2] * z) + P->t[0],
              ((P->r[3] * x + P->r[4] * y) + P->r[5] * z) + P->t[1],
              ((P->r[6] * x + P->r[7] * y) + P->r[8] * z) + P->t[2]};
  }
  OGJK_DEV D3 to_local(D3 d) const {  // R^T d
    return D3{(P->r[0] * d.x + P->r[3] * d.y) + P->r[6] * d.z,
              (P->r[1] * d.x + P->r[4] * d.y) + P->r[7] * d.z,
              (P->r[2] * d.x + P->r[5] * d.y) + P->r[8] * d.z};
  }
  OGJK_DEV D3 d(int i) const { return world(rx(i), ry(i), rz(i)); }
  OGJK_DEV double c(int i, int k) const {
    const D3 p = d(i);
    return k == 0 ? p.x : (k == 1 ? p.y : p.z);
  }
};

// Local FP32 sweep along R^T d.  Besides the FP32 error (16u r1 in scaled
// units), each candidate's FP64 world value may differ from the real
// (R x + t).d by at most u64 (45 r1 + 15 |t|_1) scaled, < 2^-46 (r1 + |t|_1):
// the window widens by twice that.
template <int LPP>
OGJK_DEV Sup support(PBody A, const Query& q, int lane) {
  // read from LDS for each query: kept across them, two poses are 24 registers
  asm volatile("" : "+v"(A.P));
  Sweep32 sw = sweep32_begin(A.to_local(q.dir));
  sweep32<LPP>(static_cast<const Body<float, 1>&>(A), lane, sw);
  const float m = group_max_f<LPP>(sw.best);
  const float t1 = (float)(fabs(A.P->t[0]) + fabs(A.P->t[1]) + fabs(A.P->t[2]));
  const float T = m - (0x1.0p-19f * A.r1 + 0x1.0p-45f * (A.r1 + t1));
  const bool multi = group_any<LPP>(sw.second >= T);
  const auto holders = lanes_where<LPP>(sw.bi >= 0 && sw.best >= T);
  if (!multi && count_lanes<LPP>(holders) == 1) {  // as in support_f
    const int src = first_lane<LPP>(holders);
    const Sup r{shfl_i<LPP>(sw.bi, src), A.world(shfl_f<LPP>(sw.bx, src), shfl_f<LPP>(sw.by, src),
                                                 shfl_f<LPP>(sw.bz, src))};
    const double v = dot(r.p, q.dir);
    if (q.has_inc && !(v > dot(q.inc_pt, q.dir))) return Sup{q.inc_idx, q.inc_pt};
    if (!q.has_inc && !(v > -1e10)) return Sup{-1, D3{0.0, 0.0, 0.0}};
    return r;
  }
  Cand c{-INFINITY, 0x7fffffff, D3{0.0, 0.0, 0.0}};
  if (!multi) {
    if (sw.bi >= 0 && sw.best >= T) {
      c.p = A.world(sw.bx, sw.by, sw.bz);
      c.v = dot(c.p, q.dir);
      c.i = sw.bi;
    }
  } else {
    for (int i = lane; i < A.n; i += LPP) {
      const float px = A.rx(i), py = A.ry(i), pz = A.rz(i);
      const float d = fmaf(px, sw.dx, fmaf(py, sw.dy, pz * sw.dz));
      if (d >= T) {
        const D3 p = A.world(px, py, pz);
        const double v = dot(p, q.dir);
        if (v > c.v) {  // ascending i within the lane keeps the lowest index
          c.v = v;
          c.i = i;
          c.p = p;
        }
      }
    }
  }
  if (!(c.v == c.v)) c.v = -INFINITY;
  return finish1<LPP>(c, q);
}

// Field-wise value selects (a select between two structs' addresses would
// put them in scratch memory).
template <class T, int STRIDE>
OGJK_DEV Body<T, STRIDE> pick(bool c, const Body<T, STRIDE>& a, const Body<T, STRIDE>& b) {
  return Body<T, STRIDE>{c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z, c ? a.n : b.n,
                         c ? a.r1 : b.r1};
}
OGJK_DEV CBody pick(bool c, const CBody& a, const CBody& b) {
  return CBody{pick(c, static_cast<const Body<float, 1>&>(a), static_cast<const Body<float, 1>&>(b)),
               a.cv, c ? a.slot : b.slot};
}
OGJK_DEV CBody2 pick(bool c, const CBody2& a, const CBody2& b) {
  return CBody2{pick(c, static_cast<const CBody&>(a), static_cast<const CBody&>(b))};
}
OGJK_DEV PBody pick(bool c, const PBody& a, const PBody& b) {
  return PBody{pick(c, static_cast<const Body<float, 1>&>(a), static_cast<const Body<float, 1>&>(b)),
               c ? a.P : b.P};
}
OGJK_DEV Query pick(bool c, const Query& a, const Query& b) {
  return Query{sel(c, a.dir, b.dir), c ? a.has_inc : b.has_inc, c ? a.inc_idx : b.inc_idx,
               sel(c, a.inc_pt, b.inc_pt), c ? a.unit : b.unit};
}

template <int LPP>
OGJK_DEV void both_halves(const Sup& r, Sup& lo, Sup& hi) {
  both_halves<LPP>(r.i, lo.i, hi.i);
  both_halves<LPP>(r.p.x, lo.p.x, hi.p.x);
  both_halves<LPP>(r.p.y, lo.p.y, hi.p.y);
  both_halves<LPP>(r.p.z, lo.p.z, hi.p.z);
}
template <int LPP>
OGJK_DEV void both_halves(const SupF& r, SupF& lo, SupF& hi) {
  both_halves<LPP>(r.i, lo.i, hi.i);
  both_halves<LPP>(r.x, lo.x, hi.x);
  both_halves<LPP>(r.y, lo.y, hi.y);
  both_halves<LPP>(r.z, lo.z, hi.z);
}

// Split the group between the two queries for bodies swept whole (small
// hulls: the reduction chains dominate); clustered bodies keep every lane on
// one query at a time (large hulls: the sweep dominates; splitting was 16%
// slower on the uneven 1M-pair workload, 8% faster on 64-vertex pairs).
template <class BT>
constexpr bool kSplitQueries = !std::is_base_of_v<CBody, BT>;
template <int LPP, class BT>
OGJK_DEV void support_pair(const BT& A, const Query& qa, const BT& B, const Query& qb, int lane,
                           Sup& ra, Sup& rb) {
  if constexpr (LPP >= 8 && kSplitQueries<BT>) {
    // the lower half of the group answers A's query, the upper half B's, at
    // the same time; then each half takes the other's result
    const bool hi = lane >= LPP / 2;
    const BT& body = pick(hi, B, A);
    const Query& q = pick(hi, qb, qa);
    if constexpr (std::is_same_v<BT, PBody>) {
      both_halves<LPP>(support<LPP / 2>(body, q, lane & (LPP / 2 - 1)), ra, rb);
    } else {
      SupF fa, fb;
      both_halves<LPP>(support_f<LPP / 2>(body, q, lane & (LPP / 2 - 1)), fa, fb);
      ra = widen(fa);
      rb = widen(fb);
    }
    return;
  }
  // one query after the other through one copy of the sweep code (two sweeps
  // in one loop keep two sweep states live; two inlined copies double the code
  // the register allocator sees)
#pragma clang loop unroll(disable)
  for (int w = 0; w < 2; w++) {
    const bool second = w != 0;
    const Sup r = support<LPP>(pick(second, B, A), pick(second, qb, qa), lane);
    if (second) {
      rb = r;
    } else {
      ra = r;
    }
  }
}

// A clustered body of a pair that two waves work on together, a block of 128:
// the first wave answers every query of A, the second of B, and they exchange
// the results.  Everything else both do alike, each in its own LDS, so their
// control flow is one and the barriers meet.
struct DuoShared {
  SupF r[2];
};
template <class BT>
struct Duo : BT {
  DuoShared* ex;
};

template <int LPP, class BT>
OGJK_DEV void support_pair(const Duo<BT>& A, const Query& qa, const Duo<BT>& B, const Query& qb,
                           int lane, Sup& ra, Sup& rb) {
  static_assert(LPP == 64, "one wave per body");
  const bool second = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) != 0;
  const BT& a = A;
  const BT& b = B;
  const Sup r = support<64>(pick(second, b, a), pick(second, qb, qa), lane);
  if (lane == 0) A.ex->r[second] = SupF{r.i, (float)r.p.x, (float)r.p.y, (float)r.p.z};
  __syncthreads();
  ra = widen(A.ex->r[0]);
  rb = widen(A.ex->r[1]);
  __syncthreads();  // read by both before the next query overwrites it
}

// Plain FP64 path over double storage: the same selection rules computed
// directly in FP64 (the comparison baseline; no FP32 pass).
template <int LPP, int STRIDE>
OGJK_DEV void support_pair(const Body<double, STRIDE>& A, const Query& qa,
                           const Body<double, STRIDE>& B, const Query& qb, int lane, Sup& ra,
                           Sup& rb) {
  Cand ca{-INFINITY, 0x7fffffff, D3{0.0, 0.0, 0.0}}, cb = ca;
  const int nmax = A.n > B.n ? A.n : B.n;
  for (int i = lane; i < nmax; i += LPP) {
    if (i < A.n) {
      const D3 p = A.d(i);
      const double v = dot(p, qa.dir);
      if (v > ca.v) ca = Cand{v, i, p};
    }
    if (i < B.n) {
      const D3 p = B.d(i);
      const double v = dot(p, qb.dir);
      if (v > cb.v) cb = Cand{v, i, p};
    }
  }
  if (!(ca.v == ca.v)) ca.v = -INFINITY;
  if (!(cb.v == cb.v)) cb.v = -INFINITY;
  ra = finish1<LPP>(ca, qa);
  rb = finish1<LPP>(cb, qb);
}

// --------------------------------------------------------------- simplex

struct Simplex {
  int n;
  D3 p[4];
  int ia[4], ib[4];
};

// Runtime-indexed access to the simplex.  LLVM would turn a select between
// two loads of the simplex into a load from a selected address, which forces
// the whole simplex into scratch memory; reading every slot and passing the
// values through an empty asm statement keeps the selects on registers.
OGJK_DEV double keep_reg(double v) {
  asm volatile("" : "+v"(v));
  return v;
}
OGJK_DEV int keep_reg(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
OGJK_DEV D3 keep_reg(D3 v) { return D3{keep_reg(v.x), keep_reg(v.y), keep_reg(v.z)}; }

OGJK_DEV D3 sp(const Simplex& s, int k) {
  const D3 p0 = keep_reg(s.p[0]), p1 = keep_reg(s.p[1]), p2 = keep_reg(s.p[2]),
           p3 = keep_reg(s.p[3]);
  return sel(k == 0, p0, sel(k == 1, p1, sel(k == 2, p2, p3)));
}
OGJK_DEV int sa(const Simplex& s, int k) {
  const int a0 = keep_reg(s.ia[0]), a1 = keep_reg(s.ia[1]), a2 = keep_reg(s.ia[2]),
            a3 = keep_reg(s.ia[3]);
  return k == 0 ? a0 : (k == 1 ? a1 : (k == 2 ? a2 : a3));
}
OGJK_DEV int sb(const Simplex& s, int k) {
  const int b0 = keep_reg(s.ib[0]), b1 = keep_reg(s.ib[1]), b2 = keep_reg(s.ib[2]),
            b3 = keep_reg(s.ib[3]);
  return k == 0 ? b0 : (k == 1 ? b1 : (k == 2 ? b2 : b3));
}
template <int DST, int SRC>
OGJK_DEV void smove(Simplex& s) {
  s.p[DST] = s.p[SRC];
  s.ia[DST] = s.ia[SRC];
  s.ib[DST] = s.ib[SRC];
}

// ---------------------------------------------------- sub-distance (FP64)
//
// S1D, S2D and S3D (GJK/cpu/openGJK.c:257-613) as one straight piece of code.
// Written as the reference's tree, with a projection at each of some twenty
// leaves, a wave of eight pairs walked nearly all of it in every iteration.  All
// leaves are of four kinds: keep the newest vertex s1, project on the line to
// one older vertex, on the plane through two, or stop inside.  So every
// predicate is evaluated once, from the edges e_x = q_x - s1 and their cross
// products, the tree is walked over the resulting bits, and one projection is
// made at the end, with one division.
//
// The values are the reference's bit for bit:
//   hff2(s1, x, y) = s1.(e_x x (e_x x e_y)) < 0, and e_y x e_x is the exact
//   negative of e_x x e_y, so both orders of a pair share one cross product;
//   projectOnPlane's normal (s1 - x) x (s1 - y) is e_x x e_y, and
//   projectOnLine's s1 - x is -e_x: a sign on both factors of X * t;
//   the determinant of (e_1, e_0, e_2) is -(e_1 . (e_2 x e_0)).
// (A zero component of v may take the other sign; no output depends on it.)
//
// The simplex itself is in LDS: four places, and a map of its slots to places
// (2 bits each), so that the reference's copies between slots, which leave the
// old vertices in the slots above the count, are changes of the map.

struct SimplexVertex {
  double x, y, z;
  int a, b;
};
struct GjkShared {
  SimplexVertex v[4];
  int pad[4];  // neighbouring groups' vertices fall on other banks
};

OGJK_DEV D3 point(const SimplexVertex& v) { return D3{v.x, v.y, v.z}; }

// hff1: GJK/cpu/openGJK.c:219-230
OGJK_DEV bool hff1(D3 p, D3 q) {
  return (p.x * p.x - p.x * q.x) + (p.y * p.y - p.y * q.y) + (p.z * p.z - p.z * q.z) > 0;
}

OGJK_DEV int map_at(int map, int slot) { return (map >> (2 * slot)) & 3; }
OGJK_DEV int map_set(int map, int slot, int place) {
  return (map & ~(3 << (2 * slot))) | (place << (2 * slot));
}

// x for label 0, 1, 2 of q[]
OGJK_DEV D3 sel3(int x, D3 q0, D3 q1, D3 q2) { return sel(x == 0, q0, sel(x == 1, q1, q2)); }

// The tree of S3D below "origin outside" (openGJK.c:390-608) over the bits of
// its predicates, for one or no face plane containing the origin's side.  H:
// hff1 of the older vertices; F bit x: hff2(s1, x, x - 1 mod 3); G bit x: hff2(s1, x,
// x + 1 mod 3); k: the reference's k (i = k - 1, j = k + 1 mod 3).  Returns x | y
// << 2 | kind << 4 with kind 2: line to x, 3: plane through x and y (slots 1 and
// 0 of the triangle).
OGJK_DEV int s3d_leaf(int H, int F, int G, int k, bool one_plane) {
  const int i = k == 0 ? 2 : k - 1, j = k == 2 ? 0 : k + 1;
  const bool hk = (H >> k) & 1, hi = (H >> i) & 1;
  const bool Tki = (F >> k) & 1, Tjk = (F >> j) & 1, Tij = (F >> i) & 1;
  const bool Tkj = (G >> k) & 1, Tji = (G >> j) & 1, Tik = (G >> i) & 1;
  const int Lk = k | 32, Li = i | 32, Lj = j | 32;
  const int Pik = i | (k << 2) | 48, Pjk = j | (k << 2) | 48, Pij = i | (j << 2) | 48;
  const int dt = __popc((unsigned)H);
  const int one = dt == 1 ? (hk ? (!Tki ? Pik : (!Tkj ? Pjk : Lk))
                                : (hi ? (!Tik ? Pik : Li) : (!Tjk ? Pjk : Lj)))
                : dt == 2 ? (hi ? (!Tki ? (!Tik ? Pik : Lk) : (!Tkj ? Pjk : Lk))
                                : (!Tkj ? (!Tjk ? Pjk : Lj) : (!Tki ? Pik : Lk)))
                          : (Tki ? (Tkj ? Lk : (Tjk ? Lj : Pjk)) : (Tik ? Li : Pik));
  const int none = dt == 1 ? (!Tij ? Pij : (!Tik ? Pik : Li))
                           : (!Tjk ? (!Tkj ? Pjk : (!Tki ? Pik : Lk)) : (!Tji ? Pij : Lj));
  return one_plane ? one : none;
}

// subalgorithm (openGJK.c:641-656) after vertex s1 (place f) joined the n older
// ones: n, map and v are updated.
OGJK_DEV void subdistance(const GjkShared& sh, D3 s1, int f, int& n, int& map, D3& v) {
  const D3 q0 = point(sh.v[map_at(map, 0)]), q1 = point(sh.v[map_at(map, 1)]),
           q2 = point(sh.v[map_at(map, 2)]);
  const D3 e0 = sub(q0, s1), e1 = sub(q1, s1), e2 = sub(q2, s1);
  int H = hff1(s1, q0) ? 1 : 0;
  // kind 0: v and the simplex stay, 1: s1 alone, 2: line to x, 3: plane x, y,
  // 4: inside.  tri: the reference reduced a tetrahedron to the triangle (s1, a, b)
  // first, or it was one.
  int kind, x = 0, y = 0, a = 1, b = 0;
  bool tri = n == 2;
  D3 c10 = e0, c20 = e0, c21 = e0;
  if (n == 1) {
    kind = H ? 2 : 1;  // S1D
  } else {
    H |= hff1(s1, q1) ? 2 : 0;
    c10 = cross(e1, e0);
    const bool T10 = dot(s1, cross(e1, c10)) < 0, T01 = dot(s1, cross(e0, c10)) > 0;
    bool Ta = T10, Tb = T01;
    kind = 0;
    if (n == 3) {
      H |= hff1(s1, q2) ? 4 : 0;
      c20 = cross(e2, e0);
      c21 = cross(e2, e1);
      const bool T20 = dot(s1, cross(e2, c20)) < 0, T02 = dot(s1, cross(e0, c20)) > 0;
      const bool T21 = dot(s1, cross(e2, c21)) < 0, T12 = dot(s1, cross(e1, c21)) > 0;
      const bool sss = dot(e1, c20) >= 0;
      const bool p2 = (dot(s1, cross(q1, q0)) <= 0) != sss;
      const bool p3 = (dot(s1, cross(q0, q2)) <= 0) != sss;
      const bool p4 = (dot(s1, cross(q2, q1)) <= 0) != sss;
      const int planes = (int)p2 + (int)p3 + (int)p4;
      const int dt = __popc((unsigned)H);
      if (dt == 0) {
        kind = 1;
      } else if (planes == 3) {
        kind = 4;
      } else if (planes == 2) {
        tri = true;
        a = !p2 ? 1 : 2;
        b = !p4 ? 1 : 0;
        Ta = !p2 ? T10 : (!p3 ? T20 : T21);
        Tb = !p2 ? T01 : (!p3 ? T02 : T12);
      } else if (planes == 1 || dt != 3) {
        const int F = (T02 ? 1 : 0) | (T10 ? 2 : 0) | (T21 ? 4 : 0);
        const int G = (T01 ? 1 : 0) | (T12 ? 2 : 0) | (T20 ? 4 : 0);
        const bool h0 = H & 1, h1 = H & 2;
        const int k = planes == 1 ? (p2 ? 2 : (p3 ? 1 : 0))
                                  : (dt == 1 ? (h1 ? 2 : (h0 ? 1 : 0)) : (!h1 ? 2 : (!h0 ? 1 : 0)));
        const int leaf = s3d_leaf(H, F, G, k, planes == 1);
        x = leaf & 3;
        y = (leaf >> 2) & 3;
        kind = leaf >> 4;
      }
    }
    if (tri) {  // S2D over (s1, a, b)
      const bool ha = (H >> a) & 1, hb = (H >> b) & 1;
      x = a;
      y = b;
      kind = !(ha || hb) ? 1 : (ha && Ta ? 2 : (hb && Tb ? 2 : 3));
      if (kind == 2 && !(ha && Ta)) x = b;
    }
  }
  if (kind == 0) {  // outside all faces and towards every vertex: no branch there
    n = 4;
    return;
  }

  // the one projection: X the edge, or the plane's normal
  const int other = 3 - x - y;  // of a plane's pair: the vertex left out
  const D3 X = sel(kind == 3, sel3(other, c21, c20, c10), sel3(x, e0, e1, e2));
  const double t = dot(s1, X) / dot(X, X);
  const D3 Xt{X.x * t, X.y * t, X.z * t};
  v = kind == 3 ? Xt : (kind == 2 ? sub(s1, Xt) : (kind == 1 ? s1 : D3{0.0, 0.0, 0.0}));

  // the slots, as the reference leaves them
  const int px = map_at(map, x), py = map_at(map, y);
  if (n == 1) {
    if (kind == 1) map = map_set(map, 0, f);
  } else if (tri) {
    const int pa = map_at(map, a), pb = map_at(map, b);
    map = map_set(map_set(map_set(map, 2, f), 1, pa), 0, pb);
    if (kind == 1 || (kind == 2 && x == a)) map = map_set(map, 0, f);
    if (kind == 2 && x == b) map = map_set(map, 1, f);
  } else if (kind == 3) {
    map = map_set(map_set(map_set(map, 2, f), 1, px), 0, py);
  } else if (kind == 2) {
    map = map_set(map_set(map, 1, f), 0, px);
  } else if (kind == 1) {
    map = map_set(map, 0, f);
  }
  n = kind;  // 1, 2, 3 or 4 vertices
}

// ------------------------------------------------------- witnesses W*D

struct Wit {
  D3 w0, w1;
};

template <class BT>
OGJK_DEV void W0D(const BT& A, const BT& B, const Simplex& s, Wit& w) {
  w.w0 = A.d(s.ia[0]);
  w.w1 = B.d(s.ib[0]);
}

// Blend of original vertices: sum_k (coord_k * a_k), left to right.
template <class BT>
OGJK_DEV double blend_c(const BT& b, const int* idx, const double* a, int m, int c) {
  double acc = 0.0;
  for (int k = 0; k < m; k++) {
    const int i = idx[k];
    const double x = b.c(i, c);
    acc = (k == 0) ? x * a[k] : acc + x * a[k];
  }
  return acc;
}

// W1D: GJK/cpu/openGJK.c:668-700 (det == 0 falls through, as the reference)
template <class BT>
OGJK_DEV void W1D(const BT& A, const BT& B, const Simplex& s, Wit& w) {
  const D3 p = s.p[0], q = s.p[1];
  const D3 pq = sub(q, p), po = neg(p);
  const double det = dot(pq, pq);
  if (det == 0.0) W0D(A, B, s, w);
  const double a1 = dot(pq, po) / det;
  const double a[2] = {1.0 - a1, a1};
  const int ia[2] = {s.ia[0], s.ia[1]}, ib[2] = {s.ib[0], s.ib[1]};
  w.w0 = D3{blend_c(A, ia, a, 2, 0), blend_c(A, ia, a, 2, 1), blend_c(A, ia, a, 2, 2)};
  w.w1 = D3{blend_c(B, ib, a, 2, 0), blend_c(B, ib, a, 2, 1), blend_c(B, ib, a, 2, 2)};
}

// W2D: GJK/cpu/openGJK.c:702-795
template <class BT>
OGJK_DEV void W2D(const BT& A, const BT& B, Simplex& s, Wit& w) {
  const D3 p = s.p[0], q = s.p[1], r = s.p[2];
  const D3 pq = sub(q, p), pr = sub(r, p), po = neg(p);
  const double T00 = dot(pq, pq), T01 = dot(pq, pr), T11 = dot(pr, pr);
  const double det = T00 * T11 - T01 * T01;
  if (det == 0.0) W1D(A, B, s, w);
  const double b0 = dot(pq, po), b1 = dot(pr, po);
  const double I00 = T11 / det, I01 = -T01 / det, I11 = T00 / det;
  const double a1 = I00 * b0 + I01 * b1;
  const double a2 = I01 * b0 + I11 * b1;
  const double a0 = 1.0 - a1 - a2;
  if (a0 < kEps64) {
    s.n = 2;
    smove<0, 2>(s);
    W1D(A, B, s, w);
  } else if (a1 < kEps64) {
    s.n = 2;
    smove<1, 2>(s);
    W1D(A, B, s, w);
  } else if (a2 < kEps64) {
    s.n = 2;
    W1D(A, B, s, w);
  }
  const double a[3] = {a0, a1, a2};
  const int ia[3] = {s.ia[0], s.ia[1], s.ia[2]}, ib[3] = {s.ib[0], s.ib[1], s.ib[2]};
  w.w0 = D3{blend_c(A, ia, a, 3, 0), blend_c(A, ia, a, 3, 1), blend_c(A, ia, a, 3, 2)};
  w.w1 = D3{blend_c(B, ib, a, 3, 0), blend_c(B, ib, a, 3, 1), blend_c(B, ib, a, 3, 2)};
}

// W3D: GJK/cpu/openGJK.c:797-929
template <class BT>
OGJK_DEV void W3D(const BT& A, const BT& B, Simplex& s, Wit& w) {
  const D3 p = s.p[0], q = s.p[1], r = s.p[2], t = s.p[3];
  const D3 pq = sub(q, p), pr = sub(r, p), ps = sub(t, p), po = neg(p);
  const double T00 = dot(pq, pq), T01 = dot(pq, pr), T02 = dot(pq, ps);
  const double T11 = dot(pr, pr), T12 = dot(pr, ps), T22 = dot(ps, ps);
  const double det00 = T11 * T22 - T12 * T12;
  const double det01 = T01 * T22 - T02 * T12;
  const double det02 = T01 * T12 - T02 * T11;
  const double det = T00 * det00 - T01 * det01 + T02 * det02;
  if (det == 0.0) W2D(A, B, s, w);
  const double b0 = dot(pq, po), b1 = dot(pr, po), b2 = dot(ps, po);
  const double det11 = T00 * T22 - T02 * T02;
  const double det12 = T00 * T12 - T01 * T02;
  const double det22 = T00 * T11 - T01 * T01;
  const double I00 = det00 / det, I01 = -det01 / det, I02 = det02 / det;
  const double I11 = det11 / det, I12 = -det12 / det, I22 = det22 / det;
  const double a1 = I00 * b0 + I01 * b1 + I02 * b2;
  const double a2 = I01 * b0 + I11 * b1 + I12 * b2;
  const double a3 = I02 * b0 + I12 * b1 + I22 * b2;
  const double a0 = 1.0 - a1 - a2 - a3;
  if (a0 < kEps64) {
    s.n = 3;
    smove<0, 3>(s);
    W2D(A, B, s, w);
  } else if (a1 < kEps64) {
    s.n = 3;
    smove<1, 3>(s);
    W2D(A, B, s, w);
  } else if (a2 < kEps64) {
    s.n = 3;
    smove<2, 3>(s);
    W2D(A, B, s, w);
  } else if (a3 < kEps64) {
    s.n = 3;
    W2D(A, B, s, w);
  }
  const double a[4] = {a0, a1, a2, a3};
  const int ia[4] = {s.ia[0], s.ia[1], s.ia[2], s.ia[3]};
  const int ib[4] = {s.ib[0], s.ib[1], s.ib[2], s.ib[3]};
  w.w0 = D3{blend_c(A, ia, a, 4, 0), blend_c(A, ia, a, 4, 1), blend_c(A, ia, a, 4, 2)};
  w.w1 = D3{blend_c(B, ib, a, 4, 0), blend_c(B, ib, a, 4, 1), blend_c(B, ib, a, 4, 2)};
}

// compute_witnesses: GJK/cpu/openGJK.c:931-950
template <class BT>
OGJK_DEV void witnesses(const BT& A, const BT& B, Simplex& s, Wit& w) {
  if (s.n == 4)
    W3D(A, B, s, w);
  else if (s.n == 3)
    W2D(A, B, s, w);
  else if (s.n == 2)
    W1D(A, B, s, w);
  else if (s.n == 1)
    W0D(A, B, s, w);
}

// ------------------------------------------------------------- GJK driver

// compute_minimum_distance: GJK/cpu/openGJK.c:952-1056.  Returns ||v||.
template <int LPP, class BT>
OGJK_DEV double gjk(const BT& A, const BT& B, Simplex& s, Wit& w, GjkShared& sh, int lane) {
  const double eps_rel = kEps64 * 1e4;  // (gkFloat)DBL_EPSILON * 1e4f
  const double eps_tot = kEps64 * 1e2;
  const double eps_rel2 = eps_rel * eps_rel;

  D3 pa = A.d(0), pb = B.d(0);
  int ia = 0, ib = 0;
  D3 v = sub(pa, pb);
  int n = 1, map = 0xE4;  // slot i in place i
  if (lane == 0) {
    sh.v[0] = SimplexVertex{v.x, v.y, v.z, 0, 0};
    for (int k = 1; k < 4; k++) sh.v[k] = SimplexVertex{0.0, 0.0, 0.0, 0, 0};
  }
  const double n0 = norm2(v);
  double norm2Wmax = 0.0;
  unsigned k = 0;
  do {
    k++;
    Sup sA, sB;
    support_pair<LPP>(A, Query{neg(v), true, ia, pa}, B, Query{v, true, ib, pb}, lane, sA, sB);
    ia = sA.i;
    pa = sA.p;
    ib = sB.i;
    pb = sB.p;
    const D3 wv = sub(pa, pb);
    const double gap = norm2(v) - dot(v, wv);
    if (gap <= eps_rel * norm2(v) || gap < eps_tot) break;
    if (norm2(v) < eps_rel2) break;

    // slot n gets the new vertex, in a place that no other slot names
    int used = 0;
#pragma unroll
    for (int t = 0; t < 4; t++) used |= t == n ? 0 : 1 << map_at(map, t);
    const int f = __builtin_ctz(~(unsigned)used);
    wave_sync();
    if (lane == 0) sh.v[f] = SimplexVertex{wv.x, wv.y, wv.z, ia, ib};
    map = map_set(map, n, f);
    wave_sync();
    subdistance(sh, wv, f, n, map, v);

    // the largest vertex of any simplex so far: the newest vertex always stays,
    // the older ones were counted when they were new, the first one in the
    // first turn if it stayed
    const double tn = norm2(wv);
    if (k == 1u && n == 2 && n0 > norm2Wmax) norm2Wmax = n0;
    if (tn > norm2Wmax) norm2Wmax = tn;
    if (norm2(v) <= eps_tot * eps_tot * norm2Wmax) break;
  } while (n != 4 && k != 25u);

  wave_sync();
  s.n = n;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    const SimplexVertex& q = sh.v[map_at(map, t)];
    s.p[t] = point(q);
    s.ia[t] = q.a;
    s.ib[t] = q.b;
  }
  witnesses(A, B, s, w);
  return sqrt(norm2(v));
}

}  // namespace ogjk
