// opengjk-amd device EPA for one pair on a group of LPP lanes (LPP <= 64).
//
// Layout: the polytope's vertex pool (<= 68 FP64 points and their body
// indices), the edge tables and the input witnesses live in LDS.  The 128 face
// slots are spread over the group's lanes, slot = q * LPP + lane.  A polytope
// seldom has more than 30 faces, so each lane holds the face of its first slot
// (q = 0) in registers and those of the others in LDS: with all of them in
// registers the 32-lane kernel wanted 190 of the 168 that three waves per SIMD
// leave it.  Nothing else of the pair stays in registers through the expansion
// loop: the starting tetrahedron is slots 0-3 of the vertex pool and is read
// back from there when the loop ends.
//
// The reference EPA (GJK/cpu/EPA.c:362-864) is sequential; its discrete
// choices are reproduced exactly with ballots:
//   * closest face: min distance, lowest slot on ties (EPA.c:608-617);
//   * horizon: edges of the faces removed this iteration, in slot order and
//     (v0v1, v1v2, v2v0) order; an edge that occurs more than once is dropped
//     (the pairwise cancellation of EPA.c:746-759 drops every occurrence), found
//     by two bit tables over the vertex pairs: met, and met again;
//   * new faces take the lowest free slots in horizon order (EPA.c:762-775);
//   * a face's normal is computed when it is created and a degenerate face is
//     retired at the start of the next iteration, which is when the reference
//     recomputes it (EPA.c:600-604) -- until then it still occupies its slot.
#pragma once

#include "ogjk_core.hpp"

namespace ogjk {

constexpr int kEpaMaxFaces = 128;
constexpr int kEpaMaxIter = 64;
// the tetrahedron and one vertex per iteration (below the reference's cap of
// 132, EPA.c:44, which therefore never ends the loop)
constexpr int kEpaMaxVerts = 4 + kEpaMaxIter;
constexpr int kEdgeWords = (kEpaMaxVerts * (kEpaMaxVerts - 1) / 2 + 31) / 32;

template <int LPP>
struct EpaShared {
  double vx[kEpaMaxVerts], vy[kEpaMaxVerts], vz[kEpaMaxVerts];
  double w_in[6];  // the witnesses EPA started from
  // faces of the slots past the first LPP
  static constexpr int kFar = kEpaMaxFaces - LPP;
  double nx[kFar], ny[kFar], nz[kFar], dist[kFar];
  int verts[kFar];
  int via[kEpaMaxVerts], vib[kEpaMaxVerts];
  // a bit per edge of the faces removed this iteration: those met, and those
  // met more than once.  All zero between iterations.
  unsigned met[kEdgeWords], again[kEdgeWords];
  unsigned short surv[kEpaMaxFaces];  // surviving horizon edges, in order
};

// Per block: 1 / (5 + i), the weights of the centroid's running mean.
struct EpaTable {
  double inv[kEpaMaxIter];
};

// Clears the edge tables: once before a group's first pair (epa() leaves them
// clear).
template <int LPP>
OGJK_DEV void epa_shared_begin(EpaShared<LPP>& sh, int lane) {
  for (int i = lane; i < kEdgeWords; i += LPP) sh.met[i] = sh.again[i] = 0u;
  wave_sync();
}
// By every thread of the block.
OGJK_DEV void epa_table_begin(EpaTable& tb) {
  if (threadIdx.x < kEpaMaxIter) tb.inv[threadIdx.x] = 1.0 / (double)(5 + (int)threadIdx.x);
  __syncthreads();
}

// Place of the edge (a, b) in the edge tables.
OGJK_DEV void edge_place(int a, int b, int& word, unsigned& bit) {
  const int lo = min(a, b), hi = max(a, b);
  const unsigned at = ((unsigned)__mul24(hi, hi - 1) >> 1) + (unsigned)lo;
  word = (int)(at >> 5);
  bit = 1u << (at & 31u);
}

// Places of a face's edges (v0v1, v1v2, v2v0), from its packed vertices.
OGJK_DEV void face_edges(int packed, int (&w)[3], unsigned (&b)[3]) {
  const int x0 = packed & 0xff, x1 = (packed >> 8) & 0xff, x2 = (packed >> 16) & 0xff;
  edge_place(x0, x1, w[0], b[0]);
  edge_place(x1, x2, w[1], b[1]);
  edge_place(x2, x0, w[2], b[2]);
}

OGJK_DEV unsigned lds_or(unsigned* p, unsigned bits) {
  return __hip_atomic_fetch_or(p, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

template <int LPP>
OGJK_DEV void mark_edges(EpaShared<LPP>& sh, const int (&w)[3], const unsigned (&b)[3]) {
  unsigned old[3];
#pragma unroll
  for (int k = 0; k < 3; k++) old[k] = lds_or(&sh.met[w[k]], b[k]);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const unsigned twice = old[k] & b[k];
    if (twice) lds_or(&sh.again[w[k]], twice);
  }
}

// Appends the edges of the lanes' removed faces (`mine`) that were met once to
// the surviving ones, of which there are n; returns how many.
template <int LPP>
OGJK_DEV int keep_edges(EpaShared<LPP>& sh, bool mine, int packed, const int (&w)[3],
                        const unsigned (&b)[3], int n, int lane) {
  bool k0 = false, k1 = false, k2 = false;
  if (mine) {
    k0 = !(sh.again[w[0]] & b[0]);
    k1 = !(sh.again[w[1]] & b[1]);
    k2 = !(sh.again[w[2]] & b[2]);
  }
  const int x0 = packed & 0xff, x1 = (packed >> 8) & 0xff, x2 = (packed >> 16) & 0xff;
  const auto m0 = lanes_where<LPP>(k0), m1 = lanes_where<LPP>(k1), m2 = lanes_where<LPP>(k2);
  int at = n + lanes_below<LPP>(m0, lane) + lanes_below<LPP>(m1, lane) + lanes_below<LPP>(m2, lane);
  // at most kEpaMaxFaces slots can take a new face
  if (k0 && at < kEpaMaxFaces) sh.surv[at] = (unsigned short)(x0 | (x1 << 8));
  at += k0;
  if (k1 && at < kEpaMaxFaces) sh.surv[at] = (unsigned short)(x1 | (x2 << 8));
  at += k1;
  if (k2 && at < kEpaMaxFaces) sh.surv[at] = (unsigned short)(x2 | (x0 << 8));
  return count_lanes<LPP>(m0) + count_lanes<LPP>(m1) + count_lanes<LPP>(m2);
}

template <int LPP>
OGJK_DEV void clear_edges(EpaShared<LPP>& sh, const int (&w)[3]) {
#pragma unroll
  for (int k = 0; k < 3; k++) sh.met[w[k]] = sh.again[w[k]] = 0u;
}

template <int LPP>
OGJK_DEV D3 lds_v(const EpaShared<LPP>& sh, int i) { return D3{sh.vx[i], sh.vy[i], sh.vz[i]}; }

// set_contact_normal: GJK/cpu/EPA.c:350-360
OGJK_DEV D3 contact_normal(D3 w1, D3 w2) {
  const D3 d = sub(w2, w1);
  const double n = sqrt(norm2(d));
  if (n > kEps64) return D3{d.x / n, d.y / n, d.z / n};
  return D3{1.0, 0.0, 0.0};
}

// compute_barycentric_origin: GJK/cpu/EPA.c:238-304
OGJK_DEV void bary_origin(D3 v0, D3 v1, D3 v2, double& a0, double& a1, double& a2) {
  const D3 e0 = sub(v1, v0), e1 = sub(v2, v0);
  const double d00 = dot(e0, e0), d01 = dot(e0, e1), d11 = dot(e1, e1);
  const double d20 = -dot(v0, e0), d21 = -dot(v0, e1);
  const double denom = d00 * d11 - d01 * d01;
  if (fabs(denom) < kEps64) {
    a0 = a1 = a2 = 1.0 / 3.0;
    return;
  }
  const double inv = 1.0 / denom;
  const double u = (d11 * d20 - d01 * d21) * inv;
  const double v = (d00 * d21 - d01 * d20) * inv;
  const double w = 1.0 - u - v;
  if (w < 0) {
    const D3 e12 = sub(v2, v1);
    double t = -dot(v1, e12) / dot(e12, e12);
    t = fmax(0.0, fmin(1.0, t));
    a0 = 0;
    a1 = 1.0 - t;
    a2 = t;
  } else if (u < 0) {
    double t = -dot(v0, e1) / dot(e1, e1);
    t = fmax(0.0, fmin(1.0, t));
    a0 = 1.0 - t;
    a1 = 0;
    a2 = t;
  } else if (v < 0) {
    double t = -dot(v0, e0) / dot(e0, e0);
    t = fmax(0.0, fmin(1.0, t));
    a0 = 1.0 - t;
    a1 = t;
    a2 = 0;
  } else {
    a0 = w;
    a1 = u;
    a2 = v;
  }
}

// A lane's faces: the first slot's in registers, and which slots are in use.
struct Faces {
  double nx, ny, nz, dist;
  int verts;       // v0 | v1 << 8 | v2 << 16
  unsigned valid;  // bit q
  unsigned pend;   // bit q: degenerate, retire at the next iteration start
};

// A built face: unit normal, plane distance, packed vertex ids, and whether
// it is degenerate (retired at the next iteration start).
struct NewFace {
  D3 n;
  double d;
  int packed;
  bool ok;
};

// A new face (v0, v1, v2): winding fixed against the centroid
// (GJK/cpu/EPA.c:204-231, 791-819), then its normal and plane distance
// (compute_face_normal_distance, GJK/cpu/EPA.c:92-129).  The winding test's
// cross product is reused for the plane: with no contraction, cross(p2 - p0,
// p1 - p0) is exactly -cross(p1 - p0, p2 - p0) (products commute exactly,
// x - y = -(y - x)), so the swapped face's normal is the negated one, bit for
// bit.
template <int LPP>
OGJK_DEV NewFace build_face(const EpaShared<LPP>& sh, int v0, int v1, int v2, D3 centroid) {
  const D3 p0 = lds_v(sh, v0);
  D3 n = cross(sub(lds_v(sh, v1), p0), sub(lds_v(sh, v2), p0));
  const bool swap = dot(n, sub(centroid, p0)) > 0;
  NewFace f;
  f.packed = swap ? (v0 | (v2 << 8) | (v1 << 16)) : (v0 | (v1 << 8) | (v2 << 16));
  if (swap) n = neg(n);
  const double nsq = norm2(n);
  f.ok = nsq > kEps64 * kEps64;
  if (f.ok) {
    const double nn = sqrt(nsq);
    n = D3{n.x / nn, n.y / nn, n.z / nn};
    f.d = dot(n, p0);
    if (f.d < 0) {
      n = neg(n);
      f.d = -f.d;
    }
  } else {
    f.d = 1e10;
  }
  f.n = n;
  return f;
}

template <int LPP>
OGJK_DEV void put_face(EpaShared<LPP>& sh, Faces& F, int q, int lane, const NewFace& f) {
  if (q == 0) {
    F.nx = f.n.x;
    F.ny = f.n.y;
    F.nz = f.n.z;
    F.dist = f.d;
    F.verts = f.packed;
  } else {
    const int k = (q - 1) * LPP + lane;
    sh.nx[k] = f.n.x;
    sh.ny[k] = f.n.y;
    sh.nz[k] = f.n.z;
    sh.dist[k] = f.d;
    sh.verts[k] = f.packed;
  }
  F.valid |= 1u << q;
  if (!f.ok) F.pend |= 1u << q;
}

// Is a bit of any lane's mask set from q on?  The loops over the far slots end
// there: with 16 lanes to a pair there are seven, and a polytope of 40 faces uses
// two (20,000 pairs of 64 vertices in plain FP64 at 16 lanes 815 -> 690 us).  With
// 64 lanes there is one, which the caller has asked for.
template <int LPP>
OGJK_DEV bool far_slots(unsigned mask, int q) {
  if constexpr (LPP == 64) return true;
  else return __ballot((mask >> q) != 0u) != 0;
}

// Closest valid face with distance in [0, 1e10), lowest slot on ties: the lanes
// with the group's least distance, then the first slot that has it.  `many`:
// slots past the first LPP are in use.
template <int LPP>
OGJK_DEV int closest_face(const EpaShared<LPP>& sh, const Faces& F, bool many, int lane) {
  constexpr int FPL = kEpaMaxFaces / LPP;
  double m = INFINITY;
  int slot = lane;
  if ((F.valid & 1u) && F.dist >= 0.0 && F.dist < 1e10) m = F.dist;
  if (many) {
#pragma clang loop unroll(disable)
    for (int q = 1; q < FPL && far_slots<LPP>(F.valid, q); q++) {
      if ((F.valid >> q) & 1u) {
        const double fd = sh.dist[(q - 1) * LPP + lane];
        if (fd >= 0.0 && fd < 1e10 && fd < m) {
          m = fd;
          slot = q * LPP + lane;
        }
      }
    }
  }
  const auto least = lanes_of_least<LPP>(m);
  const bool mine = ((least >> lane) & 1) != 0 && m < INFINITY;
  const auto hold = lanes_where<LPP>(mine);
  if (hold == 0) return -1;
  if (!many) return first_lane<LPP>(hold);
  return (int)group_min_u<LPP>(mine ? (uint32_t)slot : 0xffffffffu);
}

// Normal, distance and vertices of the face in `slot`, on every lane.
template <int LPP>
OGJK_DEV void fetch_face(const EpaShared<LPP>& sh, const Faces& F, int slot, D3& n, double& dist,
                         int& verts) {
  if (slot < LPP) {
    n = D3{shfl_d<LPP>(F.nx, slot), shfl_d<LPP>(F.ny, slot), shfl_d<LPP>(F.nz, slot)};
    dist = shfl_d<LPP>(F.dist, slot);
    verts = shfl_i<LPP>(F.verts, slot);
  } else {
    const int k = slot - LPP;
    n = D3{sh.nx[k], sh.ny[k], sh.nz[k]};
    dist = sh.dist[k];
    verts = sh.verts[k];
  }
}

// The two bodies as EPA holds them through its loop.  Where the group splits
// into halves (see kSplitQueries), a lane keeps its own half's body only (the lower
// half A, the upper half B), half the registers, and each half works on its
// body: the queries, and the blend of the witnesses, which the halves then
// exchange.  Otherwise every lane keeps both.
template <int LPP, class BT, bool SPLIT = LPP >= 16 && kSplitQueries<BT>>
struct PairView {
  BT A, B;
  OGJK_DEV PairView(const BT& a, const BT& b, int) : A(a), B(b) {}
  OGJK_DEV void query(D3 dir, bool unit, int lane, Sup& a, Sup& b) const {
    const D3 zero{0.0, 0.0, 0.0};
    support_pair<LPP>(A, Query{dir, false, 0, zero, unit}, B,
                      Query{neg(dir), false, 0, zero, unit}, lane, a, b);
    // The reference leaves its output unset when no vertex beats -1e10; such
    // coordinates are out of any physical range, fall back to vertex 0.
    if (a.i < 0) a = Sup{0, A.d(0)};
    if (b.i < 0) b = Sup{0, B.d(0)};
  }
  // indices into A and B, clamped to vertex 0
  OGJK_DEV void clamp(int& ia, int& ib) const {
    ia = (ia >= 0 && ia < A.n) ? ia : 0;
    ib = (ib >= 0 && ib < B.n) ? ib : 0;
  }
  OGJK_DEV void points(int ia, int ib, Wit& w) const {
    w.w0 = A.d(ia);
    w.w1 = B.d(ib);
  }
  OGJK_DEV void blend(const int* ia, const int* ib, const double* a, Wit& w) const {
    w.w0 = D3{blend_c(A, ia, a, 3, 0), blend_c(A, ia, a, 3, 1), blend_c(A, ia, a, 3, 2)};
    w.w1 = D3{blend_c(B, ib, a, 3, 0), blend_c(B, ib, a, 3, 1), blend_c(B, ib, a, 3, 2)};
  }
};

template <int LPP, class BT>
struct PairView<LPP, BT, true> {
  BT own;
  bool upper;
  OGJK_DEV PairView(const BT& a, const BT& b, int lane)
      : own(pick(lane >= LPP / 2, b, a)), upper(lane >= LPP / 2) {}
  OGJK_DEV void query(D3 dir, bool unit, int lane, Sup& a, Sup& b) const {
    const Query q{sel(upper, neg(dir), dir), false, 0, D3{0.0, 0.0, 0.0}, unit};
    if constexpr (std::is_same_v<BT, PBody>) {
      Sup r = support<LPP / 2>(own, q, lane & (LPP / 2 - 1));
      if (r.i < 0) r = Sup{0, own.d(0)};
      both_halves<LPP>(r, a, b);
    } else {
      SupF r = support_f<LPP / 2>(own, q, lane & (LPP / 2 - 1)), fa, fb;
      if (r.i < 0) r = SupF{0, own.rx(0), own.ry(0), own.rz(0)};
      both_halves<LPP>(r, fa, fb);
      a = widen(fa);
      b = widen(fb);
    }
  }
  OGJK_DEV void clamp(int& ia, int& ib) const {
    int na, nb;
    both_halves<LPP>(own.n, na, nb);
    ia = (ia >= 0 && ia < na) ? ia : 0;
    ib = (ib >= 0 && ib < nb) ? ib : 0;
  }
  OGJK_DEV void exchange(D3 p, Wit& w) const {
    both_halves<LPP>(p.x, w.w0.x, w.w1.x);
    both_halves<LPP>(p.y, w.w0.y, w.w1.y);
    both_halves<LPP>(p.z, w.w0.z, w.w1.z);
  }
  OGJK_DEV void points(int ia, int ib, Wit& w) const { exchange(own.d(upper ? ib : ia), w); }
  OGJK_DEV void blend(const int* ia, const int* ib, const double* a, Wit& w) const {
    const int i[3] = {upper ? ib[0] : ia[0], upper ? ib[1] : ia[1], upper ? ib[2] : ia[2]};
    exchange(D3{blend_c(own, i, a, 3, 0), blend_c(own, i, a, 3, 1), blend_c(own, i, a, 3, 2)}, w);
  }
};

// The plain FP64 path sweeps both bodies at once on the whole group.
template <int LPP, int STRIDE>
struct PairView<LPP, Body<double, STRIDE>, true> : PairView<LPP, Body<double, STRIDE>, false> {
  using PairView<LPP, Body<double, STRIDE>, false>::PairView;
};

// support_epa (GJK/cpu/EPA.c:307-344): farthest vertex of A along dir and of
// B along -dir; returns the Minkowski point A[ia] - B[ib].
template <int LPP, class PV>
OGJK_DEV D3 support_epa(const PV& V, D3 dir, bool unit, int& ia, int& ib, int lane) {
  Sup a, b;
  V.query(dir, unit, lane, a, b);
  ia = a.i;
  ib = b.i;
  return sub(a.p, b.p);
}

// Is p farther than eps from each of the first n pool vertices
// (GJK/cpu/EPA.c:453-463, 654-684)?
template <int LPP>
OGJK_DEV bool is_new_point(const EpaShared<LPP>& sh, int n, D3 p, int lane) {
  const double eps_sq = kEps64 * kEps64;
  bool near = false;
  for (int t = lane; t < n; t += LPP) {
    const double dx = p.x - sh.vx[t], dy = p.y - sh.vy[t], dz = p.z - sh.vz[t];
    if (dx * dx + dy * dy + dz * dz < eps_sq) near = true;
  }
  return !group_any<LPP>(near);
}

template <int LPP>
OGJK_DEV void put_vertex(EpaShared<LPP>& sh, int i, D3 p, int ia, int ib) {
  sh.vx[i] = p.x;
  sh.vy[i] = p.y;
  sh.vz[i] = p.z;
  sh.via[i] = ia;
  sh.vib[i] = ib;
}

// The simplex EPA returns: the tetrahedron it started from, pool slots 0-3.
template <int LPP>
OGJK_DEV void simplex_back(const EpaShared<LPP>& sh, Simplex& s, int n) {
  s.n = n;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    s.p[k] = lds_v(sh, k);
    s.ia[k] = sh.via[k];
    s.ib[k] = sh.vib[k];
  }
}

template <class PV>
OGJK_DEV void zero_depth(const PV& V, int ia, int ib, double& distance, Wit& w, D3& normal) {
  distance = 0.0;
  V.points(ia, ib, w);
  normal = contact_normal(w.w0, w.w1);
}

template <int LPP, class PV>
OGJK_DEV void face_result(const PV& V, const EpaShared<LPP>& sh, int verts, D3 n, double cdist,
                          double& distance, Wit& w, D3& normal) {
  const int v0 = verts & 0xff, v1 = (verts >> 8) & 0xff, v2 = (verts >> 16) & 0xff;
  double a[3];
  bary_origin(lds_v(sh, v0), lds_v(sh, v1), lds_v(sh, v2), a[0], a[1], a[2]);
  const int ia[3] = {sh.via[v0], sh.via[v1], sh.via[v2]};
  const int ib[3] = {sh.vib[v0], sh.vib[v1], sh.vib[v2]};
  V.blend(ia, ib, a, w);
  normal = n;
  distance = -cdist;
}

// computeCollisionInformation for one pair (GJK/cpu/EPA.c:362-864).  The edge
// tables of sh are clear before and after.
template <int LPP, class BT>
OGJK_DEV void epa(const BT& A, const BT& B, Simplex& s, double& distance, Wit& w, D3& normal,
                  EpaShared<LPP>& sh, const EpaTable& tb, int lane) {
  constexpr int FPL = kEpaMaxFaces / LPP;
  static_assert(FPL * LPP == kEpaMaxFaces, "LPP must divide 128");

  if (distance > kEps64) {
    normal = contact_normal(w.w0, w.w1);
    return;
  }
  const PairView<LPP, BT> V(A, B, lane);

  // the simplex and the witnesses wait in LDS: registers are what limits the
  // waves in flight
  if (lane < 4) put_vertex(sh, lane, sp(s, lane), sa(s, lane), sb(s, lane));
  if (lane == 0) {
    sh.w_in[0] = w.w0.x;
    sh.w_in[1] = w.w0.y;
    sh.w_in[2] = w.w0.z;
    sh.w_in[3] = w.w1.x;
    sh.w_in[4] = w.w1.y;
    sh.w_in[5] = w.w1.z;
  }
  wave_sync();

  // -------- grow a degenerate GJK simplex to a tetrahedron (EPA.c:376-583):
  // one support query per turn, along the point, across the edge, along the
  // triangle's normal, then against it
  int ns = s.n;
  bool against = false;
  while (ns >= 1 && ns < 4) {
    const D3 p0 = lds_v(sh, 0);
    D3 dir;
    if (ns == 1) {
      dir = p0;
    } else if (ns == 2) {
      const D3 edge = sub(lds_v(sh, 1), p0);
      D3 axis{1.0, 0.0, 0.0};
      const double en = sqrt(norm2(edge));
      if (en > kEps64 && fabs(edge.x) > (double)0.9f * en) axis = D3{0.0, 1.0, 0.0};
      dir = cross(edge, axis);
      if (norm2(dir) < kEps64) {
        axis = D3{0.0, 0.0, 1.0};
        dir = cross(edge, axis);
      }
    } else {
      dir = cross(sub(lds_v(sh, 1), p0), sub(lds_v(sh, 2), p0));
      if (against) dir = neg(dir);
    }
    int ia, ib;
    const D3 nv = support_epa<LPP>(V, dir, false, ia, ib, lane);
    if (is_new_point<LPP>(sh, ns, nv, lane)) {
      if (lane == 0) put_vertex(sh, ns, nv, ia, ib);
      wave_sync();
      ns++;
    } else if (ns == 3 && !against) {
      against = true;
    } else {
      zero_depth(V, ia, ib, distance, w, normal);
      simplex_back(sh, s, ns);
      return;
    }
  }
  if (ns != 4) {  // no simplex a GJK writes: caller-provided, sanitised
    int best = ns > 0 ? ns - 1 : 0;
    best = best > 3 ? 3 : best;
    int ba = sh.via[best], bb = sh.vib[best];
    V.clamp(ba, bb);
    zero_depth(V, ba, bb, distance, w, normal);
    simplex_back(sh, s, ns);
    return;
  }

  // -------- initial tetrahedron (init_epa_polytope, EPA.c:144-235)
  D3 centroid{0.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const D3 p = lds_v(sh, i);
    centroid.x += p.x * 0.25;
    centroid.y += p.y * 0.25;
    centroid.z += p.z * 0.25;
  }
  Faces F{0.0, 0.0, 0.0, 0.0, 0, 0u, 0u};
  if (lane < 4) {
    // faces (0,1,2) (0,3,1) (0,2,3) (1,3,2)
    const int a = lane == 3 ? 1 : 0;
    const int b = lane == 0 ? 1 : (lane == 1 ? 3 : (lane == 2 ? 2 : 3));
    const int c = lane == 0 ? 2 : (lane == 1 ? 1 : (lane == 2 ? 3 : 2));
    put_face(sh, F, 0, lane, build_face(sh, a, b, c, centroid));
  }

  const double tol = kEps64 * 1e2;
  int nverts = 4;
  int iteration = 0;
  int rverts = -1;  // the face whose result is returned, if any
  D3 rn{0.0, 0.0, 0.0};
  double rdist = 0.0;
  while (iteration < kEpaMaxIter) {
    iteration++;
    F.valid &= ~F.pend;  // the reference's per-iteration recompute retires them
    F.pend = 0;
    // slots past the first LPP are rarely in use: one ballot skips their share
    // of every step (wave-uniform)
    const bool many = __ballot(F.valid > 1u) != 0;

    const int cf = closest_face(sh, F, many, lane);
    if (cf < 0) break;
    D3 n;
    double cdist;
    int cverts;
    fetch_face(sh, F, cf, n, cdist, cverts);

    int ia, ib;
    const D3 nv = support_epa<LPP>(V, n, true, ia, ib, lane);
    const double improvement = dot(n, nv) - cdist;
    if (improvement < tol || !is_new_point<LPP>(sh, nverts, nv, lane)) {
      rverts = cverts;
      rn = n;
      rdist = cdist;
      break;
    }

    // add the vertex and update the running-mean centroid (EPA.c:686-699)
    const int nid = nverts;
    if (lane == 0) put_vertex(sh, nid, nv, ia, ib);
    const double inv_n = tb.inv[nverts - 4];
    nverts++;
    centroid.x += (nv.x - centroid.x) * inv_n;
    centroid.y += (nv.y - centroid.y) * inv_n;
    centroid.z += (nv.z - centroid.z) * inv_n;
    wave_sync();

    // faces visible from the new vertex (is_face_visible, EPA.c:132-140); each
    // marks its edges in the tables
    unsigned vis = 0;
    int w[3];  // the first slot's edge places; the others' are found again
    unsigned b[3];
    if ((F.valid & 1u) &&
        dot(D3{F.nx, F.ny, F.nz}, sub(nv, lds_v(sh, F.verts & 0xff))) > kEps64) {
      vis = 1u;
      face_edges(F.verts, w, b);
      mark_edges(sh, w, b);
    }
    if (many) {
#pragma clang loop unroll(disable)
      for (int q = 1; q < FPL && far_slots<LPP>(F.valid, q); q++) {
        if ((F.valid >> q) & 1u) {
          const int k = (q - 1) * LPP + lane;
          const int pv = sh.verts[k];
          if (dot(D3{sh.nx[k], sh.ny[k], sh.nz[k]}, sub(nv, lds_v(sh, pv & 0xff))) > kEps64) {
            vis |= 1u << q;
            int fw[3];
            unsigned fb[3];
            face_edges(pv, fw, fb);
            mark_edges(sh, fw, fb);
          }
        }
      }
    }
    F.valid &= ~vis;
    wave_sync();

    // horizon = edges met once, in slot order, (v0v1, v1v2, v2v0) within a face
    int nsurv = keep_edges(sh, (vis & 1u) != 0, F.verts, w, b, 0, lane);
    if (many) {
#pragma clang loop unroll(disable)
      for (int q = 1; q < FPL && far_slots<LPP>(vis, q); q++) {
        const bool mine = ((vis >> q) & 1u) != 0;
        const int pv = sh.verts[(q - 1) * LPP + lane];
        int fw[3];
        unsigned fb[3];
        face_edges(mine ? pv : 0x020100, fw, fb);
        nsurv += keep_edges(sh, mine, pv, fw, fb, nsurv, lane);
      }
    }
    wave_sync();
    // leave the tables clear
    if (vis & 1u) clear_edges(sh, w);
    if (many) {
#pragma clang loop unroll(disable)
      for (int q = 1; q < FPL && far_slots<LPP>(vis, q); q++) {
        if ((vis >> q) & 1u) {
          int fw[3];
          unsigned fb[3];
          face_edges(sh.verts[(q - 1) * LPP + lane], fw, fb);
          clear_edges(sh, fw);
        }
      }
    }

    // fan new faces into the lowest free slots (EPA.c:761-825)
    int taken = 0;
#pragma clang loop unroll(disable)
    for (int q = 0; q < FPL; q++) {
      if (__ballot(taken < nsurv) == 0) break;
      const bool fr = !((F.valid >> q) & 1u);
      const auto mf = lanes_where<LPP>(fr);
      const int rank = taken + lanes_below<LPP>(mf, lane);
      if (fr && rank < nsurv) {
        const int ed = sh.surv[rank];
        put_face(sh, F, q, lane, build_face(sh, ed & 0xff, (ed >> 8) & 0xff, nid, centroid));
      }
      taken += count_lanes<LPP>(mf);
    }
  }

  if (iteration >= kEpaMaxIter) {  // cap fallback (EPA.c:828-863)
    F.valid &= ~F.pend;
    F.pend = 0;
    const int cf = closest_face(sh, F, true, lane);
    if (cf >= 0) fetch_face(sh, F, cf, rn, rdist, rverts);
  }
  simplex_back(sh, s, 4);
  if (rverts >= 0) {
    face_result(V, sh, rverts, rn, rdist, distance, w, normal);
  } else {  // no face: the witnesses EPA started from
    w.w0 = D3{sh.w_in[0], sh.w_in[1], sh.w_in[2]};
    w.w1 = D3{sh.w_in[3], sh.w_in[4], sh.w_in[5]};
  }
}

}  // namespace ogjk
