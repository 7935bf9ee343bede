// Mesh ingestion on the device: the incremental convex hull of many point
// clouds at once, and the FP64 volume moments, centre of mass and inertia
// factors of each hull.
//
// The face list is the reference's (visualization/rendering/mesh_builder.cpp:
// 268-360): the same initial tetrahedron, points inserted in index order,
// faces with a 6x signed volume above 1e-7 (FP32) visible, visible faces
// removed in place, one new face per horizon edge appended in the order the
// visible faces and their edges are listed.  The reference runs that loop on
// one CPU thread per cloud; here 16 lanes, a wave or a block own a cloud (by its
// size and its face count) and each step is data-parallel over it: visibility
// over faces, the horizon test over the visible faces' edges, order-preserving
// compaction and appends by ballots and prefix counts.  Moments are summed in
// face order, as the reference sums them (:433-481), so they are
// bit-identical too.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "ogjk_internal.hpp"
#include "ogjk_math.hpp"
#include "opengjk/ogjk.h"

ogjk_status ogjk_fail(ogjk_status code, const char* fmt, ...);

namespace {

using ogjk::wave_sync;
using ogjk::xpair;

constexpr int kWave = 64;

// Results of d_nfaces that pass a cloud on to the next kernel of the call, to be
// started again or to go on from its saved state (no result that a caller sees:
// the last kernel leaves none of them).
constexpr int kToWave = -100, kSaved = -101;

// The arguments of a build: cloud m's points, its part of the output buffer and
// of the workspace (three words per face of its capacity in each).
struct HullArgs {
  const float* pts;
  const int64_t* off;
  const int32_t* cnt;
  int nm;
  const int64_t* face_off;
  int64_t total_faces;
  int32_t* faces;
  int32_t* nfaces;
  int32_t* scratch;
  __device__ bool range_ok(int64_t m) const {
    return face_off[m] >= 0 && face_off[m + 1] >= face_off[m] && face_off[m + 1] <= total_faces;
  }
  __device__ int64_t cap64(int64_t m) const { return face_off[m + 1] - face_off[m]; }
  __device__ int cap(int64_t m) const {
    return cap64(m) < 0x7fffffff ? (int)cap64(m) : 0x7fffffff;
  }
  __device__ const float* points(int64_t m) const { return pts + 3 * off[m]; }
  __device__ int32_t* out(int64_t m) const { return faces + 3 * face_off[m]; }
  __device__ int32_t* work(int64_t m) const { return scratch + 3 * face_off[m]; }
};

// A point of the working set and a face with its plane: the normal of
// (v0, v1, v2) as vol6 forms it, and the packed vertex ids.
struct alignas(16) Tri {
  float nx, ny, nz;
  uint32_t ids;
};

__device__ __forceinline__ Tri make_tri(float4 a, float4 b, float4 c, uint32_t ids) {
  const float bx = b.x - a.x, by = b.y - a.y, bz = b.z - a.z;
  const float cx = c.x - a.x, cy = c.y - a.y, cz = c.z - a.z;
  return Tri{by * cz - bz * cy, bz * cx - bx * cz, bx * cy - by * cx, ids};
}

// 6x signed volume of the face and q: the operations of the reference's
// signed volume in its order, with the face's normal kept from its creation
// (same operands, so the same bits).
__device__ __forceinline__ float vol6(const Tri& f, float4 a, float4 q) {
  const float dx = q.x - a.x, dy = q.y - a.y, dz = q.z - a.z;
  return f.nx * dx + f.ny * dy + f.nz * dz;
}

__device__ __forceinline__ float vol6(float4 a, float4 b, float4 c, float4 q) {
  return vol6(make_tri(a, b, c, 0u), a, q);
}

__device__ __forceinline__ uint64_t ballot(bool v) { return __ballot(v); }

__device__ __forceinline__ int rank_below(uint64_t mask, int lane) {
  return ogjk::lanes_below<kWave>(mask, lane);
}

template <int L, int M = 1>
__device__ __forceinline__ int group_min_i(int v) {
  if constexpr (M < L) {
    int a, b;
    xpair<M>(v, a, b);
    return group_min_i<L, 2 * M>(a < b ? a : b);
  } else {
    return v;
  }
}

// Of the lanes' (value, index) candidates (index < 0: none), the largest
// value's lowest index, or -1.  No value is NaN or -inf.
template <int L>
__device__ __forceinline__ int group_argmax(float v, int i) {
  const float m = ogjk::group_max_f<L>(i >= 0 ? v : -INFINITY);
  const int r = group_min_i<L>(i >= 0 && v == m ? i : 0x7fffffff);
  return r == 0x7fffffff ? -1 : r;
}

// The first four points of the hull of pt[0..n) (lane: of a group of L), in
// the reference's choice and orientation.  Returns false when there is no
// tetrahedron.  lo, hi, lo_i, hi_i: this lane's axis extremes over its points
// i = lane, lane + L, ... (first index on ties, -1 without a point).
template <int L, class Pts>
__device__ __forceinline__ bool first_tetrahedron(const Pts& pt, int n, int lane,
                                                  const float (&lo)[3], const int (&lo_i)[3],
                                                  const float (&hi)[3], const int (&hi_i)[3],
                                                  int (&id)[4]) {
  int c[6];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    c[2 * k] = group_argmax<L>(-lo[k], lo_i[k]);
    c[2 * k + 1] = group_argmax<L>(hi[k], hi_i[k]);
  }
  // most separated pair among the six, the first in (a, b) order on ties:
  // pair p = lane of 15, in chunks where the group is narrower
  int i0 = 0, i1 = 1;
  {
    float bv = 0.0f;
    int bp = -1;
    for (int p = lane; p < 15; p += L) {
      const int a = p < 5 ? 0 : p < 9 ? 1 : p < 12 ? 2 : p < 14 ? 3 : 4;
      const int b = p < 5 ? p + 1 : p < 9 ? p - 3 : p < 12 ? p - 6 : p < 14 ? p - 8 : 5;
      int ca = c[0], cb = c[1];
#pragma unroll
      for (int k = 1; k < 6; k++) {
        ca = a == k ? c[k] : ca;
        cb = b == k ? c[k] : cb;
      }
      const float4 A = pt(ca), B = pt(cb);
      const float dx = B.x - A.x, dy = B.y - A.y, dz = B.z - A.z;
      const float d = dx * dx + dy * dy + dz * dz;
      if (d > bv) {
        bv = d;
        bp = p;
      }
    }
    const int p = group_argmax<L>(bv, bp);
    if (p >= 0) {
      const int a = p < 5 ? 0 : p < 9 ? 1 : p < 12 ? 2 : p < 14 ? 3 : 4;
      const int b = p < 5 ? p + 1 : p < 9 ? p - 3 : p < 12 ? p - 6 : p < 14 ? p - 8 : 5;
      i0 = c[0];
      i1 = c[1];
#pragma unroll
      for (int k = 1; k < 6; k++) {
        i0 = a == k ? c[k] : i0;
        i1 = b == k ? c[k] : i1;
      }
    }
  }
  const float4 p0 = pt(i0), p1 = pt(i1);
  // farthest from the line i0-i1
  int i2;
  {
    const float e0 = p1.x - p0.x, e1 = p1.y - p0.y, e2 = p1.z - p0.z;
    float bv = 0.0f;
    int bi = -1;
    for (int i = lane; i < n; i += L) {
      if (i == i0 || i == i1) continue;
      const float4 p = pt(i);
      const float vx = p.x - p0.x, vy = p.y - p0.y, vz = p.z - p0.z;
      const float cx = vy * e2 - vz * e1, cy = vz * e0 - vx * e2, cz = vx * e1 - vy * e0;
      const float d = cx * cx + cy * cy + cz * cz;
      if (d > bv) {
        bv = d;
        bi = i;
      }
    }
    i2 = group_argmax<L>(bv, bi);
  }
  if (i2 < 0) return false;
  const float4 p2 = pt(i2);
  // farthest from the plane i0-i1-i2
  int i3;
  {
    const Tri t = make_tri(p0, p1, p2, 0u);
    float bv = 0.0f;
    int bi = -1;
    for (int i = lane; i < n; i += L) {
      if (i == i0 || i == i1 || i == i2) continue;
      float d = vol6(t, p0, pt(i));
      if (d < 0) d = -d;
      if (d > bv) {
        bv = d;
        bi = i;
      }
    }
    i3 = group_argmax<L>(bv, bi);
  }
  if (i3 < 0) return false;
  const bool swap = vol6(p0, p1, p2, pt(i3)) > 0;
  id[0] = i0;
  id[1] = swap ? i2 : i1;
  id[2] = swap ? i1 : i2;
  id[3] = i3;
  return true;
}

// Corner j of initial face f: (0,1,2) (0,2,3) (0,3,1) (1,3,2).
__device__ __forceinline__ int init_corner(const int (&id)[4], int f, int j) {
  const uint32_t map[4] = {0x210u, 0x320u, 0x130u, 0x231u};
  const uint32_t m = f == 0 ? map[0] : f == 1 ? map[1] : f == 2 ? map[2] : map[3];
  const int k = (m >> (4 * j)) & 3;
  return k == 0 ? id[0] : k == 1 ? id[1] : k == 2 ? id[2] : id[3];
}

// ------------------------------------------------- clouds of few points
//
// Clouds of up to 32 points, 16 lanes each, the whole working set in LDS.
// Bound by vector instructions (a step has ~20 faces and ~12 edges to look
// at), hence: as many lanes as a small hull fills (four clouds share a wave's
// instructions), the plane of each face kept from its creation (an insertion
// reads it and one corner instead of three gathered corners and a cross
// product), and the horizon test by one bit per directed edge of the visible
// faces (word = start, bit = end) instead of a search of their list.  100,000
// clouds of 8-32 points: 0.29 ms at 16 lanes, 0.33 at 32, 0.90 with one wave
// per cloud and no kept planes.
constexpr int kFewLanes = 16, kFewPoints = 32, kFewFaces = 96;

struct FewHull {
  float4 pt[kFewPoints];
  Tri face[kFewFaces];
  uint32_t vis[kFewFaces];
  uint32_t adj[kFewPoints];
};

__device__ __forceinline__ int hull_few(const float* __restrict__ P, int n, int cap, FewHull& s,
                                        int lane) {
  constexpr int L = kFewLanes;
  const auto pt = [&](int i) { return s.pt[i]; };
  float lo[3], hi[3];
  int lo_i[3], hi_i[3];
  bool bad = false;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    lo[k] = INFINITY;
    hi[k] = -INFINITY;
    lo_i[k] = hi_i[k] = -1;
  }
  wave_sync();
  for (int i = lane; i < n; i += L) {
    const float p[3] = {P[3 * i], P[3 * i + 1], P[3 * i + 2]};
    s.pt[i] = make_float4(p[0], p[1], p[2], 0.0f);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      bad |= !isfinite(p[k]);
      if (lo_i[k] < 0 || p[k] < lo[k]) { lo[k] = p[k]; lo_i[k] = i; }
      if (hi_i[k] < 0 || p[k] > hi[k]) { hi[k] = p[k]; hi_i[k] = i; }
    }
  }
  for (int i = lane; i < kFewPoints; i += L) s.adj[i] = 0u;
  if (ogjk::group_any<L>(bad)) return -2;
  wave_sync();
  int id[4];
  if (!first_tetrahedron<L>(pt, n, lane, lo, lo_i, hi, hi_i, id)) return 0;
  if (cap < 4) return -1;
  if (lane < 4) {
    const int a = init_corner(id, lane, 0), b = init_corner(id, lane, 1),
              c = init_corner(id, lane, 2);
    s.face[lane] = make_tri(s.pt[a], s.pt[b], s.pt[c], (uint32_t)(a | b << 8 | c << 16));
  }
  wave_sync();
  int nf = 4;
  const int k0 = lane / 3, e0 = lane - 3 * k0;  // the edge of this lane's first horizon test
  for (int q = 0; q < n; q++) {
    if (q == id[0] || q == id[1] || q == id[2] || q == id[3]) continue;
    const float4 Q = s.pt[q];
    // Visible faces leave the list (in place: a chunk is read before it is
    // written, and only to lower positions) and mark their edges.
    int nv = 0, w = 0;
    for (int base = 0; base < nf; base += L) {
      const int f = base + lane;
      const bool in = f < nf;
      const Tri F = s.face[in ? f : 0];
      const bool v = in && vol6(F, s.pt[F.ids & 255u], Q) > 1e-7f;
      const auto bv = ogjk::lanes_where<L>(v);
      const int left = nf - base < L ? nf - base : L;
      if (bv == 0 && nv == 0) {
        w += left;
        continue;
      }
      const int r = ogjk::lanes_below<L>(bv, lane);
      if (v) {
        s.vis[nv + r] = F.ids;
        const uint32_t a = F.ids & 255u, b = (F.ids >> 8) & 255u, c = F.ids >> 16;
        atomicOr(&s.adj[a], 1u << b);
        atomicOr(&s.adj[b], 1u << c);
        atomicOr(&s.adj[c], 1u << a);
      } else if (in) {
        s.face[w + lane - r] = F;  // lanes below that are not visible
      }
      const int c = ogjk::count_lanes<L>(bv);
      nv += c;
      w += left - c;
    }
    if (nv == 0) continue;
    wave_sync();
    // horizon: directed edges of visible faces whose reverse no visible face
    // has, in (visible face, edge) order; each is the base of a new face
    int nh = 0;
    const int ne = 3 * nv;
    for (int base = 0; base < ne; base += L) {
      const int h = base + lane;
      uint32_t a = 0u, b = 0u;
      bool hz = false;
      if (h < ne) {
        const int k = base == 0 ? k0 : h / 3, e = base == 0 ? e0 : h - 3 * k;
        const uint32_t ids = s.vis[k];
        a = (ids >> (8 * e)) & 255u;
        b = (e == 2 ? ids : ids >> (8 * e + 8)) & 255u;
        hz = !((s.adj[b] >> a) & 1u);
      }
      const auto bl = ogjk::lanes_where<L>(hz);
      const int r = w + nh + ogjk::lanes_below<L>(bl, lane);
      if (hz && r < kFewFaces)
        s.face[r] = make_tri(s.pt[a], s.pt[b], Q, a | b << 8 | (uint32_t)q << 16);
      nh += ogjk::count_lanes<L>(bl);
    }
    wave_sync();
    for (int i = lane; i < kFewPoints; i += L) s.adj[i] = 0u;
    nf = w + nh;
    if (nf > cap) return -1;
    if (nf > kFewFaces) return kToWave;
    wave_sync();
  }
  return nf;
}

// The clouds of up to kFewPoints points, 4 to a one-wave block; gridDim.x * 4
// groups take the clouds in turn.
__global__ __launch_bounds__(kWave) void k_hull_few(HullArgs h) {
  constexpr int L = kFewLanes, G = kWave / L;
  __shared__ FewHull lds[G];
  FewHull& s = lds[threadIdx.x / L];
  const int lane = threadIdx.x & (L - 1);
  const int groups = gridDim.x * G;
  const int g = blockIdx.x * G + threadIdx.x / L;
  // L clouds of this group at a time, the ones of its class by ballot
  for (int64_t first = g; first < h.nm; first += (int64_t)groups * L) {
    const int64_t mine = first + (int64_t)groups * lane;
    int n_mine = -1;
    if (mine < h.nm) n_mine = h.cnt[mine] < 0 ? 0 : h.cnt[mine];
    uint64_t todo = ogjk::group_ballot<L>(n_mine >= 0 && n_mine <= kFewPoints);
    while (todo != 0) {
      const int src = (int)__builtin_ctzll(todo);
      todo &= todo - 1;
      const int64_t m = first + (int64_t)groups * src;
      const int n = __shfl(n_mine, src, L);
      int nf;
      if (!h.range_ok(m)) {
        nf = -3;
      } else if (n < 4) {
        nf = 0;
      } else {
        nf = hull_few(h.points(m), n, h.cap(m), s, lane);
      }
      wave_sync();
      int32_t* out = h.out(m);
      for (int f = lane; f < nf; f += L) {
        const uint32_t ids = s.face[f].ids;
        out[3 * f] = (int32_t)(ids & 255u);
        out[3 * f + 1] = (int32_t)((ids >> 8) & 255u);
        out[3 * f + 2] = (int32_t)(ids >> 16);
      }
      if (lane == 0) h.nfaces[m] = nf;
    }
  }
}

// ------------------------------------------------------- a wave per cloud
//
// The faces in LDS, the points where they are.  Most insertions into a large
// cloud see no face, and then a step is one look at each face and nothing
// else; many clouds at once want as many waves as there is room for, and a
// barrier per insertion costs more than the other waves of a block bring: a
// block per cloud took 8.1 ms for 3,000 clouds of 1,024 points, most of them
// inside (0.64 ms with one wave each and the faces in global memory).  Hence:
//   * a face is 32 bytes with its plane and its first corner, so that the
//     visibility test is two LDS reads and no gather;
//   * a lane holds one of 64 points at a time, an insertion's point comes from
//     there by v_readlane;
//   * the visible faces' directed edges are listed as keys (start | end << 16)
//     and an edge is on the horizon if the list does not hold the reverse key:
//     up to 16 edges (as nearly always) are compared with all others in one
//     step, a quarter of the list per 16 lanes.
// When the list outgrows FB faces the cloud's state is saved (see load_state) and
// a kernel with more room goes on from there.
constexpr int kWavePoints = 65536;  // ids are 16 bits

template <int FB>
struct WaveHull {
  struct alignas(16) Corner {
    float y, z;
    uint32_t ab, c;  // ids: a | b << 16, c
  };
  float4 nx[FB];  // normal, x of corner a
  Corner co[FB];  // y and z of corner a
  alignas(16) uint32_t key[3 * FB + kWave];
};

// Where a cloud stands between two insertions: its faces in order in the
// output buffer, and at the start of its workspace six words: the number of
// faces, the next point, the first tetrahedron's points.  Only states of more
// faces than a wave's room are saved, so the words have a place.
__device__ __forceinline__ void load_state(const int32_t* save, int& nf, int& next, int (&id)[4]) {
  // not from the scalar cache: a wave of the same block may have written them
  const auto word = [&](int k) {
    return __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(save + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
  };
  nf = word(0);
  next = word(1);
#pragma unroll
  for (int k = 0; k < 4; k++) id[k] = word(2 + k);
}
__device__ __forceinline__ void store_state(int32_t* save, int nf, int next, const int (&id)[4]) {
  save[0] = nf;
  save[1] = next;
#pragma unroll
  for (int k = 0; k < 4; k++) save[2 + k] = id[k];
}

// The first tetrahedron's points of P[0..n), or the status that ends the build.
__device__ __forceinline__ int hull_begin(const float* __restrict__ P, int n, int cap, int lane, int (&id)[4]) {
  const auto pt = [&](int i) {
    return make_float4(P[3 * (int64_t)i], P[3 * (int64_t)i + 1], P[3 * (int64_t)i + 2], 0.0f);
  };
  float lo[3], hi[3];
  int lo_i[3], hi_i[3];
  bool bad = false;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    lo[k] = INFINITY;
    hi[k] = -INFINITY;
    lo_i[k] = hi_i[k] = -1;
  }
  for (int i = lane; i < n; i += kWave) {
    const float4 p4 = pt(i);
    const float p[3] = {p4.x, p4.y, p4.z};
#pragma unroll
    for (int k = 0; k < 3; k++) {
      bad |= !isfinite(p[k]);
      if (lo_i[k] < 0 || p[k] < lo[k]) { lo[k] = p[k]; lo_i[k] = i; }
      if (hi_i[k] < 0 || p[k] > hi[k]) { hi[k] = p[k]; hi_i[k] = i; }
    }
  }
  if (ballot(bad) != 0) return -2;
  if (!first_tetrahedron<kWave>(pt, n, lane, lo, lo_i, hi, hi_i, id)) return 0;
  return cap < 4 ? -1 : 4;
}

// Returns the face count (faces in s), a status of d_nfaces, or kSaved.
template <int FB>
__device__ __forceinline__ int hull_wave(const float* __restrict__ P, int n, int cap, WaveHull<FB>& s,
                         int32_t* out, int32_t* save, bool resume, int lane) {
  using Corner = typename WaveHull<FB>::Corner;
  const auto pt = [&](uint32_t i) { return make_float4(P[3 * i], P[3 * i + 1], P[3 * i + 2], 0.0f); };
  const auto put = [&](int f, uint32_t a, uint32_t b, uint32_t c, float4 A, float4 B, float4 C) {
    const Tri t = make_tri(A, B, C, 0u);
    s.nx[f] = make_float4(t.nx, t.ny, t.nz, A.x);
    s.co[f] = Corner{A.y, A.z, a | b << 16, c};
  };
  int id[4] = {0, 0, 0, 0};
  int nf = 4, q = 0;
  wave_sync();
  if (resume) {
    load_state(save, nf, q, id);
    if (nf > FB) return kSaved;
    for (int f = lane; f < nf; f += kWave) {
      const uint32_t a = out[3 * f], b = out[3 * f + 1], c = out[3 * f + 2];
      put(f, a, b, c, pt(a), pt(b), pt(c));
    }
  } else {
    const int st = hull_begin(P, n, cap, lane, id);
    if (st != 4) return st;
    if (lane < 4) {
      const uint32_t a = init_corner(id, lane, 0), b = init_corner(id, lane, 1),
                     c = init_corner(id, lane, 2);
      put(lane, a, b, c, pt(a), pt(b), pt(c));
    }
  }
  wave_sync();
  for (int from = q & ~(kWave - 1); from < n; from += kWave) {
    const float4 mine = pt(min(from + lane, n - 1));
    const int end = min(n, from + kWave);
    for (q = max(q, from); q < end; q++) {
      if (q == id[0] || q == id[1] || q == id[2] || q == id[3]) continue;
      const float4 Q = make_float4(ogjk::lane_value(mine.x, q - from),
                                   ogjk::lane_value(mine.y, q - from),
                                   ogjk::lane_value(mine.z, q - from), 0.0f);
      // Visible faces leave the list (in place: a chunk is read before it is
      // written, and only to lower positions) and list their edges.
      constexpr int U = 2;  // chunks in flight
      int nv = 0, w = 0;
      for (int base = 0; base < nf; base += U * kWave) {
        float4 N[U];
        Corner A[U];
        bool v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int f = min(base + u * kWave + lane, nf - 1);
          N[u] = s.nx[f];
          A[u] = s.co[f];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          const Tri t{N[u].x, N[u].y, N[u].z, 0u};
          v[u] = base + u * kWave + lane < nf &&
                 vol6(t, make_float4(N[u].w, A[u].y, A[u].z, 0.0f), Q) > 1e-7f;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          const uint64_t bv = ballot(v[u]);
          const int left = max(min(nf - base - u * kWave, kWave), 0);
          if (bv == 0 && nv == 0) {
            w += left;
            continue;
          }
          const int r = rank_below(bv, lane);
          if (v[u]) {
            uint32_t* k = s.key + 3 * (nv + r);
            const uint32_t a = A[u].ab & 0xffffu, b = A[u].ab >> 16, c = A[u].c;
            k[0] = A[u].ab;
            k[1] = b | c << 16;
            k[2] = c | a << 16;
          } else if (lane < left) {
            s.nx[w + lane - r] = N[u];  // lanes below that are not visible
            s.co[w + lane - r] = A[u];
          }
          const int c = __popcll(bv);
          nv += c;
          w += left - c;
        }
      }
      if (nv == 0) continue;
      // the list filled up to a multiple of 64 with a key that is no reverse:
      // an edge from a point to itself is on no face
      const int ne = 3 * nv;
      if (ne + lane < ((ne + kWave - 1) & ~(kWave - 1))) s.key[ne + lane] = 0u;
      wave_sync();
      // horizon: directed edges of visible faces whose reverse no visible face
      // has, in (visible face, edge) order; each is the base of a new face
      int nh = 0;
      const auto four = [&](int at) {
        uint4 k;
        __builtin_memcpy(&k, __builtin_assume_aligned(s.key + at, 16), sizeof(k));
        return k;
      };
      const auto any_of = [](uint4 k, uint32_t x) {
        return k.x == x || k.y == x || k.z == x || k.w == x;
      };
      for (int base = 0; base < ne; base += kWave) {
        uint32_t k;
        bool hz;
        if (ne <= 16) {
          k = s.key[lane & 15];
          const uint64_t b = ballot(any_of(four(lane >> 4 << 2), k << 16 | k >> 16));
          hz = lane < ne && !(((b | b >> 16 | b >> 32 | b >> 48) >> lane) & 1u);
        } else {
          k = s.key[base + lane];
          bool found = false;
          for (int j = 0; j < ne; j += 4) found |= any_of(four(j), k << 16 | k >> 16);
          hz = base + lane < ne && !found;
        }
        const uint64_t bl = ballot(hz);
        const int r = w + nh + rank_below(bl, lane);
        if (hz) {
          const uint32_t a = k & 0xffffu, b = k >> 16;
          if (r < FB) {
            put(r, a, b, (uint32_t)q, pt(a), pt(b), Q);
          } else if (r < cap) {  // straight to where the state is saved
            out[3 * r] = (int32_t)a;
            out[3 * r + 1] = (int32_t)b;
            out[3 * r + 2] = q;
          }
        }
        nh += __popcll(bl);
      }
      wave_sync();
      nf = w + nh;
      if (nf > cap) return -1;
      if (nf > FB) {
        for (int f = lane; f < FB; f += kWave) {
          out[3 * f] = (int32_t)(s.co[f].ab & 0xffffu);
          out[3 * f + 1] = (int32_t)(s.co[f].ab >> 16);
          out[3 * f + 2] = (int32_t)s.co[f].c;
        }
        if (lane == 0) store_state(save, nf, q + 1, id);
        return kSaved;
      }
    }
  }
  return nf;
}

template <int FB>
__device__ __forceinline__ void write_faces(const WaveHull<FB>& s, int nf, int32_t* out, int lane) {
  for (int f = lane; f < nf; f += kWave) {
    out[3 * f] = (int32_t)(s.co[f].ab & 0xffffu);
    out[3 * f + 1] = (int32_t)(s.co[f].ab >> 16);
    out[3 * f + 2] = (int32_t)s.co[f].c;
  }
}

// ------------------------------------------------------ over global memory
//
// Any size, one wave over the output buffer and the workspace (F: 3 * cap
// entries, vis: cap, hor: 2 * cap), from the start or from a saved state.

__device__ __forceinline__ float vol6(const float* __restrict__ p, int a, int b, int c,
                                      float qx, float qy, float qz) {
  const float ax = p[3 * a], ay = p[3 * a + 1], az = p[3 * a + 2];
  const float bx = p[3 * b] - ax, by = p[3 * b + 1] - ay, bz = p[3 * b + 2] - az;
  const float cx = p[3 * c] - ax, cy = p[3 * c + 1] - ay, cz = p[3 * c + 2] - az;
  const float dx = qx - ax, dy = qy - ay, dz = qz - az;
  const float nx = by * cz - bz * cy, ny = bz * cx - bx * cz, nz = bx * cy - by * cx;
  return nx * dx + ny * dy + nz * dz;
}

// Orders the global memory accesses of the lanes of one wave.
__device__ __forceinline__ void memory_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ int hull_global(const float* __restrict__ P, int n, int cap, int32_t* F, int32_t* vis,
                           int32_t* hor, bool resume, int lane) {
  int id[4] = {0, 0, 0, 0};
  int nf = 4, q = 0;
  memory_sync();
  if (resume) {
    load_state(vis, nf, q, id);  // it lies where the visible faces are listed
  } else {
    const int st = hull_begin(P, n, cap, lane, id);
    if (st != 4) return st;
    if (lane < 4) {
#pragma unroll
      for (int j = 0; j < 3; j++) F[3 * lane + j] = init_corner(id, lane, j);
    }
  }
  memory_sync();
  for (; q < n; q++) {
    if (q == id[0] || q == id[1] || q == id[2] || q == id[3]) continue;
    const float qx = P[3 * q], qy = P[3 * q + 1], qz = P[3 * q + 2];
    // visible faces, listed in ascending order
    int nv = 0;
    for (int base = 0; base < nf; base += kWave) {
      const int f = base + lane;
      bool v = false;
      if (f < nf) v = vol6(P, F[3 * f], F[3 * f + 1], F[3 * f + 2], qx, qy, qz) > 1e-7f;
      const uint64_t b = ballot(v);
      if (v) vis[nv + rank_below(b, lane)] = f;
      nv += __popcll(b);
    }
    if (nv == 0) continue;
    memory_sync();
    // horizon: directed edges of visible faces whose reverse no visible face
    // has, in (visible face, edge) order
    int nh = 0;
    const int ne = 3 * nv;
    for (int base = 0; base < ne; base += kWave) {
      const int h = base + lane;
      bool hz = false;
      int a = 0, b = 0;
      if (h < ne) {
        const int k = h / 3, e = h - 3 * k;
        const int g = vis[k];
        a = F[3 * g + e];
        b = F[3 * g + (e == 2 ? 0 : e + 1)];
        bool found = false;
        for (int k2 = 0; k2 < nv && !found; k2++) {
          const int g2 = vis[k2];
          const int x0 = F[3 * g2], x1 = F[3 * g2 + 1], x2 = F[3 * g2 + 2];
          found = (x0 == b && x1 == a) || (x1 == b && x2 == a) || (x2 == b && x0 == a);
        }
        hz = !found;
      }
      const uint64_t bl = ballot(hz);
      const int r = nh + rank_below(bl, lane);
      if (hz && r < cap) {
        hor[2 * r] = a;
        hor[2 * r + 1] = b;
      }
      nh += __popcll(bl);
    }
    memory_sync();
    // drop the visible faces, keeping the order of the others
    int w = 0;
    for (int base = 0; base < nf; base += kWave) {
      const int f = base + lane;
      bool alive = false;
      int x0 = 0, x1 = 0, x2 = 0;
      if (f < nf) {
        x0 = F[3 * f];
        x1 = F[3 * f + 1];
        x2 = F[3 * f + 2];
        alive = !(vol6(P, x0, x1, x2, qx, qy, qz) > 1e-7f);
      }
      const uint64_t b = ballot(alive);
      if (alive) {
        const int d = w + rank_below(b, lane);
        F[3 * d] = x0;
        F[3 * d + 1] = x1;
        F[3 * d + 2] = x2;
      }
      w += __popcll(b);
      memory_sync();
    }
    if (nh > cap || w + nh > cap) {
      return -1;
    }
    for (int r = lane; r < nh; r += kWave) {
      F[3 * (w + r)] = hor[2 * r];
      F[3 * (w + r) + 1] = hor[2 * r + 1];
      F[3 * (w + r) + 2] = q;
    }
    nf = w + nh;
    memory_sync();
  }
  return nf;
}

// RESUME: the clouds whose state was saved, else those of more than kFewPoints
// points and those of fewer that outgrew their lanes, from the start.  The waves
// of the grid take the clouds in turn.  Two steps, for the room: a compute unit
// has 22 waves of the first and 4, one to a SIMD, of the second (3 with 1,200 faces:
// 1,000 clouds of 256 points on a sphere 750 us, 460 with 880; 5 and 6 with 700 and
// 560: 2,000 clouds of 8-512 points 1.22 ms with 880, 1.38 with 1,200, 1.41, 1.64).
constexpr int kWaveFaces = 160, kWaveMoreFaces = 880;

template <int FB, bool RESUME>
__global__ __launch_bounds__(kWave) void k_hull_wave(HullArgs h) {
  __shared__ WaveHull<FB> s;
  const int lane = threadIdx.x;
  for (int64_t first = blockIdx.x; first < h.nm; first += (int64_t)gridDim.x * kWave) {
    const int64_t mine = first + (int64_t)gridDim.x * lane;
    int n_mine = 0;
    bool take = false;
    if (mine < h.nm) {
      n_mine = h.cnt[mine];
      take = RESUME ? h.nfaces[mine] == kSaved
                    : n_mine > kFewPoints || h.nfaces[mine] == kToWave;
    }
    uint64_t todo = ballot(take);
    while (todo != 0) {
      const int src = (int)__builtin_ctzll(todo);
      todo &= todo - 1;
      const int64_t m = first + (int64_t)gridDim.x * src;
      const int n = ogjk::lane_value(n_mine, src);
      int nf = -3;
      if (RESUME || (h.range_ok(m) && n <= kWavePoints)) {
        nf = hull_wave(h.points(m), n, h.cap(m), s, h.out(m), h.work(m), RESUME, lane);
        write_faces(s, nf, h.out(m), lane);
      } else if (h.range_ok(m)) {
        nf = hull_global(h.points(m), n, h.cap(m), h.out(m), h.work(m), h.work(m) + h.cap64(m),
                         false, lane);
      }
      if (lane == 0) h.nfaces[m] = nf;
    }
  }
}

// ------------------------------------------------------ a block per cloud
//
// For clouds of up to kBlockPoints points whose face list outgrows a wave's: the
// whole block tests the faces and notes the visible ones, then the first wave
// alone does the ordered part (horizon, new faces).  Two barriers per insertion,
// but a lone wave takes some 70 instructions for every 64 faces.  A face that
// leaves stays behind as a dead slot, so nothing moves: slots are in creation
// order, which is the order the reference's compaction keeps, and the first
// wave closes the gaps now and then.  Each wave tests one contiguous run of
// slots, so the waves' lists of visible faces joined together are in slot order.
// On dense, nearly coplanar surfaces the face list grows tenfold and more within
// the last insertions (a cloud of 8-512 points took 10 ms and more over global
// memory): when the faces with their planes outgrow the LDS, they are kept as
// vertex ids alone (4 bytes a face, the normal formed anew from the corners).
// A call over few clouds is one launch of this kernel: each block's first wave
// starts its cloud, and the block goes on from kAloneFaces faces, where a wave's
// insertion takes as long (512 points: 0.83 ms, 1.16 with the wave to the end,
// 1.2 with the block from 64 faces).  16 waves a block, one block to a compute
// unit: 8 are 2% faster there, but clouds that end over global memory want all
// the waves (300 clouds of 1,500 points on a sphere 58 ms with 512 blocks of 8
// waves, 37 with 256 of 16).
constexpr int kBlockThreads = 1024, kBlockWaves = kBlockThreads / kWave, kBlockPoints = 1024;
constexpr int kAloneFaces = 512;
constexpr int kBlocksAtOnce = 256;  // compute units, one block each

// Directed edges of the visible faces, in the same room: a bit per (start, end)
// for at most kBitPoints points, else a hash set.  (One type that looks at the
// point count cost the former 0.8 us an insertion.)
constexpr int kBitPoints = 512, kEdgeWords = 8192;

struct EdgeBits {
  static constexpr uint32_t kClear = 0u;
  uint32_t word[kEdgeWords];
  __device__ __forceinline__ static uint32_t place(uint32_t a, uint32_t b) {
    return a * (kBitPoints / 32) + (b >> 5);
  }
  __device__ __forceinline__ bool insert(uint32_t a, uint32_t b) {
    atomicOr(&word[place(a, b)], 1u << (b & 31u));
    return true;
  }
  __device__ __forceinline__ bool found(uint32_t a, uint32_t b) const {
    return (word[place(a, b)] >> (b & 31u)) & 1u;
  }
  // after the last look-up of a step
  __device__ __forceinline__ void erase(uint32_t a, uint32_t b) { word[place(a, b)] = kClear; }
};

struct EdgeHash {
  static constexpr uint32_t kClear = 0xffffffffu;
  static constexpr int kProbes = 32;  // an edge lies within this many places of its own, or nowhere
  uint32_t word[kEdgeWords];
  __device__ __forceinline__ static uint32_t place(uint32_t k, int p) {
    return ((k * 0x9e3779b1u >> 19) + p) & (kEdgeWords - 1);
  }
  __device__ __forceinline__ bool insert(uint32_t a, uint32_t b) {
    const uint32_t k = a << 10 | b;
    for (int p = 0; p < kProbes; p++) {
      const uint32_t was = atomicCAS(&word[place(k, p)], kClear, k);
      if (was == kClear || was == k) return true;
    }
    return false;
  }
  __device__ __forceinline__ bool found(uint32_t a, uint32_t b) const {
    const uint32_t k = a << 10 | b;
    for (int p = 0; p < kProbes; p++) {
      const uint32_t x = word[place(k, p)];
      if (x == k) return true;
      if (x == kClear) return false;
    }
    return false;
  }
  // Places of other edges may be clear already, so a clear one does not end
  // the search.
  __device__ __forceinline__ void erase(uint32_t a, uint32_t b) {
    const uint32_t k = a << 10 | b;
    for (int p = 0; p < kProbes; p++) {
      if (word[place(k, p)] == k) {
        word[place(k, p)] = kClear;
        return;
      }
    }
  }
};

template <bool PLANES, class Edges>
struct BlockHull {
  using Face = std::conditional_t<PLANES, Tri, uint32_t>;
  static constexpr int kFaces = 65536 / sizeof(Face);
  static constexpr int kRoom = kFaces / 8;  // slots an insertion finds free
  static constexpr int kSeg = 256;          // visible faces a wave lists at an insertion
  static constexpr int kRow = kWave / kBlockWaves;  // of which the first wave takes these in one go
  Face face[kFaces];  // ids: 3 x 10 bits, kDead, kLate
  float4 pt[kBlockPoints];
  Edges edges;
  uint32_t seg[kBlockWaves][kSeg];  // vertex ids of the visible faces each wave found
  int cnt[2][kBlockWaves];          // how many, by the parity of the step
  int tail, status;                 // read by every thread after an insertion
  int full;                         // an edge found no place
};
// Flags beside a slot's ids: the face has left, and it left at the insertion at
// hand and is on no wave's list.
constexpr uint32_t kDead = 0x80000000u, kLate = 0x40000000u;

__device__ __forceinline__ uint32_t& ids_of(Tri& f) { return f.ids; }
__device__ __forceinline__ uint32_t& ids_of(uint32_t& f) { return f; }

// Live slots of [0, tail) moved down in order, by one wave.  Returns their count.
template <class Face>
__device__ __forceinline__ int close_gaps(Face* face, int tail, int lane) {
  // as plain words: copies of the struct end in the stack frame
  using Words = std::conditional_t<sizeof(Face) == sizeof(uint4), uint4, uint32_t>;
  int w = 0;
  for (int base = 0; base < tail; base += kWave) {
    const int f = base + lane;
    Words F;
    __builtin_memcpy(&F, &face[min(f, tail - 1)], sizeof(F));
    const bool live = f < tail && !(ids_of(face[min(f, tail - 1)]) & kDead);
    const uint64_t b = ballot(live);
    wave_sync();
    if (live) __builtin_memcpy(&face[w + rank_below(b, lane)], &F, sizeof(F));
    wave_sync();
    w += __popcll(b);
  }
  return w;
}

__device__ __forceinline__ void write_ids(int32_t* out, uint32_t ids) {
  out[0] = (int32_t)(ids & 1023u);
  out[1] = (int32_t)((ids >> 10) & 1023u);
  out[2] = (int32_t)(ids >> 20);
}

// Whole block, from a saved state.  Returns the face count (faces in
// s.face[0..)), a status of d_nfaces, or kSaved when the slots or the edge set
// are too few: the state is then the one of the last insertion that left room
// for another, or the one it started from.
template <bool PLANES, class Edges>
__device__ __forceinline__ int hull_block(const float* __restrict__ P, int n, int cap, BlockHull<PLANES, Edges>& s,
                          int32_t* out, int32_t* save) {
  using B = BlockHull<PLANES, Edges>;
  constexpr int T = kBlockThreads, S = B::kFaces;
  static_assert(kBlockPoints <= 1024, "vertex ids are packed in 10 bits");
  const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  const auto put = [&](int f, float4 a, float4 b, float4 c, uint32_t ids) {
    if constexpr (PLANES) s.face[f] = make_tri(a, b, c, ids);
    else s.face[f] = ids;
  };
  __syncthreads();  // the block's LDS is free
  int tail, q0, id[4];
  load_state(save, tail, q0, id);
  if (tail > S - B::kRoom) return kSaved;
  int alive = tail;  // the first wave's
  for (int i = t; i < kEdgeWords; i += T) s.edges.word[i] = Edges::kClear;
  for (int i = t; i < n; i += T) s.pt[i] = make_float4(P[3 * i], P[3 * i + 1], P[3 * i + 2], 0.0f);
  if (t == 0) {
    s.full = 0;
    s.status = 4;
  }
  __syncthreads();
  for (int f = t; f < tail; f += T) {
    const uint32_t a = out[3 * f], b = out[3 * f + 1], c = out[3 * f + 2];
    put(f, s.pt[a], s.pt[b], s.pt[c], a | b << 10 | c << 20);
  }
  __syncthreads();
  float4 next = s.pt[min(q0, n - 1)];
  for (int q = q0, step = 0; q < n; q++) {
    const float4 Q = next;
    next = s.pt[q + 1 < n ? q + 1 : q];
    if (q == id[0] || q == id[1] || q == id[2] || q == id[3]) continue;
    const int run = (tail + T - 1) / T * kWave;
    const int end = min(tail, (wave + 1) * run);
    int found = 0;
    constexpr int U = 2;  // chunks in flight
    for (int base = wave * run; base < end; base += U * kWave) {
      typename B::Face F[U];
      bool v[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        F[u] = s.face[min(base + u * kWave + lane, end - 1)];
        if (base + u * kWave + lane >= end) ids_of(F[u]) = kDead;
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const uint32_t ids = ids_of(F[u]);
        const float4 a = s.pt[ids & 1023u];
        float d;
        if constexpr (PLANES) d = vol6(F[u], a, Q);
        else d = vol6(a, s.pt[(ids >> 10) & 1023u], s.pt[(ids >> 20) & 1023u], Q);
        v[u] = !(ids & kDead) && d > 1e-7f;
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const uint64_t bv = ballot(v[u]);
        if (v[u]) {
          const int f = base + u * kWave + lane;
          const uint32_t ids = ids_of(F[u]);
          const uint32_t x = ids & 1023u, y = (ids >> 10) & 1023u, z = ids >> 20;
          const int r = found + rank_below(bv, lane);
          ids_of(s.face[f]) = ids | (r < B::kSeg ? kDead : kDead | kLate);
          if (r < B::kSeg) s.seg[wave][r] = ids;
          const bool i0 = s.edges.insert(x, y), i1 = s.edges.insert(y, z),
                     i2 = s.edges.insert(z, x);
          if (!i0 || !i1 || !i2) s.full = 1;
        }
        found += __popcll(bv);
      }
    }
    int* cnt = s.cnt[step & 1];
    if (lane == 0) cnt[wave] = found;
    step++;
    __syncthreads();
    const int here = cnt[lane / B::kRow];  // found by the wave whose row this lane stands for
    if (ballot(here != 0) == 0) continue;
    if (wave == 0) {
      int status = 4, nh = 0, nv = 0, at = tail;
      if (s.full) {
        status = kSaved;
      } else {
        // Each lane takes a visible face (valid: ids), in slot order: its
        // edges whose reverse no visible face has are bases of new faces, in
        // (face, edge) order.
        const auto fan = [&](bool valid, uint32_t ids) {
          const uint32_t x[3] = {ids & 1023u, (ids >> 10) & 1023u, ids >> 20};
          float4 p[3];
          bool hz[3];
#pragma unroll
          for (int e = 0; e < 3; e++) p[e] = s.pt[x[e]];
#pragma unroll
          for (int e = 0; e < 3; e++) hz[e] = valid && !s.edges.found(x[(e + 1) % 3], x[e]);
          int r = at + nh;
#pragma unroll
          for (int e = 0; e < 3; e++) {
            const uint64_t b = ballot(hz[e]);
            r += rank_below(b, lane);
            nh += __popcll(b);
          }
#pragma unroll
          for (int e = 0; e < 3; e++) {
            if (hz[e]) {
              if (r < S)
                put(r, p[e], p[(e + 1) % 3], Q, x[e] | x[(e + 1) % 3] << 10 | (uint32_t)q << 20);
              r++;
            }
          }
        };
        const auto unmark = [&](uint32_t ids) {
          const uint32_t x0 = ids & 1023u, x1 = (ids >> 10) & 1023u, x2 = ids >> 20;
          s.edges.erase(x0, x1);
          s.edges.erase(x1, x2);
          s.edges.erase(x2, x0);
        };
        if (ballot(here > B::kRow) == 0) {
          // a few per wave, as always but on dense clouds: lane (wave, rank)
          const int w = lane / B::kRow, k = lane - w * B::kRow;
          const bool valid = k < here;
          const uint32_t ids = valid ? s.seg[w][k] : 0u;
          nv = __popcll(ballot(valid));
          fan(valid, ids);
          if (valid) unmark(ids);
        } else if (ballot(here > B::kSeg) != 0) {
          // A wave saw more than its list holds: new faces sit together at the
          // tail, so a cloud whose face list grows fast has most of its visible
          // ones in a few waves' runs.  Those past a list's end are found again
          // by their flag, in the slots of the wave's run, behind the listed ones.
          const auto each = [&](const auto& f) {
            for (int w = 0; w < kBlockWaves; w++) {
              const int c = cnt[w], listed = min(c, B::kSeg);
              for (int base = 0; base < listed; base += kWave)
                f(base + lane < listed, base + lane < listed ? s.seg[w][base + lane] : 0u, -1);
              if (c == listed) continue;
              const int stop = min(tail, (w + 1) * run);
              for (int base = w * run; base < stop; base += kWave) {
                const int slot = base + lane;
                const uint32_t ids = slot < stop ? ids_of(s.face[slot]) : 0u;
                f((ids & kLate) != 0, ids & ~(kDead | kLate), slot);
              }
            }
          };
          nv = 0;
          each([&](bool valid, uint32_t ids, int) {
            nv += __popcll(ballot(valid));
            fan(valid, ids);
          });
          each([&](bool valid, uint32_t ids, int slot) {
            if (valid) unmark(ids);
            if (valid && slot >= 0) ids_of(s.face[slot]) = ids | kDead;
          });
        } else {
          int pre[kBlockWaves + 1];  // visible faces of the waves before
          pre[0] = 0;
#pragma unroll
          for (int w = 0; w < kBlockWaves; w++) pre[w + 1] = pre[w] + cnt[w];
          nv = pre[kBlockWaves];
          const auto visible = [&](int j) {
            int w = 0, st = 0;
#pragma unroll
            for (int k = 1; k < kBlockWaves; k++) {
              w = j >= pre[k] ? k : w;
              st = j >= pre[k] ? pre[k] : st;
            }
            return s.seg[w][j - st];
          };
          for (int base = 0; base < nv; base += kWave) {
            const bool valid = base + lane < nv;
            fan(valid, valid ? visible(base + lane) : 0u);
          }
          for (int j = lane; j < nv; j += kWave) unmark(visible(j));
        }
        alive += nh - nv;
        at += nh;
        if (alive > cap) {
          status = -1;
        } else if (at > S) {
          status = kSaved;
        } else if (at > S - B::kRoom || at > alive + alive / 8 + 256) {
          wave_sync();
          at = close_gaps(s.face, at, lane);
          if (at > S - B::kRoom) {
            for (int f = lane; f < at; f += kWave) write_ids(out + 3 * f, ids_of(s.face[f]));
            if (lane == 0) store_state(save, at, q + 1, id);
            status = kSaved;
          }
        }
      }
      if (lane == 0) {
        s.tail = at;
        s.status = status;
      }
    }
    __syncthreads();
    const int status = __builtin_amdgcn_readfirstlane(s.status);
    if (status != 4) return status;
    tail = __builtin_amdgcn_readfirstlane(s.tail);
  }
  __syncthreads();
  if (wave == 0) {
    const int nf = close_gaps(s.face, tail, lane);
    if (lane == 0) s.tail = nf;
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(s.tail);
}

// One cloud from its saved state; the block writes the faces out.
template <bool PLANES, class Edges>
__device__ __forceinline__ int hull_block_out(const HullArgs& h, int64_t m, int n,
                                              BlockHull<PLANES, Edges>& s) {
  const int nf = hull_block(h.points(m), n, h.cap(m), s, h.out(m), h.work(m));
  int32_t* out = h.out(m);
  for (int f = threadIdx.x; f < nf; f += kBlockThreads) write_ids(out + 3 * f, ids_of(s.face[f]));
  return nf;
}

// ALL: every cloud of the call, from the start, else those whose state was
// saved.  The blocks of the grid take the clouds in turn; a block's clouds that
// it has no room for are spread over its waves at the end, over global memory.
template <bool ALL>
__global__ __launch_bounds__(kBlockThreads) void k_hull_block(HullArgs h) {
  __shared__ union Lds {
    WaveHull<kAloneFaces> w;
    BlockHull<true, EdgeBits> p;
    BlockHull<false, EdgeBits> b;
    BlockHull<true, EdgeHash> ph;
    BlockHull<false, EdgeHash> bh;
  } s;
  __shared__ int result;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  for (int64_t first = blockIdx.x; first < h.nm; first += (int64_t)gridDim.x * kWave) {
    const int64_t mine = first + (int64_t)gridDim.x * lane;
    const int n_mine = mine < h.nm ? h.cnt[mine] : 0;
    uint64_t todo = ballot(mine < h.nm && (ALL || h.nfaces[mine] == kSaved));
    uint64_t large = 0;  // the same in every wave, as todo is
    __syncthreads();     // every wave has read the counts that this block writes
    while (todo != 0) {
      const int src = (int)__builtin_ctzll(todo);
      todo &= todo - 1;
      const int64_t m = first + (int64_t)gridDim.x * src;
      const int n = ogjk::lane_value(n_mine, src);
      int nf = kSaved;
      if (ALL) {
        __syncthreads();  // the block's LDS is free
        if (wave == 0) {
          int r = kSaved;
          if (!h.range_ok(m)) {
            r = -3;
          } else if (n < 4) {
            r = 0;
          } else if (n <= kWavePoints) {
            r = hull_wave(h.points(m), n, h.cap(m), s.w, h.out(m), h.work(m), false, lane);
            write_faces(s.w, r, h.out(m), lane);
          }
          if (lane == 0) result = r;
        }
        __syncthreads();
        nf = __builtin_amdgcn_readfirstlane(result);
      }
      if (nf == kSaved && n <= kBitPoints) {
        nf = hull_block_out(h, m, n, s.p);
        if (nf == kSaved) nf = hull_block_out(h, m, n, s.b);
      } else if (nf == kSaved && n <= kBlockPoints) {
        nf = hull_block_out(h, m, n, s.ph);
        if (nf == kSaved) nf = hull_block_out(h, m, n, s.bh);
      }
      if (nf == kSaved) large |= 1ull << src;
      else if (threadIdx.x == 0) h.nfaces[m] = nf;
    }
    __syncthreads();
    for (int k = 0; large != 0; k++) {
      const int src = (int)__builtin_ctzll(large);
      large &= large - 1;
      if (wave != k % kBlockWaves) continue;
      const int64_t m = first + (int64_t)gridDim.x * src;
      const int n = ogjk::lane_value(n_mine, src);
      const int nf = hull_global(h.points(m), n, h.cap(m), h.out(m), h.work(m),
                                 h.work(m) + h.cap64(m), !ALL || n <= kWavePoints, lane);
      if (lane == 0) h.nfaces[m] = nf;
    }
  }
}

// Moments summed in face order (mesh_builder.cpp:433-462), centre of mass as
// center_hull_verts shifts by it (0 below volume 1e-10) and the inertia factors
// of compute_hull_inertia_k (:464-481).  L lanes per cloud work out the terms of
// L faces at a time; then lane k < 7 adds the k-th moment's terms one by one
// in face order (the sums' bits depend on it).  A wave holds 64 / 16 clouds
// of at most 64 faces, a larger cloud gets the wave to itself.  Bound by the
// gathers and the chain of additions; with one thread per cloud 100,000
// clouds of 8-32 points took 95 us (now 43), 2,000 of 8-512 points 570 (51).
constexpr int kMom = 7;

template <int L>
__device__ __forceinline__ double hull_moment(const float* __restrict__ P,
                                              const int32_t* __restrict__ F, int nf,
                                              double (*term)[kWave], int base_lane, int lane) {
  double acc = 0.0;
  for (int base = 0; base < nf; base += L) {
    const int f = base + lane;
    if (f < nf) {
      const float* a = P + 3 * (int64_t)F[3 * (int64_t)f];
      const float* b = P + 3 * (int64_t)F[3 * (int64_t)f + 1];
      const float* c = P + 3 * (int64_t)F[3 * (int64_t)f + 2];
      const double dv =
          ((double)a[0] * ((double)b[1] * (double)c[2] - (double)b[2] * (double)c[1]) -
           (double)a[1] * ((double)b[0] * (double)c[2] - (double)b[2] * (double)c[0]) +
           (double)a[2] * ((double)b[0] * (double)c[1] - (double)b[1] * (double)c[0])) /
          6.0;
      const int at = base_lane + lane;
      term[0][at] = dv;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        term[1 + k][at] = dv * (a[k] + b[k] + c[k]);
        term[4 + k][at] = dv / 10.0 *
                          ((double)a[k] * a[k] + (double)a[k] * b[k] + (double)b[k] * b[k] +
                           (double)a[k] * c[k] + (double)b[k] * c[k] + (double)c[k] * c[k]);
      }
    }
    wave_sync();
    if (lane < kMom) {
      const int m = nf - base < L ? nf - base : L;
      const double* t = term[lane] + base_lane;
      int j = 0;
      for (; j + 8 <= m; j += 8) {
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; u++) x[u] = t[j + u];
#pragma unroll
        for (int u = 0; u < 8; u++) acc += x[u];
      }
      for (; j < m; j++) acc += t[j];
    }
    wave_sync();
  }
  return acc;
}

__global__ __launch_bounds__(kWave) void k_hull_moments(const float* __restrict__ pts,
                                                        const int64_t* __restrict__ off,
                                                        const int32_t* __restrict__ faces,
                                                        const int64_t* __restrict__ face_off,
                                                        const int32_t* __restrict__ nfaces, int nm,
                                                        double* __restrict__ moments,
                                                        float* __restrict__ com,
                                                        float* __restrict__ inertia_k) {
  constexpr int L = 16, G = kWave / L;
  __shared__ double term[kMom][kWave];
  const int lane = threadIdx.x, sub = lane & (L - 1), g0 = lane & ~(L - 1);
  const int m = blockIdx.x * G + lane / L;
  int nf = 0;
  const float* P = pts;
  const int32_t* F = faces;
  if (m < nm) {
    nf = nfaces[m] > 0 ? nfaces[m] : 0;
    P = pts + 3 * off[m];
    F = faces + 3 * face_off[m];
  }
  double acc = hull_moment<L>(P, F, nf <= kWave ? nf : 0, term, g0, sub);
  for (uint64_t big = ballot(sub == 0 && nf > kWave); big != 0; big &= big - 1) {
    const int src = (int)__builtin_ctzll(big);
    const int mb = blockIdx.x * G + src / L;
    const double a = hull_moment<kWave>(pts + 3 * off[mb], faces + 3 * face_off[mb], nfaces[mb],
                                        term, 0, lane);
    const double mine = __shfl(a, sub, kWave);  // lanes 0..6 hold the moments
    if (g0 == src) acc = mine;
  }
  double mo[kMom];
#pragma unroll
  for (int k = 0; k < kMom; k++) mo[k] = __shfl(acc, k, L);
  if (m >= nm) return;
  if (sub < kMom) moments[kMom * (int64_t)m + sub] = acc;
  if (sub != 0) return;
  const double vol = mo[0];
  float* co = com + 3 * (int64_t)m;
  float* ko = inertia_k + 3 * (int64_t)m;
  if (vol < 1e-10) {
    co[0] = co[1] = co[2] = 0.0f;
    ko[0] = ko[1] = ko[2] = 1.0f / 10.0f;
    return;
  }
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const double c = mo[1 + k] / (4.0 * vol);
    co[k] = (float)c;
    ko[k] = (float)((mo[4 + k] - vol * c * c) / vol);
  }
}

// points of cloud m minus com[m], one thread per point
__global__ __launch_bounds__(256) void k_center(float* __restrict__ pts,
                                                const int32_t* __restrict__ cloud,
                                                int64_t n_points,
                                                const float* __restrict__ com) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n_points;
       i += (int64_t)gridDim.x * 256) {
    const float* c = com + 3 * (int64_t)cloud[i];
    pts[3 * i] -= c[0];
    pts[3 * i + 1] -= c[1];
    pts[3 * i + 2] -= c[2];
  }
}

ogjk_status hip_err(hipError_t e, const char* what) {
  return ogjk_fail(e == hipErrorOutOfMemory ? OGJK_ERR_NOMEM : OGJK_ERR_HIP, "%s: %s", what,
                   hipGetErrorString(e));
}

}  // namespace

extern "C" {

ogjk_status ogjk_build_hulls(const float* d_points, const int64_t* d_point_off,
                             const int32_t* d_point_cnt, int32_t n_clouds,
                             const int64_t* d_face_off, int64_t total_faces, int32_t* d_faces,
                             int32_t* d_nfaces, void* d_workspace, size_t workspace_bytes,
                             void* stream) {
  if (n_clouds < 0 || total_faces < 0)
    return ogjk_fail(OGJK_ERR_INVALID, "n_clouds and total_faces must be >= 0");
  if (n_clouds == 0) return OGJK_OK;
  if (!d_points || !d_point_off || !d_point_cnt || !d_face_off || !d_faces || !d_nfaces)
    return ogjk_fail(OGJK_ERR_INVALID, "NULL argument");
  const size_t need = (size_t)total_faces * 3 * sizeof(int32_t);
  if (!d_workspace || workspace_bytes < need)
    return ogjk_fail(OGJK_ERR_INVALID, "workspace of %zu bytes needed", need);
  const hipStream_t st = (hipStream_t)stream;
  const HullArgs h{d_points, d_point_off, d_point_cnt, n_clouds, d_face_off, total_faces,
                   d_faces, d_nfaces, (int32_t*)d_workspace};
  // Sizes are on the device, so each kernel goes over the counts and takes its
  // own clouds.  A block has room for any of them and a compute unit for one
  // such block, so up to as many clouds are one launch (10 clouds of 8 points 41
  // us, 53 as four launches); past that the launches by size, of which an idle
  // one takes about 3 us.  Waves are launched per cloud as far as an idle launch
  // stays cheap, so that the dispatcher balances them; larger batches take the
  // clouds in turn.
  const auto grid = [&](int clouds_per_block, int64_t most) {
    const int64_t b = ((int64_t)n_clouds + clouds_per_block - 1) / clouds_per_block;
    return dim3((unsigned)(b < most ? b : most));
  };
  if (n_clouds <= kBlocksAtOnce) {
    hipLaunchKernelGGL((k_hull_block<true>), dim3((unsigned)n_clouds), dim3(kBlockThreads), 0, st, h);
  } else {
    hipLaunchKernelGGL(k_hull_few, grid(kWave / kFewLanes, 1 << 20), dim3(kWave), 0, st, h);
    hipLaunchKernelGGL((k_hull_wave<kWaveFaces, false>), grid(1, 4096), dim3(kWave), 0, st, h);
    hipLaunchKernelGGL((k_hull_wave<kWaveMoreFaces, true>), grid(1, 4096), dim3(kWave), 0, st, h);
    hipLaunchKernelGGL((k_hull_block<false>), grid(1, kBlocksAtOnce), dim3(kBlockThreads), 0, st,
                       h);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? OGJK_OK : hip_err(e, "hull launch");
}

ogjk_status ogjk_hull_moments(const float* d_points, const int64_t* d_point_off,
                              const int32_t* d_faces, const int64_t* d_face_off,
                              const int32_t* d_nfaces, int32_t n_clouds, double* d_moments,
                              float* d_com, float* d_inertia_k, void* stream) {
  if (n_clouds < 0) return ogjk_fail(OGJK_ERR_INVALID, "n_clouds < 0");
  if (n_clouds == 0) return OGJK_OK;
  if (!d_points || !d_point_off || !d_faces || !d_face_off || !d_nfaces || !d_moments ||
      !d_com || !d_inertia_k)
    return ogjk_fail(OGJK_ERR_INVALID, "NULL argument");
  hipLaunchKernelGGL(k_hull_moments, dim3((unsigned)((n_clouds + 3) / 4)), dim3(kWave), 0,
                     (hipStream_t)stream, d_points, d_point_off, d_faces, d_face_off, d_nfaces,
                     n_clouds, d_moments, d_com, d_inertia_k);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? OGJK_OK : hip_err(e, "moments launch");
}

ogjk_status ogjk_center_points(float* d_points, const int32_t* d_point_cloud, int64_t n_points,
                               const float* d_com, void* stream) {
  if (n_points < 0) return ogjk_fail(OGJK_ERR_INVALID, "n_points < 0");
  if (n_points == 0) return OGJK_OK;
  if (!d_points || !d_point_cloud || !d_com) return ogjk_fail(OGJK_ERR_INVALID, "NULL argument");
  const int64_t cb = (n_points + 255) / 256;
  hipLaunchKernelGGL(k_center, dim3((unsigned)(cb < 65536 ? cb : 65536)), dim3(256), 0,
                     (hipStream_t)stream, d_points, d_point_cloud, n_points, d_com);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? OGJK_OK : hip_err(e, "centre launch");
}

}  // extern "C"
