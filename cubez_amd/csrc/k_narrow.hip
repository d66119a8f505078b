// k_narrow.hip — K2: the narrowphase over ordered pairs, with contacts
// compacted in the reference's emission order.
//
// Emission order (examples/cubedrop.go:47-64): for each body i of a world,
// first its half-space checks (planes in order, up to 8 cube vertices each
// in the `mults` order of colliders.go:319-327), then CheckForCollisions(i, j)
// for every j != i in ascending order.  Row r of a world has np + n columns
// (planes, then bodies; column j == r is never a pair), cut into 64-column
// tiles; tiles are ordered row by row, so scanning their contact totals in
// tile order gives every contact its slot in the reference's order.  An
// explicit pair list (any caller loop) uses its own order instead, 64
// consecutive entries per tile.
//
// Launches (all-pairs):
//   cull        — one wave per (column tile, 16 rows): clears the tiles and
//                 lists the candidate body pairs (i, j), i < j.  Cube-cube
//                 and cube-sphere pairs whose bounding spheres are far apart
//                 are rejected: the bound guarantees that the reference's own
//                 test reports no contact (see far_apart below), so the
//                 result is unchanged.
//   eval        — one thread per body (its planes) and per candidate: the
//                 reference's test; per tile a hit bitmask and contact total,
//                 and the hit list.  A pair is tested once for both orders:
//                 swapping the bodies negates the centre offset and the cross
//                 products and swaps the terms of sums, so every comparison
//                 of the test (colliders.go:216-254, 369-441, 445-477) comes
//                 out the same, NaNs included.
//   scan_tiles  — one wave per world: exclusive scan of tile totals.
//   scan_worlds — one block: exclusive scan of world totals.
//   emit_hits   — one thread per hit pair: recompute it and write its
//                 contacts at world offset + tile offset + in-tile prefix.
// (The explicit-list form counts and emits one wave per tile.)
// All geometry is evaluated in FP64 whatever the storage type R.
#include <algorithm>

#include "cbz_devmath.h"
#include "cbz_launch.h"
#include "cbz_types.h"
#include "cbz_wave.h"

namespace cbz {

using D3 = V3<double>;

struct Col {
  double T[12];
  double h[3];
  int shape;
};

template <typename R>
__device__ __forceinline__ void load_col(const Bodies<R>& b, int i, Col& c) {
  const int64_t S = b.stride;
#pragma unroll
  for (int k = 0; k < 12; ++k) c.T[k] = double(b.ctransform[k * S + i]);
  c.h[0] = double(b.half[i]);
  c.h[1] = double(b.half[S + i]);
  c.h[2] = double(b.half[2 * S + i]);
  c.shape = b.shape[i];
}

template <typename R>
struct NP {
  Bodies<R> b;
  Planes<R> pl;
  PairSpace ps;
  Contacts<R> c;
  const double* brad;  // conservative bounding radius per body
  int32_t* tile_cnt;
  uint64_t* tile_mask;
  int32_t* tile_off;
  int32_t* world_cnt;
  int64_t* world_coff;
  int64_t* total;
  int32_t* overflow;
  uint32_t* hits;
  int32_t* n_hits;
  uint32_t* cand;
  int32_t* n_pairs;
  int32_t* n_cand;
  int64_t cand_cap, plane_pairs;
  const int32_t* body_world;
  int32_t max_planes;
  int32_t n_worlds;
  Materials<R> mat;  // read when c.fric is set
};

// Writes one contact.  m1 names the contact's second material: body b1 for
// a body pair, -(k+1) for plane k (Bodies[1] is nil there).  With materials
// on, the contact's friction and restitution are the means of body b0's and
// m1's values (the reference gives every contact 0.9 and 0.1,
// colliders.go:201-202, 248-249, 360-361, 437-438, 511-512, 704-705).
template <typename R>
__device__ __forceinline__ void put_contact(const NP<R>& a, int64_t slot, int b0, int b1, int m1, const D3& p,
                                            const D3& n, double pen) {
  const Contacts<R>& c = a.c;
  if (slot >= c.cap) return;
  const int64_t S = c.cap;
  c.body0[slot] = b0;
  c.body1[slot] = b1;
  c.point[slot] = R(p.x);
  c.point[S + slot] = R(p.y);
  c.point[2 * S + slot] = R(p.z);
  c.normal[slot] = R(n.x);
  c.normal[S + slot] = R(n.y);
  c.normal[2 * S + slot] = R(n.z);
  c.pen[slot] = R(pen);
  if (c.fric) {
    const Materials<R>& m = a.mat;
    const R f1 = m1 >= 0 ? m.body_fric[m1] : m.plane_fric[-m1 - 1];
    const R e1 = m1 >= 0 ? m.body_rest[m1] : m.plane_rest[-m1 - 1];
    c.fric[slot] = (m.body_fric[b0] + f1) * R(0.5);
    c.rest[slot] = (m.body_rest[b0] + e1) * R(0.5);
  }
}

// GetAxis / HalfSize[i] with a run-time index, re-read from the body arrays
// (a dynamic index into a register array would put the whole collider in
// scratch memory).
template <typename R>
__device__ __forceinline__ D3 axis_g(const NP<R>& a, int body, int col) {
  const int c = col > 3 ? 3 : col;
  const int64_t S = a.b.stride;
  return D3{double(a.b.ctransform[(3 * c) * S + body]), double(a.b.ctransform[(3 * c + 1) * S + body]),
            double(a.b.ctransform[(3 * c + 2) * S + body])};
}
template <typename R>
__device__ __forceinline__ double half_g(const NP<R>& a, int body, int k) {
  return double(a.b.half[k * a.b.stride + body]);
}

// transformToAxis, colliders.go:762-770
__device__ __forceinline__ double transform_to_axis(const Col& c, const D3& a) {
  return c.h[0] * dabs(dot(a, axis(c.T, 0))) + c.h[1] * dabs(dot(a, axis(c.T, 1))) +
         c.h[2] * dabs(dot(a, axis(c.T, 2)));
}

// CollisionSphere.CheckAgainstHalfSpace, colliders.go:180-207
template <typename R, bool EMIT>
__device__ __forceinline__ int sphere_half_space(const NP<R>& a, const Col& s, int si, int pk, const D3& pn, double po,
                                                 int64_t slot) {
  D3 positionAxis = axis(s.T, 3);
  double r = s.h[0];
  double distance = dot(pn, positionAxis) - r;
  if ((distance <= po) == false) return 0;
  if (EMIT) {
    D3 p = add(mul(pn, distance + r * -1.0), positionAxis);
    put_contact(a, slot, si, -1, -pk - 1, p, pn, -distance);
  }
  return 1;
}

// CollisionCube.CheckAgainstHalfSpace, colliders.go:308-366, with
// intersectCubeAndHalfSpace (:750-760) as the early-out.
template <typename R, bool EMIT>
__device__ __forceinline__ int cube_half_space(const NP<R>& a, const Col& c, int ci, int pk, const D3& pn, double po,
                                               int64_t slot) {
  double projectedRadius = transform_to_axis(c, pn);
  double cubeDistance = dot(pn, axis(c.T, 3)) - projectedRadius;
  if (!(cubeDistance <= po)) return 0;
  int k = 0;
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    // mults[v] = (+-1, +-1, +-1): x flips on odd v, y on v&2, z on v&4
    D3 vert{(v & 1) ? -c.h[0] : c.h[0], (v & 2) ? -c.h[1] : c.h[1], (v & 4) ? -c.h[2] : c.h[2]};
    D3 vertexPos = m34v(c.T, vert);
    double vertexDistance = dot(vertexPos, pn);
    if (vertexDistance <= po) {
      if (EMIT) {
        D3 p = add(mul(pn, vertexDistance - po), vertexPos);
        put_contact(a, slot + k, ci, -1, -pk - 1, p, pn, po - vertexDistance);
      }
      ++k;
    }
  }
  return k;
}

// CollisionSphere.CheckAgainstSphere, colliders.go:216-254
template <typename R, bool EMIT>
__device__ __forceinline__ int sphere_sphere(const NP<R>& a, const Col& s1, int i1, const Col& s2, int i2, int64_t slot) {
  D3 p1 = axis(s1.T, 3), p2 = axis(s2.T, 3);
  D3 midline = sub(p1, p2);
  double size = mag(midline);
  if (size <= 0.0 || size >= s1.h[0] + s2.h[0]) return 0;
  if (EMIT) {
    D3 p = add(mul(midline, 0.5), p1);
    D3 n = mul(midline, 1.0 / size);
    put_contact(a, slot, i1, i2, i2, p, n, s1.h[0] + s2.h[0] - size);
  }
  return 1;
}

// CollisionCube.CheckAgainstSphere, colliders.go:369-441
template <typename R, bool EMIT>
__device__ __forceinline__ int cube_sphere(const NP<R>& a, const Col& c, int ci, const Col& s, int si, int64_t slot) {
  const double r = s.h[0];
  D3 position = axis(s.T, 3);
  D3 rc = m34_tinv(c.T, position);
  if (dabs(rc.x) - r > c.h[0] || dabs(rc.y) - r > c.h[1] || dabs(rc.z) - r > c.h[2]) return 0;
  double cp[3];
  const double rcv[3] = {rc.x, rc.y, rc.z};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double dist = rcv[k];
    if (dist > c.h[k]) {
      dist = c.h[k];
    } else if (dist < -c.h[k]) {
      dist = -c.h[k];
    }
    cp[k] = dist;
  }
  D3 closest{cp[0], cp[1], cp[2]};
  double dist = sqmag(sub(closest, rc));
  if (dist > r * r) return 0;
  if (EMIT) {
    D3 cw = m34v(c.T, closest);
    D3 n = sub(cw, position);
    if (real_equal(mag(n), 0.0)) {
      const int64_t S = a.b.stride;
      n = D3{double(a.b.vel[si]), double(a.b.vel[S + si]), double(a.b.vel[2 * S + si])};
    }
    n = normalize(n);
    double pen = r;
    if (!real_equal(dist, 0.0)) {
      pen -= dsqrt(dist);
    } else {
      pen = 0.0;
    }
    put_contact(a, slot, ci, si, si, cw, n, pen);
  }
  return 1;
}

// tryAxis, colliders.go:458-477 with penetrationOnAxis (:445-456)
__device__ __forceinline__ bool try_axis(const Col& one, const Col& two, D3 ax, const D3& toCenter, int index,
                                         double& smallest, int& best) {
  if (sqmag(ax) < Lim<double>::eps) return true;
  ax = normalize(ax);
  double oneProject = transform_to_axis(one, ax);
  double twoProject = transform_to_axis(two, ax);
  double distance = dabs(dot(toCenter, ax));
  double penetration = oneProject + twoProject - distance;
  if (penetration < 0) return false;
  if (penetration < smallest) {
    smallest = penetration;
    best = index;
  }
  return true;
}

// fillPointFaceBoxBox, colliders.go:481-517 (i1 = one's body index)
template <typename R>
__device__ __forceinline__ void point_face(const NP<R>& a, const Col& one, int i1, const Col& two,
                                           const D3& toCenter, int best, D3& n, D3& p) {
  n = axis_g(a, i1, best);
  if (dot(n, toCenter) > 0) n = mul(n, -1.0);
  D3 v{two.h[0], two.h[1], two.h[2]};
  if (dot(axis(two.T, 0), n) < 0) v.x = -v.x;
  if (dot(axis(two.T, 1), n) < 0) v.y = -v.y;
  if (dot(axis(two.T, 2), n) < 0) v.z = -v.z;
  p = m34v(two.T, v);
}

// contactPoint, colliders.go:519-573
__device__ __forceinline__ D3 contact_point(const D3& pOne, const D3& dOne, double oneSize, const D3& pTwo,
                                            const D3& dTwo, double twoSize, bool useOne) {
  double smOne = sqmag(dOne);
  double smTwo = sqmag(dTwo);
  double dpOneTwo = dot(dTwo, dOne);
  D3 toSt = sub(pOne, pTwo);
  double dpStaOne = dot(dOne, toSt);
  double dpStaTwo = dot(dTwo, toSt);
  double denom = smOne * smTwo - dpOneTwo * dpOneTwo;
  if (dabs(denom) < Lim<double>::eps) return useOne ? pOne : pTwo;
  double mua = (dpOneTwo * dpStaTwo - smTwo * dpStaOne) / denom;
  double mub = (smOne * dpStaTwo - dpOneTwo * dpStaOne) / denom;
  if (mua > oneSize || mua < -oneSize || mub > twoSize || mub < -twoSize) return useOne ? pOne : pTwo;
  D3 cOne = add(mul(dOne, mua), pOne);
  D3 cTwo = add(mul(dTwo, mub), pTwo);
  cOne = mul(cOne, 0.5);
  cTwo = mul(cTwo, 0.5);
  return add(cOne, cTwo);
}

// CollisionCube.CheckAgainstCube, colliders.go:576-710
template <typename R, bool EMIT>
__device__ __forceinline__ int cube_cube(const NP<R>& a, const Col& one, int i1, const Col& two, int i2, int64_t slot) {
  D3 toCenter = sub(axis(two.T, 3), axis(one.T, 3));
  double pen = Lim<double>::max_value;
  int best = 0xffffff;
  for (int i = 0; i <= 2; ++i)
    if (!try_axis(one, two, axis(one.T, i), toCenter, i, pen, best)) return 0;
  for (int i = 0; i <= 2; ++i)
    if (!try_axis(one, two, axis(two.T, i), toCenter, i + 3, pen, best)) return 0;
  const int bestSingleAxis = best;
  for (int i = 0; i <= 2; ++i)
    for (int k = 0; k <= 2; ++k)
      if (!try_axis(one, two, cross(axis(one.T, i), axis(two.T, k)), toCenter, i * 3 + 6 + k, pen, best)) return 0;
  if (!EMIT) return 1;
  D3 n, p;
  if (best < 3) {
    point_face(a, one, i1, two, toCenter, best, n, p);
    put_contact(a, slot, i1, i2, i2, p, n, pen);
  } else if (best < 6) {
    point_face(a, two, i2, one, mul(toCenter, -1.0), best - 3, n, p);
    put_contact(a, slot, i2, i1, i1, p, n, pen);
  } else {
    best -= 6;
    const int oneAxisIndex = best / 3;
    const int twoAxisIndex = best % 3;
    D3 oneAxis = axis_g(a, i1, oneAxisIndex);
    D3 twoAxis = axis_g(a, i2, twoAxisIndex);
    D3 ax = normalize(cross(oneAxis, twoAxis));
    if (dot(ax, toCenter) > 0) ax = mul(ax, -1.0);
    double p1[3] = {one.h[0], one.h[1], one.h[2]};
    double p2[3] = {two.h[0], two.h[1], two.h[2]};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (i == oneAxisIndex) {
        p1[i] = 0;
      } else if (dot(axis(one.T, i), ax) > 0) {
        p1[i] = -p1[i];
      }
      if (i == twoAxisIndex) {
        p2[i] = 0;
      } else if (dot(axis(two.T, i), ax) < 0) {
        p2[i] = -p2[i];
      }
    }
    D3 ptOnOneEdge = m34v(one.T, D3{p1[0], p1[1], p1[2]});
    D3 ptOnTwoEdge = m34v(two.T, D3{p2[0], p2[1], p2[2]});
    const bool useOne = bestSingleAxis > 2;
    // an index past 2 only arises from a NaN state; GetAxis clamps it to 3
    const double oneSize = oneAxisIndex < 3 ? half_g(a, i1, oneAxisIndex) : 0.0;
    const double twoSize = twoAxisIndex < 3 ? half_g(a, i2, twoAxisIndex) : 0.0;
    D3 cv = contact_point(ptOnOneEdge, oneAxis, oneSize, ptOnTwoEdge, twoAxis, twoSize, useOne);
    put_contact(a, slot, i1, i2, i2, cv, ax, pen);
  }
  return 1;
}

// Conservative rejection for body pairs.  For orthonormal box axes a_k,
// max_k |t.a_k| >= |t|/sqrt(3), while the projections of the two shapes on
// a_k are bounded by their bounding radii; so |t|^2 > 3 (rA+rB)^2 makes a
// face axis of A separate (tryAxis returns false) and a sphere centre
// farther than rA + rB from a box centre fails the closest-point test.
// The factors carry a 1e-3 margin for rounding and for the 1e-7 slack the
// quaternion normalisation leaves in the axes.
template <typename R>
__device__ __forceinline__ bool far_apart(const NP<R>& a, int i, int j, int si, int sj) {
  const int64_t S = a.b.stride;
  double dx = double(a.b.ctransform[9 * S + j]) - double(a.b.ctransform[9 * S + i]);
  double dy = double(a.b.ctransform[10 * S + j]) - double(a.b.ctransform[10 * S + i]);
  double dz = double(a.b.ctransform[11 * S + j]) - double(a.b.ctransform[11 * S + i]);
  double d2 = dx * dx + dy * dy + dz * dz;
  double rr = a.brad[i] + a.brad[j];
  double k = (si == SHAPE_CUBE && sj == SHAPE_CUBE) ? 3.003 : 1.001;
  return d2 > k * rr * rr;
}

// CheckForCollisions, colliders.go:720-747, including the plane delegations
// (:116-125) and the sphere-to-cube delegation (:210-213).
template <typename R, bool EMIT>
__device__ __forceinline__ int pair_eval(const NP<R>& a, int one, int two, int64_t slot) {
  if (one < 0 && two < 0) return 0;
  if (one < 0 || two < 0) {
    const int bi = one < 0 ? two : one;
    const int pk = one < 0 ? -one - 1 : -two - 1;
    const int64_t PS = a.pl.stride;
    D3 pn{double(a.pl.normal[pk]), double(a.pl.normal[PS + pk]), double(a.pl.normal[2 * PS + pk])};
    double po = double(a.pl.offset[pk]);
    Col c;
    load_col(a.b, bi, c);
    if (c.shape == SHAPE_SPHERE) return sphere_half_space<R, EMIT>(a, c, bi, pk, pn, po, slot);
    return cube_half_space<R, EMIT>(a, c, bi, pk, pn, po, slot);
  }
  const int s1 = a.b.shape[one], s2 = a.b.shape[two];
  if (!(s1 == SHAPE_SPHERE && s2 == SHAPE_SPHERE) && far_apart(a, one, two, s1, s2)) return 0;
  Col c1, c2;
  load_col(a.b, one, c1);
  load_col(a.b, two, c2);
  if (s2 == SHAPE_SPHERE) {
    if (s1 == SHAPE_SPHERE) return sphere_sphere<R, EMIT>(a, c1, one, c2, two, slot);
    return cube_sphere<R, EMIT>(a, c1, one, c2, two, slot);
  }
  if (s1 == SHAPE_SPHERE) return cube_sphere<R, EMIT>(a, c2, two, c1, one, slot);
  return cube_cube<R, EMIT>(a, c1, one, c2, two, slot);
}

// Entry q of world w's explicit pair list -> (one, two).
__device__ __forceinline__ void pair_of(const PairSpace& ps, int w, int q, int& one, int& two) {
  const int p = ps.list_off[w] + q;
  one = ps.list_one[p];
  two = ps.list_two[p];
}

// A list that a block collects in LDS and appends to a global one at its end
// with a single atomic: the atomics of a grid on one counter come one after
// another.  What does not fit in LDS is appended at once.  Entries past the
// capacity are counted and dropped.
template <int N>
struct BlockList {
  uint32_t item[N];
  int n, base;

  __device__ __forceinline__ void clear() {
    if (threadIdx.x == 0) n = 0;
    __syncthreads();
  }
  __device__ __forceinline__ void put(uint32_t v, uint32_t* list, int32_t* counter, int64_t cap) {
    const int at = atomicAdd(&n, 1);
    if (at < N) {
      item[at] = v;
    } else {
      const int64_t g = atomicAdd(counter, 1);
      if (g < cap) list[g] = v;
    }
  }
  // One entry per set bit of every lane of a wave (first + k * step for bit k),
  // reserved together; all lanes call it.
  __device__ __forceinline__ void put_bits(uint32_t bits, uint32_t first, uint32_t step, uint32_t* list,
                                           int32_t* counter, int64_t cap) {
    const int lane = threadIdx.x & 63;
    const int mine = __popc(bits), incl = wave_incl_scan_i32(mine), total = __shfl(incl, 63, 64);
    if (total == 0) return;
    int at = 0;
    if (lane == 63) at = atomicAdd(&n, total);
    at = __shfl(at, 63, 64);
    const int fit = min(max(N - at, 0), total);  // the first of them go to LDS
    int64_t g = 0;
    if (fit < total) {
      int b = 0;
      if (lane == 63) b = atomicAdd(counter, total - fit);
      g = __shfl(b, 63, 64);
    }
    for (int k = incl - mine; bits; bits &= bits - 1u, ++k) {
      const uint32_t v = first + uint32_t(__ffs(bits) - 1) * step;
      if (k < fit)
        item[at + k] = v;
      else if (g + (k - fit) < cap)
        list[g + (k - fit)] = v;
    }
  }
  __device__ __forceinline__ void flush(uint32_t* list, int32_t* counter, int64_t cap) {
    __syncthreads();
    const int m = min(n, N);
    if (threadIdx.x == 0 && m > 0) base = atomicAdd(counter, m);
    __syncthreads();
    for (int k = threadIdx.x; k < m; k += blockDim.x)
      if (base + int64_t(k) < cap) list[base + int64_t(k)] = item[k];
  }
};

// Orders a wave's LDS writes before its later reads, and the other way.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// all-pairs space
// ---------------------------------------------------------------------------
// Cull: each wave takes `per` consecutive tasks (world w, column tile c, rows
// r0 .. r0+15).  Lane l owns column 64c + l for the whole task: a plane, or
// body j whose centre, bounding radius and shape stay in registers; the 16
// row bodies are put in LDS once and read as broadcasts.  Each tile is
// cleared here; the body pairs with j > r that pass the conservative bound
// (see far_apart) go to the candidate list.
//
// The 16 tests of a lane run in FP32 on positions relative to the first row's
// body, with a margin that covers the rounding: for s = sqrt(kf) rr and an
// error e of the distance, (s + e)^2 <= 1.004 s^2 + 251 e^2, and with the
// coordinates' and the difference's rounding e <= 2^-23 (|a| + |b|) in the
// 1-norms of a and b, so 251 e^2 is below 4e-12 (|a| + |b|)^2.  What they leave (a NaN or an infinity passes) is
// tested again as far_apart does it, once per pair that is left instead of once
// per pair: the list is the same.  4096 worlds of 8 to 256 cubes take
// 97 us (183 with every ordered pair tested in FP64, rows shuffled from lane to
// lane), bound by the tests' instructions and the clearing of 1.4 million tiles.
// Tasks per wave: one while every task's wave fits the chip at once (a launch is
// then one task long: 22 to 5 us for one world of 64 cubes), up to 16 beyond, so
// that there are few blocks and with them few reservations.
constexpr int kCullWaves = 8192, kCullPer = 16;
constexpr int kCullList = 4096;  // every pair of four tasks

struct CullRow {
  float x, y, z, r;    // relative to the first row's body
  double dx, dy, dz, dr;
  float norm;          // |x| + |y| + |z|
  int shape;
};

template <typename R>
__global__ void __launch_bounds__(256) k_np_cull(NP<R> a, int per) {
  __shared__ CullRow s_row[4][kRowBlock];
  __shared__ BlockList<kCullList> s_list;
  s_list.clear();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int task0 = __builtin_amdgcn_readfirstlane((blockIdx.x * 4 + wv) * per);
  CullRow* row = s_row[wv];
  for (int task = task0; task < min(task0 + per, a.ps.n_tasks); ++task) {
    const int w = a.ps.task_world[task];
    const int b0 = a.ps.body_off[w], n = a.ps.body_off[w + 1] - b0;
    const int np = a.ps.plane_off[w + 1] - a.ps.plane_off[w];
    const int nch = (np + n + 63) >> 6;
    const int k = task - a.ps.world_task0[w];
    const int c = k % nch;
    const int r0 = (k / nch) * kRowBlock;
    const int t0 = a.ps.world_tile0[w];
    const int rows = min(n - r0, kRowBlock);
    if (lane < rows) {
      const int t = t0 + (r0 + lane) * nch + c;
      a.tile_cnt[t] = 0;
      a.tile_mask[t] = 0ull;
    }
    if (64 * c + 63 - np <= r0) continue;  // no column with j > r
    const int j = 64 * c + lane - np;
    const bool is_body = j >= 0 && j < n;
    const int64_t S = a.b.stride;
    double tj[3] = {0, 0, 0}, rj = 0;
    int sj = 0;
    if (is_body) {
      const int g = b0 + j;
      tj[0] = double(a.b.ctransform[9 * S + g]);
      tj[1] = double(a.b.ctransform[10 * S + g]);
      tj[2] = double(a.b.ctransform[11 * S + g]);
      rj = a.brad[g];
      sj = a.b.shape[g];
    }
    double ti[3] = {0, 0, 0}, ri = 0;
    int si = 0;
    if (lane < rows) {  // lane k holds row r0 + k
      const int g = b0 + r0 + lane;
      ti[0] = double(a.b.ctransform[9 * S + g]);
      ti[1] = double(a.b.ctransform[10 * S + g]);
      ti[2] = double(a.b.ctransform[11 * S + g]);
      ri = a.brad[g];
      si = a.b.shape[g];
    }
    const double ox = __shfl(ti[0], 0, 64), oy = __shfl(ti[1], 0, 64), oz = __shfl(ti[2], 0, 64);
    const float xj = float(tj[0] - ox), yj = float(tj[1] - oy), zj = float(tj[2] - oz), fj = float(rj);
    const float normj = fabsf(xj) + fabsf(yj) + fabsf(zj);
    wave_lds_fence();  // the last task's rows have been read
    if (lane < kRowBlock) {
      CullRow v;
      v.x = float(ti[0] - ox), v.y = float(ti[1] - oy), v.z = float(ti[2] - oz), v.r = float(ri);
      v.dx = ti[0], v.dy = ti[1], v.dz = ti[2], v.dr = ri;
      v.norm = fabsf(v.x) + fabsf(v.y) + fabsf(v.z);
      v.shape = si;
      row[lane] = v;
    }
    wave_lds_fence();
    // kf with its margin, for a row that is a cube and one that is not
    // (two spheres are always a candidate)
    const bool cj = sj == SHAPE_CUBE;
    const float kc = (cj ? 3.003f : 1.001f) * 1.0042f;
    const float ks = sj == SHAPE_SPHERE ? INFINITY : 1.001f * 1.0042f;
    uint32_t m = 0;
#pragma unroll
    for (int k2 = 0; k2 < kRowBlock; ++k2) {
      const CullRow& v = row[k2];
      const float dx = xj - v.x, dy = yj - v.y, dz = zj - v.z;
      const float d2 = dx * dx + dy * dy + dz * dz;
      const float rr = v.r + fj, nn = v.norm + normj;
      const float lim = (v.shape == SHAPE_CUBE ? kc : (v.shape == SHAPE_SPHERE ? ks : 1.001f * 1.0042f)) * (rr * rr);
      if (!(d2 > lim + 1e-10f * (nn * nn))) m |= 1u << k2;
    }
    // rows below the column's body only
    const int up = min(max(j - r0, 0), rows);
    m = is_body ? m & ((1u << up) - 1u) : 0u;
    uint32_t keep = 0;
    for (; m; m &= m - 1u) {
      const int k2 = __ffs(m) - 1;
      const CullRow& v = row[k2];
      const double dx = tj[0] - v.dx, dy = tj[1] - v.dy, dz = tj[2] - v.dz;
      const double d2 = dx * dx + dy * dy + dz * dz;
      const double rr = v.dr + rj;
      const bool spheres = v.shape == SHAPE_SPHERE && sj == SHAPE_SPHERE;
      const double kf = (v.shape == SHAPE_CUBE && cj) ? 3.003 : 1.001;
      if (spheres || !(d2 > kf * rr * rr)) keep |= 1u << k2;
    }
    s_list.put_bits(keep, uint32_t(t0 + r0 * nch + c) * 64u + uint32_t(lane), uint32_t(nch) * 64u, a.cand, a.n_pairs,
                    a.cand_cap);
  }
  s_list.flush(a.cand, a.n_pairs, a.cand_cap);
}

// Eval: the first workgroups take a body per thread, against its world's
// planes, the others a candidate pair per thread: the reference's test
// (contact count only); hits add to their tile's total and mask (integer
// atomics: the sums do not depend on the order) and join the hit list.  Too
// many candidates (in both orders, the planes' pairs among them) for the list
// raise the overflow flags (the step reports a capacity error).  The planes
// apart from the pairs: a wave that holds both runs both tests.
// 4096 worlds of 8 to 256 cubes take 88 us (166 with both orders tested and the
// planes among the pairs, 110 with a reservation per 256 bodies or pairs), bound by the gathers of two bodies per thread and the
// longest axis search of each wave.
constexpr int kEvalList = 2048;
template <typename R>
__global__ void __launch_bounds__(256) k_np_eval(NP<R> a, int plane_blocks) {
  __shared__ BlockList<kEvalList> s_list;
  const int64_t np2 = a.n_pairs[0], nc = 2 * np2 + a.plane_pairs;
  if (blockIdx.x == 0 && threadIdx.x == 0) a.n_cand[0] = int32_t(min(nc, int64_t(INT32_MAX)));
  if (nc > a.cand_cap) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      a.overflow[0] = 1;
      a.overflow[1] = 1;
    }
    return;  // uniform over the grid
  }
  auto hit = [&](int t, int l, int cnt) {
    atomicAdd(&a.tile_cnt[t], cnt);
    atomicOr((unsigned long long*)&a.tile_mask[t], 1ull << l);
  };
  const int64_t hcap = min(a.c.cap, int64_t(INT32_MAX));
  s_list.clear();
  if (int(blockIdx.x) < plane_blocks) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < a.b.n; i += plane_blocks * 256) {
      const int w = a.body_world[i];
      const int b0 = a.ps.body_off[w], n = a.ps.body_off[w + 1] - b0;
      const int p0 = a.ps.plane_off[w], np = a.ps.plane_off[w + 1] - p0;
      const int nch = (np + n + 63) >> 6, t0 = a.ps.world_tile0[w];
      for (int k = 0; k < np; ++k) {
        const int cnt = pair_eval<R, false>(a, i, -(p0 + k) - 1, 0);
        if (cnt <= 0) continue;
        const int t = t0 + (i - b0) * nch + (k >> 6), l = k & 63;
        hit(t, l, cnt);
        s_list.put(uint32_t(t) * 64u + uint32_t(l), a.hits, a.n_hits, hcap);
      }
    }
    s_list.flush(a.hits, a.n_hits, hcap);
    return;
  }
  const int64_t stride = int64_t(gridDim.x - plane_blocks) * blockDim.x;
  for (int64_t e0 = int64_t(blockIdx.x - plane_blocks) * blockDim.x; e0 < np2; e0 += stride) {
    const int64_t e = e0 + threadIdx.x;
    if (e >= np2) continue;
    const uint32_t code = a.cand[e];
    const int t = int(code >> 6), l = int(code & 63u);
    const int w = a.ps.tile_world[t];
    const int b0 = a.ps.body_off[w], n = a.ps.body_off[w + 1] - b0;
    const int np = a.ps.plane_off[w + 1] - a.ps.plane_off[w];
    const int nch = (np + n + 63) >> 6, t0 = a.ps.world_tile0[w];
    const int k = t - t0;
    const int r = k / nch, c = k - r * nch;
    const int j = 64 * c + l - np;
    const int cnt = pair_eval<R, false>(a, b0 + r, b0 + j, 0);  // one contact or none
    if (cnt <= 0) continue;
    const int tb = t0 + j * nch + ((np + r) >> 6), lb = (np + r) & 63;
    hit(t, l, cnt);
    hit(tb, lb, cnt);
    s_list.put(code, a.hits, a.n_hits, hcap);
    s_list.put(uint32_t(tb) * 64u + uint32_t(lb), a.hits, a.n_hits, hcap);
  }
  s_list.flush(a.hits, a.n_hits, hcap);
}

// Emit: one thread per hit pair.  Its first contact goes to world offset +
// tile offset + the contacts of the tile's earlier hit pairs: one for a body
// pair (a body pair that hit holds exactly one contact), a recount for a
// plane column (up to 8 cube vertices).
template <typename R>
__global__ void __launch_bounds__(256) k_np_emit_hits(NP<R> a) {
  if (a.overflow[0] != 0) return;
  const int H = min(a.n_hits[0], int(min(a.c.cap, int64_t(INT32_MAX))));
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < H; e += gridDim.x * blockDim.x) {
    const uint32_t code = a.hits[e];
    const int t = int(code >> 6), lane = int(code & 63u);
    const int w = a.ps.tile_world[t];
    const int b0 = a.ps.body_off[w], n = a.ps.body_off[w + 1] - b0;
    const int p0 = a.ps.plane_off[w], np = a.ps.plane_off[w + 1] - p0;
    const int nch = (np + n + 63) >> 6;
    const int k = t - a.ps.world_tile0[w];
    const int r = k / nch, c = k - r * nch;
    const int i = b0 + r;
    const uint64_t below = a.tile_mask[t] & ((1ull << lane) - 1ull);
    // lanes of this tile that are plane columns
    const int np_here = min(max(np - 64 * c, 0), 64);
    const uint64_t plane_lanes = np_here >= 64 ? ~0ull : ((1ull << np_here) - 1ull);
    int64_t prefix = __popcll(below & ~plane_lanes);
    for (uint64_t pb = below & plane_lanes; pb; pb &= pb - 1ull) {
      const int l = __ffsll((unsigned long long)pb) - 1;
      prefix += pair_eval<R, false>(a, i, -(p0 + 64 * c + l) - 1, 0);
    }
    const int64_t slot = a.world_coff[w] + a.tile_off[t] + prefix;
    const int col = 64 * c + lane;
    if (col < np)
      pair_eval<R, true>(a, i, -(p0 + col) - 1, slot);
    else
      pair_eval<R, true>(a, i, b0 + (col - np), slot);
  }
}

template <typename R>
__global__ void __launch_bounds__(256) k_np_count(NP<R> a) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= a.ps.n_tiles) return;
  const int w = a.ps.tile_world[t];
  const int q = (t - a.ps.world_tile0[w]) * 64 + lane;
  int cnt = 0;
  if (q < a.ps.world_q[w]) {
    int one, two;
    pair_of(a.ps, w, q, one, two);
    cnt = pair_eval<R, false>(a, one, two, 0);
    if (a.ps.list_cnt) a.ps.list_cnt[a.ps.list_off[w] + q] = cnt;
  }
  const uint64_t m = __ballot(cnt > 0);
  const int tot = wave_sum_i32(cnt);
  if (lane == 0) {
    a.tile_cnt[t] = tot;
    a.tile_mask[t] = m;
  }
}

// The 16-wave tile scan is launched above this many tiles in one world, or
// from a quarter of a thousand on where every world can have a CU: one wave
// takes 64 tiles per dependent step, 25 us for the 4000 of 40000 listed bodies
// where 16 waves take 5 us; with more worlds than CUs the chip is full
// either way and 16 waves per world would mostly wait.
constexpr int kWideScanTiles = 4096;
constexpr int kWideScanFew = 256;  // tiles, and worlds

// The totals over all worlds, by one thread: the sum, and the flags when it
// exceeds the capacity.
template <typename R>
__device__ __forceinline__ void put_total(const NP<R>& a, int64_t total) {
  a.total[0] = total;
  if (total > a.c.cap) {
    a.overflow[0] = 1;  // this narrowphase (read by emit and the resolver)
    a.overflow[1] = 1;  // sticky until the host clears it
  }
}

// With one world its tile scan is all there is to scan.
template <typename R>
__device__ __forceinline__ void put_world(const NP<R>& a, int w, int cnt) {
  a.world_cnt[w] = cnt;
  if (a.n_worlds == 1) {
    a.world_coff[0] = 0;
    put_total(a, cnt);
  }
}

template <typename R>
__global__ void __launch_bounds__(64) k_np_scan_tiles(NP<R> a) {
  const int w = blockIdx.x;
  const int lane = threadIdx.x;
  const int t0 = a.ps.world_tile0[w], nt = a.ps.world_tile0[w + 1] - t0;
  int carry = 0;
  for (int base = 0; base < nt; base += 64) {
    const int k = base + lane;
    const int v = k < nt ? a.tile_cnt[t0 + k] : 0;
    const int inc = wave_incl_scan_i32(v);
    if (k < nt) a.tile_off[t0 + k] = carry + inc - v;
    carry += __shfl(inc, 63, 64);
  }
  if (lane == 0) put_world(a, w, carry);
}

// The same scan for worlds of many tiles (thousands of bodies): 16 waves,
// each thread summing kScanPer consecutive tiles, take 8,192 tiles per
// pass, so the serial carry chain is 128x shorter than the one-wave scan's.
// Integer prefix sums, so the offsets equal the one-wave scan's.
constexpr int kScanPer = 8;
template <typename R>
__global__ void __launch_bounds__(1024) k_np_scan_tiles_wide(NP<R> a) {
  __shared__ int32_t wsum[16];
  __shared__ int32_t s_carry;
  const int w = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int t0 = a.ps.world_tile0[w], nt = a.ps.world_tile0[w + 1] - t0;
  if (tid == 0) s_carry = 0;
  __syncthreads();
  for (int base = 0; base < nt; base += 1024 * kScanPer) {
    const int k0 = base + kScanPer * tid;
    int v[kScanPer];
    int sum = 0;
#pragma unroll
    for (int j = 0; j < kScanPer; ++j) {
      v[j] = k0 + j < nt ? a.tile_cnt[t0 + k0 + j] : 0;
      sum += v[j];
    }
    const int inc = wave_incl_scan_i32(sum);
    if (lane == 63) wsum[wv] = inc;
    __syncthreads();
    int before = 0;
    for (int u = 0; u < wv; ++u) before += wsum[u];
    const int carry = s_carry;
    int run = carry + before + inc - sum;
#pragma unroll
    for (int j = 0; j < kScanPer; ++j) {
      if (k0 + j < nt) a.tile_off[t0 + k0 + j] = run;
      run += v[j];
    }
    __syncthreads();
    if (tid == 1023) s_carry = carry + before + inc;
    __syncthreads();
  }
  if (tid == 0) put_world(a, w, s_carry);
}

template <typename R>
__global__ void __launch_bounds__(1024) k_np_scan_worlds(NP<R> a) {
  __shared__ int64_t wsum[16];
  __shared__ int64_t s_carry;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  if (tid == 0) s_carry = 0;
  __syncthreads();
  for (int base = 0; base < a.n_worlds; base += 1024) {
    const int k = base + tid;
    const int64_t v = k < a.n_worlds ? int64_t(a.world_cnt[k]) : 0;
    const int64_t inc = wave_incl_scan_i64(v);
    if (lane == 63) wsum[wv] = inc;
    __syncthreads();
    int64_t before = 0;
    for (int u = 0; u < wv; ++u) before += wsum[u];
    const int64_t carry = s_carry;
    if (k < a.n_worlds) a.world_coff[k] = carry + before + inc - v;
    __syncthreads();
    if (tid == 1023) s_carry = carry + before + inc;
    __syncthreads();
  }
  if (tid == 0) put_total(a, s_carry);
}

template <typename R>
__global__ void __launch_bounds__(256) k_np_emit(NP<R> a) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= a.ps.n_tiles) return;
  const uint64_t m = a.tile_mask[t];
  if (m == 0) return;
  const int w = a.ps.tile_world[t];
  const int q = (t - a.ps.world_tile0[w]) * 64 + lane;
  const bool hit = (m >> lane) & 1ull;
  int one = 0, two = 0, cnt = 0;
  if (hit) {
    pair_of(a.ps, w, q, one, two);
    // a body pair that hit holds exactly one contact; only a half-space
    // check can hold several (up to 8 cube vertices)
    cnt = (one < 0 || two < 0) ? pair_eval<R, false>(a, one, two, 0) : 1;
  }
  const int inc = wave_incl_scan_i32(cnt);
  const int64_t slot = a.world_coff[w] + a.tile_off[t] + (inc - cnt);
  if (hit) pair_eval<R, true>(a, one, two, slot);
}

template <typename R>
hipError_t launch_narrowphase(const NarrowLaunch<R>& L, hipStream_t st, hipEvent_t* ev) {
  NP<R> a;
  a.b = L.b;
  a.pl = L.pl;
  a.ps = L.ps;
  a.c = L.c;
  a.brad = L.brad;
  a.tile_cnt = L.tile_cnt;
  a.tile_mask = L.tile_mask;
  a.tile_off = L.tile_off;
  a.world_cnt = L.world_cnt;
  a.world_coff = L.world_coff;
  a.total = L.total;
  a.overflow = L.overflow;
  a.hits = L.hits;
  a.n_hits = L.n_hits;
  a.cand = L.cand;
  a.n_pairs = L.n_pairs;
  a.n_cand = L.n_cand;
  a.cand_cap = L.cand_cap;
  a.plane_pairs = L.plane_pairs;
  a.body_world = L.body_world;
  a.max_planes = L.max_planes;
  a.n_worlds = L.n_worlds;
  a.mat = L.mat;
  if (a.n_worlds <= 0) return hipSuccess;
  if (a.c.fric && (!a.c.rest || !a.mat.body_fric || !a.mat.body_rest || !a.mat.plane_fric || !a.mat.plane_rest))
    return hipErrorInvalidValue;
  const bool list = a.ps.list_one != nullptr;
  if (!list && (!a.hits || !a.n_hits || !a.cand || !a.n_cand || !a.n_pairs || !a.body_world)) return hipErrorInvalidValue;
  // ev (optional): recorded before the count, after it, after the scans
  // and after the emit, for per-kernel timing on this stream.
  const int nb = (a.ps.n_tiles + 3) / 4;
  if (ev) (void)hipEventRecord(ev[0], st);
  if (list) {
    if (nb > 0) k_np_count<R><<<nb, 256, 0, st>>>(a);
  } else {
    if (a.ps.n_tasks > 0) {
      const int per = std::min(std::max(a.ps.n_tasks / kCullWaves, 1), kCullPer);
      k_np_cull<R><<<(a.ps.n_tasks + 4 * per - 1) / (4 * per), 256, 0, st>>>(a, per);
    }
    const int64_t want = std::min<int64_t>(std::max<int64_t>((a.cand_cap + 511) / 512, 1), 8192);
    // the planes' blocks: a body per thread while they are few, four beyond
    const int bodies = (a.b.n + 255) / 256;
    const int planes = a.max_planes > 0 ? (bodies > 512 ? (bodies + 3) / 4 : bodies) : 0;
    k_np_eval<R><<<planes + int(want), 256, 0, st>>>(a, planes);
  }
  if (ev) (void)hipEventRecord(ev[1], st);
  if (a.ps.max_world_tiles > kWideScanTiles || (a.ps.max_world_tiles > kWideScanFew && a.n_worlds <= kWideScanFew))
    k_np_scan_tiles_wide<R><<<a.n_worlds, 1024, 0, st>>>(a);
  else
    k_np_scan_tiles<R><<<a.n_worlds, 64, 0, st>>>(a);
  if (a.n_worlds > 1) k_np_scan_worlds<R><<<1, 1024, 0, st>>>(a);
  if (ev) (void)hipEventRecord(ev[2], st);
  if (list) {
    if (nb > 0) k_np_emit<R><<<nb, 256, 0, st>>>(a);
  } else {
    const int64_t want = (a.c.cap + 255) / 256;
    const int nbe = int(want < 8192 ? (want > 0 ? want : 1) : 8192);
    k_np_emit_hits<R><<<nbe, 256, 0, st>>>(a);
  }
  if (ev) (void)hipEventRecord(ev[3], st);
  return hipGetLastError();
}

template hipError_t launch_narrowphase<double>(const NarrowLaunch<double>&, hipStream_t, hipEvent_t*);
template hipError_t launch_narrowphase<float>(const NarrowLaunch<float>&, hipStream_t, hipEvent_t*);

}  // namespace cbz
