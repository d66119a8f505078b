// cbz_resolve.h — K3: ResolveContacts (contact.go:208-222): the pieces both
// resolver kernels are made of, and the serial one, a wave per world, for the
// worlds that the island kernel (cbz_islands.h) leaves.  Each (precision,
// kind) instantiation is compiled in a translation unit of its own
// (k_resolve_<precision>_<kind>.hip), the launch dispatch is k_resolve.hip.
//
// The reference's resolver is sequential: each iteration picks the worst
// contact (largest penetration, then largest desired velocity change; ties
// go to the lowest index because the scan uses a strict '>'), applies a
// correction to its one or two bodies, and updates every contact that
// shares one of those bodies.  Here a world runs on one wave: the
// argmax is a lane-strided scan plus a butterfly reduction, the correction
// is computed redundantly by all 64 lanes (lane 0 stores it), and the
// update scans the world's contacts lane-parallel, each contact applying
// its matches in the reference's (b, d) order.  Worlds run concurrently.
//
// The selection keys and the body indices of the world's contacts live in
// LDS when the world has at most kKeyCap contacts, otherwise in HBM.
#pragma once
#include <climits>
#include <utility>

#include "cbz_devmath.h"
#include "cbz_launch.h"
#include "cbz_mlp.h"
#include "cbz_types.h"
#include "cbz_wave.h"

namespace cbz {

constexpr int kKeyCap = 1280;

// threads of the island kernel's workgroup (half of them in large launches)
constexpr int kIslThreads = 256;
// a left world's entry: its position phase is done already
constexpr int32_t kLeftVelOnly = 1 << 30;
// RS::left_count: listed worlds, workgroups of the left kernel that are done
// with theirs, worlds that the narrow workgroups leave to whole ones
enum : int { LEFT_WORLDS = 0, LEFT_DONE = 1, LEFT_WIDE = 2, LEFT_COUNTS = 3 };

// Relative energy slack of the surrogate's acceptance test (rounding); the
// absolute slack is 1/2 tol^2 per kilogram: the kinetic energy of the
// residual closing speed the test already accepts.
constexpr double kEnergyRel = 1e-5;

// Compile-time variants of the resolver kernel, so that the plain
// resolver's hot loops carry no code (and no register pressure) of the
// others: KIND_PLAIN (ResolveContacts, or one of its phases), KIND_LABEL
// (also records every impulse's body changes and every resolved
// penetration per contact), KIND_POLISH (the surrogate's velocity polish
// with the plain fallback), KIND_MAT (KIND_PLAIN with per-contact friction
// and restitution, and the frictionless impulse for contacts whose
// friction is 0), KIND_PPOLISH (the surrogate's position polish with the
// plain fallback).
enum : int { KIND_PLAIN = 0, KIND_LABEL = 1, KIND_POLISH = 2, KIND_MAT = 3, KIND_PPOLISH = 4 };

// The position polish's separation bound: a polished world is rejected if a
// contact ends separated by more than kSepFactor times the world's deepest
// penetration at the start (+ the tolerance).  The plain phase stays within
// 1.4 times it (every world of 4096 at six points of a 600-step run; 0.1 %
// of worlds pass 1.0 times).
constexpr double kSepFactor = 2.0;
// A prediction that breaks that bound is tried once more at this fraction of
// its moves before the world is rejected: most over-separations come from
// moves that are too large, and the loop finishes what smaller ones leave.
constexpr double kPosRetryScale = 1.0 / 3.0;

template <typename R>
struct RS {
  Bodies<R> b;
  Contacts<R> c;
  const int32_t* world_cnt;
  const int64_t* world_coff;
  const int32_t* overflow;
  const int32_t* order;
  const int32_t* body_off;
  int64_t* world_iters;  // [2 * n_worlds]: position / velocity iterations
  // [4 * n_worlds] (or null): wall-clock ticks when the world's workgroup
  // started and ended, for a launch without (0, 1) and with (2, 3) RM_VEL
  int64_t* world_time;
  // the worlds the island kernel leaves: entries (world | kLeftVelOnly);
  // left_count: LEFT_*, zero between resolves
  int32_t* left_list;
  int32_t* wide_list;
  int32_t* left_count;
  // the island kernel (cbz_islands.h): per island, at its world's
  // first body + rank: contacts (offset into isl_idx from the world's first
  // slot, count), iterations, log records and where the log starts; per
  // world the class counts and the workgroup size that its islands were made for
  int32_t isl_nb;      // bodies the LDS tables hold
  int32_t isl_wide;    // the worlds are wide_list
  int32_t* isl_off;    // [n_bodies]
  int32_t* isl_cnt;    // [n_bodies]
  int32_t* isl_its;    // [n_bodies]
  int32_t* isl_nrec;   // [n_bodies]
  int64_t* isl_log;    // [n_bodies]
  int32_t* isl_cls;    // [kIslWords * n_worlds]
  int32_t* isl_idx;    // [cap]
  R* isl_save;         // [5][cap] contact velocity, desired velocity change, penetration before the phase
  // [21][n_bodies] position phase: transform and world inverse inertia of
  // sleeping bodies; velocity phase: the state table at a pause (6), with
  // its flags in isl_flag [n_bodies]
  R* isl_snap;
  uint8_t* isl_flag;
  R* log_key;          // [log_cap] the log pool: key, contact, iteration
  int32_t* log_j;
  int32_t* log_it;
  int64_t* log_head;
  int64_t log_cap;
  int32_t n_worlds;
  R dt;
  int64_t iter_mult;
  int64_t iter_fixed;
  int32_t mode;                // RM_* bits
  uint8_t* world_mask;         // velocity phase only where set (null: every world); RM_POLISH: in/out
  R* pos0;                     // [3][n_bodies] body positions at prepare time
  // [cap][kOut] per contact: accumulated velocity-phase changes (0-11) and
  // resolved penetration (12) (null: off)
  float* labels;
  // RM_POLISH: [6][n_bodies] velocity and rotation changes (RM_VEL) or
  // position and orientation changes (RM_POS)
  const float* delta;
  R polish_tol;
  int64_t polish_mult;
};


template <typename R>
__device__ __forceinline__ void add_label(const RS<R>& a, int64_t g, const V3<R> vc[2], const V3<R> rc[2]) {
  float* L = a.labels + g * kOut;
  const V3<R>* v[4] = {&vc[0], &rc[0], &vc[1], &rc[1]};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    L[3 * k + 0] += float(v[k]->x);
    L[3 * k + 1] += float(v[k]->y);
    L[3 * k + 2] += float(v[k]->z);
  }
}

// The position phase's label: the penetration resolved at the contact.
template <typename R>
__device__ __forceinline__ void add_pos_label(const RS<R>& a, int64_t g, R depth) {
  a.labels[g * kOut + kOutPos] += float(depth);
}

template <typename R>
__device__ __forceinline__ V3<R> ld3(const R* a, int64_t s, int64_t i) {
  return V3<R>{a[i], a[s + i], a[2 * s + i]};
}
template <typename R>
__device__ __forceinline__ void st3(R* a, int64_t s, int64_t i, const V3<R>& v) {
  a[i] = v.x;
  a[s + i] = v.y;
  a[2 * s + i] = v.z;
}
template <typename R>
__device__ __forceinline__ void ld9(const R* a, int64_t s, int64_t i, R* o) {
#pragma unroll
  for (int k = 0; k < 9; ++k) o[k] = a[k * s + i];
}

template <typename R>
__device__ __forceinline__ bool awake(const Bodies<R>& b, int i) {
  return (b.flags[i] & F_AWAKE) != 0;
}

// calculateLocalVelocity, contact.go:159-182
template <typename R>
__device__ __forceinline__ V3<R> local_velocity(const Bodies<R>& b, int body, const V3<R>& rel, const R* c2w,
                                                R dt) {
  const int64_t S = b.stride;
  V3<R> velocity = add(cross(ld3(b.rot, S, body), rel), ld3(b.vel, S, body));
  V3<R> cv = m3tv(c2w, velocity);
  V3<R> accv = m3tv(c2w, mul(ld3(b.last_acc, S, body), dt));
  accv.x = R(0);
  return add(cv, accv);
}

// Contact.Restitution and Contact.Friction of contact g: the reference's
// constants (colliders.go:201-202) unless the kernel is KIND_MAT.
template <typename R, int KIND>
__device__ __forceinline__ R restitution_of(const Contacts<R>& c, int64_t g) {
  if constexpr (KIND == KIND_MAT) return c.rest[g];
  return R(kRestitution);
}
template <typename R, int KIND>
__device__ __forceinline__ R friction_of(const Contacts<R>& c, int64_t g) {
  if constexpr (KIND == KIND_MAT) return c.fric[g];
  return R(kFriction);
}

// calculateDesiredDeltaVelocity, contact.go:87-112, with the contact's
// restitution e
template <typename R>
__device__ __forceinline__ R desired_dv(const Bodies<R>& b, int b0, int b1, const V3<R>& n, R cvx, R dt, R e) {
  const int64_t S = b.stride;
  R vfa = R(0);
  if (awake(b, b0)) vfa += dot(mul(ld3(b.last_acc, S, b0), dt), n);
  if (b1 >= 0 && awake(b, b1)) vfa -= dot(mul(ld3(b.last_acc, S, b1), dt), n);
  R restitution = e;
  if (dabs(cvx) < R(0.25)) restitution = R(0);
  return -cvx - restitution * (cvx - vfa);
}

// calculateContactBasis, contact.go:118-156, split in two: the scale
// s = 1/sqrt(...) (the only square root and division), and the frame built
// from the normal and s.  Rebuilding the frame from a stored s gives the
// same bits as the full computation.  Both run in FP64 whatever the storage
// type R (the FP32 variant keeps the basis in FP64; for R = double nothing
// is converted).
template <typename R>
__device__ __forceinline__ double basis_scale(const V3<R>& nr) {
  const V3<double> n{double(nr.x), double(nr.y), double(nr.z)};
  if (dabs(n.x) > dabs(n.y)) return 1.0 / dsqrt(n.z * n.z + n.x * n.x);
  return 1.0 / dsqrt(n.z * n.z + n.y * n.y);
}
template <typename R>
__device__ __forceinline__ void basis_from_scale(const V3<R>& nr, double s, R* m) {
  const V3<double> n{double(nr.x), double(nr.y), double(nr.z)};
  V3<double> ty, tz;
  if (dabs(n.x) > dabs(n.y)) {
    ty = V3<double>{n.z * s, 0.0, n.x * -s};
    tz = V3<double>{n.y * ty.x, n.z * ty.x - n.x * ty.z, -n.y * ty.x};
  } else {
    ty = V3<double>{0.0, -n.z * s, n.y * s};
    tz = V3<double>{n.y * ty.z - n.z * ty.y, -n.x * ty.z, n.x * ty.y};
  }
  // SetComponents(normal, tangentY, tangentZ), math/matrix.go:52-56
  m[0] = nr.x; m[1] = nr.y; m[2] = nr.z;
  m[3] = R(ty.x); m[4] = R(ty.y); m[5] = R(ty.z);
  m[6] = R(tz.x); m[7] = R(tz.y); m[8] = R(tz.z);
}
template <typename R>
__device__ __forceinline__ void contact_basis(const V3<R>& n, R* m) {
  basis_from_scale(n, basis_scale(n), m);
}

// A contact's record (Contacts::rec): 16 reals from one 64-byte (FP32) or
// 128-byte (FP64) aligned address, in 16-byte loads.
template <typename R>
__device__ __forceinline__ void load_rec(const R* q, R (&v)[16]) {
  if constexpr (sizeof(R) == 4) {
    const float4* p = reinterpret_cast<const float4*>(q);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float4 x = p[i];
      v[4 * i] = x.x;
      v[4 * i + 1] = x.y;
      v[4 * i + 2] = x.z;
      v[4 * i + 3] = x.w;
    }
  } else {
    const double2* p = reinterpret_cast<const double2*>(q);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const double2 x = p[i];
      v[2 * i] = x.x;
      v[2 * i + 1] = x.y;
    }
  }
}
// contactToWorld and both relative positions
template <typename R>
__device__ __forceinline__ void rec_frame(const R* q, R (&m)[9], V3<R> (&r)[2]) {
  R v[16];
  load_rec(q, v);
#pragma unroll
  for (int k = 0; k < 9; ++k) m[k] = v[k];
  r[0] = V3<R>{v[9], v[10], v[11]};
  r[1] = V3<R>{v[12], v[13], v[14]};
}
// the normal (contactToWorld's first column) and both relative positions
template <typename R>
__device__ __forceinline__ void rec_normal(const R* q, V3<R>& n, V3<R> (&r)[2]) {
  R v[16];
  load_rec(q, v);
  n = V3<R>{v[0], v[1], v[2]};
  r[0] = V3<R>{v[9], v[10], v[11]};
  r[1] = V3<R>{v[12], v[13], v[14]};
}
template <typename R>
__device__ __forceinline__ void store_rec(R* q, const R (&m)[9], const V3<R>& r0, const V3<R>& r1) {
  const R v[16] = {m[0], m[1], m[2], m[3], m[4], m[5], m[6], m[7], m[8], r0.x, r0.y, r0.z, r1.x, r1.y, r1.z, R(0)};
  if constexpr (sizeof(R) == 4) {
    float4* p = reinterpret_cast<float4*>(q);
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = float4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
  } else {
    double2* p = reinterpret_cast<double2*>(q);
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = double2{v[2 * i], v[2 * i + 1]};
  }
}

// calculateInternals, contact.go:59-85, for contact g.
// With REC, also the contact's record (Contacts::rec).
template <typename R, int KIND, bool REC = false>
__device__ __forceinline__ void prepare_contact(const RS<R>& a, int64_t g) {
  const Bodies<R>& b = a.b;
  const Contacts<R>& c = a.c;
  const int64_t S = b.stride, CS = c.cap;
  int b0 = c.body0[g], b1 = c.body1[g];
  V3<R> n = ld3(c.normal, CS, g);
  if (b0 < 0) {  // contact.go:61-65 (not produced by the narrowphase)
    n = mul(n, R(-1));
    b0 = b1;
    b1 = -1;
    c.body0[g] = b0;
    c.body1[g] = b1;
    st3(c.normal, CS, g, n);
  }
  R m[9];
  contact_basis(n, m);
  const V3<R> p = ld3(c.point, CS, g);
  const V3<R> r0 = sub(p, ld3(b.pos, S, b0));
  V3<R> cv = local_velocity(b, b0, r0, m, a.dt);
  V3<R> r1{R(0), R(0), R(0)};
  if (b1 >= 0) {
    r1 = sub(p, ld3(b.pos, S, b1));
    cv = sub(cv, local_velocity(b, b1, r1, m, a.dt));
  }
  const R ddv = desired_dv(b, b0, b1, n, cv.x, a.dt, restitution_of<R, KIND>(c, g));
#pragma unroll
  for (int k = 0; k < 9; ++k) c.c2w[k * CS + g] = m[k];
  st3(c.rel, CS, g, r0);
  st3(c.rel + 3 * CS, CS, g, r1);
  st3(c.cvel, CS, g, cv);
  c.ddv[g] = ddv;
  if constexpr (REC) store_rec(c.rec + 16 * g, m, r0, r1);
}

// matchAwakeState, contact.go:185-202.  Returns the awake states after the
// call in a0/a1 (lane 0 stores the change).
template <typename R>
__device__ __forceinline__ void match_awake(const RS<R>& a, int k0, int k1, bool& a0, bool& a1, int lane) {
  a0 = awake(a.b, k0);
  a1 = k1 >= 0 ? awake(a.b, k1) : false;
  if (k1 < 0) return;
  if ((a0 || a1) && !(a0 && a1)) {
    const int t = a0 ? k1 : k0;
    if (lane == 0) {  // SetAwake(true), rigidbody.go:183-186
      a.b.flags[t] = uint8_t(a.b.flags[t] | F_AWAKE);
      a.b.motion[t] = R(kSleepEpsilon * 2.0);
    }
    a0 = a1 = true;
  }
}

// CalculateDerivedData (rigidbody.go:268-272) for a sleeping body moved by
// applyPositionChange (contact.go:380-382); IW: its world inverse inertia.
template <typename R>
__device__ __forceinline__ void rederive(const Bodies<R>& b, int i, const V3<R>& pos, Q4<R>& q, int lane, R (&IW)[9]) {
  const int64_t S = b.stride;
  q = q_normalize(q);
  R T[12], IB[9];
  set_as_transform(pos, q, T);
  ld9(b.iit_body, S, i, IB);
  transform_inertia(IB, T, IW);
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < 12; ++k) b.transform[k * S + i] = T[k];
#pragma unroll
    for (int k = 0; k < 9; ++k) b.iit_world[k * S + i] = IW[k];
  }
}

// applyPositionChange, contact.go:286-386
template <typename R>
__device__ __forceinline__ void apply_position_change(const RS<R>& a, const int kb[2], const bool aw[2], const V3<R>& n,
                                      const V3<R> rel[2], R penetration, V3<R> lin[2], V3<R> ang[2], int lane) {
  const Bodies<R>& b = a.b;
  const int64_t S = b.stride;
  const R angularLimit = R(0.2);
  R angI[2] = {R(0), R(0)}, linI[2] = {R(0), R(0)};
  R total = R(0);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    lin[i] = V3<R>{R(0), R(0), R(0)};
    ang[i] = V3<R>{R(0), R(0), R(0)};
    if (kb[i] < 0) continue;
    R iw[9];
    ld9(b.iit_world, S, kb[i], iw);
    V3<R> aiw = cross(rel[i], n);
    aiw = m3v(iw, aiw);
    aiw = cross(aiw, rel[i]);
    angI[i] = dot(aiw, n);
    linI[i] = b.inv_mass[kb[i]];
    total += linI[i] + angI[i];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int bi = kb[i];
    if (bi < 0) continue;
    R sign = R(1);
    if (i != 0) sign = R(-1);
    R angM = sign * penetration * (angI[i] / total);
    R linM = sign * penetration * (linI[i] / total);
    V3<R> projection = add_scaled(rel[i], n, -dot(rel[i], n));
    R maxMagnitude = angularLimit * mag(projection);
    if (angM < -maxMagnitude) {
      R totalMove = angM + linM;
      angM = -maxMagnitude;
      linM = totalMove - angM;
    } else if (angM > maxMagnitude) {
      R totalMove = angM + linM;
      angM = maxMagnitude;
      linM = totalMove - angM;
    }
    if (angM == R(0)) {
      ang[i] = V3<R>{R(0), R(0), R(0)};
    } else {
      V3<R> tad = cross(rel[i], n);
      R iw[9];
      ld9(b.iit_world, S, bi, iw);
      ang[i] = mul(m3v(iw, tad), angM / angI[i]);
    }
    lin[i] = mul(n, linM);
    V3<R> pos = add_scaled(ld3(b.pos, S, bi), n, linM);
    Q4<R> q{b.quat[bi], b.quat[S + bi], b.quat[2 * S + bi], b.quat[3 * S + bi]};
    q = q_add_scaled_vector(q, ang[i], R(1));
    q = q_normalize(q);
    R iwn[9];
    if (!aw[i]) rederive(b, bi, pos, q, lane, iwn);
    if (lane == 0) {
      st3(b.pos, S, bi, pos);
      b.quat[bi] = q.w;
      b.quat[S + bi] = q.x;
      b.quat[2 * S + bi] = q.y;
      b.quat[3 * S + bi] = q.z;
    }
  }
}

// setSkewSymmetric, contact.go:612-616
template <typename R>
__device__ __forceinline__ void skew(const V3<R>& v, R* m) {
  m[0] = R(0); m[3] = -v.z; m[6] = v.y;
  m[1] = v.z;  m[4] = R(0); m[7] = -v.x;
  m[2] = -v.y; m[5] = v.x;  m[8] = R(0);
}

// calculateFrictionlessImpulse, contact.go:498-531, taken by contacts
// whose friction is 0 (contact.go:459-461; only KIND_MAT has such
// contacts): the impulse is (desiredDeltaVelocity / deltaVelocity, 0, 0)
// with this deltaVelocity, which depends only on quantities the velocity
// phase does not change.  ContactNormal is column 0 of contactToWorld.  The
// reference's test at :512 is inverted (Bodies[1] == nil): a two-body
// contact never adds its second body's terms, and a half-space contact
// dereferences nil there (a Go panic; here the absent body adds nothing).
// two_body (RM_FRICTIONLESS2) adds the second body's terms when it exists.
// im: the two bodies' inverse masses (im[1] unused without a second body).
template <typename R>
__device__ __forceinline__ R frictionless_delta_velocity(const R im[2], bool has1, const R* iit0, const R* iit1,
                                                         const V3<R> rel[2], const R* c2w, bool two_body) {
  const V3<R> n{c2w[0], c2w[1], c2w[2]};
  V3<R> dvw = cross(rel[0], n);
  dvw = m3v(iit0, dvw);
  dvw = cross(dvw, rel[0]);
  R deltaVelocity = dot(dvw, n);
  deltaVelocity += im[0];
  if (two_body && has1) {
    dvw = cross(rel[1], n);
    dvw = m3v(iit1, dvw);
    dvw = cross(dvw, rel[1]);
    deltaVelocity += dot(dvw, n);
    deltaVelocity += im[1];
  }
  return deltaVelocity;
}

// calculateFrictionImpulse, contact.go:535-606, in two parts.  The first
// builds the contact-frame matrix deltaVelocity (the velocity change per
// unit impulse, :537-578) and its inverse impulseMatrix (:581); they depend
// only on contactToWorld, the relative contact positions, both bodies'
// world inverse inertia and inverse masses, none of which the velocity
// phase changes, so the island kernel computes them once per
// phase for every contact.  It keeps the inverse (9) and deltaVelocity's
// entries 0, 3, 6 (the only ones the friction cone reads).
template <typename R>
__device__ __forceinline__ void friction_matrices(const R invm[2], bool has1, const R* iit0, const R* iit1,
                                                  const V3<R> rel[2], const R* c2w, R* im, R* dvcol) {
  R inverseMass = invm[0];
  R sk[9], t[9], dvw[9];
  skew(rel[0], sk);
  m3mul(sk, iit0, t);
  m3mul(t, sk, dvw);
#pragma unroll
  for (int k = 0; k < 9; ++k) dvw[k] *= R(-1);
  if (has1) {
    R d2[9];
    skew(rel[1], sk);
    m3mul(sk, iit1, t);
    m3mul(t, sk, d2);
#pragma unroll
    for (int k = 0; k < 9; ++k) d2[k] *= R(-1);
#pragma unroll
    for (int k = 0; k < 9; ++k) dvw[k] += d2[k];
    inverseMass += invm[1];
  }
  R ct[9] = {c2w[0], c2w[3], c2w[6], c2w[1], c2w[4], c2w[7], c2w[2], c2w[5], c2w[8]};
  R dv[9];
  m3mul(ct, dvw, t);
  m3mul(t, c2w, dv);
  dv[0] += inverseMass;
  dv[4] += inverseMass;
  dv[8] += inverseMass;
  m3inv(dv, im);
  dvcol[0] = dv[0];
  dvcol[1] = dv[3];
  dvcol[2] = dv[6];
}

// The second part (:582-606): the impulse that removes the desired normal
// velocity change and the tangential velocity, projected onto the friction
// cone when it leaves it.
template <typename R>
__device__ __forceinline__ V3<R> friction_impulse_from(const R* im, const R* dvcol, R ddv, const V3<R>& cvel,
                                                       R friction) {
  V3<R> velKill{ddv, -cvel.y, -cvel.z};
  V3<R> ic = m3v(im, velKill);
  R planar = dsqrt(ic.y * ic.y + ic.z * ic.z);
  if (planar > ic.x * friction) {
    ic.y /= planar;
    ic.z /= planar;
    ic.x = dvcol[0] + dvcol[1] * friction * ic.y + dvcol[2] * friction * ic.z;
    ic.x = ddv / ic.x;
    ic.y *= friction * ic.x;
    ic.z *= friction * ic.x;
  }
  return ic;
}

// The per-contact data of the velocity phase that the phase does not
// change: impulseMatrix (9) and deltaVelocity's entries 0, 3, 6 (3) of
// calculateFrictionImpulse, or, for a contact of friction 0 (KIND_MAT),
// calculateFrictionlessImpulse's deltaVelocity in entry 0.
constexpr int kImpPlanes = 12;

// From the bodies' world inverse inertia and inverse masses as given.
template <typename R, int KIND>
__device__ __forceinline__ void impulse_data_from(int32_t mode, const R* iit0, const R* iit1, const R invm[2], bool has1,
                                                  const V3<R> rel[2], const R* c2w, R friction, R* out) {
  if (KIND == KIND_MAT && friction == R(0)) {
    out[0] = frictionless_delta_velocity(invm, has1, iit0, iit1, rel, c2w, (mode & RM_FRICTIONLESS2) != 0);
#pragma unroll
    for (int k = 1; k < kImpPlanes; ++k) out[k] = R(0);
  } else {
    friction_matrices(invm, has1, iit0, iit1, rel, c2w, out, out + 9);
  }
}

template <typename R, int KIND>
__device__ __forceinline__ void impulse_data(const RS<R>& a, const int kb[2], const V3<R> rel[2], const R* c2w,
                                             R friction, R* out) {
  const Bodies<R>& b = a.b;
  const int64_t S = b.stride;
  R iit0[9], iit1[9];
  ld9(b.iit_world, S, kb[0], iit0);
#pragma unroll
  for (int k = 0; k < 9; ++k) iit1[k] = R(0);
  if (kb[1] >= 0) ld9(b.iit_world, S, kb[1], iit1);
  const R invm[2] = {b.inv_mass[kb[0]], kb[1] >= 0 ? b.inv_mass[kb[1]] : R(0)};
  impulse_data_from<R, KIND>(a.mode, iit0, iit1, invm, kb[1] >= 0, rel, c2w, friction, out);
}

// applyVelocityChange, contact.go:448-494, for a contact of the given
// friction, from its impulse data (impulse_data): the impulse in contact
// coordinates (the frictionless branch of :459-461 exists in KIND_MAT only),
// then the velocity and rotation changes of both bodies (:463-494).
template <typename R, int KIND>
__device__ __forceinline__ void apply_velocity_change(const RS<R>& a, const int kb[2], const V3<R> rel[2],
                                                      const R* c2w, R ddv, const V3<R>& cvel, const R* imp,
                                                      V3<R> vc[2], V3<R> rc[2], int lane, R friction) {
  const Bodies<R>& b = a.b;
  const int64_t S = b.stride;
  V3<R> ic;
  if (KIND == KIND_MAT && friction == R(0))
    ic = V3<R>{ddv / imp[0], R(0), R(0)};
  else
    ic = friction_impulse_from(imp, imp + 9, ddv, cvel, friction);
  const V3<R> impulse = m3v(c2w, ic);
  const V3<R> zero{R(0), R(0), R(0)};
  R iw[9];
  ld9(b.iit_world, S, kb[0], iw);
  V3<R> torque = cross(rel[0], impulse);
  rc[0] = m3v(iw, torque);
  vc[0] = add_scaled(zero, impulse, b.inv_mass[kb[0]]);
  rc[1] = zero;
  vc[1] = zero;
  const V3<R> v0 = add(ld3(b.vel, S, kb[0]), vc[0]);
  const V3<R> w0 = add(ld3(b.rot, S, kb[0]), rc[0]);
  if (lane == 0) {
    st3(b.vel, S, kb[0], v0);
    st3(b.rot, S, kb[0], w0);
  }
  if (kb[1] >= 0) {
    ld9(b.iit_world, S, kb[1], iw);
    torque = cross(impulse, rel[1]);
    rc[1] = m3v(iw, torque);
    vc[1] = add_scaled(zero, impulse, -b.inv_mass[kb[1]]);
    const V3<R> v1 = add(ld3(b.vel, S, kb[1]), vc[1]);
    const V3<R> w1 = add(ld3(b.rot, S, kb[1]), rc[1]);
    if (lane == 0) {
      st3(b.vel, S, kb[1], v1);
      st3(b.rot, S, kb[1], w1);
    }
  }
}

template <typename R, bool LDS, int KIND>
__device__ __forceinline__ void resolve_world(const RS<R>& a, int w, int C, int64_t base, R* key, int32_t* kb0, int32_t* kb1,
                              int lane) {
  const Bodies<R>& b = a.b;
  const Contacts<R>& c = a.c;
  const int64_t CS = c.cap;
  const int64_t maxIter = a.iter_fixed > 0 ? a.iter_fixed : a.iter_mult * int64_t(C);

  const bool do_pos = (a.mode & RM_POS) != 0;
  const bool do_prep = do_pos && !(a.mode & RM_PREPARED);
  const bool do_vel = (a.mode & RM_VEL) != 0 && (KIND == KIND_POLISH || !a.world_mask || a.world_mask[w]);
  // worlds this path takes are never polished: the plain phase
  if ((KIND == KIND_POLISH || KIND == KIND_PPOLISH) && lane == 0) a.world_mask[w] = 1;
  // prepareContacts, contact.go:225-229
  for (int j = lane; j < C; j += 64) {
    if (do_prep) prepare_contact<R, KIND>(a, base + j);
    if (LDS) {
      key[j] = c.pen[base + j];
      kb0[j] = c.body0[base + j];
      kb1[j] = c.body1[base + j];
    }
  }
  __syncthreads();

  // adjustPositions, contact.go:233-283
  int64_t used = 0;
  while (do_pos && used < maxIter) {
    R best = R(kPositionEpsilon);
    int bi = INT_MAX;
    for (int j = lane; j < C; j += 64) {
      const R p = key[j];
      if (p > best) {
        best = p;
        bi = j;
      }
    }
    wave_argmax_dpp(best, bi);
    if (bi == INT_MAX) break;
    const int64_t g = base + bi;
    const int kb[2] = {kb0[bi], kb1[bi]};
    const V3<R> n = ld3(c.normal, CS, g);
    const V3<R> rel[2] = {ld3(c.rel, CS, g), ld3(c.rel + 3 * CS, CS, g)};
    bool aw[2];
    match_awake(a, kb[0], kb[1], aw[0], aw[1], lane);
    V3<R> lin[2], ang[2];
    apply_position_change(a, kb, aw, n, rel, best, lin, ang, lane);
    if constexpr (KIND == KIND_LABEL)
      if (lane == 0) add_pos_label(a, g, best);
    for (int j = lane; j < C; j += 64) {
      const int jb[2] = {kb0[j], kb1[j]};
      bool any = false;
#pragma unroll
      for (int bb = 0; bb < 2; ++bb)
#pragma unroll
        for (int d = 0; d < 2; ++d) any |= (jb[bb] >= 0 && jb[bb] == kb[d]);
      if (!any) continue;
      R p = key[j];
      const V3<R> nj = ld3(c.normal, CS, base + j);
#pragma unroll
      for (int bb = 0; bb < 2; ++bb) {
        if (jb[bb] < 0) continue;
        const V3<R> rj = ld3(c.rel + 3 * bb * CS, CS, base + j);
        // a side is at most one of the two moved bodies: its change is
        // selected and applied once
        if (jb[bb] == kb[0] || jb[bb] == kb[1]) {
          const bool d0 = jb[bb] == kb[0];
          V3<R> dp = add(cross(sel3(d0, ang[0], ang[1]), rj), sel3(d0, lin[0], lin[1]));
          R sign = R(1);
          if (bb == 0) sign = R(-1);
          p += dot(dp, nj) * sign;
        }
      }
      key[j] = p;
    }
    __syncthreads();
    ++used;
  }
  const int64_t pos_iters = used;
  if (LDS) {
    for (int j = lane; j < C; j += 64) {
      if (do_pos) c.pen[base + j] = key[j];
      key[j] = c.ddv[base + j];
    }
    __syncthreads();
  }
  R* dkey = LDS ? key : c.ddv + base;

  // adjustVelocities, contact.go:390-445
  used = 0;
  while (do_vel && used < maxIter) {
    R best = R(kVelocityEpsilon);
    int bi = INT_MAX;
    for (int j = lane; j < C; j += 64) {
      const R p = dkey[j];
      if (p > best) {
        best = p;
        bi = j;
      }
    }
    wave_argmax_dpp(best, bi);
    if (bi == INT_MAX) break;
    const int64_t g = base + bi;
    const int kb[2] = {kb0[bi], kb1[bi]};
    const V3<R> rel[2] = {ld3(c.rel, CS, g), ld3(c.rel + 3 * CS, CS, g)};
    R m[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) m[k] = c.c2w[k * CS + g];
    const V3<R> cv = ld3(c.cvel, CS, g);
    bool aw[2];
    match_awake(a, kb[0], kb[1], aw[0], aw[1], lane);
    V3<R> vc[2], rc[2];
    const R fr = friction_of<R, KIND>(c, g);
    R imp[kImpPlanes];
    impulse_data<R, KIND>(a, kb, rel, m, fr, imp);
    apply_velocity_change<R, KIND>(a, kb, rel, m, best, cv, imp, vc, rc, lane, fr);
    if constexpr (KIND == KIND_LABEL)
      if (lane == 0) add_label(a, g, vc, rc);
    for (int j = lane; j < C; j += 64) {
      const int jb[2] = {kb0[j], kb1[j]};
      bool any = false;
#pragma unroll
      for (int bb = 0; bb < 2; ++bb)
#pragma unroll
        for (int d = 0; d < 2; ++d) any |= (jb[bb] >= 0 && jb[bb] == kb[d]);
      if (!any) continue;
      const int64_t gj = base + j;
      R mj[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) mj[k] = c.c2w[k * CS + gj];
      V3<R> cvj = ld3(c.cvel, CS, gj);
#pragma unroll
      for (int bb = 0; bb < 2; ++bb) {
        if (jb[bb] < 0) continue;
        const V3<R> rj = ld3(c.rel + 3 * bb * CS, CS, gj);
        // a side is at most one of the two moved bodies: its change is
        // selected and applied once
        if (jb[bb] == kb[0] || jb[bb] == kb[1]) {
          const bool d0 = jb[bb] == kb[0];
          V3<R> dv = add(cross(sel3(d0, rc[0], rc[1]), rj), sel3(d0, vc[0], vc[1]));
          R sign = R(1);
          if (bb == 1) sign = R(-1);
          cvj = add(cvj, mul(m3tv(mj, dv), sign));
        }
      }
      st3(c.cvel, CS, gj, cvj);
      const V3<R> nj = ld3(c.normal, CS, gj);
      dkey[j] = desired_dv(b, jb[0], jb[1], nj, cvj.x, a.dt, restitution_of<R, KIND>(c, gj));
    }
    __syncthreads();
    ++used;
  }
  if (LDS && do_vel) {
    for (int j = lane; j < C; j += 64) c.ddv[base + j] = dkey[j];
  }
  if (lane == 0 && a.world_iters) {
    if (do_pos) a.world_iters[2 * w] = pos_iters;
    if (do_vel) a.world_iters[2 * w + 1] = used;
  }
}

// worlds the surrogate's polish takes; beyond them, the plain phases
constexpr int kPolishBodies = 256;
constexpr int kPolishContacts = 2048;

// A value that is the same in every lane, in scalar registers: loaded behind
// stores, it would be a vector register's, and every address made of it.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uniform(int64_t v) {
  return int64_t(uint64_t(uint32_t(uniform(int(v >> 32)))) << 32 | uint32_t(uniform(int(v))));
}

// One world on one wave, its state in HBM: selection keys and body ids in
// LDS when the world has at most kKeyCap contacts.
template <typename R, int KIND>
__device__ __forceinline__ void resolve_hbm(const RS<R>& a, int w, int C, char* lds, int lane) {
  if (a.world_iters && lane == 0) {
    if (a.mode & RM_POS) a.world_iters[2 * w] = 0;
    if (a.mode & RM_VEL) a.world_iters[2 * w + 1] = 0;
  }
  // ResolveContacts' guard, contact.go:210-212
  if (a.overflow[0] != 0 || C <= 0 || a.dt <= R(0)) return;
  const int64_t base = uniform(a.world_coff[w]);
  if (C <= kKeyCap) {
    R* s_key = (R*)lds;
    int32_t* s_b0 = (int32_t*)(lds + kKeyCap * sizeof(R));
    int32_t* s_b1 = s_b0 + kKeyCap;
    resolve_world<R, true, KIND>(a, w, C, base, s_key, s_b0, s_b1, lane);
  } else {
    resolve_world<R, false, KIND>(a, w, C, base, a.c.pen + base, a.c.body0 + base, a.c.body1 + base, lane);
  }
}

// ---------------------------------------------------------------------------
// pieces of the island kernel (cbz_islands.h)
// ---------------------------------------------------------------------------
// A contact's body ids, world-local, packed 16 + 16 bits.
constexpr uint32_t kNoBody = 0xFFFFu;

// Kinetic energy of a body, 1/2 (m |v|^2 + w . I w) with I the inverse of
// the world inverse inertia tensor (a zero matrix for an infinite tensor,
// math/matrix.go:133-137), in FP64; 0 for an infinite mass.  Also returns m.
template <typename R>
__device__ __forceinline__ double kinetic_energy(const V3<R>& v, const V3<R>& w, R inv_mass, const R* iit,
                                                 double& mass) {
  mass = 0.0;
  if (!(inv_mass > R(0))) return 0.0;
  mass = 1.0 / double(inv_mass);
  double m[9], I[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) m[k] = double(iit[k]);
  m3inv(m, I);
  const V3<double> wd{double(w.x), double(w.y), double(w.z)};
  const V3<double> Iw = m3v(I, wd);
  const double vv = double(v.x) * double(v.x) + double(v.y) * double(v.y) + double(v.z) * double(v.z);
  return 0.5 * (mass * vv + dot(wd, Iw));
}

__device__ __forceinline__ int id_lo(uint32_t id) { return int(id & 0xFFFFu); }
__device__ __forceinline__ int id_hi(uint32_t id) { return (id >> 16) == kNoBody ? -1 : int(id >> 16); }

// Broadcast of lane l's value (l uniform) by readlane.
__device__ __forceinline__ float lane_value(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_value(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}
// Marks the slots' packed body ids as redefined, so that values derived from
// them (decoded ids, comparison masks: one 64-bit scalar mask per slot) are
// recomputed in each iteration instead of being hoisted out of the loop, where
// they would be spilled.
template <int N>
__device__ __forceinline__ void opaque_ids(uint32_t (&ids)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) asm volatile("" : "+v"(ids[k]));
}

// A lane's index as a value redefined at the point of the call: the addresses
// computed from it are then recomputed there instead of being hoisted out of
// the loop.
__device__ __forceinline__ int opaque_lane(int lane) {
  asm volatile("" : "+v"(lane));
  return lane;
}

// Element s (uniform) of a register array, as a chain of selects with
// compile-time indexes (an indexed loop would keep the array in scratch).
template <typename T, int N, int... K>
__device__ __forceinline__ T pick_impl(const T (&a)[N], int s, std::integer_sequence<int, K...>) {
  T v = a[0];
  ((v = (K == s) ? a[K] : v), ...);
  return v;
}
template <typename R, int N, int... K>
__device__ __forceinline__ V3<R> pick_impl(const V3<R> (&a)[N], int s, std::integer_sequence<int, K...>) {
  // component by component: a select of the structs would go through memory
  R x = a[0].x, y = a[0].y, z = a[0].z;
  ((x = (K == s) ? a[K].x : x, y = (K == s) ? a[K].y : y, z = (K == s) ? a[K].z : z), ...);
  return V3<R>{x, y, z};
}
template <typename T, int N>
__device__ __forceinline__ T pick(const T (&a)[N], int s) {
  return pick_impl(a, s, std::make_integer_sequence<int, N>{});
}
// a if c else b, component by component
template <typename R>
__device__ __forceinline__ V3<R> sel3(bool c, const V3<R>& a, const V3<R>& b) {
  return V3<R>{c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z};
}


// Both bodies' world inverse inertia and inverse mass (zeros for an absent
// second body).
template <typename R>
__device__ __forceinline__ void body_inertia(const Bodies<R>& b, const int kb[2], R (&iw)[2][9], R im[2]) {
  const int64_t S = b.stride;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
#pragma unroll
    for (int k = 0; k < 9; ++k) iw[i][k] = R(0);
    im[i] = R(0);
  }
  ld9(b.iit_world, S, kb[0], iw[0]);
  im[0] = b.inv_mass[kb[0]];
  if (kb[1] >= 0) {
    ld9(b.iit_world, S, kb[1], iw[1]);
    im[1] = b.inv_mass[kb[1]];
  }
}

// Entry e of a left list: the world, and the phases it still needs.
template <typename R>
__device__ __forceinline__ int left_world(RS<R>& a, int32_t e) {
  if (e & kLeftVelOnly) a.mode &= ~(RM_POS | RM_PREPARED);
  return e & ~kLeftVelOnly;
}

// The worlds the island kernel leaves, a wave each.  The last workgroup that
// had one clears the counters for the next resolve (without any, the first).
template <typename R, int KIND>
__device__ __forceinline__ void resolve_left_block(const RS<R>& args) {
  __shared__ __align__(16) char lds[kKeyCap * (sizeof(R) + 2 * sizeof(int32_t))];
  const int lane = threadIdx.x;
  const int left = uniform(args.left_count[LEFT_WORLDS]);
  for (int k = blockIdx.x; k < left; k += gridDim.x) {
    RS<R> a = args;
    const int w = left_world(a, uniform(args.left_list[k]));
    int64_t* wt = a.world_time ? a.world_time + 4 * int64_t(w) + ((a.mode & RM_VEL) ? 2 : 0) : nullptr;
    if (wt && lane == 0) wt[0] = int64_t(wall_clock64());
    resolve_hbm<R, KIND>(a, w, uniform(a.world_cnt[w]), lds, lane);
    __syncthreads();
    if (wt && lane == 0) wt[1] = int64_t(wall_clock64());
  }
  const int with = left < int(gridDim.x) ? left : int(gridDim.x);  // workgroups that had a world
  if (lane != 0 || int(blockIdx.x) >= (with > 0 ? with : 1)) return;
  __threadfence();
  if (with == 0 || atomicAdd(&args.left_count[LEFT_DONE], 1) == with - 1) {
    for (int q = 0; q < LEFT_COUNTS; ++q) args.left_count[q] = 0;
    *args.log_head = 0;
  }
}

template <typename R, int KIND>
__global__ void __launch_bounds__(64) k_resolve_left(RS<R> a) {
  resolve_left_block<R, KIND>(a);
}

// A workgroup for every world that can be left: the world's bodies or the
// contacts of one of its islands exceed the tables, which takes more than
// kLeftBodies bodies unless they are packed into each other.  Workgroups beyond
// the list end at once.  450 worlds of 2100 bodies, 60 of them in contact, take
// 1.47 ms; with 256 workgroups, and the world's place in vector registers, 2.0.
constexpr int kLeftGrid = 256;
template <typename R, int KIND>
void launch_left_kind(const RS<R>& a, int grid, hipStream_t st) {
  k_resolve_left<R, KIND><<<grid, 64, 0, st>>>(a);
}

// Every instantiation lives in one translation unit of its own
// (k_resolve_<precision>_<kind>.hip); other units only declare them.
#define CBZ_RESOLVE_KIND(EXT, R, KIND)                                          \
  EXT template void launch_left_kind<R, KIND>(const RS<R>&, int, hipStream_t); \
  EXT template hipError_t launch_islands_kind<R, KIND>(const RS<R>&, bool, hipStream_t); \
  EXT template hipError_t islands_occupancy<R, KIND>(int, int*);

}  // namespace cbz
