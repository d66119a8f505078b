// cbz_islands.h — K3 by islands: ResolveContacts (contact.go:208-222) with
// one workgroup per world and the world's islands side by side.
//
// An island is a set of bodies joined by contacts (half-space contacts join
// nothing).  An iteration of the reference's worst-first loop reads and
// writes only the selected contact's island, so the selections that fall
// into one island, in their order, are exactly those the same loop makes on
// that island alone: its largest key, the lowest contact index on a tie.
// The islands of a world can therefore run at the same time and give the
// same bits, as long as the world's iterations together stay within the
// iteration budget (maxIter is the world's, contact.go:235 and :392).
//
// What that buys.  As one chain (one wavefront per world, or four for the
// largest), a settled world of 470 contacts ran about 1000 iterations of
// 3-4 us, each a scan of every contact of the world; it has about 100
// islands, most of them one cube with its four ground contacts (3-5
// iterations), the largest of 10-60 contacts (50-300 iterations).  A step of
// the exact path, before and after (ms):
//   1000 batched worlds FP64            7.4 -> 1.0
//   2048 batched worlds FP32            7.4 -> 1.05
//   1 world of 301 cubes landing FP32   1.3 -> 0.18
//   1024 bodies, spheres and cubes      0.82 -> 0.18
//   1024 worlds of towers, standing     1.7 -> 0.47; collapsed into piles of
//     200-500 contacts, up to half of the worlds over their budget, 5.2 -> 5.3
// and of the surrogate over 4096 worlds 4.5 -> 2.4 (narrowphase and order of
// the worlds included).
//
// The work of an island: a power-of-two group of lanes, one contact per
// lane, all of a contact's data in its lane's registers; several groups share
// a wave.  (Islands of more than 64 contacts: the whole workgroup.)  An
// iteration: the group's argmax by DPP, the lane that owns the selected contact
// computes the correction alone (the wave would spend the same instructions if
// every lane did) and puts the two bodies' changes into LDS, from where the
// group's lanes update their own contacts.  The bodies' state is in LDS for the
// phase.  Islands are handed out by size,
// the largest first, so that the islands that share a wave run for similar
// times.
//
// The budget.  Each phase first runs every island to its end and counts.  If
// the world's sum exceeds the budget, the serial loop would have stopped in
// the middle: the islands' selections are logged, the logs merged as the serial
// loop orders them (always the island whose next selection has the largest key)
// up to the budget, and each island runs to its share.  The merge needs only the
// selections at which an island's running minimum falls (or is met again):
// between two of those the island's next key is above every other island's,
// so the serial loop stays in it.
//
// What a world over its budget waits for is, as a rule, one island that does not
// settle.  Three runs of that (to count, to log, to its share) take longer than
// the serial chain did, so in the velocity phase an island that has run for a
// quarter of the budget logs from there on and keeps two checkpoints: the second
// run is of the first quarter, the third starts from the last checkpoint before
// the share.  1000 landing worlds take 0.40 ms a resolve (0.71 with three whole
// runs, 0.53 as serial chains), 1000 of 8 to 32 bodies 0.51 (0.75, 0.53).  The
// registers this takes cost every launch 1.4 us (one landing world of 64 bodies:
// 26.5 instead of 25.0).
//
// A budget that is small for the world is not worth it: a world whose budget is
// below half (with more than 512 contacts a quarter) of its contacts, or whose
// budget of at most 96 is exceeded, runs as one island of all its contacts, which
// makes its selections in the serial order; so does a world whose logs find no
// room.  20 iterations of 1000 worlds of 350 contacts take 0.34 ms (0.92 in three
// runs, 0.32 as serial chains).
//
// Worlds this does not take (more bodies than the LDS tables hold, an island
// of more than 2048 contacts, contacts that name bodies of another world, more
// than 2048 contacts and no room for the logs) are left to the serial kernel of
// cbz_resolve.h.
#pragma once
#include "cbz_resolve.h"

namespace cbz {

// Size classes by contact count: above 4 T, 2 T, T and 64 (the whole workgroup
// of T threads, 8, 8 or 4, 2 or 1 contacts per thread), then one contact per lane
// in groups of 64, 32, 16, 8 and 4 lanes.  RS::isl_cls holds kIslWords words per
// world: the counts, and at kIslTaken the workgroup size the islands were made
// for (0: not taken).
constexpr int kIslClasses = 9, kIslBigClasses = 4, kIslTaken = 9;
// contacts of the largest island taken
template <int T>
constexpr int isl_max_contacts() { return 8 * T; }
template <int T>
__device__ __forceinline__ int isl_class(int c) {
  return c > 4 * T ? 0 : c > 2 * T ? 1 : c > T ? 2 : c > 64 ? 3 : c > 32 ? 4 : c > 16 ? 5 : c > 8 ? 6 : c > 4 ? 7 : 8;
}
__device__ __forceinline__ int isl_class_lg(int k) { return 10 - k; }  // log2 lanes per island of a small class

enum : int { ISL_FREE = 0, ISL_LOG = 1, ISL_LIMIT = 2 };

// LDS: the fixed part, then the body tables (NB bodies): R[NB][8] state
// (position and orientation, or velocity and rotation; the island search
// and the merge use the space before and between), uint8[NB] flags.
template <typename R>
struct IslBest {
  R key;
  int32_t j;
  uint32_t id;
};
template <typename R, int T>
struct IslFixed {
  static constexpr int kWaves = T / 64;
  R x[kWaves][16][12];         // the two bodies' changes of each group's iteration
  uint32_t xi[kWaves][16][2];  // packed body ids, rederived bits
  double sum[kWaves];
  // each wave's best contact of a big island (two iterations' worth), with
  // what its correction would change: the two bodies' changes 12, their new
  // velocity and rotation 12 (position and orientation 14)
  IslBest<R> best[2][kWaves];
  R bx[2][kWaves][28];
  unsigned long long total;       // the phase's iterations
  int32_t cls[kIslWords];         // class counts, then cursors
  int32_t next, over, bad, off, ok;
  int32_t big, bigs, bigoff;      // contacts and number of the big islands, the next one's place
  int32_t lates;                  // islands that log late
  int32_t paused, at;             // the big island the budget stopped (-1: none), its iterations there
  int32_t runj;                   // and where its running minimum stood: contact, key
  R runkey;
};
template <typename R, int T>
constexpr size_t isl_fixed_bytes() {
  return (sizeof(IslFixed<R, T>) + 15) & ~size_t(15);
}

// Stores of one lane of a wave before loads of others, through LDS (which a
// wave's operations reach in program order): the compiler must not move
// them across.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename R>
__device__ __forceinline__ R dpp_xor1(R v) { return dpp::mov<0xB1, 0xF>(v, v); }         // quad_perm 1,0,3,2
template <typename R>
__device__ __forceinline__ R dpp_xor2(R v) { return dpp::mov<0x4E, 0xF>(v, v); }         // quad_perm 2,3,0,1
template <typename R>
__device__ __forceinline__ R dpp_half_mirror(R v) { return dpp::mov<0x141, 0xF>(v, v); } // i <-> 7 - i
template <typename R>
__device__ __forceinline__ R dpp_mirror(R v) { return dpp::mov<0x140, 0xF>(v, v); }      // i <-> 15 - i

__device__ __forceinline__ int lane_of(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float lane_of(float v, int l) { return lane_value(v, l); }
__device__ __forceinline__ double lane_of(double v, int l) { return lane_value(v, l); }

// op over each group of 2^lg lanes (lg 2..6, the same for the whole wave);
// every lane of the group gets it.  All lanes are active.  Within a row of 16
// by DPP, across rows through scalar registers (readlane): no LDS round trip
// in an iteration's serial chain.
template <typename T, typename OP>
__device__ __forceinline__ T group_reduce(T v, int lg, OP op) {
  v = op(v, dpp_xor1(v));
  v = op(v, dpp_xor2(v));
  if (lg > 2) v = op(v, dpp_half_mirror(v));
  if (lg > 3) v = op(v, dpp_mirror(v));
  if (lg > 4) {
    const T lo = op(lane_of(v, 0), lane_of(v, 16)), hi = op(lane_of(v, 32), lane_of(v, 48));
    v = lg > 5 ? op(lo, hi) : (threadIdx.x & 32) ? hi : lo;
  }
  return v;
}

// The lane of each group whose key is the group's greatest (m); among equal keys
// the lowest index j.  gm: the group's lanes.  The second reduction is made
// only when some group has equal keys.
template <typename R>
__device__ __forceinline__ bool group_owner(bool top, int j, int lg, uint64_t gm) {
  const uint64_t g = __ballot(top) & gm;
  if (!__any(__popcll(g) > 1)) return top;
  const int jm = group_reduce(top ? j : INT_MAX, lg, [](int p, int q) { return q < p ? q : p; });
  return top && j == jm;
}
__device__ __forceinline__ uint64_t group_lanes(int lg) {
  const int lane = int(threadIdx.x & 63);
  return lg == 6 ? ~uint64_t(0) : ((uint64_t(1) << (1 << lg)) - 1) << (lane >> lg << lg);
}

// Body i's entry in the state table: 8 reals, position 0-2 and orientation
// 3-6, or velocity 0-2 and rotation 3-5 (one address per body; the rest of
// the address is an immediate).
constexpr int kIslSt = 8;
// Body i's entry in the inertia table, which a launch has when its worlds are
// of at most kIslIwBodies bodies (20 KB in FP64; beyond, it would cost the
// second workgroup of a CU its place).
constexpr int kIslIw = 10, kIslIwBodies = 256;
template <typename R>
__device__ __forceinline__ V3<R> tab3(const R* e) {
  return V3<R>{e[0], e[1], e[2]};
}
template <typename R>
__device__ __forceinline__ void tab3_store(R* e, const V3<R>& v) {
  e[0] = v.x;
  e[1] = v.y;
  e[2] = v.z;
}

// One world as the workgroup sees it.
template <typename R, int T>
struct IslWorld {
  int w, C, b0w, n, NB, t;
  int64_t base;
  IslFixed<R, T>* f;
  R* st;
  R* iw;  // [n][kIslIw] world inverse inertia 9, inverse mass, or null: no table in this launch
  uint8_t* fl;
};

// Sum / extreme over the workgroup, in a fixed order.
template <typename R, typename OP, int T>
__device__ __forceinline__ double isl_reduce(const IslWorld<R, T>& W, double v, OP op) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = op(v, __shfl_xor(v, o, 64));
  if ((W.t & 63) == 0) W.f->sum[W.t >> 6] = v;
  __syncthreads();
  double r = W.f->sum[0];
#pragma unroll
  for (int k = 1; k < (T / 64); ++k) r = op(r, W.f->sum[k]);
  __syncthreads();
  return r;
}

// ---------------------------------------------------------------------------
// the islands of a world
// ---------------------------------------------------------------------------
// Union-find over the bodies in LDS, then per island its contacts as a list
// (any order: ties are broken by the contact's index, which travels with
// the key).  Writes isl_off / isl_cnt [b0w + rank] with ranks ordered by
// class, isl_idx [base ..], and the class counts with a "taken" mark.
template <typename R, int T>
__device__ __forceinline__ void isl_build(const RS<R>& a, const IslWorld<R, T>& W) {
  int32_t* par = (int32_t*)W.st;
  int32_t* cnt = par + W.NB;
  const Contacts<R>& c = a.c;
  for (int i = W.t; i < W.n; i += T) {
    par[i] = i;
    cnt[i] = 0;
  }
  if (W.t < kIslWords) W.f->cls[W.t] = 0;
  if (W.t == 0) W.f->bad = W.f->off = W.f->big = W.f->bigs = 0;
  __syncthreads();
  volatile int32_t* vp = par;
  auto root = [&](int i) {
    int p = vp[i];
    while (p != i) {
      i = p;
      p = vp[i];
    }
    return i;
  };
  for (int j = W.t; j < W.C; j += T) {
    const int c0 = c.body0[W.base + j], c1 = c.body1[W.base + j];
    const int l0 = c0 - W.b0w, l1 = c1 - W.b0w;
    if (l0 < 0 || l0 >= W.n || (c1 >= 0 && (l1 < 0 || l1 >= W.n))) {
      W.f->bad = 1;
      continue;
    }
    if (c1 < 0) continue;
    int ra = root(l0), rb = root(l1);
    while (ra != rb) {  // hook the larger root under the smaller
      if (ra < rb) {
        const int x = ra;
        ra = rb;
        rb = x;
      }
      const int old = atomicCAS(&par[ra], ra, rb);
      if (old == ra) break;
      ra = root(old);
      rb = root(rb);
    }
  }
  __syncthreads();
  if (W.f->bad) {
    if (W.t == 0) a.isl_cls[kIslWords * int64_t(W.w) + kIslTaken] = 0;
    return;
  }
  for (int i = W.t; i < W.n; i += T) {
    const int r = root(i);
    vp[i] = r;  // a root keeps itself; others' chains only get shorter
  }
  __syncthreads();
  for (int j = W.t; j < W.C; j += T) atomicAdd(&cnt[par[c.body0[W.base + j] - W.b0w]], 1);
  __syncthreads();
  for (int i = W.t; i < W.n; i += T) {
    if (cnt[i] > isl_max_contacts<T>()) W.f->bad = 1;
    if (cnt[i] > 64) {
      atomicAdd(&W.f->big, cnt[i]);
      atomicAdd(&W.f->bigs, 1);
    }
    if (cnt[i] > 0) atomicAdd(&W.f->cls[isl_class<T>(cnt[i])], 1);
  }
  __syncthreads();
  // The big islands run one after another on the whole workgroup; together
  // they run as many iterations as one island of all their contacts, whose
  // loop makes their selections in the serial order.  So they are one, where
  // that is not too large: one island per world can be paused at the budget.
  const bool one = W.f->bigs > 0 && W.f->big <= isl_max_contacts<T>();
  if (W.t == 0) {
    if (one) {
#pragma unroll
      for (int k = 0; k < kIslBigClasses; ++k) W.f->cls[k] = 0;
      W.f->cls[isl_class<T>(W.f->big)] = 1;
      W.f->bigoff = 0;
      W.f->off = W.f->big;
      a.isl_off[W.b0w] = 0;
      a.isl_cnt[W.b0w] = W.f->big;
    }
    int32_t at = 0;
#pragma unroll
    for (int k = 0; k < kIslClasses; ++k) {
      const int32_t m = W.f->cls[k];
      a.isl_cls[kIslWords * int64_t(W.w) + k] = m;
      W.f->cls[k] = at;
      at += m;
    }
    a.isl_cls[kIslWords * int64_t(W.w) + kIslTaken] = W.f->bad ? 0 : T;
  }
  __syncthreads();
  if (W.f->bad) return;
  for (int i = W.t; i < W.n; i += T) {
    const int m = cnt[i];
    if (m <= 0) continue;
    if (one && m > 64) {
      cnt[i] = atomicAdd(&W.f->bigoff, m);
      continue;
    }
    const int k = atomicAdd(&W.f->cls[isl_class<T>(m)], 1);
    const int o = atomicAdd(&W.f->off, m);
    a.isl_off[W.b0w + k] = o;
    a.isl_cnt[W.b0w + k] = m;
    cnt[i] = o;
  }
  __syncthreads();
  for (int j = W.t; j < W.C; j += T) {
    const int p = atomicAdd(&cnt[par[c.body0[W.base + j] - W.b0w]], 1);
    a.isl_idx[W.base + p] = j;
  }
}

// prepareContacts (contact.go:225-229), a thread per contact, with every
// contact's record, the bodies' prepare-time positions and the islands.
template <typename R, int KIND, int T>
__device__ __forceinline__ void isl_prepare(const RS<R>& a, const IslWorld<R, T>& W, bool islands) {
  const int64_t S = a.b.stride;
  for (int i = W.t; i < W.n; i += T) st3(a.pos0, S, W.b0w + i, ld3(a.b.pos, S, W.b0w + i));
  for (int j = W.t; j < W.C; j += T) prepare_contact<R, KIND, true>(a, W.base + j);
  __syncthreads();
  if (islands) isl_build(a, W);
  __syncthreads();
}

// ---------------------------------------------------------------------------
// one batch: the islands of one class that share a wave
// ---------------------------------------------------------------------------
// Iteration budgets are counted in 32 bits per island.
__device__ __forceinline__ int64_t isl_budget(int64_t n) { return n < (int64_t(1) << 30) ? n : int64_t(1) << 30; }

struct IslPass {
  int pass;        // ISL_FREE, ISL_LOG or ISL_LIMIT
  bool saved;      // the contacts' values before the phase are in isl_save already
  int64_t budget;  // ISL_FREE, ISL_LOG: no island runs longer
  bool pause;      // ISL_FREE: the last island stops where the world's budget is spent
  int resume;      // ISL_LOG, ISL_LIMIT: the island that goes on from its pause (-1: none)
  bool only;       // ... alone
  bool one;        // ISL_FREE: the world's contacts as one island, the serial loop itself
  // ISL_FREE: iterations after which an island logs (0: never), with checkpoints at
  // two and three times as many; ISL_LIMIT: it starts from the last one before its
  // share
  int late;
};
// isl_nrec: the log was begun in the free pass, after IslPass::late iterations,
// with room for isl_late_records (a record is a new running minimum, of the log's
// part here; it takes several iterations to one, as a rule).  Those before them
// are logged later, in front: entry 0 holds how many, and how many of the later
// ones are above them, then there is room for `late` of them.  At most kIslLates
// of a world's islands do so.
constexpr int kIslLate = 1 << 30, kIslLates = 3;
__device__ __forceinline__ int isl_late_records(int64_t budget) { return int(budget >> 1); }
__device__ __forceinline__ bool isl_is_late(int nrec) { return nrec >= kIslLate; }

// An island's log: record r is entry place(r).
struct IslLog {
  int64_t at;
  int n, gap_at, gap;
  __device__ __forceinline__ int64_t place(int r) const { return at + r + (r >= gap_at ? gap : 0); }
};
template <typename R>
__device__ __forceinline__ IslLog isl_log_of(const RS<R>& a, int g, int late) {
  const int64_t at = a.isl_log[g];
  const int n = a.isl_nrec[g];
  if (!isl_is_late(n)) return IslLog{at, n, INT_MAX, 0};
  const int before = a.log_it[at], skip = a.log_j[at];
  return IslLog{at + 1, before + n - kIslLate - skip, before, late - before + skip};
}

// The first of records lo .. hi of a log whose key is not above tau (hi if there
// is none).
template <typename R>
__device__ __forceinline__ int isl_first(const RS<R>& a, const IslLog& L, int lo, int hi, R tau) {
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (a.log_key[L.place(mid)] > tau)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// Ends of a batch: the islands' iteration counts, the world's sum.
template <typename R, int T>
__device__ __forceinline__ void isl_count(const RS<R>& a, const IslWorld<R, T>& W, const IslPass& P, int k, bool first,
                                          int it, int nrec, bool over, R runmin) {
  if (!first) return;
  if (P.pass == ISL_FREE) {
    a.isl_its[W.b0w + k] = it;
    a.isl_nrec[W.b0w + k] = nrec < 0 ? -1 : kIslLate + nrec;
    if (it > 0) atomicAdd(&W.f->total, (unsigned long long)it);
    if (over) W.f->over = 1;
  } else if (P.pass == ISL_LOG) {
    const int n = a.isl_nrec[W.b0w + k];
    if (P.late > 0 && isl_is_late(n)) {  // the free pass's records from this running minimum on
      const int64_t at = a.isl_log[W.b0w + k];
      const int skip = isl_first(a, IslLog{at + 1 + P.late, n - kIslLate, INT_MAX, 0}, 0, n - kIslLate, runmin);
      a.log_it[at] = nrec;
      a.log_j[at] = skip;
      return;
    }
    a.isl_its[W.b0w + k] = it;
    a.isl_nrec[W.b0w + k] = nrec;
  }
}

template <typename R>
__device__ __forceinline__ void isl_log(const RS<R>& a, int64_t at, R key, int j, int it) {
  a.log_key[at] = key;
  a.log_j[at] = j;
  a.log_it[at] = it;
}

// `need` entries of the log pool: where they start, or -1 (and they stay free
// for worlds that need less).
template <typename R>
__device__ __forceinline__ int64_t isl_reserve(const RS<R>& a, int64_t need) {
  unsigned long long* head = (unsigned long long*)a.log_head;
  const int64_t at = int64_t(atomicAdd(head, (unsigned long long)need));
  if (at + need <= a.log_cap) return at;
  atomicAdd(head, (unsigned long long)-need);
  return -1;
}

// What applyPositionChange (contact.go:286-386) computes of a contact that
// does not depend on its penetration: the shares of the angular and linear
// move, the angular limit, and the rotation per unit of angular inertia.  It
// changes only with a body's world inverse inertia (a sleeping body's derived
// data).  Kept per contact it takes three divisions, a square root and three
// matrix products out of every iteration, and fewer registers than the two
// tensors.  With it, with the sides of a touched contact side by side and with
// one barrier per iteration of a big island, 301 cubes in one world (FP32) take
// 10% less per step, 1000 worlds (FP64) 5%.
template <typename R>
struct IslMove {
  R ai[2], ra[2], rl[2], mm[2];  // angular inertia, shares, limit
  V3<R> td[2];
};
template <typename R>
__device__ __forceinline__ void isl_move_of(bool has1, const V3<R>& n, const V3<R> rel[2], const R (&iw)[2][9],
                                            const R im[2], IslMove<R>& mv) {
  const R angularLimit = R(0.2);
  R linI[2] = {R(0), R(0)}, total = R(0);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    mv.ai[i] = R(0);
    if (i == 1 && !has1) continue;
    V3<R> aiw = cross(rel[i], n);
    aiw = m3v(iw[i], aiw);
    aiw = cross(aiw, rel[i]);
    mv.ai[i] = dot(aiw, n);
    linI[i] = im[i];
    total += linI[i] + mv.ai[i];
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    mv.ra[i] = mv.ai[i] / total;
    mv.rl[i] = linI[i] / total;
    V3<R> projection = add_scaled(rel[i], n, -dot(rel[i], n));
    mv.mm[i] = angularLimit * mag(projection);
    mv.td[i] = m3v(iw[i], cross(rel[i], n));
  }
}

// The rest of it: the moves of the two bodies for a penetration, and their new
// position and orientation from the tables (st: 7 reals per body).
template <typename R, int T>
__device__ __forceinline__ void isl_position_change(const IslWorld<R, T>& W, const int kl[2], const V3<R>& n,
                                                    R penetration, const IslMove<R>& mv, V3<R> lin[2], V3<R> ang[2],
                                                    R (&st)[2][7]) {
  const int l1 = kl[1] >= 0 ? kl[1] : kl[0];
#pragma unroll
  for (int q = 0; q < 7; ++q) st[0][q] = W.st[kIslSt * kl[0] + q];
#pragma unroll
  for (int q = 0; q < 7; ++q) st[1][q] = W.st[kIslSt * l1 + q];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    lin[i] = V3<R>{R(0), R(0), R(0)};
    ang[i] = V3<R>{R(0), R(0), R(0)};
    if (i == 1 && kl[1] < 0) continue;
    R sign = R(1);
    if (i != 0) sign = R(-1);
    R angM = sign * penetration * mv.ra[i];
    R linM = sign * penetration * mv.rl[i];
    const R maxMagnitude = mv.mm[i];
    if (angM < -maxMagnitude) {
      R totalMove = angM + linM;
      angM = -maxMagnitude;
      linM = totalMove - angM;
    } else if (angM > maxMagnitude) {
      R totalMove = angM + linM;
      angM = maxMagnitude;
      linM = totalMove - angM;
    }
    if (angM != R(0)) ang[i] = mul(mv.td[i], angM / mv.ai[i]);
    lin[i] = mul(n, linM);
    if (i == 1 && kl[1] == kl[0])  // a body against itself: from what the first side left
#pragma unroll
      for (int q = 0; q < 7; ++q) st[1][q] = st[0][q];
    const V3<R> pos = add_scaled(V3<R>{st[i][0], st[i][1], st[i][2]}, n, linM);
    Q4<R> q{st[i][3], st[i][4], st[i][5], st[i][6]};
    q = q_add_scaled_vector(q, ang[i], R(1));
    q = q_normalize(q);
    st[i][0] = pos.x; st[i][1] = pos.y; st[i][2] = pos.z;
    st[i][3] = q.w; st[i][4] = q.x; st[i][5] = q.y; st[i][6] = q.z;
  }
}

// World inverse inertia and inverse mass of a contact's bodies, from the LDS
// table where the launch has one.
template <typename R, int T>
__device__ __forceinline__ void isl_inertia(const Bodies<R>& b, const IslWorld<R, T>& W, const int kl[2], R (&iw)[2][9],
                                            R im[2]) {
  if (W.iw) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const R* e = W.iw + kIslIw * (kl[i] >= 0 ? kl[i] : kl[0]);
#pragma unroll
      for (int q = 0; q < 9; ++q) iw[i][q] = e[q];
      im[i] = e[9];
    }
  } else {
    const int kb[2] = {W.b0w + kl[0], kl[1] >= 0 ? W.b0w + kl[1] : -1};
    body_inertia(b, kb, iw, im);
  }
}

// The derived data of the sleeping bodies of `red` (bit i: kl[i]), from the
// state just stored, to HBM and to the table (rare, and large: one copy of the
// code).
template <typename R, int T>
__device__ __forceinline__ void isl_rederive(const Bodies<R>& b, const IslWorld<R, T>& W, const int kl[2], uint32_t red) {
#pragma unroll 1
  for (int i = 0; i < 2 && red; ++i) {
    if (!(red >> i & 1u)) continue;
    const int l = i == 0 ? kl[0] : kl[1];
    R* e = W.st + kIslSt * l;
    Q4<R> q{e[3], e[4], e[5], e[6]};
    R iw[9];
    rederive(b, W.b0w + l, tab3(e), q, 0, iw);
    e[3] = q.w;
    e[4] = q.x;
    e[5] = q.y;
    e[6] = q.z;
    if (W.iw) {
#pragma unroll
      for (int k = 0; k < 9; ++k) W.iw[kIslIw * l + k] = iw[k];
    }
  }
}
// Contacts of a body whose derived data changed take their part of it again.
// Out of the table that is a few LDS reads; from HBM, where the store has to be
// waited for as well, such an iteration takes three times as long (3.6 us).
template <typename R, int T>
__device__ __forceinline__ void isl_move_again(const Bodies<R>& b, const IslWorld<R, T>& W, const int jb[2],
                                               const V3<R>& n, const V3<R> rel[2], IslMove<R>& mv) {
  R iw[2][9], im[2];
  if (W.iw) {
    isl_inertia(b, W, jb, iw, im);
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int l = W.b0w + opaque_lane(jb[i] >= 0 ? jb[i] : jb[0]);
      const volatile R* src = b.iit_world + l;
#pragma unroll
      for (int q = 0; q < 9; ++q) iw[i][q] = src[q * b.stride];
      im[i] = b.inv_mass[l];
    }
  }
  isl_move_of(jb[1] >= 0, n, rel, iw, im, mv);
}

// matchAwakeState (contact.go:185-202) on the flag table, in two parts: the
// flags of a contact's bodies, read with the rest of what a correction needs,
// and the store.  The motion a woken body gets is written when the phase ends
// (isl_commit).  The result has bit i for a body i that stays asleep.
struct IslAwake {
  uint8_t f0, f1;
};
template <typename R, int T>
__device__ __forceinline__ IslAwake isl_awake_of(const IslWorld<R, T>& W, const int kl[2]) {
  return IslAwake{W.fl[kl[0]], W.fl[kl[1] >= 0 ? kl[1] : kl[0]]};
}
template <typename R, int T>
__device__ __forceinline__ uint32_t isl_match_awake(const IslWorld<R, T>& W, const int kl[2], IslAwake f, bool store) {
  const bool a0 = (f.f0 & F_AWAKE) != 0, a1 = (f.f1 & F_AWAKE) != 0;
  if (kl[1] < 0) return a0 ? 0u : 1u;
  if (a0 != a1 && store) W.fl[a0 ? kl[1] : kl[0]] = uint8_t((a0 ? f.f1 : f.f0) | F_AWAKE);
  return a0 || a1 ? 0u : 3u;
}

// calculateDesiredDeltaVelocity (contact.go:87-112) from the products of
// lastFrameAccelleration * dt with the normal (d0, d1), which the phase does
// not change, and the flags, which it does.
template <typename R>
__device__ __forceinline__ R isl_desired_dv(IslAwake f, bool has1, R d0, R d1, R cvx, R e) {
  R vfa = R(0);
  if (f.f0 & F_AWAKE) vfa += d0;
  if (has1 && (f.f1 & F_AWAKE)) vfa -= d1;
  R restitution = e;
  if (dabs(cvx) < R(0.25)) restitution = R(0);
  return -cvx - restitution * (cvx - vfa);
}

// The two bodies' changes through LDS: written by the owner, read by the
// group (u: rotation or angular, v: velocity or linear).
template <typename R>
__device__ __forceinline__ void isl_put(R* x, const V3<R> v[2], const V3<R> u[2]) {
  x[0] = v[0].x; x[1] = v[0].y; x[2] = v[0].z; x[3] = u[0].x; x[4] = u[0].y; x[5] = u[0].z;
  x[6] = v[1].x; x[7] = v[1].y; x[8] = v[1].z; x[9] = u[1].x; x[10] = u[1].y; x[11] = u[1].z;
}
// the change of side d (0: the selected contact's body 0)
template <typename R>
__device__ __forceinline__ void isl_get(const R* x, int d, V3<R>& v, V3<R>& u) {
  x += 6 * d;
  v = V3<R>{x[0], x[1], x[2]};
  u = V3<R>{x[3], x[4], x[5]};
}

// What a correction of the bodies kl (their changes at x: velocity and
// rotation) does to the closing velocity of a contact of the bodies jb: side 0,
// then side 1.  Both terms are computed whatever the sides are: they overlap,
// where under conditions each would wait for its own reads.  Returns whether
// the contact is touched.
template <typename R>
__device__ __forceinline__ bool isl_touch_velocity(const R* x, const int jb[2], const int kl[2], const R* m9,
                                                   const V3<R> rel[2], V3<R>& cv) {
  const bool h0 = jb[0] >= 0 && (jb[0] == kl[0] || jb[0] == kl[1]);
  const bool h1 = jb[1] >= 0 && (jb[1] == kl[0] || jb[1] == kl[1]);
  V3<R> v0, u0, v1, u1;
  isl_get(x, jb[0] == kl[0] ? 0 : 1, v0, u0);
  isl_get(x, jb[1] == kl[0] ? 0 : 1, v1, u1);
  const V3<R> t0 = m3tv(m9, add(cross(u0, rel[0]), v0));
  const V3<R> t1 = mul(m3tv(m9, add(cross(u1, rel[1]), v1)), R(-1));
  cv = sel3(h0, add(cv, t0), cv);
  cv = sel3(h1, add(cv, t1), cv);
  return h0 || h1;
}
// The same for a penetration (changes: linear and angular moves).
template <typename R>
__device__ __forceinline__ void isl_touch_position(const R* x, const int jb[2], const int kl[2], const V3<R>& n,
                                                   const V3<R> rel[2], R& key) {
  const bool h0 = jb[0] >= 0 && (jb[0] == kl[0] || jb[0] == kl[1]);
  const bool h1 = jb[1] >= 0 && (jb[1] == kl[0] || jb[1] == kl[1]);
  V3<R> v0, u0, v1, u1;
  isl_get(x, jb[0] == kl[0] ? 0 : 1, v0, u0);
  isl_get(x, jb[1] == kl[0] ? 0 : 1, v1, u1);
  const R t0 = dot(add(cross(u0, rel[0]), v0), n) * R(-1);
  const R t1 = dot(add(cross(u1, rel[1]), v1), n);
  key = h0 ? key + t0 : key;
  key = h1 ? key + t1 : key;
}

// applyVelocityChange (contact.go:448-494) by the lane that owns the
// selected contact, the bodies' velocity and rotation in the tables; their
// new velocity and rotation come back in nv, nw.
template <typename R, int KIND, int T>
__device__ __forceinline__ void isl_velocity_change(const IslWorld<R, T>& W, const int kl[2], const V3<R> rel[2],
                                                    const R* c2w, R ddv, const V3<R>& cvel, const R* imp,
                                                    const R (&iw)[2][9], const R im[2], V3<R> vc[2], V3<R> rc[2],
                                                    V3<R> nv[2], V3<R> nw[2], R friction) {
  // the bodies' state first: its reads overlap with what follows
  const R* e0 = W.st + kIslSt * kl[0];
  const R* e1 = W.st + kIslSt * (kl[1] >= 0 ? kl[1] : kl[0]);
  const V3<R> v0 = tab3(e0), w0 = tab3(e0 + 3), v1 = tab3(e1), w1 = tab3(e1 + 3);
  V3<R> ic;
  if (KIND == KIND_MAT && friction == R(0))
    ic = V3<R>{ddv / imp[0], R(0), R(0)};
  else
    ic = friction_impulse_from(imp, imp + 9, ddv, cvel, friction);
  const V3<R> impulse = m3v(c2w, ic);
  const V3<R> zero{R(0), R(0), R(0)};
  V3<R> torque = cross(rel[0], impulse);
  rc[0] = m3v(iw[0], torque);
  vc[0] = add_scaled(zero, impulse, im[0]);
  rc[1] = vc[1] = nv[1] = nw[1] = zero;
  nv[0] = add(v0, vc[0]);
  nw[0] = add(w0, rc[0]);
  if (kl[1] >= 0) {
    torque = cross(impulse, rel[1]);
    rc[1] = m3v(iw[1], torque);
    vc[1] = add_scaled(zero, impulse, -im[1]);
    nv[1] = add(v1, vc[1]);
    nw[1] = add(w1, rc[1]);
  }
}

__device__ __forceinline__ uint32_t isl_ids(int c0, int c1, int b0w) {
  return uint32_t(c0 - b0w) | (uint32_t(c1 >= 0 ? c1 - b0w : int(kNoBody)) << 16);
}

// adjustPositions (contact.go:233-283) on islands k0 .. of one class, one
// contact per lane.
template <typename R, int KIND, int T>
__device__ __forceinline__ void isl_pos_batch(const RS<R>& a, const IslWorld<R, T>& W, const IslPass& P, int lg, int k0, int kend, R eps,
                              R& kmin) {
  const Contacts<R>& c = a.c;
  const int64_t CS = c.cap;
  const int lane = W.t & 63, wave = W.t >> 6, grp = lane >> lg, li = lane & ((1 << lg) - 1);
  const int k = k0 + grp;
  bool live = k < kend && !(P.pass != ISL_FREE && a.isl_its[W.b0w + k] < 0);
  const int cnt = !live ? 0 : P.one ? W.C : a.isl_cnt[W.b0w + k];
  const bool has = li < cnt;
  int j = INT_MAX;
  R key = R(0);
  uint32_t id = 0xFFFFFFFFu;
  V3<R> n{R(0), R(0), R(0)}, rel[2] = {n, n};
  IslMove<R> mv{};
  if (has) {
    j = P.one ? li : a.isl_idx[W.base + a.isl_off[W.b0w + k] + li];
    const int64_t g = W.base + j;
    const int c0 = c.body0[g], c1 = c.body1[g];
    id = isl_ids(c0, c1, W.b0w);
    rec_normal(c.rec + 16 * g, n, rel);
    const int kl[2] = {id_lo(id), id_hi(id)};
    R iw[2][9], im[2];
    isl_inertia(a.b, W, kl, iw, im);
    isl_move_of(c1 >= 0, n, rel, iw, im, mv);
    if (P.pass == ISL_FREE) {
      key = c.pen[g];
      if (!P.saved) a.isl_save[4 * CS + g] = key;
    } else {
      key = a.isl_save[4 * CS + g];
    }
  }
  const int64_t lim = P.pass == ISL_LIMIT ? (live ? int64_t(a.isl_its[W.b0w + k]) : 0) : P.budget;
  int64_t logat = P.pass == ISL_LOG && live ? a.isl_log[W.b0w + k] : 0;
  R* x = W.f->x[wave][grp];
  volatile uint32_t* xi = W.f->xi[wave][grp];
  const uint64_t gm = group_lanes(lg);
  const int jb[2] = {id_lo(id), id_hi(id)};
  int it = 0, nrec = 0;
  R runmin = R(__builtin_inf());
  bool over = false;
  while (true) {
    const R kk = (has && live && key > eps) ? key : R(-__builtin_inf());
    const R m = group_reduce(kk, lg, [](R p, R q) { return q > p ? q : p; });
    const bool any = m > R(-__builtin_inf());
    const bool top = group_owner<R>(any && kk == m, j, lg, gm);
    live = live && any;
    if (live && it >= lim) {
      over = true;
      live = false;
    }
    if (!__any(live)) break;
    const bool owner = live && top;
    if (P.pass == ISL_LOG && live && (nrec == 0 || m <= runmin)) {
      runmin = m;
      if (owner) isl_log(a, logat + nrec, m, j, it);
      ++nrec;
    }
    if (owner) {
      const int kl[2] = {jb[0], jb[1]};
      const IslAwake f = isl_awake_of(W, kl);
      V3<R> lin[2], ang[2];
      R st[2][7];
      isl_position_change(W, kl, n, key, mv, lin, ang, st);
      isl_put(x, lin, ang);
      const uint32_t red = isl_match_awake(W, kl, f, true);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (kl[i] < 0) continue;
#pragma unroll
        for (int q = 0; q < 7; ++q) W.st[kIslSt * kl[i] + q] = st[i][q];
      }
      if (red) {
        // opaque: the addresses of the rare sleeping body's data are computed
        // here and not kept for the whole loop
        const int ko[2] = {opaque_lane(kl[0]), opaque_lane(kl[1])};
        isl_rederive(a.b, W, ko, red);
      }
      xi[0] = id;
      xi[1] = red;
      if constexpr (KIND == KIND_LABEL)
        if (P.pass != ISL_LOG) add_pos_label(a, W.base + j, key);
    }
    wave_fence();
    const uint32_t kid = xi[0], red = xi[1];
    const int kl[2] = {id_lo(kid), id_hi(kid)};
    R p = key;
    isl_touch_position(x, jb, kl, n, rel, p);
    key = live ? p : key;
    it += live ? 1 : 0;
    // a sleeping body's new world inverse inertia
    if (__any(live && red != 0)) {
      if (!W.iw) __threadfence_block();
      bool hit = false;
#pragma unroll
      for (int bb = 0; bb < 2; ++bb)
        hit |= jb[bb] >= 0 && ((jb[bb] == kl[0] && (red & 1)) || (jb[bb] == kl[1] && (red & 2)));
      if (live && has && hit) isl_move_again(a.b, W, jb, n, rel, mv);
    }
    wave_fence();
  }
  if (has && P.pass != ISL_LOG) {
    c.pen[W.base + j] = key;
    kmin = key < kmin ? key : kmin;
  }
  isl_count(a, W, P, k, k < kend && li == 0, it, nrec, over, runmin);
}

// Checkpoint q (2 or 3) of a small island in the velocity phase: the contact's
// key and closing velocity where a big island's impulse data would be, its
// bodies' velocity, rotation and flag where the position phase kept the
// sleepers.  SAVE, or back.
template <typename R, bool SAVE, int T>
__device__ __forceinline__ void isl_checkpoint(const RS<R>& a, const IslWorld<R, T>& W, int j, const int jb[2], int q,
                                               R& key, V3<R>& cv) {
  const int64_t S = a.b.stride;
  R* e = a.c.imp + kImpPlanes * (W.base + j) + 4 * (q - 2);
  if constexpr (SAVE) {
    e[0] = key, e[1] = cv.x, e[2] = cv.y, e[3] = cv.z;
  } else {
    key = e[0];
    cv = V3<R>{e[1], e[2], e[3]};
  }
#pragma unroll 1
  for (int i = 0; i < 2; ++i) {
    const int l = opaque_lane(i == 0 ? jb[0] : jb[1]);
    if (l < 0) continue;
    R* p = a.isl_snap + W.b0w + l + 7 * (q - 2) * S;
#pragma unroll 1
    for (int k = 0; k < 6; ++k) {
      if constexpr (SAVE)
        p[k * S] = W.st[kIslSt * l + k];
      else
        W.st[kIslSt * l + k] = p[k * S];
    }
    if constexpr (SAVE)
      p[6 * S] = R(W.fl[l]);
    else
      W.fl[l] = uint8_t(p[6 * S]);
  }
}

// adjustVelocities (contact.go:390-445) on islands k0 .. of one class, one
// contact per lane.
template <typename R, int KIND, int T>
__device__ __forceinline__ void isl_vel_batch(const RS<R>& a, const IslWorld<R, T>& W, const IslPass& P, int lg, int k0, int kend, R eps) {
  const Bodies<R>& b = a.b;
  const Contacts<R>& c = a.c;
  const int64_t CS = c.cap, S = b.stride;
  constexpr bool LATE = KIND != KIND_LABEL;
  const int lane = W.t & 63, wave = W.t >> 6, grp = lane >> lg, li = lane & ((1 << lg) - 1);
  const int k = k0 + grp;
  bool live = k < kend && !(P.pass != ISL_FREE && a.isl_its[W.b0w + k] < 0);
  const int cnt = !live ? 0 : P.one ? W.C : a.isl_cnt[W.b0w + k];
  const bool has = li < cnt;
  const V3<R> zero{R(0), R(0), R(0)};
  int j = INT_MAX;
  R key = R(0);
  uint32_t id = 0xFFFFFFFFu;
  V3<R> cv = zero, rel[2] = {zero, zero};
  R m9[9], imp[kImpPlanes], iw[2][9], im[2], d0 = R(0), d1 = R(0);
  R fr = R(kFriction), rs = R(kRestitution);
#pragma unroll
  for (int q = 0; q < 9; ++q) m9[q] = iw[0][q] = iw[1][q] = R(0);
#pragma unroll
  for (int q = 0; q < kImpPlanes; ++q) imp[q] = R(0);
  im[0] = im[1] = R(0);
  if (has) {
    j = P.one ? li : a.isl_idx[W.base + a.isl_off[W.b0w + k] + li];
    const int64_t g = W.base + j;
    const int c0 = c.body0[g], c1 = c.body1[g];
    id = isl_ids(c0, c1, W.b0w);
    rec_frame(c.rec + 16 * g, m9, rel);
    const int kb[2] = {c0, c1};
    body_inertia(b, kb, iw, im);
    if constexpr (KIND == KIND_MAT) {
      fr = c.fric[g];
      rs = c.rest[g];
    }
    impulse_data_from<R, KIND>(a.mode, iw[0], iw[1], im, c1 >= 0, rel, m9, fr, imp);
    const V3<R> nn{m9[0], m9[1], m9[2]};
    d0 = dot(mul(ld3(b.last_acc, S, c0), a.dt), nn);
    if (c1 >= 0) d1 = dot(mul(ld3(b.last_acc, S, c1), a.dt), nn);
    if (P.pass == ISL_FREE) {
      key = c.ddv[g];
      cv = ld3(c.cvel, CS, g);
      if (!P.saved) {
        st3(a.isl_save, CS, g, cv);
        a.isl_save[3 * CS + g] = key;
      }
    } else {
      key = a.isl_save[3 * CS + g];
      cv = ld3(a.isl_save, CS, g);
    }
  }
  int lim = P.pass == ISL_LIMIT ? (live ? a.isl_its[W.b0w + k] : 0) : int(P.budget);
  int64_t logat = P.pass == ISL_LOG && live ? a.isl_log[W.b0w + k] : 0;
  if (LATE && P.pass == ISL_LOG && P.late > 0 && live && isl_is_late(a.isl_nrec[W.b0w + k])) {
    lim = P.late;  // what the free pass did not log
    ++logat;
  }
  R* x = W.f->x[wave][grp];
  volatile uint32_t* xi = W.f->xi[wave][grp];
  const uint64_t gm = group_lanes(lg);
  const int jb[2] = {id_lo(id), id_hi(id)};
  bool logs = P.pass == ISL_LOG;  // the wave's islands log
  int it = 0, nrec = logs ? 0 : -1;  // records: -1 as long as the island does not
  R runmin = R(__builtin_inf());
  bool over = false;
  if constexpr (LATE) {
    if (P.pass == ISL_FREE && P.late > 0) lim = P.late;  // where something is kept, and on from there
    if (P.pass == ISL_LIMIT && P.late > 0) {
      const int q = live ? min((lim - 1) / P.late, 3) : 0;
      if (q > 1) {
        it = q * P.late;
        if (has) isl_checkpoint<R, false>(a, W, j, jb, q, key, cv);
      }
      wave_fence();
    }
  }
  while (true) {
    const R kk = (has && live && key > eps) ? key : R(-__builtin_inf());
    const R m = group_reduce(kk, lg, [](R p, R q) { return q > p ? q : p; });
    const bool any = m > R(-__builtin_inf());
    const bool top = group_owner<R>(any && kk == m, j, lg, gm);
    live = live && any;
    const bool stop = live && it >= lim;
    if (__any(stop)) {
      if (LATE && P.pass == ISL_FREE && P.late > 0 && __any(stop && it < int(P.budget))) {
        // every live island of the wave has made as many iterations
        if (stop && it > P.late) {
          if (has) isl_checkpoint<R, true>(a, W, j, jb, it / P.late, key, cv);
        } else if (stop) {
          if (li == 0)
            logat = atomicAdd(&W.f->lates, 1) < kIslLates ? isl_reserve(a, 1 + P.late + isl_late_records(P.budget)) : -1;
        }
        if (!logs) {
          logs = true;
          logat = __shfl(logat, grp << lg, 64);
          if (stop && logat >= 0) {
            if (li == 0) a.isl_log[W.b0w + k] = logat;
            logat += 1 + P.late;
            nrec = 0;
          }
        }
        lim = it < 3 * P.late ? it + P.late : int(P.budget);
      } else if (stop) {
        over = true;
        live = false;
      }
    }
    if (!__any(live)) break;
    const bool owner = live && top;
    if (logs && live && m <= runmin) {
      runmin = m;
      if (LATE && P.pass == ISL_FREE && nrec >= isl_late_records(P.budget)) {
        nrec = -1;  // no room for more: no log
      } else if (nrec >= 0) {
        if (owner) isl_log(a, logat + nrec, m, j, it);
        ++nrec;
      }
    }
    if (owner) {
      const int kl[2] = {jb[0], jb[1]};
      const IslAwake f = isl_awake_of(W, kl);
      V3<R> vc[2], rc[2], nv[2], nw[2];
      isl_velocity_change<R, KIND>(W, kl, rel, m9, key, cv, imp, iw, im, vc, rc, nv, nw, fr);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (kl[i] < 0) continue;
        tab3_store(W.st + kIslSt * kl[i], nv[i]);
        tab3_store(W.st + kIslSt * kl[i] + 3, nw[i]);
      }
      isl_match_awake(W, kl, f, true);
      isl_put(x, vc, rc);
      xi[0] = id;
      if constexpr (KIND == KIND_LABEL)
        if (P.pass != ISL_LOG) add_label(a, W.base + j, vc, rc);
    }
    wave_fence();
    const uint32_t kid = xi[0];
    // a lane without a contact has no bodies: it reads the first one's flags
    const int kl[2] = {id_lo(kid), id_hi(kid)}, jo[2] = {has ? jb[0] : 0, jb[1]};
    const IslAwake f = isl_awake_of(W, jo);
    V3<R> cn = cv;
    if (isl_touch_velocity(x, jb, kl, m9, rel, cn) && live) {
      cv = cn;
      key = isl_desired_dv(f, jb[1] >= 0, d0, d1, cn.x, rs);
    }
    it += live ? 1 : 0;
    wave_fence();
  }
  if (has && P.pass != ISL_LOG) {
    c.ddv[W.base + j] = key;
    st3(c.cvel, CS, W.base + j, cv);
  }
  isl_count(a, W, P, k, k < kend && li == 0, it, nrec, over, runmin);
}

// A contact's impulse data (Contacts::imp), in 16-byte accesses.
template <typename R>
__device__ __forceinline__ void isl_imp_store(R* q, const R (&v)[kImpPlanes]) {
  if constexpr (sizeof(R) == 4) {
    float4* p = reinterpret_cast<float4*>(q);
#pragma unroll
    for (int i = 0; i < 3; ++i) p[i] = float4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
  } else {
    double2* p = reinterpret_cast<double2*>(q);
#pragma unroll
    for (int i = 0; i < 6; ++i) p[i] = double2{v[2 * i], v[2 * i + 1]};
  }
}
template <typename R>
__device__ __forceinline__ void isl_imp_load(const R* q, R (&v)[kImpPlanes]) {
  if constexpr (sizeof(R) == 4) {
    const float4* p = reinterpret_cast<const float4*>(q);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const float4 x = p[i];
      v[4 * i] = x.x;
      v[4 * i + 1] = x.y;
      v[4 * i + 2] = x.z;
      v[4 * i + 3] = x.w;
    }
  } else {
    const double2* p = reinterpret_cast<const double2*>(q);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const double2 x = p[i];
      v[2 * i] = x.x;
      v[2 * i + 1] = x.y;
    }
  }
}

// The same for one island of more than 64 contacts on the whole workgroup:
// thread t holds contacts t + 256 s of the island's list (s < SL).  With one
// contact per thread everything is in registers, as in the batches; with two,
// the impulse data come from HBM (written when the island is loaded) and the
// bodies' inertia from an LDS table where the launch has one; with eight, the
// records from HBM too.  An iteration has one barrier, after the waves' best
// contacts and the corrections these would make (two more where a sleeping
// body's derived data change).
template <typename R, int KIND, bool VEL, int SL, int T>
__device__ __forceinline__ void isl_big(const RS<R>& a, const IslWorld<R, T>& W, const IslPass& P, int k, bool last, R eps,
                                        R& kmin) {
  const Bodies<R>& b = a.b;
  const Contacts<R>& c = a.c;
  const int64_t CS = c.cap, S = b.stride;
  const int t = W.t, wave = t >> 6;
  const int cnt = P.one ? W.C : a.isl_cnt[W.b0w + k];
  const int32_t* idx = a.isl_idx + W.base + (P.one ? 0 : a.isl_off[W.b0w + k]);
  const V3<R> zero{R(0), R(0), R(0)};
  constexpr bool REG = SL == 1;
  constexpr bool MOVE = !VEL && SL <= 2;  // what a position change keeps is in registers
  IslMove<R> mv[MOVE ? SL : 1];
  const bool resume = VEL && k == P.resume;
  if (P.pass != ISL_FREE && a.isl_its[W.b0w + k] < 0) return;
  R rimp[kImpPlanes], riw[2][9], rim[2];  // REG
  constexpr bool REC = SL <= 2;           // the records are in registers
  R rm[REC ? SL : 1][9];
  V3<R> rrel[REC ? SL : 1][2];
  R key[SL];
  uint32_t js[SL];
  uint32_t ids[SL];
  V3<R> cv[VEL ? SL : 1];
  // lastFrameAccelleration * dt along the normal, both bodies (8 contacts per
  // thread: not kept, no registers left)
  constexpr bool DN = VEL && SL <= 2;
  R dn[DN ? SL : 1][2];
  constexpr bool MAT = VEL && KIND == KIND_MAT && SL <= 2;
  R fr[MAT ? SL : 1], rs[MAT ? SL : 1];
#pragma unroll
  for (int s = 0; s < SL; ++s) {
    key[s] = R(0);
    js[s] = uint32_t(INT_MAX);
    ids[s] = 0xFFFFFFFFu;
    if constexpr (VEL) {
      cv[s] = zero;
      if constexpr (DN) dn[s][0] = dn[s][1] = R(0);
      if constexpr (MAT) fr[s] = rs[s] = R(0);
    }
    if (T * s + t >= cnt) continue;
    asm volatile("" ::: "memory");
    js[s] = uint32_t(P.one ? T * s + t : idx[T * s + t]);
    const int64_t g = W.base + int(js[s]);
    const int c0 = c.body0[g], c1 = c.body1[g];
    ids[s] = isl_ids(c0, c1, W.b0w);
    if constexpr (MAT) {
      fr[s] = c.fric[g];
      rs[s] = c.rest[g];
    }
    if constexpr (MOVE) {
      rec_frame(c.rec + 16 * g, rm[s], rrel[s]);
      const int kl[2] = {id_lo(ids[s]), id_hi(ids[s])};
      R iw[2][9], im[2];
      isl_inertia(b, W, kl, iw, im);
      isl_move_of(c1 >= 0, V3<R>{rm[s][0], rm[s][1], rm[s][2]}, rrel[s], iw, im, mv[s]);
    }
    if constexpr (VEL) {
      R mj[9];
      V3<R> rj[2];
      rec_frame(c.rec + 16 * g, mj, rj);
      const int kb[2] = {c0, c1};
      if constexpr (REC) {
#pragma unroll
        for (int q = 0; q < 9; ++q) rm[s][q] = mj[q];
        rrel[s][0] = rj[0];
        rrel[s][1] = rj[1];
      }
      if constexpr (REG) {
        body_inertia(b, kb, riw, rim);
        impulse_data_from<R, KIND>(a.mode, riw[0], riw[1], rim, c1 >= 0, rj, mj, friction_of<R, KIND>(c, g), rimp);
      }
      if constexpr (DN) {
        const V3<R> nj{mj[0], mj[1], mj[2]};
        dn[s][0] = dot(mul(ld3(b.last_acc, S, c0), a.dt), nj);
        if (c1 >= 0) dn[s][1] = dot(mul(ld3(b.last_acc, S, c1), a.dt), nj);
      }
      if (P.pass == ISL_FREE || resume) {
        key[s] = c.ddv[g];
        cv[s] = ld3(c.cvel, CS, g);
        if (P.pass == ISL_FREE && !P.saved) {
          st3(a.isl_save, CS, g, cv[s]);
          a.isl_save[3 * CS + g] = key[s];
        }
        if constexpr (!REG) {
          if (P.pass == ISL_FREE) {
            R imp[kImpPlanes];
            impulse_data<R, KIND>(a, kb, rj, mj, friction_of<R, KIND>(c, g), imp);
            isl_imp_store(c.imp + kImpPlanes * g, imp);
          }
        }
      } else {
        key[s] = a.isl_save[3 * CS + g];
        cv[s] = ld3(a.isl_save, CS, g);
      }
    } else {
      if (P.pass == ISL_FREE) {
        key[s] = c.pen[g];
        if (!P.saved) a.isl_save[4 * CS + g] = key[s];
      } else {
        key[s] = a.isl_save[4 * CS + g];
      }
    }
  }
  // the owner of a contact reads the impulse data it wrote itself
  const bool pause = VEL && P.pause && last;
  int64_t lim = P.pass == ISL_LIMIT ? int64_t(a.isl_its[W.b0w + k]) : P.budget;
  if (pause) {  // what the other islands left of the budget
    const int64_t left = P.budget - int64_t(W.f->total);
    lim = left > 0 ? left : 0;
  }
  const int64_t logat = P.pass == ISL_LOG ? a.isl_log[W.b0w + k] : 0;
  int par = 0;
  int it = resume ? W.f->at : 0, nrec = 0;
  R runmin = resume ? W.f->runkey : R(__builtin_inf());
  int runj = resume ? W.f->runj : INT_MAX;
  int jm = INT_MAX;
  __syncthreads();  // the pause's words are read, the island before is done
  while (true) {
    opaque_ids(ids);
    opaque_ids(js);
    R best = R(-__builtin_inf());
    int bj = INT_MAX, bs = 0;
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      const bool up = key[s] > eps && (key[s] > best || (key[s] == best && int(js[s]) < bj));
      best = up ? key[s] : best;
      bj = up ? int(js[s]) : bj;
      bs = up ? s : bs;
    }
    const R wm = group_reduce(best, 6, [](R p, R q) { return q > p ? q : p; });
    // the lowest index among the lanes with that key: one lane, as a rule
    const unsigned long long tie = __ballot(bj != INT_MAX && best == wm);
    int wj = __builtin_amdgcn_readlane(bj, tie ? __builtin_ctzll(tie) : 0);
    if (tie & (tie - 1)) wj = group_reduce(bj != INT_MAX && best == wm ? bj : INT_MAX, 6, [](int p, int q) { return q < p ? q : p; });
    IslBest<R>* bb4 = W.f->best[par];
    if (tie ? bj == wj : (t & 63) == 0) bb4[wave] = IslBest<R>{wm, tie ? wj : INT_MAX, pick(ids, bs)};
    // The best of the waves' best, in each quad of lanes: before the corrections
    // in the launches that fill the chip (narrow workgroups), where those of the
    // other waves would cost others their turns, and after them else.
    constexpr bool FULL = T < kIslThreads;
    int bw = 0;
    R m = R(0);
    uint32_t kid = 0;
    auto winner = [&]() {
      static_assert(T / 64 <= 4, "a quad holds one offer per wave");
      const IslBest<R> e = bb4[t & ((T / 64) - 1)];
      m = group_reduce(e.key, 2, [](R p, R q) { return q > p ? q : p; });
      jm = __builtin_amdgcn_readfirstlane(
          group_reduce(e.key == m ? e.j : INT_MAX, 2, [](int p, int q) { return q < p ? q : p; }));
      bw = __builtin_ctzll(__ballot(e.j == jm)) & ((T / 64) - 1);
      kid = uint32_t(__builtin_amdgcn_readlane(int(e.id), bw));
    };
    if constexpr (FULL) {
      __syncthreads();
      winner();
      if (jm == INT_MAX || it >= lim) break;
    }
    const bool mine = FULL ? bj == jm : tie && bj == wj;
    if constexpr (VEL) {
      // else every wave's best contact computes its correction, the winner's is
      // taken: the other waves would wait
      if (mine) {
        const uint32_t id = pick(ids, bs);
        const int64_t g = W.base + wj;
        const int kl[2] = {id_lo(id), id_hi(id)};
        V3<R> v[2], u[2], nv[2], nw[2];
        R fk;
        if constexpr (MAT)
          fk = pick(fr, bs);
        else
          fk = friction_of<R, KIND>(c, g);
        if constexpr (REG) {
          isl_velocity_change<R, KIND>(W, kl, rrel[0], rm[0], wm, cv[0], rimp, riw, rim, v, u, nv, nw, fk);
        } else {
          R iw[2][9], im[2], mj[9], imp[kImpPlanes];
          V3<R> rel[2];
          isl_imp_load(c.imp + kImpPlanes * g, imp);
          isl_inertia(b, W, kl, iw, im);
          if constexpr (REC) {
#pragma unroll
            for (int q = 0; q < 9; ++q) mj[q] = bs ? rm[SL - 1][q] : rm[0][q];
            rel[0] = sel3(bs != 0, rrel[SL - 1][0], rrel[0][0]);
            rel[1] = sel3(bs != 0, rrel[SL - 1][1], rrel[0][1]);
          } else {
            rec_frame(c.rec + 16 * g, mj, rel);
          }
          isl_velocity_change<R, KIND>(W, kl, rel, mj, wm, pick(cv, bs), imp, iw, im, v, u, nv, nw, fk);
        }
        isl_put(W.f->bx[par][wave], v, u);
        isl_put(W.f->bx[par][wave] + 12, nv, nw);
      }
    } else if (mine) {
      const uint32_t id = pick(ids, bs);
      const int kl[2] = {id_lo(id), id_hi(id)};
      V3<R> v[2], u[2], nj;
      R st[2][7];
      IslMove<R> mj;
      if constexpr (MOVE) {
        nj = sel3(bs != 0, V3<R>{rm[SL - 1][0], rm[SL - 1][1], rm[SL - 1][2]}, V3<R>{rm[0][0], rm[0][1], rm[0][2]});
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          mj.ai[i] = bs ? mv[SL - 1].ai[i] : mv[0].ai[i];
          mj.ra[i] = bs ? mv[SL - 1].ra[i] : mv[0].ra[i];
          mj.rl[i] = bs ? mv[SL - 1].rl[i] : mv[0].rl[i];
          mj.mm[i] = bs ? mv[SL - 1].mm[i] : mv[0].mm[i];
          mj.td[i] = sel3(bs != 0, mv[SL - 1].td[i], mv[0].td[i]);
        }
      } else {
        R iw[2][9], im[2], m9[9];
        V3<R> rel[2];
        rec_frame(c.rec + 16 * (W.base + wj), m9, rel);
        isl_inertia(b, W, kl, iw, im);
        nj = V3<R>{m9[0], m9[1], m9[2]};
        isl_move_of(kl[1] >= 0, nj, rel, iw, im, mj);
      }
      isl_position_change(W, kl, nj, pick(key, bs), mj, v, u, st);
      R* o = W.f->bx[par][wave];
      isl_put(o, v, u);
#pragma unroll
      for (int q = 0; q < 7; ++q) {
        o[12 + q] = st[0][q];
        o[19 + q] = st[1][q];
      }
    }
    __syncthreads();
    if constexpr (!FULL) {
      winner();
      if (jm == INT_MAX || it >= lim) break;
    }
    const int kl[2] = {id_lo(kid), id_hi(kid)};
    const bool owner = bj == jm;
    const bool low = m <= runmin;
    if (low) {
      runmin = m;
      runj = jm;
    }
    if (P.pass == ISL_LOG && (nrec == 0 || low)) {
      if (owner) isl_log(a, logat + nrec, runmin, runj, it);
      ++nrec;
    }
    // Every wave stores the bodies' new state and the woken body's flag (the
    // same values), so each reads its own stores in the next iteration and
    // one barrier per iteration is enough; the offers alternate between two
    // sets.
    const R* x = W.f->bx[par][bw];
    constexpr int NS = VEL ? 6 : 7;
    const int l = t & 63;
    const IslAwake fa = isl_awake_of(W, kl);
    if (l < NS) {
      if (kl[0] != kl[1]) W.st[kIslSt * kl[0] + l] = x[12 + l];
    } else if (l < 2 * NS && kl[1] >= 0) {
      W.st[kIslSt * kl[1] + l - NS] = x[12 + l];
    }
    const uint32_t red = isl_match_awake(W, kl, fa, l == 0);
    if constexpr (KIND == KIND_LABEL) {
      if (owner && P.pass != ISL_LOG) {
        if constexpr (VEL) {
          const V3<R> v[2] = {V3<R>{x[0], x[1], x[2]}, V3<R>{x[6], x[7], x[8]}};
          const V3<R> u[2] = {V3<R>{x[3], x[4], x[5]}, V3<R>{x[9], x[10], x[11]}};
          add_label(a, W.base + jm, v, u);
        } else {
          add_pos_label(a, W.base + jm, m);
        }
      }
    }
    wave_fence();
    if constexpr (!VEL) {
      // Another wave may have stored a woken body's flag before this one read
      // it; asleep it stays only if no wave wakes it, so all agree.
      if (__any(red != 0)) {
        __syncthreads();  // every wave has stored the state the owner now corrects
        if (owner) isl_rederive(b, W, kl, red);
        __syncthreads();
        if constexpr (MOVE) {
#pragma unroll
          for (int s = 0; s < SL; ++s) {
            const int jb[2] = {id_lo(ids[s]), id_hi(ids[s])};
            bool hit = false;
#pragma unroll
            for (int bb = 0; bb < 2; ++bb)
              hit |= jb[bb] >= 0 && ((jb[bb] == kl[0] && (red & 1)) || (jb[bb] == kl[1] && (red & 2)));
            if (hit) isl_move_again(b, W, jb, V3<R>{rm[s][0], rm[s][1], rm[s][2]}, rrel[s], mv[s]);
          }
        }
      }
    }
    par ^= 1;
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      if (T * s >= cnt) break;
      const int jb[2] = {id_lo(ids[s]), id_hi(ids[s])};
      bool hit = false;
#pragma unroll
      for (int bb = 0; bb < 2; ++bb) hit |= jb[bb] >= 0 && (jb[bb] == kl[0] || jb[bb] == kl[1]);
      if (!hit || js[s] == uint32_t(INT_MAX)) continue;
      R mj[9];
      V3<R> rj[2];
      if constexpr (REC) {
#pragma unroll
        for (int q = 0; q < 9; ++q) mj[q] = rm[s][q];
        rj[0] = rrel[s][0];
        rj[1] = rrel[s][1];
      } else {
        rec_frame(c.rec + 16 * (W.base + int(js[s])), mj, rj);
      }
      const V3<R> nj{mj[0], mj[1], mj[2]};
      if constexpr (VEL)
        isl_touch_velocity(x, jb, kl, mj, rj, cv[s]);
      else
        isl_touch_position(x, jb, kl, nj, rj, key[s]);
      if constexpr (VEL) {
        R d0, d1 = R(0);
        if constexpr (DN) {
          d0 = dn[s][0];
          d1 = dn[s][1];
        } else {
          d0 = dot(mul(ld3(b.last_acc, S, W.b0w + jb[0]), a.dt), nj);
          if (jb[1] >= 0) d1 = dot(mul(ld3(b.last_acc, S, W.b0w + jb[1]), a.dt), nj);
        }
        R e;
        if constexpr (MAT)
          e = rs[s];
        else
          e = restitution_of<R, KIND>(c, W.base + int(js[s]));
        key[s] = isl_desired_dv(isl_awake_of(W, jb), jb[1] >= 0, d0, d1, cv[s].x, e);
      }
    }
    ++it;
  }
  const bool over = jm != INT_MAX;  // the budget stopped it
  if (P.pass != ISL_LOG) {
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      if (js[s] == uint32_t(INT_MAX)) continue;
      const int64_t g = W.base + int(js[s]);
      if constexpr (VEL) {
        c.ddv[g] = key[s];
        st3(c.cvel, CS, g, cv[s]);
      } else {
        c.pen[g] = key[s];
        kmin = key[s] < kmin ? key[s] : kmin;
      }
    }
  }
  if (t == 0 && pause && over) {
    W.f->paused = k;
    W.f->at = it;
    W.f->runkey = runmin;
    W.f->runj = runj;
  }
  isl_count(a, W, P, k, t == 0, it, nrec, over, runmin);
  __syncthreads();  // the waves' best contacts are read, the counts made
}

// Every island of the world once: the waves take batches of the small ones in
// class order, then the whole workgroup the big ones, one after another, the
// one of the largest class last.
template <typename R, int KIND, bool VEL, int T>
__device__ __forceinline__ void isl_run(const RS<R>& a, const IslWorld<R, T>& W, const IslPass& P, R eps, R& kmin) {
  if (W.t == 0) {
    W.f->next = 0;
    if (P.pass == ISL_FREE) {
      W.f->total = 0;
      W.f->over = 0;
      W.f->paused = -1;
      W.f->lates = 0;
    }
  }
  if (W.t < kIslWords) W.f->cls[W.t] = a.isl_cls[kIslWords * int64_t(W.w) + W.t];
  __syncthreads();
  const int32_t* cls = W.f->cls;
  // islands of eight, of four and of two contacts per thread, and all big ones
  constexpr bool FOUR = T < 256;
  int n8 = cls[0] + (FOUR ? 0 : cls[1]), n4 = FOUR ? cls[1] : 0, n2 = cls[2], nbig = n8 + n4 + n2 + cls[3];
  if (P.one) {
    const int k = isl_class<T>(W.C);
    n8 = k == 0 || (!FOUR && k == 1) ? 1 : 0;
    n4 = FOUR && k == 1 ? 1 : 0;
    n2 = k == 2 ? 1 : 0;
    nbig = W.C > 64 ? 1 : 0;
  }
  if (W.iw && (!VEL || n8 + n4 + n2 > 0)) {
    for (int i = opaque_lane(W.t); i < W.n; i += T) {
      R iw[9];
      ld9(a.b.iit_world, a.b.stride, W.b0w + i, iw);
#pragma unroll
      for (int q = 0; q < 9; ++q) W.iw[kIslIw * i + q] = iw[q];
      W.iw[kIslIw * i + 9] = a.b.inv_mass[W.b0w + i];
    }
  }
  if constexpr (!VEL) __syncthreads();
  while (!P.only) {
    // One lane takes the wave's ticket.  Its index is opaque: with a branch that
    // is the same in every turn, the compiler makes the other lanes a loop of
    // their own, which never sees the first lane's value.
    int q = 0;
    if ((opaque_lane(W.t) & 63) == 0) q = atomicAdd(&W.f->next, 1);
    __builtin_amdgcn_wave_barrier();
    q = __builtin_amdgcn_readfirstlane(q);
    int at = nbig, k = kIslBigClasses, m = 0, per = 1, lg = 6;
    if (P.one) {
      if (q > 0 || W.C > 64) break;
      m = 1;
    }
    for (; !P.one && k < kIslClasses; ++k) {
      m = cls[k];
      lg = isl_class_lg(k);
      per = 64 >> lg;
      const int nb = (m + per - 1) >> (6 - lg);
      if (q < nb) break;
      q -= nb;
      at += m;
    }
    if (k == kIslClasses) break;
    if constexpr (VEL)
      isl_vel_batch<R, KIND>(a, W, P, lg, at + q * per, at + m, eps);
    else
      isl_pos_batch<R, KIND>(a, W, P, lg, at + q * per, at + m, eps, kmin);
  }
  __syncthreads();
  // ranks are in class order, the largest class first
  for (int i = nbig - 1; i >= 0; --i) {
    if (P.only ? i != P.resume : P.pass == ISL_LOG && i == P.resume) continue;
    const bool last = i == 0;
    if (i < n8) {
      isl_big<R, KIND, VEL, 8>(a, W, P, i, last, eps, kmin);
    } else if (i < n8 + n4) {
      if constexpr (FOUR) isl_big<R, KIND, VEL, 4>(a, W, P, i, last, eps, kmin);
    } else if (i < n8 + n4 + n2) {
      isl_big<R, KIND, VEL, 2>(a, W, P, i, last, eps, kmin);
    } else {
      isl_big<R, KIND, VEL, 1>(a, W, P, i, last, eps, kmin);
    }
  }
}

// ---------------------------------------------------------------------------
// a phase of a world
// ---------------------------------------------------------------------------
// The body tables as the phase starts.  (Here and below the thread index is
// opaque, so that the addresses of one loop over the bodies are not kept in
// registers through a phase for the next.)
template <typename R, bool VEL, int T>
__device__ __forceinline__ void isl_load(const RS<R>& a, const IslWorld<R, T>& W) {
  const Bodies<R>& b = a.b;
  const int64_t S = b.stride;
  for (int i = opaque_lane(W.t); i < W.n; i += T) {
    const int g = W.b0w + i;
    W.fl[i] = b.flags[g];
    if constexpr (VEL) {
      tab3_store(W.st + kIslSt * i, ld3(b.vel, S, g));
      tab3_store(W.st + kIslSt * i + 3, ld3(b.rot, S, g));
    } else {
      tab3_store(W.st + kIslSt * i, ld3(b.pos, S, g));
#pragma unroll
      for (int k = 0; k < 4; ++k) W.st[kIslSt * i + 3 + k] = b.quat[k * S + g];
    }
  }
  __syncthreads();
}

// The position phase writes a sleeping body's derived data in HBM when it
// moves one (contact.go:380-382): kept, and put back.
template <typename R, int T>
__device__ __forceinline__ void isl_sleepers(const RS<R>& a, const IslWorld<R, T>& W, bool put_back) {
  const Bodies<R>& b = a.b;
  const int64_t S = b.stride;
  for (int i = opaque_lane(W.t); i < W.n; i += T) {
    const int g = W.b0w + i;
    if (b.flags[g] & F_AWAKE) continue;
#pragma unroll
    for (int k = 0; k < 12; ++k) {
      if (put_back)
        b.transform[k * S + g] = a.isl_snap[k * S + g];
      else
        a.isl_snap[k * S + g] = b.transform[k * S + g];
    }
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      if (put_back)
        b.iit_world[k * S + g] = a.isl_snap[(12 + k) * S + g];
      else
        a.isl_snap[(12 + k) * S + g] = b.iit_world[k * S + g];
    }
  }
  __syncthreads();
}

// The phase's result to HBM: the tables, the awake flags and the motion
// matchAwakeState gives a woken body (SetAwake(true), rigidbody.go:183-186).
template <typename R, bool VEL, int T>
__device__ __forceinline__ void isl_commit(const RS<R>& a, const IslWorld<R, T>& W) {
  const Bodies<R>& b = a.b;
  const int64_t S = b.stride;
  for (int i = opaque_lane(W.t); i < W.n; i += T) {
    const int g = W.b0w + i;
    if constexpr (VEL) {
      st3(b.vel, S, g, tab3(W.st + kIslSt * i));
      st3(b.rot, S, g, tab3(W.st + kIslSt * i + 3));
    } else {
      st3(b.pos, S, g, tab3(W.st + kIslSt * i));
#pragma unroll
      for (int k = 0; k < 4; ++k) b.quat[k * S + g] = W.st[kIslSt * i + 3 + k];
    }
    const uint8_t f = W.fl[i];
    if (f != b.flags[g]) {
      b.motion[g] = R(kSleepEpsilon * 2.0);
      b.flags[g] = f;
    }
  }
  __syncthreads();
}

// The world's labels of a phase that is run again.
template <typename R, bool VEL, int T>
__device__ __forceinline__ void isl_clear_labels(const RS<R>& a, const IslWorld<R, T>& W) {
  for (int j = opaque_lane(W.t); j < W.C; j += T) {
    float* L = a.labels + (W.base + j) * kOut;
    if constexpr (VEL) {
      for (int q = 0; q < 12; ++q) L[q] = 0.f;
    } else {
      L[kOutPos] = 0.f;
    }
  }
}

// Non-negative reals ordered as their bits.
__device__ __forceinline__ float real_of_bits(uint32_t u) { return __int_as_float(int(u)); }
__device__ __forceinline__ double real_of_bits(uint64_t u) {
  return __hiloint2double(int(uint32_t(u >> 32)), int(uint32_t(u)));
}
template <typename R>
struct BitsOf {
  typedef uint64_t type;
  static constexpr type inf = 0x7FF0000000000000ull;
};
template <>
struct BitsOf<float> {
  typedef uint32_t type;
  static constexpr type inf = 0x7F800000u;
};

constexpr double kIslDeal = 16;  // records that are dealt out one by one rather than searched for a level
// Merges the islands' logs in the serial loop's order up to `budget`
// iterations; leaves each island's share in isl_its (-1 with `skip` where the
// island is not cut short).  The serial loop has run every selection above
// a level before the first at or below it: the lowest level whose selections
// above it fit the budget is found by bisection over the keys' bits, and what
// is left of the budget is dealt out from there by picking the island with
// the largest key.  (A paused island's log starts at its pause, where
// `at_pause` of its iterations are done.)  The heads are in the state tables'
// space.
template <typename R, int T>
__device__ __forceinline__ void isl_merge(const RS<R>& a, const IslWorld<R, T>& W, int nisl, int64_t budget, int paused,
                                          int at_pause, bool skip, int late) {
  typedef typename BitsOf<R>::type U;
  R* hkey = W.st;
  int32_t* hj = (int32_t*)(hkey + W.NB);
  int32_t* hp = hj + W.NB;
  auto plus = [](double p, double q) { return p + q; };
  auto its = [&](int k, const IslLog& L, int r) {  // of island k before record r of its log
    return (r < L.n ? a.log_it[L.place(r)] : a.isl_its[W.b0w + k]) - (k == paused ? at_pause : 0);
  };
  auto above = [&](R tau) {  // iterations above a level
    double n = 0.0;
    for (int k = W.t; k < nisl; k += T) {
      const IslLog L = isl_log_of(a, W.b0w + k, late);
      n += double(its(k, L, isl_first(a, L, 0, L.n, tau)));
    }
    return int64_t(isl_reduce(W, n, plus));
  };
  int64_t rem = budget - at_pause;
  U lo = 0, hi = BitsOf<R>::inf;
  if (nisl <= T) {
    // One island per thread (up to 64: per lane, and every wave does the same).
    // The thread keeps which of its records may be the first at or below the
    // level, so that a step costs a load or two, and when few are left in the
    // range they are dealt out below.
    const bool wave = nisl <= 64;
    const int k = wave ? W.t & 63 : W.t;
    const bool has = k < nisl;
    const IslLog L = has ? isl_log_of(a, W.b0w + k, late) : IslLog{0, 0, INT_MAX, 0};
    int r0 = 0, r1 = L.n;
    while (lo < hi) {
      const U mid = lo + ((hi - lo) >> 1);
      const int r = isl_first(a, L, r0, r1, real_of_bits(mid));
      // the iterations above the level, and (times 2^32) the records still in question
      double sum = has ? double(its(k, L, r)) + double(r1 - r) * 0x1p32 : 0.0;
      if (wave) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
      } else {
        sum = isl_reduce(W, sum, plus);
      }
      const double records = floor(sum * 0x1p-32);
      if (int64_t(sum - records * 0x1p32) <= rem) {
        hi = mid;
        r0 = r;
        if (records <= kIslDeal) break;
      } else {
        lo = mid + 1;
        r1 = r;
      }
    }
  } else {
    while (lo < hi) {
      const U mid = lo + ((hi - lo) >> 1);
      if (above(real_of_bits(mid)) <= rem)
        hi = mid;
      else
        lo = mid + 1;
    }
  }
  const R tau = real_of_bits(hi);
  rem -= above(tau);
  for (int k = W.t; k < nisl; k += T) {
    const IslLog L = isl_log_of(a, W.b0w + k, late);
    const int r = isl_first(a, L, 0, L.n, tau);
    hkey[k] = r < L.n ? a.log_key[L.place(r)] : R(-__builtin_inf());
    hj[k] = r < L.n ? a.log_j[L.place(r)] : INT_MAX;
    hp[k] = r;
  }
  __syncthreads();
  const int lane = W.t;
  if (W.t < 64) {
    while (!__any(rem <= 0)) {
      R best = R(-__builtin_inf());
      int bj = INT_MAX, bk = -1;
      for (int k = lane; k < nisl; k += 64) {
        const R h = hkey[k];
        if (h > best || (h == best && hj[k] < bj)) {
          best = h;
          bj = hj[k];
          bk = k;
        }
      }
      const R m = group_reduce(best, 6, [](R p, R q) { return q > p ? q : p; });
      if (!__any(m > R(-__builtin_inf()))) break;
      const int jm = group_reduce(best == m ? bj : INT_MAX, 6, [](int p, int q) { return q < p ? q : p; });
      int run = 0;
      if (bk >= 0 && best == m && bj == jm) {  // this lane's island goes on to its next record
        const IslLog L = isl_log_of(a, W.b0w + bk, late);
        const int r = hp[bk], from = a.log_it[L.place(r)];
        const int end = r + 1 < L.n ? a.log_it[L.place(r + 1)] : a.isl_its[W.b0w + bk];
        run = end - from;
        if (int64_t(run) >= rem) {
          run = int(rem);
          hp[bk] = -1 - (from + run);  // settled: its share
          hkey[bk] = R(-__builtin_inf());
        } else {
          hp[bk] = r + 1;
          hkey[bk] = r + 1 < L.n ? a.log_key[L.place(r + 1)] : R(-__builtin_inf());
          hj[bk] = r + 1 < L.n ? a.log_j[L.place(r + 1)] : INT_MAX;
        }
      }
      rem -= group_reduce(run, 6, [](int p, int q) { return q > p ? q : p; });
      wave_fence();
    }
  }
  __syncthreads();
  for (int k = W.t; k < nisl; k += T) {
    const int g = W.b0w + k, r = hp[k], all = a.isl_its[g];
    const IslLog L = isl_log_of(a, g, late);
    const int share = r < 0 ? -1 - r : r < L.n ? a.log_it[L.place(r)] : all;
    a.isl_its[g] = skip && k != paused && share == all ? -1 : share;
  }
  __syncthreads();
}

// The body tables to HBM scratch, and back.
template <typename R, int T>
__device__ __forceinline__ void isl_tables(const RS<R>& a, const IslWorld<R, T>& W, bool put_back) {
  const int64_t S = a.b.stride;
  for (int i = opaque_lane(W.t); i < W.n; i += T) {
    const int g = W.b0w + i;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      if (put_back)
        W.st[kIslSt * i + k] = a.isl_snap[(14 + k) * S + g];
      else
        a.isl_snap[(14 + k) * S + g] = W.st[kIslSt * i + k];
    }
    if (put_back)
      W.fl[i] = a.isl_flag[g];
    else
      a.isl_flag[g] = W.fl[i];
  }
  __syncthreads();
}

// The bodies of the islands that were cut short, as the velocity phase starts
// (a wave per island; a body of several contacts is written several times).
template <typename R, int T>
__device__ __forceinline__ void isl_cut_bodies(const RS<R>& a, const IslWorld<R, T>& W, int nisl, int paused) {
  const Bodies<R>& b = a.b;
  const int64_t S = b.stride;
  for (int k = W.t >> 6; k < nisl; k += (T / 64)) {
    if (k == paused || a.isl_its[W.b0w + k] < 0) continue;
    const int cnt = a.isl_cnt[W.b0w + k];
    const int32_t* idx = a.isl_idx + W.base + a.isl_off[W.b0w + k];
    for (int q = W.t & 63; q < cnt; q += 64) {
      const int64_t gj = W.base + idx[q];
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const int g = d == 0 ? a.c.body0[gj] : a.c.body1[gj];
        if (g < 0) continue;
        R* e = W.st + kIslSt * (g - W.b0w);
        tab3_store(e, ld3(b.vel, S, g));
        tab3_store(e + 3, ld3(b.rot, S, g));
        W.fl[g - W.b0w] = b.flags[g];
      }
    }
  }
  __syncthreads();
}

// The surrogate's position polish of the world (KIND_PPOLISH, mask byte 0):
// the predicted moves are added to the awake bodies and every contact's
// penetration updated for them by the loop's own formula, a thread per
// contact.  The plain phase stays within 1.4 times the world's deepest
// penetration of separating a contact; a prediction that separates one beyond
// kSepFactor times it (sep_floor) is tried again at a third of its moves, and
// given up (false) if that still does.
template <typename R, int T>
__device__ __forceinline__ bool isl_take_moves(const RS<R>& a, const IslWorld<R, T>& W, R& sep_floor) {
  const Bodies<R>& b = a.b;
  const Contacts<R>& c = a.c;
  const int64_t S = b.stride, CS = c.cap;
  const float* dl = a.delta;
  R pmax = R(0);
  for (int j = W.t; j < W.C; j += T) {
    const R p = c.pen[W.base + j];
    a.isl_save[4 * CS + W.base + j] = p;
    pmax = p > pmax ? p : pmax;
  }
  pmax = R(isl_reduce(W, double(pmax), [](double p, double q) { return q > p ? q : p; }));
  sep_floor = -(R(kSepFactor) * pmax + a.polish_tol);
  for (int attempt = 0; attempt < 2; ++attempt) {
    // the moves times `scale`, from the phase's starting state
    const R scale = attempt == 0 ? R(1) : R(kPosRetryScale);
    for (int i = W.t; i < W.n; i += T) {
      const int g = W.b0w + i;
      if (!(W.fl[i] & F_AWAKE)) continue;
      const V3<R> dx = mul(V3<R>{R(dl[g]), R(dl[S + g]), R(dl[2 * S + g])}, scale);
      const V3<R> dq = mul(V3<R>{R(dl[3 * S + g]), R(dl[4 * S + g]), R(dl[5 * S + g])}, scale);
      if (dx.x == R(0) && dx.y == R(0) && dx.z == R(0) && dq.x == R(0) && dq.y == R(0) && dq.z == R(0)) continue;
      R* e = W.st + kIslSt * i;
      tab3_store(e, add(ld3(b.pos, S, g), dx));
      Q4<R> q{b.quat[g], b.quat[S + g], b.quat[2 * S + g], b.quat[3 * S + g]};
      q = q_normalize(q_add_scaled_vector(q, dq, R(1)));
      e[3] = q.w;
      e[4] = q.x;
      e[5] = q.y;
      e[6] = q.z;
    }
    R kmin = R(0);
    for (int j = W.t; j < W.C; j += T) {
      const int64_t gj = W.base + j;
      const int kb[2] = {c.body0[gj], c.body1[gj]};
      V3<R> nj, rj[2];
      rec_normal(c.rec + 16 * gj, nj, rj);
      R pen = a.isl_save[4 * CS + gj];
#pragma unroll
      for (int bb = 0; bb < 2; ++bb) {
        const int g = kb[bb];
        if (g < 0) continue;
        const V3<R> dx = mul(V3<R>{R(dl[g]), R(dl[S + g]), R(dl[2 * S + g])}, scale);
        const V3<R> dq = mul(V3<R>{R(dl[3 * S + g]), R(dl[4 * S + g]), R(dl[5 * S + g])}, scale);
        if (dx.x == R(0) && dx.y == R(0) && dx.z == R(0) && dq.x == R(0) && dq.y == R(0) && dq.z == R(0)) continue;
        const V3<R> dp = add(cross(dq, rj[bb]), dx);
        R sign = R(1);
        if (bb == 0) sign = R(-1);
        pen += dot(dp, nj) * sign;
      }
      c.pen[gj] = pen;
      kmin = pen < kmin ? pen : kmin;
    }
    __syncthreads();
    kmin = R(isl_reduce(W, double(kmin), [](double p, double q) { return q < p ? q : p; }));
    if (kmin >= sep_floor) return true;
  }
  return false;
}

// Kinetic energy of the world from the tables (KIND_POLISH); with it the
// world's mass.
template <typename R, int T>
__device__ __forceinline__ double isl_energy(const RS<R>& a, const IslWorld<R, T>& W, double& mass) {
  double ke = 0.0, m = 0.0;
  for (int i = opaque_lane(W.t); i < W.n; i += T) {
    const int g = W.b0w + i;
    R iw[9];
    ld9(a.b.iit_world, a.b.stride, g, iw);
    double mi;
    ke += kinetic_energy(tab3(W.st + kIslSt * i), tab3(W.st + kIslSt * i + 3), a.b.inv_mass[g], iw, mi);
    m += mi;
  }
  auto plus = [](double p, double q) { return p + q; };
  mass = isl_reduce(W, m, plus);
  return isl_reduce(W, ke, plus);
}

// The surrogate's velocity polish of the world (KIND_POLISH, mask byte 0):
// the predicted changes are added to the
// bodies, and every contact of a changed body gets its contact velocity by
// the update of contact.go:424-441 and its desired velocity change anew.
template <typename R, int T>
__device__ __forceinline__ void isl_take_changes(const RS<R>& a, const IslWorld<R, T>& W) {
  const Bodies<R>& b = a.b;
  const Contacts<R>& c = a.c;
  const int64_t S = b.stride, CS = c.cap;
  const float* dl = a.delta;
  for (int i = W.t; i < W.n; i += T) {
    const int g = W.b0w + i;
    const V3<R> dv{R(dl[g]), R(dl[S + g]), R(dl[2 * S + g])};
    const V3<R> dw{R(dl[3 * S + g]), R(dl[4 * S + g]), R(dl[5 * S + g])};
    if (dv.x != R(0) || dv.y != R(0) || dv.z != R(0) || dw.x != R(0) || dw.y != R(0) || dw.z != R(0)) {
      R* e = W.st + kIslSt * i;
      tab3_store(e, add(tab3(e), dv));
      tab3_store(e + 3, add(tab3(e + 3), dw));
    }
  }
  for (int j = W.t; j < W.C; j += T) {
    const int64_t gj = W.base + j;
    const int kb[2] = {c.body0[gj], c.body1[gj]};
    V3<R> cvj = ld3(c.cvel, CS, gj);
    st3(a.isl_save, CS, gj, cvj);
    a.isl_save[3 * CS + gj] = c.ddv[gj];
    R mj[9];
    V3<R> rj[2];
    rec_frame(c.rec + 16 * gj, mj, rj);
    bool moved = false;
#pragma unroll
    for (int bb = 0; bb < 2; ++bb) {
      const int g = kb[bb];
      if (g < 0) continue;
      const V3<R> dv{R(dl[g]), R(dl[S + g]), R(dl[2 * S + g])};
      const V3<R> dw{R(dl[3 * S + g]), R(dl[4 * S + g]), R(dl[5 * S + g])};
      if (dv.x == R(0) && dv.y == R(0) && dv.z == R(0) && dw.x == R(0) && dw.y == R(0) && dw.z == R(0)) continue;
      moved = true;
      R sign = R(1);
      if (bb == 1) sign = R(-1);
      cvj = add(cvj, mul(m3tv(mj, add(cross(dw, rj[bb]), dv)), sign));
    }
    if (moved) {  // a contact neither of whose bodies changed keeps prepare's key
      const V3<R> nj{mj[0], mj[1], mj[2]};
      const R d0 = dot(mul(ld3(b.last_acc, S, kb[0]), a.dt), nj);
      const R d1 = kb[1] >= 0 ? dot(mul(ld3(b.last_acc, S, kb[1]), a.dt), nj) : R(0);
      st3(c.cvel, CS, gj, cvj);
      const int jl[2] = {kb[0] - W.b0w, kb[1] >= 0 ? kb[1] - W.b0w : -1};
      c.ddv[gj] = isl_desired_dv(isl_awake_of(W, jl), kb[1] >= 0, d0, d1, cvj.x, restitution_of<R, KIND_POLISH>(c, gj));
    }
  }
  __syncthreads();
}

// The contacts' values before the phase, put back.
template <typename R, bool VEL, int T>
__device__ __forceinline__ void isl_contacts_back(const RS<R>& a, const IslWorld<R, T>& W) {
  const Contacts<R>& c = a.c;
  const int64_t CS = c.cap;
  for (int j = opaque_lane(W.t); j < W.C; j += T) {
    const int64_t g = W.base + j;
    if constexpr (VEL) {
      st3(c.cvel, CS, g, ld3(a.isl_save, CS, g));
      c.ddv[g] = a.isl_save[3 * CS + g];
    } else {
      c.pen[g] = a.isl_save[4 * CS + g];
    }
  }
  __syncthreads();
}

// Room in the log pool for the world's logs, an island's being at most the
// iterations it ran (a paused one's: what it may still run); false when there
// is none.
template <typename R, int T>
__device__ __forceinline__ bool isl_log_room(const RS<R>& a, const IslWorld<R, T>& W, int nisl, int paused,
                                             int64_t paused_room, int late) {
  if (W.t < 64) {
    // an island that is run again whole logs at most its iterations so far,
    // or, stopped by the budget as part of the world's, up to the budget
    int64_t need = 0;
    for (int k = W.t; k < nisl; k += 64) {
      const int64_t its = late > 0 && isl_is_late(a.isl_nrec[W.b0w + k]) ? 0 : a.isl_its[W.b0w + k];
      need += k == paused ? its + paused_room : its;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) need += __shfl_xor(need, o, 64);
    int64_t at = 0;
    if (W.t == 0) at = isl_reserve(a, need);
    at = __shfl(at, 0, 64);
    const bool ok = at >= 0;
    if (W.t == 0) W.f->ok = ok ? 1 : 0;
    for (int k0 = 0; ok && k0 < nisl; k0 += 64) {
      const int k = k0 + W.t;
      const bool mine = k < nisl && !(late > 0 && isl_is_late(a.isl_nrec[W.b0w + k]));
      const int64_t its = mine ? a.isl_its[W.b0w + k] : 0;
      const int64_t m = k == paused ? its + paused_room : its;
      const int64_t inc = wave_incl_scan_i64(m);
      if (mine) a.isl_log[W.b0w + k] = at + inc - m;
      at += __shfl(inc, 63, 64);
    }
  }
  __syncthreads();
  return W.f->ok != 0;
}

// A budget that is a small part of what the islands would run (below
// C / kIslSerial) or short altogether, once it is exceeded, is spent on one chain
// of all the world's contacts: the logs and their merge would cost more.
constexpr int64_t kIslSerial = 2, kIslShort = 96;
// After a free pass over the budget: whether every island that ran for more than
// `late` iterations logged from there on, and there is room for the logs of the
// rest, which is short.  Not with big islands, which log late only when paused.
template <typename R, int T>
__device__ __forceinline__ bool isl_late(const RS<R>& a, const IslWorld<R, T>& W, int nisl, int late) {
  if (W.f->lates == 0 || W.f->lates > kIslLates || W.f->cls[0] + W.f->cls[1] + W.f->cls[2] + W.f->cls[3] > 0)
    return false;
  double bad = 0.0;
  for (int k = W.t; k < nisl; k += T)
    if (!isl_is_late(a.isl_nrec[W.b0w + k]) && a.isl_its[W.b0w + k] > late) bad = 1.0;
  if (isl_reduce(W, bad, [](double p, double q) { return p + q; }) > 0.0) return false;
  return isl_log_room(a, W, nisl, -1, 0, late);
}

// One phase of the world: the tables are loaded, the contacts are as
// prepared; `polish` first tries the surrogate's polish (its mask byte is
// set when that is rejected).  A world that exceeds its budget and finds no
// room in the log pool starts again as one island of all its contacts.
// Returns false when that has more than isl_max_contacts<T>() of them: the phase is
// undone, for the serial kernel to do.
template <typename R, int KIND, bool VEL, int T>
__device__ __forceinline__ bool isl_phase(const RS<R>& a, const IslWorld<R, T>& W, int64_t budget, bool polish,
                                          int64_t& used) {
  constexpr bool POLISH = VEL ? KIND == KIND_POLISH : KIND == KIND_PPOLISH;
  const R plain_eps = VEL ? R(kVelocityEpsilon) : R(kPositionEpsilon);
  constexpr bool LATE = VEL && KIND != KIND_LABEL;
  const int late = LATE && budget >= 16 && budget < kIslLate ? int(budget >> 2) : 0;
  const bool one = W.C <= isl_max_contacts<T>() && budget * (W.C > 2 * T ? 2 * kIslSerial : kIslSerial) < W.C;
  IslPass P{ISL_FREE, false, budget, !one, -1, false, one, late};
  R eps = plain_eps, sep_floor = R(0);
  double ke = 0.0, mass = 0.0;
  bool rejected = false;
  if constexpr (POLISH) {
    if (polish) {
      if constexpr (VEL) {
        ke = isl_energy(a, W, mass);
        isl_take_changes(a, W);
      } else {
        rejected = !isl_take_moves(a, W, sep_floor);
      }
      P.saved = true;
      P.pause = P.one = false;
      P.late = 0;
      P.budget = isl_budget(a.polish_mult * int64_t(W.C));
      eps = plain_eps + a.polish_tol;
    }
  }
  int nisl = 0, paused = -1, at_pause = 0;
  while (true) {
    R kmin = R(0);
    if (!rejected) isl_run<R, KIND, VEL>(a, W, P, eps, kmin);
    if constexpr (POLISH) {
      if (polish) {
        used = int64_t(W.f->total);
        bool ok = !rejected && used <= P.budget && !W.f->over;
        if constexpr (VEL) {
          // The plain phase applies only compressive impulses inside the
          // friction cone with restitution below 1, so it never adds kinetic
          // energy; a polished world that ends with more than it started
          // with, beyond a slack of 1/2 tol^2 per kilogram (which also covers
          // the acceleration term of the restitution target,
          // contact.go:87-112), is rejected.  This is what stops a wrong
          // prediction from pushing bodies apart.
          if (ok) {
            double m2;
            const double after = isl_energy(a, W, m2), tol = double(a.polish_tol);
            ok = after <= ke * (1.0 + kEnergyRel) + 0.5 * tol * tol * mass;
          }
        } else {
          const R least = R(isl_reduce(W, double(kmin), [](double p, double q) { return q < p ? q : p; }));
          ok = ok && least >= sep_floor;
        }
        if (ok) return true;
        // the plain phase instead, from the state the phase found
        if constexpr (!VEL) isl_sleepers(a, W, true);
        isl_contacts_back<R, VEL>(a, W);
        isl_load<R, VEL>(a, W);
        if (W.t == 0) a.world_mask[W.w] = 1;
        polish = rejected = false;
        P = IslPass{ISL_FREE, true, budget, !one, -1, false, one, late};
        eps = plain_eps;
        if (budget <= 0) {
          used = 0;
          return true;
        }
        continue;
      }
    }
    if (P.pass == ISL_LIMIT) return true;
    if (P.pass == ISL_FREE) {
      const int64_t total = int64_t(W.f->total);
      used = total;
      if (P.one || (total <= budget && !W.f->over)) return true;
      used = budget;
      for (int k = 0; k < kIslClasses; ++k) nisl += W.f->cls[k];
      paused = W.f->paused;
      at_pause = paused >= 0 ? W.f->at : 0;
      if (LATE && P.late > 0 && budget > kIslShort && isl_late(a, W, nisl, P.late)) {
        isl_tables(a, W, false);
        P.pass = ISL_LOG;
        P.pause = false;
        isl_load<R, VEL>(a, W);
        continue;
      }
      P.late = 0;
      // log the selections, merge them, and run each island to its share; a
      // paused island logs what it goes on to run, at most to the budget
      const bool large = W.C > isl_max_contacts<T>();
      const bool ok = (budget > kIslShort || large) && isl_log_room(a, W, nisl, paused, budget - at_pause, 0);
      if constexpr (KIND == KIND_LABEL) {
        isl_clear_labels<R, VEL>(a, W);
        paused = -1;  // its labels would have to be kept
      }
      if (!ok) {
        if constexpr (!VEL) isl_sleepers(a, W, true);
        isl_contacts_back<R, VEL>(a, W);
        if (large) return false;
        P = IslPass{ISL_FREE, true, budget, false, -1, false, true, 0};
        isl_load<R, VEL>(a, W);
        continue;
      }
      P.pass = ISL_LOG;
      P.pause = false;
      if (VEL && paused >= 0) {
        isl_tables(a, W, false);
        P.resume = paused;
      }
    } else if (VEL && paused >= 0 && !P.only) {
      // the others have logged; the paused island goes on alone
      isl_tables(a, W, true);
      P.only = true;
      continue;
    } else {
      // islands that ended are as their end left them, the paused one as its
      // pause did, the others start again
      const bool keep = VEL && (paused >= 0 || P.late > 0);
      isl_merge(a, W, nisl, budget, keep ? paused : -1, keep && paused >= 0 ? at_pause : 0, keep, P.late);
      P.pass = ISL_LIMIT;
      P.only = false;
      if (keep) {
        isl_tables(a, W, true);
        isl_cut_bodies(a, W, nisl, paused);
        continue;
      }
    }
    if constexpr (!VEL) isl_sleepers(a, W, true);
    isl_load<R, VEL>(a, W);
  }
}

// Hands the world to the left kernel; vel_only: its position phase is done.
template <typename R, int T>
__device__ __forceinline__ void isl_leave(const RS<R>& a, const IslWorld<R, T>& W, bool vel_only) {
  if (W.t == 0) a.left_list[atomicAdd(&a.left_count[LEFT_WORLDS], 1)] = W.w | (vel_only ? kLeftVelOnly : 0);
}

template <typename R, int KIND, int T>
__device__ __forceinline__ void isl_world(const RS<R>& a, const IslWorld<R, T>& W) {
  const int w = W.w;
  const bool do_pos = (a.mode & RM_POS) != 0;
  const bool do_prep = do_pos && !(a.mode & RM_PREPARED);
  const bool do_vel = (a.mode & RM_VEL) != 0 && (KIND == KIND_POLISH || !a.world_mask || a.world_mask[w]);
  if (a.world_iters && W.t == 0) {
    if (do_pos) a.world_iters[2 * w] = 0;
    if (a.mode & RM_VEL) a.world_iters[2 * w + 1] = 0;
  }
  // ResolveContacts' guard, contact.go:210-212
  if (a.overflow[0] != 0 || W.C <= 0 || a.dt <= R(0)) return;
  if (!do_pos && !do_vel) return;
  const int64_t maxIter = isl_budget(a.iter_fixed > 0 ? a.iter_fixed : a.iter_mult * int64_t(W.C));
  if (W.n > W.NB) {
    isl_leave(a, W, false);
    return;
  }
  if (do_prep) isl_prepare<R, KIND>(a, W, true);
  if (a.isl_wide && !do_prep) {  // left by the narrow workgroups: its islands are theirs
    isl_build(a, W);
    __syncthreads();
  }
  if (a.isl_cls[kIslWords * int64_t(w) + kIslTaken] != T) {
    if (T < kIslThreads) {
      if (W.t == 0) a.wide_list[atomicAdd(&a.left_count[LEFT_WIDE], 1)] = w;
    } else {
      isl_leave(a, W, false);
    }
    return;
  }
  // worlds beyond the polish's reach take the plain phase
  bool polish = (KIND == KIND_POLISH || KIND == KIND_PPOLISH) && a.world_mask[w] == 0;
  if (polish && (W.n > kPolishBodies || W.C > kPolishContacts)) {
    __syncthreads();
    polish = false;
    if (W.t == 0) a.world_mask[w] = 1;
  }
  if (do_pos) {
    int64_t used = 0;
    isl_sleepers(a, W, false);
    isl_load<R, false>(a, W);
    if ((polish || maxIter > 0) && !isl_phase<R, KIND, false>(a, W, maxIter, polish, used)) {
      isl_leave(a, W, false);
      return;
    }
    isl_commit<R, false>(a, W);
    if (W.t == 0 && a.world_iters) a.world_iters[2 * w] = used;
  }
  if (do_vel) {
    int64_t used = 0;
    isl_load<R, true>(a, W);
    if ((polish || maxIter > 0) && !isl_phase<R, KIND, true>(a, W, maxIter, polish, used)) {
      isl_leave(a, W, do_pos);
      return;
    }
    isl_commit<R, true>(a, W);
    if (W.t == 0 && a.world_iters) a.world_iters[2 * w + 1] = used;
  }
}

template <typename R, int T>
__device__ __forceinline__ IslWorld<R, T> isl_world_of(const RS<R>& a, char* lds, int w) {
  IslWorld<R, T> W;
  W.w = w;
  W.t = threadIdx.x;
  W.C = a.world_cnt[w];
  W.b0w = a.body_off[w];
  W.n = a.body_off[w + 1] - W.b0w;
  W.base = a.world_coff[w];
  W.NB = a.isl_nb;
  W.f = (IslFixed<R, T>*)lds;
  W.st = (R*)(lds + isl_fixed_bytes<R, T>());
  R* after = W.st + kIslSt * int64_t(W.NB);
  W.iw = W.NB <= kIslIwBodies ? after : nullptr;
  W.fl = (uint8_t*)(W.NB <= kIslIwBodies ? after + kIslIw * int64_t(W.NB) : after);
  return W;
}

template <typename R, int KIND, int T>
__device__ __forceinline__ void isl_block(const RS<R>& a) {
  extern __shared__ __align__(16) char isl_lds[];
  if (a.isl_wide && int(blockIdx.x) >= a.left_count[LEFT_WIDE]) return;
  const int w = a.isl_wide ? a.wide_list[blockIdx.x] : a.order ? a.order[blockIdx.x] : int(blockIdx.x);
  const IslWorld<R, T> W = isl_world_of<R, T>(a, isl_lds, w);
  int64_t* wt = a.world_time ? a.world_time + 4 * int64_t(w) + ((a.mode & RM_VEL) ? 2 : 0) : nullptr;
  if (wt && W.t == 0) wt[0] = int64_t(wall_clock64());
  isl_world<R, KIND>(a, W);
  if (wt) {
    __syncthreads();
    if (W.t == 0) wt[1] = int64_t(wall_clock64());
  }
}

// Bound by the longest island's chain of dependent arithmetic in small
// launches, by instruction issue in large ones.
template <int KIND, int T>
__global__ void __launch_bounds__(T, 2) k_resolve_islands_f64(RS<double> a) {
  isl_block<double, KIND, T>(a);
}
template <int KIND, int T>
__global__ void __launch_bounds__(T, 3) k_resolve_islands_f32(RS<float> a) {
  isl_block<float, KIND, T>(a);
}

template <typename R, int T>
size_t isl_lds_bytes(int nb) {
  return isl_fixed_bytes<R, T>() + size_t(nb) * ((kIslSt + (nb <= kIslIwBodies ? kIslIw : 0)) * sizeof(R) + 1);
}

template <typename R, int KIND, int T>
constexpr void (*isl_kernel())(RS<R>) {
  if constexpr (sizeof(R) == 8)
    return k_resolve_islands_f64<KIND, T>;
  else
    return k_resolve_islands_f32<KIND, T>;
}

// Dynamic LDS beyond the default limit (worlds of more than about 880 bodies
// in FP64) has to be asked for.
template <typename R>
hipError_t isl_allow_lds(void (*kernel)(RS<R>), size_t lds) {
  if (lds <= 64 * 1024) return hipSuccess;
  return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
}

template <typename R, int KIND, int T>
hipError_t isl_launch(const RS<R>& a, hipStream_t st) {
  const size_t lds = isl_lds_bytes<R, T>(a.isl_nb);
  const hipError_t e = isl_allow_lds<R>(isl_kernel<R, KIND, T>(), lds);
  if (e != hipSuccess) return e;
  isl_kernel<R, KIND, T>()<<<a.n_worlds, T, lds, st>>>(a);
  return hipGetLastError();
}

// narrow: half the threads per world, and what these leave on whole workgroups.
template <typename R, int KIND>
hipError_t launch_islands_kind(const RS<R>& a, bool narrow, hipStream_t st) {
  if (!narrow) return isl_launch<R, KIND, kIslThreads>(a, st);
  const hipError_t e = isl_launch<R, KIND, kIslThreads / 2>(a, st);
  if (e != hipSuccess) return e;
  RS<R> wide = a;
  wide.isl_wide = 1;
  return isl_launch<R, KIND, kIslThreads>(wide, st);
}

// Worlds (workgroups) of one kind's island kernel resident per CU, from its
// register and LDS use.
template <typename R, int KIND>
hipError_t islands_occupancy(int nb, int* worlds_per_cu) {
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(worlds_per_cu,
                                                      (const void*)isl_kernel<R, KIND, kIslThreads>(), kIslThreads,
                                                      isl_lds_bytes<R, kIslThreads>(nb));
}

#ifndef CBZ_RESOLVE_INSTANTIATE
CBZ_RESOLVE_KIND(extern, double, KIND_PLAIN)
CBZ_RESOLVE_KIND(extern, double, KIND_LABEL)
CBZ_RESOLVE_KIND(extern, double, KIND_POLISH)
CBZ_RESOLVE_KIND(extern, double, KIND_MAT)
CBZ_RESOLVE_KIND(extern, double, KIND_PPOLISH)
CBZ_RESOLVE_KIND(extern, float, KIND_PLAIN)
CBZ_RESOLVE_KIND(extern, float, KIND_LABEL)
CBZ_RESOLVE_KIND(extern, float, KIND_POLISH)
CBZ_RESOLVE_KIND(extern, float, KIND_MAT)
CBZ_RESOLVE_KIND(extern, float, KIND_PPOLISH)
#endif

}  // namespace cbz
