// k_resolve.hip — launch dispatch of the resolver (K3): picks the
// compile-time kind of the kernel for the requested phases and materials.
// The kernels are in cbz_islands.h and cbz_resolve.h, instantiated by k_resolve_<precision>_<kind>.hip.
#include <algorithm>

#include "cbz_islands.h"

namespace cbz {

// prepareContacts alone (a position launch without iterations): one
// workgroup per world, a thread per contact, from the bodies' state in HBM,
// with every contact's record and the world's islands.
template <typename R, int KIND, int T>
__global__ void __launch_bounds__(T) k_prepare(RS<R> a) {
  extern __shared__ __align__(16) char isl_lds[];
  const IslWorld<R, T> W = isl_world_of<R, T>(a, isl_lds, int(blockIdx.x));
  if (a.overflow[0] != 0 || W.C <= 0) return;  // the resolver's guard
  isl_prepare<R, KIND>(a, W, W.n <= W.NB);
}
template <typename R, int T>
hipError_t launch_prepare(const RS<R>& a, hipStream_t st) {
  const size_t lds = isl_lds_bytes<R, T>(a.isl_nb);
  void (*kernel)(RS<R>) = a.c.fric ? k_prepare<R, KIND_MAT, T> : k_prepare<R, KIND_PLAIN, T>;
  const hipError_t e = isl_allow_lds<R>(kernel, lds);
  if (e != hipSuccess) return e;
  kernel<<<a.n_worlds, T, lds, st>>>(a);
  return hipGetLastError();
}

// The order in which the worlds start: those that took longest in the last
// launch of the same phase first.  A launch of more worlds than fit the chip
// ends with whatever started last, and what a world costs is not its size: one
// that runs into its iteration budget takes several times as long as its
// neighbours, and does so step after step.  In FP64, 1000 worlds whose times add
// up to 380 us on the whole chip took 990 us with the largest worlds first and
// take 670 now, the time of the longest; 2048 in FP32 830 and 750.  Only the order depends on the clock, no result.
// A world's cost is the greater of its last time and three quarters of the cost
// before (what takes long comes and goes), by its bodies as long as it has no
// time.  Counting sort, 5 us (512 ticks) per bucket.
__global__ void __launch_bounds__(1024) k_order(const int64_t* time, const int32_t* body_off, int n_worlds,
                                                int32_t* cost, int32_t* order) {
  constexpr int kBuckets = 256;
  __shared__ int32_t s_at[kBuckets];
  __shared__ int32_t s_wave[4];
  const int t = threadIdx.x;
  auto bucket = [&](int w) { return kBuckets - 1 - min(cost[w] >> 9, kBuckets - 1); };
  if (t < kBuckets) s_at[t] = 0;
  __syncthreads();
  for (int w = t; w < n_worlds; w += 1024) {
    const int64_t from = time[4 * int64_t(w)], to = time[4 * int64_t(w) + 1];
    const int32_t old = cost[w];
    cost[w] = from >= 0 && to >= from ? max(int32_t(min(to - from, int64_t(1) << 30)), old - old / 4)
                                      : (body_off[w + 1] - body_off[w]) << 7;
    atomicAdd(&s_at[bucket(w)], 1);
  }
  __syncthreads();
  int32_t v = 0, inc = 0;
  if (t < kBuckets) {
    v = s_at[t];
    inc = wave_incl_scan_i32(v);
    if ((t & 63) == 63) s_wave[t >> 6] = inc;
  }
  __syncthreads();
  if (t < kBuckets) {
    for (int u = 0; u < t >> 6; ++u) inc += s_wave[u];
    s_at[t] = inc - v;
  }
  __syncthreads();
  for (int w = t; w < n_worlds; w += 1024) order[atomicAdd(&s_at[bucket(w)], 1)] = w;
}
// Worlds up to which all start at once, one per CU, whatever their order (the
// scene's own: larger worlds first).  That one also serves the polish, whose
// times say less of the next step's (correlation 0.58 against 0.69 of the
// bodies, and 0.82 against 0.76 in the plain phases).
constexpr int kOrderWorlds = 256;

// Worlds whose whole workgroups fit the chip (two per CU in FP64, three in FP32).
template <typename R>
constexpr int32_t kResident = 256 * (sizeof(R) == 8 ? 2 : 3);
// Launches of many times that are bound by how many worlds are in flight, not by
// the longest one's chain: they get workgroups of half the threads, twice as many
// of them resident, and the few worlds of larger islands whole ones behind.  A
// step of 4096 worlds of towers, collapsed, takes 9.8 ms in FP64 (13.8 with whole
// workgroups) and 7.0 in FP32 (8.9), of 16384 in FP32 19 (30); of 2048 batched
// worlds in FP32 1.13 against 1.02, so the line lies above.
template <typename R>
bool isl_narrow(int32_t n_worlds) {
  return n_worlds > 4 * kResident<R>;
}

// The island kernel, then the kernel for the worlds it leaves (none, as a
// rule: its workgroups end at once).
template <typename R, int KIND>
hipError_t launch_all(const RS<R>& plain, const ResolveLaunch<R>& L, hipStream_t st) {
  int32_t* cost = L.cost;
  RS<R> a = plain;
  if (a.n_worlds > kOrderWorlds && cost && (a.mode & (RM_POS | RM_VEL | RM_POLISH)) == (RM_POS | RM_VEL)) {
    k_order<<<1, 1024, 0, st>>>(a.world_time + 2, a.body_off, a.n_worlds, cost, cost + a.n_worlds);
    a.order = cost + a.n_worlds;
  }
  const hipError_t e = launch_islands_kind<R, KIND>(a, isl_narrow<R>(a.n_worlds), st);
  if (e != hipSuccess) return e;
  launch_left_kind<R, KIND>(a, std::min(a.n_worlds, std::max(kLeftGrid, L.isl.large)), st);
  return hipGetLastError();
}

template <typename R>
hipError_t launch_resolve(const ResolveLaunch<R>& L, hipStream_t st) {
  RS<R> a;
  a.b = L.b;
  a.c = L.c;
  a.world_cnt = L.world_cnt;
  a.world_coff = L.world_coff;
  a.overflow = L.overflow;
  a.order = L.order;
  a.body_off = L.body_off;
  a.world_iters = L.world_iters;
  a.world_time = L.world_time;
  a.left_list = L.isl.left_list;
  a.wide_list = L.isl.wide_list;
  a.left_count = L.isl.left_count;
  a.isl_nb = L.isl.nb;
  a.isl_wide = 0;
  a.isl_off = L.isl.off;
  a.isl_cnt = L.isl.cnt;
  a.isl_its = L.isl.its;
  a.isl_nrec = L.isl.nrec;
  a.isl_log = L.isl.log;
  a.isl_cls = L.isl.cls;
  a.isl_idx = L.isl.idx;
  a.isl_save = (R*)L.isl.save;
  a.isl_snap = (R*)L.isl.snap;
  a.isl_flag = L.isl.flag;
  a.log_key = (R*)L.isl.log_key;
  a.log_j = L.isl.log_j;
  a.log_it = L.isl.log_it;
  a.log_head = L.isl.log_head;
  a.log_cap = L.isl.log_cap;
  a.n_worlds = L.n_worlds;
  a.dt = L.dt;
  a.iter_mult = L.iter_mult;
  a.iter_fixed = L.iter_fixed;
  a.mode = L.mode;
  a.world_mask = L.world_mask;
  a.pos0 = L.pos0;
  a.labels = L.labels;
  a.delta = L.delta;
  a.polish_tol = L.polish_tol;
  a.polish_mult = L.polish_mult;
  if (a.mode & RM_POLISH) {
    // one phase per polish launch
    const bool pos = (a.mode & RM_POS) != 0, vel = (a.mode & RM_VEL) != 0;
    if (pos == vel || !a.world_mask || !a.delta) return hipErrorInvalidValue;
  }
  if ((a.mode & RM_PREPARED) && !(a.mode & RM_POS)) return hipErrorInvalidValue;
  if ((a.mode & RM_LABEL) && !a.labels) return hipErrorInvalidValue;
  // per-contact materials: the plain resolver only
  if (a.c.fric && (!a.c.rest || (a.mode & (RM_POLISH | RM_LABEL)))) return hipErrorInvalidValue;
  if (a.n_worlds <= 0) return hipSuccess;
  if (a.iter_mult == 0 && a.iter_fixed == 0 && (a.mode & ~RM_FRICTIONLESS2) == RM_POS) {
    if (!a.pos0 || !a.c.rec) return hipErrorInvalidValue;  // k_prepare writes both
    return isl_narrow<R>(a.n_worlds) ? launch_prepare<R, kIslThreads / 2>(a, st) : launch_prepare<R, kIslThreads>(a, st);
  }
  if (a.c.fric) return launch_all<R, KIND_MAT>(a, L, st);
  if (a.mode & RM_POLISH)
    return (a.mode & RM_POS) ? launch_all<R, KIND_PPOLISH>(a, L, st) : launch_all<R, KIND_POLISH>(a, L, st);
  if (a.mode & RM_LABEL) return launch_all<R, KIND_LABEL>(a, L, st);
  return launch_all<R, KIND_PLAIN>(a, L, st);
}

// Worlds (workgroups) of the plain island kernel resident per CU, from its
// register and LDS use with tables for 256 bodies.
hipError_t resolver_occupancy(bool f64, int* worlds_per_cu) {
  return f64 ? islands_occupancy<double, KIND_PLAIN>(256, worlds_per_cu)
             : islands_occupancy<float, KIND_PLAIN>(256, worlds_per_cu);
}

template hipError_t launch_resolve<double>(const ResolveLaunch<double>&, hipStream_t);
template hipError_t launch_resolve<float>(const ResolveLaunch<float>&, hipStream_t);

}  // namespace cbz
