// k_broad.hip — sort-and-sweep broadphase in front of the explicit-list
// narrowphase, for worlds of thousands of bodies where the all-pairs space
// grows as n^2.
//
// Every body gets an axis-aligned box of half-width kBroadGrow * bounding
// radius around its collider centre.  The narrowphase's own far-pair test
// (k_narrow.hip, far_apart) rejects a body pair only when
// |t|^2 > k (rA + rB)^2 with k <= 3.003, so a pair it keeps has
// |t| <= sqrt(3.003) (rA + rB): its boxes overlap.  A body whose centre or
// radius is not finite overlaps everything (the reference still emits
// contacts for NaN states).  The kept ordered pairs (i, j) and (j, i) of
// every overlap, plus every body-plane pair, are sorted into the order of
// examples/cubedrop.go:47-64 (row i ascending, its planes first, then j
// ascending) and handed to the explicit-list narrowphase: its contacts are
// those of the all-pairs narrowphase, in the same order.  Both sorts are
// the stable radix sort of k_sort.hip.
#include "cbz_broad.h"
#include "cbz_launch.h"
#include "cbz_sort.h"
#include "cbz_wave.h"

namespace cbz {

// sqrt(3.003) = 1.73291..., rounded up with a margin for the rounding of
// the distance and radius sums
constexpr double kBroadGrow = 1.7330;

// float nearest to x in the direction of -inf / +inf (x finite)
__device__ __forceinline__ float f32_down(double x) {
  float f = float(x);
  if (double(f) > x) f = nextafterf(f, -INFINITY);
  return f;
}
__device__ __forceinline__ float f32_up(double x) {
  float f = float(x);
  if (double(f) < x) f = nextafterf(f, INFINITY);
  return f;
}
// order-preserving map of a float onto uint32 (-inf first)
__device__ __forceinline__ uint32_t f32_order(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float f32_unorder(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// bits of the numbers 0 .. n-1
static int bits_for(int64_t n) {
  int b = 0;
  while ((int64_t(1) << b) < n) ++b;
  return b;
}

// Boxes and the sort keys (world << 32 | ordered lower x bound, rounded down).
template <typename R>
__global__ void __launch_bounds__(256) k_bp_bounds(BroadArgs<R> a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.nb) return;
  const int64_t S = a.stride;
  const double cx = double(a.ctransform[9 * S + i]);
  const double cy = double(a.ctransform[10 * S + i]);
  const double cz = double(a.ctransform[11 * S + i]);
  const double r = kBroadGrow * a.brad[i];
  // a body that is not finite spans every axis
  BroadBox box{-INFINITY, -INFINITY, INFINITY, INFINITY};
  float hx = INFINITY;
  uint32_t kx = f32_order(-INFINITY);
  if (isfinite(cx) && isfinite(cy) && isfinite(cz) && isfinite(r)) {
    box = BroadBox{cy - r, cz - r, cy + r, cz + r};
    hx = f32_up(cx + r);
    kx = f32_order(f32_down(cx - r));
  }
  a.box[i] = box;
  a.hix[i] = hx;
  a.key_in[i] = (uint64_t(uint32_t(a.body_world[i])) << 32) | kx;
  a.val_in[i] = i;
}

// The body-plane pairs of every body: planes first in each row.
__global__ void __launch_bounds__(256) k_bp_planes(BroadPlanes p) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p.nb) return;
  const int w = p.body_world[i];
  const int b0 = p.body_off[w], np = p.plane_off[w + 1] - p.plane_off[w];
  const int64_t at = p.plane_pair_base[w] + int64_t(i - b0) * np;
  for (int k = 0; k < np; ++k) p.pkey[at + k] = (uint64_t(uint32_t(i)) << 32) | uint32_t(k);
}

// Sweep along x over each world's sorted boxes: position p meets the
// positions after it up to the first lower bound past its upper bound, y and z
// are tested, and both ordered pairs of every overlap are appended; entries
// past the capacity are counted and dropped.
//
// A workgroup takes 64 positions, one per lane of each of its 4 waves, and
// passes over what follows them in tiles of 128 boxes in LDS, a wave every
// fourth box: a box is one broadcast read for 64 tests.  Overlaps are collected
// in LDS, so that one atomic per workgroup reserves their places (a workgroup
// with more of them appends the rest one by one).  40000 bodies with about 300
// boxes each in reach along x take 36 us; with a thread per position walking them
// by itself, twice (to count, then to write), they took 1063.
constexpr int kSweepTile = 128;
constexpr int kSweepHits = 2048;

template <typename R>
__global__ void __launch_bounds__(256) k_bp_sweep(BroadArgs<R> a) {
  __shared__ BroadBox s_box[kSweepTile];
  __shared__ float s_lo[kSweepTile];
  __shared__ int s_j[kSweepTile];
  __shared__ int2 s_hit[kSweepHits];
  __shared__ int s_n;
  __shared__ long long s_base;
  const int t = threadIdx.x, wv = t >> 6;
  const int first = blockIdx.x * 64, p = first + (t & 63);
  if (t == 0) s_n = 0;
  // both keys of a pair, i's row first
  auto append = [&](int64_t at, int i, int j) {
    const int w = a.body_world[i], b0 = a.body_off[w];
    const int np = a.plane_off[w + 1] - a.plane_off[w];
    if (at < a.pcap) a.pkey[at] = (uint64_t(uint32_t(i)) << 32) | uint32_t(np + (j - b0));
    if (at + 1 < a.pcap) a.pkey[at + 1] = (uint64_t(uint32_t(j)) << 32) | uint32_t(np + (i - b0));
  };
  int i = 0, end = 0;
  float hx = 0.f;
  BroadBox b{};
  if (p < a.nb) {
    i = a.val_out[p];
    end = a.body_off[int(a.key_out[p] >> 32) + 1];
    hx = a.hix[i];
    b = a.box[i];
  }
  for (int q0 = first + 1;; q0 += kSweepTile) {
    __syncthreads();  // every wave is done with the last tile
    if (t < kSweepTile && q0 + t < a.nb) {
      const int j = a.val_out[q0 + t];
      s_j[t] = j;
      s_lo[t] = f32_unorder(uint32_t(a.key_out[q0 + t]));
      s_box[t] = a.box[j];
    }
    __syncthreads();
    // the same in every wave; false for all once q0 is past the last world
    if (!__any(p < a.nb && (p >= q0 || (q0 < end && s_lo[0] <= hx)))) break;
#pragma unroll 4
    for (int k = wv; k < kSweepTile; k += 4) {
      const BroadBox c = s_box[k];
      const int q = q0 + k;
      const bool keep = (q > p) & (q < end) & (s_lo[k] <= hx) & (c.lo_y <= b.hi_y) & (b.lo_y <= c.hi_y) &
                        (c.lo_z <= b.hi_z) & (b.lo_z <= c.hi_z);
      if (keep) {
        const int n = atomicAdd(&s_n, 1);
        if (n < kSweepHits)
          s_hit[n] = int2{i, s_j[k]};
        else
          append(a.plane_pairs + int64_t(atomicAdd((unsigned long long*)a.pcount, 2ull)), i, s_j[k]);
      }
    }
  }
  const int n = min(s_n, kSweepHits);
  if (t == 0 && n > 0) s_base = (long long)atomicAdd((unsigned long long*)a.pcount, 2ull * (unsigned long long)n);
  __syncthreads();
  for (int h = t; h < n; h += 256) append(a.plane_pairs + s_base + 2 * h, s_hit[h].x, s_hit[h].y);
}

// Sorted pair keys -> the explicit list (one, two); a plane is -(k+1).
__global__ void __launch_bounds__(256) k_bp_unpack(BroadList L) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= L.n) return;
  const uint64_t key = L.pkey[t];
  const int i = int(key >> 32);
  const int jk = int(uint32_t(key));
  const int w = L.body_world[i];
  const int np = L.plane_off[w + 1] - L.plane_off[w];
  L.one[t] = i;
  L.two[t] = jk < np ? -(L.plane_off[w] + jk + 1) : L.body_off[w] + (jk - np);
}

// World w's pairs start at the first key of its first body.
__global__ void __launch_bounds__(256) k_bp_world_off(BroadList L) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w > L.nw) return;
  const uint64_t want = uint64_t(uint32_t(L.body_off[w])) << 32;
  int64_t lo = 0, hi = L.n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (L.pkey[mid] < want)
      lo = mid + 1;
    else
      hi = mid;
  }
  L.list_off[w] = int32_t(lo);
}

template <typename R>
hipError_t launch_bp_bounds_sort(const BroadArgs<R>& a, void* tmp, size_t tmp_bytes, hipStream_t st) {
  if (a.nb <= 0) return hipSuccess;
  k_bp_bounds<R><<<(a.nb + 255) / 256, 256, 0, st>>>(a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return radix_sort_u64(a.key_in, a.key_out, a.val_in, a.val_out, a.nb, tmp, tmp_bytes, st, 32, bits_for(a.nw));
}

template <typename R>
hipError_t launch_bp_sweep(const BroadArgs<R>& a, const BroadPlanes& p, hipStream_t st) {
  if (a.nb <= 0) return hipSuccess;
  hipError_t e = launch_fill_i32((int32_t*)a.pcount, 2, 0, st);
  if (e != hipSuccess) return e;
  k_bp_planes<<<(p.nb + 255) / 256, 256, 0, st>>>(p);
  k_bp_sweep<R><<<(a.nb + 63) / 64, 256, 0, st>>>(a);
  return hipGetLastError();
}

hipError_t launch_bp_list(const BroadList& L, void* tmp, size_t tmp_bytes, hipStream_t st) {
  hipError_t e = hipSuccess;
  if (L.n > 0) {
    e = radix_sort_u64(L.pkey_in, L.pkey, nullptr, nullptr, L.n, tmp, tmp_bytes, st, bits_for(L.slots), bits_for(L.nb));
    if (e != hipSuccess) return e;
    k_bp_unpack<<<int((L.n + 255) / 256), 256, 0, st>>>(L);
  }
  k_bp_world_off<<<(L.nw + 1 + 255) / 256, 256, 0, st>>>(L);
  return hipGetLastError();
}

// Temporary storage the two radix sorts need for n bodies and m pair keys.
hipError_t bp_sort_bytes(int32_t n, int64_t m, size_t* bytes) {
  if (m >= (int64_t(1) << 31)) return hipErrorInvalidValue;
  const size_t b1 = radix_sort_bytes(n, true), b2 = radix_sort_bytes(m, false);
  *bytes = b1 > b2 ? b1 : b2;
  return hipSuccess;
}

template hipError_t launch_bp_bounds_sort<double>(const BroadArgs<double>&, void*, size_t, hipStream_t);
template hipError_t launch_bp_bounds_sort<float>(const BroadArgs<float>&, void*, size_t, hipStream_t);
template hipError_t launch_bp_sweep<double>(const BroadArgs<double>&, const BroadPlanes&, hipStream_t);
template hipError_t launch_bp_sweep<float>(const BroadArgs<float>&, const BroadPlanes&, hipStream_t);

}  // namespace cbz
