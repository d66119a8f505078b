// k_sort.hip — stable LSD radix sort of 64-bit keys for wave64, 8 bits a
// pass:
//   k_radix_hist     per tile of keys, the digit histogram ([tile][digit]);
//   k_radix_scatter  per tile, each key's rank among the tile's earlier keys
//                    of its digit.  A tile is four waves, each a contiguous
//                    run of ROUNDS rounds of 64 keys; within a round the lanes
//                    with the same digit are found with eight ballots, so a
//                    key's rank is the popcount of its group below its lane
//                    plus the running count of the digit in its wave, and
//                    a wave starts at its tile's offset plus the earlier
//                    waves' counts.  Equal digits keep the input order, so
//                    the sort is stable.
//
// The keys it is given are some 10^4 to 10^6: a pass moves less than a launch
// takes, so what counts is launches and the length of each one's serial part.
// A pass is two launches, since a tile adds up the histograms before it itself;
// with many tiles that is more work than one workgroup's scan of all of
// them, which is then a third launch (k_radix_scan).  Small sorts get tiles of
// 1024 keys instead of 4096: 40 workgroups for 40000 keys.
// 40000 keys with values: 10.5 us a pass; some 200000 pair keys: 20 us a pass.
// With tiles of 4096, a scan launch and each digit matched twice a pass of
// either took 32 us, and all eight digits had one; four have now.
#include <algorithm>

#include "cbz_sort.h"
#include "cbz_wave.h"

namespace cbz {

constexpr int kSortWaves = 4, kSortThreads = 64 * kSortWaves;
constexpr int kRadix = 256;
static_assert(kSortThreads == kRadix, "one thread per digit in the per-tile steps");
constexpr int kSortDirect = 128;                  // most tiles whose offsets the tiles add up
constexpr int64_t kSortSmall = kSortDirect << 10;  // keys: tiles of 1024 up to here, of 4096 above

static int sort_rounds(int64_t n) { return n <= kSortSmall ? 4 : 16; }
static int32_t sort_tiles(int64_t n) {
  const int64_t tile = int64_t(kSortThreads) * sort_rounds(n);
  return int32_t((n + tile - 1) / tile);
}

// The lanes of the wave whose digit equals this lane's (valid lanes only).
__device__ __forceinline__ uint64_t match_digit(uint32_t d, bool valid) {
  uint64_t m = __ballot(valid);
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const bool bit = (d >> b) & 1u;
    const uint64_t bb = __ballot(valid && bit);
    m &= bit ? bb : ~bb;
  }
  return m;
}

// Exclusive prefix of v over the 256 threads of a group of four waves (all
// threads of the workgroup call it; s: 4 words of LDS per group).
__device__ __forceinline__ uint32_t excl_256(uint32_t v, uint32_t* s) {
  const int t = threadIdx.x & 255, wv = t >> 6;
  const uint32_t inc = uint32_t(wave_incl_scan_i32(int(v)));
  if ((t & 63) == 63) s[wv] = inc;
  __syncthreads();
  uint32_t pre = inc - v;
  for (int u = 0; u < wv; ++u) pre += s[u];
  return pre;
}

template <int ROUNDS>
__global__ void __launch_bounds__(kSortThreads) k_radix_hist(const uint64_t* keys, int64_t n, int shift, uint32_t* hist) {
  __shared__ uint32_t s_cnt[kRadix];
  const int t = threadIdx.x;
  s_cnt[t] = 0;
  __syncthreads();
  const int64_t base = int64_t(blockIdx.x) * kSortThreads * ROUNDS;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int64_t i = base + int64_t(r) * kSortThreads + t;
    if (i < n) atomicAdd(&s_cnt[uint32_t(keys[i] >> shift) & 255u], 1u);
  }
  __syncthreads();
  hist[int64_t(blockIdx.x) * kRadix + t] = s_cnt[t];
}

// The histograms -> every (tile, digit)'s output offset, in place: one
// workgroup, a thread per digit and quarter of the tiles.
__global__ void __launch_bounds__(1024) k_radix_scan(uint32_t* hist, int32_t tiles) {
  __shared__ uint32_t s_sum[4][kRadix];
  __shared__ uint32_t s_wave[4][4];
  const int d = threadIdx.x & 255, g = threadIdx.x >> 8;
  const int64_t per = (tiles + 3) / 4;
  const int64_t b0 = min(g * per, int64_t(tiles)), b1 = min(b0 + per, int64_t(tiles));
  uint32_t sum = 0;
#pragma unroll 8
  for (int64_t i = b0; i < b1; ++i) sum += hist[i * kRadix + d];
  s_sum[g][d] = sum;
  __syncthreads();
  uint32_t tot = 0, pre = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    tot += s_sum[u][d];
    if (u < g) pre += s_sum[u][d];
  }
  pre += excl_256(tot, s_wave[g]);
#pragma unroll 8
  for (int64_t i = b0; i < b1; ++i) {
    const uint32_t h = hist[i * kRadix + d];
    hist[i * kRadix + d] = pre;
    pre += h;
  }
}

// hist: offsets (SCANNED), or the histograms of all tiles
template <int ROUNDS, bool VALS, bool SCANNED>
__global__ void __launch_bounds__(kSortThreads)
    k_radix_scatter(const uint64_t* kin, uint64_t* kout, const int32_t* vin, int32_t* vout, int64_t n, int shift,
                    const uint32_t* hist, int32_t tiles) {
  __shared__ uint32_t s_cnt[kSortWaves][kRadix];  // each wave's digit counts, then its first position per digit
  __shared__ uint32_t s_wave[4];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  for (int v = 0; v < kSortWaves; ++v) s_cnt[v][t] = 0;
  const int64_t wbase = (int64_t(blockIdx.x) * kSortWaves + wv) * ROUNDS * 64 + lane;
  uint64_t key[ROUNDS];
  int32_t val[ROUNDS];
  uint32_t rank[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int64_t i = wbase + r * 64;
    key[r] = i < n ? kin[i] : 0;
    if constexpr (VALS) val[r] = i < n ? vin[i] : 0;
  }
  uint32_t off = 0;
  if constexpr (SCANNED) {
    off = hist[int64_t(blockIdx.x) * kRadix + t];
    __syncthreads();
  } else {
    uint32_t tot = 0;
#pragma unroll 16
    for (int i = 0; i < tiles; ++i) {
      const uint32_t h = hist[i * kRadix + t];
      tot += h;
      off += i < int(blockIdx.x) ? h : 0u;
    }
    off += excl_256(tot, s_wave);
  }
  const uint64_t below = (uint64_t(1) << lane) - 1;
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const bool valid = wbase + r * 64 < n;
    const uint32_t d = uint32_t(key[r] >> shift) & 255u;
    const uint64_t m = match_digit(d, valid);
    // every lane of the group reads the running count before its lowest
    // lane advances it (one wave: the read precedes the write)
    rank[r] = s_cnt[wv][d] + uint32_t(__popcll(m & below));
    if (valid && (m & below) == 0) s_cnt[wv][d] += uint32_t(__popcll(m));
  }
  __syncthreads();
  for (int v = 0; v < kSortWaves; ++v) {
    const uint32_t c = s_cnt[v][t];
    s_cnt[v][t] = off;
    off += c;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    if (wbase + r * 64 >= n) break;
    const uint32_t pos = s_cnt[wv][uint32_t(key[r] >> shift) & 255u] + rank[r];
    kout[pos] = key[r];
    if constexpr (VALS) vout[pos] = val[r];
  }
}

static size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// One pass: histograms, their scan where there are many, and the scatter.
template <int ROUNDS, bool VALS>
static void radix_pass(const uint64_t* ks, uint64_t* kd, const int32_t* vs, int32_t* vd, int64_t n, int shift,
                       uint32_t* hist, int32_t tiles, hipStream_t st) {
  k_radix_hist<ROUNDS><<<tiles, kSortThreads, 0, st>>>(ks, n, shift, hist);
  if (tiles > kSortDirect) {
    k_radix_scan<<<1, 1024, 0, st>>>(hist, tiles);
    k_radix_scatter<ROUNDS, VALS, true><<<tiles, kSortThreads, 0, st>>>(ks, kd, vs, vd, n, shift, hist, tiles);
  } else {
    k_radix_scatter<ROUNDS, VALS, false><<<tiles, kSortThreads, 0, st>>>(ks, kd, vs, vd, n, shift, hist, tiles);
  }
}

size_t radix_sort_bytes(int64_t n, bool with_values) {
  if (n <= 0) return 256;
  size_t b = align256(size_t(n) * sizeof(uint64_t));
  if (with_values) b += align256(size_t(n) * sizeof(int32_t));
  // any smaller sort fits too: no more than kSortDirect tiles up to kSortSmall keys
  const size_t tiles = size_t(std::max<int64_t>(sort_tiles(n), n > kSortSmall ? kSortDirect : 0));
  return b + align256(kRadix * tiles * sizeof(uint32_t));
}

hipError_t radix_sort_u64(const uint64_t* keys_in, uint64_t* keys_out, const int32_t* vals_in, int32_t* vals_out,
                          int64_t n, void* tmp, size_t tmp_bytes, hipStream_t st, int lo_bits, int hi_bits) {
  if (n <= 0) return hipSuccess;
  const bool vals = vals_in != nullptr;
  if (n >= (int64_t(1) << 31) || (vals != (vals_out != nullptr)) || !tmp ||
      tmp_bytes < radix_sort_bytes(n, vals))
    return hipErrorInvalidValue;
  char* p = (char*)tmp;
  uint64_t* ktmp = (uint64_t*)p;
  p += align256(size_t(n) * sizeof(uint64_t));
  int32_t* vtmp = nullptr;
  if (vals) {
    vtmp = (int32_t*)p;
    p += align256(size_t(n) * sizeof(int32_t));
  }
  uint32_t* hist = (uint32_t*)p;
  const int lo = std::max(1, (lo_bits + 7) / 8), passes = lo + (hi_bits + 7) / 8;
  const int32_t tiles = sort_tiles(n);
  const bool small = sort_rounds(n) == 4;
  // each pass from the last one's output; the last writes out, the others
  // tmp and out alternately
  const uint64_t* ks = keys_in;
  const int32_t* vs = vals_in;
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = pass < lo ? 8 * pass : 32 + 8 * (pass - lo);
    const bool to_tmp = (passes - 1 - pass) & 1;
    uint64_t* kd = to_tmp ? ktmp : keys_out;
    int32_t* vd = to_tmp ? vtmp : vals_out;
    auto* run = vals ? (small ? radix_pass<4, true> : radix_pass<16, true>)
                     : (small ? radix_pass<4, false> : radix_pass<16, false>);
    run(ks, kd, vs, vd, n, shift, hist, tiles, st);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    ks = kd;
    vs = vd;
  }
  return hipSuccess;
}

}  // namespace cbz
