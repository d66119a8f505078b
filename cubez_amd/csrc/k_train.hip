// k_train.hip — one optimiser step of the surrogate network in two launches:
// the rows (forward, and back through the activations), then the weight
// gradients with the update.  No counterpart in the reference.
//
// A step moves little (a batch of 4096 rows is 0.9 MB of features and labels,
// the weights with their optimiser state 4 MB) and multiplies 3.5 GFLOP, so
// what it costs is launches, passes over the activations and serial sums.
// Layer by layer it was 27 launches and 3.83 ms, 3.43 of them the bias
// gradients: a thread per column adding 4096 rows in order, each load waiting
// for the last.  An optimiser's trajectory keeps no rounding error small (a
// gradient near zero is divided by its own size), so every sum here still
// runs in the order it had; what changed is how many run side by side and
// how far ahead of them the loads are.  A step of 4096 rows now takes 40 us
// (k_train_rows 21, k_train_update 18), one of 33 rows 22 us.
#include "cbz_devmath.h"
#include "cbz_mfma.h"
#include "cbz_mlp.h"
#include "cbz_wave.h"

namespace cbz {

// Row i of training step `step` is SplitMix64(seed, step * n + i) mod rows
// (uniform with replacement).
__device__ __forceinline__ int64_t sample_row(uint64_t seed, uint64_t step, int n, int i, int64_t rows) {
  uint64_t z = seed * 0xD1B54A32D192ED03ull + (step * uint64_t(n) + uint64_t(i) + 1ull) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return int64_t(z % uint64_t(rows));
}

__device__ __forceinline__ float silu_grad(float z) {
  const float s = 1.0f / (1.0f + __expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

// A barrier for what waves exchange through LDS: global loads and stores stay in
// flight across it (__syncthreads waits for them).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ---------------------------------------------------------------------------
// forward and backward of the rows
// ---------------------------------------------------------------------------
// One workgroup of 8 waves takes 32 or 16 rows (one MFMA row tile, or half of
// one) through all layers and back.  Wave w owns features 32 w .. 32 w + 31 of
// every hidden layer; rows are the first operand, so a lane holds one feature
// of 16 (8) rows.  Its pre-activations of all three hidden layers stay in
// registers for the backward pass, where the same lane gets the gradients of the
// same feature and rows.  Activations pass from layer to layer through one LDS
// tile; a layer's weights, one contiguous 1 KB fragment per 16 inputs, are
// asked for before the tile is ready.  HBM sees the sampled rows in, and
// out what the weight gradients need: every layer's input and its dL/dZ as their
// fragments, 8 bytes (4 rows of a feature) per store.  The order of every dot
// product is that of k_gemm.  Bound by the chain of seven products with their
// barriers, and by the weights (0.6 MB per workgroup, from L2): 21 us at 4096
// rows.  Barriers that wait for global memory and loads under a condition
// (each then waits by itself) were 4 us of that together, products by
// row-major weights and 2-byte stores another 17.
constexpr int kTrainWaves = 8;
constexpr int kTrainThreads = 64 * kTrainWaves;
constexpr int kXStride = 72;  // LDS feature rows: 16-byte fragments, rows in different banks
constexpr int kDStride = 40;  // LDS rows of the output layer's gradient

// the fragments of 32 rows of a [rows][K] operand
template <int K>
__device__ __forceinline__ void load_frags(const __bf16* W, int row0, int lane, bf16x8 (&w)[kHidden / 16]) {
#pragma unroll
  for (int k = 0; k < K / 16; ++k) w[k] = *(const bf16x8*)(W + frag_at(row0, 16 * k, K) + 8 * lane);
}
// rows (LDS, element (r, k) at addr(r, k)) times those fragments
template <int K, typename Addr>
__device__ __forceinline__ f32x16 mul_frags(Addr addr, int r, int h, const bf16x8 (&w)[kHidden / 16]) {
  f32x16 acc = {};
#pragma unroll
  for (int k = 0; k < K / 16; ++k)  // the upper half of half a tile repeats the lower
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)addr(r, 16 * k + 8 * h), w[k], acc, 0, 0, 0);
  return acc;
}

template <int ROWS>
__global__ void __launch_bounds__(kTrainThreads) k_train_rows(TrainArgs f) {
  __shared__ __align__(16) __bf16 X[ROWS * kXStride];
  __shared__ __align__(16) __bf16 H[ROWS * kHidden];
  __shared__ __align__(16) __bf16 D[ROWS * kDStride];
  __shared__ float Y[ROWS * 16], T[ROWS * 16], E2[ROWS * 16];
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, r = lane & 31, h = lane >> 5;
  const int m0 = blockIdx.x * ROWS;
  const int col = wave * 32 + r;  // this lane's feature of the hidden layers
  const int ar = r & (ROWS - 1);  // this lane's row of the first operand
  auto x_at = [&](int row, int k) { return X + row * kXStride + k; };
  auto h_at = [&](int row, int k) { return H + fswz(row, k); };
  auto d_at = [&](int row, int k) { return D + row * kDStride + k; };
  // 4 rows (8q + 4h ..) of the lane's feature
  auto store_rows = [&](__bf16* P, int q, bf16x4 v) { *(bf16x4*)(P + batch_at(col, m0 + 8 * q + 4 * h, kHidden)) = v; };

  bf16x8 w[kHidden / 16];
  load_frags<kFeatPad>(f.Wf[0], wave * 32, lane, w);
  float bias[kLayers];
#pragma unroll
  for (int l = 0; l < kLayers; ++l) bias[l] = f.bias[l][l < kLayers - 1 ? col : min(r, kOut - 1)];
  if (t < 16 * ROWS) {  // the sampled rows, normalised; 16 threads per row
    const int row = t >> 4, q = t & 15, i = m0 + row;
    const bool v = i < f.M;
    const int64_t s = v ? (f.sample ? sample_row(f.seed, f.step, f.M, i, f.rows) : int64_t(i)) : 0;
    bf16x4 x;
    float raw[4], mean[4], inv[4];  // asked for together, whatever holds data (row 0 exists)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = min(4 * q + j, kFeat - 1);
      raw[j] = f.Xraw[s * kFeat + k], mean[j] = f.in_mean[k], inv[j] = f.in_inv_std[k];
    }
    const int y = min(q, kOut - 1);
    const float label = f.Yraw[s * kOut + y], ymean = f.out_mean[y], yinv = f.out_inv_std[y];
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = __bf16(v && 4 * q + j < kFeat ? (raw[j] - mean[j]) * inv[j] : 0.f);
    *(bf16x4*)x_at(row, 4 * q) = x;
    T[t] = v && q < kOut ? (label - ymean) * yinv : 0.f;
  }
  lds_barrier();
  if (t < 8 * ROWS) {  // the features' fragments: 64 features x groups of 8 rows
    const int k = t & 63, g = t >> 6;
    bf16x8 x;
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = *x_at(8 * g + j, k);
    *(bf16x8*)(f.At[0] + batch_at(k, m0 + 8 * g, layer_in_frag(0))) = x;
  }

  float Z[kLayers - 1][ROWS / 2];
#pragma unroll
  for (int l = 0; l < kLayers - 1; ++l) {
    const f32x16 acc = l == 0 ? mul_frags<kFeatPad>(x_at, ar, h, w) : mul_frags<kHidden>(h_at, ar, h, w);
    if (l < kLayers - 2) load_frags<kHidden>(f.Wf[l + 1], wave * 32, lane, w);
    if (l == kLayers - 2 && wave == 0) load_frags<kHidden>(f.Wf[l + 1], 0, lane, w);
    if (l > 0) lds_barrier();  // every wave has read the tile
#pragma unroll
    for (int q = 0; q < ROWS / 8; ++q) {
      bf16x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = 8 * q + 4 * h + j;
        const float z = acc[4 * q + j] + bias[l];
        Z[l][4 * q + j] = z;
        const float y = silu(z);
        v[j] = __bf16(m0 + row < f.M ? y : 0.f);
        *h_at(row, col) = v[j];
      }
      store_rows(f.At[l + 1], q, v);
    }
    lds_barrier();
  }
  // the output layer (one tile, wave 0), its error and its gradient
  if (wave == 0) {
    const f32x16 y = mul_frags<kHidden>(h_at, ar, h, w);
    if (r < 16) {
#pragma unroll
      for (int j = 0; j < ROWS / 2; ++j) Y[(8 * (j >> 2) + 4 * h + (j & 3)) * 16 + r] = y[j] + bias[kLayers - 1];
    }
  }
  load_frags<kOutPad>(f.Wb[kLayers - 1], wave * 32, lane, w);
  lds_barrier();
  const float scale = float(f.M * kOut);
  if (t < 16 * ROWS) {
    const int row = t >> 4, k = t & 15;
    float d = 0.f, e2 = 0.f;
    if (k < kOut && m0 + row < f.M) {
      const float e = Y[t] - T[t];
      e2 = e * e;
      d = 2.0f * e / scale;
    }
    E2[t] = e2;
    *d_at(row, k) = __bf16(d);
    *d_at(row, k + 16) = __bf16(0.f);
  }
  lds_barrier();
  if (t < ROWS) {
    float acc = 0.f;
    for (int k = 0; k < kOut; ++k) acc += E2[t * 16 + k];
    f.row_loss[m0 + t] = m0 + t < f.M ? acc / scale : 0.f;
  }
  if (t >= kTrainThreads - 4 * ROWS) {  // 32 outputs x groups of 8 rows
    const int k = t & 31, g = (t >> 5) & (ROWS / 8 - 1);
    bf16x8 d;
#pragma unroll
    for (int j = 0; j < 8; ++j) d[j] = *d_at(8 * g + j, k);
    *(bf16x8*)(f.dZt[kLayers - 1] + batch_at(k, m0 + 8 * g, kOutPad)) = d;
  }
  // back: dL/dA of layer l's input = dZ_l * W_l, times SiLU'(Z)
#pragma unroll
  for (int l = kLayers - 1; l > 0; --l) {
    const f32x16 acc = l == kLayers - 1 ? mul_frags<kOutPad>(d_at, ar, h, w) : mul_frags<kHidden>(h_at, ar, h, w);
    if (l > 1) load_frags<kHidden>(f.Wb[l - 1], wave * 32, lane, w);
    if (l < kLayers - 1) lds_barrier();
#pragma unroll
    for (int q = 0; q < ROWS / 8; ++q) {
      bf16x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = 8 * q + 4 * h + j;
        const float dz = acc[4 * q + j] * silu_grad(Z[l - 1][4 * q + j]);
        v[j] = __bf16(m0 + row < f.M ? dz : 0.f);
        if (l > 1) *h_at(row, col) = v[j];
      }
      store_rows(f.dZt[l - 1], q, v);
    }
    if (l > 1) lds_barrier();
  }
}

// ---------------------------------------------------------------------------
// weight gradients and the update
// ---------------------------------------------------------------------------
// One workgroup per 32 x 32 tile of a layer's dW = dZ^T * A over the whole
// batch (152 tiles), one per 64 bias gradients (13) and one for the loss, so
// every sum runs at the rate of its own dependent chain: Mpad / 16 matrix
// instructions for a tile, Mpad additions for a bias gradient.  What the chains
// wait for is the operands, written by other XCDs a moment ago and about a
// microsecond away: one wave of a workgroup runs the chain out of LDS, four keep
// the loads of the next stages in flight (96 KB for a tile, straight into LDS).
// A gradient is complete in its lane, so Adam on the FP32 master and the
// BF16 copies of the weight follow there.
//
// Each XCD has its own L2, and workgroups go to the XCDs in turn: XCD x takes
// a quarter of one of the two 256 x 256 layers as 4 x 4 tiles (half of its
// dZ and half of its A, 2 MB at 4096 rows, instead of all 4 MB of both layers),
// and an eighth of the rest.  18 us at 4096 rows; with the chain's own wave loading
// one stage of registers ahead it was 33, and 33 again as one product split over
// the batch with a reduction behind it, in another order.
constexpr int kDwBias = (3 * kHidden + kOut + 63) / 64;  // workgroups of bias gradients
constexpr int kDwFirst = (kDwBias + 1 + 7) / 8;          // of them and the loss, per XCD
constexpr int kDwTasks = kDwFirst + 16 + 2 + 1;          // workgroups per XCD
constexpr int kDwLoaders = 4;                            // waves that load; the last one computes
constexpr int kDwThreads = 64 * (kDwLoaders + 1);
constexpr int kDwStage = 16;                             // fragments of either operand per stage
constexpr int kDwSlots = 4;                              // stages in LDS
constexpr int kDbStage = 128;                            // rows per stage of a bias gradient
constexpr int kDbAhead = 4;                              // its stages in registers
constexpr int kDwLds = kDwSlots * kDwStage * 2 * 1024;
static_assert(kDwLds >= 2 * kDbStage * 64 * 4, "the bias gradients' two stages");

// Adam on parameter i, whose old value and moments are at hand
struct AdamStep {
  const UpdateArgs& f;
  __device__ __forceinline__ float operator()(int64_t i, float g, float p, float m, float v) const {
    f.grad[i] = g;
    if (!f.update) return p;
    const float mi = f.b1 * m + (1.f - f.b1) * g;
    const float vi = f.b2 * v + (1.f - f.b2) * g * g;
    f.m[i] = mi;
    f.v[i] = vi;
    p = p - f.lr * (mi * f.c1) / (sqrtf(vi * f.c2) + f.eps);
    f.p[i] = p;
    return p;
  }
};

typedef __attribute__((address_space(1))) const void gvoid;
typedef __attribute__((address_space(3))) void lvoid;

__device__ void dw_tile(const UpdateArgs& f, int l, int mt, int nt, char* lds) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int F = layer_out_pad(l), G = layer_in_frag(l), steps = f.Mpad / 16;
  const int stages = (steps + kDwStage - 1) / kDwStage;
  constexpr int kSlot = kDwStage * 2 * 1024;
  if (wave < kDwLoaders) {
    // two waves per operand, half a stage each: 8 fragments, one load each
    constexpr int kEach = kDwStage / 2;
    const bool second = wave >= 2;
    const __bf16* src = (second ? f.At[l] + nt * 512 : f.dZt[l] + mt * 512) + 8 * lane;
    const int64_t ld = 16 * (second ? G : F);
    const int k0 = (wave & 1) * kEach;
    char* dst = lds + (second ? kDwStage * 1024 : 0) + k0 * 1024;
    auto stage = [&](int s) {
      char* d = dst + (s % kDwSlots) * kSlot;
#pragma unroll
      for (int k = 0; k < kEach; ++k) {
        const int64_t q = min(s * kDwStage + k0 + k, steps - 1);  // past the end: any fragment, it is not used
        __builtin_amdgcn_global_load_lds((gvoid*)(src + q * ld), (lvoid*)(d + k * 1024), 16, 0, 0);
      }
    };
    for (int s = 0; s < kDwSlots - 1; ++s) stage(s);
    for (int s = 0; s < stages; ++s) {
      // this wave's part of stage s has landed: those of s+1 and s+2 may be out
      static_assert(kEach == 8 && kDwSlots == 4, "the count of loads that may be out");
      asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
      lds_barrier();  // stage s is in LDS; stage s-1 has been read
      stage(s + kDwSlots - 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }
  const int K = layer_in(l), N = layer_out(l), k = nt * 32 + r;
  float p[16], m[16], v[16];
  int64_t at[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int n = mt * 32 + 8 * (j >> 2) + 4 * h + (j & 3);
    at[j] = ((k < K) & (n < N)) ? f.off_w[l] + int64_t(n) * K + k : -1;
    const int64_t i = f.off_w[l] + int64_t(min(n, N - 1)) * K + min(k, K - 1);
    p[j] = f.p[i], m[j] = f.m[i], v[j] = f.v[i];
  }
  f32x16 acc = {};
  for (int s = 0; s < stages; ++s) {
    lds_barrier();
    const char* d = lds + (s % kDwSlots) * kSlot + 16 * lane;
    const int n = min(steps - s * kDwStage, kDwStage);
    bf16x8 a[kDwStage], b[kDwStage];
#pragma unroll
    for (int k = 0; k < kDwStage; ++k) {
      a[k] = *(const bf16x8*)(d + k * 1024);
      b[k] = *(const bf16x8*)(d + (kDwStage + k) * 1024);
    }
    auto mul = [&](int k) { acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[k], b[k], acc, 0, 0, 0); };
    if (n == kDwStage) {
#pragma unroll
      for (int k = 0; k < kDwStage; ++k) mul(k);
    } else {
#pragma unroll
      for (int k = 0; k < kDwStage; ++k)
        if (k < n) mul(k);
    }
  }
  const AdamStep adam{f};
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    if (at[j] < 0) continue;
    const int n = mt * 32 + 8 * (j >> 2) + 4 * h + (j & 3);
    const float w = adam(at[j], acc[j], p[j], m[j], v[j]);
    if (!f.update) continue;
    f.Wf[l][frag_at(n, k, layer_in_pad(l))] = __bf16(w);
    if (l > 0) f.Wb[l][frag_at(k, n, F)] = __bf16(w);
  }
}

// 64 bias gradients: the loading waves widen the rows to FP32 in LDS (4 rows of
// a column per 16 bytes), so that the chain is additions alone.
__device__ void db_columns(const UpdateArgs& f, int c, char* lds) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  c += lane;
  int l = 0;
  while (l < kLayers - 1 && c >= kHidden) c -= kHidden, ++l;
  const int F = layer_out_pad(l);
  const int groups = f.Mpad / 8, stages = (f.Mpad + kDbStage - 1) / kDbStage;
  constexpr int kSlot = kDbStage * 64 * 4, kEach = kDbStage / 8 / kDwLoaders;
  const bool valid = c < layer_out(l);
  if (wave < kDwLoaders) {
    const __bf16* a = f.dZt[l] + batch_at(valid ? c : 0, 0, F);
    bf16x8 x[kDbAhead][kEach];
    auto load = [&](int b, int s) {
#pragma unroll
      for (int g = 0; g < kEach; ++g) {
        const int64_t q = min(s * (kDbStage / 8) + wave * kEach + g, groups - 1);
        x[b][g] = *(const bf16x8*)(a + (q >> 1) * 16 * F + (q & 1) * 256);
      }
    };
#pragma unroll
    for (int s = 0; s < kDbAhead; ++s) load(s, s);
    for (int s0 = 0; s0 < stages; s0 += kDbAhead)
#pragma unroll
      for (int b = 0; b < kDbAhead; ++b) {
        const int s = s0 + b;
        if (s >= stages) break;
        float4* d = (float4*)(lds + (s & 1) * kSlot) + wave * kEach * 2 * 64 + lane;
#pragma unroll
        for (int g = 0; g < kEach; ++g) {
          const bf16x8 v = x[b][g];
          d[(2 * g) * 64] = float4{float(v[0]), float(v[1]), float(v[2]), float(v[3])};
          d[(2 * g + 1) * 64] = float4{float(v[4]), float(v[5]), float(v[6]), float(v[7])};
        }
        load(b, s + kDbAhead);
        lds_barrier();  // stage s is in LDS; stage s-1 has been read
      }
    return;
  }
  const int64_t i = f.off_b[l] + (valid ? c : 0);
  const float p = f.p[i], m = f.m[i], v = f.v[i];
  float sum = 0.f;
  for (int s = 0; s < stages; ++s) {
    lds_barrier();
    const float4* d = (const float4*)(lds + (s & 1) * kSlot) + lane;
    const int n = min(f.Mpad - s * kDbStage, kDbStage) / 32;
    float4 x[kDbStage / 4];
#pragma unroll
    for (int g = 0; g < kDbStage / 4; ++g) x[g] = d[g * 64];
#pragma unroll
    for (int q = 0; q < kDbStage / 32; ++q)
      if (q < n) {
#pragma unroll
        for (int g = 0; g < 8; ++g) {
          const float4 y = x[8 * q + g];
          sum += y.x;
          sum += y.y;
          sum += y.z;
          sum += y.w;
        }
      }
  }
  if (valid) AdamStep{f}(i, sum, p, m, v);
}

// The rows' losses: 256 strided sums, then halves.
__device__ void loss_sum(const UpdateArgs& f) {
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  float s[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    s[q] = 0.f;
    for (int k = lane + 64 * q; k < f.Mpad; k += 256) s[q] += f.row_loss[k];
  }
  float a = (s[0] + s[2]) + (s[1] + s[3]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
  if (lane == 0) f.loss[0] = a;
}

__global__ void __launch_bounds__(kDwThreads) k_train_update(UpdateArgs f) {
  __shared__ __align__(16) char lds[kDwLds];
  const int x = blockIdx.x & 7;
  int i = blockIdx.x >> 3;
  if (i < kDwFirst) {
    const int b = i * 8 + x;
    if (b < kDwBias)
      db_columns(f, b * 64, lds);
    else if (b == kDwBias)
      loss_sum(f);
    return;
  }
  i -= kDwFirst;
  int l = kLayers - 1, mt = 0, nt = x;
  if (i < 16)  // quarter x & 3 of layer 1 or 2
    l = 1 + (x >> 2), mt = (x & 1) * 4 + (i & 3), nt = ((x >> 1) & 1) * 4 + (i >> 2);
  else if (i < 18)
    l = 0, mt = x, nt = i - 16;
  dw_tile(f, l, mt, nt, lds);
}

hipError_t launch_train_rows(const TrainArgs& f, hipStream_t st) {
  if (f.M <= 0 || f.Mpad % 32 || f.Mpad < f.M) return hipErrorInvalidValue;
  // A workgroup fills a CU.  Up to 4096 rows half tiles have one each and
  // take less time than whole ones (20.8 against 23.2 us at 4096: half the
  // activations per lane); beyond that the chip is full, and half tiles would load and multiply twice as much.
  if (f.Mpad <= 4096)
    k_train_rows<16><<<f.Mpad / 16, kTrainThreads, 0, st>>>(f);
  else
    k_train_rows<32><<<f.Mpad / 32, kTrainThreads, 0, st>>>(f);
  return hipGetLastError();
}
hipError_t launch_train_update(const UpdateArgs& f, hipStream_t st) {
  static_assert(kHidden == 256 && kLayers == 4 && layer_in_frag(0) == 64 && kOutPad == 32, "the tasks of an XCD");
  if (f.Mpad <= 0 || f.Mpad % 32) return hipErrorInvalidValue;
  k_train_update<<<8 * kDwTasks, kDwThreads, 0, st>>>(f);
  return hipGetLastError();
}

}  // namespace cbz
