// cbz_mlp.h — shapes and launch interfaces of the resolver surrogate MLP.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cbz_types.h"

namespace cbz {

constexpr int kFeat = 40;      // input features per contact
constexpr int kFeatPad = 48;   // padded to the MFMA K step (16)
constexpr int kHidden = 256;   // hidden width
constexpr int kOutVel = 12;    // outputs 0-11: dv0, dw0, dv1, dw1 (the velocity phase's changes)
constexpr int kOutPos = 12;    // output 12: the penetration the position phase resolves at the contact
constexpr int kOut = 13;       // outputs per contact
constexpr int kOutPad = 32;    // padded to the MFMA tile (32)
constexpr int kLayers = 4;
constexpr int kSurBodies = 256;     // bodies per world the surrogate takes
constexpr int kSurContacts = 2048;  // contacts per world the surrogate takes
// contacts per world the position polish takes; larger worlds get the plain
// position phase
constexpr int kSurPosContacts = 2048;

// layer l maps kIn[l] -> kOutL[l] features (unpadded)
__host__ __device__ constexpr int layer_in(int l) { return l == 0 ? kFeat : kHidden; }
__host__ __device__ constexpr int layer_out(int l) { return l == kLayers - 1 ? kOut : kHidden; }
__host__ __device__ constexpr int layer_in_pad(int l) { return l == 0 ? kFeatPad : kHidden; }
__host__ __device__ constexpr int layer_out_pad(int l) { return l == kLayers - 1 ? kOutPad : kHidden; }

// Matrix operands are stored as the MFMA fragments that the kernels load: 32
// rows x 16 contraction elements are 512 consecutive elements, lane r + 32 h
// of a wave taking the 16 bytes of row r, elements 8h .. 8h+7, so a fragment is
// one contiguous 1 KB load.  Element (row, k) of a [rows][K] operand (rows a
// multiple of 32, K of 16):
__host__ __device__ constexpr int64_t frag_at(int64_t row, int64_t k, int64_t K) {
  return ((row >> 5) * (K >> 4) + (k >> 4)) * 512 + ((k >> 3) & 1) * 256 + (row & 31) * 8 + (k & 7);
}
// The batch's transposed activations, feature f of F (a multiple of 32) and
// batch row i: the same fragments, those of 16 batch rows side by side.
__host__ __device__ constexpr int64_t batch_at(int64_t f, int64_t i, int64_t F) {
  return ((i >> 4) * (F >> 5) + (f >> 5)) * 512 + ((i >> 3) & 1) * 256 + (f & 31) * 8 + (i & 7);
}
// features of a layer's input in whole fragments
__host__ __device__ constexpr int layer_in_frag(int l) { return (layer_in_pad(l) + 31) / 32 * 32; }

struct GemmArgs {
  int M, N, K;                  // padded sizes: M, N multiples of 32, K of 16
  const __bf16* A;              // [M x K] row-major
  int64_t lda;
  const __bf16* Bt;             // [N x K] (B transposed) in fragments, see frag_at
  const float* bias;            // [N] or null
  int act;                      // 1: SiLU
  float* Y;                     // activation FP32 (or null)
  int64_t ldy;
  const float* y_scale;         // Y = act * scale + shift per column (or null)
  const float* y_shift;
  __bf16* H;                    // activation BF16 row-major (or null)
  int64_t ldh;
  int m_valid, n_valid;         // rows / columns that hold data
};

// fused inference forward: all four layers per block of rows
// Grid sizes of the grid-stride kernels of the surrogate step: whatever the
// contact count, one launch of at most this many workgroups covers it.
constexpr int kGridStrideBlocks = 8192;  // 256-thread workgroups (features)
constexpr int kMlpGridBlocks = 1024;     // fused-forward workgroups (2 per CU fit its LDS)

struct MlpArgs {
  int64_t M;                      // rows (the capacity when M_dev is set)
  const int64_t* M_dev = nullptr; // rows counted on the device (clamped to M), or null
  const __bf16* X;                // [M][kFeatPad] normalised features
  const __bf16* W[kLayers];       // per layer [Npad][Kpad] in fragments (the k_gemm Bt operand)
  const float* bias[kLayers];
  const float* y_scale;           // output = y * scale + shift (denormalisation)
  const float* y_shift;
  float* Y;                       // [M][kOut]
};

template <typename R>
struct SurApply {
  Bodies<R> b;
  Contacts<R> c;
  const int32_t* world_cnt;
  const int64_t* world_coff;
  const int32_t* body_off;
  const int32_t* overflow;
  const float* Y;               // [contacts][kOut] predictions
  float* delta;                 // out: [6][n_bodies] summed velocity and rotation change per body
  uint8_t* mask;                // out: 1 = plain velocity phase, 0 = polish
  float* dpos;                  // out: [6][n_bodies] summed position and orientation change per body
  uint8_t* pmask;               // out: 1 = plain position phase, 0 = polish (null: no position polish)
  int max_contacts;
};

// One optimiser step (k_train.hip).  Mpad: the rows rounded up to 32.
struct TrainArgs {
  int M, Mpad;
  const float* Xraw;  // [rows][kFeat] features, [rows][kOut] labels: sampled, or rows 0 .. M-1
  const float* Yraw;
  int64_t rows;
  int sample;
  uint64_t seed, step;
  const float *in_mean, *in_inv_std, *out_mean, *out_inv_std;
  const __bf16* Wf[kLayers];
  const __bf16* Wb[kLayers];
  const float* bias[kLayers];
  __bf16* At[kLayers];   // out: layer inputs, transposed, see batch_at
  __bf16* dZt[kLayers];  // out: dL/dZ, transposed
  float* row_loss;       // out: [Mpad]
};
struct UpdateArgs {
  int Mpad, update;  // update 0: the gradient and the loss alone
  const __bf16* At[kLayers];
  const __bf16* dZt[kLayers];
  const float* row_loss;
  int64_t off_w[kLayers], off_b[kLayers];
  float *loss, *grad, *p, *m, *v;
  __bf16* Wf[kLayers];
  __bf16* Wb[kLayers];
  float lr, b1, b2, eps, c1, c2;
};
hipError_t launch_train_rows(const TrainArgs& f, hipStream_t st);
hipError_t launch_train_update(const UpdateArgs& f, hipStream_t st);

hipError_t launch_gemm(const GemmArgs& g, hipStream_t st);
hipError_t launch_mlp_forward(const MlpArgs& f, hipStream_t st);
template <typename R>
hipError_t launch_features(const Bodies<R>& b, const Contacts<R>& c, int64_t n_cap, const int64_t* n_dev,
                           int32_t* deg, const float* mean, const float* inv_std, __bf16* X, float* raw,
                           hipStream_t st);
// The feature rows of the step's contacts (normalised BF16 rows into X and/or
// raw FP32 rows into raw, either may be null), one workgroup per world, the
// per-body contact counts in LDS; worlds of at most 4096 bodies (else
// hipErrorInvalidValue: use launch_features).
template <typename R>
hipError_t launch_features_world(const Bodies<R>& b, const Contacts<R>& c, const int32_t* world_cnt,
                                 const int64_t* world_coff, const int32_t* body_off, const int32_t* overflow,
                                 int n_worlds, int max_world_bodies, const float* mean, const float* inv_std,
                                 __bf16* X, float* raw, hipStream_t st);
template <typename R>
hipError_t launch_sur_scatter(const SurApply<R>& a, int n_worlds, hipStream_t st);
hipError_t launch_normalise_rows(const float* Xraw, int rows, int valid_rows, const float* in_mean,
                                 const float* in_inv_std, __bf16* X, hipStream_t st);
hipError_t launch_col_stats(const float* A, int64_t rows, int cols, float* mean, float* stdv, hipStream_t st);
// count of worlds whose byte is set in m or (when not null) in m2
hipError_t launch_count_u8(const uint8_t* m, int n, int32_t* out, hipStream_t st, const uint8_t* m2 = nullptr);
hipError_t launch_fill_f32(float* p, int64_t n, float v, hipStream_t st);
hipError_t launch_record_count(const int32_t* value, int32_t* hist, int32_t* ctr, int64_t cap, hipStream_t st);
hipError_t launch_pack_weights(const float* W, int N, int K, __bf16* Wf, int kpad, __bf16* Wb, int npad,
                               hipStream_t st);

}  // namespace cbz
