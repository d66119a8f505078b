// The part of the HIP device language that the resolver's headers use, for one
// workgroup at a time on the CPU: a fiber per thread, wave operations and
// barriers as the points where the fibers meet.
#pragma once
#include <math.h>
#include <setjmp.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <vector>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
using std::max;
using std::min;

typedef int hipError_t;
typedef void* hipStream_t;
typedef void* hipEvent_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipFuncAttributeMaxDynamicSharedMemorySize = 0 };
inline int hipGetLastError() { return 0; }
inline int hipFuncSetAttribute(const void*, int, int) { return 0; }
inline int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* p, const void*, int, size_t) { return *p = 1, 0; }
struct Index3 {
  unsigned x = 0, y = 0, z = 0;
};
inline Index3 threadIdx, blockIdx, blockDim, gridDim;
struct float4 {
  float x, y, z, w;
};
struct double2 {
  double x, y;
};

namespace emu {
// entered once through its context, then switched by jumps, which save no
// signal mask
struct Fiber {
  ucontext_t ctx;
  jmp_buf at;
  char* stack = nullptr;
  bool begun = false, done = false;
};
// a meeting point: who has arrived, of how many, and how often all had
struct Meet {
  int arrived = 0, alive = 0;
  long round = 0;
  void close() {
    if (alive > 0 && arrived >= alive) arrived = 0, ++round;
  }
};
constexpr int kWaves = 16;
inline std::vector<Fiber> fibers;
inline int cur;
inline jmp_buf scheduler;
inline Meet wave[kWaves], block;
inline uint64_t lanes[kWaves][2][64];

inline void meet(Meet& m) {
  const long r = m.round;
  ++m.arrived;
  m.close();
  while (m.round == r)
    if (!_setjmp(fibers[cur].at)) _longjmp(scheduler, 1);
}
inline void wave_sync() { meet(wave[cur >> 6]); }
// every lane's value of one wave operation
inline uint64_t* wave_put(uint64_t v) {
  const int w = cur >> 6;
  uint64_t* b = lanes[w][wave[w].round & 1];
  b[cur & 63] = v;
  wave_sync();
  return b;
}
template <class T>
uint64_t bits(T v) {
  uint64_t u = 0;
  memcpy(&u, &v, sizeof v);
  return u;
}
template <class T>
T of_bits(uint64_t u) {
  T v;
  memcpy(&v, &u, sizeof v);
  return v;
}
inline void fence(int, const char*) {}
inline int readlane(int v, int l) { return int(uint32_t(wave_put(uint32_t(v))[l & 63])); }
inline int readfirstlane(int v) { return readlane(v, 0); }
inline int update_dpp(int old, int v, int ctrl, int rows, int, bool) {
  const uint64_t* b = wave_put(uint32_t(v));
  const int l = cur & 63, r = l & 15, row = l & ~15;
  int s = -1;
  if (ctrl < 0x100)  // quad_perm
    s = (l & ~3) | ((ctrl >> (2 * (l & 3))) & 3);
  else if (ctrl > 0x110 && ctrl < 0x120)  // row_shr
    s = r >= (ctrl & 15) ? l - (ctrl & 15) : -1;
  else if (ctrl == 0x141)  // row_half_mirror
    s = row | (r & 8) | (7 - (r & 7));
  else if (ctrl == 0x140)  // row_mirror
    s = row | (15 - r);
  else if (ctrl == 0x142)  // row_bcast15
    s = l >= 16 ? row - 1 : -1;
  else if (ctrl == 0x143)  // row_bcast31
    s = l >= 32 ? 31 : -1;
  else
    abort();
  if (!((rows >> (l >> 4)) & 1) || s < 0) return old;
  return int(uint32_t(b[s]));
}
}  // namespace emu

#define __builtin_amdgcn_fence emu::fence
#define __builtin_amdgcn_wave_barrier emu::wave_sync
#define __builtin_amdgcn_readlane emu::readlane
#define __builtin_amdgcn_readfirstlane emu::readfirstlane
#define __builtin_amdgcn_update_dpp emu::update_dpp
#define __popcll(x) __builtin_popcountll(x)
inline void __syncthreads() { emu::meet(emu::block); }
inline void __threadfence() {}
inline void __threadfence_block() {}
template <class T>
T __shfl(T v, int l, int = 64) {
  return emu::of_bits<T>(emu::wave_put(emu::bits(v))[l & 63]);
}
template <class T>
T __shfl_xor(T v, int m, int = 64) {
  return __shfl(v, (emu::cur & 63) ^ m);
}
template <class T>
T __shfl_up(T v, int o, int = 64) {
  const int l = emu::cur & 63;
  return __shfl(v, l >= o ? l - o : l);
}
inline unsigned long long __ballot(int p) {
  const uint64_t* b = emu::wave_put(p != 0);
  unsigned long long r = 0;
  for (int i = 0; i < 64; ++i) r |= (unsigned long long)(b[i] & 1) << i;
  return r;
}
inline int __any(int p) { return __ballot(p) != 0; }
inline int __double2loint(double d) { return int(uint32_t(emu::bits(d))); }
inline int __double2hiint(double d) { return int(uint32_t(emu::bits(d) >> 32)); }
inline double __hiloint2double(int h, int l) { return emu::of_bits<double>(uint64_t(uint32_t(h)) << 32 | uint32_t(l)); }
inline int __float_as_int(float f) { return emu::of_bits<int>(emu::bits(f)); }
inline float __int_as_float(int i) { return emu::of_bits<float>(emu::bits(i)); }
template <class T>
T atomicAdd(T* p, T v) {
  const T o = *p;
  *p = o + v;
  return o;
}
template <class T>
T atomicCAS(T* p, T c, T v) {
  const T o = *p;
  if (o == c) *p = v;
  return o;
}
inline long long wall_clock64() { return 0; }
