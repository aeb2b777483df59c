// Shared helpers for the gfx950 kernels: storage types, wave64 and block reductions, error reporting.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

typedef __bf16 bf16;

#define TIS_WAVE 64

// dtype codes shared with the Python binding
#define TIS_F32 0
#define TIS_BF16 1

template <typename T> __device__ __forceinline__ float to_f(T v);
template <> __device__ __forceinline__ float to_f<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_f<bf16>(bf16 v) { return static_cast<float>(v); }

template <typename T> __device__ __forceinline__ T from_f(float v);
template <> __device__ __forceinline__ float from_f<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16 from_f<bf16>(float v) { return static_cast<bf16>(v); }

// What lane i ^ O holds of a value, in a butterfly over the wave (O = 32, 16, 8, 4, 2, 1 in turn): for O = 4 the value may by then depend on
// the lane's number modulo 8 alone, and a turn by four lanes brings the same. By lane swaps and moves between lanes, no trip through LDS, of
// which a butterfly by __shfl_xor makes six in a row (us, with those trips / without: the sum behind a layer and its norm, 5 rows of 1,024, 3.7 / 3.1; the
// choice of two experts of nine 6.7 / 4.9; a gate behind a head's norm 3.0 / 2.6). The same sums in the same order.
template <int O> __device__ __forceinline__ uint32_t butterfly_bits(uint32_t v) {
  if constexpr (O == 32) {
    auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return threadIdx.x & 32 ? s[0] : s[1];
  } else if constexpr (O == 16) {
    auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return threadIdx.x & 16 ? s[0] : s[1];
  } else {
    static_assert(O == 8 || O == 4 || O == 2 || O == 1, "a step of the butterfly");
    constexpr int MOVE = O == 8 ? 0x128 : O == 4 ? 0x124 : O == 2 ? 0x4E : 0xB1;      // row_ror:8, row_ror:4, quad_perm [2,3,0,1], [1,0,3,2]
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, MOVE, 0xF, 0xF, true);
  }
}
template <int O> __device__ __forceinline__ float butterfly(float v) { return __uint_as_float(butterfly_bits<O>(__float_as_uint(v))); }

// Sum and maximum over a wave whose 64 lanes are all there; every lane gets it.
__device__ __forceinline__ float wave_sum(float v) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  v += butterfly<8>(v);
  v += butterfly<4>(v);
  v += butterfly<2>(v);
  return v + butterfly<1>(v);
}
__device__ __forceinline__ float wave_max(float v) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
  v = fmaxf(v, butterfly<8>(v));
  v = fmaxf(v, butterfly<4>(v));
  v = fmaxf(v, butterfly<2>(v));
  return fmaxf(v, butterfly<1>(v));
}

// The largest value of a wave and its number, the lowest of those that share it; every lane gets both. (No value: -inf, 0x7fffffff.)
template <int O> __device__ __forceinline__ void argmax_step(float& v, int& at) {
  const float ov = butterfly<O>(v);
  const int oa = (int)butterfly_bits<O>((uint32_t)at);
  if (ov > v || (ov == v && oa < at)) { v = ov; at = oa; }
}
__device__ __forceinline__ void wave_argmax(float& v, int& at) {
  argmax_step<32>(v, at);
  argmax_step<16>(v, at);
  argmax_step<8>(v, at);
  argmax_step<4>(v, at);
  argmax_step<2>(v, at);
  argmax_step<1>(v, at);
}

// Sum over a block of up to 1024 threads. `scratch` holds 16 floats of LDS. Every thread gets the result.
// The order of additions depends only on the block size, never on the data or the grid.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  const int wave = threadIdx.x / TIS_WAVE, lane = threadIdx.x % TIS_WAVE;
  const int nw = (blockDim.x + TIS_WAVE - 1) / TIS_WAVE;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float r = 0.f;
  if (nw == 4) {               // (a loop of unknown length reads one at a time)
#pragma unroll
    for (int i = 0; i < 4; ++i) r += scratch[i];
    return r;
  }
  for (int i = 0; i < nw; ++i) r += scratch[i];
  return r;
}
__device__ __forceinline__ float block_max(float v, float* scratch) {
  v = wave_max(v);
  const int wave = threadIdx.x / TIS_WAVE, lane = threadIdx.x % TIS_WAVE;
  const int nw = (blockDim.x + TIS_WAVE - 1) / TIS_WAVE;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float r = scratch[0];
  if (nw == 4) {
#pragma unroll
    for (int i = 1; i < 4; ++i) r = fmaxf(r, scratch[i]);
    return r;
  }
  for (int i = 1; i < nw; ++i) r = fmaxf(r, scratch[i]);
  return r;
}

// ---- error reporting: every entry point returns 0 or a negative code and leaves a message here ----
static thread_local char tis_error_text[512];

static inline int tis_fail(const char* fmt, ...) __attribute__((format(printf, 1, 2)));
#include <stdarg.h>
static inline int tis_fail(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(tis_error_text, sizeof(tis_error_text), fmt, ap);
  va_end(ap);
  return -1;
}
static inline int tis_launch_status(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return tis_fail("%s: launch failed: %s", what, hipGetErrorString(e));
  return 0;
}
#define TIS_EXPORT extern "C" __attribute__((visibility("default")))
#define TIS_DEFINE_LAST_ERROR(prefix) \
  TIS_EXPORT const char* prefix##_last_error() { return tis_error_text; }

// The gate of a clamped gated feed-forward: g sigmoid(1.702 g) (u + 1) with g capped from above and u from both sides at `limit`.
__device__ __forceinline__ float clamped_swish(float g, float u, float limit) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.f + expf(-1.702f * g)) * (u + 1.f);
}
