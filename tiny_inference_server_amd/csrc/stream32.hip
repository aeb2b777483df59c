// Row-wise kernels for models whose residual stream is kept in 32-bit whatever the compute type: scaled embedding,
// the gated sum followed by an RMS norm (norm after the sum), the closing RMS norm, the per-head norm and output gate
// of recurrent mixers, and the low-rank decay of gated linear attention.
//
// The RMS norm here is x / sqrt(mean(x^2) + eps) * gain, eps under the root. Every sum is taken in 32-bit in an order
// that depends on the row's width and on whether rows are read in fours (alignment, strides) alone; residual_norm's beyond 1,024
// columns also on whether the step has more than 64 rows. `T` is the compute type (float or bf16): what the next matrix product reads.
#include "common.h"

TIS_DEFINE_LAST_ERROR(tis_stream32)

static constexpr int S32_THREADS = 256;

__device__ __forceinline__ float sigmoid_f(float z) { return 1.f / (1.f + expf(-z)); }
__device__ __forceinline__ float log_sigmoid_f(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// x32[r] = table[token[r]] * scale, and the same rows in the compute type
template <typename T>
__global__ __launch_bounds__(S32_THREADS) void embed_scale_kernel(const T* __restrict__ table, const int* __restrict__ tokens,
                                                                   float scale, float* __restrict__ out32,
                                                                   T* __restrict__ outT, int D) {
  const long r = blockIdx.x;
  const T* src = table + (long)tokens[r] * D;
  for (int c = threadIdx.x; c < D; c += S32_THREADS) {
    const float v = to_f(src[c]) * scale;
    out32[r * D + c] = v;
    if (outT) outT[r * D + c] = from_f<T>(v);
  }
}

// r = alpha * x + sigmoid(gate + bias) * (s0 * y0 + s1 * y1);  out = r / sqrt(mean(r^2) + eps) * gain
// y1 and gate may be null (one branch; no gate).
template <typename T, int PER>      // PER: values a thread keeps in registers (width <= 256 * PER); 0: any width, through memory
__global__ __launch_bounds__(S32_THREADS) void gated_postnorm_kernel(
    const float* __restrict__ x, const float* __restrict__ y0, long ld0, float s0, const float* __restrict__ y1, long ld1,
    float s1, const float* __restrict__ gate, long ldg, const float* __restrict__ bias, float alpha,
    const float* __restrict__ gain, float eps, float* __restrict__ out32, T* __restrict__ outT, int D) {
  __shared__ float red[16];
  const long r = blockIdx.x;
  float ss = 0.f;
  float keep[PER > 0 ? PER : 1];
  auto summed = [&](int c) {
    float y = s0 * y0[r * ld0 + c];
    if (y1) y += s1 * y1[r * ld1 + c];
    if (gate) y *= sigmoid_f(gate[r * ldg + c] + (bias ? bias[c] : 0.f));
    return alpha * x[r * D + c] + y;
  };
  if (PER > 0) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int c = threadIdx.x + k * S32_THREADS;
      keep[k] = c < D ? summed(c) : 0.f;
      ss += keep[k] * keep[k];
    }
  } else {
    for (int c = threadIdx.x; c < D; c += S32_THREADS) {
      const float v = summed(c);
      out32[r * D + c] = v;
      ss += v * v;
    }
  }
  ss = block_sum(ss, red);      // (the order of this sum depends on the width alone, whichever way the values are kept)
  const float inv = 1.f / sqrtf(ss / (float)D + eps);
  if (PER > 0) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int c = threadIdx.x + k * S32_THREADS;
      if (c < D) {
        const float v = keep[k] * inv * gain[c];
        out32[r * D + c] = v;
        if (outT) outT[r * D + c] = from_f<T>(v);
      }
    }
  } else {
    for (int c = threadIdx.x; c < D; c += S32_THREADS) {
      const float v = out32[r * D + c] * inv * gain[c];
      out32[r * D + c] = v;
      if (outT) outT[r * D + c] = from_f<T>(v);
    }
  }
}

// Four neighbouring values at a time, 32-bit or in the compute type (16- or 8-byte pieces).
__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
__device__ __forceinline__ float4 load4(const bf16* p) {
  const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
  return make_float4((float)v[0], (float)v[1], (float)v[2], (float)v[3]);
}
__device__ __forceinline__ void store4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
__device__ __forceinline__ void store4(bf16* p, float4 v) {
  *reinterpret_cast<bf16x4*>(p) = (bf16x4){static_cast<__bf16>(v.x), static_cast<__bf16>(v.y), static_cast<__bf16>(v.z), static_cast<__bf16>(v.w)};
}
__device__ __forceinline__ float4 add4(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }
__device__ __forceinline__ float4 mul4(float4 a, float4 b) { return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w); }
__device__ __forceinline__ float4 scale4(float f, float4 a) { return make_float4(f * a.x, f * a.y, f * a.z, f * a.w); }
__device__ __forceinline__ float sum4(float4 a) { return (a.x + a.y) + (a.z + a.w); }
__device__ __forceinline__ float square4(float4 a) { return (a.x * a.x + a.y * a.y) + (a.z * a.z + a.w * a.w); }
// whether rows of 32-bit numbers at p, `ld` apart, may be read in such pieces (a null pointer may: it is not read)
static inline bool fours32(const void* p, long ld) { return !p || ((uintptr_t)p % 16 == 0 && ld % 4 == 0); }
static inline bool foursT(const void* p, long ld, int dtype) { return !p || ((uintptr_t)p % (dtype == TIS_F32 ? 16 : 8) == 0 && ld % 4 == 0); }

// The same for a width that is a multiple of four, PER pieces of four values a thread (width <= 4 PER THREADS): what bounds it
// is memory, and a lane's 4-byte loads of five arrays kept too little under way. us, 2,048 wide, before / now:
// 8 rows 7.2 / 3.4, 300 rows of 1,024 4.8 / 3.3, 1,531 rows 17.4 / 13.1, 2,048 rows 18.2 / 15.4.
template <typename T, int PER>
__global__ __launch_bounds__(S32_THREADS) void gated_postnorm_fours_kernel(
    const float* __restrict__ x, const float* __restrict__ y0, long ld0, float s0, const float* __restrict__ y1, long ld1,
    float s1, const float* __restrict__ gate, long ldg, const float* __restrict__ bias, float alpha,
    const float* __restrict__ gain, float eps, float* __restrict__ out32, T* __restrict__ outT, int D) {
  __shared__ float red[16];
  const long r = blockIdx.x;
  float4 xv[PER], y0v[PER], y1v[PER], zv[PER], gv[PER];
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (threadIdx.x + k * S32_THREADS) * 4;
    const bool in = c < D;
    xv[k] = in ? load4(x + r * D + c) : zero;
    y0v[k] = in ? load4(y0 + r * ld0 + c) : zero;
    y1v[k] = y1 && in ? load4(y1 + r * ld1 + c) : zero;
    zv[k] = gate && in ? load4(gate + r * ldg + c) : zero;
    if (gate && bias && in) zv[k] = add4(zv[k], load4(bias + c));
    gv[k] = in ? load4(gain + c) : zero;
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    float4 y = scale4(s0, y0v[k]);
    if (y1) y = add4(y, scale4(s1, y1v[k]));
    if (gate) y = mul4(y, make_float4(sigmoid_f(zv[k].x), sigmoid_f(zv[k].y), sigmoid_f(zv[k].z), sigmoid_f(zv[k].w)));
    xv[k] = add4(scale4(alpha, xv[k]), y);
    ss += square4(xv[k]);
  }
  const float inv = 1.f / sqrtf(block_sum(ss, red) / (float)D + eps);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (threadIdx.x + k * S32_THREADS) * 4;
    if (c >= D) continue;
    const float4 v = mul4(scale4(inv, xv[k]), gv[k]);
    store4(out32 + r * D + c, v);
    if (outT) store4(outT + r * D + c, v);
  }
}

// out = x / sqrt(mean(x^2) + eps) * gain, from the 32-bit stream into the compute type
template <typename T>
__global__ __launch_bounds__(S32_THREADS) void rmsnorm32_kernel(const float* __restrict__ x, long ldx, const float* __restrict__ gain,
                                                                 float eps, T* __restrict__ out, long ldo, int D) {
  __shared__ float red[16];
  const long r = blockIdx.x;
  float ss = 0.f;
  for (int c = threadIdx.x; c < D; c += S32_THREADS) {
    const float v = x[r * ldx + c];
    ss += v * v;
  }
  ss = block_sum(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)D + eps);
  for (int c = threadIdx.x; c < D; c += S32_THREADS) out[r * ldo + c] = from_f<T>(x[r * ldx + c] * inv * gain[c]);
}

// One wave per (row, head): o / sqrt(mean_over_V(o^2) + eps) * gain * act(g). gain is [V] shared by the heads or
// [H * V]; act 0: g * sigmoid(g), 1: sigmoid(g).
template <typename T>
__global__ __launch_bounds__(TIS_WAVE) void head_norm_gate_kernel(const float* __restrict__ o, long ldo,
                                                                   const float* __restrict__ g, long ldg,
                                                                   const float* __restrict__ gain, int gain_per_head,
                                                                   int act, float eps, T* __restrict__ out, long ldout,
                                                                   int V) {
  const long r = blockIdx.x;
  const int h = blockIdx.y;
  const float* src = o + r * ldo + (long)h * V;
  float ss = 0.f;
  for (int j = threadIdx.x; j < V; j += TIS_WAVE) ss += src[j] * src[j];
  ss = wave_sum(ss);
  const float inv = 1.f / sqrtf(ss / (float)V + eps);
  for (int j = threadIdx.x; j < V; j += TIS_WAVE) {
    const float z = g[r * ldg + (long)h * V + j];
    const float a = act == 0 ? z * sigmoid_f(z) : sigmoid_f(z);
    out[r * ldout + (long)h * V + j] = from_f<T>(src[j] * inv * gain[gain_per_head ? h * V + j : j] * a);
  }
}

// The same for channels that are a multiple of four, PER pieces of four a lane (V <= 256 PER): everything a head needs is asked for
// at once, where single values went to memory twice, one after the other. us, single values /
// fours: 8 rows of 8 heads of 256 2.9 / 2.3, 1,531 rows 8.5 / 6.1, 2,048 rows of 16 heads of 128 12.5 / 11.3.
template <typename T, int PER>
__global__ __launch_bounds__(TIS_WAVE) void head_norm_gate_fours_kernel(const float* __restrict__ o, long ldo,
                                                                         const float* __restrict__ g, long ldg,
                                                                         const float* __restrict__ gain, int gain_per_head,
                                                                         int act, float eps, T* __restrict__ out, long ldout,
                                                                         int V) {
  const long r = blockIdx.x;
  const int h = blockIdx.y;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 x[PER], z[PER], gn[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (threadIdx.x + k * TIS_WAVE) * 4;
    const bool in = c < V;
    x[k] = in ? load4(o + r * ldo + (long)h * V + c) : zero;
    z[k] = in ? load4(g + r * ldg + (long)h * V + c) : zero;
    gn[k] = in ? load4(gain + (gain_per_head ? h * V : 0) + c) : zero;
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) ss += square4(x[k]);
  const float inv = 1.f / sqrtf(wave_sum(ss) / (float)V + eps);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (threadIdx.x + k * TIS_WAVE) * 4;
    if (c >= V) continue;
    const float4 q = make_float4(sigmoid_f(z[k].x), sigmoid_f(z[k].y), sigmoid_f(z[k].z), sigmoid_f(z[k].w));
    store4(out + r * ldout + (long)h * V + c, mul4(mul4(scale4(inv, x[k]), gn[k]), act == 0 ? mul4(z[k], q) : q));
  }
}

// Layer norm of a 32-bit row into the compute type: (x - mean) / sqrt(var + eps) * gain + bias, the variance being the
// mean of the squared deviations (two passes over the row; bias may be null).
template <typename T>
__global__ __launch_bounds__(S32_THREADS) void layernorm32_kernel(const float* __restrict__ x, const float* __restrict__ gain,
                                                                   const float* __restrict__ bias, float eps,
                                                                   T* __restrict__ out, long ldo, int D) {
  __shared__ float red[16];
  const long r = blockIdx.x;
  float s = 0.f;
  for (int c = threadIdx.x; c < D; c += S32_THREADS) s += x[r * D + c];
  const float mean = block_sum(s, red) / (float)D;
  float ss = 0.f;
  for (int c = threadIdx.x; c < D; c += S32_THREADS) {
    const float d = x[r * D + c] - mean;
    ss += d * d;
  }
  const float inv = 1.f / sqrtf(block_sum(ss, red) / (float)D + eps);
  for (int c = threadIdx.x; c < D; c += S32_THREADS)
    out[r * ldo + c] = from_f<T>((x[r * D + c] - mean) * inv * gain[c] + (bias ? bias[c] : 0.f));
}

// The residual sum of a 32-bit stream, with what usually follows it, in one pass over the row:
//   v = x + y                                  (y_gain null)
//   v = x + y / sqrt(mean(y^2) + y_eps) * y_gain   (an RMS norm on the branch before the sum)
// v goes to out32 (which may be x itself); `copy` (nullable) gets v in the compute type; `normed` (nullable) gets the
// norm of v in the compute type: kind 1 layer norm (gain, bias), kind 2 RMS norm (gain), eps under the root in both.
// Where the branch is a routed feed-forward's result that has not been summed yet: y then holds a line per (row, choice),
// and the branch's value at row r is sum_k weights[r][k] * (y[r * top + k] if ids[r][k] < n_experts else rows[r]): an
// id from n_experts on is an identity expert, whose result is the row it was given. ids null: y is the branch itself.
struct ChosenSum {
  const int* ids;
  const float* weights;
  int top, n_experts;
  const void* rows;      // [rows][ldr] in the compute type: what the feed-forward read
  long ldr;
  const float* extra = nullptr;        // [rows][lde]: what every row adds beside its choices (a shared expert's result),
  long lde = 0;                        // times sigmoid(extra_gate[row * ldg]); null: nothing
  const float* extra_gate = nullptr;
  long ldg = 0;
};

// PER: values a thread keeps in registers (width <= 256 * PER), so that the row is read once and the sums follow one
// another without a trip to memory between them; 0: any width, through out32.
template <typename T, int PER, int THREADS>
__global__ __launch_bounds__(THREADS) void residual_norm_kernel(
    const float* __restrict__ x, const float* __restrict__ y_in, long ldy, const float* __restrict__ y_gain, float y_eps,
    float* __restrict__ out32, T* __restrict__ copy, long ldc, int norm_kind, const float* __restrict__ gain,
    const float* __restrict__ bias, float eps, T* __restrict__ normed, long ldn, int D, ChosenSum cs) {
  __shared__ float red[16];
  const long r = blockIdx.x;
  constexpr int P = PER > 0 ? PER : 1;
  const bool y = y_in != nullptr || cs.ids != nullptr;        // whether there is a branch at all
  // a row's choices and their weights, once for all its columns (up to 64 choices; beyond, from memory every time)
  __shared__ int chosen_id[64];
  __shared__ float chosen_w[64];
  const bool kept = cs.ids && cs.top <= 64;
  if (kept) {
    if (threadIdx.x < cs.top) {
      chosen_id[threadIdx.x] = cs.ids[r * cs.top + threadIdx.x];
      chosen_w[threadIdx.x] = cs.weights[r * cs.top + threadIdx.x];
    }
    __syncthreads();
  }
  auto y_at = [&](int c) {
    if (!cs.ids) return y_in[r * ldy + c];
    float v = 0.f;
    for (int k = 0; k < cs.top; ++k) {
      const int e = kept ? chosen_id[k] : cs.ids[r * cs.top + k];
      const float w = kept ? chosen_w[k] : cs.weights[r * cs.top + k];
      v += w * (e < cs.n_experts ? y_in[(r * cs.top + k) * ldy + c] : to_f(static_cast<const T*>(cs.rows)[r * cs.ldr + c]));
    }
    if (cs.extra) v += (cs.extra_gate ? sigmoid_f(cs.extra_gate[r * cs.ldg]) : 1.f) * cs.extra[r * cs.lde + c];
    return v;
  };
  // (everything the row's columns need is asked for at once: the gains and the bias too, which are only used after
  // the sums, so that no trip to memory stands between two of them)
  float xv[P], yv[P], ygv[P], gv[P], bv[P];
  if (PER > 0) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int c = threadIdx.x + k * THREADS;
      xv[k] = c < D ? x[r * D + c] : 0.f;
      yv[k] = (y && c < D) ? y_at(c) : 0.f;
      ygv[k] = (y && y_gain && c < D) ? y_gain[c] : 1.f;
      gv[k] = (norm_kind && c < D) ? gain[c] : 0.f;
      bv[k] = (norm_kind == 1 && bias && c < D) ? bias[c] : 0.f;
    }
  }
  float y_inv = 1.f;
  if (y && y_gain) {
    float ss = 0.f;
    if (PER > 0) {
#pragma unroll
      for (int k = 0; k < PER; ++k) ss += yv[k] * yv[k];
    } else {
      for (int c = threadIdx.x; c < D; c += THREADS) {
        const float v = y_at(c);
        ss += v * v;
      }
    }
    y_inv = 1.f / sqrtf(block_sum(ss, red) / (float)D + y_eps);
  }
  float s = 0.f;
  if (PER > 0) {
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int c = threadIdx.x + k * THREADS;
      if (c >= D) continue;
      float v = xv[k];
      if (y) v += y_gain ? yv[k] * y_inv * ygv[k] : yv[k];
      xv[k] = v;
      out32[r * D + c] = v;
      if (copy) copy[r * ldc + c] = from_f<T>(v);
      s += norm_kind == 2 ? v * v : v;
    }
  } else {
    for (int c = threadIdx.x; c < D; c += THREADS) {
      float v = x[r * D + c];
      if (y) v += y_gain ? y_at(c) * y_inv * y_gain[c] : y_at(c);
      out32[r * D + c] = v;          // (each thread reads back only what it wrote itself)
      if (copy) copy[r * ldc + c] = from_f<T>(v);
      s += norm_kind == 2 ? v * v : v;
    }
  }
  if (!normed || norm_kind == 0) return;
  // every value of the row that this thread holds (with its gain and bias), from its registers or from memory
  auto each = [&](auto fn) {
    if (PER > 0) {
#pragma unroll
      for (int k = 0; k < P; ++k) {
        const int c = threadIdx.x + k * THREADS;
        if (c < D) fn(xv[k], c, gv[k], bv[k]);
      }
    } else {
      for (int c = threadIdx.x; c < D; c += THREADS) fn(out32[r * D + c], c, gain[c], (norm_kind == 1 && bias) ? bias[c] : 0.f);
    }
  };
  if (norm_kind == 2) {
    const float inv = 1.f / sqrtf(block_sum(s, red) / (float)D + eps);
    each([&](float v, int c, float g, float) { normed[r * ldn + c] = from_f<T>(v * inv * g); });
    return;
  }
  const float mean = block_sum(s, red) / (float)D;
  float ss = 0.f;
  each([&](float v, int, float, float) { ss += (v - mean) * (v - mean); });
  const float inv = 1.f / sqrtf(block_sum(ss, red) / (float)D + eps);
  each([&](float v, int c, float g, float b) { normed[r * ldn + c] = from_f<T>((v - mean) * inv * g + b); });
}

// The same for a width that is a multiple of four, PER pieces of four values a thread (width <= 4 PER THREADS): a lane's
// 4-byte loads kept too little under way for many rows, and a row alone waits for fewer of the wider ones. us, 2,048 wide,
// before / now: a branch with a norm of its own, copy and next norm: 1 row 4.6 / 3.1, 1,531 rows 14.5 / 9.2, 2,048 rows
// 17.9 / 11.6; two chosen experts and a shared term: 8 rows 6.2 / 3.8, 65 rows 11.0 / 4.8, 2,048 rows 36.9 / 15.8.
template <typename T, int PER, int THREADS>
__global__ __launch_bounds__(THREADS) void residual_norm_fours_kernel(
    const float* __restrict__ x, const float* __restrict__ y_in, long ldy, const float* __restrict__ y_gain, float y_eps,
    float* __restrict__ out32, T* __restrict__ copy, long ldc, int norm_kind, const float* __restrict__ gain,
    const float* __restrict__ bias, float eps, T* __restrict__ normed, long ldn, int D, ChosenSum cs) {
  __shared__ float red[16];
  const long r = blockIdx.x;
  const bool y = y_in != nullptr || cs.ids != nullptr;        // whether there is a branch at all
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f), one = make_float4(1.f, 1.f, 1.f, 1.f);
  float4 xv[PER], yv[PER], ygv[PER], gv[PER], bv[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (threadIdx.x + k * THREADS) * 4;
    const bool in = c < D;
    xv[k] = in ? load4(x + r * D + c) : zero;
    yv[k] = y && !cs.ids && in ? load4(y_in + r * ldy + c) : zero;
    ygv[k] = y && y_gain && in ? load4(y_gain + c) : one;
    gv[k] = norm_kind && in ? load4(gain + c) : zero;
    bv[k] = norm_kind == 1 && bias && in ? load4(bias + c) : zero;
  }
  if (cs.ids) {                    // (a row's choices are the same for all its threads: scalar loads)
    for (int i = 0; i < cs.top; ++i) {
      const int e = cs.ids[r * cs.top + i];
      const float w = cs.weights[r * cs.top + i];
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int c = (threadIdx.x + k * THREADS) * 4;
        if (c < D)
          yv[k] = add4(yv[k], scale4(w, e < cs.n_experts ? load4(y_in + (r * cs.top + i) * ldy + c)
                                                         : load4(static_cast<const T*>(cs.rows) + r * cs.ldr + c)));
      }
    }
    if (cs.extra) {
      const float w = cs.extra_gate ? sigmoid_f(cs.extra_gate[r * cs.ldg]) : 1.f;
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int c = (threadIdx.x + k * THREADS) * 4;
        if (c < D) yv[k] = add4(yv[k], scale4(w, load4(cs.extra + r * cs.lde + c)));
      }
    }
  }
  float y_inv = 1.f;
  if (y && y_gain) {
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < PER; ++k) ss += square4(yv[k]);
    y_inv = 1.f / sqrtf(block_sum(ss, red) / (float)D + y_eps);
  }
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (threadIdx.x + k * THREADS) * 4;
    if (c >= D) continue;
    if (y) xv[k] = add4(xv[k], y_gain ? mul4(scale4(y_inv, yv[k]), ygv[k]) : yv[k]);
    store4(out32 + r * D + c, xv[k]);
    if (copy) store4(copy + r * ldc + c, xv[k]);
    s += norm_kind == 2 ? square4(xv[k]) : sum4(xv[k]);
  }
  if (!normed || norm_kind == 0) return;
  float mean = 0.f;
  if (norm_kind == 1) {
    mean = block_sum(s, red) / (float)D;
    s = 0.f;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int c = (threadIdx.x + k * THREADS) * 4;
      if (c < D) s += square4(add4(xv[k], make_float4(-mean, -mean, -mean, -mean)));
    }
  }
  const float inv = 1.f / sqrtf(block_sum(s, red) / (float)D + eps);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (threadIdx.x + k * THREADS) * 4;
    if (c >= D) continue;
    const float4 v = norm_kind == 2 ? xv[k] : add4(xv[k], make_float4(-mean, -mean, -mean, -mean));
    store4(normed + r * ldn + c, add4(mul4(scale4(inv, v), gv[k]), bv[k]));
  }
}

__device__ __forceinline__ float gelu_tanh_f(float z) {
  return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// out[r][j] = act(z[r][j]) * table[token[r]][j]: a gate on a row of a per-token table. act 0: tanh-form gelu, 1: silu,
// 2: sigmoid. z is 32-bit (a strided view is fine), table and out are in the compute type.
template <typename T>
__global__ __launch_bounds__(S32_THREADS) void gate_table_kernel(const float* __restrict__ z, long ldz,
                                                                  const T* __restrict__ table, long ldt,
                                                                  const int* __restrict__ tokens, int act,
                                                                  T* __restrict__ out, long ldo, int rows, int W) {
  const long i = (long)blockIdx.x * S32_THREADS + threadIdx.x;
  if (i >= (long)rows * W) return;
  const long r = i / W;
  const int j = (int)(i % W);
  const float v = z[r * ldz + j];
  const float a = act == 0 ? gelu_tanh_f(v) : act == 1 ? v * sigmoid_f(v) : sigmoid_f(v);
  out[r * ldo + j] = from_f<T>(a * to_f(table[(long)tokens[r] * ldt + j]));
}

// In place on the columns [0, W) of 32-bit rows: act 1 silu, 2 sigmoid, 0 tanh-form gelu.
__global__ __launch_bounds__(S32_THREADS) void activate32_kernel(float* __restrict__ z, long ldz, int act, int rows, int W) {
  const long i = (long)blockIdx.x * S32_THREADS + threadIdx.x;
  if (i >= (long)rows * W) return;
  float* p = z + (i / W) * ldz + (i % W);
  const float v = *p;
  *p = act == 0 ? gelu_tanh_f(v) : act == 1 ? v * sigmoid_f(v) : sigmoid_f(v);
}

// x[r][h * V + j] *= sigmoid(gate[r][h]), in place
template <typename T>
__global__ __launch_bounds__(S32_THREADS) void head_gate_kernel(T* __restrict__ x, long ldx, const float* __restrict__ gate,
                                                                 long ldg, int rows, int H, int V) {
  const long i = (long)blockIdx.x * S32_THREADS + threadIdx.x;
  const long W = (long)H * V;
  if (i >= rows * W) return;
  const long r = i / W;
  const int c = (int)(i % W);
  x[r * ldx + c] = from_f<T>(to_f(x[r * ldx + c]) * sigmoid_f(gate[r * ldg + c / V]));
}

#define S32_DISPATCH(call_f32, call_bf16)                 \
  if (dtype == TIS_F32) { call_f32; }                     \
  else if (dtype == TIS_BF16) { call_bf16; }              \
  else return tis_fail("unknown dtype code %d", dtype);

TIS_EXPORT int tis_embed_scale(int dtype, const void* table, const int* tokens, float scale, float* out32, void* outT,
                               int rows, int D, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || D < 1) return tis_fail("embed_scale: bad size rows=%d width=%d", rows, D);
  S32_DISPATCH((embed_scale_kernel<float><<<rows, S32_THREADS, 0, stream>>>((const float*)table, tokens, scale, out32, (float*)outT, D)),
               (embed_scale_kernel<bf16><<<rows, S32_THREADS, 0, stream>>>((const bf16*)table, tokens, scale, out32, (bf16*)outT, D)))
  return tis_launch_status("embed_scale");
}

TIS_EXPORT int tis_gated_postnorm(int dtype, const float* x, const float* y0, long ld0, float s0, const float* y1, long ld1,
                                  float s1, const float* gate, long ldg, const float* bias, float alpha, const float* gain,
                                  float eps, float* out32, void* outT, int rows, int D, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || D < 1 || !x || !y0 || !gain || !out32) return tis_fail("gated_postnorm: bad arguments rows=%d width=%d", rows, D);
#define S32_POSTNORM(T, PER)                                                                                           \
  gated_postnorm_kernel<T, PER><<<rows, S32_THREADS, 0, stream>>>(x, y0, ld0, s0, y1, ld1, s1, gate, ldg, bias, alpha, gain, \
                                                                  eps, out32, (T*)outT, D)
#define S32_POSTNORM4(T, PER)                                                                                          \
  gated_postnorm_fours_kernel<T, PER><<<rows, S32_THREADS, 0, stream>>>(x, y0, ld0, s0, y1, ld1, s1, gate, ldg, bias, alpha, \
                                                                        gain, eps, out32, (T*)outT, D)
  const bool fours = D % 4 == 0 && D <= 16 * S32_THREADS && fours32(x, D) && fours32(y0, ld0) && fours32(y1, ld1) &&
                     fours32(gate, ldg) && fours32(bias, 0) && fours32(gain, 0) && fours32(out32, D) && foursT(outT, D, dtype);
#define S32_POSTNORM_BY_WIDTH(T)                         \
  if (fours && D <= 4 * S32_THREADS) { S32_POSTNORM4(T, 1); }      \
  else if (fours && D <= 8 * S32_THREADS) { S32_POSTNORM4(T, 2); } \
  else if (fours) { S32_POSTNORM4(T, 4); }                \
  else if (D <= 4 * S32_THREADS) { S32_POSTNORM(T, 4); } \
  else if (D <= 16 * S32_THREADS) { S32_POSTNORM(T, 16); } \
  else { S32_POSTNORM(T, 0); }
  S32_DISPATCH(S32_POSTNORM_BY_WIDTH(float), S32_POSTNORM_BY_WIDTH(bf16))
#undef S32_POSTNORM_BY_WIDTH
#undef S32_POSTNORM4
#undef S32_POSTNORM
  return tis_launch_status("gated_postnorm");
}

TIS_EXPORT int tis_rmsnorm32(int dtype, const float* x, long ldx, const float* gain, float eps, void* out, long ldo, int rows, int D,
                             hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || D < 1) return tis_fail("rmsnorm32: bad size rows=%d width=%d", rows, D);
  S32_DISPATCH((rmsnorm32_kernel<float><<<rows, S32_THREADS, 0, stream>>>(x, ldx, gain, eps, (float*)out, ldo, D)),
               (rmsnorm32_kernel<bf16><<<rows, S32_THREADS, 0, stream>>>(x, ldx, gain, eps, (bf16*)out, ldo, D)))
  return tis_launch_status("rmsnorm32");
}

TIS_EXPORT int tis_head_norm_gate(int dtype, const float* o, long ldo, const float* g, long ldg, const float* gain,
                                  int gain_per_head, int act, float eps, void* out, long ldout, int rows, int H, int V,
                                  hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || H < 1 || H > 65535 || V < 1 || (act != 0 && act != 1))
    return tis_fail("head_norm_gate: bad size rows=%d heads=%d vdim=%d act=%d", rows, H, V, act);
  dim3 grid(rows, H);
  if (V % 4 == 0 && V <= 1024 && fours32(o, ldo) && fours32(g, ldg) && fours32(gain, 0) && foursT(out, ldout, dtype)) {
#define S32_HEADS(T, PER) \
  head_norm_gate_fours_kernel<T, PER><<<grid, TIS_WAVE, 0, stream>>>(o, ldo, g, ldg, gain, gain_per_head, act, eps, (T*)out, ldout, V)
    if (V <= 256) {
      S32_DISPATCH(S32_HEADS(float, 1), S32_HEADS(bf16, 1))
    } else {
      S32_DISPATCH(S32_HEADS(float, 4), S32_HEADS(bf16, 4))
    }
#undef S32_HEADS
    return tis_launch_status("head_norm_gate");
  }
  S32_DISPATCH((head_norm_gate_kernel<float><<<grid, TIS_WAVE, 0, stream>>>(o, ldo, g, ldg, gain, gain_per_head, act, eps, (float*)out, ldout, V)),
               (head_norm_gate_kernel<bf16><<<grid, TIS_WAVE, 0, stream>>>(o, ldo, g, ldg, gain, gain_per_head, act, eps, (bf16*)out, ldout, V)))
  return tis_launch_status("head_norm_gate");
}

static void launch_lowrank(const float* low, long ldl, int rank, const float* w2, const float* bias, int kind, float tau,
                           const float* rate, int group, float* out, int rows, int C, hipStream_t stream);

// sigmoid(z)^(1/tau), as exp(log_sigmoid(z) / tau), of z = low . w2^T + bias
TIS_EXPORT int tis_lowrank_decay(const float* low, long ldl, int rank, const float* w2, const float* bias, float tau,
                                 float* out, int rows, int C, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || rank < 1 || rank > 8192 || C < 1 || !(tau > 0.f))
    return tis_fail("lowrank_decay: bad size rows=%d rank=%d channels=%d tau=%g", rows, rank, C, (double)tau);
  launch_lowrank(low, ldl, rank, w2, bias, 0, tau, nullptr, 1, out, rows, C, stream);
  return tis_launch_status("lowrank_decay");
}

TIS_EXPORT int tis_layernorm32(int dtype, const float* x, const float* gain, const float* bias, float eps, void* out, long ldo,
                               int rows, int D, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || D < 1 || !x || !gain || !out) return tis_fail("layernorm32: bad arguments rows=%d width=%d", rows, D);
  S32_DISPATCH((layernorm32_kernel<float><<<rows, S32_THREADS, 0, stream>>>(x, gain, bias, eps, (float*)out, ldo, D)),
               (layernorm32_kernel<bf16><<<rows, S32_THREADS, 0, stream>>>(x, gain, bias, eps, (bf16*)out, ldo, D)))
  return tis_launch_status("layernorm32");
}

TIS_EXPORT int tis_residual_norm(int dtype, const float* x, const float* y, long ldy, const float* y_gain, float y_eps,
                                 float* out32, void* copy, long ldc, int norm_kind, const float* gain, const float* bias,
                                 float eps, void* normed, long ldn, int rows, int D, const int* ids, const float* weights,
                                 int top, int n_experts, const void* chosen_rows, long ldr, const float* extra, long lde,
                                 const float* extra_gate, long ldg, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || D < 1 || !x || !out32) return tis_fail("residual_norm: bad arguments rows=%d width=%d", rows, D);
  if (ids && (!weights || top < 1 || n_experts < 0 || (n_experts > 0 && !y) || !chosen_rows))
    return tis_fail("residual_norm: a sum over chosen experts needs ids, weights, the experts' results and the rows they read");
  if (extra && !ids) return tis_fail("residual_norm: a shared term goes with chosen experts");
  const ChosenSum cs{ids, weights, top, n_experts, chosen_rows, ldr, extra, lde, extra_gate, ldg};
  if (norm_kind < 0 || norm_kind > 2 || (norm_kind && (!gain || !normed)))
    return tis_fail("residual_norm: norm kind %d needs a gain and an output", norm_kind);
#define S32_RESIDUAL(T, PER, THREADS)                                                                                      \
  residual_norm_kernel<T, PER, THREADS><<<rows, THREADS, 0, stream>>>(x, y, ldy, y_gain, y_eps, out32, (T*)copy, ldc, norm_kind, \
                                                                      gain, bias, eps, (T*)normed, ldn, D, cs)
#define S32_RESIDUAL4(T, PER, THREADS)                                                                                     \
  residual_norm_fours_kernel<T, PER, THREADS><<<rows, THREADS, 0, stream>>>(x, y, ldy, y_gain, y_eps, out32, (T*)copy, ldc, \
                                                                            norm_kind, gain, bias, eps, (T*)normed, ldn, D, cs)
  const bool fours = D % 4 == 0 && D <= 4096 && fours32(x, D) && fours32(y, ldy) && fours32(y_gain, 0) && fours32(out32, D) &&
                     foursT(copy, ldc, dtype) && fours32(gain, 0) && fours32(bias, 0) && foursT(normed, ldn, dtype) &&
                     foursT(chosen_rows, ldr, dtype) && fours32(extra, lde);
  // (a step of few rows leaves most of the chip idle: the widest workgroups then, for the shortest chains. What cannot be
  // read in fours, or is wider than a thread's registers hold, goes through the kernel of single values.)
#define S32_RESIDUAL_BY_WIDTH(T)                                                        \
  if (fours && D <= 1024) { S32_RESIDUAL4(T, 1, 256); }                                 \
  else if (fours && rows <= 64 && D <= 2048) { S32_RESIDUAL4(T, 1, 512); }              \
  else if (fours && rows <= 64) { S32_RESIDUAL4(T, 1, 1024); }                          \
  else if (fours && D <= 2048) { S32_RESIDUAL4(T, 2, 256); }                            \
  else if (fours) { S32_RESIDUAL4(T, 4, 256); }                                         \
  else if (rows <= 64 && D > 1024 && D <= 4096) { S32_RESIDUAL(T, 4, 1024); }                  \
  else if (D <= 4 * S32_THREADS) { S32_RESIDUAL(T, 4, S32_THREADS); }                     \
  else if (D <= 16 * S32_THREADS) { S32_RESIDUAL(T, 16, S32_THREADS); }                   \
  else { S32_RESIDUAL(T, 0, S32_THREADS); }
  S32_DISPATCH(S32_RESIDUAL_BY_WIDTH(float), S32_RESIDUAL_BY_WIDTH(bf16))
#undef S32_RESIDUAL_BY_WIDTH
#undef S32_RESIDUAL4
#undef S32_RESIDUAL
  return tis_launch_status("residual_norm");
}

TIS_EXPORT int tis_gate_table(int dtype, const float* z, long ldz, const void* table, long ldt, const int* tokens, int act,
                              void* out, long ldo, int rows, int W, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || W < 1 || act < 0 || act > 2) return tis_fail("gate_table: bad size rows=%d width=%d act=%d", rows, W, act);
  const long blocks = ((long)rows * W + S32_THREADS - 1) / S32_THREADS;
  S32_DISPATCH((gate_table_kernel<float><<<blocks, S32_THREADS, 0, stream>>>(z, ldz, (const float*)table, ldt, tokens, act, (float*)out, ldo, rows, W)),
               (gate_table_kernel<bf16><<<blocks, S32_THREADS, 0, stream>>>(z, ldz, (const bf16*)table, ldt, tokens, act, (bf16*)out, ldo, rows, W)))
  return tis_launch_status("gate_table");
}

TIS_EXPORT int tis_activate32(float* z, long ldz, int act, int rows, int W, hipStream_t stream) {
  if (rows == 0 || W == 0) return 0;
  if (rows < 0 || W < 0 || act < 0 || act > 2) return tis_fail("activate32: bad size rows=%d width=%d act=%d", rows, W, act);
  const long blocks = ((long)rows * W + S32_THREADS - 1) / S32_THREADS;
  activate32_kernel<<<blocks, S32_THREADS, 0, stream>>>(z, ldz, act, rows, W);
  return tis_launch_status("activate32");
}

TIS_EXPORT int tis_head_gate(int dtype, void* x, long ldx, const float* gate, long ldg, int rows, int H, int V,
                             hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || H < 1 || V < 1) return tis_fail("head_gate: bad size rows=%d heads=%d vdim=%d", rows, H, V);
  const long blocks = ((long)rows * H * V + S32_THREADS - 1) / S32_THREADS;
  S32_DISPATCH((head_gate_kernel<float><<<blocks, S32_THREADS, 0, stream>>>((float*)x, ldx, gate, ldg, rows, H, V)),
               (head_gate_kernel<bf16><<<blocks, S32_THREADS, 0, stream>>>((bf16*)x, ldx, gate, ldg, rows, H, V)))
  return tis_launch_status("head_gate");
}

// ---- blocks whose sublayers all read one norm of the stream and are summed with a factor per channel ---------------

// Dynamic tanh: out = tanh(alpha * x) * gain + bias, element by element (no mean, no variance), in the compute type.
template <typename T>
__global__ __launch_bounds__(S32_THREADS) void dyt32_kernel(const float* __restrict__ x, float alpha,
                                                             const float* __restrict__ gain, const float* __restrict__ bias,
                                                             T* __restrict__ out, long ldo, int D, int row_blocks) {
  const long r = blockIdx.x / row_blocks;      // grid (rows * blocks of columns, a row's side by side): a few rows still fill the chip
  const int c = (blockIdx.x % row_blocks) * S32_THREADS + threadIdx.x;
  if (c < D) out[r * ldo + c] = from_f<T>(tanhf(alpha * x[r * D + c]) * gain[c] + (bias ? bias[c] : 0.f));
}

// One branch of a scaled sum: s[c] * (y[r][c] + b[c]); s and b may be null (1 and 0). With `cs.ids` the branch is the
// not yet summed result of a routed feed-forward (see ChosenSum; weights may be null: every choice counts once).
struct ScaledBranch {
  const float* y;
  long ld;
  const float* scale;
  const float* bias;
};

// x <- x + sum over the branches, in place or into out32; `normed` (nullable) gets the dynamic tanh of the new row in
// the compute type (the norm that the next block, or the model's end, reads the stream through). grid (rows * blocks of
// columns, a row's blocks side by side): every element is on its own, and a step of a few rows still spreads over the chip.
template <typename T>
__global__ __launch_bounds__(S32_THREADS) void scaled_sum_kernel(const float* __restrict__ x, ScaledBranch a, ScaledBranch b,
                                                                  ChosenSum cs, float* __restrict__ out32, int norm_kind,
                                                                  float alpha, const float* __restrict__ gain,
                                                                  const float* __restrict__ nbias, T* __restrict__ normed,
                                                                  long ldn, int D, int row_blocks) {
  const long r = blockIdx.x / row_blocks;
  __shared__ int chosen_id[64];
  __shared__ float chosen_w[64];
  const bool kept = cs.ids && cs.top <= 64;
  if (kept) {
    if (threadIdx.x < cs.top) {
      chosen_id[threadIdx.x] = cs.ids[r * cs.top + threadIdx.x];
      chosen_w[threadIdx.x] = cs.weights ? cs.weights[r * cs.top + threadIdx.x] : 1.f;
    }
    __syncthreads();
  }
  const int c = (blockIdx.x % row_blocks) * S32_THREADS + threadIdx.x;
  if (c < D) {
    float v = x[r * D + c];
    if (a.y) v += (a.scale ? a.scale[c] : 1.f) * (a.y[r * a.ld + c] + (a.bias ? a.bias[c] : 0.f));
    if (cs.ids) {
      float y = 0.f;
      for (int k = 0; k < cs.top; ++k) {
        const int e = kept ? chosen_id[k] : cs.ids[r * cs.top + k];
        const float w = kept ? chosen_w[k] : (cs.weights ? cs.weights[r * cs.top + k] : 1.f);
        y += w * (e < cs.n_experts ? b.y[(r * cs.top + k) * b.ld + c] : to_f(static_cast<const T*>(cs.rows)[r * cs.ldr + c]));
      }
      v += (b.scale ? b.scale[c] : 1.f) * (y + (b.bias ? b.bias[c] : 0.f));
    } else if (b.y) {
      v += (b.scale ? b.scale[c] : 1.f) * (b.y[r * b.ld + c] + (b.bias ? b.bias[c] : 0.f));
    }
    out32[r * D + c] = v;
    if (norm_kind == 3) normed[r * ldn + c] = from_f<T>(tanhf(alpha * v) * gain[c] + (nbias ? nbias[c] : 0.f));
  }
}

// out[r][j] = act(w_r * (z[r][j] + gb[j])) * (w_r * (z[r][F + j] + ub[j])): the gate of a gated feed-forward on a
// 32-bit product whose first F columns are the gate's and whose next F the other factor's. Biases and the factor per
// row (a router's weight on the row that an expert read) may be null. act 0: tanh-form gelu, 1: silu, 2: see below. pairs: the
// columns alternate instead, gate 0, factor 0, gate 1, ...
template <typename T>
__global__ __launch_bounds__(S32_THREADS) void gated_act_kernel(const float* __restrict__ z, long ldz, int F,
                                                                 const float* __restrict__ gb, const float* __restrict__ ub,
                                                                 const float* __restrict__ row_scale, int act,
                                                                 T* __restrict__ out, long ldo, int rows, float limit, int pairs) {
  const long i = (long)blockIdx.x * S32_THREADS + threadIdx.x;
  if (i >= (long)rows * F) return;
  const long r = i / F;
  const int j = (int)(i % F);
  const float w = row_scale ? row_scale[r] : 1.f;
  const long at = r * ldz + (pairs ? 2 * j : j);
  float g = w * (z[at] + (gb ? gb[j] : 0.f)), u = w * (z[at + (pairs ? 1 : F)] + (ub ? ub[j] : 0.f));
  if (act == 2) {      // g sigmoid(1.702 g) (u + 1) with g capped from above and u from both sides at `limit`
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    out[r * ldo + j] = from_f<T>(g * sigmoid_f(1.702f * g) * (u + 1.f));
    return;
  }
  out[r * ldo + j] = from_f<T>((act == 0 ? gelu_tanh_f(g) : g * sigmoid_f(g)) * u);
}

// z <- cap * tanh(z / cap) on 32-bit rows, in place
__global__ __launch_bounds__(S32_THREADS) void softcap_kernel(float* __restrict__ z, long ldz, float cap, int rows, int W) {
  const long i = (long)blockIdx.x * S32_THREADS + threadIdx.x;
  if (i >= (long)rows * W) return;
  float* p = z + (i / W) * ldz + (i % W);
  *p = cap * tanhf(*p / cap);
}

TIS_EXPORT int tis_dyt32(int dtype, const float* x, float alpha, const float* gain, const float* bias, void* out, long ldo,
                         int rows, int D, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || D < 1 || !x || !gain || !out) return tis_fail("dyt32: bad arguments rows=%d width=%d", rows, D);
  const int row_blocks = (D + S32_THREADS - 1) / S32_THREADS;
  if ((long)rows * row_blocks > 0x7fffffffL) return tis_fail("dyt32: %d rows of %d in one call", rows, D);
  S32_DISPATCH((dyt32_kernel<float><<<rows * row_blocks, S32_THREADS, 0, stream>>>(x, alpha, gain, bias, (float*)out, ldo, D, row_blocks)),
               (dyt32_kernel<bf16><<<rows * row_blocks, S32_THREADS, 0, stream>>>(x, alpha, gain, bias, (bf16*)out, ldo, D, row_blocks)))
  return tis_launch_status("dyt32");
}

TIS_EXPORT int tis_scaled_sum(int dtype, const float* x, const float* y0, long ld0, const float* s0, const float* b0,
                              const float* y1, long ld1, const float* s1, const float* b1, const int* ids,
                              const float* weights, int top, int n_experts, const void* chosen_rows, long ldr,
                              float* out32, int norm_kind, float alpha, const float* gain, const float* nbias, void* normed,
                              long ldn, int rows, int D, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || D < 1 || !x || !out32) return tis_fail("scaled_sum: bad arguments rows=%d width=%d", rows, D);
  if (ids && (top < 1 || n_experts < 0 || (n_experts > 0 && !y1) || !chosen_rows))
    return tis_fail("scaled_sum: a sum over chosen experts needs ids, the experts' results and the rows they read");
  if ((norm_kind != 0 && norm_kind != 3) || (norm_kind && (!gain || !normed)))
    return tis_fail("scaled_sum: norm kind %d (0: none, 3: dynamic tanh, with a gain and an output)", norm_kind);
  const ScaledBranch a{y0, ld0, s0, b0}, b{y1, ld1, s1, b1};
  const ChosenSum cs{ids, weights, top, n_experts, chosen_rows, ldr};
  const int row_blocks = (D + S32_THREADS - 1) / S32_THREADS;
  if ((long)rows * row_blocks > 0x7fffffffL) return tis_fail("scaled_sum: %d rows of %d in one call", rows, D);
  const int grid = rows * row_blocks;
  S32_DISPATCH((scaled_sum_kernel<float><<<grid, S32_THREADS, 0, stream>>>(x, a, b, cs, out32, norm_kind, alpha, gain, nbias, (float*)normed, ldn, D, row_blocks)),
               (scaled_sum_kernel<bf16><<<grid, S32_THREADS, 0, stream>>>(x, a, b, cs, out32, norm_kind, alpha, gain, nbias, (bf16*)normed, ldn, D, row_blocks)))
  return tis_launch_status("scaled_sum");
}

TIS_EXPORT int tis_gated_act(int dtype, const float* z, long ldz, int F, const float* gate_bias, const float* up_bias,
                             const float* row_scale, int act, void* out, long ldo, int rows, float limit, int pairs,
                             hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || F < 1 || act < 0 || act > 2 || (act == 2 && !(limit > 0.f)))
    return tis_fail("gated_act: bad size rows=%d hidden=%d act=%d limit=%g", rows, F, act, (double)limit);
  const long blocks = ((long)rows * F + S32_THREADS - 1) / S32_THREADS;
  S32_DISPATCH((gated_act_kernel<float><<<blocks, S32_THREADS, 0, stream>>>(z, ldz, F, gate_bias, up_bias, row_scale, act, (float*)out, ldo, rows, limit, pairs)),
               (gated_act_kernel<bf16><<<blocks, S32_THREADS, 0, stream>>>(z, ldz, F, gate_bias, up_bias, row_scale, act, (bf16*)out, ldo, rows, limit, pairs)))
  return tis_launch_status("gated_act");
}

TIS_EXPORT int tis_softcap(float* z, long ldz, float cap, int rows, int W, hipStream_t stream) {
  if (rows == 0 || W == 0) return 0;
  if (rows < 0 || W < 0 || !(cap > 0.f)) return tis_fail("softcap: bad arguments rows=%d width=%d cap=%g", rows, W, (double)cap);
  const long blocks = ((long)rows * W + S32_THREADS - 1) / S32_THREADS;
  softcap_kernel<<<blocks, S32_THREADS, 0, stream>>>(z, ldz, cap, rows, W);
  return tis_launch_status("softcap");
}

// ---- blocks with a norm on both sides of a sublayer, several mixers side by side -----------------------------------

// out[r][c] = act(z) with z = sum_k low[r][k] * w2[c][k] + bias[c] (bias may be null): the second half of a low-rank
// projection, in 32-bit. kind 0: sigmoid(z)^(1/tau); 1: exp(-rate[c / group] * softplus(z)), a decay whose rate is one
// number per run of `group` channels; 2: z itself.
// A workgroup takes 32 channels and 8 RT rows, a thread one channel of RT of them, and both factors come through LDS in chunks of LR_K of
// the rank, read in whole runs (a thread that walked its channel's line of w2 by itself touched a line of memory per lane and
// term, and 5 rows of 512 channels were two workgroups). k in rising order for every row, whatever RT. us before / now, rank 64: 5 rows
// x 1,024 7.0 / 4.3, 64 x 1,024 8.5 / 4.4, 1,531 x 1,024 15.4 / 12.4, 1,531 x 2,048 25.0 / 22.4; with all of a chunk's loads under way
// together (before, each waited for the one before it), traced inside a pass, before / now: 5 rows 7.0 / 4.0, 1,531 rows, the two widths' mean, 20.1 / 13.1.
static constexpr int LR_COLS = 32, LR_BY = S32_THREADS / LR_COLS;
struct LowRank {
  const float* low;
  long ldl;
  int rank;
  const float *w2, *bias;
  int kind;
  float tau;
  const float* rate;
  int group;
  float* out;
  int C, col_blocks;
};
// x, y: the products of one launch; y's workgroups follow x's, of which there are `of_x` (one product: all)
template <int RT, int LR_K, int V>
__global__ __launch_bounds__(S32_THREADS) void lowrank_act_kernel(LowRank x, LowRank y, int of_x, int rows) {
  const bool first = (int)blockIdx.x < of_x;
  const int block = first ? blockIdx.x : blockIdx.x - of_x;
  const float *__restrict__ low = first ? x.low : y.low, *__restrict__ w2 = first ? x.w2 : y.w2, *__restrict__ bias = first ? x.bias : y.bias;
  const float* __restrict__ rate = first ? x.rate : y.rate;
  float* __restrict__ out = first ? x.out : y.out;
  const long ldl = first ? x.ldl : y.ldl;
  const int rank = first ? x.rank : y.rank, kind = first ? x.kind : y.kind, group = first ? x.group : y.group, C = first ? x.C : y.C;
  const int col_blocks = first ? x.col_blocks : y.col_blocks;
  const float tau = first ? x.tau : y.tau;
  __shared__ __attribute__((aligned(16))) float w[LR_COLS][LR_K + 4], a[LR_BY * RT][LR_K];
  typedef __attribute__((ext_vector_type(V))) float floats;
  constexpr int LINE = LR_K / V, WS = LR_COLS * LINE, AS = LR_BY * RT * LINE;      // pieces a line, of w's tile and of a's
  constexpr int WN = (WS + S32_THREADS - 1) / S32_THREADS, AN = (AS + S32_THREADS - 1) / S32_THREADS;
  // grid (blocks of rows * blocks of channels, a row block's side by side)
  const long r0 = (long)(block / col_blocks) * (LR_BY * RT);
  const int n = (int)min((long)LR_BY * RT, rows - r0);
  const int c0 = (block % col_blocks) * LR_COLS, cl = threadIdx.x % LR_COLS, rl = threadIdx.x / LR_COLS, c = c0 + cl;
  const float b = bias && c < C ? bias[c] : 0.f;
  const float rt = kind == 1 && c < C ? rate[c / group] : 0.f;
  float z[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) z[i] = 0.f;
  for (int k0 = 0; k0 < rank; k0 += LR_K) {
    // all of a chunk's loads at once, from addresses that always hold something (a load under a condition is waited for before the next)
    floats hw[WN], ha[AN];
#pragma unroll
    for (int i = 0; i < WN; ++i) {
      const int at = i * S32_THREADS + threadIdx.x, row = c0 + at / LINE, k = k0 + at % LINE * V;
      hw[i] = *reinterpret_cast<const floats*>(w2 + (long)min(row, C - 1) * rank + min(k, rank - V));
      if (row >= C || k >= rank) hw[i] = (floats)0.f;
    }
#pragma unroll
    for (int i = 0; i < AN; ++i) {
      const int at = i * S32_THREADS + threadIdx.x, row = at / LINE, k = k0 + at % LINE * V;
      ha[i] = *reinterpret_cast<const floats*>(low + (r0 + min(row, n - 1)) * ldl + min(k, rank - V));
      if (row >= n || k >= rank) ha[i] = (floats)0.f;
    }
    if (k0) __syncthreads();
#pragma unroll
    for (int i = 0; i < WN; ++i) {
      const int at = i * S32_THREADS + threadIdx.x;
      if (WS % S32_THREADS == 0 || at < WS) *reinterpret_cast<floats*>(&w[at / LINE][at % LINE * V]) = hw[i];
    }
#pragma unroll
    for (int i = 0; i < AN; ++i) {
      const int at = i * S32_THREADS + threadIdx.x;
      if (AS % S32_THREADS == 0 || at < AS) *reinterpret_cast<floats*>(&a[at / LINE][at % LINE * V]) = ha[i];
    }
    __syncthreads();
    const int kc = min(LR_K, rank - k0);
    for (int k = 0; k < kc; k += 4) {            // (terms past the rank are zeros)
      const float4 wk = *reinterpret_cast<const float4*>(&w[cl][k]);
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const float4 ak = *reinterpret_cast<const float4*>(&a[rl + i * LR_BY][k]);
        z[i] = fmaf(ak.w, wk.w, fmaf(ak.z, wk.z, fmaf(ak.y, wk.y, fmaf(ak.x, wk.x, z[i]))));
      }
    }
  }
  if (c >= C) return;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    if (rl + i * LR_BY >= n) break;
    float v = z[i] + b;
    if (kind == 0) v = expf(log_sigmoid_f(v) / tau);
    else if (kind == 1) v = expf(-rt * (v > 20.f ? v : log1pf(expf(v))));
    out[(r0 + rl + i * LR_BY) * C + c] = v;
  }
}

// Eight rows a workgroup while the chip holds all of them at a time, eight a unit of up to 64 terms of the rank (four where a rank of up to
// 32 leaves little to do but the results): the shortest chain. 32 rows beyond, which read w2 a quarter as often. And a chunk of the rank is no longer than a
// short rank is, or copying zeros is most of the work. us, eight rows / 32: rank 64, 256 rows x 1,024 6.3 / 8.1, 256 x 2,048 8.5 / 9.0, 257 x 2,048
// 10.9 / 8.9, 2,048 x 2,048 52 / 31; 2,048 x 32 4.6 / 7.7; rank 16, 256 x 1,024 4.6 / 4.7, 1,000 x 512 7.1 / 5.5, 2,048 x 4,096 71 / 34 (43
// in chunks of 64; a channel's line of w2 walked by one thread: 31); 1 row x 1,024 3.3 (4.1 in chunks of 64).
// Which of the kernel's forms a product takes: rows a thread, chunk of the rank, values a load.
struct LowRankForm {
  bool few, fours;
  int chunk;
  long blocks;
  bool operator==(const LowRankForm& o) const { return few == o.few && fours == o.fours && chunk == o.chunk; }
};
static LowRankForm lowrank_form(const LowRank& p, int rows) {
  const long small = ((long)rows + LR_BY - 1) / LR_BY * p.col_blocks;
  const bool few = small <= (p.rank > 32 ? 2048 : 1024);
  // lines that start on 16 bytes are read 16 at a time
  return {few, p.rank % 4 == 0 && p.ldl % 4 == 0 && ((uintptr_t)p.low | (uintptr_t)p.w2) % 16 == 0, p.rank <= 16 ? 16 : p.rank <= 32 ? 32 : 64,
          few ? small : ((long)rows + 4 * LR_BY - 1) / (4 * LR_BY) * p.col_blocks};
}
static void launch_lowrank(const LowRank& x, const LowRank* y, int rows, hipStream_t stream) {
  const LowRankForm f = lowrank_form(x, rows);
  const long blocks = f.blocks + (y ? lowrank_form(*y, rows).blocks : 0);
#define LOWRANK(RT, K, V) lowrank_act_kernel<RT, K, V><<<blocks, S32_THREADS, 0, stream>>>(x, y ? *y : x, (int)f.blocks, rows)
#define LOWRANK_BY_ROWS(K) { if (f.fours) { if (f.few) LOWRANK(1, K, 4); else LOWRANK(4, K, 4); } else { if (f.few) LOWRANK(1, K, 1); else LOWRANK(4, K, 1); } }
  if (f.chunk == 16) LOWRANK_BY_ROWS(16)
  else if (f.chunk == 32) LOWRANK_BY_ROWS(32)
  else LOWRANK_BY_ROWS(64)
#undef LOWRANK_BY_ROWS
#undef LOWRANK
}
static void launch_lowrank(const float* low, long ldl, int rank, const float* w2, const float* bias, int kind, float tau,
                           const float* rate, int group, float* out, int rows, int C, hipStream_t stream) {
  launch_lowrank(LowRank{low, ldl, rank, w2, bias, kind, tau, rate, group, out, C, (C + LR_COLS - 1) / LR_COLS}, nullptr, rows, stream);
}

// out[r] = (1 / n) * sum_i y_i[r] / sqrt(mean(y_i[r]^2) + eps) * gain_i: the mean of one or two RMS-normed rows, 32-bit.
// One workgroup a row; the sums' order depends on the width (and on whether it can be read in fours, see below) alone.
__global__ __launch_bounds__(S32_THREADS) void normed_mean_kernel(const float* __restrict__ y0, long ld0,
                                                                   const float* __restrict__ g0,
                                                                   const float* __restrict__ y1, long ld1,
                                                                   const float* __restrict__ g1, float eps,
                                                                   float* __restrict__ out, int D) {
  __shared__ float red[16];
  const long r = blockIdx.x;
  float s0 = 0.f, s1 = 0.f;
  for (int c = threadIdx.x; c < D; c += S32_THREADS) {
    const float a = y0[r * ld0 + c];
    s0 += a * a;
    if (y1) {
      const float b = y1[r * ld1 + c];
      s1 += b * b;
    }
  }
  const float i0 = 1.f / sqrtf(block_sum(s0, red) / (float)D + eps);
  const float i1 = y1 ? 1.f / sqrtf(block_sum(s1, red) / (float)D + eps) : 0.f;
  const float share = y1 ? 0.5f : 1.f;
  for (int c = threadIdx.x; c < D; c += S32_THREADS) {
    float v = y0[r * ld0 + c] * i0 * g0[c];
    if (y1) v += y1[r * ld1 + c] * i1 * g1[c];
    out[r * D + c] = v * share;
  }
}

// The same for a width that is a multiple of four, PER pieces of four a thread (width <= 4 PER THREADS): both rows and gains are
// asked for at once and stay in registers, and both sums meet in one pass through LDS: every wave sums runs of 256 columns, and the runs'
// sums are added in the order of the columns, whichever threads they come from, so a row's bits are the same on workgroups of any
// size. us, 2,048 wide, single values / fours: 8 rows 5.3 / 2.5, 1,531 rows 10.7 / 7.1, 2,048 rows 13.6 / 8.6 (added in the order of the
// threads, which tells 64 rows from 65: 2.5, 6.4, 8.7; workgroups of 512 for every number of rows: 2.5, 7.4, 9.6).
template <int PER, int THREADS>
__global__ __launch_bounds__(THREADS) void normed_mean_fours_kernel(const float* __restrict__ y0, long ld0,
                                                                     const float* __restrict__ g0,
                                                                     const float* __restrict__ y1, long ld1,
                                                                     const float* __restrict__ g1, float eps,
                                                                     float* __restrict__ out, int D) {
  constexpr int WAVES = THREADS / TIS_WAVE;
  __shared__ float2 red[PER * WAVES];
  const long r = blockIdx.x;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  // (multiply-adds spelled out: which of two products the compiler takes into one may differ from kernel to kernel)
  auto squares = [](float4 v) { return fmaf(v.y, v.y, v.x * v.x) + fmaf(v.w, v.w, v.z * v.z); };
  auto both = [](float p, float g, float q, float h) { return fmaf(p, g, q * h); };
  float4 a[PER], b[PER], ga[PER], gb[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (threadIdx.x + k * THREADS) * 4;
    const bool in = c < D;
    a[k] = in ? load4(y0 + r * ld0 + c) : zero;
    b[k] = y1 && in ? load4(y1 + r * ld1 + c) : zero;
    ga[k] = in ? load4(g0 + c) : zero;
    gb[k] = y1 && in ? load4(g1 + c) : zero;
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const float2 run = make_float2(wave_sum(squares(a[k])), wave_sum(squares(b[k])));
    if (threadIdx.x % TIS_WAVE == 0) red[k * WAVES + threadIdx.x / TIS_WAVE] = run;
  }
  __syncthreads();
  float s0 = 0.f, s1 = 0.f;
#pragma unroll
  for (int i = 0; i < PER * WAVES; ++i) {
    s0 += red[i].x;
    s1 += red[i].y;
  }
  const float i0 = 1.f / sqrtf(s0 / (float)D + eps), i1 = y1 ? 1.f / sqrtf(s1 / (float)D + eps) : 0.f;
  const float share = y1 ? 0.5f : 1.f;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = (threadIdx.x + k * THREADS) * 4;
    if (c >= D) continue;
    const float4 p = scale4(i0, a[k]), q = scale4(i1, b[k]);
    float4 v = mul4(p, ga[k]);
    if (y1) v = make_float4(both(p.x, ga[k].x, q.x, gb[k].x), both(p.y, ga[k].y, q.y, gb[k].y), both(p.z, ga[k].z, q.z, gb[k].z), both(p.w, ga[k].w, q.w, gb[k].w));
    store4(out + r * D + c, scale4(share, v));
  }
}

// out = act(z) in the compute type, z 32-bit (a strided view is fine). act 0: tanh-form gelu, 1: silu, 2: sigmoid,
// 3: the square of relu.
template <typename T>
__global__ __launch_bounds__(S32_THREADS) void activate_rows_kernel(const float* __restrict__ z, long ldz, int act,
                                                                     T* __restrict__ out, long ldo, int rows, int W) {
  const long i = (long)blockIdx.x * S32_THREADS + threadIdx.x;
  if (i >= (long)rows * W) return;
  const long r = i / W;
  const int j = (int)(i % W);
  const float v = z[r * ldz + j];
  const float p = fmaxf(v, 0.f);
  out[r * ldo + j] = from_f<T>(act == 0 ? gelu_tanh_f(v) : act == 1 ? v * sigmoid_f(v) : act == 2 ? sigmoid_f(v) : p * p);
}

TIS_EXPORT int tis_lowrank_act(const float* low, long ldl, int rank, const float* w2, const float* bias, int kind, float tau,
                               const float* rate, int group, float* out, int rows, int C, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || rank < 1 || rank > 8192 || C < 1 || kind < 0 || kind > 2 || (kind == 0 && !(tau > 0.f)) ||
      (kind == 1 && (!rate || group < 1)))
    return tis_fail("lowrank_act: bad arguments rows=%d rank=%d channels=%d kind=%d", rows, rank, C, kind);
  if (rank > 1024) return tis_fail("lowrank_act: rank %d (at most 1024)", rank);
  launch_lowrank(low, ldl, rank, w2, bias, kind, tau, rate, group, out, rows, C, stream);
  return tis_launch_status("lowrank_act");
}

// Two such products of the same rows, at most 2^31 workgroups together, in one launch where both take the same form (a mixer's decays and gates: a launch less, and
// one tail; 5 rows of 64 against 512 and 1,024, us: 8.2 / 4.2; 1,531 rows against 1,024 and 2,048 27.2 / 22.0), else in two.
TIS_EXPORT int tis_lowrank_act_pair(const float* low0, long ldl0, int rank0, const float* w0, const float* bias0, int kind0, float tau0, const float* rate0, int group0,
                                    float* out0, int C0, const float* low1, long ldl1, int rank1, const float* w1, const float* bias1, int kind1, float tau1,
                                    const float* rate1, int group1, float* out1, int C1, int rows, hipStream_t stream) {
  if (rows == 0) return 0;
  const LowRank p[2] = {{low0, ldl0, rank0, w0, bias0, kind0, tau0, rate0, group0, out0, C0, (C0 + LR_COLS - 1) / LR_COLS},
                        {low1, ldl1, rank1, w1, bias1, kind1, tau1, rate1, group1, out1, C1, (C1 + LR_COLS - 1) / LR_COLS}};
  for (const LowRank& q : p)
    if (rows < 0 || q.rank < 1 || q.rank > 1024 || q.C < 1 || q.kind < 0 || q.kind > 2 || (q.kind == 0 && !(q.tau > 0.f)) || (q.kind == 1 && (!q.rate || q.group < 1)))
      return tis_fail("lowrank_act: bad arguments rows=%d rank=%d channels=%d kind=%d", rows, q.rank, q.C, q.kind);
  const LowRankForm a = lowrank_form(p[0], rows), b = lowrank_form(p[1], rows);
  if (a == b && a.blocks + b.blocks < (1L << 31)) {
    launch_lowrank(p[0], &p[1], rows, stream);
  } else {
    launch_lowrank(p[0], nullptr, rows, stream);
    launch_lowrank(p[1], nullptr, rows, stream);
  }
  return tis_launch_status("lowrank_act_pair");
}

TIS_EXPORT int tis_normed_mean(const float* y0, long ld0, const float* g0, const float* y1, long ld1, const float* g1, float eps,
                               float* out, int rows, int D, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || D < 1 || !y0 || !g0 || (y1 && !g1) || !out) return tis_fail("normed_mean: bad arguments rows=%d width=%d", rows, D);
  if (D % 4 == 0 && D <= 4096 && fours32(y0, ld0) && fours32(y1, ld1) && fours32(g0, 0) && fours32(g1, 0) && fours32(out, 0)) {
#define S32_MEAN(PER, THREADS) normed_mean_fours_kernel<PER, THREADS><<<rows, THREADS, 0, stream>>>(y0, ld0, g0, y1, ld1, g1, eps, out, D)
    if (D <= 1024) S32_MEAN(1, 256);
    else if (rows <= 64 && D <= 2048) S32_MEAN(1, 512);
    else if (rows <= 64) S32_MEAN(1, 1024);
    else if (D <= 2048) S32_MEAN(2, 256);
    else S32_MEAN(4, 256);
#undef S32_MEAN
    return tis_launch_status("normed_mean");
  }
  normed_mean_kernel<<<rows, S32_THREADS, 0, stream>>>(y0, ld0, g0, y1, ld1, g1, eps, out, D);
  return tis_launch_status("normed_mean");
}

TIS_EXPORT int tis_activate_rows(int dtype, const float* z, long ldz, int act, void* out, long ldo, int rows, int W,
                                 hipStream_t stream) {
  if (rows == 0 || W == 0) return 0;
  if (rows < 0 || W < 0 || act < 0 || act > 3) return tis_fail("activate_rows: bad size rows=%d width=%d act=%d", rows, W, act);
  const long blocks = ((long)rows * W + S32_THREADS - 1) / S32_THREADS;
  S32_DISPATCH((activate_rows_kernel<float><<<blocks, S32_THREADS, 0, stream>>>(z, ldz, act, (float*)out, ldo, rows, W)),
               (activate_rows_kernel<bf16><<<blocks, S32_THREADS, 0, stream>>>(z, ldz, act, (bf16*)out, ldo, rows, W)))
  return tis_launch_status("activate_rows");
}
