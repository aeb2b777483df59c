// A gated delta rule: a matrix state per head that is corrected towards each new value, with a decay per key channel.
//
//   S <- diag(a_t) S;  u = beta_t (v_t - S^T k_t);  S <- S + k_t u^T;  o_t = S^T q_t
//
// per head and row, S being 32-bit floats in the request's state line, laid out [head][block of 16 value channels]
// [key channel][16] (value channels rounded up to a multiple of 16; the channels beyond stay zero), so that the part
// of a line that one workgroup of the walk owns is one run of memory. The kernels: the
// step before the walk (a short causal convolution with silu over the q, k and v columns of a 32-bit input product,
// unit q and k per head, beta); the walk, row by row; and for a request's many rows the walk in chunks of 16, with
// the step before it. Everything is 32-bit.
//
// A request's state line holds S and, from float `conv_at` on, the convolution's last taps - 1
// inputs [taps - 1][channels], oldest first. Rows of the step are grouped by request: request s owns the rows
// [cu_rows[s], cu_rows[s + 1]) in order of position and the line seq_slots[s].
#include <type_traits>

#include "common.h"

TIS_DEFINE_LAST_ERROR(tis_delta_rule)

static constexpr int DR_MAX_TAPS = 16;
static constexpr int DR_PER = 4;         // channels of a head a lane keeps in the step before the walk: dim <= 256

__device__ __forceinline__ float dr_sigmoid(float z) { return 1.f / (1.f + expf(-z)); }

// One convolved channel of row r: sum_j taps[ch][j] * input(i - (K - 1) + j), i the row's index among its request's rows
// of this step; inputs before the step's first row come from the state line, which is zero before a request's first row.
// KT: the number of taps where it is known at compile time (0: K): then all loads of a channel are under way at once, where a loop of unknown length
// waits for each input before it asks for the next. Same sums in the same order. 1,531 rows of 2 heads of 128, 8 of 256, four taps, us: 26 / 20; 5 rows 6.0 / 4.5.
// KEEP: the row is its request's only one, and the line moves on by it (entry k becomes what entry k + 1 was, the last one this row's input): a
// channel belongs to one thread, so nobody else reads what it overwrites, and a decoded step saves the kernel that would do this for requests of any number of rows
// (3 us).
template <int KT, bool KEEP>
__device__ __forceinline__ float dr_conv(const float* __restrict__ proj, long ldp, int col, const float* __restrict__ taps,
                                         int K, int ch, int C, float* line, long first_row, int i) {
  float acc = 0.f;
  if constexpr (KT > 0) {
    float x[KT], tap[KT];
#pragma unroll
    for (int j = 0; j < KT; ++j) {
      const int at = i - (KT - 1) + j;
      x[j] = *(at >= 0 ? proj + (first_row + at) * ldp + col : line + (long)(i + j) * C + ch);
      tap[j] = taps[(long)ch * KT + j];
    }
#pragma unroll
    for (int j = 0; j < KT; ++j) acc += tap[j] * x[j];
    if constexpr (KEEP)
#pragma unroll
      for (int j = 0; j + 1 < KT; ++j) line[(long)j * C + ch] = x[j + 1];
  } else {                // (a load on either side of the condition: with the address chosen first, 3 to 6 % slower at 2, 3, 5 and 8 taps)
    for (int j = 0; j < K; ++j) {
      const int at = i - (K - 1) + j;
      const float x = at >= 0 ? proj[(first_row + at) * ldp + col] : line[(long)(i + j) * C + ch];
      acc += taps[(long)ch * K + j] * x;
      if (KEEP && j > 0) line[(long)(j - 1) * C + ch] = x;
    }
  }
  return acc * dr_sigmoid(acc);
}

// grid (rows, units), one wave each. Units: the G query heads (unit vectors times dim^-1/2), the G key heads (unit
// vectors), blocks of 64 value channels, and one for the heads' beta = sigmoid(.). out: [rows][C + H], C = 2 G D + H V.
template <int KT, bool KEEP>
__global__ __launch_bounds__(TIS_WAVE) void delta_prepare_kernel(
    const float* __restrict__ proj, long ldp, int conv_off, int beta_off, const float* __restrict__ taps, int K,
    float* state, long lds, int conv_at, const int* __restrict__ row_seq, const int* __restrict__ cu_rows,
    const int* __restrict__ seq_slots, float* __restrict__ out, long ldo, int H, int G, int D, int V) {
  const long r = blockIdx.x;
  const int unit = blockIdx.y, lane = threadIdx.x;
  const int C = 2 * G * D + H * V;
  const int s = row_seq[r];
  const long first_row = cu_rows[s];
  const int i = (int)(r - first_row);
  float* line = state + (long)seq_slots[s] * lds + conv_at;
  if (unit < 2 * G) {
    float y[DR_PER];
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < DR_PER; ++u) {
      const int e = lane + u * TIS_WAVE;
      y[u] = 0.f;
      if (e < D) {
        const int ch = unit * D + e;
        y[u] = dr_conv<KT, KEEP>(proj, ldp, conv_off + ch, taps, K, ch, C, line, first_row, i);
        ss += y[u] * y[u];
      }
    }
    ss = wave_sum(ss);
    const float mul = (unit < G ? 1.f / sqrtf((float)D) : 1.f) / sqrtf(ss + 1e-6f);
#pragma unroll
    for (int u = 0; u < DR_PER; ++u) {
      const int e = lane + u * TIS_WAVE;
      if (e < D) out[r * ldo + unit * D + e] = y[u] * mul;
    }
    return;
  }
  const int v_blocks = (H * V + TIS_WAVE - 1) / TIS_WAVE;
  if (unit < 2 * G + v_blocks) {
    const int e = (unit - 2 * G) * TIS_WAVE + lane;
    if (e < H * V) {
      const int ch = 2 * G * D + e;
      out[r * ldo + ch] = dr_conv<KT, KEEP>(proj, ldp, conv_off + ch, taps, K, ch, C, line, first_row, i);
    }
    return;
  }
  for (int h = lane; h < H; h += TIS_WAVE) out[r * ldo + C + h] = dr_sigmoid(proj[r * ldp + beta_off + h]);
}

// Sum over the 16 lanes of a row of lanes (lanes 16 r .. 16 r + 15), every lane gets it: four data-parallel moves
// inside the row (two inside quads, then the half row and the row mirrored), no trip through LDS. One fixed order.
__device__ __forceinline__ float dr_row_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));    // quad_perm [2,3,0,1]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));   // row_half_mirror
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, true));   // row_mirror
  return v;
}

// The walk. grid (blocks of 16 value channels, heads, requests), 256 threads: thread (c, l) = (t / 16, t % 16) owns, for
// value channel c, the state's key channels [l * R, (l + 1) * R) in registers from the line before the first row to the
// line after the last (the line goes through LDS both ways, so that memory sees whole runs of 16 channels). With
// S' = diag(a) S, a token needs S'^T k for its write and (S' + k w^T)^T q = S'^T q + (k . q) w for its read: the three
// sums over the key channels (S'^T k, S'^T q, k . q) are R terms a lane each and then one pass over the 16 lanes of a
// column for all three together. Every state element sees its rows strictly in order and every sum has one fixed
// order: a row's result does not depend on what else is in the step. Requests of `from` rows and more are left to the chunks below.
// Rows come through LDS 16 at a time (8 where a lane holds 16 key channels): [rows][k: Dp | decay: Dp | q: Dp | v: 16 | beta | 3 unused].
template <int R>
__global__ __launch_bounds__(256) void delta_scan_kernel(
    const float* __restrict__ u, long ldu, int q_off, int k_off, int v_off, int beta_off, const float* __restrict__ decay,
    long ldd, float* __restrict__ state, long lds, const int* __restrict__ cu_rows, const int* __restrict__ seq_slots,
    float* __restrict__ out, long ldo, int H, int G, int D, int V, int from) {
  extern __shared__ __attribute__((aligned(16))) float dr_lds[];
  const int s = blockIdx.z, h = blockIdx.y, vb = blockIdx.x, t = threadIdx.x;
  const int first = cu_rows[s], n_rows = cu_rows[s + 1] - first;
  if (n_rows <= 0 || n_rows >= from) return;
  const int cl = t / 16, l = t % 16;
  const int c = vb * 16 + cl;
  const bool live = c < V;
  const int hq = h / (H / G);
  constexpr int Dp = 16 * R;                 // key channels as the lanes hold them (those from D on are zeros)
  constexpr int stride = 3 * Dp + 20;
  // this block's [D][16] part of the line: one run of memory, into LDS 16 bytes a lane, then each lane's own elements
  float* S_line = state + (long)seq_slots[s] * lds + ((long)h * gridDim.x + vb) * D * 16;
  for (int e = t; e < D * 4; e += 256)
    reinterpret_cast<float4*>(dr_lds)[e] = reinterpret_cast<const float4*>(S_line)[e];
  __syncthreads();
  float S[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int d = l * R + i;
    S[i] = d < D ? dr_lds[d * 16 + cl] : 0.f;
  }
  // Rows go through two LDS buffers: while one chunk of rows is walked, the next one's loads are in flight in registers
  // and are put into the other buffer afterwards, so one barrier a chunk and no wait for memory between chunks.
  constexpr int TOK = R <= 8 ? 16 : 8;       // rows a chunk
  constexpr int NI = TOK * Dp / 256;         // k, decay and q elements a thread fetches for a chunk
  float pk[NI], pa[NI], pq[NI], pv[2];
  auto fetch = [&](int r0) {
    const int n = min(TOK, n_rows - r0);
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int i = t + 256 * j, tt = i / Dp, d = i % Dp;
      const long row = first + r0 + tt;
      const bool ok = tt < n && d < D;
      pk[j] = ok ? u[row * ldu + k_off + hq * D + d] : 0.f;
      pa[j] = ok ? decay[row * ldd + h * D + d] : 0.f;
      pq[j] = ok ? u[row * ldu + q_off + hq * D + d] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = t + 256 * j, tt = i / 17, e = i % 17;
      const long row = first + r0 + tt;
      const int cc = vb * 16 + e;
      pv[j] = tt < n ? (e == 16 ? u[row * ldu + beta_off + h] : (cc < V ? u[row * ldu + v_off + h * V + cc] : 0.f)) : 0.f;
    }
  };
  auto commit = [&](float* buf) {
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int i = t + 256 * j, tt = i / Dp, d = i % Dp;
      float* dst = buf + tt * stride;
      dst[d] = pk[j];
      dst[Dp + d] = pa[j];
      dst[2 * Dp + d] = pq[j];
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = t + 256 * j, tt = i / 17, e = i % 17;
      if (tt < TOK) buf[tt * stride + 3 * Dp + e] = pv[j];
    }
  };
  __syncthreads();               // every lane has taken its part of the line out of LDS
  fetch(0);
  commit(dr_lds);
  __syncthreads();
  int which = 0;
  for (int r0 = 0; r0 < n_rows; r0 += TOK, which ^= 1) {
    const int n = min(TOK, n_rows - r0);
    const bool more = r0 + TOK < n_rows;
    if (more) fetch(r0 + TOK);
    const float* rows_lds = dr_lds + which * (TOK * stride);
    for (int tt = 0; tt < n; ++tt) {
      const float* src = rows_lds + tt * stride;
      float kv[R], av[R], qv[R];
      if constexpr (R % 4 == 0) {
#pragma unroll
        for (int i = 0; i < R; i += 4) {
          const float4 a = *reinterpret_cast<const float4*>(src + l * R + i);
          const float4 b = *reinterpret_cast<const float4*>(src + Dp + l * R + i);
          const float4 q4 = *reinterpret_cast<const float4*>(src + 2 * Dp + l * R + i);
          kv[i] = a.x, kv[i + 1] = a.y, kv[i + 2] = a.z, kv[i + 3] = a.w;
          av[i] = b.x, av[i + 1] = b.y, av[i + 2] = b.z, av[i + 3] = b.w;
          qv[i] = q4.x, qv[i + 1] = q4.y, qv[i + 2] = q4.z, qv[i + 3] = q4.w;
        }
      } else {
#pragma unroll
        for (int i = 0; i < R; ++i) {
          kv[i] = src[l * R + i];
          av[i] = src[Dp + l * R + i];
          qv[i] = src[2 * Dp + l * R + i];
        }
      }
      float dk = 0.f, dq = 0.f, kq = 0.f;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        S[i] *= av[i];
        dk += S[i] * kv[i];
        dq += S[i] * qv[i];
        kq += kv[i] * qv[i];
      }
      dk = dr_row_sum(dk);
      dq = dr_row_sum(dq);
      kq = dr_row_sum(kq);
      const float w = src[3 * Dp + 16] * (src[3 * Dp + cl] - dk);
#pragma unroll
      for (int i = 0; i < R; ++i) S[i] += kv[i] * w;
      if (live && l == 0) out[(long)(first + r0 + tt) * ldo + h * V + c] = dq + kq * w;
    }
    if (more) commit(dr_lds + (which ^ 1) * (TOK * stride));
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int d = l * R + i;
    if (d < D) dr_lds[d * 16 + cl] = S[i];
  }
  __syncthreads();
  // (channels beyond vdim have seen values of zero only and are still zero)
  for (int e = t; e < D * 4; e += 256)
    reinterpret_cast<float4*>(S_line)[e] = reinterpret_cast<const float4*>(dr_lds)[e];
}

// ---- a request's many rows: the walk in chunks of 16 ------------------------------------------------------------------
//
// The walk above is one serial chain: every row waits for three sums over the key channels of the state that the row before left
// (270 ns a row, on one wave a SIMD of half the chip). Sixteen rows at a time the sums of all of them against the state at the
// chunk's beginning, S0, are matrix products, and what the rows of a chunk do to one another needs no state at all. With
// A(i, j) = the decays of rows i + 1 .. j multiplied up per channel (products of numbers up to 1: nothing is ever divided by),
//   G(i, j) = sum_d k_i k_j A(i, j),  Q(j, i) = sum_d k_i q_j A(i, j)  (i <= j)
//   w_j = beta_j (v_j - S0^T (k_j A(-1, j)) - sum_{i<j} G(i, j) w_i)            that is  W = T (V - K~ S0)
//   o_j = S0^T (q_j A(-1, j)) + sum_{i<=j} Q(j, i) w_i                                   O = Q~ S0 + Q W
//   S <- A(-1, 15) S0 + sum_i (k_i A(i, 15)) w_i^T                                       S = A S0 + K^ W
// with T = (I + beta G)^-1 beta, solved column by column. delta_chunks_kernel makes K~, Q~, K^, A, T and Q of every chunk and head,
// all chunks at once; delta_chunk_walk_kernel walks them with S in registers, all products on v_mfma_f32_16x16x4_f32 (32-bit
// multiply-adds). Rows past a request's last have k = q = 0, decay 1 and beta 0 and change nothing. MI355X, 8 heads of 128 x 256,
// us row by row / in chunks with the step before them: 2,048 rows 546 / 153, 1,531 410 / 121, 512 141 / 49, 128 38 / 22. Off from 64 bits, row
// by row / in chunks, by decays from 0.5, 0.9 and 0.995 on: results 0.99e-7 / 0.98e-7, 1.39e-7 / 1.40e-7, 3.3e-7 / 3.0e-7, states 0.62e-7 / 0.62e-7,
// 1.16e-7 / 1.19e-7, 3.6e-7 / 3.2e-7. (With rows four apart in a product, the newest among the first, 1.15e-7 and 0.87e-7 at the strongest
// decays, where the newest are the largest; with one sum over a wave's channels 5 % more, and 162 us where the four take 155.)
typedef __attribute__((ext_vector_type(4))) float f32x4;
static constexpr int DC = 16;                    // rows of a chunk
static constexpr int DR_CHUNK_FROM = 48;         // rows of a request from which on its rows are walked in chunks (us, row by row / in
                                                 // chunks: 32 rows 13.3 / 14.5, 48 17.9 / 16.1, 128 39 / 24)

__host__ __device__ constexpr int dc_floats(int Dp) { return 3 * DC * Dp + Dp + 2 * DC * DC; }   // of a chunk and head: K~, Q~, K^ [d][row], A, T, Q

// Where row i of a chunk lies in the products: register r of lane (g, n) is place 4 g + r and row 4 r + g, so that a product over rows adds
// them four at a time in their order, oldest first, as the walk row by row does (its own inverse).
__host__ __device__ constexpr int dc_place(int i) { return i % 4 * 4 + i / 4; }

__device__ __forceinline__ int dc_chunks(int n) { return n >= DR_CHUNK_FROM ? (n + DC - 1) / DC : 0; }

// grid (chunks, heads), 256 threads: thread (i, l) = (t / 16, t % 16) takes row i and the key channels l, l + 16, ...
template <int Dp>
__global__ __launch_bounds__(256) void delta_chunks_kernel(const float* __restrict__ u, long ldu, int q_off, int k_off, int beta_off,
                                                           const float* __restrict__ decay, long ldd,
                                                           const int* __restrict__ cu_rows, int n_seqs, float* __restrict__ work,
                                                           int H, int G, int D) {
  __shared__ __attribute__((aligned(16))) float k[DC][Dp], q[DC][Dp], a[DC][Dp], L[DC][DC], beta[DC];
  const int h = blockIdx.y, hq = h / (H / G), t = threadIdx.x, lane = t % 64;
  // which request's, and which of its chunks: the requests' chunks numbered through (a lane a request, 64 at a time)
  int first = -1, n = 0, before = 0;
  for (int s0 = 0; s0 < n_seqs && first < 0; s0 += 64) {
    const int s = s0 + lane;
    const int rows = s < n_seqs ? cu_rows[s + 1] - cu_rows[s] : 0;
    const int own = dc_chunks(rows);
    int upto = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o, 64);
      if (lane >= o) upto += v;
    }
    const unsigned long long holds = __ballot(before + upto > (int)blockIdx.x);
    if (holds) {
      const int at = __ffsll(holds) - 1;
      const int c = (int)blockIdx.x - before - __shfl(upto - own, at, 64);
      first = cu_rows[s0 + at] + c * DC;
      n = min(DC, __shfl(rows, at, 64) - c * DC);
    } else {
      before += __shfl(upto, 63, 64);
    }
  }
  if (first < 0) return;                         // the grid is as wide as there could be chunks
  // all of the chunk's loads at once, from addresses that always hold something (a load under a condition is waited for before the next;
  // 1,531 rows of 8 heads of 128, us: 23 / 20)
  constexpr int PER = DC * Dp / 256;
  float hk[PER], hq4[PER], ha[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = t + 256 * j, r = e / Dp, d = min(e % Dp, D - 1);
    const long row = first + min(r, n - 1);
    hk[j] = u[row * ldu + k_off + hq * D + d];
    hq4[j] = u[row * ldu + q_off + hq * D + d];
    ha[j] = decay[row * ldd + h * D + d];
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int e = t + 256 * j, r = e / Dp, d = e % Dp;
    const bool ok = r < n && d < D;
    k[r][d] = ok ? hk[j] : 0.f;
    q[r][d] = ok ? hq4[j] : 0.f;
    a[r][d] = ok ? ha[j] : 1.f;
  }
  if (t < DC) beta[t] = t < n ? u[(long)(first + t) * ldu + beta_off + h] : 0.f;
  __syncthreads();
  float* mine = work + ((long)blockIdx.x * H + h) * dc_floats(Dp);
  float *Kt = mine, *Qt = mine + DC * Dp, *Kh = mine + 2 * DC * Dp, *A = mine + 3 * DC * Dp, *T = A + Dp, *Q = T + DC * DC;
  const int i = t / 16, l = t % 16;
  float g[DC], p[DC];                            // (of rows that do not follow i: numbers that nobody reads)
#pragma unroll
  for (int j = 0; j < DC; ++j) g[j] = p[j] = 0.f;
#pragma unroll 1
  for (int d = l * 4; d < Dp; d += 64) {
    const f32x4 ki = *reinterpret_cast<const f32x4*>(&k[i][d]), qi = *reinterpret_cast<const f32x4*>(&q[i][d]);
    f32x4 upto = {1.f, 1.f, 1.f, 1.f}, ka = ki;  // the decays of rows 0 .. i; k_i times those of rows i + 1 .. j
#pragma unroll
    for (int j = 0; j < DC; ++j) {
      const f32x4 aj = *reinterpret_cast<const f32x4*>(&a[j][d]), kj = *reinterpret_cast<const f32x4*>(&k[j][d]);
      const f32x4 qj = *reinterpret_cast<const f32x4*>(&q[j][d]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        upto[e] *= j <= i ? aj[e] : 1.f;
        ka[e] *= j > i ? aj[e] : 1.f;
        g[j] = fmaf(ka[e], kj[e], g[j]);
        p[j] = fmaf(ka[e], qj[e], p[j]);
      }
    }
    *reinterpret_cast<f32x4*>(Kt + dc_place(i) * Dp + d) = ki * upto;
    *reinterpret_cast<f32x4*>(Qt + dc_place(i) * Dp + d) = qi * upto;
#pragma unroll
    for (int e = 0; e < 4; ++e) Kh[(d + e) * DC + dc_place(i)] = ka[e];
    if (i == DC - 1) *reinterpret_cast<f32x4*>(A + d) = upto;
  }
#pragma unroll
  for (int j = 0; j < DC; ++j) {
    const float gs = dr_row_sum(g[j]), ps = dr_row_sum(p[j]);
    if (l == j) {
      L[j][i] = gs;
      Q[dc_place(j) * DC + dc_place(i)] = i <= j ? ps : 0.f;
    }
  }
  __syncthreads();
  if (t < DC) {                                  // column t of T: x_j = beta_j ((j == t) - sum of G(m, j) x_m over t <= m < j)
    float x[DC];
#pragma unroll
    for (int j = 0; j < DC; ++j) {
      float v = j == t ? 1.f : 0.f;
#pragma unroll
      for (int m = 0; m < j; ++m) v = m >= t ? fmaf(-L[j][m], x[m], v) : v;
      x[j] = j >= t ? beta[j] * v : 0.f;
      T[dc_place(j) * DC + dc_place(t)] = x[j];
    }
  }
}

// grid (heads, blocks of 16 value channels, requests), five waves. Wave w < 4 keeps key channels [16 NT w, 16 NT (w + 1)) of S as NT
// result tiles of 16 channels x 16 value channels: lane (g, n) = (lane / 16, lane % 16) holds channels 16 t + 4 g + r of value
// channel n in register r of tile t. As the second operand of a product over channels, register r of tile t is what the four channels
// 16 t + 4 g + r (g = 0 .. 3) make up, so S goes into the products as it lies; the same holds for V - K~ S0 and W, whose rows are
// 4 r + g (see dc_place). The waves' parts of K~ S0 meet in LDS, one barrier a chunk; each then makes W for itself. Q~ S0 is worked out while the parts
// are on their way, and the fifth wave, which makes W too, adds up the rows' results a chunk later. Three chunks' operands are
// under way (one ahead, a chunk took what memory takes), or one where a head's channels leave no more registers. Workgroups of one head follow one another by `heads`, so that with 8 heads
// (or 16, ...) an XCD's L2 serves a head to all of its value channels. What bounds it is a chunk's chain (1.05 us): the products with S, LDS, W, and
// the products that change S. The loop over the chunks is one straight stretch, whose waits let the later chunks' loads be under way; with loads
// under conditions and the way out for rows that are not finite inside it, every fourth chunk waited for all of them, and a chunk took 1.38 us
// (1,531 rows of 8 heads of 128 x 256, with the step before them, 151 / 121 us; of 256 x 128 264 / 208).
template <int NT>
__global__ __launch_bounds__(320) void delta_chunk_walk_kernel(const float* __restrict__ u, long ldu, int v_off,
                                                               const float* __restrict__ work, float* __restrict__ state, long lds,
                                                               const int* __restrict__ cu_rows, const int* __restrict__ seq_slots,
                                                               float* __restrict__ out, long ldo, int H, int D, int V) {
  constexpr int SETS = NT <= 2 ? 4 : 2;          // chunks whose operands are held or under way
  constexpr int Dp = 64 * NT, OFF_A = 3 * DC * Dp, OFF_T = OFF_A + Dp, OFF_Q = OFF_T + DC * DC;
  __shared__ f32x4 ks_parts[2][4][64], qs_parts[2][4][64];       // turn, wave, lane
  __shared__ int poisoned[5];
  const int h = blockIdx.x, vb = blockIdx.y, s = blockIdx.z, t = threadIdx.x;
  const int first = cu_rows[s], n_rows = cu_rows[s + 1] - first;
  if (n_rows < DR_CHUNK_FROM) return;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, g = lane >> 4, n = lane & 15;
  int chunk0 = 0;                                // the chunks of the requests before
  for (int s0 = 0; s0 < s; s0 += 64) {
    int c = s0 + lane < s ? dc_chunks(cu_rows[s0 + lane + 1] - cu_rows[s0 + lane]) : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) c += __shfl_xor(c, o, 64);
    chunk0 += __builtin_amdgcn_readfirstlane(c);
  }
  const int c_v = vb * 16 + n;
  const bool live = c_v < V;
  const int chunks = (n_rows + DC - 1) / DC;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

  // Everything of a chunk lies at a scalar address (the same on all lanes) plus each lane's own offset in bytes, which never changes; `ahead` is the
  // chunk that is asked for next, at the last one it stays (its numbers are then asked for again and not used: loads without conditions).
  const long stride = (long)H * dc_floats(Dp) * 4, v_stride = (long)DC * ldu * 4;
  const unsigned char* const base = reinterpret_cast<const unsigned char*>(work + ((long)chunk0 * H + h) * dc_floats(Dp));
  const unsigned char* const v_base = reinterpret_cast<const unsigned char*>(u + (long)first * ldu + v_off + h * V);
  const unsigned v_row = (unsigned)ldu * 4, v_col = (unsigned)min(c_v, V - 1) * 4;
  const unsigned t_off = (n * DC + g * 4) * 4;
  auto four = [](const unsigned char* at, unsigned lane_off) { return *reinterpret_cast<const f32x4*>(at + lane_off); };
  int ahead;
  const unsigned char *p, *pv;
  auto rewind = [&] { ahead = 0, p = base, pv = v_base; };
  // (rows past the last: the last one's values, which T's zeros keep out)
  auto fetch_v = [&] {
    const int last = n_rows - 1 - ahead * DC;      // of the chunk's rows
    f32x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = *reinterpret_cast<const float*>(pv + ((unsigned)min(r * 4 + g, last) * v_row + v_col));
    return v;
  };
  auto advance = [&] {
    const bool more = ahead + 1 < chunks;
    ahead += more ? 1 : 0;
    p += more ? stride : 0;
    pv += more ? v_stride : 0;
  };

  // T and Q are triangular, but a product takes their zeros times every row: a row that is not finite must not reach the rows before it.
  // A walk that meets one therefore notes it (`poison` is no number from then on) and is done again, `careful`, where such chunks go without the
  // matrix product. (With that way out inside the one loop the compiler waits for all loads under way at its beginning, and the loop is four
  // times as long.)
  float poison = 0.f;
  auto triangle = [&](auto careful, f32x4 m, f32x4 x, f32x4 sum) {   // sum + M x, M [16][16], m: the lane's four, row n, columns 4 g .. 4 g + 3
    const float none = fmaf(x[3], 0.f, fmaf(x[2], 0.f, fmaf(x[1], 0.f, x[0] * 0.f)));
    if constexpr (!careful) poison += none;
    if (!careful || __all(none == 0.f)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(m[r], x[r], sum, 0, 0, 0);
      return sum;
    }
#pragma unroll 1
    for (int i = 0; i < DC; ++i) {                 // (dc_place(i) is 4 (i % 4) + i / 4)
      const int e = i / 4, from = i % 4 * 16;
      const float xe = e == 0 ? x[0] : e == 1 ? x[1] : e == 2 ? x[2] : x[3], me = e == 0 ? m[0] : e == 1 ? m[1] : e == 2 ? m[2] : m[3];
      const float xi = __shfl(xe, from + n, 64);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float mi = __shfl(me, from + g * 4 + r, 64);
        if (i <= r * 4 + g) sum[r] += mi * xi;
      }
    }
    return sum;
  };
  // W of chunk c from the four parts of K~ S0 in LDS
  auto make_w = [&](auto careful, int c, f32x4 m, f32x4 v) {
    const f32x4 k0 = ks_parts[c & 1][0][lane], k1 = ks_parts[c & 1][1][lane], k2 = ks_parts[c & 1][2][lane], k3 = ks_parts[c & 1][3][lane];
    f32x4 x = v - ((k0 + k1) + (k2 + k3));
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = live ? x[r] : 0.f;
    return triangle(careful, m, x, zero);
  };
  // (not __syncthreads, which also waits for what is under way from memory)
  auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); };
  // turns(c, set) for every chunk, with the SETS - 1 after it on their way
  auto walk = [&](auto& sets, auto&& fetch, auto&& turn) {
    rewind();
#pragma unroll
    for (int e = 0; e < SETS - 1; ++e) fetch(sets[e]), advance();
    int c0 = 0;
    for (; c0 + SETS <= chunks; c0 += SETS) {
#pragma unroll
      for (int e = 0; e < SETS; ++e) {
        fetch(sets[(e + SETS - 1) % SETS]), advance();
        __builtin_amdgcn_sched_barrier(0);
        turn(c0 + e, sets[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < SETS - 1; ++e)
      if (c0 + e < chunks) turn(c0 + e, sets[e]);
  };

  const int d0 = wave * NT * 16;                 // the wave's first key channel
  float* S_line = state + (long)seq_slots[s] * lds + ((long)h * gridDim.y + vb) * D * 16;
  f32x4 S[NT];

  auto results_wave = [&](auto careful) {        // the rows' results
    struct Operands { f32x4 t, q, v; } sets[SETS];
    f32x4 W = zero, q = zero;                    // of the chunk before
    auto results = [&](int c) {
      const f32x4 a = qs_parts[c & 1][0][lane], b = qs_parts[c & 1][1][lane], d = qs_parts[c & 1][2][lane], e = qs_parts[c & 1][3][lane];
      const f32x4 o = triangle(careful, q, W, (a + b) + (d + e));
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = c * DC + r * 4 + g;
        if (row < n_rows && live) out[(long)(first + row) * ldo + h * V + c_v] = o[r];
      }
    };
    walk(sets, [&](Operands& o) { o.t = four(p + OFF_T * 4, t_off), o.q = four(p + OFF_Q * 4, t_off), o.v = fetch_v(); },
         [&](int c, const Operands& own) {
           meet();
           const f32x4 now = make_w(careful, c, own.t, own.v);
           if (c) results(c - 1);
           W = now;
           q = own.q;
         });
    meet();
    results(chunks - 1);
  };
  auto state_waves = [&](auto careful) {
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = d0 + k * 16 + g * 4 + r;
        S[k][r] = d < D ? S_line[d * 16 + n] : 0.f;
      }
    struct Operands { f32x4 kt[NT], qt[NT], kh[NT], a[NT], t, v; } sets[SETS];
    const unsigned row_off = (n * Dp + d0 + g * 4) * 4, kh_off = ((d0 + n) * DC + g * 4) * 4, a_off = (d0 + g * 4) * 4;
    // the wave's part of a product with S, in four sums, so that none is a longer chain than the walk row by row has
    auto against = [&](const f32x4 (&rows)[NT]) {
      f32x4 part[4];
#pragma unroll
      for (int k = 0; k < NT; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(rows[k][r], S[k][r], k ? part[r] : zero, 0, 0, 0);
      return (part[0] + part[1]) + (part[2] + part[3]);
    };
    walk(sets,
         [&](Operands& o) {
#pragma unroll
           for (int k = 0; k < NT; ++k) {
             o.kt[k] = four(p + k * 64, row_off);
             o.qt[k] = four(p + DC * Dp * 4 + k * 64, row_off);
             o.kh[k] = four(p + 2 * DC * Dp * 4 + k * 16 * DC * 4, kh_off);
             o.a[k] = four(p + OFF_A * 4 + k * 64, a_off);
           }
           o.t = four(p + OFF_T * 4, t_off);
           o.v = fetch_v();
         },
         [&](int c, const Operands& now) {
           ks_parts[c & 1][wave][lane] = against(now.kt);
           meet();
           const f32x4 k0 = ks_parts[c & 1][0][lane], k1 = ks_parts[c & 1][1][lane], k2 = ks_parts[c & 1][2][lane], k3 = ks_parts[c & 1][3][lane];
           __builtin_amdgcn_sched_barrier(0);
           const f32x4 qs = against(now.qt);
           __builtin_amdgcn_sched_barrier(0);
           f32x4 x = now.v - ((k0 + k1) + (k2 + k3));
#pragma unroll
           for (int r = 0; r < 4; ++r) x[r] = live ? x[r] : 0.f;
           const f32x4 W = triangle(careful, now.t, x, zero);
           qs_parts[c & 1][wave][lane] = qs;
#pragma unroll
           for (int k = 0; k < NT; ++k) S[k] *= now.a[k];
#pragma unroll
           for (int r = 0; r < 4; ++r)
#pragma unroll
             for (int k = 0; k < NT; ++k) S[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.kh[k][r], W[r], S[k], 0, 0, 0);
         });
    meet();                                      // the fifth wave's last results
  };

  if (wave == 4) results_wave(std::false_type{});
  else state_waves(std::false_type{});
  poisoned[t >> 6] = __any(!(poison == 0.f)) ? 1 : 0;
  meet();
  if (poisoned[0] | poisoned[1] | poisoned[2] | poisoned[3] | poisoned[4]) {      // the same for all waves
    if (wave == 4) results_wave(std::true_type{});
    else state_waves(std::true_type{});
  }
  if (wave == 4) return;
  // (channels beyond vdim have seen values of zero only and are still zero)
#pragma unroll
  for (int k = 0; k < NT; ++k)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = d0 + k * 16 + g * 4 + r;
      if (d < D) S_line[d * 16 + n] = S[k][r];
    }
}

// keep: every request of the step has one row, and its line's convolution inputs move on by it; 0: the lines stay as they are.
TIS_EXPORT int tis_delta_prepare_keep(const float* proj, long ldp, int conv_off, int beta_off, const float* taps, int K,
                                 float* state, long lds, int conv_at, const int* row_seq, const int* cu_rows,
                                 const int* seq_slots, float* out, long ldo, int rows, int H, int G, int D, int V, int keep,
                                 hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || H < 1 || G < 1 || H % G || D < 1 || D > DR_PER * TIS_WAVE || V < 1 || K < 1 || K > DR_MAX_TAPS)
    return tis_fail("delta_prepare: bad size rows=%d heads=%d qk_heads=%d dim=%d (at most %d) vdim=%d taps=%d (at most %d)",
                    rows, H, G, D, DR_PER * TIS_WAVE, V, K, DR_MAX_TAPS);
  const int units = 2 * G + (H * V + TIS_WAVE - 1) / TIS_WAVE + 1;
  if (units > 65535) return tis_fail("delta_prepare: %d units a row are too many", units);
  const auto kernel = keep ? (K == 4 ? delta_prepare_kernel<4, true> : delta_prepare_kernel<0, true>)
                           : (K == 4 ? delta_prepare_kernel<4, false> : delta_prepare_kernel<0, false>);
  kernel<<<dim3(rows, units), TIS_WAVE, 0, stream>>>(proj, ldp, conv_off, beta_off, taps, K, state, lds, conv_at, row_seq, cu_rows, seq_slots,
                                                     out, ldo, H, G, D, V);
  return tis_launch_status("delta_prepare");
}

// The most chunks that `rows` rows can have, over all requests of DR_CHUNK_FROM rows and more (each begins one that it may not fill).
static long dc_most(long rows) { return rows / DC + rows / DR_CHUNK_FROM + 1; }

// Floats of work space that tis_delta_scan wants for the walk in chunks; 0: no request (the longest has `longest` rows) is long enough for it.
TIS_EXPORT long tis_delta_scan_work(int rows, int longest, int H, int D) {
  return longest < DR_CHUNK_FROM ? 0 : dc_most(rows) * H * dc_floats((D + 63) / 64 * 64);
}

// longest: the rows of the longest request, as the host knows it. work: null, or tis_delta_scan_work floats, 16-byte aligned: requests of
// DR_CHUNK_FROM rows and more are then walked in chunks. A step without such a request (decoded tokens, however many) launches the
// walk row by row alone: the kernels of the chunks would find nothing to do in thousands of workgroups (64 single rows of 128 x 256,
// us with / without them: 8 heads 59 / 53, 16 heads 108 / 99; two requests of 47 rows 20 / 17).
TIS_EXPORT int tis_delta_scan(const float* u, long ldu, int q_off, int k_off, int v_off, int beta_off, const float* decay,
                              long ldd, float* state, long lds, const int* cu_rows, const int* seq_slots, int n_seqs, int rows,
                              int longest, float* work, float* out, long ldo, int H, int G, int D, int V, hipStream_t stream) {
  if (n_seqs == 0) return 0;
  if (n_seqs < 0 || n_seqs > 65535 || rows < 0 || H < 1 || H > 65535 || G < 1 || H % G || D < 1 || D > 256 || V < 1 || lds % 4 ||
      ((uintptr_t)state % 16) || ((uintptr_t)work % 16))
    return tis_fail("delta_scan: bad size requests=%d heads=%d qk_heads=%d dim=%d (at most 256) vdim=%d, or state lines that are "
                    "not 16 bytes aligned", n_seqs, H, G, D, V);
  // (ldu: a chunk's rows are read at 32-bit offsets from its first)
  const bool chunks = work && longest >= DR_CHUNK_FROM && (V + 15) / 16 <= 65535 && dc_most(rows) < (1L << 31) && ldu < (1L << 26);
  const int from = chunks ? DR_CHUNK_FROM : 0x7fffffff;
  if (!(chunks && n_seqs == 1 && longest == rows)) {      // (a single request of that many rows leaves none for the walk row by row)
    const int R = D <= 16 ? 1 : D <= 32 ? 2 : D <= 64 ? 4 : D <= 128 ? 8 : 16;
    const int tokens = R <= 8 ? 16 : 8;
    size_t lds_bytes = 2 * (size_t)tokens * (3 * 16 * R + 20) * sizeof(float);      // two buffers of rows
    if (lds_bytes < (size_t)D * 16 * sizeof(float)) lds_bytes = (size_t)D * 16 * sizeof(float);      // the line's way in and out
    dim3 grid((V + 15) / 16, H, n_seqs);
#define DR_SCAN(RR)                                                                                                        \
  delta_scan_kernel<RR><<<grid, 256, lds_bytes, stream>>>(u, ldu, q_off, k_off, v_off, beta_off, decay, ldd, state, lds,   \
                                                          cu_rows, seq_slots, out, ldo, H, G, D, V, from)
    switch (R) {
      case 1: DR_SCAN(1); break;
      case 2: DR_SCAN(2); break;
      case 4: DR_SCAN(4); break;
      case 8: DR_SCAN(8); break;
      default: DR_SCAN(16); break;
    }
#undef DR_SCAN
  }
  if (chunks) {
    const dim3 each((unsigned)dc_most(rows), H), walk(H, (V + 15) / 16, n_seqs);
#define DR_CHUNKS(NT)                                                                                                        \
  {                                                                                                                         \
    delta_chunks_kernel<64 * NT><<<each, 256, 0, stream>>>(u, ldu, q_off, k_off, beta_off, decay, ldd, cu_rows, n_seqs, work, H, G, D);  \
    delta_chunk_walk_kernel<NT><<<walk, 320, 0, stream>>>(u, ldu, v_off, work, state, lds, cu_rows, seq_slots, out, ldo, H, D, V);      \
  }
    switch ((D + 63) / 64) {
      case 1: DR_CHUNKS(1); break;
      case 2: DR_CHUNKS(2); break;
      case 3: DR_CHUNKS(3); break;
      default: DR_CHUNKS(4); break;
    }
#undef DR_CHUNKS
  }
  return tis_launch_status("delta_scan");
}
