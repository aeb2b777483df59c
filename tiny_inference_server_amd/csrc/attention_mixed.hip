// Attention whose weights are sigmoids mixed across the heads, on the matrix cores (bfloat16, pages of 16 slots).
//
// For the row at position p and every key j it sees (j <= p, and with chunk c > 0 only j >= p - p % c):
//   s_g = q_g . k_kv(g) * scale;  s_g <- cap * tanh(s_g / cap) (cap 0: as it is);  w_g = sigmoid(s_g + head_bias[g]);
//   m_h = sum_g talk[h][g] * w_g;  out_h = sum_j m_h(j) * v_kv(h)(j).
// Nothing is normalised over the keys: a row's result is a plain sum over its keys and may be cut anywhere.
//
// A workgroup of four waves takes an item of up to 16 consecutive rows of one request, all heads, and every
// `n_splits`-th step of 32 keys (two pages). Wave w owns the heads [w * HPW, (w + 1) * HPW):
//   S^T[key, row] = K[key, :] . Q[row, :]     v_mfma_f32_16x16x32_bf16, A = keys straight from the page, B = the rows'
//                                              queries kept in registers; lane (c, g) = (lane % 16, lane / 16) gets the
//                                              keys g * 4 .. g * 4 + 3 of both pages for row c
//   w = sigmoid(cap(S * scale) + bias)         32-bit, masked by position; into LDS [head][lane][8]
//   m_h = sum_g talk[h][g] w_g                 every wave reads all heads' weights of its own lanes and mixes for its heads
//   O^T[channel, row] += V^T[channel, key] m_h^T[key, row]     the same instruction, A = transposed values from the page,
//                                              B = the lane's own eight mixed weights: they never leave its registers
// Scores, weights and the mixture are 32-bit; the mixture is rounded to bfloat16 only as the value product's operand.
// Slots past the item's last position and pages past its range are never weighted merely by zero: their values are set
// to zero before the product, so what a reused page holds there, finite or not, cannot reach a result.
//
// Built per (key size, value size, heads a wave): TIS_AMX = key * 100000 + value * 100 + heads_per_wave.
#include "common.h"

TIS_DEFINE_LAST_ERROR(tis_attention_mixed)

#ifndef TIS_AMX
#define TIS_AMX 12812804
#endif
static constexpr int KD = TIS_AMX / 100000;
static constexpr int VD = (TIS_AMX / 100) % 1000;
static constexpr int HPW = TIS_AMX % 100;
static_assert(KD >= 8 && KD % 8 == 0 && KD <= 512, "key size: a multiple of 8 up to 512");
static_assert(VD >= 16 && VD % 16 == 0 && VD <= 512, "value size: a multiple of 16 up to 512");
static_assert(HPW >= 1 && HPW <= 16, "heads a wave: 1 to 16");
static constexpr int DC = (KD + 31) / 32;      // steps of 32 key channels
static constexpr int DB = VD / 16;             // blocks of 16 value channels
static constexpr int PAGE = 16;

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ bf16x8 amx_load8(const bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }
__device__ __forceinline__ bf16x4 amx_load4(const bf16* p) { return *reinterpret_cast<const bf16x4*>(p); }

__device__ __forceinline__ float amx_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
// 1 / x for x >= 1 and infinity: the instruction's quotient is off by up to a unit in the last place; one Newton step rounds it as a
// division does (but for the rare quotient next to the middle of two numbers) in two multiply-adds instead of a division's ten instructions. The step would
// make NaN of infinity, which keeps its 0; NaN stays NaN.
__device__ __forceinline__ float amx_inverse(float x) {
  const float r = __builtin_amdgcn_rcpf(x), better = fmaf(fmaf(-x, r, 1.f), r, r);
  return x == INFINITY ? 0.f : better;
}
// the same where x is known to be finite
__device__ __forceinline__ float amx_inverse_finite(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.f), r, r);
}

// items: (first row, rows) pairs, or null: item i is row i alone. LDS (floats): talk [4 HPW][4 HPW], heads that are mixed from outside,
// wave's heads inside | weights [H][64][8].
//
// What bounds it: a wave's instructions (a step of 32 keys: 64 products, two exponentials and two reciprocals for each of 8 weights
// of 4 heads, 512 multiply-adds of the mixture), as 16 heads' results and queries leave one wave a SIMD; so nothing may wait
// for memory either: the next step's pages are looked up a step ahead, its first head's keys are fetched as soon as this
// step's scores are made and the values before this step's weights meet, once for the heads that share them. us, 16
// heads of 128 in chunks of 1,024, with the sum of the cuts: 1,531 rows 203 before that (and with divisions), 98 now (92 with bare reciprocals).
__global__ __launch_bounds__(256) void attention_mixed_mfma_kernel(
    const bf16* __restrict__ q, long ldq, const bf16* __restrict__ plane, const int* __restrict__ block_tables, int bt_ld,
    const int* __restrict__ row_seq, const int* __restrict__ positions, const int* __restrict__ items,
    bf16* __restrict__ out, long ldo, float* __restrict__ partial, int n_splits, int H, int G, int chunk, float scale,
    float softcap, const float* __restrict__ head_bias, const float* __restrict__ talk) {
  constexpr int HM = 4 * HPW;                    // heads there is room for
  extern __shared__ __attribute__((aligned(16))) float amx_lds[];
  float* tk = amx_lds;                           // [from head][to head]
  float* wl = amx_lds + HM * HM;
  const int item = blockIdx.x, split = blockIdx.y;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TIS_WAVE), lane = threadIdx.x % TIS_WAVE;
  const int c16 = lane % 16, g4 = lane / 16;
  const int first = items ? items[2 * item] : item;
  const int n_rows = items ? items[2 * item + 1] : 1;
  const int pos0 = positions[first];
  const int p_hi = pos0 + n_rows - 1;
  const int* bt = block_tables + (long)row_seq[first] * bt_ld;
  const int k_first = chunk > 0 ? pos0 - pos0 % chunk : 0;
  const int group_size = H / G;
  for (int i = threadIdx.x; i < HM * HM; i += 256) {
    const int from = i / HM, to = i % HM;
    tk[i] = from < H && to < H ? talk[to * H + from] : 0.f;
  }
  // the lane's row: its position, its first visible key, whether it is a row at all
  const bool row_ok = c16 < n_rows;
  const int p_row = row_ok ? pos0 + c16 : -1;    // (no row: no key lies before it)
  const int lo_row = chunk > 0 && row_ok ? p_row - p_row % chunk : 0;
  const bf16* q_row = q + (long)(first + (row_ok ? c16 : 0)) * ldq;
  // this wave's heads: queries as B operands, biases
  constexpr float LOG2E = 1.4426950408889634f;
  bf16x8 qb[HPW][DC];
  float hb[HPW];
#pragma unroll
  for (int u = 0; u < HPW; ++u) {
    const int h = wave * HPW + u;
    hb[u] = h < H ? -LOG2E * head_bias[h] : 0.f;
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) {
      const int d = dc * 32 + g4 * 8;
      const bool ok = h < H && d < KD;
      const bf16x8 v = amx_load8(q_row + (long)(ok ? h : 0) * KD + (ok ? d : 0));
      qb[u][dc] = ok ? v : (bf16x8){0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  f32x4 o[HPW][DB];
#pragma unroll
  for (int u = 0; u < HPW; ++u)
#pragma unroll
    for (int db = 0; db < DB; ++db) o[u][db] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const long page_stride = (long)G * PAGE * (KD + VD);
  const long v_base = (long)G * PAGE * KD;
  // tanh(y) = 1 - 2 / (1 + exp(2 y)), |y| capped so that exp stays finite; sigmoid(x) = 1 / (1 + exp(-x)); both on base 2
  const float to_cap = softcap > 0.f ? 2.f * LOG2E * scale / softcap : 0.f, from_cap = -LOG2E * softcap, plain = -LOG2E * scale;
  const int s_first = k_first / 32, s_last = p_hi / 32;
  // a step's two pages; one past the item's last position is not looked up
  auto page_of = [&](int s, int t) { return bt[min(s * 32 + t * 16, p_hi) / PAGE]; };
  auto load_keys = [&](bf16x8 (&ka)[2][DC], const int (&page)[2], int kv_head) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const bf16* kp = plane + (long)page[t] * page_stride + (long)kv_head * PAGE * KD + (long)c16 * KD;
#pragma unroll
      for (int dc = 0; dc < DC; ++dc) {
        const int d = dc * 32 + g4 * 8;
        const bool ok = d < KD;
        const bf16x8 kv = amx_load8(kp + (ok ? d : 0));
        ka[t][dc] = ok ? kv : (bf16x8){0, 0, 0, 0, 0, 0, 0, 0};
      }
    }
  };
  bf16x4 va[DB][2];
  auto load_values = [&](const int (&page)[2], int kv_head) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const bf16* vp = plane + (long)page[t] * page_stride + v_base + (long)kv_head * VD * PAGE + (long)c16 * PAGE + g4 * 4;
#pragma unroll
      for (int db = 0; db < DB; ++db) va[db][t] = amx_load4(vp + (long)db * 16 * PAGE);
    }
  };
  const int kv_first = min(wave * HPW, H - 1) / group_size;      // the key/value head of the wave's first head
  int page[2], page_next[2];
  bf16x8 ka[2][DC];
  int s = s_first + split;
  if (s <= s_last) {
    page[0] = page_of(s, 0);
    page[1] = page_of(s, 1);
    load_keys(ka, page, kv_first);
  }
  for (; s <= s_last; s += n_splits) {
    const bool more = s + n_splits <= s_last;
    if (more) {
      page_next[0] = page_of(s + n_splits, 0);
      page_next[1] = page_of(s + n_splits, 1);
    }
    bool seen[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int j = s * 32 + (e / 4) * 16 + g4 * 4 + e % 4;
      seen[e] = j <= p_row && j >= lo_row;
    }
    // scores and weights of this wave's heads; the keys of a key/value head are fetched once for the heads that share it
    int kv_have = kv_first;
#pragma unroll
    for (int u = 0; u < HPW; ++u) {
      const int h = wave * HPW + u;
      if (h < H) {
        if (h / group_size != kv_have) {
          kv_have = h / group_size;
          load_keys(ka, page, kv_have);
        }
        float* dst = wl + ((long)h * TIS_WAVE + lane) * 8;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          f32x4 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int dc = 0; dc < DC; ++dc) st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[t][dc], qb[u][dc], st, 0, 0, 0);
          f32x4 w;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float x;               // minus the capped score with its bias, times log2 e
            if (softcap > 0.f) {
              const float e2 = amx_exp2(fminf(fmaxf(st[i] * to_cap, -30.f * LOG2E), 30.f * LOG2E));
              x = fmaf(from_cap, fmaf(-2.f, amx_inverse_finite(1.f + e2), 1.f), hb[u]);
            } else {
              x = fmaf(st[i], plain, hb[u]);
            }
            w[i] = seen[t * 4 + i] ? amx_inverse(1.f + amx_exp2(x)) : 0.f;
          }
          *reinterpret_cast<f32x4*>(dst + t * 4) = w;
        }
      }
    }
    if (more) load_keys(ka, page_next, kv_first);
    load_values(page, kv_first);
    // (not __syncthreads, which also waits for what is under way from memory)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
    // the mixture for this wave's heads, from all heads' weights of the lane's own keys and row
    float m[HPW][8];
#pragma unroll
    for (int u = 0; u < HPW; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) m[u][e] = 0.f;
#pragma unroll 4
    for (int gg = 0; gg < H; ++gg) {
      const float* src = wl + ((long)gg * TIS_WAVE + lane) * 8;
      const f32x4 a = *reinterpret_cast<const f32x4*>(src), b = *reinterpret_cast<const f32x4*>(src + 4);
      float tt[HPW];
#pragma unroll
      for (int u = 0; u < HPW; ++u) tt[u] = tk[gg * HM + wave * HPW + u];
#pragma unroll
      for (int u = 0; u < HPW; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          m[u][e] = fmaf(tt[u], a[e], m[u][e]);
          m[u][4 + e] = fmaf(tt[u], b[e], m[u][4 + e]);
        }
    }
    // O^T += V^T . m^T
    int v_have = -1;
#pragma unroll
    for (int u = 0; u < HPW; ++u) {
      const int h = wave * HPW + u;
      if (h < H) {
        if (h / group_size != v_have) {
          if (v_have >= 0) load_values(page, h / group_size);
          v_have = h / group_size;
          if (s * 32 + 31 > p_hi) {              // slots past the item's last position
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
              for (int e = 0; e < 8; ++e)
                if (s * 32 + (e / 4) * 16 + g4 * 4 + e % 4 > p_hi) va[db][e / 4][e % 4] = static_cast<__bf16>(0.f);
          }
        }
        bf16x8 pb;
#pragma unroll
        for (int e = 0; e < 8; ++e) pb[e] = static_cast<__bf16>(m[u][e]);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const bf16x8 v8 = __builtin_shufflevector(va[db][0], va[db][1], 0, 1, 2, 3, 4, 5, 6, 7);
          o[u][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v8, pb, o[u][db], 0, 0, 0);
        }
      }
    }
    page[0] = page_next[0];
    page[1] = page_next[1];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");      // the next step's weights overwrite this step's
  }
  // O^T[channel = db * 16 + g4 * 4 + i][row = c16]
  if (!row_ok) return;
  const long row = first + c16;
  const int n_out = H * VD;
#pragma unroll
  for (int u = 0; u < HPW; ++u) {
    const int h = wave * HPW + u;
    if (h >= H) continue;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int c = h * VD + db * 16 + g4 * 4;
      if (n_splits > 1) {
        *reinterpret_cast<f32x4*>(partial + (row * n_splits + split) * n_out + c) = o[u][db];
      } else {
        bf16x4 w;
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = static_cast<__bf16>(o[u][db][i]);
        *reinterpret_cast<bf16x4*>(out + row * ldo + c) = w;
      }
    }
  }
}

// (eight parts are asked for at a time: with a runtime count one after the other, 33 parts of 5 rows took 9.4 us, now 4.1)
__global__ __launch_bounds__(256) void attention_mixed_sum_kernel(const float* __restrict__ partial, int n_splits,
                                                                  bf16* __restrict__ out, long ldo, int rows, int n_out) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long)rows * n_out) return;
  const long r = i / n_out;
  const int c = (int)(i % n_out);
  float a = 0.f;
  const float* mine = partial + r * n_splits * n_out + c;
  int s = 0;
  for (; s + 8 <= n_splits; s += 8) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = mine[(long)(s + i) * n_out];
#pragma unroll
    for (int i = 0; i < 8; ++i) a += v[i];
  }
  for (; s < n_splits; ++s) a += mine[(long)s * n_out];
  out[r * ldo + c] = static_cast<bf16>(a);
}

TIS_EXPORT int tis_attention_mixed_sizes(int* kd, int* vd, int* hpw) {
  *kd = KD;
  *vd = VD;
  *hpw = HPW;
  return 0;
}

static size_t lds_bytes(int H) { return ((size_t)16 * HPW * HPW + (size_t)H * TIS_WAVE * 8) * sizeof(float); }

// How many workgroups of the kernel a compute unit holds at a time for H heads (1 where the runtime cannot tell).
TIS_EXPORT int tis_attention_mixed_resident(int H) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, attention_mixed_mfma_kernel, 256, lds_bytes(H)) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  return n < 1 ? 1 : n;
}

// items: n_items (first row, rows <= 16) pairs of consecutive rows of one request each, or null: every row by itself.
// partial: [rows * n_splits * H * VD] floats where n_splits > 1. q, out: bfloat16 with 16-byte aligned rows.
TIS_EXPORT int tis_attention_mixed_mfma(const void* q, long ldq, const void* plane, const int* block_tables, int bt_ld,
                                        const int* row_seq, const int* positions, const int* items, int n_items, void* out,
                                        long ldo, float* partial, int n_splits, int rows, int H, int G, int key_dim,
                                        int value_dim, int page_size, int chunk, float scale, float softcap,
                                        const float* head_bias, const float* talk, hipStream_t stream) {
  if (rows == 0 || n_items == 0) return 0;
  if (key_dim != KD || value_dim != VD || page_size != PAGE)
    return tis_fail("attention_mixed_mfma: built for keys of %d, values of %d and pages of %d, called with %d, %d, %d", KD, VD,
                    PAGE, key_dim, value_dim, page_size);
  if (rows < 0 || n_items < 0 || H < 1 || G < 1 || H % G || H > 4 * HPW || chunk < 0 || n_splits < 1 || n_splits > 65535 ||
      !head_bias || !talk || softcap < 0.f)
    return tis_fail("attention_mixed_mfma: bad size rows=%d items=%d heads=%d (at most %d) kv_heads=%d chunk=%d splits=%d", rows,
                    n_items, H, 4 * HPW, G, chunk, n_splits);
  if (ldq % 8 || ldo % 4 || ((uintptr_t)q % 16) || ((uintptr_t)out % 8))
    return tis_fail("attention_mixed_mfma: rows of q and out must be 16 and 8 bytes aligned");
  if (n_splits > 1 && (!partial || ((uintptr_t)partial % 16))) return tis_fail("attention_mixed_mfma: key splits without a workspace");
  const size_t lds = lds_bytes(H);
  if (lds > 64 * 1024) return tis_fail("attention_mixed_mfma: %d heads need %zu bytes of LDS", H, lds);
  attention_mixed_mfma_kernel<<<dim3(n_items, n_splits), 256, lds, stream>>>(
      (const bf16*)q, ldq, (const bf16*)plane, block_tables, bt_ld, row_seq, positions, items, (bf16*)out, ldo, partial, n_splits,
      H, G, chunk, scale, softcap, head_bias, talk);
  if (n_splits > 1) {
    const long blocks = ((long)rows * H * VD + 255) / 256;
    attention_mixed_sum_kernel<<<blocks, 256, 0, stream>>>(partial, n_splits, (bf16*)out, ldo, rows, H * VD);
  }
  return tis_launch_status("attention_mixed_mfma");
}
