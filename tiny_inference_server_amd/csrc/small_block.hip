// A pre-norm block of a small 32-bit model (norm, queries, keys and values with their rotation and cache write, attention, output
// projection, norm, gated feed-forward) in one kernel, for steps in which every request brings one row.
//
// One workgroup takes one row through the whole block: a row's block reads no other row of such a step, so nothing crosses workgroups
// and the block needs no second launch. What it replaces are six dependent launches that do next to nothing.
//
// What bounds it is a compute unit's way from memory: 176 KB of matrices at some 30 bytes a nanosecond (the L2s begin a kernel empty).
// So all of it is asked for when the kernel begins, in the order in which it is needed, into registers that the products take it from (sixteen
// lanes share a row of a matrix: its pieces of 16 bytes lie side by side, the lanes' sums are added by lane moves; a thread holds SB_QKV + SB_O + SB_GU +
// SB_DOWN pieces, which sets the sizes that the kernel takes); the row's keys and values go to LDS beside them. A head's attention is one wave's and every
// wave norms the row for itself, so that four barriers are left.
// us a block in a graph, separate kernels / this one, 64 wide, 8 heads of 8 over 2, 176 hidden: rows that see 40 keys, 3 of them 21.5 / 10.0, 64 24.6 / 10.5, 512
// 36.1 / 20.9; 250 keys, 3 rows 22.6 / 15.6, 512 43.0 / 32.2; 512 keys, 1 row 24.7 / 21.6, 256 39.9 / 23.7, 300 46.5 / 44.1, 512 57.6 / 45.8. (Matrices through LDS and sums in one chain
// over K, the bits of the separate kernels: 22.7 for 3 rows of 40.)
// Which steps it takes. A head's attention is one wave's, 64 / HD keys at a time, and beyond 256 rows a compute unit has two workgroups one after the other; the separate kernels
// walk keys on many waves. So up to 256 rows, 128 keys for each of a wave's groups (separate / this one, 1 row: heads of 32, 256 keys 29.0 / 25.7, 384 33.4 / 33.8, 512 37.0 / 41.9; of 24, 256 26.8 / 24.2,
// 384 30.1 / 31.8; of 40, 128 25.5 / 22.9, 192 27.4 / 30.0; of 16, 512 28.4 / 27.3); beyond, 8 for each group and head, as many heads are what the separate kernels
// take long for (260 rows: 4 heads of 8 over 4, 256 keys 1.00 of their time, 384 1.11; 5 of 12, 192 keys 0.94, 256 1.08; 2 of 16, 128 keys 0.92, 256 1.10; 2 of 32, 64 keys 0.89, 128 1.02; 8 of 8 over 2, 512 keys
// 0.97, over 4 1.02; 16 of 4, 512 keys 0.95). The keys are the most that a row may see: in a captured step, and in the launch before it, what its block tables hold (64 pages at least) or the rotary table, whichever is
// shorter, not what the requests are long. So a model of more positions than SB_KEYS, or one without a rotary table, has its decoded steps run by the separate kernels.
//
// Sums are 32-bit: a product's sixteen partial sums of up to 12 terms added up in pairs, where the separate kernels have one chain.
#include <mutex>

#include "common.h"

TIS_DEFINE_LAST_ERROR(tis_small_block)

static constexpr int SB_THREADS = 1024, SB_WAVES = SB_THREADS / TIS_WAVE, SB_LANES = 16, SB_ROWS = SB_THREADS / SB_LANES;    // lanes a matrix row, rows a turn
static constexpr int SB_QKV = 2, SB_O = 1, SB_GU = 6, SB_DOWN = 3, SB_KV = 2;        // pieces of each matrix that a thread holds, and of the cache
static constexpr int SB_WIDTH = SB_LANES * 4;                                       // most of D and of all heads' channels together
static constexpr int SB_HIDDEN = SB_DOWN * SB_LANES * 4;                            // most of F
static constexpr int SB_KEYS = 512, SB_ROWS_MOST = 512, SB_ROWS_ROUND = 256;          // (a workgroup a compute unit)
static constexpr long SB_LDS = 160 * 1024;
static_assert(SB_WIDTH == TIS_WAVE && SB_WIDTH == SB_ROWS && 2 * SB_HIDDEN == SB_GU * SB_ROWS, "a row of the stream is a wave's, an output a turn's");

struct SmallBlock {
  const float* x; long x_ld;                     // [rows, D]
  float* out; long out_ld;
  const float *gain_a, *gain_f; float eps_a, eps_f;
  const float *w_qkv, *w_o, *w_gu, *w_down;      // [(H + 2 G) HD, D], [D, H HD], [2 F, D], [D, F]
  const float2* table;                           // [positions][HD / 2] (cos, sin), or null
  const int *positions, *row_seq, *write_slots, *block_tables;
  float* plane;
  int bt_ld, D, F, H, G, HD, page_size, window, interleaved, cap;
  float scale;
};

// LDS, in floats: the request's pages as the cache has them, the heads' scores, the row's vectors
struct SbLayout { int pages, scores, x, h, q, kv, attn, hidden, parts, end; };
__host__ __device__ static inline SbLayout sb_layout(int H, int G, int HD, int page_size, int cap) {
  SbLayout l;
  l.pages = 0;
  l.scores = cap / page_size * 2 * G * page_size * HD;
  l.x = l.scores + H * cap;
  l.x = (l.x + 3) / 4 * 4;
  l.h = l.x + SB_WIDTH;
  l.q = l.h + SB_WAVES * SB_WIDTH;               // (a copy a wave)
  l.kv = l.q + SB_WIDTH;
  l.attn = l.kv + 2 * SB_WIDTH;
  l.hidden = l.attn + SB_WIDTH;
  l.parts = l.hidden + SB_HIDDEN;
  l.end = l.parts + SB_WAVES * TIS_WAVE;
  return l;
}

__device__ __forceinline__ float sb_dot(const float4& w, const float4& v, float acc) {
  acc = fmaf(w.x, v.x, acc);
  acc = fmaf(w.y, v.y, acc);
  acc = fmaf(w.z, v.z, acc);
  return fmaf(w.w, v.w, acc);
}
// over the sixteen lanes of a matrix row; each gets it
__device__ __forceinline__ float sb_row_sum(float v) {
  v += butterfly<8>(v);
  v += butterfly<4>(v);
  v += butterfly<2>(v);
  return v + butterfly<1>(v);
}
// a barrier that waits for LDS but not for what is still on its way from memory
__device__ __forceinline__ void sb_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); }

__global__ __launch_bounds__(SB_THREADS) void small_block_kernel(SmallBlock a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), row = t / SB_LANES, l16 = t % SB_LANES;
  const int D = a.D, F = a.F, H = a.H, G = a.G, HD = a.HD, Q = H * HD, N = Q + 2 * G * HD, ps = a.page_size;
  const long r = blockIdx.x;
  const int pos = a.positions[r], slot = a.write_slots[r];
  const int* bt = a.block_tables + (long)a.row_seq[r] * a.bt_ld;
  const SbLayout l = sb_layout(H, G, HD, ps, a.cap);

  // ---- from memory, in the order in which it is needed
  // (addresses past an end are moved inside, and no load waits behind a branch: the compiler would wait for all of them where it joins)
  const int own_lane = min(lane, D - 1);
  const float x_at = a.x[r * a.x_ld + own_lane], gain_a = a.gain_a[own_lane], gain_f = a.gain_f[own_lane];
  auto piece = [&](const float* w, int at, int rows, int p, int K) {
    return *reinterpret_cast<const float4*>(w + (unsigned)(min(at, rows - 1) * K + min(p * 4, K - 4)));
  };
  float4 qkv[SB_QKV], o[SB_O], gu[SB_GU], down[SB_DOWN], kv_held[SB_KV];
  float2 turn[SB_QKV];
#pragma unroll
  for (int s = 0; s < SB_QKV; ++s) qkv[s] = piece(a.w_qkv, s * SB_ROWS + row, N, l16, D);
  o[0] = piece(a.w_o, row, D, l16, Q);
  const float2* angles = a.table ? a.table + (long)pos * (HD / 2) : reinterpret_cast<const float2*>(a.w_qkv);
#pragma unroll
  for (int s = 0; s < SB_QKV; ++s) turn[s] = angles[a.table ? (s * SB_ROWS + row) % HD / 2 : 0];
  const int first = a.window > 0 && pos - a.window + 1 > 0 ? pos - a.window + 1 : 0, n = pos + 1 - first;
  const int page0 = first / ps, per_page = 2 * G * ps * HD / 4, kv_pieces = (pos / ps + 1 - page0) * per_page;
  const float4* plane4 = reinterpret_cast<const float4*>(a.plane);
  auto kv_from = [&](int i) {
    const int at = min(i, kv_pieces - 1), pg = at / per_page;
    return plane4 + (long)bt[page0 + pg] * per_page + (at - pg * per_page);
  };
#pragma unroll
  for (int s = 0; s < SB_KV; ++s) kv_held[s] = *kv_from(t + s * SB_THREADS);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < SB_GU; ++s) gu[s] = piece(a.w_gu, s * SB_ROWS + row, 2 * F, l16, D);
#pragma unroll
  for (int s = 0; s < SB_DOWN; ++s) down[s] = piece(a.w_down, row, D, l16 + s * SB_LANES, F);
  __builtin_amdgcn_sched_barrier(0);
  const float x_own = lane < D ? x_at : 0.f;
  auto dot = [&](const float4& w, const float4& v, int p, int K, float acc) {       // (a piece past the row's end counts for nothing, whatever stands there)
    const float sum = sb_dot(w, v, acc);
    return p * 4 < K ? sum : acc;
  };

  // x * sqrt(D) / (||x|| + eps) * gain, every wave for itself
  float* hs = lds + l.h + wave * SB_WIDTH;
  auto norm = [&](float x, float gain, float eps) {
    const float sum = wave_sum(x * x);
    hs[lane] = x * (sqrtf((float)D) / (sqrtf(sum) + eps)) * gain;
    return *reinterpret_cast<const float4*>(hs + l16 * 4);
  };

  // ---- queries, keys and values: rows 2j and 2j + 1 are a pair of channels, sixteen lanes apart; turned, and the new key and value into the cache
  if (t < SB_HIDDEN) lds[l.hidden + t] = 0.f;
  if (t < SB_WIDTH) lds[l.attn + t] = 0.f;
  const float4 h_a = norm(x_own, gain_a, a.eps_a);
  const long page_elems = (long)ps * HD;
  const int wpage = slot / ps, woff = slot - wpage * ps;
  float* qs = lds + l.q;
  float* kvs = lds + l.kv;                       // the row's own keys [G][HD], then values
  float sums[SB_QKV];
#pragma unroll
  for (int s = 0; s < SB_QKV; ++s) sums[s] = sb_row_sum(dot(qkv[s], h_a, l16, D, 0.f));
  float4* pages = reinterpret_cast<float4*>(lds + l.pages);
#pragma unroll
  for (int s = 0; s < SB_KV; ++s)                // (before the stores below, which not every lane makes: behind them the wait would be for all loads)
    if (t + s * SB_THREADS < kv_pieces) pages[t + s * SB_THREADS] = kv_held[s];
  for (int i = t + SB_KV * SB_THREADS; i < kv_pieces; i += SB_THREADS) pages[i] = *kv_from(i);
#pragma unroll
  for (int s = 0; s < SB_QKV; ++s) {
    const int c = s * SB_ROWS + row;
    const float own = sums[s], other = butterfly<16>(own);
    if (c >= N || l16) continue;
    const int head = c / HD, e = c - head * HD;
    if (head >= H + G) {
      const int kv = head - H - G;
      kvs[(G + kv) * HD + e] = own;
      a.plane[(((long)wpage * 2 + 1) * G + kv) * page_elems + (long)e * ps + woff] = own;
      continue;
    }
    const int j = e / 2, at = a.interleaved ? e : e % 2 == 0 ? j : j + HD / 2;
    float y = own;
    if (a.table) {
      const float2 cs = turn[s];
      y = e % 2 == 0 ? fmaf(own, cs.x, -(other * cs.y)) : fmaf(own, cs.x, other * cs.y);
    }
    if (head < H) qs[head * HD + at] = y * a.scale;
    else {
      kvs[(head - H) * HD + at] = y;
      a.plane[((long)wpage * 2 * G + head - H) * page_elems + (long)woff * HD + at] = y;
    }
  }
  sb_barrier();

  // ---- attention: a head a wave
  for (int head = wave; head < H; head += SB_WAVES) {
    const int kv = head / (H / G), from = first - page0 * ps;       // (key first + i lies at place from + i of the pages in LDS)
    const float* qh = qs + head * HD;
    const float* mine = lds + l.pages;
    float* sc = lds + l.scores + head * a.cap;
    float top = -INFINITY;
    for (int i = lane; i < n; i += TIS_WAVE) {
      const int j = from + i, pg = j / ps;
      const float* kp = i == n - 1 ? kvs + kv * HD : mine + ((long)pg * 2 * G + kv) * page_elems + (j - pg * ps) * HD;
      float s = 0.f;
      for (int e = 0; e < HD; e += 4) s = sb_dot(*reinterpret_cast<const float4*>(qh + e), *reinterpret_cast<const float4*>(kp + e), s);
      sc[i] = s;
      top = fmaxf(top, s);
    }
    top = wave_max(top);
    float sum = 0.f;
    for (int i = lane; i < n; i += TIS_WAVE) {
      const float p = expf(sc[i] - top);
      sc[i] = p;
      sum += p;
    }
    sum = wave_sum(sum);
    const int groups = TIS_WAVE / HD, g = lane / HD, d = lane - g * HD;
    const float* own_value = kvs + (G + kv) * HD + d;
    float acc = 0.f;
    if (g < groups)
#pragma unroll 4
      for (int i = g; i < n; i += groups) {
        const int j = from + i, pg = j / ps;
        const float* vp = i == n - 1 ? own_value : mine + (((long)pg * 2 + 1) * G + kv) * page_elems + (long)d * ps + (j - pg * ps);
        acc = fmaf(sc[i], *vp, acc);
      }
    float* parts = lds + l.parts + wave * TIS_WAVE;
    parts[lane] = acc;
    if (lane < HD) {
      float out = 0.f;
      for (int k = 0; k < groups; ++k) out += parts[k * HD + lane];
      lds[l.attn + head * HD + lane] = out / sum;
    }
  }
  sb_barrier();

  // ---- output projection and residual
  const float proj = sb_row_sum(dot(o[0], *reinterpret_cast<const float4*>(lds + l.attn + l16 * 4), l16, Q, 0.f));
  // (lane i of wave w has row 4 w + i / 16 of this sum and element i of the row itself)
  if (l16 == 0) lds[l.x + row] = proj;
  sb_barrier();
  const float mid = lds[l.x + lane] + x_own;

  // ---- norm and feed-forward: rows in pairs (gate, up)
  const float4 h_f = norm(lane < D ? mid : 0.f, gain_f, a.eps_f);
#pragma unroll
  for (int s = 0; s < SB_GU; ++s) {
    const int c = s * SB_ROWS + row;
    const float g = sb_row_sum(dot(gu[s], h_f, l16, D, 0.f)), up = butterfly<16>(g);
    if (c < 2 * F && c % 2 == 0 && l16 == 0) lds[l.hidden + c / 2] = g / (1.f + expf(-g)) * up;
  }
  sb_barrier();
  float y = 0.f;
#pragma unroll
  for (int s = 0; s < SB_DOWN; ++s) y = dot(down[s], *reinterpret_cast<const float4*>(lds + l.hidden + (l16 + s * SB_LANES) * 4), l16 + s * SB_LANES, F, y);
  y = sb_row_sum(y);
  const float res = __shfl(mid, row, TIS_WAVE);
  if (row < D && l16 == 0) a.out[r * a.out_ld + row] = y + res;
}

// Whether this kernel takes a block of these sizes, whose rows see up to `keys` keys: its matrices in the threads' registers, its keys and values in LDS, and
// no more rows and keys than it is the faster one for (see the figures above).
TIS_EXPORT int tis_small_block_takes(int rows, int D, int F, int H, int G, int HD, int keys, int page_size) {
  if (rows < 1 || rows > SB_ROWS_MOST || D < 4 || D > SB_WIDTH || D % 4 || F < 4 || F % 4 || F > SB_HIDDEN || H < 1 || G < 1 || H % G || HD < 4 || HD % 4 ||
      H > SB_WIDTH || HD > SB_WIDTH || H * HD > SB_WIDTH || (H + 2 * G) * HD > SB_QKV * SB_ROWS || keys < 1 || keys > SB_KEYS || page_size < 1 || page_size > SB_KEYS)
    return 0;
  const int groups = TIS_WAVE / HD;              // keys that a wave's value sums take at a time
  if (keys > (rows <= SB_ROWS_ROUND ? 128 : 8 * H) * groups) return 0;
  const long cap = ((long)keys + page_size - 1) / page_size * page_size;
  if (cap * (2L * G * HD + H) * 4 > SB_LDS) return 0;
  return sb_layout(H, G, HD, page_size, (int)cap).end * 4L <= SB_LDS;
}

// The dynamic LDS that the kernel may be launched with on this device, -1 where the runtime does not say.
TIS_EXPORT int tis_small_block_lds() {
  hipFuncAttributes got;
  return hipFuncGetAttributes(&got, (const void*)small_block_kernel) == hipSuccess ? got.maxDynamicSharedSizeBytes : -1;
}

// The kernel may be launched with all of a compute unit's LDS, said once a device: said for each call's own size it would be lowered by a smaller call, under a
// larger one that another thread is about to launch.
static hipError_t sb_allow_lds() {
  static std::mutex lock;
  static unsigned long long allowed = 0;         // a bit a device
  int device = 0;
  if (hipError_t e = hipGetDevice(&device); e != hipSuccess) return e;
  const unsigned long long bit = device < 64 ? 1ull << device : 0;
  std::lock_guard<std::mutex> held(lock);
  if (allowed & bit) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute((const void*)small_block_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)SB_LDS);
  if (e == hipSuccess) allowed |= bit;
  return e;
}

// x, out: [rows, D] 32-bit, row strides x_ld, out_ld; the matrices as the separate kernels take them (rows of query and key heads in rotary pairs, gate
// and up rows in turn), on 16 bytes; keys: the most a row sees of its request's (its position is below). Launches only: safe under stream capture.
TIS_EXPORT int tis_small_block(const float* x, long x_ld, float* out, long out_ld, const float* gain_a, float eps_a, const float* w_qkv, const float* w_o,
                               const float* gain_f, float eps_f, const float* w_gu, const float* w_down, const float* table, int interleaved,
                               const int* positions, const int* row_seq, const int* write_slots, const int* block_tables, int bt_ld, float* plane, int rows,
                               int D, int F, int H, int G, int HD, int page_size, int window, float scale, int keys, hipStream_t stream) {
  if (rows == 0) return 0;
  if (!tis_small_block_takes(rows, D, F, H, G, HD, keys, page_size))
    return tis_fail("small_block: %d rows of %d, %d hidden, %d heads of %d over %d, %d keys: not a block that a compute unit holds", rows, D, F, H, HD, G, keys);
  const int pages = (keys + page_size - 1) / page_size, cap = pages * page_size;
  if (x_ld < D || out_ld < D || window < 0 || !positions || !row_seq || !write_slots || !block_tables || !plane || bt_ld < pages)
    return tis_fail("small_block: row strides %ld, %ld for %d values, or block tables of %d pages for %d keys", x_ld, out_ld, D, bt_ld, keys);
  if (((uintptr_t)w_qkv | (uintptr_t)w_o | (uintptr_t)w_gu | (uintptr_t)w_down | (uintptr_t)plane) % 16 || (uintptr_t)table % 8)
    return tis_fail("small_block: matrices and cache start on 16 bytes");
  const SmallBlock a{x, x_ld, out, out_ld, gain_a, gain_f, eps_a, eps_f, w_qkv, w_o, w_gu, w_down, (const float2*)table, positions, row_seq, write_slots,
                     block_tables, plane, bt_ld, D, F, H, G, HD, page_size, window, interleaved, cap, scale};
  const size_t bytes = sb_layout(H, G, HD, page_size, cap).end * sizeof(float);
  if (hipError_t e = sb_allow_lds(); e != hipSuccess) return tis_fail("small_block: %ld bytes of LDS: %s", SB_LDS, hipGetErrorString(e));
  small_block_kernel<<<rows, SB_THREADS, bytes, stream>>>(a);
  return tis_launch_status("small_block");
}
