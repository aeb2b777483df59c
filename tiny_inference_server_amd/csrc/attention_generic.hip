// Attention of query rows over paged keys and values: the kernel for every head size and for 32-bit.
//
// One workgroup per (row, query head). The row at position p of a request sees the keys at positions
// [max(0, p - window + 1), p] of that request (window 0: all of them), found through the request's block
// table. Query head h reads key/value head h / group_size (reference paged_attention_kernels.py:49).
// Scores, maximum, sum and the output accumulate in 32-bit (reference paged_attention_kernels.py:86-108);
// masked keys are never read, so what a reused page still holds cannot reach the result.
// A page holds a head's keys as [slot][head_dim] and its values as [head_dim][slot].
// A position encoding that works on the scores brings one slope per query head: the score of key j for the row at
// position p gets slope[h] * (j - p) added (a bias linear in the distance; null: none).
// Keys are walked in chunks of a fixed size with a running maximum, so the order of every sum depends on
// the row's own length only, not on what else is in the batch.
//
// What bounds it is the chain of trips to memory and through LDS of one small workgroup: the row's position and request, the block table, a
// key's channels and the values, which are asked for together (rows of up to 50 keys, 8 heads of 8, 32-bit, traced in replayed steps,
// us: one channel and one value after the other 5.7, AG_AHEAD pieces of 16 bytes of a key and AG_AHEAD values of a thread at a time 5.0). The sums keep their
// order.
#include <algorithm>
#include <utility>
#include <vector>

#include "common.h"

TIS_DEFINE_LAST_ERROR(tis_attention_generic)

static constexpr int AG_THREADS = 256;
static constexpr int AG_CHUNK = 1024;
static constexpr int AG_MAX_HD = 256;
static constexpr int AG_AHEAD = 4;

// WIDE: a key is read 16 bytes at a time
template <typename T> struct alignas(16) AgPiece { T v[16 / sizeof(T)]; };

template <typename T, bool WIDE>
__global__ __launch_bounds__(AG_THREADS) void attention_generic_kernel(
    const T* __restrict__ q, long q_ld, const T* __restrict__ plane, const int* __restrict__ block_tables, int bt_ld,
    const int* __restrict__ row_seq, const int* __restrict__ positions, T* __restrict__ out, long out_ld,
    int group_size, int n_kv_heads, int HD, int page_size, int window, float scale, const float* __restrict__ slopes) {
  __shared__ float qs[AG_MAX_HD];
  __shared__ float sc[AG_CHUNK];
  __shared__ float red[16];
  __shared__ float accm[AG_THREADS];

  const long r = blockIdx.x;
  const int h = blockIdx.y;
  const int kvh = h / group_size;
  const int t = threadIdx.x;
  const int pos = positions[r];
  const int* bt = block_tables + (long)row_seq[r] * bt_ld;
  const int first = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
  const int kv_end = pos + 1;
  const float slope = slopes ? slopes[h] : 0.f;

  for (int d = t; d < HD; d += AG_THREADS) qs[d] = to_f(q[r * q_ld + (long)h * HD + d]) * scale;
  __syncthreads();

  const long page_stride = 2L * n_kv_heads * page_size * HD;
  const long k_off = (long)kvh * page_size * HD;
  const long v_off = ((long)n_kv_heads + kvh) * page_size * HD;

  const int groups = AG_THREADS / HD;  // HD <= 256 so at least 1
  const int g = t / HD, d = t % HD;
  const bool pv_thread = g < groups;

  float m = -INFINITY, l = 0.f, acc = 0.f;
  for (int c0 = first; c0 < kv_end; c0 += AG_CHUNK) {
    const int n = min(AG_CHUNK, kv_end - c0);
    // a thread's values of the keys g + u groups, u from u0 on (past the chunk's last: that one's)
    float ahead[AG_AHEAD];
    auto values = [&](int u0) {
#pragma unroll
      for (int u = 0; u < AG_AHEAD; ++u) {
        const int j = c0 + min(g + (u0 + u) * groups, n - 1);
        const T* vp = plane + (long)bt[j / page_size] * page_stride + v_off + (j % page_size);
        ahead[u] = to_f(vp[(long)d * page_size]);  // values lie transposed: [head_dim][slot]
      }
    };
    values(0);                                     // under way while the scores are worked out
    float cmax = -INFINITY;
    for (int i = t; i < n; i += AG_THREADS) {
      const int j = c0 + i;
      const T* kp = plane + (long)bt[j / page_size] * page_stride + k_off + (long)(j % page_size) * HD;
      float s = 0.f;
      if constexpr (WIDE) {
        constexpr int PIECE = 16 / sizeof(T);
        for (int e0 = 0; e0 < HD; e0 += AG_AHEAD * PIECE) {
          AgPiece<T> piece[AG_AHEAD];
#pragma unroll
          for (int u = 0; u < AG_AHEAD; ++u) piece[u] = *reinterpret_cast<const AgPiece<T>*>(kp + min(e0 + u * PIECE, HD - PIECE));
#pragma unroll
          for (int u = 0; u < AG_AHEAD; ++u) {
            if (e0 + u * PIECE >= HD) break;
#pragma unroll
            for (int e = 0; e < PIECE; ++e) s += qs[e0 + u * PIECE + e] * to_f(piece[u].v[e]);
          }
        }
      } else {
        for (int e = 0; e < HD; ++e) s += qs[e] * to_f(kp[e]);
      }
      if (slopes) s += slope * (float)(j - pos);
      sc[i] = s;
      cmax = fmaxf(cmax, s);
    }
    cmax = block_max(cmax, red);
    const float m_new = fmaxf(m, cmax);
    float csum = 0.f;
    for (int i = t; i < n; i += AG_THREADS) {
      const float p = expf(sc[i] - m_new);
      sc[i] = p;
      csum += p;
    }
    csum = block_sum(csum, red);  // its barriers also publish sc[]
    const float rescale = expf(m - m_new);  // 0 on the first chunk (m = -inf)
    l = l * rescale + csum;
    acc *= rescale;
    m = m_new;
    for (int u0 = 0; g + u0 * groups < n; u0 += AG_AHEAD) {
      if (u0) values(u0);
#pragma unroll
      for (int u = 0; u < AG_AHEAD; ++u) {
        const int i = g + (u0 + u) * groups;
        if (pv_thread && i < n) acc += sc[i] * ahead[u];
      }
    }
    __syncthreads();  // sc[] is rewritten by the next chunk
  }
  accm[t] = pv_thread ? acc : 0.f;
  __syncthreads();
  if (t < HD) {
    float o = 0.f;
#pragma unroll 8
    for (int gg = 0; gg < groups; ++gg) o += accm[gg * HD + t];
    out[r * out_ld + (long)h * HD + t] = from_f<T>(o / l);
  }
}

TIS_EXPORT int tis_attention_generic(int dtype, const void* q, long q_ld, const void* plane, const int* block_tables,
                                     int bt_ld, const int* row_seq, const int* positions, void* out, long out_ld,
                                     int rows, int n_heads, int n_kv_heads, int head_dim, int page_size, int window,
                                     float scale, const float* slopes, hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || n_heads < 1 || n_kv_heads < 1 || n_heads % n_kv_heads || page_size < 1 || window < 0)
    return tis_fail("attention: bad size rows=%d heads=%d kv_heads=%d page=%d window=%d", rows, n_heads, n_kv_heads,
                    page_size, window);
  if (head_dim < 1 || head_dim > AG_MAX_HD)
    return tis_fail("attention: head size %d is outside this kernel's range 1..%d", head_dim, AG_MAX_HD);
  if (n_heads > 65535) return tis_fail("attention: %d heads exceed the grid", n_heads);
  dim3 grid(rows, n_heads);
  const int group = n_heads / n_kv_heads;
  const bool wide = (uintptr_t)plane % 16 == 0 && head_dim * (dtype == TIS_F32 ? 4 : 2) % 16 == 0;     // keys start on 16 bytes
#define LAUNCH(T, W)                                                                                                          \
  attention_generic_kernel<T, W><<<grid, AG_THREADS, 0, stream>>>((const T*)q, q_ld, (const T*)plane, block_tables, bt_ld, row_seq,       \
                                                                  positions, (T*)out, out_ld, group, n_kv_heads, head_dim, page_size,  \
                                                                  window, scale, slopes)
  if (dtype == TIS_F32) {
    if (wide) LAUNCH(float, true);
    else LAUNCH(float, false);
  } else if (dtype == TIS_BF16) {
    if (wide) LAUNCH(bf16, true);
    else LAUNCH(bf16, false);
  } else {
    return tis_fail("unknown dtype code %d", dtype);
  }
#undef LAUNCH
  return tis_launch_status("attention_generic");
}

// ---- host planning -----------------------------------------------------------------------------------------
//
// (Here, because every engine loads this library once; the tile kernel's source is built once a head size.)
// The parts that the tile kernel of attention_mfma.hip cuts its tiles into, those with the longest chains of steps first (those alike in the order
// of their tiles): (first row, rows + 256 * split, position of the first row, block-table line) each, into out [capacity][4]. rows: (first row, first
// position, rows) of each request; tiles: (first row, rows) each. The counts are the kernel's own: a tile of n steps of 32 keys, from a multiple of 32
// at or before the first key that any row sees, has min(splits, ceil(n / most)) parts of ceil(n / parts) steps, the last what is left. The host's
// work before a prompt's first launch: 64 tiles cut in five 9 us with the call, 50 as array operations. Returns the parts, or -1.
TIS_EXPORT int tis_attention_tile_pieces(const long* rows, int n_rows, const int* tiles, int n_tiles, int splits, int most, int window, int* out, int capacity) {
  if (n_rows < 0 || n_tiles < 0 || splits < 1 || most < 1) return tis_fail("tile_pieces: %d tiles of %d requests, %d parts of %d steps", n_tiles, n_rows, splits, most), -1;
  try {
    struct Piece {
      long steps;
      int first, rows, pos, line;
    };
    std::vector<std::pair<long, int>> live;
    for (int i = 0; i < n_rows; ++i)
      if (rows[3 * i + 2] > 0) live.emplace_back(rows[3 * i], i);          // (first rows rise)
    std::vector<Piece> pieces;
    pieces.reserve(std::min((long)capacity, (long)n_tiles * splits));
    for (int t = 0; t < n_tiles; ++t) {
      const int first = tiles[2 * t], count = tiles[2 * t + 1];
      auto after = std::upper_bound(live.begin(), live.end(), std::make_pair((long)first, n_rows));
      if (after == live.begin()) return tis_fail("tile_pieces: the tile at row %d is no request's", first), -1;
      const int line = (--after)->second;
      const long pos = rows[3 * line + 1] + first - after->first;
      const long seen = window > 0 ? std::max(0L, pos - window + 1) : window < 0 ? pos - pos % -(long)window : 0;
      const long steps = (pos + count - (seen & ~31L) + 31) / 32;
      const long parts = std::min((long)splits, std::max(1L, (steps + most - 1) / most)), per = (steps + parts - 1) / parts;
      for (long s = 0; s < parts; ++s) pieces.push_back({std::min(per, steps - s * per), first, count + 256 * (int)s, (int)pos, line});
    }
    if (pieces.size() > (size_t)std::max(0, capacity)) return tis_fail("tile_pieces: %zu parts for %d places", pieces.size(), capacity), -1;
    std::stable_sort(pieces.begin(), pieces.end(), [](const Piece& a, const Piece& b) { return a.steps > b.steps; });
    for (const Piece& p : pieces) {
      *out++ = p.first;
      *out++ = p.rows;
      *out++ = p.pos;
      *out++ = p.line;
    }
    return (int)pieces.size();
  } catch (...) {
    return tis_fail("tile_pieces: no memory"), -1;
  }
}
