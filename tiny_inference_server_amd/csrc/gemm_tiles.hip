// C[M,N] = X[M,K] . W[N,K]^T (+ R[M,N]) in bfloat16 for many rows at widths where the library's product is not used:
// a product tiled in both directions on v_mfma_f32_32x32x16_bf16 (gfx950), operands through LDS by direct loads.
// (The few-row kernel takes such a product in panels of 32 rows, each of which streams all of W again: 0.25 to 0.3
// PFLOP/s at 2,048 rows. This kernel reaches 0.75 to 1.0 on the same shapes; the library's kernels, where they may be
// used, 0.5 to 1.3.) The reference's engine uses a library product here (x @ W, main_models_new.py:19-20).
//
// tile_loop.h holds the loop. A row's sums run over K in the same order whatever M is and whichever tile is taken: its result does not depend on the other rows.
#include <climits>
#include <type_traits>

#include "tile_loop.h"

TIS_DEFINE_LAST_ERROR(tis_gemm_tiles)

// BM x BN: the workgroup's tile; WM x WN: its waves, each with (BM / WM) x (BN / WN) of it
// ACT: what becomes of a sum before it is rounded (0 nothing; 1 the tanh form of gelu, 0.5 z (1 + tanh(u)) written as
// z / (1 + exp(-2u)); 2 the square of relu; of the columns' pairs (2j, 2j + 1), for a C of N / 2 columns: 3 clamped_swish, 4 silu(g) u)
template <int ACT> __device__ __forceinline__ float gt_activated(float z) {
  if (ACT == 1) return z / (1.f + __expf(-1.5957691216057308f * (z + 0.044715f * z * z * z)));
  if (ACT == 2) { const float p = fmaxf(z, 0.f); return p * p; }
  return z;
}
template <int ACT> __device__ __forceinline__ float gt_gated(float g, float u, float limit) {
  if (ACT == 3) return clamped_swish(g, u, limit);
  // the gate of the rounded product, as the kernel that reads a stored one takes it: the same bits whichever way a step went
  g = static_cast<float>(static_cast<__bf16>(g));
  u = static_cast<float>(static_cast<__bf16>(u));
  return g / (1.f + expf(-g)) * u;
}

// acc = the tile's sums over K
template <typename Loop, int BM>
__device__ __forceinline__ void tile_sums(unsigned char* lds, const bf16* X, long x_ld, const bf16* W, long m0, long n0, int M, int N, int K,
                                          f32x16 (&acc)[Loop::TM][Loop::TN]) {
  constexpr int LPW = Loop::LPW;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  // Rows past the matrix's last are the last row again (their results are not stored).
  const unsigned char* first[LPW];
  unsigned lane_off[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int row0 = Loop::row_of(wave, 0, j), row = Loop::row_of(wave, lane, j);
    const bool of_x = row0 < BM;
    const long ld = of_x ? x_ld : (long)K;
    const long last = of_x ? (long)M - 1 : (long)N - 1;
    const long g_first = min(last, of_x ? m0 + row0 : n0 + (row0 - BM));
    const long g_row = min(last, of_x ? m0 + row : n0 + (row - BM));
    first[j] = (const unsigned char*)(of_x ? X : W) + g_first * ld * 2;
    lane_off[j] = (unsigned)((g_row - g_first) * ld * 2 + Loop::piece_of(lane, row) * 16);
  }
#pragma unroll
  for (int i = 0; i < Loop::TM; ++i)
#pragma unroll
    for (int j = 0; j < Loop::TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  Loop::run(lds, first, lane_off, K, acc);
}

template <int BM, int BN, int WM, int WN, int NSTAGE, int AHEAD, bool RESIDUAL, typename TO, int ACT = 0>
__global__ __launch_bounds__(WM * WN * 64) void gemm_tiles_kernel(
    const bf16* __restrict__ X, long x_ld, const bf16* __restrict__ W, const bf16* R, long r_ld, TO* C, long c_ld,
    int M, int N, int K, float limit, int wide) {
  typedef TileLoop<BM, BN, WM, WN, NSTAGE, AHEAD> Loop;
  constexpr int TM = Loop::TM, TN = Loop::TN;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[NSTAGE * Loop::STAGE];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r32 = lane & 31, h = lane >> 5;
  const int wm = wave / WN, wn = wave % WN;
  const GtTile tile = gt_tile(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN);
  const long m0 = (long)tile.m * BM, n0 = (long)tile.n * BN;
  // The residual's four of every eight columns, asked for before the first step where they find room: behind the last one they would be a trip to memory
  // that nothing hides. (R may be C: a wave reads its own results' places before it writes them; what lanes past an end read nobody looks at.)
  constexpr bool EARLY = RESIDUAL && TM * TN <= 4;
  bf16x4 res[EARLY ? TM : 1][EARLY ? TN : 1][4];
  if constexpr (EARLY)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          res[i][j][q] = *(const bf16x4*)(R + min(m0 + wm * (BM / WM) + i * 32 + r32, (long)M - 1) * r_ld + min(n0 + wn * (BN / WN) + j * 32 + q * 8 + h * 4, (long)N - 4));
  f32x16 acc[TM][TN];
  tile_sums<Loop, BM>(lds, X, x_ld, W, m0, n0, M, N, K, acc);

  // Accumulator 4 q + e of block (i, j): row m0 + wm * (BM / WM) + i * 32 + r32, column n0 + wn * (BN / WN) + j * 32 + 8 q + 4 h + e. A lane's four columns are
  // 4 (gated), 8 or 16 bytes of a row; stored as they are, an instruction reaches 32 rows with 8 to 32 bytes each. Where the result's rows lie on 16 bytes
  // they pass through LDS, 32 rows of the wave at a time, and leave 16 bytes a lane, a row's side by side. us, stored as they are with a late residual / so, matrices from
  // memory: 2,048 rows of 1,536 x 1,536 with a residual 16.6 / 14.7, of 1,536 x 4,096 34.8 / 33.6, of 2,304 x 1,536 21.8 / 19.7; 3,000 of 2,816 x 1,024 28.3 / 24.6; 32-bit
  // results 1,800 of 32,000 x 2,048 252 / 242, 2,048 of 3,072 x 2,048 32.4 / 30.3; gated 600 of 8,192 x 1,536 23.8 / 22.6. At 30 sizes none slower by more than 0.5 %.
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  using Four = std::conditional_t<(ACT >= 3), bf16x2, std::conditional_t<sizeof(TO) == 4, f32x4, bf16x4>>;
  auto four = [&](int i, int j, int q, long m, long n) {
    Four o;
    if constexpr (ACT >= 3) {
      o = (bf16x2){static_cast<__bf16>(gt_gated<ACT>(acc[i][j][q * 4], acc[i][j][q * 4 + 1], limit)),
                   static_cast<__bf16>(gt_gated<ACT>(acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3], limit))};
    } else {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = gt_activated<ACT>(acc[i][j][q * 4 + e]);
      if constexpr (RESIDUAL) {
        bf16x4 r;
        if constexpr (EARLY) r = res[i][j][q];
        else r = *(const bf16x4*)(R + min(m, (long)M - 1) * r_ld + min(n, (long)N - 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += (float)r[e];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (sizeof(TO) == 4) o[e] = v[e];       // the 32-bit sums as they are
        else o[e] = static_cast<__bf16>(v[e]);
      }
    }
    return o;
  };
  constexpr int ROW = TN * 8 * sizeof(Four), PITCH = ROW + 16, PIECES = ROW / 16, COLUMNS = 64 / sizeof(Four);      // bytes of a wave's row, 16-byte pieces, W's rows a piece
  const long out_n0 = n0 + wn * (BN / WN);
  const int per = ACT >= 3 ? 2 : 1;
  if (wide) {
    static_assert(32 * PITCH * WM * WN <= NSTAGE * Loop::STAGE, "the waves' rows in the operands' place");
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");      // every wave has its last operands
    unsigned char* mine = lds + wave * 32 * PITCH;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const long row0 = m0 + wm * (BM / WM) + i * 32;
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *(Four*)(mine + r32 * PITCH + ((j * 4 + q) * 2 + h) * sizeof(Four)) = four(i, j, q, row0 + r32, out_n0 + j * 32 + q * 8 + h * 4);
      asm volatile("" : : : "memory");
#pragma unroll
      for (int k = 0; k < PIECES / 2; ++k) {
        const int p = k * 64 + lane, row = p / PIECES, at = p % PIECES;
        const f32x4 v = *(const f32x4*)(mine + row * PITCH + at * 16);
        if (row0 + row < M && out_n0 + at * COLUMNS < N) *(f32x4*)(C + (row0 + row) * c_ld + (out_n0 + at * COLUMNS) / per) = v;
      }
      asm volatile("" : : : "memory");
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const long m = m0 + wm * (BM / WM) + i * 32 + r32;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const long n = out_n0 + j * 32 + q * 8 + h * 4;
        if (n < N) *(Four*)(C + m * c_ld + n / per) = four(i, j, q, m, n);        // (N is a multiple of 4: the four columns are inside or outside together)
      }
  }
}

// The product that makes a prompt's queries, keys and values: W's rows are the heads' channels, the queries' and keys' in pairs (2j, 2j + 1 of a
// head: channels j and j + head_dim / 2). A lane holds two whole pairs of a row, so they are turned by the row's position where they lie, in 32 bits
// from the product rounded to bfloat16, as the kernel that reads a stored product takes it (the same bits). Queries go to q_out, keys to the row's slot
// of the cache's pages, values there transposed. What it saves is that kernel: its launch and the product's way to memory and back (2,048 rows of 18 heads of
// 128 against 1,536, us: 29.2 / 24.7; 1,532 rows of 24 against 2,048 33.8 / 30.0). The rows' cosines and sines are asked for before the first step, where they find room.
struct RopeOut {
  const int* positions;
  const int* write_slots;     // null: keys and values have no reader
  const float2* table;        // [positions][head_dim / 2] (cos, sin)
  bf16* plane;                // [page][keys, values][kv head][page_size * head_dim]
  int n_heads, n_kv_heads, head_dim, page_size;
};
template <int BM, int BN, int WM, int WN, int NSTAGE, int AHEAD>
__global__ __launch_bounds__(WM * WN * 64) void gemm_tiles_rope_kernel(const bf16* __restrict__ X, long x_ld, const bf16* __restrict__ W,
                                                                       bf16* __restrict__ q_out, long q_ld, int M, int N, int K, RopeOut a) {
  typedef TileLoop<BM, BN, WM, WN, NSTAGE, AHEAD> Loop;
  constexpr int TM = Loop::TM, TN = Loop::TN;
  constexpr bool EARLY = TM * TN <= 4;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[NSTAGE * Loop::STAGE];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r32 = lane & 31, h = lane >> 5;
  const int wm = wave / WN, wn = wave % WN;
  const GtTile tile = gt_tile(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN);
  const long m0 = (long)tile.m * BM, n0 = (long)tile.n * BN;
  const int HD = a.head_dim, half = HD / 2;
  int head[TN], d0[TN];                          // of a block of 32 columns (head sizes are multiples of 32): its head, its first channel
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = (int)n0 + wn * (BN / WN) + j * 32;
    head[j] = __builtin_amdgcn_readfirstlane(n / HD);
    d0[j] = n - head[j] * HD;
  }
  int pos[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) pos[i] = a.positions[min(m0 + wm * (BM / WM) + i * 32 + r32, (long)M - 1)];
  // (cos, sin) of the lane's two pairs of every eight columns
  auto factors = [&](int i, int j, float4 (&cs)[4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) cs[q] = *reinterpret_cast<const float4*>(a.table + (long)pos[i] * half + d0[j] / 2 + q * 4 + h * 2);
  };
  float4 held[EARLY ? TM : 1][EARLY ? TN : 1][4];
  if constexpr (EARLY)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) factors(i, j, held[i][j]);
  f32x16 acc[TM][TN];
  tile_sums<Loop, BM>(lds, X, x_ld, W, m0, n0, M, N, K, acc);

  const long page_elems = (long)a.page_size * HD;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const long m = m0 + wm * (BM / WM) + i * 32 + r32;
    const bool row = m < M;
    int page = 0, slot = 0;
    if (a.write_slots) {
      const int at = a.write_slots[min(m, (long)M - 1)];
      page = at / a.page_size;
      slot = at - page * a.page_size;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if (n0 + wn * (BN / WN) + j * 32 >= N) continue;       // (the same for the wave, as the head is)
      const int kv = head[j] - a.n_heads, value = kv - a.n_kv_heads;
      if (kv >= 0 && !a.write_slots) continue;
      if (value >= 0) {
        bf16* dst = a.plane + (((long)page * 2 + 1) * a.n_kv_heads + value) * page_elems + slot;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (row) dst[(long)(d0[j] + q * 8 + h * 4 + e) * a.page_size] = static_cast<__bf16>(acc[i][j][q * 4 + e]);
        continue;
      }
      float4 late[4];
      if constexpr (!EARLY) factors(i, j, late);
      uint32_t lo[4], hi[4];                     // of the head's halves: the lane's two channels of every four
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
        const float4 cs = EARLY ? held[EARLY ? i : 0][EARLY ? j : 0][q] : late[q];
        const float c[2] = {cs.x, cs.z}, sn[2] = {cs.y, cs.w};
        bf16x2 y1, y2;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float x1 = static_cast<float>(static_cast<__bf16>(acc[i][j][q * 4 + 2 * e])), x2 = static_cast<float>(static_cast<__bf16>(acc[i][j][q * 4 + 2 * e + 1]));
          // (which of the two products is rounded before the sum is spelled out, as the rotary kernel has it: the compiler's choice differs)
          y1[e] = static_cast<__bf16>(fmaf(x1, c[e], -(x2 * sn[e])));
          y2[e] = static_cast<__bf16>(fmaf(x1, sn[e], x2 * c[e]));
        }
        lo[q] = __builtin_bit_cast(uint32_t, y1);
        hi[q] = __builtin_bit_cast(uint32_t, y2);
      }
      bf16* dst = kv < 0 ? q_out + m * q_ld + (long)head[j] * HD : a.plane + ((long)page * 2 * a.n_kv_heads + kv) * page_elems + (long)slot * HD;
#pragma unroll
      for (int q = 0; q < 4; q += 2) {           // the lane beside it (32 on) has the other two of four: each takes four of one piece, 8 bytes
        const auto l = __builtin_amdgcn_permlane32_swap(lo[q], lo[q + 1], false, false), u = __builtin_amdgcn_permlane32_swap(hi[q], hi[q + 1], false, false);
        bf16* at = dst + d0[j] / 2 + (q + h) * 4;
        if (row) *reinterpret_cast<uint2*>(at) = make_uint2(l[0], l[1]);
        if (row) *reinterpret_cast<uint2*>(at + half) = make_uint2(u[0], u[1]);
      }
    }
  }
}

static int g_units = 256;      // compute units of the device: set by whoever knows (the default is an MI355X)
TIS_EXPORT void tis_gemm_tiles_units(int n) { if (n > 0) g_units = n; }

// The tiles, and what a product is estimated to take with each, us: a beginning and end, and the time of a step of 64 by r, the tiles a
// compute unit. Measured with matrices that come from memory (none that a cache still holds), 129 to 8,000 rows, widths of 256 to 48,000. Over
// 617 such products the one picked here took 1.006 times the fastest's time on average while results left as they lay. The estimates are as they were then: as results leave
// now (see gemm_tiles_kernel) it takes 1.02 times over 132 products, 90 of them drawn, and 25 of the 132 take more than 3 % longer than with the fastest
// (159 rows of 32,928 x 1,792 49 / 43, 1,172 of 3,016 x 832 13.5 / 11.6).
//
// What bounds a product of few hundred rows is the way of its matrix from memory: a tile's copies reach two to five steps ahead (what
// its buffers hold; two for the 256 x 256 and the 128 x 192 tile, 5 instead of 4 buffers of 64 x 64, 6 of 64 x 32 and 128 x 64), and there are tiles enough for the chip. us before
// (tiles of 64 x 64 up to 256 x 256, three steps ahead) / now, and the library's product: 300 rows of 1,536 x 1,536 11.1 / 7.7 (10.6), of
// 2,304 x 1,536 11.4 / 9.3 (16.6), of 1,536 x 4,096 26 / 15.3 (21.1); 140 rows of 1,536 x 4,096 24.6 / 14.9 (15.6); 700 rows of 2,304 x 1,536
// 15.2 / 11.0 (16.4); 2,048 rows of 2,304 x 1,536 33 / 21.1 (23.7), of 2,816 x 2,048 41.1 / 28.7 (30.4), of 3,072 x 2,048 41.0 / 31.2 (30.5).
// (K in two parts by two sets of waves, for products of less than a tile a unit: 1 to 2.5 us less, but other sums than every other tile's,
// and than the library's, with which all of these agree to the bit.)
// Beyond one tile a unit a tile's LDS says how many share one: two of 128 x 192, 64 x 64 and 64 x 32, else one.
// Tiles of less than 256 x 256 that are alone on their unit are bound by the unit's way from the L2 into LDS, some 60 bytes a nanosecond whatever their size
// and waves; so for a product of two to three million results, one tile a unit, the smaller the rows of a step the better: 128 x 96 (96 x 128 where only that many
// fit) in place of 128 x 128, four waves of three 32 x 32 results each. us, 128 x 128 / these, and the library's product: 1,900 rows of 1,536 x 4,096 38.4 / 34.1
// (35.6), 1,605 34.2 / 31.1 (31.9), 2,048 38.5 / 34.7 (35.8); of 2,048 x 5,632 1,195 46.5 / 40.0 (47.6), 1,482 50.5 / 45.8 (44.0); 1,060 rows of 2,304 x 1,536 15.1 / 14.6
// (19.9), of 2,048 x 2,048 18.4 / 17.2 (22.9).
struct TileShape { int bm, bn; };
static constexpr int GT_SHAPES = 10;
static const TileShape g_shapes[GT_SHAPES] = {{256, 256}, {256, 128}, {192, 128}, {128, 192}, {128, 128}, {128, 64}, {64, 64}, {64, 32}, {128, 96}, {96, 128}};
// DO(BM, BN, WM, WN, NSTAGE, AHEAD) for tile `pick`
#define GT_EACH_TILE(pick, DO)                   \
  switch (pick) {                                \
    case 0: DO(256, 256, 2, 4, 2, 1) break;      \
    case 1: DO(256, 128, 4, 2, 3, 1) break;      \
    case 2: DO(192, 128, 2, 4, 4, 2) break;      \
    case 3: DO(128, 192, 2, 2, 2, 1) break;      \
    case 4: DO(128, 128, 2, 4, 5, 2) break;      \
    case 5: DO(128, 64, 4, 2, 6, 2) break;       \
    case 6: DO(64, 64, 2, 2, 5, 2) break;        \
    case 7: DO(64, 32, 2, 1, 6, 2) break;        \
    case 8: DO(128, 96, 4, 1, 5, 2) break;       \
    default: DO(96, 128, 1, 4, 5, 2) break;      \
  }
static long tiles_of(int i, int M, int N) {
  return (long)((M + g_shapes[i].bm - 1) / g_shapes[i].bm) * ((N + g_shapes[i].bn - 1) / g_shapes[i].bn);
}
static float tile_estimate(int i, int M, int N, int K) {
  const float r = (float)tiles_of(i, M, N) / g_units, steps = (float)((K + GT_BK - 1) / GT_BK), part = r - floorf(r);
  // The results' own way to memory, a million of them: tiles that are alone on their unit store while no product runs there. (The time that all
  // tiles have in common is left out.) It decides where outputs are many and steps few, us with / without: 3,000 rows of 2,816 x 1,024 26.0 / 30.6, 7,321 of
  // 9,088 x 704 109 / 118, 1,531 of 48,000 x 1,536 241 / 267, 3,492 of 15,104 x 384 59 / 64. Of the 132 products above 25 instead of 33 take more than 3 % longer than with
  // the fastest tile. (While results left as they lay, 617 products together took 0.933 of what they did with the first four tiles there were, 256 x 256, 128 x 192, 128 x 128, 64 x 64.)
  const float out = 1e-6f * (float)M * (float)N;
  switch (i) {
    case 0: return 5.0f + steps * (1.85f * floorf(r) + (part > 0.f ? fmaxf(1.5f, 1.5f + 1.2f * (part - 0.6f)) : 0.f));
    case 1: return 4.5f + 0.11f * out + steps * (r <= 0.75f ? 0.82f : r <= 1.f ? 1.05f : 0.55f + 0.95f * r);
    case 2: return 4.2f + 0.14f * out + steps * (r <= 0.75f ? 0.63f : r <= 1.f ? 0.77f : 0.45f + 0.72f * r);
    case 3: return 4.5f + steps * (r <= 1.f ? 1.1f : r <= 2.f ? fmaxf(1.42f, 0.79f * r) : fmaxf(2.3f, 0.78f * r));
    case 4: return 4.0f + 0.05f * out + steps * (r <= 1.f ? 0.53f : 0.2f + 0.6f * r);
    case 5: return 4.0f + steps * (r <= 0.75f ? 0.32f : r <= 1.f ? 0.37f : 0.03f + 0.36f * ceilf(r));
    case 6: return 3.4f + steps * (r <= 1.f ? 0.25f : r <= 1.25f ? 0.36f : 0.22f * ceilf(r));
    // (up to eight steps the wider tile: 448 x 512, 129 to 600 rows, 4.7 / 4.4)
    case 7: return 4.1f + steps * (r <= 1.f ? 0.17f : 0.29f * ceilf(0.5f * r));
    // (beyond one a unit: none)
    case 8: return 7.5f + steps * (r <= 0.9f ? 0.36f : r <= 1.f ? 0.42f : 1e3f);
    default: return 7.8f + steps * (r <= 1.f ? 0.44f : 1e3f);
  }
}

// The tile that a product takes, an index into g_shapes.
TIS_EXPORT int tis_gemm_tiles_pick(int M, int N, int K) {
  int pick = 0;
  float best = tile_estimate(0, M, N, K);
  for (int i = 1; i < GT_SHAPES; ++i) {
    const float t = tile_estimate(i, M, N, K);
    if (t < best) best = t, pick = i;
  }
  return pick;
}

// How many workgroups that tile makes of the product.
TIS_EXPORT int tis_gemm_tiles_count(int M, int N, int K) {
  const long n = tiles_of(tis_gemm_tiles_pick(M, N, K), M, N);
  return n < INT_MAX ? (int)n : INT_MAX;
}

// W: [N, K] contiguous. R: null, or the residual (bfloat16) added to the product; it may be C itself: an element is read by the wave that writes it, and a wave
// has read 32 rows of its own before it writes the first of them (through LDS another lane may write what one has read). out_f32: C holds 32-bit floats, the sums as they are (the output table's
// logits), and takes no residual. act: 1 the tanh form of gelu, 2 the square of relu, 3 clamped_swish of pairs of columns at
// `limit`, 4 silu(g) u of pairs of columns of the rounded product
// (3 and 4: C has N / 2 columns), the others applied to the 32-bit sums; a bfloat16 result without a residual.
// Sizes: K and x_ld multiples of 8, N, c_ld and r_ld multiples of 4; X and W 16-byte
// aligned, C and R 8-byte aligned (a 32-bit C 16-byte). Launches only: safe under stream capture.
TIS_EXPORT int tis_gemm_tiles(const void* X, long x_ld, const void* W, const void* R, long r_ld, void* C, long c_ld,
                              int M, int N, int K, int out_f32, int act, float limit, hipStream_t stream) {
  if (M < 0 || N < 0 || K < 1) return tis_fail("gemm_tiles: bad size M=%d N=%d K=%d", M, N, K);
  if (M == 0 || N == 0) return 0;
  if (K % 8 || x_ld % 8 || x_ld < K) return tis_fail("gemm_tiles: K=%d and the input's row stride %ld must be multiples of 8", K, x_ld);
  if (N % 4 || c_ld % (act >= 3 ? 2 : 4) || c_ld < (act >= 3 ? N / 2 : N) || (R && (r_ld % 4 || r_ld < N)))
    return tis_fail("gemm_tiles: N=%d and the row strides of the output (%ld) and residual (%ld) must be multiples of 4", N, c_ld, r_ld);
  if (((uintptr_t)X | (uintptr_t)W) % 16 || ((uintptr_t)C | (uintptr_t)R) % 8 || (out_f32 && (uintptr_t)C % 16))
    return tis_fail("gemm_tiles: inputs must be 16-byte aligned, output and residual 8-byte aligned (a 32-bit output 16-byte)");
  if (act == 3 && !(limit > 0.f)) return tis_fail("gemm_tiles: a clamp at %g", (double)limit);
  if (act < 0 || act > 4 || (act && (out_f32 || R))) return tis_fail("gemm_tiles: an activation (%d) goes with a plain bfloat16 result", act);
  if (out_f32 && R) return tis_fail("gemm_tiles: a 32-bit result takes no residual");
  if ((long)x_ld * 16 >= (1L << 31) || (long)K * 16 >= (1L << 31)) return tis_fail("gemm_tiles: rows of %ld elements are too long for 32-bit offsets", x_ld);
  const int pick = tis_gemm_tiles_pick(M, N, K);
  const long tiles = tiles_of(pick, M, N);
  if (tiles >= (1L << 31)) return tis_fail("gemm_tiles: %ld tiles are more than a grid holds", tiles);
  // whether the result's rows are whole pieces of 16 bytes
  const int piece = out_f32 ? 4 : 8;
  const bool wide = (uintptr_t)C % 16 == 0 && c_ld % piece == 0 && N % (act >= 3 ? 16 : piece) == 0;
#define LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, RV, TOV, ACTV)                                                               \
  gemm_tiles_kernel<BMV, BNV, WMV, WNV, NSV, AHV, RV, TOV, ACTV><<<dim3((unsigned)tiles), WMV * WNV * 64, 0, stream>>>(   \
      (const bf16*)X, x_ld, (const bf16*)W, (const bf16*)R, r_ld, (TOV*)C, c_ld, M, N, K, limit, wide)
#define PICK(BMV, BNV, WMV, WNV, NSV, AHV)                                     \
  {                                                                             \
    if (out_f32) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, float, 0);       \
    else if (R) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, true, bf16, 0);          \
    else if (act == 1) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, bf16, 1);  \
    else if (act == 2) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, bf16, 2);  \
    else if (act == 3) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, bf16, 3);  \
    else if (act == 4) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, bf16, 4);  \
    else LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, bf16, 0);                \
  }
  GT_EACH_TILE(pick, PICK)
#undef PICK
#undef LAUNCH
  return tis_launch_status("gemm_tiles");
}

// q_out = the queries of X . W^T, turned; keys and values into the cache (see gemm_tiles_rope_kernel). W: [(n_heads + 2 n_kv_heads) head_dim, K], the rows
// of query and key heads in pairs. write_slots and plane null: keys and values are not kept. Sizes: K, x_ld multiples of 8, head_dim of 32, q_ld of 4; X, W
// and the table 16-byte aligned, q_out and the plane 8-byte. Launches only: safe under stream capture.
TIS_EXPORT int tis_gemm_tiles_qkv_rope(const void* X, long x_ld, const void* W, void* q_out, long q_ld, int M, int K, const int* positions,
                                       const int* write_slots, const float* table, void* plane, int n_heads, int n_kv_heads, int head_dim,
                                       int page_size, hipStream_t stream) {
  if (M < 0 || K < 1 || n_heads < 1 || n_kv_heads < 1 || head_dim < 32 || head_dim % 32 || page_size < 1 || (long)(n_heads + 2L * n_kv_heads) * head_dim >= (1L << 31))
    return tis_fail("gemm_tiles_qkv_rope: bad size M=%d K=%d heads=%d kv_heads=%d head_dim=%d page=%d", M, K, n_heads, n_kv_heads, head_dim, page_size);
  if (M == 0) return 0;
  const int N = (n_heads + 2 * n_kv_heads) * head_dim;
  if (K % 8 || x_ld % 8 || x_ld < K || q_ld % 4 || q_ld < (long)n_heads * head_dim)
    return tis_fail("gemm_tiles_qkv_rope: K=%d and the row strides %ld, %ld must be multiples of 8, 8 and 4", K, x_ld, q_ld);
  if (((uintptr_t)X | (uintptr_t)W | (uintptr_t)table) % 16 || ((uintptr_t)q_out | (uintptr_t)plane) % 8 || !positions || !table || !write_slots != !plane)
    return tis_fail("gemm_tiles_qkv_rope: inputs and table must be 16-byte aligned, queries and cache 8-byte, and slots go with a cache");
  if ((long)x_ld * 16 >= (1L << 31) || (long)K * 16 >= (1L << 31)) return tis_fail("gemm_tiles: rows of %ld elements are too long for 32-bit offsets", x_ld);
  const int pick = tis_gemm_tiles_pick(M, N, K);
  const long tiles = tiles_of(pick, M, N);
  if (tiles >= (1L << 31)) return tis_fail("gemm_tiles: %ld tiles are more than a grid holds", tiles);
  const RopeOut a{positions, write_slots, (const float2*)table, (bf16*)plane, n_heads, n_kv_heads, head_dim, page_size};
#define ROPE(BMV, BNV, WMV, WNV, NSV, AHV)                                                                                   \
  gemm_tiles_rope_kernel<BMV, BNV, WMV, WNV, NSV, AHV><<<dim3((unsigned)tiles), WMV * WNV * 64, 0, stream>>>((const bf16*)X, x_ld, (const bf16*)W, (bf16*)q_out, q_ld, M, N, K, a);
  GT_EACH_TILE(pick, ROPE)
#undef ROPE
  return tis_launch_status("gemm_tiles_qkv_rope");
}
