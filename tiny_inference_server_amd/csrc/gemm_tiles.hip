// C[M,N] = X[M,K] . W[N,K]^T (+ R[M,N]) in bfloat16 for many rows at widths where the library's product is not used:
// a product tiled in both directions on v_mfma_f32_32x32x16_bf16 (gfx950), operands through LDS by direct loads.
// (The few-row kernel takes such a product in panels of 32 rows, each of which streams all of W again: 0.25 to 0.3
// PFLOP/s at 2,048 rows. This kernel reaches 0.75 to 1.0 on the same shapes; the library's kernels, where they may be
// used, 0.5 to 1.3.) The reference's engine uses a library product here (x @ W, main_models_new.py:19-20).
//
// tile_loop.h holds the loop. A row's sums run over K in the same order whatever M is: its result does not depend on the other rows.
// With operands fetched where they are used and copies one step ahead (before) and as the loop is now, us: 2,048 rows x 2,048 x 2,048
// 28.0 / 22.7; inner 5,632 62.9 / 48.0; 2,048 x 5,632 x 2,048 54.0 / 49.6; 1,800 x 32,000 x 2,048 271 / 247; 1,531 x 2,048 x 2,048
// 24.1 / 18.2; 300 x 1,024 x 1,024 12.1 / 6.8; 8 columns 14.9 / 7.9.
#include "tile_loop.h"

TIS_DEFINE_LAST_ERROR(tis_gemm_tiles)

// BM x BN: the workgroup's tile; WM x WN: its waves, each with (BM / WM) x (BN / WN) of it
// ACT: what becomes of a sum before it is rounded (0 nothing; 1 the tanh form of gelu, 0.5 z (1 + tanh(u)) written as
// z / (1 + exp(-2u)); 2 the square of relu; 3 clamped_swish of the columns' pairs (2j, 2j + 1): C has N / 2 columns)
template <int ACT> __device__ __forceinline__ float gt_activated(float z) {
  if (ACT == 1) return z / (1.f + __expf(-1.5957691216057308f * (z + 0.044715f * z * z * z)));
  if (ACT == 2) { const float p = fmaxf(z, 0.f); return p * p; }
  return z;
}

template <int BM, int BN, int WM, int WN, int NSTAGE, int AHEAD, bool RESIDUAL, typename TO, int ACT = 0>
__global__ __launch_bounds__(WM * WN * 64) void gemm_tiles_kernel(
    const bf16* __restrict__ X, long x_ld, const bf16* __restrict__ W, const bf16* R, long r_ld, TO* C, long c_ld,
    int M, int N, int K, float limit) {
  typedef TileLoop<BM, BN, WM, WN, NSTAGE, AHEAD> Loop;
  constexpr int LPW = Loop::LPW, TM = Loop::TM, TN = Loop::TN;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[NSTAGE * Loop::STAGE];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r32 = lane & 31, h = lane >> 5;
  const int wm = wave / WN, wn = wave % WN;
  const GtTile tile = gt_tile(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN);
  const long m0 = (long)tile.m * BM, n0 = (long)tile.n * BN;

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
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  Loop::run(lds, first, lane_off, K, acc);

  // accumulator 4 q + e of block (i, j): row m0 + wm * (BM / WM) + i * 32 + r32, column n0 + wn * (BN / WN) + j * 32 + 8 q + 4 h + e
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const long m = m0 + wm * (BM / WM) + i * 32 + r32;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const long n = n0 + wn * (BN / WN) + j * 32 + q * 8 + h * 4;
        if (n >= N) continue;                 // (N is a multiple of 4: the four columns are inside or outside together)
        if constexpr (ACT == 3) {
          typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
          *(bf16x2*)(C + m * c_ld + n / 2) =
              (bf16x2){static_cast<__bf16>(clamped_swish(acc[i][j][q * 4], acc[i][j][q * 4 + 1], limit)),
                       static_cast<__bf16>(clamped_swish(acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3], limit))};
          continue;
        }
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gt_activated<ACT>(acc[i][j][q * 4 + e]);
        if (RESIDUAL) {
          const bf16x4 r = *(const bf16x4*)(R + m * r_ld + n);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += (float)r[e];
        }
        if constexpr (sizeof(TO) == 4) {
          *(f32x4*)(C + m * c_ld + n) = (f32x4){v[0], v[1], v[2], v[3]};       // the 32-bit sums as they are
        } else {
          bf16x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = static_cast<__bf16>(v[e]);
          *(bf16x4*)(C + m * c_ld + n) = o;
        }
      }
  }
}

static int g_units = 256;      // compute units of the device: set by whoever knows (the default is an MI355X)
TIS_EXPORT void tis_gemm_tiles_units(int n) { if (n > 0) g_units = n; }

// W: [N, K] contiguous. R: null, or the residual (bfloat16) added to the product; it may be C itself (every element is
// read and then written by the same lane). out_f32: C holds 32-bit floats, the sums as they are (the output table's
// logits), and takes no residual. act: 1 the tanh form of gelu, 2 the square of relu, 3 clamped_swish of pairs of columns at
// `limit` (C has N / 2 columns), applied to the 32-bit sums of a bfloat16 result without a residual. Sizes: K and x_ld multiples of 8, N, c_ld and r_ld multiples of 4; X and W 16-byte
// aligned, C and R 8-byte aligned (a 32-bit C 16-byte). Launches only: safe under stream capture.
TIS_EXPORT int tis_gemm_tiles(const void* X, long x_ld, const void* W, const void* R, long r_ld, void* C, long c_ld,
                              int M, int N, int K, int out_f32, int act, float limit, hipStream_t stream) {
  if (M < 0 || N < 0 || K < 1) return tis_fail("gemm_tiles: bad size M=%d N=%d K=%d", M, N, K);
  if (M == 0 || N == 0) return 0;
  if (K % 8 || x_ld % 8 || x_ld < K) return tis_fail("gemm_tiles: K=%d and the input's row stride %ld must be multiples of 8", K, x_ld);
  if (N % 4 || c_ld % (act == 3 ? 2 : 4) || c_ld < (act == 3 ? N / 2 : N) || (R && (r_ld % 4 || r_ld < N)))
    return tis_fail("gemm_tiles: N=%d and the row strides of the output (%ld) and residual (%ld) must be multiples of 4", N, c_ld, r_ld);
  if (((uintptr_t)X | (uintptr_t)W) % 16 || ((uintptr_t)C | (uintptr_t)R) % 8 || (out_f32 && (uintptr_t)C % 16))
    return tis_fail("gemm_tiles: inputs must be 16-byte aligned, output and residual 8-byte aligned (a 32-bit output 16-byte)");
  if (act == 3 && !(limit > 0.f)) return tis_fail("gemm_tiles: a clamp at %g", (double)limit);
  if (act < 0 || act > 3 || (act && (out_f32 || R))) return tis_fail("gemm_tiles: an activation (%d) goes with a plain bfloat16 result", act);
  if (out_f32 && R) return tis_fail("gemm_tiles: a 32-bit result takes no residual");
  if ((long)x_ld * 16 >= (1L << 31) || (long)K * 16 >= (1L << 31)) return tis_fail("gemm_tiles: rows of %ld elements are too long for 32-bit offsets", x_ld);
  // The tile: the one that is estimated to end first, by the microseconds a step of 64 takes with one or more workgroups a
  // compute unit (measured at K of 1,408 to 5,632; the clock falls as more of the chip works, hence 1.36 to 1.85 for the largest):
  //   256 x 256, eight waves, two buffers    1.36 up to 0.7 workgroups a unit, then to 1.72 at one; 1.85 a full round
  //   128 x 192, four waves, two buffers     0.79 up to one a unit; two share one: from 1.25 on, 0.79 for each on average
  //   128 x 128, eight waves, four buffers   0.47, and 0.6 a further round
  //   64 x 64, four waves, four buffers      0.21 up to one a unit; two share one: from 0.42 on, 0.21 for each on average
  // (us, 256 / 192 / 128 / 64, 2,048 inner columns: 2,048 x 2,048 48.4, 31.4, 22.7, 30.5; 2,048 x 2,816 47.0, 31.3, 33.0, 39.2;
  // 2,048 x 5,120 49.0, 48.6, 51.9, 66.5; 1,800 x 8,192 62.8, 71.3, 70.8, 98.2; 1,536 x 11,264 102.9, 75.1, 84.9, 110.0;
  // 1,800 x 32,000 247, 280, 333, 420; 700 x 1,024 x 2,816 59.4, 37.4, 20.6, 13.8.)
  struct { int bm, bn; } const shapes[4] = {{256, 256}, {128, 192}, {128, 128}, {64, 64}};
  int pick = 0;
  float best = 0.f;
  long tiles = 0;
  for (int i = 0; i < 4; ++i) {
    const long n = (long)((M + shapes[i].bm - 1) / shapes[i].bm) * ((N + shapes[i].bn - 1) / shapes[i].bn);
    const float r = (float)n / g_units, full = floorf(r), part = r - full;
    float t;
    if (i == 0) t = 1.85f * full + (part > 0.f ? fmaxf(1.36f, 1.36f + 1.2f * (part - 0.7f)) : 0.f);
    else if (i == 2) t = 0.47f + 0.6f * (ceilf(r) - 1.f);
    else if (i == 1) t = r <= 1.f ? 0.79f : fmaxf(1.25f, 0.79f * r);
    else t = r <= 1.f ? 0.21f : fmaxf(0.42f, 0.21f * r);
    if (i == 0 || t < best) best = t, pick = i, tiles = n;
  }
  if (tiles >= (1L << 31)) return tis_fail("gemm_tiles: %ld tiles are more than a grid holds", tiles);
#define LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, RV, TOV, ACTV)                                                     \
  gemm_tiles_kernel<BMV, BNV, WMV, WNV, NSV, AHV, RV, TOV, ACTV><<<dim3((unsigned)tiles), WMV * WNV * 64, 0, stream>>>(    \
      (const bf16*)X, x_ld, (const bf16*)W, (const bf16*)R, r_ld, (TOV*)C, c_ld, M, N, K, limit)
#define PICK(BMV, BNV, WMV, WNV, NSV, AHV)                                     \
  {                                                                             \
    if (out_f32) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, float, 0);   \
    else if (R) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, true, bf16, 0);      \
    else if (act == 1) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, bf16, 1); \
    else if (act == 2) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, bf16, 2); \
    else if (act == 3) LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, bf16, 3); \
    else LAUNCH(BMV, BNV, WMV, WNV, NSV, AHV, false, bf16, 0);            \
  }
  if (pick == 0) PICK(256, 256, 2, 4, 2, 1)
  else if (pick == 1) PICK(128, 192, 2, 2, 2, 1)
  else if (pick == 2) PICK(128, 128, 2, 4, 4, 2)
  else PICK(64, 64, 2, 2, 4, 2)
#undef PICK
#undef LAUNCH
  return tis_launch_status("gemm_tiles");
}
