// C[M,N] = X[M,K] . W[N,K]^T (+ R[M,N]) in bfloat16 for many rows at widths where the library's product is not used:
// a product tiled in both directions on v_mfma_f32_32x32x16_bf16 (gfx950), operands through LDS by direct loads.
// (The few-row kernel takes such a product in panels of 32 rows, each of which streams all of W again: 0.25 to 0.3
// PFLOP/s at 2,048 rows. This kernel reaches 0.45 to 0.95 on the same shapes; the library's kernels, where they may be
// used, 0.5 to 1.3.) The reference's engine uses a library product here (x @ W, main_models_new.py:19-20).
//
// A workgroup owns a tile of BM rows x BN columns and walks K in steps of 64. A step's
// operand rows, 128 bytes each, are copied into LDS by global_load_lds_dwordx4 (no registers; eight lanes read one
// row's 128 bytes) into a ring of NSTAGE buffers, one to three steps ahead of the products. A row's eight 16-byte pieces lie in LDS with their index XORed by half the row's number:
// an operand fetch reads one piece index of 32 rows, LDS serves sixteen lanes at a time, and sixteen rows of 128
// bytes are eight such indices at each of two offsets in the 256 bytes that the banks span, so no two of them meet
// (XORed by the row's number itself, rows r and r + 8 did: half of the LDS's busy cycles were bank conflicts). The
// copying lane picks the piece that belongs in its slot. The result tile is computed transposed (W's rows are the first operand), so that a
// lane ends up with four consecutive columns of one row: 8-byte stores, and the residual read the same way.
// A row's sums run over K in the same order whatever M is: its result does not depend on the other rows.
//
// What bounds it: the clock under load (8,192 cubed runs at 1.42 PFLOP/s here: 1.5 us for a step of a 256 x 256 tile on every
// compute unit), for tiles of 64 x 64 and 128 x 128 the LDS, whose reads and writes take 1.5 to 2 times the products' cycles, and for
// products of one tile a unit the beginning and end (4 us, and 16 or 32 MB of results at 5 TB/s). Operands are fetched from LDS one
// or two 16-wide slices ahead of their products (a wave alone on its SIMD waits 230 cycles for four fetches that all waves issue at
// once, and its products take 128), and a slice's instructions keep a pinned order. Before that (operands fetched where they are
// used, one step ahead into two buffers) and now, us: 2,048 rows x 2,048 x 2,048 28.0 / 22.7; inner 5,632 62.9 / 48.0; 2,048 x 5,632
// x 2,048 54.0 / 49.6; 1,800 x 32,000 x 2,048 271 / 247; 1,531 x 2,048 x 2,048 24.1 / 18.2; 300 x 1,024 x 1,024 12.1 / 6.8; 8
// columns 14.9 / 7.9.
#include "common.h"

TIS_DEFINE_LAST_ERROR(tis_gemm_tiles)

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;

static constexpr int GT_BK = 64, GT_PIECES = GT_BK / 8;

// what lanes past the end of K read in the last step: zeros
static __device__ __attribute__((aligned(16))) unsigned char gt_zeros[16];

#pragma clang diagnostic ignored "-Winline-asm"   // M0 in a clobber list: meant
// One 16-byte piece per lane from global memory straight into LDS: lane i's piece lands at lds_addr + 16 * i. In
// assembly, because the compiler would order every later LDS read behind such a load, whichever buffer it reads; so
// the compiler does not count these loads either, and whoever reads the pieces waits for them (vmcnt) and for the
// other waves (barrier).
__device__ __forceinline__ void gt_copy16(const void* scalar_src, unsigned lane_bytes, unsigned lds_addr) {
  const uint64_t a = (uint64_t)scalar_src;
  const uint64_t sc = ((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32) |
                      (unsigned)__builtin_amdgcn_readfirstlane((int)a);
  const unsigned base = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_addr);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(lane_bytes), "s"(sc), "s"(base) : "memory", "m0");
}
// the same with every lane's own address
__device__ __forceinline__ void gt_copy16(const void* lane_src, unsigned lds_addr) {
  const unsigned base = (unsigned)__builtin_amdgcn_readfirstlane((int)lds_addr);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(lane_src), "s"(base) : "memory", "m0");
}

// BM x BN: the workgroup's tile; WM x WN: its waves, each with (BM / WM) x (BN / WN) of it
// ACT: what becomes of a sum before it is rounded (0 nothing; 1 the tanh form of gelu, 0.5 z (1 + tanh(u)) written as
// z / (1 + exp(-2u)); 2 the square of relu; 3 clamped_swish of the columns' pairs (2j, 2j + 1): C has N / 2 columns)
template <int ACT> __device__ __forceinline__ float gt_activated(float z) {
  if (ACT == 1) return z / (1.f + __expf(-1.5957691216057308f * (z + 0.044715f * z * z * z)));
  if (ACT == 2) { const float p = fmaxf(z, 0.f); return p * p; }
  return z;
}

template <int V> struct IntC { constexpr operator int() const { return V; } };

// Which tile a workgroup takes. Workgroups go to the eight XCDs in turn, each with an L2 of its own: an XCD gets a run of
// neighbouring tiles, in an order that walks four rows of tiles side by side, so that what its workgroups read at a time
// is few rows of X and of W.
struct GtTile { int m, n; };
__device__ __forceinline__ GtTile gt_tile(unsigned id, int tiles_m, int tiles_n) {
  const unsigned total = (unsigned)tiles_m * (unsigned)tiles_n, xcd = id % 8, per = total / 8, more = total % 8;
  const unsigned t = xcd * per + min(xcd, more) + id / 8;
  const unsigned band = 4u * (unsigned)tiles_n, g = t / band, in = t - g * band;
  const unsigned rows = min(4u, (unsigned)tiles_m - g * 4);
  return {(int)(g * 4 + in % rows), (int)(in / rows)};
}

// NSTAGE: buffers of LDS; AHEAD: slices of 16 of K that operands are fetched from LDS before their products
template <int BM, int BN, int WM, int WN, int NSTAGE, int AHEAD, bool RESIDUAL, typename TO, int ACT = 0>
__global__ __launch_bounds__(WM * WN * 64) void gemm_tiles_kernel(
    const bf16* __restrict__ X, long x_ld, const bf16* __restrict__ W, const bf16* R, long r_ld, TO* C, long c_ld,
    int M, int N, int K, float limit) {
  constexpr int BK = GT_BK, PCS = GT_PIECES, ROWS = BM + BN, GT_WAVES = WM * WN, KS = BK / 16;
  constexpr int STAGE = ROWS * BK * 2;                  // bytes of a buffer: X's rows, then W's
  constexpr int LPW = ROWS * PCS / 64 / GT_WAVES;       // loads of a step that each wave issues, 8 rows each
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;   // 32 x 32 result tiles of a wave
  static_assert(ROWS * PCS % (64 * GT_WAVES) == 0 && TM >= 1 && TN >= 1 && NSTAGE * STAGE <= 160 * 1024, "tile sizes");
  constexpr int FLIGHT = AHEAD == 1 ? NSTAGE : NSTAGE - 1;   // steps that are copied ahead
  constexpr int SETS = AHEAD == 1 ? 2 : KS;             // operand registers: a set a slice, in turn
  static_assert((AHEAD == 1 || AHEAD == 2) && FLIGHT >= 2 && FLIGHT <= 3 && KS == 4, "what the loop below is written for");
  static_assert((FLIGHT - 1) * LPW <= 63, "more loads in flight than the counter counts");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[NSTAGE * STAGE];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r32 = lane & 31, h = lane >> 5;
  const int wm = wave / WN, wn = wave % WN;
  const GtTile tile = gt_tile(blockIdx.x, (M + BM - 1) / BM, (N + BN - 1) / BN);
  const long m0 = (long)tile.m * BM, n0 = (long)tile.n * BN;
  const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)lds;

  // The wave's loads of a step: load j brings rows 8 (wave * LPW + j) .. +7 of the buffer, lane (row, slot) the piece
  // slot ^ ((row >> 1) & 7) of its row. Rows past the matrix's last are the last row again (their results are not
  // stored).
  const unsigned char* first_row[LPW];       // of the load's first row, at K offset 0 (the same on all lanes)
  unsigned lane_off[LPW];                    // the lane's piece from there, in bytes
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int row0 = (wave * LPW + j) * 8, row = row0 + (lane >> 3);
    const bool of_x = row0 < BM;
    const long ld = of_x ? x_ld : (long)K;
    const long last = of_x ? (long)M - 1 : (long)N - 1;
    const long g_first = min(last, of_x ? m0 + row0 : n0 + (row0 - BM));
    const long g_row = min(last, of_x ? m0 + row : n0 + (row - BM));
    first_row[j] = (const unsigned char*)(of_x ? X : W) + g_first * ld * 2;
    lane_off[j] = (unsigned)((g_row - g_first) * ld * 2 + ((lane & 7) ^ ((row >> 1) & 7)) * 16);
  }
  const int nk = (K + BK - 1) / BK;
  const bool ragged = K % BK != 0;                      // the last step's pieces past the end of K come from a block of zeros
  auto load = [&](int kt, unsigned at, int j) {         // at: where the buffer begins
    gt_copy16(first_row[j] + (long)kt * (BK * 2), lane_off[j], at + (wave * LPW + j) * 1024);
  };
  auto load_ragged = [&](int kt, unsigned at, int j) {
    const int row = (wave * LPW + j) * 8 + (lane >> 3);
    const bool inside = kt * BK + ((lane & 7) ^ ((row >> 1) & 7)) * 8 < K;
    gt_copy16(inside ? first_row[j] + (long)kt * (BK * 2) + lane_off[j] : gt_zeros, at + (wave * LPW + j) * 1024);
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // operand pieces: row r of the buffer, elements 16 ks + 8 h .. of the step, lie at r * 128 + ((2 ks + h) ^ ((r >> 1) & 7)) * 16:
  // 32 rows on, the same piece; two pieces on (the next ks), the address with bits 5 and 6 changed
  const unsigned a_row = wm * (BM / WM) + r32, b_row = BM + wn * (BN / WN) + r32;
  const unsigned a_at = a_row * 128 + ((h ^ ((a_row >> 1) & 7)) * 16), b_at = b_row * 128 + ((h ^ ((b_row >> 1) & 7)) * 16);
  bf16x8 a[SETS][TM], b[SETS][TN];
  auto fetch = [&](int ks, unsigned at) {               // at: where the buffer begins, from the first
#pragma unroll
    for (int i = 0; i < TM; ++i) a[ks % SETS][i] = *(const bf16x8*)(lds + (at + (a_at ^ (ks * 32)) + i * 4096));
#pragma unroll
    for (int j = 0; j < TN; ++j) b[ks % SETS][j] = *(const bf16x8*)(lds + (at + (b_at ^ (ks * 32)) + j * 4096));
  };

  // The loop. While a slice's products run, the operands of the slice AHEAD of it are on their way out of LDS, also across
  // steps: AHEAD slices before its end, step kt waits until step kt + 1 is in LDS for every wave (the barrier) and fetches from there.
  // After that barrier a buffer is free for copies: with AHEAD 2 step kt - 1's, whose last operands every wave has used; with
  // AHEAD 1 step kt's own, whose last operands every wave has in registers, because it waited for them too. Each gives FLIGHT
  // steps that are under way. The order of a slice's instructions is pinned: the first product, the LDS reads, the other products with
  // the copies between them, so that a wave that has its SIMD to itself keeps the matrix core busy while it issues them.
  // MODE 0: copies a whole step; 1: the ragged last one; 2: none. LEFT: the steps beyond the next that are under way meanwhile.
  unsigned at = 0, prev = (NSTAGE - 1) * STAGE;
  auto step = [&](int kt, auto mode, auto left, auto last) {
    constexpr int MODE = mode, LEFT = left;
    constexpr bool LAST = last;
    const unsigned next = at + STAGE == NSTAGE * STAGE ? 0 : at + STAGE;
    const unsigned into = lds0 + (AHEAD == 1 ? at : prev);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks == KS - AHEAD && !LAST) {
        if (AHEAD == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(LEFT * LPW) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(LEFT * LPW) : "memory");
      }
#pragma unroll
      for (int m = 0; m < TM * TN; ++m) {
        acc[m / TN][m % TN] =
            __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[ks % SETS][m % TN], a[ks % SETS][m / TN], acc[m / TN][m % TN], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (m == 0) {
          if (ks + AHEAD < KS) fetch(ks + AHEAD, at);
          else if (!LAST) fetch(ks + AHEAD - KS, next);
        }
        if (MODE < 2 && ks >= KS - AHEAD) {
          constexpr int SLOTS = AHEAD * TM * TN;
          const int slot = (ks - (KS - AHEAD)) * TM * TN + m;
#pragma unroll
          for (int j = slot * LPW / SLOTS; j < (slot + 1) * LPW / SLOTS; ++j) {
            if (MODE == 0) load(kt + FLIGHT, into, j);
            else load_ragged(kt + FLIGHT, into, j);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    prev = at;
    at = next;
  };
  const int whole = ragged ? nk - 1 : nk;
#pragma unroll
  for (int s = 0; s < FLIGHT; ++s) {
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
      if (s < whole) load(s, lds0 + s * STAGE, j);
      else if (s < nk) load_ragged(s, lds0 + s * STAGE, j);
    }
  }
  if (nk >= FLIGHT) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((FLIGHT - 1) * LPW) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" : : : "memory");
#pragma unroll
  for (int ks = 0; ks < AHEAD; ++ks) fetch(ks, 0);
  int kt = 0;
  for (; kt + FLIGHT < whole; ++kt) step(kt, IntC<0>{}, IntC<FLIGHT - 2>{}, IntC<0>{});
  if (kt + FLIGHT < nk) {
    step(kt, IntC<1>{}, IntC<FLIGHT - 2>{}, IntC<0>{});
    ++kt;
  }
  // the last steps, whose copies are all under way
  if constexpr (FLIGHT == 3)
    if (nk >= 3) step(kt++, IntC<2>{}, IntC<1>{}, IntC<0>{});
  if (nk >= 2) step(kt++, IntC<2>{}, IntC<0>{}, IntC<0>{});
  step(kt, IntC<2>{}, IntC<0>{}, IntC<1>{});

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
  //   128 x 192, four waves, two buffers     0.79 up to one a unit, two share one: 0.79 for each on average
  //   128 x 128, eight waves, four buffers   0.47, and 0.6 a further round
  //   64 x 64, four waves, four buffers      0.21 up to one a unit, two share one: 0.21 for each on average
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
    else t = (i == 1 ? 0.79f : 0.21f) * fmaxf(r, 1.f);
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
