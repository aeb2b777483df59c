// The loop of the products tiled in both directions (gemm_tiles.hip, experts.hip): operands through LDS by direct loads, products on
// v_mfma_f32_32x32x16_bf16.
//
// A workgroup owns a tile of BM rows of X x BN rows of W and walks K in steps of 64. A step's
// operand rows, 128 bytes each, are copied into LDS by global_load_lds_dwordx4 (no registers; eight lanes read one
// row's 128 bytes) into a ring of NSTAGE buffers, two to five steps ahead of the products. A row's eight 16-byte pieces lie in LDS with their index XORed by half the row's number:
// an operand fetch reads one piece index of 32 rows, LDS serves sixteen lanes at a time, and sixteen rows of 128
// bytes are eight such indices at each of two offsets in the 256 bytes that the banks span, so no two of them meet
// (XORed by the row's number itself, rows r and r + 8 did: half of the LDS's busy cycles were bank conflicts). The
// copying lane picks the piece that belongs in its slot. The result tile is computed transposed (W's rows are the first operand), so that a
// lane ends up with four consecutive columns of one row; how they leave is the kernels' business.
// A row's sums run over K in the same order whatever M is: its result does not depend on the other rows.
//
// What bounds it: the clock under load (8,192 cubed runs at 1.42 PFLOP/s here: 1.5 us for a step of a 256 x 256 tile on every
// compute unit), for tiles of 64 x 64 and 128 x 128 the LDS, whose reads and writes take 1.5 to 2 times the products' cycles, and for
// products of one tile a unit the beginning and end (4 us, and 16 or 32 MB of results at 5 TB/s). Operands are fetched from LDS one
// or two 16-wide slices ahead of their products (a wave alone on its SIMD waits 230 cycles for four fetches that all waves issue at
// once, and its products take 128), and a slice's instructions keep a pinned order.
#pragma once
#include "common.h"

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

// WM x WN: the workgroup's waves, each with (BM / WM) x (BN / WN) of the tile; NSTAGE: buffers of LDS; AHEAD: slices of 16 of K that
// operands are fetched from LDS before their products
template <int BM, int BN, int WM, int WN, int NSTAGE, int AHEAD>
struct TileLoop {
  static constexpr int BK = GT_BK, PCS = GT_PIECES, ROWS = BM + BN, WAVES = WM * WN, KS = BK / 16;
  static constexpr int STAGE = ROWS * BK * 2;                  // bytes of a buffer: X's rows, then W's
  static constexpr int LPW = ROWS * PCS / 64 / WAVES;          // loads of a step that each wave issues, 8 rows each
  static constexpr int TM = BM / WM / 32, TN = BN / WN / 32;   // 32 x 32 result tiles of a wave
  static constexpr int FLIGHT = AHEAD == 1 ? NSTAGE : NSTAGE - 1;   // steps that are copied ahead
  static constexpr int SETS = AHEAD == 1 ? 2 : KS;             // operand registers: a set a slice, in turn
  static_assert(ROWS * PCS % (64 * WAVES) == 0 && TM >= 1 && TN >= 1 && NSTAGE * STAGE <= 160 * 1024, "tile sizes");
  static_assert((AHEAD == 1 || AHEAD == 2) && FLIGHT >= 2 && KS == 4, "what the loop below is written for");
  static_assert((FLIGHT - 1) * LPW <= 63, "more loads in flight than the counter counts");

  // the row of the buffer that a lane's piece of load j belongs to, and which of the row's pieces it is
  static __device__ __forceinline__ int row_of(int wave, int lane, int j) { return (wave * LPW + j) * 8 + (lane >> 3); }
  static __device__ __forceinline__ int piece_of(int lane, int row) { return (lane & 7) ^ ((row >> 1) & 7); }

  // acc += the tile's products over the whole of K. first[j] (the same on all lanes) + lane_off[j]: the lane's piece of load j, at K
  // offset 0, its piece's own 16 bytes included.
  static __device__ __forceinline__ void run(unsigned char* lds, const unsigned char* const (&first)[LPW],
                                             const unsigned (&lane_off)[LPW], int K, f32x16 (&acc)[TM][TN]) {
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r32 = lane & 31, h = lane >> 5;
    const int wm = wave / WN, wn = wave % WN;
    const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)lds;
    const int nk = (K + BK - 1) / BK;
    const bool ragged = K % BK != 0;                      // the last step's pieces past the end of K come from a block of zeros
    auto load = [&](int kt, unsigned at, int j) {         // at: where the buffer begins
      gt_copy16(first[j] + (long)kt * (BK * 2), lane_off[j], at + (wave * LPW + j) * 1024);
    };
    auto load_ragged = [&](int kt, unsigned at, int j) {
      const bool inside = kt * BK + piece_of(lane, row_of(wave, lane, j)) * 8 < K;
      gt_copy16(inside ? first[j] + (long)kt * (BK * 2) + lane_off[j] : gt_zeros, at + (wave * LPW + j) * 1024);
    };

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
    // the last steps, whose copies are all under way: while `remain` are left, remain - 2 beyond the next
    auto last_steps = [&](auto self, auto remain) {
      constexpr int REMAIN = remain;
      if (nk >= REMAIN) step(kt++, IntC<2>{}, IntC<REMAIN - 2>{}, IntC<0>{});
      if constexpr (REMAIN > 2) self(self, IntC<REMAIN - 1>{});
    };
    last_steps(last_steps, IntC<FLIGHT>{});
    step(kt, IntC<2>{}, IntC<0>{}, IntC<1>{});
  }
};
