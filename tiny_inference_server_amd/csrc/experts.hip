// Routed feed-forwards (mixtures of experts) and other products that come in groups: the router's choice, the lists of
// rows per expert, a grouped product C_g = act(A_g . W_g^T), and the weighted sum of a row's chosen experts.
//
// Router: s = softmax(z) over all of a row's router outputs in 32-bit; the `top` outputs with the largest s + correction
// are chosen (the lower index wins a tie); a chosen output's weight is s * scale, taken without the correction and not
// renormalised. (score kinds: 0 this softmax; 1 a sigmoid per output; 2 the largest z + correction are chosen and their weights
// are the softmax over the chosen z alone.) Outputs from n_experts on are identity experts: they have no matrices, their result is the row itself.
//
// An assignment is a (row, k-th choice) pair, numbered row * top + k. The lists kernel gives every expert the
// assignments that chose it, in rising order, in a line of `rows` entries of its own (an expert is chosen at most once
// a row), so nothing needs a prefix sum or an atomic and the order never depends on timing.
//
// The grouped product walks, for group g, tiles of 16 list entries against tiles of 64 output columns of the group's
// matrix W[g] ([N][K]). Entry e's input row is A + (e / a_div) * lda + g * a_group, its output row C + e * ldc +
// g * c_group: with a_div = top the input rows are the step's rows and the outputs lie by assignment (an expert's first
// product), with a_div = 1 both lie by assignment (its second); without lists every group takes all rows, and a_group /
// c_group move from one group's columns to the next (a product per head on a head's own columns). Sums are 32-bit in
// an order that depends on K and on the kernel: the products straight from memory add steps of 32, in one chain or in four (tis_grouped_split), the tiles steps of 16.
// Within one of them a row's result does not depend on what else is in the step; which of them a step takes hangs on its entries (tis_grouped_tile), and a
// row's last bits may differ from one to the other.
#include "tile_loop.h"

TIS_DEFINE_LAST_ERROR(tis_experts)

static constexpr int EX_MAX_PER_LANE = 16;      // router outputs a lane keeps: up to 1,024 outputs a row

__device__ __forceinline__ float gelu_erf_f(float z) { return 0.5f * z * (1.f + erff(z * 0.7071067811865476f)); }

// one wave per row; PER: router outputs a lane keeps
template <int PER>
__global__ __launch_bounds__(TIS_WAVE) void route_topk_kernel(const float* __restrict__ z, long ldz,
                                                              const float* __restrict__ correction, float scale,
                                                              int n_out, int top, int score, int* __restrict__ ids,
                                                              float* __restrict__ weights, int n_groups, int keep,
                                                              int renorm) {
  const long r = blockIdx.x;
  const int lane = threadIdx.x;
  float s[PER], c[PER];
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = lane + u * TIS_WAVE;
    s[u] = e < n_out ? z[r * ldz + e] : -INFINITY;
    m = fmaxf(m, s[u]);
  }
  m = wave_max(m);
  float sum = 0.f;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = lane + u * TIS_WAVE;
    const float zu = s[u];
    if (score == 1) s[u] = e < n_out ? 1.f / (1.f + expf(-s[u])) : 0.f;      // a sigmoid per output, no sum over them
    else s[u] = e < n_out ? expf(s[u] - m) : 0.f;
    sum += s[u];
    c[u] = zu;
  }
  sum = wave_sum(sum);
  const float inv = score == 0 ? 1.f / sum : 1.f;
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = lane + u * TIS_WAVE;
    s[u] *= inv;
    c[u] = e < n_out ? (score == 2 ? c[u] : s[u]) + (correction ? correction[e] : 0.f) : -INFINITY;
  }
  if (n_groups > 1 && keep < n_groups) {
    // The outputs form n_groups equal runs of neighbours; a group's score is its largest c. Only outputs of the `keep`
    // best groups (the lower group keeps a tie) stay in the choice; the others' c become -inf. Up to 64 groups: lane g
    // holds group g's score.
    const int per = n_out / n_groups;
    float gs = -INFINITY;
    for (int g = 0; g < n_groups; ++g) {
      float m = -INFINITY;
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int e = lane + u * TIS_WAVE;
        if (e < n_out && e / per == g) m = fmaxf(m, c[u]);
      }
      m = wave_max(m);
      if (lane == g) gs = m;
    }
    // a group's rank: how many groups beat it
    int rank = 0;
    for (int g = 0; g < n_groups; ++g) {
      const float og = __shfl(gs, g, TIS_WAVE);
      if (og > gs || (og == gs && g < lane)) ++rank;
    }
    const unsigned long long kept = __ballot(lane < n_groups && rank < keep);
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = lane + u * TIS_WAVE;
      if (e < n_out && !((kept >> (e / per)) & 1ull)) c[u] = -INFINITY;
    }
  }
  float total = 0.f;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int at = 0x7fffffff;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = lane + u * TIS_WAVE;
      if (e < n_out && c[u] > best) { best = c[u]; at = e; }       // rising e within a lane: the lower index keeps a tie
    }
    wave_argmax(best, at);
    float w = 0.f;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      if (lane + u * TIS_WAVE == at) { w = s[u]; c[u] = -INFINITY; }
    }
    w = wave_sum(w);          // only the owner's lane holds it
    total += w;
    if (lane == 0) {
      ids[r * top + k] = at;
      weights[r * top + k] = w * scale;
    }
  }
  // renorm: the chosen weights divided by their sum (lane 0 reads back what it wrote itself)
  if (renorm && lane == 0) {
    const float inv = 1.f / (total + 1e-20f);
    for (int k = 0; k < top; ++k) weights[r * top + k] *= inv;
  }
}

// one workgroup per expert: the assignments that chose it, in rising order
__global__ __launch_bounds__(256) void expert_lists_kernel(const int* __restrict__ ids, int n_assign, int line,
                                                           int* __restrict__ lists, int* __restrict__ counts) {
  __shared__ int wave_count[4];
  __shared__ int base;
  const int e = blockIdx.x, t = threadIdx.x, lane = t % TIS_WAVE, wave = t / TIS_WAVE;
  if (t == 0) base = 0;
  __syncthreads();
  for (int a0 = 0; a0 < n_assign; a0 += 256) {
    const int a = a0 + t;
    const bool mine = a < n_assign && ids[a] == e;
    const unsigned long long vote = __ballot(mine);
    const int before = __popcll(vote & ((1ull << lane) - 1ull));
    if (lane == 0) wave_count[wave] = __popcll(vote);
    __syncthreads();
    int off = base;
    for (int w = 0; w < wave; ++w) off += wave_count[w];
    if (mine) lists[(long)e * line + off + before] = a;
    __syncthreads();
    if (t == 0) base += wave_count[0] + wave_count[1] + wave_count[2] + wave_count[3];
    __syncthreads();
  }
  if (t == 0) counts[e] = base;
}

struct GroupedArgs {
  const int* lists;     // [groups][line] entries, or null: every group takes the entries 0 .. rows-1
  const int* counts;    // [groups], with lists
  int line, rows, a_div;
  long lda, a_group, ldc, c_group;
  int N, K, act;        // act 0: none, 1: erf-form gelu, 2: the matrix's rows alternate gate 0, factor 0, gate 1, ...: C has N / 2
                        // columns, clamped_swish of each pair's two sums
  const float* gate = nullptr;      // [rows][ldg], N columns a group: a result times sigmoid of its number; null: as it is
  long ldg = 0;
  float limit = 0.f;                // act 2
};

// plain multiply-adds, any type and any alignment: 16 entries x 64 columns a workgroup, K in steps of 32 through LDS
// What becomes of entry e's sum for column n of group g.
__device__ __forceinline__ float grouped_result(const GroupedArgs& p, float v, int e, int g, int n) {
  if (p.act == 1) v = gelu_erf_f(v);
  if (p.gate) v *= 1.f / (1.f + expf(-p.gate[(long)e * p.ldg + (long)g * p.N + n]));
  return v;
}

template <typename TA, typename TO>
__global__ __launch_bounds__(256) void grouped_plain_kernel(const TA* __restrict__ A, const TA* __restrict__ W,
                                                            TO* __restrict__ C, GroupedArgs p) {
  __shared__ float As[16][33];
  __shared__ float Ws[64][33];
  __shared__ int entry[16];
  const int g = blockIdx.z, m0 = blockIdx.y * 16, n0 = blockIdx.x * 64, t = threadIdx.x;
  const int count = p.lists ? p.counts[g] : p.rows;
  if (m0 >= count) return;
  if (t < 16) entry[t] = m0 + t < count ? (p.lists ? p.lists[(long)g * p.line + m0 + t] : m0 + t) : -1;
  __syncthreads();
  const TA* Wg = W + (long)g * p.N * p.K;
  const int tx = t % 64, ty = t / 64;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < p.K; k0 += 32) {
    for (int i = t; i < 16 * 32; i += 256) {
      const int row = i / 32, kk = i % 32, e = entry[row];
      As[row][kk] = (e >= 0 && k0 + kk < p.K) ? to_f(A[(long)(e / p.a_div) * p.lda + (long)g * p.a_group + k0 + kk]) : 0.f;
    }
    for (int i = t; i < 64 * 32; i += 256) {
      const int col = i / 32, kk = i % 32;
      Ws[col][kk] = (n0 + col < p.N && k0 + kk < p.K) ? to_f(Wg[(long)(n0 + col) * p.K + k0 + kk]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 32; ++kk) {
      const float w = Ws[tx][kk];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += As[ty * 4 + i][kk] * w;
    }
    __syncthreads();
  }
  if (p.act == 2) {          // a pair's two sums lie on neighbouring lanes
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float other = __shfl_xor(acc[i], 1, TIS_WAVE);
      const int e = entry[ty * 4 + i];
      if (e >= 0 && tx % 2 == 0 && n0 + tx < p.N)
        C[(long)e * p.ldc + (long)g * p.c_group + (n0 + tx) / 2] = from_f<TO>(clamped_swish(acc[i], other, p.limit));
    }
    return;
  }
  if (n0 + tx >= p.N) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = entry[ty * 4 + i];
    if (e < 0) continue;
    const float v = grouped_result(p, acc[i], e, g, n0 + tx);
    C[(long)e * p.ldc + (long)g * p.c_group + n0 + tx] = from_f<TO>(v);
  }
}

// bfloat16 on the matrix cores. A workgroup of four waves, WM x WN of them, owns 16 RM WM entries x 16 RN WN columns; a
// wave owns RM x RN tiles of 16 x 16. A matrix row and an input row are the two operands of v_mfma_f32_16x16x32_bf16
// straight from memory, 16 bytes a lane (rows 16-byte aligned, K a multiple of 8); a wave's RM + RN loads of a step feed
// RM RN products, and what the waves of a workgroup share meets in the caches. Each result is one wave's sum over K in
// steps of 32, or the sum of KS waves' such sums, of every KS-th batch each. Three shapes are built: 16 entries x 64 columns, or x 16 with the sum over K
// split (tis_grouped_split), for groups of a few rows (decoded tokens: the job is to stream the matrices once), 64 x 128 for groups of many that the tiles
// below do not take.
// grid (blocks of columns, groups, tiles of entries): every group's first tile, then every group's second, most of which have no entries and
// end at once. With a group's tiles behind one another the ones that work were every second, fourth .. workgroup, and those go to the same
// compute units: 64 groups of 512 of 1,024, two choices a row, us, so / as it is: 17 rows 22 / 14, 40 21 / 14.5, 64 43 / 15, 127 47 / 16;
// 8 groups of 5,632 of 2,048, 17 rows 52 / 43; 16 of 4,096 of 1,536, 24 rows 50 / 43.
template <typename TO, int WM, int WN, int RM, int RN, int KS>
__global__ __launch_bounds__(256) void grouped_mfma_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                           TO* __restrict__ C, GroupedArgs p) {
  static_assert(WM * WN * KS == 4 && (KS == 1 || WM * RM * RN == 1), "four waves a workgroup");
  const int g = blockIdx.y, t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int part = KS > 1 ? wave / WN : 0;
  const int m0 = blockIdx.z * (16 * RM * WM) + (KS > 1 ? 0 : (wave / WN) * (16 * RM));
  const int n0 = blockIdx.x * (16 * RN * WN) + (wave % WN) * (16 * RN);
  const int c16 = lane & 15, kg = lane >> 4;
  // The count by itself: a workgroup without entries ends on it, and with many groups those are most of the grid. us, the entries asked for beside the count / behind it: 128
  // groups, 8 choices a row, 1 row 5,632 of 2,048 47.7 / 38.2, 3 rows 2,048 of 1,536 34.6 / 28.3, 5 rows 2,048 of 1,024 37.0 / 31.4; 8 groups of 2, 8 rows 2,048 of 2,816
  // 17.6 / 17.8.
  const int count = p.lists ? p.counts[g] : p.rows;
  if (m0 >= count || (KS == 1 && n0 >= p.N)) return;
  int mine[RM];
  const bf16* arow[RM];
#pragma unroll
  for (int i = 0; i < RM; ++i) {
    const int m = m0 + i * 16 + c16;
    mine[i] = m < count ? (p.lists ? p.lists[(long)g * p.line + m] : m) : -1;
    arow[i] = A + (long)(mine[i] < 0 ? 0 : mine[i] / p.a_div) * p.lda + (long)g * p.a_group + kg * 8;
  }
  bool w_ok[RN];
  const bf16* wrow[RN];
#pragma unroll
  for (int j = 0; j < RN; ++j) {
    w_ok[j] = n0 + j * 16 + c16 < p.N;
    wrow[j] = W + ((long)g * p.N + (w_ok[j] ? n0 + j * 16 + c16 : 0)) * p.K + kg * 8;
  }
  f32x4 acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  // A batch is U steps of 32; SETS batches of operands, so that while one is multiplied the next are on their way. A whole batch is read
  // without a condition: lanes without an entry or a column read the group's first, and nobody looks at what becomes of it. What bounds a few
  // entries a group is the matrices' way from memory, of which a wave saw 16 trips one after the other. 8 groups, two choices a row, us, one set and
  // loads under conditions / two sets / three: 8 rows, 5,632 of 2,048 44 / 41 / 40, 2,048 of 2,816 25.0 / 19.6 / 20.1; 5 rows 2,816 of 1,024
  // 12.4 / 12.8 / 12.9, 1,024 of 1,408 12.7 / 10.1 / 10.0; 1 row 5,632 of 2,048 18.4 / 14.7 / 15.1. (161 MB in 41 us: 4 TB/s.)
  constexpr int U = 4, SETS = RM + RN <= 2 ? 2 : 1;
  bf16x8 av[SETS][U][RM], wv[SETS][U][RN];
  const int batches = p.K / (32 * U), whole = KS > 1 ? (batches - part + KS - 1) / KS : batches;      // (in all, and this wave's: every KS-th)
  auto load = [&](int set, int b) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = ((KS > 1 ? b * KS + part : b) * U + u) * 32;
#pragma unroll
      for (int i = 0; i < RM; ++i) av[set][u][i] = *reinterpret_cast<const bf16x8*>(arow[i] + k);
#pragma unroll
      for (int j = 0; j < RN; ++j) wv[set][u][j] = *reinterpret_cast<const bf16x8*>(wrow[j] + k);
    }
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[set][u][j], av[set][u][i], acc[i][j], 0, 0, 0);
  };
#pragma unroll
  for (int e = 0; e < SETS - 1; ++e)
    if (e < whole) load(e, e);
  for (int b0 = 0; b0 < whole; b0 += SETS) {
#pragma unroll
    for (int e = 0; e < SETS; ++e) {
      const int b = b0 + e;
      if (b >= whole) break;
      if (b + SETS - 1 < whole) load((e + SETS - 1) % SETS, b + SETS - 1);
      multiply(e);
    }
  }
  if (batches * 32 * U < p.K && (KS == 1 || batches % KS == part)) {                    // the last, begun batch: zeros past the end of K
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = (batches * U + u) * 32;
      const bool k_ok = k + kg * 8 < p.K;
#pragma unroll
      for (int i = 0; i < RM; ++i) av[0][u][i] = k_ok ? *reinterpret_cast<const bf16x8*>(arow[i] + k) : zero;
#pragma unroll
      for (int j = 0; j < RN; ++j) wv[0][u][j] = k_ok ? *reinterpret_cast<const bf16x8*>(wrow[j] + k) : zero;
    }
    multiply(0);
  }
  if constexpr (KS > 1) {                        // the waves' parts of a column block added in order
    __shared__ f32x4 parts[KS - 1][WN][64];
    if (part > 0) parts[part - 1][wave % WN][lane] = acc[0][0];
    __syncthreads();
    if (part > 0) return;
#pragma unroll
    for (int s = 0; s < KS - 1; ++s) acc[0][0] += parts[s][wave % WN][lane];
  }
  // the lane holds, of tile (i, j), the columns n0 + 16 j + 4 kg + e of entry i * 16 + c16
#pragma unroll
  for (int i = 0; i < RM; ++i) {
    if (mine[i] < 0) continue;
#pragma unroll
    for (int j = 0; j < RN; ++j) {
      if (p.act == 2) {
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          const int n = n0 + j * 16 + 4 * kg + e;
          if (n < p.N)
            C[(long)mine[i] * p.ldc + (long)g * p.c_group + n / 2] = from_f<TO>(clamped_swish(acc[i][j][e], acc[i][j][e + 1], p.limit));
        }
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = n0 + j * 16 + 4 * kg + e;
        if (n >= p.N) continue;
        const float v = grouped_result(p, acc[i][j][e], mine[i], g, n);
        C[(long)mine[i] * p.ldc + (long)g * p.c_group + n] = from_f<TO>(v);
      }
    }
  }
}

// Groups of many rows: the same product tiled in both directions with both operands through LDS, by the loop of the tiled product
// (tile_loop.h). What differs: a tile's rows are list entries, each with an address of its own for reading and for writing,
// the matrix is the group's, and the epilogue may apply the activation. A grid row of tiles per group would be as tall as the
// largest group could be, and most of its workgroups would leave at once; here the row tiles of all groups are numbered through,
// and a workgroup finds its group from the groups' counts (a lane a group, 64 at a time). us, 8 groups, before (4,096 entries: tiles
// of 128 x 128 or 64 in a grid as tall as a group; fewer: 64 x 128 straight from memory) / now: 5,632 columns of 2,048, 4,096 entries
// 162 / 133, 2,000 301 / 101, 1,000 322 / 73, 260 115 / 53; 2,048 of 2,816 93 / 74, 185 / 47, 176 / 28, 73 / 20.
template <typename TO, int BM, int BN, int WM, int WN, int NSTAGE, int AHEAD>
__global__ __launch_bounds__(WM * WN * 64) void grouped_tiles_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                                     TO* __restrict__ C, GroupedArgs p, int groups) {
  typedef TileLoop<BM, BN, WM, WN, NSTAGE, AHEAD> Loop;
  constexpr int LPW = Loop::LPW, TM = Loop::TM, TN = Loop::TN;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[NSTAGE * Loop::STAGE];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r32 = lane & 31, h = lane >> 5;
  const int wm = wave / WN, wn = wave % WN;
  // row tiles of all groups, and then this workgroup's tile and group
  int tiles_m = 0;
  if (p.lists) {
    for (int g0 = 0; g0 < groups; g0 += 64) {
      int n = g0 + lane < groups ? (p.counts[g0 + lane] + BM - 1) / BM : 0;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) n += __shfl_xor(n, o, 64);
      tiles_m += n;
    }
  } else {
    tiles_m = groups * ((p.rows + BM - 1) / BM);
  }
  tiles_m = __builtin_amdgcn_readfirstlane(tiles_m);
  const int tiles_n = (p.N + BN - 1) / BN;
  if (blockIdx.x >= (unsigned)tiles_m * (unsigned)tiles_n) return;
  const GtTile tile = gt_tile(blockIdx.x, tiles_m, tiles_n);
  int g = 0, before = 0;                                // the group, and the row tiles before it
  if (p.lists) {
    for (int g0 = 0; g0 < groups; g0 += 64) {
      int upto = g0 + lane < groups ? (p.counts[g0 + lane] + BM - 1) / BM : 0;
      const int own = upto;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(upto, o, 64);
        if (lane >= o) upto += v;
      }
      const unsigned long long holds = __ballot(before + upto > tile.m);
      if (holds) {
        const int at = __ffsll(holds) - 1;
        g = g0 + at;
        before += __shfl(upto - own, at, 64);
        break;
      }
      before += __shfl(upto, 63, 64);
    }
  } else {
    const int per = (p.rows + BM - 1) / BM;
    g = tile.m / per;
    before = g * per;
  }
  g = __builtin_amdgcn_readfirstlane(g);
  const int m0 = (tile.m - __builtin_amdgcn_readfirstlane(before)) * BM, n0 = tile.n * BN;
  const int count = p.lists ? p.counts[g] : p.rows;
  const bf16* Wg = W + (long)g * p.N * p.K;
  const bf16* Ag = A + (long)g * p.a_group;
  auto entry = [&](int m) {                             // the list entry of the tile's row m (the last one again past the count)
    const int e = min(m0 + m, count - 1);
    return p.lists ? p.lists[(long)g * p.line + e] : e;
  };
  const unsigned char* first[LPW];
  unsigned lane_off[LPW];                               // (the host has seen that they fit)
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const int row0 = Loop::row_of(wave, 0, j), row = Loop::row_of(wave, lane, j);
    if (row0 < BM) {
      first[j] = (const unsigned char*)Ag;
      lane_off[j] = (unsigned)(entry(row) / p.a_div) * (unsigned)(p.lda * 2);
    } else {
      const int r0 = min(p.N - 1, n0 + row0 - BM), r = min(p.N - 1, n0 + row - BM);
      first[j] = (const unsigned char*)(Wg + (long)r0 * p.K);
      lane_off[j] = (unsigned)((r - r0) * p.K * 2);
    }
    lane_off[j] += Loop::piece_of(lane, row) * 16;
  }
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  Loop::run(lds, first, lane_off, p.K, acc);

  // accumulator 4 q + e of block (i, j): entry wm * (BM / WM) + i * 32 + r32 of the tile, column n0 + wn * (BN / WN) + j * 32 + 8 q + 4 h + e
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = wm * (BM / WM) + i * 32 + r32;
    if (m0 + m >= count) continue;
    TO* dst = C + (long)entry(m) * p.ldc + (long)g * p.c_group;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + wn * (BN / WN) + j * 32 + q * 8 + h * 4;
        if (n >= p.N) continue;               // (N is a multiple of 4: the four columns are inside or outside together)
        if (p.act == 2) {
          const float a0 = clamped_swish(acc[i][j][q * 4], acc[i][j][q * 4 + 1], p.limit);
          const float a1 = clamped_swish(acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3], p.limit);
          if constexpr (sizeof(TO) == 4) {
            *(float2*)(dst + n / 2) = make_float2(a0, a1);
          } else {
            typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
            *(bf16x2*)(dst + n / 2) = (bf16x2){static_cast<__bf16>(a0), static_cast<__bf16>(a1)};
          }
          continue;
        }
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = grouped_result(p, acc[i][j][q * 4 + e], entry(m), g, n + e);
        if constexpr (sizeof(TO) == 4) {
          *(f32x4*)(dst + n) = (f32x4){v[0], v[1], v[2], v[3]};
        } else {
          bf16x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = static_cast<__bf16>(v[e]);
          *(bf16x4*)(dst + n) = o;
        }
      }
  }
}

// out[r] = sum_k weight[r][k] * (y[r * top + k] if ids[r][k] < n_experts else x[r]), in 32-bit
template <typename T>
__global__ __launch_bounds__(256) void experts_combine_kernel(const float* __restrict__ y, long ldy, const T* __restrict__ x,
                                                              long ldx, const int* __restrict__ ids,
                                                              const float* __restrict__ weights, int top, int n_experts,
                                                              float* __restrict__ out, long ldo, int D) {
  const long r = blockIdx.x;
  for (int c = threadIdx.x; c < D; c += 256) {
    float v = 0.f;
    for (int k = 0; k < top; ++k) {
      const int e = ids[r * top + k];
      const float w = weights[r * top + k];
      v += w * (e < n_experts ? y[(r * top + k) * ldy + c] : to_f(x[r * ldx + c]));
    }
    out[r * ldo + c] = v;
  }
}

TIS_EXPORT int tis_route_topk(const float* z, long ldz, const float* correction, float scale, int rows, int n_out, int top, int score,
                              int* ids, float* weights, int n_groups, int keep, int renorm, hipStream_t stream) {
  if (rows == 0) return 0;
  if (n_groups < 1 || n_groups > TIS_WAVE || n_out % n_groups || keep < 1 || keep > n_groups || top > keep * (n_out / n_groups))
    return tis_fail("route_topk: %d outputs in %d groups (at most %d) of which %d are kept, top %d", n_out, n_groups, TIS_WAVE, keep, top);
  if (rows < 0 || n_out < 1 || n_out > EX_MAX_PER_LANE * TIS_WAVE || top < 1 || top > n_out)
    return tis_fail("route_topk: bad size rows=%d outputs=%d (at most %d) top=%d", rows, n_out, EX_MAX_PER_LANE * TIS_WAVE, top);
  if (score < 0 || score > 2) return tis_fail("route_topk: score kind %d (0: softmax, 1: sigmoid, 2: softmax over the chosen)", score);
  if (score == 2) renorm = 1;
  if (n_out <= TIS_WAVE)
    route_topk_kernel<1><<<rows, TIS_WAVE, 0, stream>>>(z, ldz, correction, scale, n_out, top, score, ids, weights, n_groups, keep, renorm);
  else
    route_topk_kernel<EX_MAX_PER_LANE><<<rows, TIS_WAVE, 0, stream>>>(z, ldz, correction, scale, n_out, top, score, ids, weights, n_groups, keep, renorm);
  return tis_launch_status("route_topk");
}

TIS_EXPORT int tis_expert_lists(const int* ids, int n_assign, int n_experts, int line, int* lists, int* counts,
                                hipStream_t stream) {
  if (n_experts == 0) return 0;
  if (n_assign < 0 || n_experts < 0 || line < 1) return tis_fail("expert_lists: bad size assignments=%d experts=%d", n_assign, n_experts);
  expert_lists_kernel<<<n_experts, 256, 0, stream>>>(ids, n_assign, line, lists, counts);
  return tis_launch_status("expert_lists");
}

static int g_units = 256;      // compute units of the device: set by whoever knows (the default is an MI355X)
TIS_EXPORT void tis_experts_units(int n) { if (n > 0) g_units = n; }

// The tiles of grouped_tiles_kernel, and the microseconds a step of 64 takes with r workgroups a compute unit:
//   128 x 192, four waves, two buffers, two a unit     1.05 r, at least 1.15
//   64 x 64, four waves, five buffers, two a unit      0.3 r, at least 0.33   (four below 256 inner columns: gated, 64 heads of 128 x 128 and of
//                                                      128 x 192, 1,531 rows 50.2 and 51.5, with five 51.2 and 52.8)
//   128 x 128, eight waves, five buffers               0.58 a round
//   256 x 256, eight waves, two buffers                1.85 a round
//   128 x 128, four waves, two buffers, two a unit     0.78 r, at least 0.8
//   64 x 64, four waves, two buffers, five a unit      (not by this estimate: for products of few steps)
//   128 x 64, eight waves, six buffers                 0.42 a round        (these three from ten steps on: what they gain is
//   256 x 128, eight waves, three buffers              1.1 a round          in the steps, and their buffers take longer to fill)
//   192 x 128, eight waves, four buffers               0.95 a round
// us before the last three / with them, 8 groups, two choices a row: 1,531 rows, 5,632 of 2,048 124 / 106, 2,048 of 2,816 70 / 56; 1,000 rows
// 100 / 88, 60 / 44; 2,048 rows 1,024 of 1,408 37 / 29; 600 rows 2,816 of 1,024 27 / 22, 1,024 of 1,408 18 / 15. A result is the same sum in any tile.
struct GroupedShape { int bm, bn; float step, least; bool rounds; };
static const GroupedShape g_shapes[9] = {{128, 192, 1.05f, 1.15f, false}, {64, 64, 0.3f, 0.33f, false}, {128, 128, 0.58f, 0.58f, true},
                                         {256, 256, 1.85f, 1.85f, true}, {128, 128, 0.78f, 0.8f, false}, {64, 64, 0.f, 0.f, false},
                                         {128, 64, 0.42f, 0.42f, true}, {256, 128, 1.1f, 1.1f, true}, {192, 128, 0.95f, 0.95f, true}};

// The tile that a grouped product of bfloat16 rows that lie as it needs them takes, an index into g_shapes; -1: the products straight from memory.
// lists: most_rows is the most entries a group can have, most_entries the most that all groups have together.
// Without lists: from 64 rows of every group on (16 groups of 512 of 128, us, straight from memory / tiles: 48 rows 4.4 / 4.7, 64 8.7 / 4.8).
// With lists, what counts is the entries a group: while they are few both ways are bound by the matrices' way from memory, where 16 x 64
// straight from memory waits least. Up to 16 rows in the step no group can need a second tile of 16 there, and it is as fast or faster
// for any groups (16 groups, 64 entries: 2,816 of 1,024 20.9 / 28.3; 64 groups, 128 entries: 5,632 of 2,048 221 / 246, 2,048 of 704 36 / 47).
// Beyond, from 48 entries and 4 a group on (12 below 1,024 inner columns, where a tile's few steps do not hide its beginning), us
// straight from memory / tiles at 1, 2, 4, 6, 8, 12 entries a group, 64 groups of 8 choices a row: 5,632 of 2,048 189 / 193, 221 / 246, 277 / 281, 281 / 267,
// 322 / 290, 370 / 293; 2,048 of 2,816 106 / 96, 127 / 127, 140 / 135, 152 / 137, 164 / 140, 204 / 140; 2,048 of 704 26 / 35, 36 / 47, 39 / 49, 42 / 49,
// 44 / 49, 55 / 51. 8 groups of 2, at 4, 6, 8, 12: 5,632 of 2,048 43 / 52, 54 / 52, 54 / 52, 108 / 52; 2,048 of 2,816 25 / 24, 35 / 24, 35 / 24, 31 / 24.
// (Those figures are from when a group's tiles lay behind one another in the grid of the way straight from memory, which cost it up to twice the
// time beyond 16 rows. As it lies now it may be the faster one further up: the line has stayed where nothing became slower.)
// A product per head of few steps (K below 256) is bound by its results' way to memory and by the beginnings and ends of its tiles: the small tile
// of which most fit a unit. us, the tiles before the loop / as the estimate picks them / so: 4,096 rows of 64 heads of 128 x 128 46 / 59 / 42,
// 1,531 rows of 16 of 512 x 128 21 / 20 / 17, 300 of 16 of 512 x 128 7.3 / 8.5 / 6.3, 1,531 of 64 of 64 x 64 9.3 / 13.1 / 10.5. With a gate and heads no
// wider than 128, thousands of such tiles at a time read and write short pieces of rows that lie far apart, and fewer of them are faster: 4,096 rows of 64
// heads of 128 x 128 159 / 177 / 229, with four buffers (two a unit) 130; 1,531 rows 45 / 55 / 58, 49.
TIS_EXPORT int tis_grouped_tile(int lists, int groups, int most_rows, long most_entries, int N, int K, int gate) {
  if (lists ? most_rows <= 16 || most_entries < 48 || most_entries < (K < 1024 ? 12L : 4L) * groups : most_rows < 64) return -1;
  if (!lists && K < 256)
    return gate && N <= 128 && (long)groups * ((most_rows + 63) / 64) * ((N + 63) / 64) > 2048 ? 1 : 5;
  int pick = 0;
  float best = INFINITY;
  // The last three tiles, and what a further round takes below, are for many steps and for groups that the estimate of row tiles fits: sixteen at
  // most, or of 200 entries on average. us, with the first five alone / with all, at lists that an even and an uneven router makes: 64 groups of 6
  // choices, 512 of 1,024, 1,200 rows 36 / 52; 128 of 8, 768 of 2,048, 800 rows 132 / 161; 32 of 4, 1,536 of 2,048, 450 rows 64 / 75. Of 918 sizes of 4 to 128
  // groups 24 now take more than 3 % longer than with those five (before, 87), and all together 0.985 of their time (before, 0.993).
  const bool all = K > 9 * 64 && (!lists || groups <= 16 || most_entries >= 200L * groups);
  for (int i = 0; i < 9; ++i) {
    if (i == 5 || (i > 5 && !all)) continue;
    if (K < 256 && i != 1 && i != 4) continue;     // few steps: what counts is a tile's beginning and end
    const GroupedShape& q = g_shapes[i];
    // a tile of 192 or 256 rows only where the groups fill three quarters of one on average: below, a tile a group is nearly all there is, most of it
    // padding that the estimate's half a tile does not see (us with / without: 64 groups of 8 choices, 1,024 of 1,408, 1,000 rows 123 / 80; 16 of 2, 4,096 of
    // 1,536, 1,000 rows 128 / 81; 32 of 2, 2,048 of 704, 2,048 rows 83 / 65)
    if (lists && q.bm > 128 && most_entries < (long)groups * q.bm * 3 / 4) continue;
    const long tn = (N + q.bn - 1) / q.bn;
    // (with lists, entries / bm row tiles and half a tile more in every group)
    const float r = (lists ? (float)most_entries / q.bm + 0.5f * groups : (float)((long)groups * ((most_rows + q.bm - 1) / q.bm))) * tn / g_units;
    float t = fmaxf(q.least, q.step * (q.rounds ? ceilf(r) : r));
    // from ten steps on, with more tiles than units: what a step takes then (us, 8 groups, two choices a row, 128 x 192 / 128 x 128 / 256 x 128 /
    // 192 x 128: 1,531 rows, 5,632 of 2,048 122 / 124 / 106 / 125; 1,000 rows 110 / 99 / 82 / 88; 600 rows 64 / 70 / 77 / 72; 1,531 rows, 2,048 of 2,816
    // 79 / 68 / 56 / 83)
    if (all && r > 1.f) {
      if (i == 0) t = r <= 2.f ? 1.83f : 0.4f + 1.2f * r;
      else if (i == 2) t = 0.7f * ceilf(r);
      else if (i == 4) t = fmaxf(1.15f * fminf(r, 2.3f), 0.85f * r);
      else if (i == 8) t = ceilf(r);
    }
    if (t < best) best = t, pick = i;
  }
  return pick;
}

// Whether, where no tile takes a product of a few rows a group, a column block's sum over K is split over a workgroup's four waves (16 columns a workgroup) or every wave sums
// its own 16 (64 a workgroup). Split, the chip has more loads under way and compute units differ less in what they get; but there are four times the workgroups, each with a
// beginning and an end, groups without entries among them. So: K long enough that each wave but one gets a batch; from 1,536 on always, below only while the blocks of 64
// columns in all are few. us, matrices from memory, whole / split: 8 groups, two choices a row, 2,048 of 2,816, 1 row 15.5 / 9.2, 3 rows 19.2 / 14.0, 8 20.2 / 17.8, 16 21.0 / 20.3;
// 5,632 of 2,048, 3 rows 31.6 / 23.9, 16 42.2 / 38.8, 1 row 13.9 / 15.3 alone but a decode step with it 325 / 306; 16 of 4, 16 rows 5,632 of 2,048 74.6 / 67.1; 64 of 8, 16 rows 2,048 of
// 2,048 91.8 / 85.0; 128 of 8, 8 rows 2,048 of 1,536 60.4 / 56.3, 16 rows 2,048 of 4,096 254 / 227. Where the line lies, 256 blocks (16 of 4, 16 rows) / 512 (the same, twice the columns): K = 384
// 5.7 / 5.7 and 8.0 / 8.7, 512 6.6 / 6.4 and 9.5 / 10.4, 704 8.1 / 7.4 and 12.2 / 13.2, 1,024 9.6 / 9.2 and 15.6 / 16.1; 640 blocks of 1,024 (64 of 8, 5 rows) 22.1 / 16.1, of 512 12.6 / 11.2; 1,280
// of 384 13.9 / 16.1. Without lists every group has all rows and the blocks are as many as
// they are counted: split where quarters of blocks take at most 0.85 of the rounds over the units that whole ones take. 128 heads of 128 of 1,024, 16 rows (256 blocks, a round either way) 10.5 / 12.9, 32
// (two) 17.8 / 22.2; 64, 16 rows (half a round for one) 10.0 / 7.1; 64 of 192 of 512, 32 rows (384: one and a half for two) 10.5 / 9.0; at 510 sizes of 4 to 128 heads never slower than whole, and 1.005 of
// the faster one's time. Four shorter chains are also the more exact ones: relative error against 64 bits, whole / split, K = 384 1.1e-7 / 0.7e-7, 1,024 1.8e-7 /
// 1.0e-7, 2,048 2.7e-7 / 1.3e-7, 5,632 4.7e-7 / 2.2e-7.
TIS_EXPORT int tis_grouped_split(int lists, int groups, int most_rows, long most_entries, int N, int K) {
  const long blocks = (lists ? (most_entries < groups ? most_entries : groups) : (long)groups * ((most_rows + 15) / 16)) * ((N + 63) / 64);
  if (!lists) {
    const long whole = (blocks + g_units - 1) / g_units, quarters = (4 * blocks + g_units - 1) / g_units;
    return K >= 384 && 5 * quarters <= 17 * whole;
  }
  return K >= 384 && (K >= 1536 || 2 * blocks <= (K >= 1024 ? 6L : 3L) * g_units);
}

// in_dtype / out_dtype: 0 float, 1 bfloat16 (a bfloat16 input may give a 32-bit output). most_rows: the most entries a
// group can have (the grid's height); most_entries: the most that all groups' lists can have together.
TIS_EXPORT int tis_grouped_linear(int in_dtype, int out_dtype, const void* A, long lda, long a_group, int a_div, const void* W,
                                  void* C, long ldc, long c_group, const int* lists, const int* counts, int line,
                                  int groups, int most_rows, long most_entries, int N, int K, int act, const float* gate, long ldg,
                                  float limit, hipStream_t stream) {
  if (groups == 0 || most_rows == 0) return 0;
  if (groups < 0 || groups > 65535 || most_rows < 0 || N < 1 || K < 1 || a_div < 1 || act < 0 || act > 2 ||
      (act == 2 && (N % 2 || !(limit > 0.f))))
    return tis_fail("grouped_linear: bad size groups=%d rows=%d N=%d K=%d", groups, most_rows, N, K);
  if (gate && (lists || act)) return tis_fail("grouped_linear: a gate goes with groups of all rows and no activation");
  if ((lists == nullptr) != (counts == nullptr)) return tis_fail("grouped_linear: lists and counts go together");
  const int tiles_m = (most_rows + 15) / 16;
  if (tiles_m > 65535) return tis_fail("grouped_linear: %d rows are too many for one call", most_rows);
  GroupedArgs p{lists, counts, line, most_rows, a_div, lda, a_group, ldc, c_group, N, K, act, gate, ldg, limit};
  dim3 grid((N + 63) / 64, tiles_m, groups);
  if (in_dtype == TIS_BF16) {
    const bool aligned = K % 8 == 0 && lda % 8 == 0 && a_group % 8 == 0 && ((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0;
    // what a lane stores four columns at a time must be aligned for it
    const int oa = out_dtype == TIS_BF16 ? 8 : 16;
    const bool wide_ok = aligned && N % 4 == 0 && ldc % 4 == 0 && c_group % 4 == 0 && ((uintptr_t)C % oa) == 0 && K >= 64;
    // an entry's row lies within 32 bits of the group's first, and so does a tile's last matrix row of its first
    const bool near = ((lists ? most_entries : most_rows) / a_div + 1) * (lda * 2) < (1L << 32) && (long)K * 512 < (1L << 31);
    const int pick = wide_ok && near ? tis_grouped_tile(lists ? 1 : 0, groups, most_rows, most_entries, N, K, gate ? 1 : 0) : -1;
    if (pick >= 0) {
      // the most row tiles there can be: the entries' own, and one that is begun in every group
      const int bm = g_shapes[pick].bm, bn = g_shapes[pick].bn;
      const long tiles = (lists ? most_entries / bm + groups : (long)groups * ((most_rows + bm - 1) / bm)) * ((N + bn - 1) / bn);
      if (tiles >= (1L << 31)) return tis_fail("grouped_linear: %ld tiles are more than a grid holds", tiles);
#define TILES(BM, BN, WM, WN, NS, AH)                                                                                     \
  {                                                                                                                       \
    if (out_dtype == TIS_BF16) grouped_tiles_kernel<bf16, BM, BN, WM, WN, NS, AH><<<dim3((unsigned)tiles), WM * WN * 64, 0, stream>>>(  \
        (const bf16*)A, (const bf16*)W, (bf16*)C, p, groups);                                                             \
    else grouped_tiles_kernel<float, BM, BN, WM, WN, NS, AH><<<dim3((unsigned)tiles), WM * WN * 64, 0, stream>>>(                       \
        (const bf16*)A, (const bf16*)W, (float*)C, p, groups);                                                            \
  }
      if (pick == 0) TILES(128, 192, 2, 2, 2, 1)
      else if (pick == 1 && K < 256) TILES(64, 64, 2, 2, 4, 2)
      else if (pick == 1) TILES(64, 64, 2, 2, 5, 2)
      else if (pick == 2) TILES(128, 128, 2, 4, 5, 2)
      else if (pick == 3) TILES(256, 256, 2, 4, 2, 1)
      else if (pick == 4) TILES(128, 128, 2, 2, 2, 1)
      else if (pick == 5) TILES(64, 64, 2, 2, 2, 1)
      else if (pick == 6) TILES(128, 64, 4, 2, 6, 2)
      else if (pick == 7) TILES(256, 128, 4, 2, 3, 1)
      else TILES(192, 128, 2, 4, 4, 2)
#undef TILES
    } else if (aligned && most_rows >= 64 * (lists ? groups : 1)) {
      // 64 entries x 128 columns a workgroup, operands straight from memory
      const dim3 big((N + 127) / 128, groups, (most_rows + 63) / 64);
      if (out_dtype == TIS_BF16) grouped_mfma_kernel<bf16, 2, 2, 2, 4, 1><<<big, 256, 0, stream>>>((const bf16*)A, (const bf16*)W, (bf16*)C, p);
      else grouped_mfma_kernel<float, 2, 2, 2, 4, 1><<<big, 256, 0, stream>>>((const bf16*)A, (const bf16*)W, (float*)C, p);
    } else if (aligned) {
#define FEW(WN, KS)                                                                                                       \
  {                                                                                                                       \
    const dim3 few((N + 16 * WN - 1) / (16 * WN), groups, tiles_m);                                                       \
    if (out_dtype == TIS_BF16) grouped_mfma_kernel<bf16, 1, WN, 1, 1, KS><<<few, 256, 0, stream>>>((const bf16*)A, (const bf16*)W, (bf16*)C, p);  \
    else grouped_mfma_kernel<float, 1, WN, 1, 1, KS><<<few, 256, 0, stream>>>((const bf16*)A, (const bf16*)W, (float*)C, p);            \
  }
      if (tis_grouped_split(lists ? 1 : 0, groups, most_rows, most_entries, N, K)) FEW(1, 4)
      else FEW(4, 1)
#undef FEW
    } else {
      if (out_dtype == TIS_BF16) grouped_plain_kernel<bf16, bf16><<<grid, 256, 0, stream>>>((const bf16*)A, (const bf16*)W, (bf16*)C, p);
      else grouped_plain_kernel<bf16, float><<<grid, 256, 0, stream>>>((const bf16*)A, (const bf16*)W, (float*)C, p);
    }
  } else if (in_dtype == TIS_F32 && out_dtype == TIS_F32) {
    grouped_plain_kernel<float, float><<<grid, 256, 0, stream>>>((const float*)A, (const float*)W, (float*)C, p);
  } else {
    return tis_fail("grouped_linear: dtype codes %d -> %d", in_dtype, out_dtype);
  }
  return tis_launch_status("grouped_linear");
}

TIS_EXPORT int tis_experts_combine(int dtype, const float* y, long ldy, const void* x, long ldx, const int* ids,
                                   const float* weights, int top, int n_experts, float* out, long ldo, int rows, int D,
                                   hipStream_t stream) {
  if (rows == 0) return 0;
  if (rows < 0 || D < 1 || top < 1) return tis_fail("experts_combine: bad size rows=%d width=%d top=%d", rows, D, top);
  if (dtype == TIS_F32)
    experts_combine_kernel<float><<<rows, 256, 0, stream>>>(y, ldy, (const float*)x, ldx, ids, weights, top, n_experts, out, ldo, D);
  else if (dtype == TIS_BF16)
    experts_combine_kernel<bf16><<<rows, 256, 0, stream>>>(y, ldy, (const bf16*)x, ldx, ids, weights, top, n_experts, out, ldo, D);
  else
    return tis_fail("unknown dtype code %d", dtype);
  return tis_launch_status("experts_combine");
}
