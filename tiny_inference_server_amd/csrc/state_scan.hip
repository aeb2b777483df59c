// Recurrent mixers whose state is a matrix per head, S [key channels D][value channels V], walked token by token:
//
//   kind 0, decay per key channel:   S_t = diag(a_t) S_(t-1) + k_t v_t^T,                 o_t = S_t^T q_t
//   kind 1, scalar gates (log input gate i, log forget gate f) with a running maximum m that starts at 0:
//           m_t = max(f_t + m_(t-1), i_t);   S_t = exp(f_t + m_(t-1) - m_t) S_(t-1) + exp(i_t - m_t) k_t v_t^T;
//           n_t the same with k_t alone;      o_t = S_t^T q_t / (max(|n_t . q_t|, exp(-m_t)) + 1e-6),
//           with i = cap tanh((x_i + b_i) / cap), f = log sigmoid(cap tanh((x_f + b_f) / cap)).
//
// One workgroup per (request of the step, head, block of 16 value channels). Thread (s, j) owns the state's column j
// for the NS key channels from s * NS on in registers (a token's q, k and decays lie in LDS rows of 16 * NS floats,
// zeros beyond the head's channels, so a thread reads its share in 16-byte pieces), from the request's state slot before the first token to
// the slot after the last. Tokens are taken in chunks: a chunk's q, k, v and gates go into LDS, the 16 threads of a
// column leave a partial o per token there, and one pass adds them up. Each state element sees its tokens strictly in
// order with nothing else mixed in, so among steps that are walked so (no portion of two segments and more in them) the result of a token
// does not depend on how a prompt was cut into steps, on the chunk size or on what else is in the batch, bit for bit. State, gates and sums
// are 32-bit. Kind 1 keeps n and m once per block of value channels (every block needs them, none may read what another has already advanced).
//
// Long portions of prompts are cut into segments of `seg_len` tokens that run side by side (`segments` > 0): up to 128 key
// channels by products of matrices, 64 tokens at most a segment (see there); beyond that the same kernel walks every segment from an
// empty state and leaves the segment's own state, its outputs as if nothing had come before, and what ties them to the past (kind 0: the product of the decays from the segment's start to each
// token; kind 1: the running maximum, the sum of log forget gates and n . q from the segment's start). A second kernel
// then walks the segments of a request in order, element by element, to the state at every segment's start and the
// request's new state; a third adds to every token's output what the state at its segment's start contributes:
//   kind 0: o_t += (q_t * decay product to t)^T S_start
//   kind 1: m_t = max(m'_t, F_t + m_start); numerator and n . q are sums of the segment's own part scaled by
//           exp(m'_t - m_t) and the start's part scaled by exp(F_t + m_start - m_t); o_t as above.
// Everything is still 32-bit; only the order of additions differs from the token-by-token walk, for every request of such a step, the
// ones of a single token too: a token's last bits depend on whether a long portion was in its step.
#include "common.h"
#include <algorithm>
#include <type_traits>

TIS_DEFINE_LAST_ERROR(tis_state_scan)

static constexpr int SC_THREADS = 256;
static constexpr int SC_VB = 16;       // value channels of a workgroup
static constexpr int SC_R = 16;        // threads that share a column
static constexpr int SC_LDS_BYTES = 60 * 1024;

__device__ __forceinline__ float sc_log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// Workspace of a segmented call, per (request, segment) pair v and head h:
//   seg_state [v][h][D*V + D + 2]   the segment's own S, n and m (kernel 1); kernel 2 puts the S and n at the segment's
//                                   start in their place and the m at its start into the last float
//   cum       [row][H*D]            kind 0: product of the decays from the segment's start to the row
//   aux       [row][H][3]           kind 1: m', F and n . q of the segment alone
// Where a head finds its columns: `qk_group` consecutive heads share one set of query and key columns (1: every head
// has its own); head h's decay for key channel i lies at h * decay_hs + i * decay_cs of a row's decays (D and 1: one per
// key channel; 1 and 0: one per head).
// With one decay per head (decay_cs 0) a row's decays are one number a head: the walk reads that one number from LDS
// instead of a line of equal ones, keeps one running product instead of one per key channel, and the workspace's
// `cum` holds [row][H] numbers instead of [row][H*D].
struct ScanLayout {
  int qk_group, decay_hs, decay_cs;
};
__device__ __forceinline__ long cum_at(const ScanLayout& lay, long row, int H, int D, int h, int i) {
  return lay.decay_cs ? (row * H + h) * D + i : row * H + h;
}

struct SegArgs {
  int segments;      // most segments of one request in this call; 0: not segmented
  int seg_len;
  float* seg_state;
  float* cum;
  float* aux;
};

// SC_VB value channels a workgroup, SC_R threads a column. A request's state line keeps n and m once per 16 value
// channels, a segment's own state once per head.
template <int KIND, int NS, bool SEG>
__global__ __launch_bounds__(SC_THREADS) void state_scan_kernel(
    const float* __restrict__ proj, long ldp, int q_off, int k_off, int v_off, float q_scale,
    const float* __restrict__ decay, long ldd, int i_off, int f_off, const float* __restrict__ bias_i,
    const float* __restrict__ bias_f, float cap, float* __restrict__ state, long state_ld,
    const int* __restrict__ cu_rows, const int* __restrict__ seq_slots, float* __restrict__ out, long ldo, int H, int D,
    int V, int n_vb, int chunk, SegArgs sg, ScanLayout lay) {
  constexpr int VB = SC_VB, R = SC_R;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int DP = R * NS;                         // a token's row in LDS: the head's channels, then zeros
  float* sq = lds;                                   // [chunk][DP]
  float* sk = sq + chunk * DP;                       // [chunk][DP]
  float* sa = sk + chunk * DP;                       // kind 0: [chunk][DP] decays; kind 1: [chunk][4] gates i, f and m
  float* sv = sa + (KIND == 0 ? chunk * DP : chunk * 4);  // [chunk][VB]
  float* part = sv + chunk * VB;                     // [chunk][R][VB + 1]

  const int seq = SEG ? blockIdx.x / sg.segments : blockIdx.x, h = blockIdx.y, vb = blockIdx.z, t = threadIdx.x;
  int r0 = cu_rows[seq], r1 = cu_rows[seq + 1];
  if (SEG) {
    r0 += (blockIdx.x % sg.segments) * sg.seg_len;
    r1 = min(r1, r0 + sg.seg_len);
  }
  if (r0 >= r1) return;
  float* st = SEG ? sg.seg_state + ((long)blockIdx.x * H) * ((long)D * V + D + 2) : state + (long)seq_slots[seq] * state_ld;
  float* S = st + (long)h * (SEG ? (long)D * V + D + 2 : (long)D * V);
  // kind 1: n [D], then m; once per block of value channels in a request's state line, once per head in a segment's
  float* nm = SEG ? S + (long)D * V : st + (long)H * D * V + ((long)h * n_vb + vb) * (D + 1);
  const int j = t % VB, s = t / VB;
  const int col = vb * VB + j;
  const bool col_ok = col < V;

  const bool per_head = KIND == 0 && lay.decay_cs == 0;
  float Sreg[NS], nreg[NS], creg[NS];
  float m = SEG ? -INFINITY : 0.f, fsum = 0.f, cprod = 1.f;
#pragma unroll
  for (int e = 0; e < NS; ++e) {
    const int i = s * NS + e;
    Sreg[e] = (!SEG && i < D && col_ok) ? S[(long)i * V + col] : 0.f;
    nreg[e] = (!SEG && KIND == 1 && i < D) ? nm[i] : 0.f;
    creg[e] = 1.f;
  }
  if (!SEG && KIND == 1) m = nm[D];

  for (int c0 = r0; c0 < r1; c0 += chunk) {
    const int nc = min(chunk, r1 - c0);
    __syncthreads();
    for (int idx = t; idx < nc * DP; idx += SC_THREADS) {
      const int c = idx / DP, i = idx - c * DP;
      const float* row = proj + (long)(c0 + c) * ldp;
      const bool in = i < D;
      sq[idx] = in ? row[q_off + (h / lay.qk_group) * D + i] * q_scale : 0.f;
      sk[idx] = in ? row[k_off + (h / lay.qk_group) * D + i] : 0.f;
      if (KIND == 0 && (!per_head || i == 0))
        sa[idx] = in ? decay[(long)(c0 + c) * ldd + h * lay.decay_hs + i * lay.decay_cs] : 0.f;
    }
    for (int idx = t; idx < nc * VB; idx += SC_THREADS) {
      const int c = idx / VB, jj = idx - c * VB;
      sv[idx] = (vb * VB + jj < V) ? proj[(long)(c0 + c) * ldp + v_off + h * V + vb * VB + jj] : 0.f;
    }
    if (KIND == 1 && t < nc) {
      const float* row = proj + (long)(c0 + t) * ldp;
      const float xi = row[i_off + h] + bias_i[h], xf = row[f_off + h] + bias_f[h];
      sa[t * 4] = cap * tanhf(xi / cap);
      sa[t * 4 + 1] = sc_log_sigmoid(cap * tanhf(xf / cap));
    }
    __syncthreads();
    for (int c = 0; c < nc; ++c) {
      float keep = 1.f, take = 1.f;
      if (KIND == 1) {
        const float gi = sa[c * 4], gf = sa[c * 4 + 1];
        const float m_new = fmaxf(gf + m, gi);
        keep = expf(gf + m - m_new);      // (an empty segment's m is -inf: nothing is kept of nothing)
        take = expf(gi - m_new);
        m = m_new;
        fsum += gf;
      }
      const float vj = sv[c * VB + j];
      float acc = 0.f, nq = 0.f;
      const int at = c * DP + s * NS;
      // (channels beyond the head's are zeros in k and q: their state stays zero and adds nothing)
      constexpr int STEP = NS % 4 == 0 ? 4 : 1;      // a thread reads its channels in 16-byte pieces where they allow
      if (per_head) {
        const float a = sa[c * DP];                  // the head's one decay of this token
        cprod *= a;
#pragma unroll
        for (int e0 = 0; e0 < NS; e0 += STEP) {
          float kk[STEP], qq[STEP];
          if (STEP == 4) {
            *reinterpret_cast<float4*>(kk) = *reinterpret_cast<const float4*>(sk + at + e0);
            *reinterpret_cast<float4*>(qq) = *reinterpret_cast<const float4*>(sq + at + e0);
          } else {
            kk[0] = sk[at + e0];
            qq[0] = sq[at + e0];
          }
#pragma unroll
          for (int u = 0; u < STEP; ++u) {
            const int e = e0 + u;
            Sreg[e] = a * Sreg[e] + kk[u] * vj;
            acc += Sreg[e] * qq[u];
          }
        }
        if (SEG && vb == 0 && t == 0) sg.cum[cum_at(lay, c0 + c, H, D, h, 0)] = cprod;
      } else {
#pragma unroll
        for (int e0 = 0; e0 < NS; e0 += STEP) {
          float kk[STEP], qq[STEP], aa[STEP];
          if (STEP == 4) {
            *reinterpret_cast<float4*>(kk) = *reinterpret_cast<const float4*>(sk + at + e0);
            *reinterpret_cast<float4*>(qq) = *reinterpret_cast<const float4*>(sq + at + e0);
            if (KIND == 0) *reinterpret_cast<float4*>(aa) = *reinterpret_cast<const float4*>(sa + at + e0);
          } else {
            kk[0] = sk[at + e0];
            qq[0] = sq[at + e0];
            if (KIND == 0) aa[0] = sa[at + e0];
          }
#pragma unroll
          for (int u = 0; u < STEP; ++u) {
            const int e = e0 + u;
            if (KIND == 0) {
              Sreg[e] = aa[u] * Sreg[e] + kk[u] * vj;
              if (SEG) creg[e] *= aa[u];
            } else {
              Sreg[e] = keep * Sreg[e] + take * (kk[u] * vj);
              nreg[e] = keep * nreg[e] + take * kk[u];
              nq += nreg[e] * qq[u];
            }
            acc += Sreg[e] * qq[u];
          }
        }
        if (KIND == 0 && SEG && vb == 0 && j == 0) {
#pragma unroll
          for (int e = 0; e < NS; ++e)
            if (s * NS + e < D) sg.cum[cum_at(lay, c0 + c, H, D, h, s * NS + e)] = creg[e];
        }
      }
      part[(c * R + s) * (VB + 1) + j] = acc;
      if (KIND == 1) {
        if (j == 0) part[(c * R + s) * (VB + 1) + VB] = nq;
        if (t == 0) sa[c * 4 + 2] = m;
        if (SEG && t == 0 && vb == 0) sg.aux[((long)(c0 + c) * H + h) * 3 + 1] = fsum;
      }
    }
    __syncthreads();
    for (int idx = t; idx < nc * VB; idx += SC_THREADS) {
      const int c = idx / VB, jj = idx - c * VB;
      float o = 0.f, nq = 0.f;
      for (int ss = 0; ss < R; ++ss) {
        o += part[(c * R + ss) * (VB + 1) + jj];
        if (KIND == 1) nq += part[(c * R + ss) * (VB + 1) + VB];
      }
      if (KIND == 1 && !SEG) o /= fmaxf(fabsf(nq), expf(-sa[c * 4 + 2])) + 1e-6f;
      if (KIND == 1 && SEG && vb == 0 && jj == 0) {
        sg.aux[((long)(c0 + c) * H + h) * 3] = sa[c * 4 + 2];
        sg.aux[((long)(c0 + c) * H + h) * 3 + 2] = nq;
      }
      if (vb * VB + jj < V) out[(long)(c0 + c) * ldo + h * V + vb * VB + jj] = o;
    }
  }
#pragma unroll
  for (int e = 0; e < NS; ++e) {
    const int i = s * NS + e;
    if (i < D && col_ok) S[(long)i * V + col] = Sreg[e];
    if (KIND == 1 && j == 0 && i < D && (!SEG || vb == 0)) nm[i] = nreg[e];
  }
  if (KIND == 1 && t == 0 && (!SEG || vb == 0)) nm[D] = m;
}

// Kernel 2 of a segmented call: one thread per element of a head's S (and of n), segment after segment in order. What
// the first kernel left as a segment's own state is replaced by the state at the segment's start; the request's state
// line receives the state after its last row, but for kind 1's m, which every workgroup here reads: kernel 3 writes it.
template <int KIND>
__global__ __launch_bounds__(SC_THREADS) void segment_states_kernel(float* __restrict__ state, long state_ld,
                                                                    const int* __restrict__ cu_rows,
                                                                    const int* __restrict__ seq_slots, int H, int D,
                                                                    int V, int n_vb, SegArgs sg, ScanLayout lay) {
  const int seq = blockIdx.x, h = blockIdx.y;
  const int r0 = cu_rows[seq], r1 = cu_rows[seq + 1];
  if (r0 >= r1) return;
  const int el = blockIdx.z * SC_THREADS + threadIdx.x;      // [0, D*V): S; [D*V, D*V + D): n
  if (el >= D * V + (KIND == 1 ? D : 0)) return;
  const bool is_n = el >= D * V;
  const int i = is_n ? el - D * V : el / V;
  float* st = state + (long)seq_slots[seq] * state_ld;
  const long per = (long)D * V + D + 2;
  float x = is_n ? st[(long)H * D * V + (long)h * n_vb * (D + 1) + i] : st[(long)h * D * V + el];
  float m = KIND == 1 ? st[(long)H * D * V + (long)h * n_vb * (D + 1) + D] : 0.f;
  const int n_seg = (r1 - r0 + sg.seg_len - 1) / sg.seg_len;
  for (int g = 0; g < n_seg; ++g) {
    float* own = sg.seg_state + (((long)seq * sg.segments + g) * H + h) * per;
    const int last = min(r1, r0 + (g + 1) * sg.seg_len) - 1;
    const float mine = own[el];
    float next, m_next = 0.f;
    if (KIND == 0) {
      next = sg.cum[cum_at(lay, last, H, D, h, i)] * x + mine;
    } else {
      const float m_own = own[per - 2], f_all = sg.aux[((long)last * H + h) * 3 + 1];
      m_next = fmaxf(f_all + m, m_own);
      next = expf(f_all + m - m_next) * x + expf(m_own - m_next) * mine;
    }
    own[el] = x;
    if (KIND == 1 && el == 0) own[per - 1] = m;
    x = next;
    m = m_next;
  }
  if (is_n) {
    for (int b = 0; b < n_vb; ++b) st[(long)H * D * V + ((long)h * n_vb + b) * (D + 1) + i] = x;
  } else {
    st[(long)h * D * V + el] = x;
  }
}

// Kernel 3 of a segmented call: what the state at a segment's start adds to its rows. One workgroup per (request and
// segment, head, 64 value channels); rows in tiles of 32, a thread owns one channel for 8 rows.
static constexpr int SG_COLS = 64, SG_ROWS = 32;

template <int KIND>
__global__ __launch_bounds__(SC_THREADS) void segment_outputs_kernel(const float* __restrict__ proj, long ldp, int q_off,
                                                                     float q_scale, float* __restrict__ state, long state_ld,
                                                                     const int* __restrict__ cu_rows,
                                                                     const int* __restrict__ seq_slots,
                                                                     float* __restrict__ out, long ldo, int H, int D,
                                                                     int V, int n_vb, SegArgs sg, ScanLayout lay) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* s0 = lds;                       // [D][SG_COLS]
  float* qt = s0 + D * SG_COLS;          // [SG_ROWS][D + 1]
  float* qn = qt + SG_ROWS * (D + 1);    // [SG_ROWS] kind 1: q . n_start
  const int seq = blockIdx.x / sg.segments, g = blockIdx.x % sg.segments, h = blockIdx.y, t = threadIdx.x;
  const int r0 = cu_rows[seq] + g * sg.seg_len, r1 = min(cu_rows[seq + 1], r0 + sg.seg_len);
  if (r0 >= r1) return;
  const long per = (long)D * V + D + 2;
  const float* start = sg.seg_state + ((long)blockIdx.x * H + h) * per;
  const int c0 = blockIdx.z * SG_COLS, cg = t % 16, rg = t / 16;      // columns cg*4 .. cg*4+3, rows rg*2, rg*2+1
  for (int idx = t; idx < D * SG_COLS; idx += SC_THREADS) {
    const int i = idx / SG_COLS, cc = idx - i * SG_COLS;
    s0[idx] = c0 + cc < V ? start[(long)i * V + c0 + cc] : 0.f;
  }
  const float m0 = KIND == 1 ? start[per - 1] : 0.f;
  if (KIND == 1 && blockIdx.z == 0 && t < n_vb && r1 == cu_rows[seq + 1]) {      // after the request's last row
    const float m = fmaxf(sg.aux[((long)(r1 - 1) * H + h) * 3 + 1] + m0, start[per - 2]);
    for (int b = t; b < n_vb; b += SC_THREADS)
      state[(long)seq_slots[seq] * state_ld + (long)H * D * V + ((long)h * n_vb + b) * (D + 1) + D] = m;
  }
  for (int t0 = r0; t0 < r1; t0 += SG_ROWS) {
    const int nr = min(SG_ROWS, r1 - t0);
    __syncthreads();
    for (int idx = t; idx < nr * D; idx += SC_THREADS) {
      const int r = idx / D, i = idx - r * D;
      float q = proj[(long)(t0 + r) * ldp + q_off + (h / lay.qk_group) * D + i] * q_scale;
      if (KIND == 0) q *= sg.cum[cum_at(lay, t0 + r, H, D, h, i)];
      qt[r * (D + 1) + i] = q;
    }
    __syncthreads();
    if (KIND == 1 && t < nr) {
      float a = 0.f;
      for (int i = 0; i < D; ++i) a += qt[t * (D + 1) + i] * start[(long)D * V + i];
      qn[t] = a;
    }
    float acc[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = 0.f;
    for (int i = 0; i < D; ++i) {
      const float4 sv = *reinterpret_cast<const float4*>(s0 + i * SG_COLS + cg * 4);
      const float qa = qt[(rg * 2) * (D + 1) + i], qb = qt[(rg * 2 + 1) * (D + 1) + i];
      acc[0] += qa * sv.x; acc[1] += qa * sv.y; acc[2] += qa * sv.z; acc[3] += qa * sv.w;
      acc[4] += qb * sv.x; acc[5] += qb * sv.y; acc[6] += qb * sv.z; acc[7] += qb * sv.w;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int r = rg * 2 + k / 4, col = cg * 4 + k % 4;
      if (r < nr && c0 + col < V) {
        float* o = out + (long)(t0 + r) * ldo + h * V + c0 + col;
        if (KIND == 0) {
          *o += acc[k];
        } else {
          const float* a = sg.aux + ((long)(t0 + r) * H + h) * 3;
          const float m_own = a[0], m_t = fmaxf(m_own, a[1] + m0);
          const float w_own = expf(m_own - m_t), w_start = expf(a[1] + m0 - m_t);
          const float nq = w_own * a[2] + w_start * qn[r];
          *o = (w_own * *o + w_start * acc[k]) / (fmaxf(fabsf(nq), expf(-m_t)) + 1e-6f);
        }
      }
    }
  }
}

// ---- segments by matrix products --------------------------------------------------------------------------------------
//
// For up to 128 key channels, in segments of up to 64 rows. Row by row a segment's walk is bound by LDS: every thread reads its
// share of a row's q, k and decays for each of its own state elements, and all that is done with them is one multiply-add each.
// As sums over a segment's rows (S_0 the state at its start, P lower triangular, all in 32 bits, nothing divided by a decay),
//   kind 0:  o_t = (q_t A(-1, t)) S_0 + sum_{i<=t} P(t, i) v_i,  P(t, i) = sum_d q_t k_i A(i, t);   S <- A(-1, last) S_0 + sum_i (k_i A(i, last)) v_i^T
//            with A(i, t) the decays of rows i + 1 .. t multiplied up per channel;
//   kind 1:  P(t, i) = (q_t . k_i) exp(f_(i+1) + .. + f_t + i_i - m'_t), each such sum of forget gates taken from row i on; the own
//            and the start's part put together as in the segments above
// they are products on v_mfma_f32_16x16x4_f32 (32-bit multiply-adds). Three kernels: segment_rows makes P, the scaled queries and
// keys and a segment's decay (or its gates' sums) for every segment and head; segment_walk takes 16 value channels of a head
// through a request's segments in order with S in registers, and leaves S at every segment's start; segment_results makes the
// rows' outputs, all segments at once. Operands lie in the workspace as the products read them, 16 bytes a lane. A request's segments
// are numbered through over the requests of the step, so a step of one long and many short ones needs no more room than its rows.
// MI355X, 8 heads of 128 x 256, us row by row in segments / by products:
// 2,048 rows 233 / 81 (kind 1: 250 / 86), two requests of 1,216 and 584 rows 229 / 70 (250 / 71), 512 rows 124 / 39, 128 rows
// 110 / 30, eight requests of 512 rows 417 / 136. Inside a prompt step of 1,200 and 600 rows, traced kernel by kernel, the rows' kernel takes 28.9
// (LDS, pair by pair; kind 1: 16.6), the walk 26.0 (30.1; a chain of one segment after another, 1.4 us each) and the results 26.9 (32.1; memory:
// the states at the starts twice over). The workspace is 3,360 bytes a row and head of these sizes (the row by row segments' was 2,570 for
// one request, and more than this for requests of unequal lengths). Off from 64 bits, row by row in segments / by products, 130 rows of these
// heads, decays from 0.5, 0.9 and 0.995 on: results 1.26e-7 / 1.01e-7, 1.51e-7 / 1.35e-7, 2.22e-7 / 1.83e-7, states 0.49e-7 / 0.54e-7, 0.87e-7 /
// 0.96e-7, 1.76e-7 / 1.67e-7: sums of products run in four accumulators each, which keeps their chains short, but the decays up to a row's
// segment's end are multiplied up before they meet the row. (One sum in the order of the rows: states 0.49e-7, 1.08e-7, 2.02e-7, results as here;
// a sum for each 16 rows 0.51e-7, 1.02e-7, 1.68e-7, and 92 us where these take 83.) Kind 1 by 0.2e-6 to 2e-6 both ways (its division).
typedef __attribute__((ext_vector_type(4))) float f32x4;
static constexpr int SP_ROWS = 64;               // rows a segment can have: four tiles of 16

// What the workspace holds of a segment and head, in floats, Dp = 64 or 128 the head's channels as they are multiplied.
// Tiles of 16 x 16 are kept as lanes hold them, [lane (g, n)][4]: P and q have row n and columns 4 g .. 4 g + 3 there, k and S
// rows 4 g .. 4 g + 3 of column n.
struct SegmentBlock {
  int q, k, a, x, n, s;        // P [row tile][row tile] lies at 0; scaled q [row tile][channel tile]; scaled k [channel tile][row tile];
                               // decays (kind 0) or the segment's own n [Dp]; m', sums of f, own n . q [64] each and m at the start;
                               // n at the start [Dp]; S at the start [block of 16 value channels][channel tile]
  long floats;
  __host__ __device__ SegmentBlock(int D, int V) {
    const int Dp = D <= 64 ? 64 : 128;
    q = SP_ROWS * SP_ROWS;
    k = q + SP_ROWS * Dp;
    a = k + SP_ROWS * Dp;
    x = a + Dp;
    n = x + 4 * SP_ROWS;      // (every piece begins on a whole line of memory)
    s = n + Dp;
    floats = s + (long)((V + 15) / 16) * 16 * Dp;
  }
};
// The most segments that `rows` rows of `n_seqs` requests can have.
__host__ __device__ constexpr long sp_most(long rows, int seg_len, int n_seqs) { return rows / seg_len + n_seqs; }

struct Segment {
  int first, n;                // its first row of the step, its rows; n 0: there is none of this number
};
// The segment numbered `at` (a lane a request, 64 at a time).
__device__ __forceinline__ Segment find_segment(const int* __restrict__ cu_rows, int n_seqs, int seg_len, int at) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int s0 = 0; s0 < n_seqs; s0 += 64) {
    const int s = s0 + lane;
    const int rows = s < n_seqs ? cu_rows[s + 1] - cu_rows[s] : 0;
    const int own = (rows + seg_len - 1) / seg_len;
    int upto = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o, 64);
      if (lane >= o) upto += v;
    }
    const unsigned long long holds = __ballot(before + upto > at);
    if (holds) {
      const int which = __ffsll(holds) - 1;
      const int c = at - before - __shfl(upto - own, which, 64);
      return {__builtin_amdgcn_readfirstlane(cu_rows[s0 + which] + c * seg_len),
              __builtin_amdgcn_readfirstlane(min(seg_len, __shfl(rows, which, 64) - c * seg_len))};
    }
    before += __shfl(upto, 63, 64);
  }
  return {0, 0};
}

// Sum over the 16 lanes 16 r .. 16 r + 15, every lane gets it, by moves inside the row of lanes.
__device__ __forceinline__ float sp_row_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));    // quad_perm [1,0,3,2]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));    // quad_perm [2,3,0,1]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));   // row_half_mirror
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, true));   // row_mirror
  return v;
}

// grid (heads, segments), eight waves. Kind 0 has to take the decays between two rows per channel, which no product of matrices
// can where it may not divide: inside 16 rows that is done pair by pair (as thread (i, l): row i, channels 4 l .. 4 l + 3 and
// so on by 64), between tiles of 16 rows by a product of q scaled from its tile's start with k scaled to its tile's end, with the tiles
// between them multiplied into q. LDS rows are 4 floats longer than the channels: 16 lanes read 16 rows at one column.
template <int KIND, int NT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void segment_rows_kernel(const float* __restrict__ proj, long ldp, int q_off, int k_off,
                                                           float q_scale, const float* __restrict__ decay, long ldd, int i_off,
                                                           int f_off, const float* __restrict__ bias_i,
                                                           const float* __restrict__ bias_f, float cap,
                                                           const int* __restrict__ cu_rows, int n_seqs, int seg_len,
                                                           float* __restrict__ work, int H, int D, int V, ScanLayout lay) {
  constexpr int Dp = 64 * NT, LD = Dp + 4, LP = SP_ROWS + 4;
  __shared__ __attribute__((aligned(16))) float sq[SP_ROWS][LD], sk[SP_ROWS][LD], sp[SP_ROWS][LP];
  __shared__ __attribute__((aligned(16))) float sa[KIND == 0 ? SP_ROWS : 1][LD], total[4][Dp];     // decays; their products over a tile's rows
  __shared__ float sw[KIND == 1 ? SP_ROWS : 1][LP], gate_i[SP_ROWS], gate_f[SP_ROWS], gate_m[SP_ROWS];
  const Segment seg = find_segment(cu_rows, n_seqs, seg_len, blockIdx.y);
  if (seg.n <= 0) return;                        // (the grid is as wide as there could be segments)
  const int h = blockIdx.x, hq = h / lay.qk_group, t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, g = lane >> 4, n = lane & 15;
  const int nc = (seg.n + 15) / 16;              // tiles of rows
  const SegmentBlock at(D, V);
  float* mine = work + ((long)blockIdx.y * H + h) * at.floats;
  {
    constexpr int STEP = 512 / Dp, PER = SP_ROWS / STEP;   // a thread's rows, STEP apart, of one channel: all loads under way at once
    const int d = t % Dp, r0 = t / Dp;
    // (channels and rows past the last lie behind the buffers' ends: zeros)
    const int at_p = d < D ? (r0 * (int)ldp + d) * 4 : -4, at_d = d < D ? (r0 * (int)ldd + d * lay.decay_cs) * 4 : -4;
    const int bytes = ((seg.n - 1) * (int)ldp + D) * 4;
    const float* row = proj + (long)seg.first * ldp + hq * D;
    auto q_rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(row + q_off), 0, bytes, 0x00020000);
    auto k_rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(row + k_off), 0, bytes, 0x00020000);
    auto d_rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(KIND == 0 ? decay + (long)seg.first * ldd + h * lay.decay_hs : row), 0,
        KIND == 0 ? ((seg.n - 1) * (int)ldd + (D - 1) * lay.decay_cs + 1) * 4 : 0, 0x00020000);
    float q[PER], k[PER], a[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int more = d < D ? e * STEP * (int)ldp * 4 : 0;
      q[e] = __builtin_bit_cast(float, (int)__builtin_amdgcn_raw_buffer_load_b32(q_rows, at_p + more, 0, 0));
      k[e] = __builtin_bit_cast(float, (int)__builtin_amdgcn_raw_buffer_load_b32(k_rows, at_p + more, 0, 0));
      if (KIND == 0)
        a[e] = __builtin_bit_cast(float, (int)__builtin_amdgcn_raw_buffer_load_b32(
                                             d_rows, at_d + (d < D ? e * STEP * (int)ldd * 4 : 0), 0, 0));
    }
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int r = r0 + e * STEP;
      sq[r][d] = q[e] * q_scale;
      sk[r][d] = r < seg.n ? k[e] : 0.f;         // (rows may lie one over the other: a step of 0)
      if (KIND == 0) sa[r][d] = r < seg.n && d < D ? a[e] : 1.f;
    }
  }
  if (KIND == 1 && t < 64) {                     // rows past the last take nothing and keep everything
    const float* row = proj + (long)(seg.first + min(t, seg.n - 1)) * ldp;
    const float xi = row[i_off + h] + bias_i[h], xf = row[f_off + h] + bias_f[h];
    const float gi = t < seg.n ? cap * tanhf(xi / cap) : -INFINITY;
    const float gf = t < seg.n ? sc_log_sigmoid(cap * tanhf(xf / cap)) : 0.f;
    float m = gi, f = gf;                        // the running maximum and the sum of f up to this row
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float mu = __shfl_up(m, o, 64), fu = __shfl_up(f, o, 64);
      if (lane >= o) {
        m = fmaxf(f + mu, m);
        f += fu;
      }
    }
    gate_i[t] = gi;
    gate_f[t] = gf;
    gate_m[t] = m;
    mine[at.x + t] = m;
    mine[at.x + SP_ROWS + t] = f;
  }
  __syncthreads();
  if (KIND == 1) {                               // lane i, rows 8 w .. 8 w + 7: the weight of row i in row t
    const float gi = gate_i[lane];
    float f = 0.f;
    for (int u = 0; u < wave * 8; ++u) f += u > lane ? gate_f[u] : 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int u = wave * 8 + e;
      f += u > lane ? gate_f[u] : 0.f;
      sw[u][lane] = lane <= u ? expf(f + gi - gate_m[u]) : 0.f;
    }
    __syncthreads();
  } else {
    const int i = (t % 256) / 16, l = t % 16;
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
      const int c = t / 256 * 2 + pass;
      f32x4 qt[NT], kt[NT], upto[NT];
      if (c < nc) {
        float p[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) p[j] = 0.f;
#pragma unroll
        for (int v = 0; v < NT; ++v) {
          const int d = l * 4 + v * 64;
          f32x4 up = {1.f, 1.f, 1.f, 1.f}, ka = *reinterpret_cast<const f32x4*>(&sk[c * 16 + i][d]);
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const f32x4 aj = *reinterpret_cast<const f32x4*>(&sa[c * 16 + j][d]);
            const f32x4 qj = *reinterpret_cast<const f32x4*>(&sq[c * 16 + j][d]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              up[e] *= j <= i ? aj[e] : 1.f;
              ka[e] *= j > i ? aj[e] : 1.f;
              p[j] = fmaf(ka[e], qj[e], p[j]);
            }
          }
          qt[v] = *reinterpret_cast<const f32x4*>(&sq[c * 16 + i][d]) * up;
          kt[v] = ka;
          upto[v] = up;
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float ps = sp_row_sum(p[j]);
          if (l == j) sp[c * 16 + j][c * 16 + i] = i <= j ? ps : 0.f;
        }
      }
      __syncthreads();                           // the tile's rows have been read
      if (c < nc) {
#pragma unroll
        for (int v = 0; v < NT; ++v) {
          const int d = l * 4 + v * 64;
          *reinterpret_cast<f32x4*>(&sq[c * 16 + i][d]) = qt[v];
          *reinterpret_cast<f32x4*>(&sk[c * 16 + i][d]) = kt[v];
          if (i == 15) *reinterpret_cast<f32x4*>(&total[c][d]) = upto[v];
        }
      }
    }
    __syncthreads();
  }
  for (int idx = wave; idx < 16; idx += 8) {     // P between tiles of rows (kind 1: and inside them)
    const int J = idx / 4, I = idx % 4;
    if (J >= nc || I > J || (KIND == 0 && I == J)) continue;
    f32x4 part[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) part[r] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int tt = 0; tt < 4 * NT; ++tt) {
      f32x4 qf = *reinterpret_cast<const f32x4*>(&sq[J * 16 + n][tt * 16 + g * 4]);
      const f32x4 kf = *reinterpret_cast<const f32x4*>(&sk[I * 16 + n][tt * 16 + g * 4]);
      if (KIND == 0)
        for (int m = I + 1; m < J; ++m) qf *= *reinterpret_cast<const f32x4*>(&total[m][tt * 16 + g * 4]);
#pragma unroll
      for (int r = 0; r < 4; ++r) part[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[r], kf[r], part[r], 0, 0, 0);
    }
    const f32x4 acc = (part[0] + part[1]) + (part[2] + part[3]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = J * 16 + g * 4 + r, col = I * 16 + n;
      sp[row][col] = KIND == 0 ? acc[r] : col <= row ? acc[r] * sw[row][col] : 0.f;
    }
  }
  __syncthreads();
  const int last = nc * 16 - 1;
  if (KIND == 1) {
    const int row = t / 8;
    if (row < nc * 16) {
      float a = 0.f;
      for (int i = t % 8; i <= row; i += 8) a += sp[row][i];
      a += __shfl_xor(a, 1, 64);
      a += __shfl_xor(a, 2, 64);
      a += __shfl_xor(a, 4, 64);
      if (t % 8 == 0) mine[at.x + 2 * SP_ROWS + row] = a;
    }
    if (t < Dp) {
      float a[4] = {0.f, 0.f, 0.f, 0.f};
      for (int i = 0; i <= last; i += 4)
#pragma unroll
        for (int r = 0; r < 4; ++r) a[r] += sw[last][i + r] * sk[i + r][t];
      mine[at.a + t] = (a[0] + a[1]) + (a[2] + a[3]);
    }
  } else if (t < Dp) {
    float a = 1.f;
    for (int c = 0; c < nc; ++c) a *= total[c][t];
    mine[at.a + t] = a;
  }
  for (int e = wave; e < nc * 4; e += 8) {
    const int J = e / 4, I = e % 4;
    if (I <= J) *reinterpret_cast<f32x4*>(mine + (e * 64 + lane) * 4) = *reinterpret_cast<const f32x4*>(&sp[J * 16 + n][I * 16 + g * 4]);
  }
  for (int e = wave; e < nc * 4 * NT; e += 8) {
    const int J = e / (4 * NT), d = e % (4 * NT) * 16 + g * 4;
    f32x4 qf = *reinterpret_cast<const f32x4*>(&sq[J * 16 + n][d]);
    if (KIND == 0)
      for (int m = 0; m < J; ++m) qf *= *reinterpret_cast<const f32x4*>(&total[m][d]);
    *reinterpret_cast<f32x4*>(mine + at.q + (e * 64 + lane) * 4) = qf;
  }
  for (int e = wave; e < nc * 4 * NT; e += 8) {
    const int tt = e / nc, rt = e % nc, d = tt * 16 + n;
    float scale = 1.f;
    if (KIND == 0)
      for (int m = rt + 1; m < nc; ++m) scale *= total[m][d];
    f32x4 kf;
#pragma unroll
    for (int r = 0; r < 4; ++r) kf[r] = sk[rt * 16 + g * 4 + r][d] * (KIND == 0 ? scale : sw[last][rt * 16 + g * 4 + r]);
    *reinterpret_cast<f32x4*>(mine + at.k + ((tt * 4 + rt) * 64 + lane) * 4) = kf;
  }
}

// The rows 4 g .. 4 g + 3 of every tile of 16 of a segment's values, one column of 16 at `block`: through a buffer that ends behind
// the segment's last value there, so that rows past the last read as zeros and an address is one register that stays (as 64-bit
// addresses, worked out for each of 16 loads, this was most of what the walk did). Columns past the head's are other numbers of the row.
struct ValueRows {
  int offset[4][4];
  int ldp4;
  __device__ __forceinline__ ValueRows(long ldp, int g, int n) : ldp4((int)ldp * 4) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) offset[c][r] = (c * 16 + g * 4 + r) * ldp4 + n * 4;
  }
  __device__ __forceinline__ void fetch(f32x4 (&v)[4], const float* __restrict__ block, int cols, const Segment& seg) const {
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(block + (long)seg.first * (ldp4 / 4)), 0,
                                                  (seg.n - 1) * ldp4 + cols * 4, 0x00020000);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        v[c][r] = __builtin_bit_cast(float, (int)__builtin_amdgcn_raw_buffer_load_b32(rsrc, offset[c][r], 0, 0));
  }
};

// grid (heads, blocks of 16 value channels, requests), four waves of NT tiles of 16 channels each: register r of lane (g, n) in a
// tile is channel 4 g + r of value channel n, as results of products lie. The next segment's operands are under way while
// one is multiplied. Every block of value channels keeps n and m for itself, as a state line does. Workgroups of one head follow one
// another by `heads`: with 8 heads an XCD's L2 serves a head's keys to all of its value channels.
template <int KIND, int NT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void segment_walk_kernel(const float* __restrict__ proj, long ldp, int v_off,
                                                           float* __restrict__ state, long state_ld,
                                                           const int* __restrict__ cu_rows, const int* __restrict__ seq_slots,
                                                           int seg_len, float* __restrict__ work, int H, int D, int V) {
  constexpr int Dp = 64 * NT, SETS = 4;
  const int h = blockIdx.x, vb = blockIdx.y, s = blockIdx.z, t = threadIdx.x, n_vb = gridDim.y;
  const int first = cu_rows[s], n_rows = cu_rows[s + 1] - first;
  if (n_rows <= 0) return;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, g = lane >> 4, n = lane & 15;
  int before = 0;                                // the segments of the requests before
  for (int s0 = 0; s0 < s; s0 += 64) {
    int c = s0 + lane < s ? (cu_rows[s0 + lane + 1] - cu_rows[s0 + lane] + seg_len - 1) / seg_len : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) c += __shfl_xor(c, o, 64);
    before += c;
  }
  const SegmentBlock at(D, V);
  float* base = work + ((long)before * H + h) * at.floats;
  const long stride = (long)H * at.floats;
  const int n_seg = (n_rows + seg_len - 1) / seg_len;
  const int col = vb * 16 + n;
  const float* block = proj + v_off + h * V + vb * 16;
  const int cols = min(16, V - vb * 16);
  const ValueRows values(ldp, g, n);
  float* st = state + (long)seq_slots[s] * state_ld;
  float* S_line = st + (long)h * D * V;
  float* nm = st + (long)H * D * V + ((long)h * n_vb + vb) * (D + 1);
  f32x4 S[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = (wave * NT + u) * 16 + g * 4 + r;
      S[u][r] = d < D && col < V ? S_line[(long)d * V + col] : 0.f;
    }
  float n_mine = KIND == 1 && t < D ? nm[t] : 0.f, m = KIND == 1 ? nm[D] : 0.f;

  if (KIND == 1) __syncthreads();                // m has been read before the first thread is through and writes it
  struct Operands { f32x4 k[NT][4], v[4], a[NT]; float own, m, f; } sets[SETS];
  auto rows_of = [&](int c) { return Segment{first + c * seg_len, min(seg_len, n_rows - c * seg_len)}; };
  auto fetch = [&](Operands& o, int c) {
    const float* p = base + c * stride;
    const Segment seg = rows_of(c);
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)             // (of tiles that the segment does not have: memory that nobody uses)
        o.k[u][rt] = *reinterpret_cast<const f32x4*>(p + at.k + (((wave * NT + u) * 4 + rt) * 64 + lane) * 4);
    if (KIND == 0) {
#pragma unroll
      for (int u = 0; u < NT; ++u) o.a[u] = *reinterpret_cast<const f32x4*>(p + at.a + (wave * NT + u) * 16 + g * 4);
    } else {
      const int last = (seg.n + 15) / 16 * 16 - 1;
      o.own = p[at.a + min(t, Dp - 1)];
      o.m = p[at.x + last];
      o.f = p[at.x + SP_ROWS + last];
    }
    values.fetch(o.v, block, cols, seg);
  };
  auto walk = [&](int c, Operands& o) {
    float* p = base + c * stride;
    const Segment seg = rows_of(c);
    const int nc = (seg.n + 15) / 16;
#pragma unroll
    for (int u = 0; u < NT; ++u)
      *reinterpret_cast<f32x4*>(p + at.s + (((long)vb * 4 * NT + wave * NT + u) * 64 + lane) * 4) = S[u];
    if (KIND == 0) {
#pragma unroll
      for (int u = 0; u < NT; ++u) S[u] *= o.a[u];
    } else {
      if (vb == 0 && t < Dp) p[at.n + t] = n_mine;
      if (vb == 0 && t == 0) p[at.x + 3 * SP_ROWS] = m;
      const float m_next = fmaxf(o.f + m, o.m), keep = expf(o.f + m - m_next), take = expf(o.m - m_next);
      m = m_next;
      n_mine = keep * n_mine + take * o.own;
#pragma unroll
      for (int u = 0; u < NT; ++u) S[u] *= keep;
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) o.v[rt] *= take;
    }
    f32x4 own[NT][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int u = 0; u < NT; ++u)
        own[u][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.k[u][0][r], o.v[0][r], (f32x4){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
    for (int rt = 1; rt < 4; ++rt)
      if (rt < nc) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int u = 0; u < NT; ++u) own[u][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.k[u][rt][r], o.v[rt][r], own[u][r], 0, 0, 0);
      }
#pragma unroll
    for (int u = 0; u < NT; ++u) S[u] += (own[u][0] + own[u][1]) + (own[u][2] + own[u][3]);
  };
#pragma unroll
  for (int c = 0; c < SETS - 1; ++c) fetch(sets[c], min(c, n_seg - 1));
  for (int c0 = 0; c0 < n_seg; c0 += SETS) {
#pragma unroll
    for (int e = 0; e < SETS; ++e) {
      const int c = c0 + e;
      if (c >= n_seg) break;
      fetch(sets[(e + SETS - 1) % SETS], min(c + SETS - 1, n_seg - 1));
      walk(c, sets[e]);
    }
  }
#pragma unroll
  for (int u = 0; u < NT; ++u)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = (wave * NT + u) * 16 + g * 4 + r;
      if (d < D && col < V) S_line[(long)d * V + col] = S[u][r];
    }
  if (KIND == 1 && t < D) nm[t] = n_mine;
  if (KIND == 1 && t == 0) nm[D] = m;
}

// grid (heads, blocks of 64 value channels, segments), a wave 16 value channels of all the segment's rows: the operands that hang
// on the value channels (S at the start, v) stay in registers, P and q go through LDS once for the four waves; everything is under
// way at once.
template <int KIND, int NT>
__global__ __launch_bounds__(256) void segment_results_kernel(const float* __restrict__ proj, long ldp, int v_off,
                                                              const int* __restrict__ cu_rows, int n_seqs, int seg_len,
                                                              const float* __restrict__ work, float* __restrict__ out, long ldo,
                                                              int H, int D, int V, int n_vb) {
  __shared__ f32x4 q_lds[16 * NT][64], p_lds[10][64];
  __shared__ float w_own[SP_ROWS], w_start[SP_ROWS], below[SP_ROWS];
  const Segment seg = find_segment(cu_rows, n_seqs, seg_len, blockIdx.z);
  if (seg.n <= 0) return;
  const int h = blockIdx.x, t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, g = lane >> 4, n = lane & 15;
  const int nc = (seg.n + 15) / 16, vb = blockIdx.y * 4 + wave, col = vb * 16 + n;
  const SegmentBlock at(D, V);
  const float* mine = work + ((long)blockIdx.z * H + h) * at.floats;
  f32x4 S[4 * NT], v[4], q_in[4 * NT], p_in[3];   // (of tiles that the segment does not have: its last ones)
#pragma unroll
  for (int e = 0; e < 4 * NT; ++e)
    q_in[e] = *reinterpret_cast<const f32x4*>(mine + at.q + (min(e * 4 + wave, nc * 4 * NT - 1) * 64 + lane) * 4);
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    const int tile = min(e * 4 + wave, nc * (nc + 1) / 2 - 1), J = tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3;
    p_in[e] = *reinterpret_cast<const f32x4*>(mine + ((J * 4 + tile - J * (J + 1) / 2) * 64 + lane) * 4);
  }
  const int vb_in = min(vb, n_vb - 1);
#pragma unroll
  for (int tt = 0; tt < 4 * NT; ++tt)
    S[tt] = *reinterpret_cast<const f32x4*>(mine + at.s + (((long)vb_in * 4 * NT + tt) * 64 + lane) * 4);
  const float* block = proj + v_off + h * V + vb_in * 16;
  ValueRows(ldp, g, n).fetch(v, block, min(16, V - vb_in * 16), seg);
#pragma unroll
  for (int e = 0; e < 4 * NT; ++e) q_lds[e * 4 + wave][lane] = q_in[e];
#pragma unroll
  for (int e = 0; e < 3; ++e)
    if (e * 4 + wave < 10) p_lds[e * 4 + wave][lane] = p_in[e];
  __syncthreads();
  if (KIND == 1) {
    if (wave < nc) {
      float a = 0.f;                             // q . n at the start, of row n of the wave's tile
#pragma unroll
      for (int tt = 0; tt < 4 * NT; ++tt) {
        const f32x4 x = q_lds[wave * 4 * NT + tt][lane] *
                        *reinterpret_cast<const f32x4*>(mine + at.n + tt * 16 + g * 4);
        a += (x[0] + x[1]) + (x[2] + x[3]);
      }
      a += __shfl_xor(a, 16, 64);
      a += __shfl_xor(a, 32, 64);
      if (g == 0) {
        const int row = wave * 16 + n;
        const float m_own = mine[at.x + row], from = mine[at.x + SP_ROWS + row] + mine[at.x + 3 * SP_ROWS];
        const float m = fmaxf(m_own, from), own = expf(m_own - m), start = expf(from - m);
        w_own[row] = own;
        w_start[row] = start;
        below[row] = fmaxf(fabsf(own * mine[at.x + 2 * SP_ROWS + row] + start * a), expf(-m)) + 1e-6f;
      }
    }
    __syncthreads();
  }
  if (vb >= n_vb) return;
  // P is triangular, but a product takes its zeros times every row: a row that is not finite must not reach the rows before it, so such
  // a segment goes without the matrix product.
  float none = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) none = fmaf(v[c][r], 0.f, none);
  const bool finite = __all(col >= V || none == 0.f);
  auto to = __builtin_amdgcn_make_buffer_rsrc(out + (long)seg.first * ldo + h * V + vb * 16, 0,
                                              ((seg.n - 1) * (int)ldo + min(16, V - vb * 16)) * 4, 0x00020000);
  auto rows = [&](auto count, int j0) {          // the tiles of rows j0 .. j0 + count - 1
    constexpr int N = decltype(count)::value;
    f32x4 part[N][4], acc[N];
    auto clear = [&] {
#pragma unroll
      for (int j = 0; j < N; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[j][r] = (f32x4){0.f, 0.f, 0.f, 0.f};
    };
    clear();
    if (finite) {
#pragma unroll
      for (int I = 0; I < 4; ++I)
#pragma unroll
        for (int j = 0; j < N; ++j)
          if (I <= j0 + j) {
            const f32x4 p = p_lds[(j0 + j) * (j0 + j + 1) / 2 + I][lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) part[j][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[r], v[I][r], part[j][r], 0, 0, 0);
          }
    } else {
#pragma unroll
      for (int j = 0; j < N; ++j)
#pragma unroll 1
        for (int i = 0; i < min((j0 + j) * 16 + 16, seg.n); ++i) {
          const float vi = col < V ? block[(long)(seg.first + i) * ldp + n] : 0.f;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (i <= (j0 + j) * 16 + g * 4 + r)
              part[j][0][r] += mine[(((j0 + j) * 4 + i / 16) * 64 + i % 16 / 4 * 16 + g * 4 + r) * 4 + i % 4] * vi;
        }
    }
    float start[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      acc[j] = (part[j][0] + part[j][1]) + (part[j][2] + part[j][3]);
      start[j] = 1.f;
      if (KIND == 1) {
        start[j] = w_start[(j0 + j) * 16 + n];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[j][r] *= w_own[(j0 + j) * 16 + g * 4 + r];
      }
    }
    clear();
#pragma unroll
    for (int tt = 0; tt < 4 * NT; ++tt) {
      f32x4 q[N];
#pragma unroll
      for (int j = 0; j < N; ++j) {
        q[j] = q_lds[(j0 + j) * 4 * NT + tt][lane];
        if (KIND == 1) q[j] *= start[j];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < N; ++j) part[j][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(q[j][r], S[tt][r], part[j][r], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < N; ++j) acc[j] += (part[j][0] + part[j][1]) + (part[j][2] + part[j][3]);
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {              // (rows past the last lie behind the buffer's end)
        const int row = (j0 + j) * 16 + g * 4 + r;
        const float o = KIND == 1 ? acc[j][r] / below[row] : acc[j][r];
        if (col < V) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, o), to, row * (int)ldo * 4 + n * 4, 0, 0);
      }
  };
  if (nc == 4) rows(std::integral_constant<int, 4>{}, 0);
  else
    for (int j = 0; j < nc; ++j) rows(std::integral_constant<int, 1>{}, j);
}

template <int KIND, int NT>
static int launch_products(const float* proj, long ldp, int q_off, int k_off, int v_off, float q_scale, const float* decay, long ldd,
                           int i_off, int f_off, const float* bias_i, const float* bias_f, float cap, float* state, long state_ld,
                           const int* cu_rows, const int* seq_slots, int n_seqs, float* out, long ldo, int H, int D, int V,
                           int seg_len, int rows, float* work, ScanLayout lay, hipStream_t stream) {
  const unsigned most = (unsigned)sp_most(rows, seg_len, n_seqs);
  const int n_vb = (V + 15) / 16;
  segment_rows_kernel<KIND, NT><<<dim3(H, most), 512, 0, stream>>>(proj, ldp, q_off, k_off, q_scale, decay, ldd, i_off, f_off, bias_i,
                                                                   bias_f, cap, cu_rows, n_seqs, seg_len, work, H, D, V, lay);
  if (tis_launch_status("segment_rows")) return -1;
  segment_walk_kernel<KIND, NT><<<dim3(H, n_vb, n_seqs), 256, 0, stream>>>(proj, ldp, v_off, state, state_ld, cu_rows, seq_slots,
                                                                          seg_len, work, H, D, V);
  if (tis_launch_status("segment_walk")) return -1;
  segment_results_kernel<KIND, NT><<<dim3(H, (n_vb + 3) / 4, most), 256, 0, stream>>>(proj, ldp, v_off, cu_rows, n_seqs, seg_len, work,
                                                                                      out, ldo, H, D, V, n_vb);
  return tis_launch_status("segment_results");
}

template <int KIND>
static int launch_scan(int ns, dim3 grid, size_t lds, hipStream_t stream, const float* proj, long ldp, int q_off, int k_off,
                       int v_off, float q_scale, const float* decay, long ldd, int i_off, int f_off, const float* bias_i,
                       const float* bias_f, float cap, float* state, long state_ld, const int* cu_rows,
                       const int* seq_slots, float* out, long ldo, int H, int D, int V, int n_vb, int chunk, SegArgs sg,
                       ScanLayout lay) {
#define SC_LAUNCH(NS)                                                                                                   \
  if (sg.segments)                                                                                                      \
    state_scan_kernel<KIND, NS, true><<<grid, SC_THREADS, lds, stream>>>(                                        \
        proj, ldp, q_off, k_off, v_off, q_scale, decay, ldd, i_off, f_off, bias_i, bias_f, cap, state, state_ld,        \
        cu_rows, seq_slots, out, ldo, H, D, V, n_vb, chunk, sg, lay);                                                   \
  else                                                                                                                  \
    state_scan_kernel<KIND, NS, false><<<grid, SC_THREADS, lds, stream>>>(                                       \
        proj, ldp, q_off, k_off, v_off, q_scale, decay, ldd, i_off, f_off, bias_i, bias_f, cap, state, state_ld,        \
        cu_rows, seq_slots, out, ldo, H, D, V, n_vb, chunk, sg, lay)
  if (ns <= 1) { SC_LAUNCH(1); }
  else if (ns <= 2) { SC_LAUNCH(2); }
  else if (ns <= 4) { SC_LAUNCH(4); }
  else if (ns <= 8) { SC_LAUNCH(8); }
  else { SC_LAUNCH(16); }
#undef SC_LAUNCH
  if (tis_launch_status("state_scan")) return -1;
  if (!sg.segments) return 0;
  const int n_seqs = grid.x / sg.segments;
  const int elems = D * V + (KIND == 1 ? D : 0);
  segment_states_kernel<KIND><<<dim3(n_seqs, H, (elems + SC_THREADS - 1) / SC_THREADS), SC_THREADS, 0, stream>>>(
      state, state_ld, cu_rows, seq_slots, H, D, V, n_vb, sg, lay);
  if (tis_launch_status("segment_states")) return -1;
  const size_t lds3 = sizeof(float) * ((size_t)D * SG_COLS + (size_t)SG_ROWS * (D + 1) + SG_ROWS);
  segment_outputs_kernel<KIND><<<dim3(grid.x, H, (V + SG_COLS - 1) / SG_COLS), SC_THREADS, lds3, stream>>>(
      proj, ldp, q_off, q_scale, state, state_ld, cu_rows, seq_slots, out, ldo, H, D, V, n_vb, sg, lay);
  return tis_launch_status("segment_outputs");
}

// Whether heads of D key channels can be run in segments (the third kernel keeps 64 columns of a state in LDS).
TIS_EXPORT int tis_state_scan_segmentable(int D) {
  return sizeof(float) * ((size_t)D * SG_COLS + (size_t)SG_ROWS * (D + 1) + SG_ROWS) <= 64 * 1024;
}

// Whether a segmented call goes through the kernels of matrix products, whose addresses inside a segment are 32-bit (ld: the longest
// distance between two rows). Longer segments are cut into theirs of SP_ROWS rows: what was gained by longer ones, fewer states
// to carry, was the row by row kernels'. Segments of
// 128, us, row by row / cut: 2,048 rows of 8 heads of 128 x 256 277 / 83 (kind 1: 269 / 86), 300 rows 124 / 35.
static bool by_products(int n_seqs, int seg_len, int D, long rows, long ld) {
  return D <= 128 && ld >= 0 && ld < (1L << 22) && n_seqs <= 65535 && sp_most(rows, std::min(seg_len, SP_ROWS), n_seqs) <= 65535;
}

// 32-bit floats of the workspace a segmented call needs (ld: the longest row distance of projections, decays and results): a block
// for every segment and head; or, off the matrix products, the states, then `rows` lines of decay products or gate sums.
TIS_EXPORT long tis_state_scan_workspace(int kind, int n_seqs, int segments, int seg_len, int rows, int H, int D, int V,
                                         long ld) {
  if (by_products(n_seqs, seg_len, D, rows, ld)) return sp_most(rows, std::min(seg_len, SP_ROWS), n_seqs) * H * SegmentBlock(D, V).floats;
  return (long)n_seqs * segments * H * ((long)D * V + D + 2) + (kind == 0 ? (long)rows * H * D : (long)rows * H * 3);
}

// Floats of one request's state: S for every head, and for kind 1 also n and m per head and block of value channels.
TIS_EXPORT long tis_state_scan_floats(int kind, int H, int D, int V) {
  const long n_vb = (V + SC_VB - 1) / SC_VB;
  return (long)H * D * V + (kind == 1 ? (long)H * n_vb * (D + 1) : 0);
}

TIS_EXPORT int tis_state_scan(int kind, const float* proj, long ldp, int q_off, int k_off, int v_off, float q_scale,
                              const float* decay, long ldd, int i_off, int f_off, const float* bias_i,
                              const float* bias_f, float cap, float* state, long state_ld, const int* cu_rows,
                              const int* seq_slots, int n_seqs, float* out, long ldo, int H, int D, int V,
                              int segments, int seg_len, int rows, float* workspace, int qk_group, int decay_per_head,
                              hipStream_t stream) {
  if (n_seqs == 0) return 0;
  if (qk_group < 1 || H % qk_group) return tis_fail("state_scan: %d heads in groups of %d", H, qk_group);
  const ScanLayout lay = {qk_group, decay_per_head ? 1 : D, decay_per_head ? 0 : 1};
  if (n_seqs < 0 || H < 1 || H > 65535 || D < 1 || D > SC_R * 16 || V < 1)
    return tis_fail("state_scan: bad size requests=%d heads=%d key channels=%d (at most %d) value channels=%d", n_seqs, H,
                    D, SC_R * 16, V);
  if (kind != 0 && kind != 1) return tis_fail("state_scan: unknown kind %d", kind);
  if (kind == 0 && !decay) return tis_fail("state_scan: kind 0 needs the decays");
  if (kind == 1 && (!bias_i || !bias_f || !(cap > 0.f))) return tis_fail("state_scan: kind 1 needs gate biases and a cap");
  const int n_vb = (V + SC_VB - 1) / SC_VB;
  if (n_vb > 65535) return tis_fail("state_scan: %d value channels exceed the grid", V);
  if (state_ld < tis_state_scan_floats(kind, H, D, V))
    return tis_fail("state_scan: a state line of %ld floats is too short for %ld", state_ld, tis_state_scan_floats(kind, H, D, V));
  int chunk = 16;
  const int ns = (D + SC_R - 1) / SC_R, ns_built = ns <= 1 ? 1 : ns <= 2 ? 2 : ns <= 4 ? 4 : ns <= 8 ? 8 : 16;
  const size_t dp = (size_t)SC_R * ns_built;      // a token's row in LDS (see the kernel)
  auto bytes = [&](int c) {
    return sizeof(float) * ((size_t)c * dp * 2 + (kind == 0 ? (size_t)c * dp : (size_t)c * 4) + (size_t)c * SC_VB +
                            (size_t)c * SC_R * (SC_VB + 1));
  };
  while (chunk > 1 && bytes(chunk) > SC_LDS_BYTES) chunk /= 2;
  if (bytes(chunk) > SC_LDS_BYTES) return tis_fail("state_scan: %d key channels do not fit the chunk buffers", D);
  SegArgs sg = {0, 0, nullptr, nullptr, nullptr};
  if (segments > 0) {
    if (seg_len < 1 || rows < 1 || !workspace || (long)n_seqs * segments > 0x7fffffffL)
      return tis_fail("state_scan: %d segments of %d rows need a workspace", segments, seg_len);
    if (by_products(n_seqs, seg_len, D, rows, std::max(ldo, std::max(ldp, ldd)))) {
      if ((uintptr_t)workspace % 16) return tis_fail("state_scan: the workspace is not 16 bytes aligned");
#define SP_LAUNCH(KIND, NT)                                                                                                       \
  return launch_products<KIND, NT>(proj, ldp, q_off, k_off, v_off, q_scale, decay, ldd, i_off, f_off, bias_i, bias_f, cap, state, \
                                   state_ld, cu_rows, seq_slots, n_seqs, out, ldo, H, D, V, std::min(seg_len, SP_ROWS), rows, workspace, lay, \
                                   stream)
      if (kind == 0 && D <= 64) SP_LAUNCH(0, 1);
      if (kind == 0) SP_LAUNCH(0, 2);
      if (D <= 64) SP_LAUNCH(1, 1);
      SP_LAUNCH(1, 2);
#undef SP_LAUNCH
    }
    sg.segments = segments;
    sg.seg_len = seg_len;
    sg.seg_state = workspace;
    float* lines = workspace + (long)n_seqs * segments * H * ((long)D * V + D + 2);
    sg.cum = kind == 0 ? lines : nullptr;
    sg.aux = kind == 1 ? lines : nullptr;
    if (sizeof(float) * ((size_t)D * SG_COLS + (size_t)SG_ROWS * (D + 1) + SG_ROWS) > 64 * 1024)
      return tis_fail("state_scan: %d key channels do not fit the segment kernels (see tis_state_scan_segmentable)", D);
  }
  dim3 grid(segments > 0 ? n_seqs * segments : n_seqs, H, n_vb);
  if (kind == 0)
    return launch_scan<0>(ns, grid, bytes(chunk), stream, proj, ldp, q_off, k_off, v_off, q_scale, decay, ldd, i_off, f_off,
                          bias_i, bias_f, cap, state, state_ld, cu_rows, seq_slots, out, ldo, H, D, V, n_vb, chunk, sg, lay);
  return launch_scan<1>(ns, grid, bytes(chunk), stream, proj, ldp, q_off, k_off, v_off, q_scale, decay, ldd, i_off, f_off,
                        bias_i, bias_f, cap, state, state_ld, cu_rows, seq_slots, out, ldo, H, D, V, n_vb, chunk, sg, lay);
}
