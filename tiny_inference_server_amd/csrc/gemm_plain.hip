// C[M,N] = A[M,K] . W[N,K]^T (+ R[M,N]) with plain 32-bit multiply-adds: the matrix product of the true
// 32-bit path, and of any shape the faster kernels refuse. No matrix-core instruction and no reduced
// precision mode is used here; inputs may be stored as float or bfloat16 and are widened exactly.
// Each output element sums its K products in the same order whatever M is, so a row's result does not
// depend on the other rows of the batch.
#include <type_traits>

#include "common.h"

TIS_DEFINE_LAST_ERROR(tis_gemm_plain)

static constexpr int GP_BM = 64, GP_BN = 64, GP_BK = 16, GP_THREADS = 256;

template <typename TI, typename TO>
__global__ __launch_bounds__(GP_THREADS) void gemm_plain_kernel(const TI* __restrict__ A, long lda,
                                                                const TI* __restrict__ W, long ldw,
                                                                const TO* __restrict__ R, long ldr, TO* __restrict__ C,
                                                                long ldc, int M, int N, int K) {
  __shared__ float As[GP_BK][GP_BM + 4];
  __shared__ float Ws[GP_BK][GP_BN + 4];
  const int t = threadIdx.x;
  const int tx = t % 16, ty = t / 16;
  const long m0 = (long)blockIdx.y * GP_BM, n0 = (long)blockIdx.x * GP_BN;
  const int lrow = t / 4, lk = (t % 4) * 4;

  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  for (int k0 = 0; k0 < K; k0 += GP_BK) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = k0 + lk + e;
      const long am = m0 + lrow, wn = n0 + lrow;
      As[lk + e][lrow] = (am < M && k < K) ? to_f(A[am * lda + k]) : 0.f;
      Ws[lk + e][lrow] = (wn < N && k < K) ? to_f(W[wn * ldw + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < GP_BK; ++k) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[k][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Ws[k][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const long m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const long n = n0 + tx * 4 + j;
      if (n >= N) continue;
      float v = acc[i][j];
      if (R) v += to_f(R[m * ldr + n]);
      C[m * ldc + n] = from_f<TO>(v);
    }
  }
}

// The same product for few rows or few columns, where tiles of 64 x 64 leave most compute units idle and their chunks of 16
// are one trip to memory each: a workgroup owns 16 rows and 16 columns, a thread one output, and K comes through LDS in
// chunks of 256, the next chunk's loads in flight in registers while one is summed. Same order of sums as above, so the
// results are the same bits. What bounds it is the chain of K multiply-adds and two LDS reads for every four of them.
// A row of LDS is four floats longer than a chunk: the 16 columns a read takes 16 bytes of lie in 16 different bank groups.
// VEC: rows of A and W start on 16 bytes and K is a multiple of 4. MI355X, float, us, tiles of 64 x 64 / these:
// 3 rows 64 x 64 8.9 / 3.2, 64 x 176 17.7 / 3.8; 1 row 1536 x 1536 136 / 15; 8 rows 1536 x 4096 365 / 35, 48000 x 1536 253 / 97;
// 100 rows 1536 x 4096 436 / 74.
static constexpr int GS_BM = 16, GS_BN = 16, GS_BK = 256, GS_LD = GS_BK + 4;

// NORM: A's rows are RMS-normed on the way in, x * sqrt(K) / (||x|| + eps) * gain with the sum of squares added up in the order of the
// norm's own kernel (256 threads a row, four waves); GATE: C has N / 2 columns, silu(g) u of the columns' pairs (2j, 2j + 1). Both give the
// bits of the separate kernels. GATE saves a kernel (us, product and gate's kernel / one: 16 x 64 x 352 5.2 / 3.5, 128 x 1,024 x 2,048 26 / 24; faster at all
// of 370 sizes). NORM saves a launch, and little time on the GPU: every column tile sums its 16 rows' squares again before its first product (see
// tis_gemm_plain_norms).
template <bool VEC, typename TI, typename TO, bool NORM = false, bool GATE = false>
__global__ __launch_bounds__(GS_BM * GS_BN) void gemm_plain_few_kernel(const TI* __restrict__ A, long lda, const TI* __restrict__ W,
                                                                   long ldw, const TO* __restrict__ R, long ldr,
                                                                   TO* __restrict__ C, long ldc, int M, int N, int K,
                                                                   const float* __restrict__ gain, float eps) {
  static_assert(!NORM || (VEC && sizeof(TI) == 4), "normed rows are 32-bit and read 16 bytes at a time");
  constexpr int THREADS = GS_BM * GS_BN, ROWS = GS_BN + GS_BM, PER = ROWS * (GS_BK / 4) / THREADS;   // groups of four a thread copies
  __shared__ __attribute__((aligned(16))) float lds[2][ROWS][GS_LD];                           // W's rows, then A's
  const int t = threadIdx.x, tx = t % GS_BN, ty = t / GS_BN;
  const long m0 = (long)blockIdx.y * GS_BM, n0 = (long)blockIdx.x * GS_BN;
  __shared__ float row_mul[NORM ? GS_BM : 1];
  float4 held[PER], held_gain[NORM ? PER : 1];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int row = (i * THREADS + t) / (GS_BK / 4), at = (i * THREADS + t) % (GS_BK / 4);
      const bool is_w = row < GS_BN;
      const long r = is_w ? n0 + row : m0 + row - GS_BN;
      const bool ok = r < (is_w ? N : M);
      const TI* src = is_w ? W + (ok ? r : 0) * ldw : A + (ok ? r : 0) * lda;
      held[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if constexpr (VEC && sizeof(TI) == 4) {
        if (ok && k0 + at * 4 < K) held[i] = *reinterpret_cast<const float4*>(src + k0 + at * 4);
        if constexpr (NORM)
          held_gain[i] = !is_w && k0 + at * 4 < K ? *reinterpret_cast<const float4*>(gain + k0 + at * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
      } else {               // elements at, at + 64, ...: neighbouring threads read neighbours
        float* h = reinterpret_cast<float*>(&held[i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = k0 + at + e * (GS_BK / 4);
          if (ok && k < K) h[e] = to_f(src[k]);
        }
      }
    }
  };
  auto commit = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int row = (i * THREADS + t) / (GS_BK / 4), at = (i * THREADS + t) % (GS_BK / 4);
      if constexpr (VEC && sizeof(TI) == 4) {
        if constexpr (NORM) {
          if (row >= GS_BN) {
            const float mul = row_mul[row - GS_BN];
            held[i] = make_float4(held[i].x * mul * held_gain[i].x, held[i].y * mul * held_gain[i].y, held[i].z * mul * held_gain[i].z,
                                  held[i].w * mul * held_gain[i].w);
          }
        }
        *reinterpret_cast<float4*>(&lds[buf][row][at * 4]) = held[i];
      } else {
        const float* h = reinterpret_cast<const float*>(&held[i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) lds[buf][row][at + e * (GS_BK / 4)] = h[e];
      }
    }
  };
  const long m = m0 + ty, n = n0 + tx;
  const bool live = m < M && n < N;
  float res = 0.f;
  if (R && live) res = to_f(R[m * ldr + n]);
  float acc = 0.f;
  fetch(0);
  if constexpr (NORM) {
    const int lane = t % TIS_WAVE, wave = t / TIS_WAVE;
    // NV: of the four waves that would share a row, those that have values (64 a turn); the others' sums are zeros. A wave's four rows are asked
    // for at once, from addresses that always hold something (3 rows of 64 against 192 or 352 columns, traced in replayed steps, us: 6.6 row after row, 16 sums a wave; 4.5 so).
    auto squares = [&](auto nv) {
      constexpr int NV = nv;
      float ss[4][NV];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int v = 0; v < NV; ++v) ss[r][v] = 0.f;
      for (int k0 = 0; k0 < K; k0 += 4 * TIS_WAVE) {
        float x[4][NV];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int v = 0; v < NV; ++v)
            x[r][v] = to_f(A[min(m0 + wave * 4 + r, (long)M - 1) * lda + min(k0 + v * TIS_WAVE + lane, K - 1)]);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            const float in = k0 + v * TIS_WAVE + lane < K ? x[r][v] : 0.f;
            ss[r][v] += in * in;
          }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float sum = 0.f;
#pragma unroll
        for (int v = 0; v < NV; ++v) sum += wave_sum(ss[r][v]);
        if (lane == 0) row_mul[wave * 4 + r] = sqrtf((float)K) / (sqrtf(sum) + eps);
      }
    };
    if (K <= TIS_WAVE) squares(std::integral_constant<int, 1>{});
    else if (K <= 2 * TIS_WAVE) squares(std::integral_constant<int, 2>{});
    else squares(std::integral_constant<int, 4>{});
    __syncthreads();
  }
  commit(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += GS_BK, buf ^= 1) {
    const bool more = k0 + GS_BK < K;
    if (more) fetch(k0 + GS_BK);
    const float* wr = lds[buf][tx];
    const float* ar = lds[buf][GS_BN + ty];
    const int kc = min(GS_BK, (K - k0 + 15) / 16 * 16);
    for (int k = 0; k < kc; k += 16) {
#pragma unroll
      for (int j = 0; j < 16; j += 4) {
        const float4 a = *reinterpret_cast<const float4*>(ar + k + j), b = *reinterpret_cast<const float4*>(wr + k + j);
        acc = fmaf(a.x, b.x, acc);
        acc = fmaf(a.y, b.y, acc);
        acc = fmaf(a.z, b.z, acc);
        acc = fmaf(a.w, b.w, acc);
      }
    }
    if (more) commit(buf ^ 1);
    __syncthreads();
  }
  if constexpr (GATE) {
    const float u = __shfl_xor(acc, 1, TIS_WAVE);        // the odd column beside this one
    if (live && n % 2 == 0) C[m * ldc + n / 2] = from_f<TO>(acc / (1.f + expf(-acc)) * u);
  } else if (live) {
    C[m * ldc + n] = from_f<TO>(R ? acc + res : acc);
  }
}

// Whether a product of M rows takes the tiles of 16 x 16; wide: its rows are read 16 bytes at a time. What counts is how many tiles of 64 x 64
// there would be: few of them are a chain of K / 16 trips to memory on a chip that is mostly idle, many fill the chip and read each row a
// quarter as often. us, tiles of 64 x 64 / of 16 x 16, read wide (float): K = 1536, 384 tiles 248 / 187, 512 tiles 243 / 252, 768 tiles
// 297 / 371; K = 176, 32 tiles 20.2 / 4.9; K = 64, 256 tiles 11.7 / 19.9, 120 tiles 10.8 / 12.3, 64 tiles 10.6 / 7.8. Up to 16 rows most of
// a 64 x 64 tile's rows are not there: 16 rows of 48,000 columns (750 tiles) K = 1536 260 / 111, K = 176 31 / 23, but K = 64 15.0 / 17.3.
// Read value by value (bfloat16, rows that do not start on 16 bytes) a small tile costs more: K = 1537, 120 tiles 172 / 149, 128 tiles of 2,048 x 200
// 178 / 223, 320 tiles 214 / 369, 384 tiles 234 / 550; K = 65, 64 tiles 11.0 / 10.6, 120 tiles 11.1 / 19.3; 16 rows of 48,000 columns
// K = 1537 272 / 348, K = 4097 845 / 1,266.
TIS_EXPORT int tis_gemm_plain_few(int wide, int M, int N, int K) {
  const long tiles = (long)((N + GP_BN - 1) / GP_BN) * ((M + GP_BM - 1) / GP_BM);
  if (wide) return (M <= 16 && K >= 128) || tiles < (K >= 512 ? 512 : K >= 128 ? 128 : 96);
  return tiles < (K >= 512 ? 128 : 96);
}

template <typename TI, typename TO>
static void launch_plain(const void* A, long lda, const void* W, long ldw, const void* R, long ldr, void* C, long ldc, int M,
                         int N, int K, hipStream_t stream) {
  const bool vec = sizeof(TI) == 4 && K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
  if (tis_gemm_plain_few(vec, M, N, K)) {
    const dim3 grid((N + GS_BN - 1) / GS_BN, (M + GS_BM - 1) / GS_BM);
    const auto kernel = vec ? gemm_plain_few_kernel<true, TI, TO> : gemm_plain_few_kernel<false, TI, TO>;
    kernel<<<grid, GS_BM * GS_BN, 0, stream>>>((const TI*)A, lda, (const TI*)W, ldw, (const TO*)R, ldr, (TO*)C, ldc, M, N, K, nullptr, 0.f);
    return;
  }
  const dim3 grid((N + GP_BN - 1) / GP_BN, (M + GP_BM - 1) / GP_BM);
  gemm_plain_kernel<TI, TO><<<grid, GP_THREADS, 0, stream>>>((const TI*)A, lda, (const TI*)W, ldw, (const TO*)R, ldr, (TO*)C,
                                                             ldc, M, N, K);
}

// in_dtype / out_dtype: 0 float, 1 bfloat16. Supported: (0,0), (1,1), (1,0).
TIS_EXPORT int tis_gemm_plain(int in_dtype, int out_dtype, const void* A, long lda, const void* W, long ldw,
                              const void* R, long ldr, void* C, long ldc, int M, int N, int K, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  if (M < 0 || N < 0 || K < 1) return tis_fail("gemm: bad size M=%d N=%d K=%d", M, N, K);
  if ((M + GP_BM - 1) / GP_BM > 65535) return tis_fail("gemm: %d rows exceed the grid", M);
  if (in_dtype == TIS_F32 && out_dtype == TIS_F32)
    launch_plain<float, float>(A, lda, W, ldw, R, ldr, C, ldc, M, N, K, stream);
  else if (in_dtype == TIS_BF16 && out_dtype == TIS_BF16)
    launch_plain<bf16, bf16>(A, lda, W, ldw, R, ldr, C, ldc, M, N, K, stream);
  else if (in_dtype == TIS_BF16 && out_dtype == TIS_F32)
    launch_plain<bf16, float>(A, lda, W, ldw, R, ldr, C, ldc, M, N, K, stream);
  else
    return tis_fail("gemm: unsupported dtype pair in=%d out=%d", in_dtype, out_dtype);
  return tis_launch_status("gemm_plain");
}

// The product of 32-bit rows with the gate behind it and the norm before it (see the kernel): whether it takes M rows of K values against N columns.
TIS_EXPORT int tis_gemm_plain_fuses(int M, int N, int K) {
  return M > 0 && N > 0 && K > 0 && K % 4 == 0 && K <= 1024 && tis_gemm_plain_few(1, M, N, K) && (M + GS_BM - 1) / GS_BM <= 65535;
}

// Whether such a product is worth taking the norm inside. On the GPU the norm's own kernel is the faster at every size, us in a graph of such pairs, norm and
// product / one kernel: 4 rows of 176 x 64 5.3 / 5.6, 128 of 1,024 x 64 6.1 / 7.5, 16 of 2,048 x 128 6.0 / 7.2. But each kernel is the host's time, which
// steps of models of this size wait for: launched prompts of a 64 wide model, norms inside / apart, 600 / 640 us; replayed, as fast either way.
// Beyond 128 inner columns, or 256 tiles, it costs more than a launch: 16 rows of 2,048 x 512 9.3 / 12.8, 128 of 2,048 x 128 9.4 / 15.3, 512 of 2,048 x 1,024
// 93 / 216.
TIS_EXPORT int tis_gemm_plain_norms(int M, int N, int K) {
  return tis_gemm_plain_fuses(M, N, K) && K <= 128 && (long)((N + GS_BN - 1) / GS_BN) * ((M + GS_BM - 1) / GS_BM) <= 256;
}

// gain: null, or the norm's gain [K] (eps is added to the norm); gate: C has N / 2 columns. A, W and gain start on 16 bytes, lda and ldw in steps of 4.
TIS_EXPORT int tis_gemm_plain_fused(const float* A, long lda, const float* gain, float eps, const float* W, long ldw, const float* R, long ldr,
                                    float* C, long ldc, int M, int N, int K, int gate, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  if (!tis_gemm_plain_fuses(M, N, K)) return tis_fail("gemm: no fused product of M=%d N=%d K=%d", M, N, K);
  if (lda % 4 || ldw % 4 || ((uintptr_t)A | (uintptr_t)W | (uintptr_t)gain) % 16) return tis_fail("gemm: a fused product's rows start on 16 bytes");
  if (!gain && !gate) return tis_fail("gemm: a fused product has a norm or a gate");
  if (gate && (R || N % 2)) return tis_fail("gemm: a gate goes with pairs of columns and no residual");
  const dim3 grid((N + GS_BN - 1) / GS_BN, (M + GS_BM - 1) / GS_BM);
#define FUSED(NORM, GATE) gemm_plain_few_kernel<true, float, float, NORM, GATE><<<grid, GS_BM * GS_BN, 0, stream>>>( \
    A, lda, W, ldw, R, ldr, C, ldc, M, N, K, gain, eps)
  if (gain && gate) FUSED(true, true);
  else if (gain) FUSED(true, false);
  else FUSED(false, true);
#undef FUSED
  return tis_launch_status("gemm_plain_fused");
}
