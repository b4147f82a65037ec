// Decode: a layer's last product with the residual's add and the next norm's row sums behind it.
//
//   h[m, n] += x W^T[m, n]            (operands on the matrix cores, float sums, h float32)
//   y[m, n]  = h[m, n] * gamma[n]     (rounded once, to x's type)
//   sums[m, b] = the sum of h[m, n]^2 over the columns of block b
//
// The norm's factor 1 / sqrt(mean(h^2) + eps) is one number a row, so the product that reads y multiplies its own float sums by it
// (row_scale.h) and no kernel stands between the two products.  Up to eight rows, bfloat16 or float32.
//
// A decode step's norm is a kernel of a block per row whose 2.6 to 3.5 us are a launch and trips to memory.  What bounds this kernel is
// the weights' stream, as without the norm; for the sums to be whole where they meet, a block has all of K for its columns, as few
// of them as make a block for every compute unit (2,048 columns in 256 blocks of eight, 3,072 of twelve, 4,096 of sixteen).
// Weights are packed for tiles of 16 columns (gemv_mfma.hip): eight columns are 128 bytes of every 256, whole cache lines.  Blocks of
// eight columns and rows take two steps along K in one matrix instruction: rows 8 to 15 of the first operand are the same rows one step on,
// columns 8 to 15 of the second the same columns one step on, and the result's two diagonal quarters are the two steps' products.
// Output projection, gate/up, down and q/k/v of a layer with both norms, us, norms as kernels / here (graph of 16 layers' weights):
// width 2048, inner 8192 1 row 34.8 / 29.6, 4 rows 36.4 / 31.2, 8 rows 37.4 / 33.2; width 3072 50.5 / 43.6, 52.4 / 45.6, 54.5 / 48.0;
// width 4096, inner 14336 87.0 / 80.0, 87.9 / 80.7, 90.0 / 82.6; width 1024, inner 4096 20.9 / 16.3, 22.5 / 18.1, 22.9 / 19.9.  This kernel
// alone against the planes of two groups of K: [2048, 2048] 4.13 / 4.14, 8 rows 4.19 / 4.45; [2048, 8192] 8.2 / 8.2, 8 rows 8.9 / 9.6 (4.2
// and 3.9 TB/s); [3072, 8192] 11.6 / 10.8 and 12.2 / 11.6 (4.7 and 4.3 TB/s).
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t gj_piece;      // 16 bytes

#define GJ_ROWS 8
#define GJ_BLOCKS 256
#define GJ_WAVES 8

// CH fragments of 16 bytes of both operands, added to the sums
template <int CH>
__device__ __forceinline__ f32x4_t gj_multiply(const gj_piece (&a)[CH], const gj_piece (&w)[CH], f32x4_t sum, bf16) {
#pragma unroll
  for (int s = 0; s < CH; ++s)
    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[s]), __builtin_bit_cast(bf16x8_t, w[s]), sum, 0, 0, 0);
  return sum;
}
// float32 in eight chains, as gemv_f32 (gemm_f32.hip) sums: no more than 16 to 32 products in a row before they meet their neighbours
template <int CH>
__device__ __forceinline__ f32x4_t gj_multiply(const gj_piece (&a)[CH], const gj_piece (&w)[CH], f32x4_t sum, float) {
  f32x4_t acc[8];
#pragma unroll
  for (int x = 0; x < 8; ++x) acc[x] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < CH; ++s) {
    const f32x4_t x = __builtin_bit_cast(f32x4_t, a[s]), y = __builtin_bit_cast(f32x4_t, w[s]);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[(s & 1) * 4 + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], acc[(s & 1) * 4 + e], 0, 0, 0);
  }
#pragma unroll
  for (int x = 4; x; x >>= 1)
#pragma unroll
    for (int y = 0; y < x; ++y) acc[y] += acc[y + x];
  return sum + acc[0];
}

// (What the first loads need stands in the arguments' first fourteen dwords, which come in registers.)
// STEPS: steps along K per wavefront, of four fragments' 16 bytes (32 bfloat16, 16 float32), two at once with PAIR; CH: loaded at once; WHOLE: the
// wavefronts' steps are all there
template <typename T, bool PAIR, int STEPS, int CH, bool WHOLE>
__global__ void __launch_bounds__(GJ_WAVES* BLM_WAVE)
    gemv_join_kernel(const T* __restrict__ A, const T* __restrict__ Wp, int M, int K, int lda, int k_steps, int columns, int blocks,
                     int n_waves, int N, float* __restrict__ h, const float* __restrict__ gamma, T* __restrict__ y, float* __restrict__ sums) {
  constexpr int EACH = PAIR ? 2 : 1, NC = STEPS / CH, E = 16 / sizeof(T), STEP = 4 * E;
  __shared__ float red[GJ_WAVES][EACH][GJ_ROWS][16 / EACH];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / BLM_WAVE), lane = threadIdx.x & (BLM_WAVE - 1);
  const int i16 = lane & 15, kg = lane >> 4;
  const int sub = PAIR ? i16 >> 3 : 0;                         // the step of a pair that this lane brings
  const int row = PAIR ? i16 & 7 : i16;                        // (rows past the last are the last once more; their sums go nowhere)
  // neighbouring blocks, which may share lines of the weights, on one die
  const int block = blocks % 8 == 0 ? (blockIdx.x % 8) * (blocks / 8) + blockIdx.x / 8 : blockIdx.x;
  const int n0 = block * columns, n = n0 + (PAIR ? i16 & 7 : min(i16, columns - 1));
  const T* wt = Wp + ((size_t)(n >> 4) * k_steps * 64 + kg * 16 + (n & 15)) * E;
  const T* ap = A + (size_t)min(row, M - 1) * lda;
  const int first = wave * STEPS * EACH, step0 = first + sub;
  // the block's outputs: a thread each, 16 to a row
  const int om = threadIdx.x >> 4, oc = threadIdx.x & 15;
  const bool own = om < M && oc < columns;
  f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
  float h_old = 0.f, g = 0.f;
  gj_piece a[2][CH], w[2][CH];
  auto at = [](int place, int last) { return WHOLE ? place : min(place, last); };
  auto load = [&](int c, int to) {
#pragma unroll
    for (int s = 0; s < CH; ++s) a[to][s] = *reinterpret_cast<const gj_piece*>(ap + at((step0 + (c * CH + s) * EACH) * STEP + kg * E, K - E));
#pragma unroll
    for (int s = 0; s < CH; ++s) w[to][s] = __builtin_nontemporal_load(reinterpret_cast<const gj_piece*>(wt + (size_t)at(step0 + (c * CH + s) * EACH, k_steps - 1) * (64 * E)));
  };
  load(0, 0);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (c + 1 < NC) load(c + 1, (c + 1) & 1);
    else if (own) {
      h_old = h[(size_t)om * N + n0 + oc];
      g = gamma[n0 + oc];
    }
    __builtin_amdgcn_sched_barrier(0);
    if (!WHOLE && (first + (c + 1) * CH * EACH) * STEP > K) {      // behind the end of K both count as zeros (an infinite one would make no number)
      const gj_piece zero = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int s = 0; s < CH; ++s) {
        const bool keep = (step0 + (c * CH + s) * EACH) * STEP + kg * E < K;
        a[c & 1][s] = keep ? a[c & 1][s] : zero;
        w[c & 1][s] = keep ? w[c & 1][s] : zero;
      }
    }
    sum = gj_multiply<CH>(a[c & 1], w[c & 1], sum, T{});
    asm volatile("" : "+v"(sum));          // added up here: left alone, the chains of all chunks wait in registers for the end
    __builtin_amdgcn_sched_barrier(0);
  }
  // sum[r]: row kg * 4 + r, column i16 of the result
  if (PAIR ? (kg >> 1) == sub : kg < 2) {
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][sub][(kg & 1) * 4 + r][PAIR ? i16 & 7 : i16] = sum[r];
  }
  __syncthreads();
  if (threadIdx.x < GJ_ROWS * 16) {
    float t = 0.f;
    for (int x = 0; x < n_waves; ++x) {
      const float* r = &red[x][0][om][PAIR ? oc & 7 : oc];
      t += PAIR ? r[0] + r[GJ_ROWS * 8] : r[0];
    }
    t += h_old;
    float ss = own ? t * t : 0.f;
    ss += blm_dpp<BLM_DPP_XOR1>(ss);
    ss += blm_dpp<BLM_DPP_XOR2>(ss);
    ss += blm_dpp<BLM_DPP_HALF_MIRROR>(ss);
    ss += blm_dpp<BLM_DPP_MIRROR>(ss);
    if (own) {
      h[(size_t)om * N + n0 + oc] = t;
      y[(size_t)om * N + n0 + oc] = from_float<T>(t * g);
      if (oc == 0) sums[(size_t)om * blocks + block] = ss;
    }
  }
}

// Columns of a block, which has all of K: the fewest from eight to sixteen that cut N into at most GJ_BLOCKS blocks, a multiple of
// four of them; 0: none.
extern "C" int blm_gemv_join_columns(int dtype, int M, int N, int K) {
  const int piece = dtype == BLM_F32 ? 4 : 8;
  if (M < 1 || M > GJ_ROWS || N < 16 || N % 16 != 0 || K < piece || K % piece != 0 || K > 16384) return 0;
  for (int c = 8; c <= 16; ++c)
    if (N % (4 * c) == 0 && N / c <= GJ_BLOCKS) return c;
  return 0;
}

template <typename T, int CH>
static void gj_launch(const void* A, const void* Wp, float* h, const float* gamma, void* y, float* sums, int M, int N, int K, int lda,
                      int columns, hipStream_t stream) {
  const int step = 64 / (int)sizeof(T), k_steps = (K + step - 1) / step;
#define BLM_GJ(PAIR, STEPS, CH)                                                                                              \
  do {                                                                                                                       \
    const int per = STEPS * (PAIR ? 2 : 1), waves = (k_steps + per - 1) / per;                                               \
    const int blocks = N / columns, at_work = waves < 2 ? 2 : waves;                                                         \
    if (waves > 1 && waves * per * step == K)                                                                                \
      hipLaunchKernelGGL((gemv_join_kernel<T, PAIR, STEPS, CH, true>), dim3(blocks), dim3(at_work * BLM_WAVE), 0, stream,    \
                         (const T*)A, (const T*)Wp, M, K, lda, k_steps, columns, blocks, at_work, N, h, gamma, (T*)y, sums); \
    else                                                                                                                     \
      hipLaunchKernelGGL((gemv_join_kernel<T, PAIR, STEPS, CH, false>), dim3(blocks), dim3(at_work * BLM_WAVE), 0, stream,   \
                         (const T*)A, (const T*)Wp, M, K, lda, k_steps, columns, blocks, at_work, N, h, gamma, (T*)y, sums); \
  } while (0)
  if (columns == 8) {
    if (k_steps <= 128) BLM_GJ(true, 8, 8);
    else if (k_steps <= 256) BLM_GJ(true, 16, CH);
    else if (k_steps <= 512) BLM_GJ(true, 32, 8);
    else BLM_GJ(true, 64, 8);
  } else {
    if (k_steps <= 64) BLM_GJ(false, 8, 8);
    else if (k_steps <= 128) BLM_GJ(false, 16, CH);
    else if (k_steps <= 256) BLM_GJ(false, 32, 8);
    else if (k_steps <= 512) BLM_GJ(false, 64, 8);
    else BLM_GJ(false, 128, 8);
  }
#undef BLM_GJ
}

// Wp: the packed copy of W[N, K] (gemv_mfma.hip, gemm_f32.hip).  h [M, N] and gamma [N] float32, y [M, N] of the operands' type, sums
// [M, N / columns].
extern "C" int blm_gemv_join(const void* A, int dtype, const void* Wp, float* h, const float* gamma, void* y, float* sums, int M, int N,
                             int K, int lda, hipStream_t stream) {
  BLM_REQUIRE(dtype == BLM_F32 || dtype == BLM_BF16, "gemv_join: unsupported dtype %d", dtype);
  const int columns = blm_gemv_join_columns(dtype, M, N, K);
  BLM_REQUIRE(columns > 0, "gemv_join: M=%d N=%d K=%d not supported", M, N, K);
  BLM_REQUIRE(lda % (dtype == BLM_F32 ? 4 : 8) == 0 && lda >= K, "gemv_join: bad stride lda=%d", lda);
  BLM_REQUIRE(((uintptr_t)A % 16) == 0 && ((uintptr_t)Wp % 16) == 0, "gemv_join: operands must be 16-byte aligned");
  if (dtype == BLM_F32) gj_launch<float, 8>(A, Wp, h, gamma, y, sums, M, N, K, lda, columns, stream);
  else gj_launch<bf16, 16>(A, Wp, h, gamma, y, sums, M, N, K, lda, columns, stream);
  BLM_LAUNCH_CHECK("gemv_join");
  return 0;
}
