// Matrix product for long prompts: C[M, N] = A[M, K] * W[N, K]^T, bf16 operands, float accumulation, in tiles of 256x256 by eight
// wavefronts of which four multiply while the other four read shared memory.
//
// What bounds it: the card's power.  With every compute unit busy on random operands the clock falls until a product takes the same
// energy a second; the same code on zeros runs 1.3 to 1.4 times as fast (1.9 PFLOP/s), and on 64 units alone at 0.9 us a stage of 64 k,
// 96 % of the matrix cores' rate.  So what pays is less energy a product:
//   * 16x16x32 instructions instead of 32x32x16 (half the reads and writes of accumulators for twice the operand reads):
//     9,681 rows x 8,192 gated x K = 3,072 722 -> 684 us, though on 64 units it is 6 % slower;
//   * neighbouring instructions share the activations' fragment and change the weights': -> 669 (the other way round 683);
//   * no raised priority for the wavefronts that multiply: 693 -> 684.
// Tiles are 256x256 since a wavefront of 128x64 reads the least shared memory that its registers (128 of accumulators, 96 of
// fragments) allow.  The tile's two operands are staged as four regions of a stage, 128 rows of 64 k each: a region is free, and asked
// for again, as soon as its fragments are in registers, 3.5 to 4.5 of a stage's four phases before it is needed.  Wavefronts w and
// w + 4 share a SIMD and run half a phase apart: a phase is the reads of six fragments of the next ones, a barrier, 16 instructions
// with the region's loads in the middle, a barrier.  Bytes go straight from global into shared memory; the waits are the kernel's own.
// Before (gemm_mfma's 256x256 tile: one barrier a stage, all wavefronts in step): 2,048 rows, 8,192 gated, K = 2,048 118 us, now 100;
// with K = 3,072 and 9,681 rows 824 us, now 665 (1.46 PFLOP/s).  Walking 4 row tiles together instead of 8: equal;
// 16: gated 2,048 rows equal, 9,681 rows 663 against 652, 8,192 cubed 780 against 720.
#include "gemm_duo.h"

// x * sigmoid(x) with the hardware's exponential and reciprocal, as gemm_mfma has it: off by at most 2^-23 (|x| + 2) of itself, an ulp of
// each and the rounding of x * log2(e) in front of the first, far below the rounding to bfloat16 behind it.  Gate and up are float here;
// the library's product and the pass behind it round them to bfloat16 first (2,048 rows, K = 3,072, against 64 bits: 1.66e-3, so 3.09e-3;
// of gates below -4 alone 1.5e-3 and 6.1e-3).
__device__ __forceinline__ float gd_silu(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.4426950408889634f));
}
// the tanh form of GELU, z/2 (1 + tanh(a)) with a = sqrt(2/pi) (z + 0.044715 z^3): (1 + tanh(a)) / 2 = sigmoid(2a)
__device__ __forceinline__ float gd_gelu(float x) {
  const float a = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(a * -2.8853900817779268f));
}

// mode 3: the columns are query heads, then key heads and value heads of hd lanes each; queries and keys turn in adjacent pairs
// behind the product, keys and values go to their pages.
struct GdRope {
  const int *positions, *token_seq, *block_table;
  const float* cos_sin;                      // [positions][hd / 2][2]
  bf16 *kcache, *vcache;
  int table_width, page_size, nh, nkv, hd, store;
};

template <int MODE>
struct GdTile {
  const char *a, *b;
  int rows, columns;                         // that exist, from the tile's first on: those beyond are the last one again
  uint32_t up;                               // bytes from a gate row to its up row
  int lda, ldw;
  bool gated;
  __device__ __forceinline__ uint32_t row(int m) const { return (uint32_t)(min(m, rows - 1) * lda) * 2u; }
  __device__ __forceinline__ uint32_t column(int r, int h) const {
    const int n = min(gated ? r : r / 32 * 64 + h * 32 + r % 32, columns - 1);
    return (uint32_t)n * (uint32_t)ldw * 2u + (gated && h ? up : 0u);
  }
};

template <int MODE, int TILES, typename TC>
__device__ __forceinline__ void gd_store(const gd_f32x4 (&acc)[TILES][4], TC* C, int ldc, int m0, int M, int n0, int N, int l16, int quad) {
#pragma unroll
  for (int i = 0; i < TILES; ++i) {
    const int m = m0 + i * 16 + l16;
    if (sizeof(TC) == 4) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + j * 16 + quad * 4;
        if (m < M && n < N) *reinterpret_cast<float4*>(C + (size_t)m * ldc + n) = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < (MODE != 0 ? 2 : 4); j += 2) {
      float v[2][4];
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float z = acc[i][j + x][e];
          v[x][e] = MODE == 1 ? gd_silu(z) * acc[i][2 + x][e] : MODE == 2 ? gd_gelu(z) * acc[i][2 + x][e] : z;
        }
      const uint4 eight = gd_eight(v);
      const int n = n0 + (j + (quad & 1)) * 16 + (quad >> 1) * 8;
      if (m < M && n < N) *reinterpret_cast<uint4*>(C + (size_t)m * ldc + n) = eight;
    }
  }
}

// Rows of 16 lanes are tokens: their positions and pages lie in shared memory (page < 0: not stored).  A tile of 16 columns is of one
// head (head sizes are multiples of 16).  Queries and keys leave as eight neighbours a lane like every other result; a value's store is
// a run of 16 tokens, two bytes each.
template <int TILES>
__device__ __forceinline__ void gd_store_rope(const gd_f32x4 (&acc)[TILES][4], bf16* C, int ldc, const int* pos_of, const int* page_of, int first,
                                              int m0, int M, int n0, int N, const GdRope& rope, int l16, int quad) {
  const int hd = rope.hd, n_turning = (rope.nh + rope.nkv) * hd, ps = rope.page_size;
  // the next rows' angles are asked for ahead of these rows' stores (one after another they took 12 us a tile)
  int lane_of[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) lane_of[j] = (n0 + j * 16) % hd + quad * 4;
  float4 angles[2][4];
  auto ask = [&](int i) {
    const float* row = rope.cos_sin + (size_t)pos_of[first + i * 16 + l16] * hd;
#pragma unroll
    for (int j = 0; j < 4; ++j) angles[i & 1][j] = *reinterpret_cast<const float4*>(row + lane_of[j]);
  };
  ask(0);
#pragma unroll
  for (int i = 0; i < TILES; ++i) {
    const int r = first + i * 16 + l16, m = m0 + r;
    const int pos = pos_of[r], page = page_of[r], slot = pos % ps;
    if (i + 1 < TILES) ask(i + 1);
#pragma unroll
    for (int j = 0; j < 4; j += 2) {
      float v[2][4];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const int tile = n0 + (j + x) * 16, head = tile / hd, d = lane_of[j + x];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[x][e] = acc[i][j + x][e];
        if (tile < n_turning) {
          const float4 cs = angles[i & 1][j + x];
          v[x][0] = acc[i][j + x][0] * cs.x - acc[i][j + x][1] * cs.y;
          v[x][1] = acc[i][j + x][0] * cs.y + acc[i][j + x][1] * cs.x;
          v[x][2] = acc[i][j + x][2] * cs.z - acc[i][j + x][3] * cs.w;
          v[x][3] = acc[i][j + x][2] * cs.w + acc[i][j + x][3] * cs.z;
        } else if (tile < N && m < M && page >= 0) {
          bf16* to = rope.vcache + (((size_t)page * rope.nkv + (head - rope.nh - rope.nkv)) * hd + d) * ps + slot;
#pragma unroll
          for (int e = 0; e < 4; ++e) to[(size_t)e * ps] = from_float<bf16>(v[x][e]);
        }
      }
      const uint4 eight = gd_eight(v);
      const int n = n0 + (j + (quad & 1)) * 16 + (quad >> 1) * 8, head = n / hd;
      if (m >= M || n >= n_turning) continue;
      if (head < rope.nh) *reinterpret_cast<uint4*>(C + (size_t)m * ldc + n) = eight;
      else if (page >= 0) *reinterpret_cast<uint4*>(rope.kcache + (((size_t)page * rope.nkv + (head - rope.nh)) * ps + slot) * hd + (n - head * hd)) = eight;
    }
  }
}

// Gated modes: columns of tiles from `gate_tiles` on are a plain product of the rows behind the up rows, C2 [M, N2] (n_tiles counts both).
struct GdBeside {
  bf16* C;
  int N, ldc, gate_tiles;
};

// Tiles in the order in which they are walked: [0, whole) as whole ones, the rest of the m_tiles x n_tiles as two halves each, and
// behind them, where `tail`, a row of halves below the last row of tiles.
template <int MODE, typename TC>
__global__ void __launch_bounds__(512, 2)
    gemm_duo_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W, TC* __restrict__ C, int M, int N, int K, int lda, int ldw,
                    int ldc, int m_tiles, int n_tiles, int whole, int k_per_group, GdRope rope, GdBeside beside) {
  constexpr bool GATED = MODE == 1 || MODE == 2;
  constexpr int OUT = GATED ? GD_TILE / 2 : GD_TILE;       // output columns of a tile
  __shared__ __attribute__((aligned(1024))) unsigned char lds[9 * GD_REGION];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / BLM_WAVE), lane = tid & (BLM_WAVE - 1);
  const int l16 = lane & 15, quad = lane >> 4, wm = wave >> 2, wn = wave & 3;      // wavefronts w and w + 4 share a SIMD

  // neighbouring blocks go to different dies: each die gets a run of the tiles
  const bool half = (int)blockIdx.x >= whole;
  int tm, tn, below = 0;
  {
    const int total = half ? (int)gridDim.x - whole : whole, b = half ? (int)blockIdx.x - whole : (int)blockIdx.x;
    const int die = b & 7, q = total >> 3, r = total & 7;
    int t = die * q + min(die, r) + (b >> 3);
    if (half) {
      below = (t & 1) * 128;
      t = whole + (t >> 1);
    }
    if (t >= m_tiles * n_tiles) {            // the tail's halves: two indices of t a column each
      tm = m_tiles;
      tn = (t - m_tiles * n_tiles) * 2 + below / 128;
      below = 0;
    } else {
      const int in_group = GD_GROUP * n_tiles, group = t / in_group, first = group * GD_GROUP;
      const int height = min(GD_GROUP, m_tiles - first);
      tm = first + (t - group * in_group) % height;
      tn = (t - group * in_group) / height;
    }
  }
  const bool plain = GATED && tn >= beside.gate_tiles;
  if (plain) tn -= beside.gate_tiles;
  const int m0 = tm * GD_TILE + below, n0 = tn * (plain ? GD_TILE : OUT), k0 = blockIdx.y * k_per_group, stages = min(k_per_group, K - k0) / GD_BK;
  if (m0 >= M) return;                       // a second half that has no rows
  C += (size_t)blockIdx.y * M * ldc;
  const GdTile<MODE> t = {reinterpret_cast<const char*>(A + (size_t)m0 * lda + k0), reinterpret_cast<const char*>(W + (size_t)(n0 + (plain ? 2 * N : 0)) * ldw + k0),
                          M - m0, (plain ? beside.N : N) - n0, (uint32_t)N * (uint32_t)ldw * 2u, lda, ldw, GATED && !plain};
  const int n = n0 + wn * (GATED && !plain ? 32 : 64);
  if constexpr (MODE == 3) {
    __shared__ int pos_of[GD_TILE], page_of[GD_TILE];
    if (tid < GD_TILE) {
      const int m = min(m0 + tid, M - 1), seq = rope.token_seq[m], pos = rope.positions[m];
      pos_of[tid] = pos;
      page_of[tid] = seq < 0 || !rope.store ? -1 : rope.block_table[(size_t)seq * rope.table_width + pos / rope.page_size];
    }
    if (!half) {                             // the product's first barriers lie between these writes and the reads behind it
      gd_f32x4 acc[8][4];
      gd_whole(acc, t, stages, lds, wave, lane);
      gd_store_rope(acc, C, ldc, pos_of, page_of, wm * 128, m0, M, n, N, rope, l16, quad);
    } else {
      gd_f32x4 acc[4][4];
      gd_part<4>(acc, t, stages, lds, wave, lane);
      gd_store_rope(acc, C, ldc, pos_of, page_of, wm * 64, m0, M, n, N, rope, l16, quad);
    }
  } else if (!half) {
    gd_f32x4 acc[8][4];
    gd_whole(acc, t, stages, lds, wave, lane);
    if (GATED && plain) gd_store<0, 8, bf16>(acc, beside.C, beside.ldc, m0 + wm * 128, M, n, beside.N, l16, quad);
    else gd_store<MODE, 8, TC>(acc, C, ldc, m0 + wm * 128, M, n, N, l16, quad);
  } else {
    gd_f32x4 acc[4][4];
    gd_part<4>(acc, t, stages, lds, wave, lane);
    if (GATED && plain) gd_store<0, 4, bf16>(acc, beside.C, beside.ldc, m0 + wm * 64, M, n, beside.N, l16, quad);
    else gd_store<MODE, 4, TC>(acc, C, ldc, m0 + wm * 64, M, n, N, l16, quad);
  }
}

// A plain product in tiles of 160 rows and 256 columns: 0.71 of a whole tile's time, for rounds that neither whole tiles nor halves fill
// (2,166 rows of 2,048 columns in two groups of K are 272 halves for 256 units, or 224 of these).  Products of planes, us: [2048, 8192], 2,166
// rows, two groups 64.9 (1.12 PFLOP/s; halves 97.8, the library's product without planes 74.7), 1,200 rows, four groups 42.3 (55.3; 53.9).
template <typename TC>
__global__ void __launch_bounds__(512, 2)
    gemm_five_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W, TC* __restrict__ C, int M, int N, int K, int lda, int ldw,
                     int ldc, int m_tiles, int n_tiles, int k_per_group) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[3 * GdPart<5>::STAGE];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / BLM_WAVE), lane = tid & (BLM_WAVE - 1);
  const int total = gridDim.x, die = blockIdx.x & 7, q = total >> 3, r = total & 7, at = die * q + min(die, r) + (blockIdx.x >> 3);
  const int in_group = GD_GROUP * n_tiles, group = at / in_group, first = group * GD_GROUP, height = min(GD_GROUP, m_tiles - first);
  const int m0 = (first + (at - group * in_group) % height) * GdPart<5>::ROWS, n0 = (at - group * in_group) / height * GD_TILE;
  const int k0 = blockIdx.y * k_per_group, stages = min(k_per_group, K - k0) / GD_BK;
  C += (size_t)blockIdx.y * M * ldc;
  const GdTile<0> t = {reinterpret_cast<const char*>(A + (size_t)m0 * lda + k0), reinterpret_cast<const char*>(W + (size_t)n0 * ldw + k0), M - m0, N - n0, 0, lda, ldw, false};
  gd_f32x4 acc[5][4];
  gd_part<5>(acc, t, stages, lds, wave, lane);
  gd_store<0, 5, TC>(acc, C, ldc, m0 + (wave >> 2) * 80, M, n0 + (wave & 3) * 64, N, lane & 15, lane >> 4);
}

// mode 0: C[M, N] = A W^T, W [N, K].  mode 1: W [2N, K] = [gate rows; up rows], C[M, N] = silu(gate) * up; mode 2: the tanh form of
// GELU in place of silu.  k_groups > 1: C is float [k_groups, M, ldc], a partial product over each group's stretch of K (a multiple
// of 128).  whole: how many of the tiles are run as whole ones, the others as halves.  fives (mode 0): tiles of 160 rows, whole is 0.
static int gd_run(const void* A, const void* W, void* C, int c_dtype, int M, int N, int K, int lda, int ldw, int ldc, int mode,
                  int k_groups, int whole, bool fives, const GdRope* rope, GdBeside beside, hipStream_t stream) {
  BLM_REQUIRE(M >= 1 && N >= 8 && N % 8 == 0 && K >= 256 && K % 128 == 0, "gemm_duo: sizes M=%d N=%d K=%d not supported", M, N, K);
  BLM_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && ldc % 8 == 0 && lda >= K && ldw >= K && ldc >= (rope ? rope->nh * rope->hd : N), "gemm_duo: bad strides lda=%d ldw=%d ldc=%d",
              lda, ldw, ldc);
  BLM_REQUIRE(((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0 && ((uintptr_t)C % 16) == 0, "gemm_duo: operands must be 16-byte aligned");
  BLM_REQUIRE(mode >= 0 && mode <= 2 && (c_dtype == BLM_BF16 || (c_dtype == BLM_F32 && mode == 0)), "gemm_duo: mode %d, dtype %d", mode, c_dtype);
  const int k_per_group = k_groups >= 1 ? ((K + k_groups - 1) / k_groups + 127) / 128 * 128 : 0;
  BLM_REQUIRE(k_groups >= 1 && k_groups <= 64 && (k_groups == 1 || c_dtype == BLM_F32) && K - (k_groups - 1) * k_per_group >= 256,
              "gemm_duo: %d groups of K=%d need 256 each and a float output", k_groups, K);
  BLM_REQUIRE((size_t)256 * lda * 2 < ((size_t)1 << 32) && ((size_t)(mode != 0 ? 2 : 1) * N + beside.N) * ldw * 2 < ((size_t)1 << 32),
              "gemm_duo: matrices of 4 GiB and more are not supported (lda=%d, N=%d, ldw=%d)", lda, N, ldw);
  const int columns = mode != 0 ? GD_TILE / 2 : GD_TILE;
  beside.gate_tiles = (N + columns - 1) / columns;
  const int n_tiles = beside.gate_tiles + (beside.N + GD_TILE - 1) / GD_TILE;
  if (fives) {
    BLM_REQUIRE(whole == 0 && mode == 0, "gemm_duo: %d whole tiles of 0, mode %d", whole, mode);
    const int rows = GdPart<5>::ROWS, five_tiles = (M + rows - 1) / rows;
    BLM_REQUIRE((long long)five_tiles * n_tiles < (1LL << 30), "gemm_duo: too many tiles");
    const dim3 grid((unsigned)(five_tiles * n_tiles), (unsigned)k_groups);
    if (c_dtype == BLM_F32)
      hipLaunchKernelGGL(gemm_five_kernel<float>, grid, dim3(512), 0, stream, (const bf16*)A, (const bf16*)W, (float*)C, M, N, K, lda, ldw, ldc,
                         five_tiles, n_tiles, k_per_group);
    else
      hipLaunchKernelGGL(gemm_five_kernel<bf16>, grid, dim3(512), 0, stream, (const bf16*)A, (const bf16*)W, (bf16*)C, M, N, K, lda, ldw, ldc,
                         five_tiles, n_tiles, k_per_group);
    BLM_LAUNCH_CHECK("gemm_five");
    return 0;
  }
  const bool tail = M % GD_TILE != 0 && M % GD_TILE <= GD_TILE / 2;
  const int m_tiles = tail ? M / GD_TILE : (M + GD_TILE - 1) / GD_TILE;
  BLM_REQUIRE((long long)(m_tiles + 1) * n_tiles < (1LL << 29), "gemm_duo: too many tiles");
  BLM_REQUIRE(whole >= 0 && whole <= m_tiles * n_tiles, "gemm_duo: %d whole tiles of %d", whole, m_tiles * n_tiles);
  const int halves = 2 * (m_tiles * n_tiles - whole) + (tail ? n_tiles : 0);
  const dim3 grid((unsigned)(whole + halves), (unsigned)k_groups), block(512);
#define GD_LAUNCH(MODE, TC)                                                                                                        \
  hipLaunchKernelGGL((gemm_duo_kernel<MODE, TC>), grid, block, 0, stream, (const bf16*)A, (const bf16*)W, (TC*)C, M, N, K, lda, ldw, \
                     ldc, m_tiles, n_tiles, whole, k_per_group, rope ? *rope : GdRope{}, beside)
  if (rope) GD_LAUNCH(3, bf16);
  else if (mode == 1) GD_LAUNCH(1, bf16);
  else if (mode == 2) GD_LAUNCH(2, bf16);
  else if (c_dtype == BLM_F32) GD_LAUNCH(0, float);
  else GD_LAUNCH(0, bf16);
#undef GD_LAUNCH
  BLM_LAUNCH_CHECK("gemm_duo");
  return 0;
}

extern "C" int blm_gemm_duo(const void* A, const void* W, void* C, int c_dtype, int M, int N, int K, int lda, int ldw, int ldc, int mode,
                            int k_groups, int whole, int fives, hipStream_t stream) {
  return gd_run(A, W, C, c_dtype, M, N, K, lda, ldw, ldc, mode, k_groups, whole, fives != 0, nullptr, GdBeside{}, stream);
}

// A gated product (mode 1 or 2) with a plain one of the same rows beside it: W [2N + N2, K], C2[M, N2] the product with the last N2
// rows.  Its tiles fill what the gated ones leave of the last round (2,166 rows, 8,192 gated and 2,048 beside, K = 2,048: 118 us
// and 31 apart).
extern "C" int blm_gemm_duo_beside(const void* A, const void* W, void* C, void* C2, int M, int N, int N2, int K, int lda, int ldw, int ldc, int ldc2,
                                   int mode, int whole, hipStream_t stream) {
  BLM_REQUIRE((mode == 1 || mode == 2) && N2 > 0 && N2 % 8 == 0 && ldc2 >= N2 && ldc2 % 8 == 0 && ((uintptr_t)C2 % 16) == 0,
              "gemm_duo_beside: mode %d, %d columns in rows of %d not supported", mode, N2, ldc2);
  return gd_run(A, W, C, BLM_BF16, M, N, K, lda, ldw, ldc, mode, 1, whole, false, nullptr, GdBeside{(bf16*)C2, N2, ldc2, 0}, stream);
}

// The q/k/v projection with the rotation of queries and keys (on the float results) and the write of keys and values into their
// pages.  qkv_out [M][ldq]: the queries.  Instead of a pass of its own over queries, keys and values (2,048 rows of 3,072: 8.9 us).
extern "C" int blm_gemm_duo_qkv_rope(const void* A, const void* W, void* qkv_out, const int* positions, const int* token_seq,
                                     const int* block_table, int table_width, const float* cos_sin, void* kcache, void* vcache, int page_size,
                                     int M, int K, int lda, int ldw, int ldq, int nh, int nkv, int hd, int store, int whole, hipStream_t stream) {
  BLM_REQUIRE(nh > 0 && nkv > 0 && hd > 0 && hd % 16 == 0 && page_size > 0 && table_width > 0, "gemm_duo_qkv_rope: head size %d not supported (a multiple of 16)", hd);
  BLM_REQUIRE(((uintptr_t)kcache % 16) == 0 && ((uintptr_t)cos_sin % 16) == 0, "gemm_duo_qkv_rope: pages and angles must be 16-byte aligned");
  const GdRope rope{positions, token_seq, block_table, cos_sin, (bf16*)kcache, (bf16*)vcache, table_width, page_size, nh, nkv, hd, store};
  return gd_run(A, W, qkv_out, BLM_BF16, M, (nh + 2 * nkv) * hd, K, lda, ldw, ldq, 0, 1, whole, false, &rope, GdBeside{}, stream);
}
