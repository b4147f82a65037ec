// The true 32-bit product C[M,N] = A[M,K] * W[N,K]^T on the matrix cores' float instructions (float operands, float
// products, float sums, nothing narrowed), with W as the checkpoint stores it (K contiguous).
//   gemm_f32 : many rows.  A block of four wavefronts owns a tile of 128x128, 128x64, 64x128 or 64x64 (gated:
//              128x128 or 64x128); K in steps of 32.
//   gemv_f32 : up to 16 rows (decode).  Streams a packed copy of the weights once, whole lines at a time.
// Both want K, lda and the rows' addresses in units of 16 bytes; other operands take gemm_tiled.
#include "common.h"
#include "row_scale.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

__device__ __forceinline__ float silu_times(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// ---------------------------------------------------------------------------------------------------------------------
// many rows: v_mfma_f32_32x32x2_f32.  Lane l supplies A[l % 32][l / 32] and B[l / 32][l % 32] and holds
// C[8 (v / 4) + 4 (l / 32) + v % 4][l % 32], v < 16.  Which two elements of K an instruction takes is free as long as both
// operands agree, so the lower half of a wavefront takes elements 8 s + 0..3 of a row and the upper half 8 s + 4..7: one
// 16-byte read of shared memory per row feeds four instructions.  Rows of 32 floats are unpadded, their 16-byte pieces
// permuted (piece j of row r at j ^ (r / 2 % 8)) so that the 16 rows that a quarter of a wavefront reads meet every bank.
// An instruction takes 64 cycles of a SIMD, a step of a 64x64 wavefront tile 64 of them, so loads through registers and one
// barrier per step hide behind the products; what bounds the kernel is the instructions' rate (157 TFLOP/s) and how evenly
// the tiles fill the compute units, which is why there are four tiles and K may be cut into groups (partial planes).
// Sums in two levels: the products of GC_CHUNK elements of K, then the chunks, so that the rounding error does not grow with
// K additions in a row.
// Direct loads from global into shared memory: staged through registers the same tiles took 12 % longer (the conversions of
// addresses, the zeroing and the writes stand in the wavefronts' instruction streams: 122 TFLOP/s against 139 at 2,048 rows).
// Measured (us, before: 128x128 tiles of eight wavefronts, scalar loads, whole K): 1,000 rows, [16384, 2048] with the gating
// that was a pass of its own 844 -> 502 (134 TFLOP/s); [2048, 8192] 960 -> 256 in two or four groups; [3072, 2048] 255 ->
// 101; 2,048 rows, [16384, 2048] 1,509 -> 984 (140 TFLOP/s).
// ---------------------------------------------------------------------------------------------------------------------
#define GC_BK 32
#define GC_CHUNK 128

// GATED: W is [gate rows; up rows] ([2 N, K]); the second half of a wavefront's columns are the up rows of its first half,
// and C = silu(gate) * up.
template <int WM, int WN, bool GATED>
__global__ void __launch_bounds__(256, 2)
    gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N, int K,
                    int lda, int ldc, int k_group, long long plane, int m_tiles, int n_tiles) {
  static_assert(!GATED || WN == 2, "a gated tile holds a gate and an up part per wavefront");
  constexpr int BM = 64 * WM, BN = 64 * WN, ROWS = BM + BN;
  constexpr int PER = ROWS / 32;                     // direct loads per wavefront and step: eight rows each
  __shared__ __attribute__((aligned(1024))) float tile[2][ROWS * GC_BK];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / BLM_WAVE), lane = tid & (BLM_WAVE - 1);
  // the row tiles of one column tile follow each other on one die (blocks go to the eight dies in turn), so that its L2
  // brings the weights of a column tile once
  const int die = blockIdx.x & 7, at = blockIdx.x >> 3;
  const int nt = (at / m_tiles) * 8 + die, mt = at % m_tiles;
  if (nt >= n_tiles) return;
  const int m0 = mt * BM, n0 = nt * (GATED ? BN / 2 : BN);
  const int k_begin = blockIdx.y * k_group, k_end = min(K, k_begin + k_group);

  // Rows (4 i + wave) 8 + 0..7 of the tile are this wavefront's i-th load; a lane brings 16 bytes.  Rows past the end of a
  // matrix are its last row again; nothing stores what comes of them.
  uint32_t lane_offset[PER];
  const char* base[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int r0 = (i * 4 + wave) * 8, r = r0 + lane / 8, piece = (lane & 7) ^ ((r >> 1) & 7);
    if (r0 < BM) {
      base[i] = reinterpret_cast<const char*>(A + (size_t)m0 * lda);
      lane_offset[i] = (uint32_t)min(r, M - 1 - m0) * (uint32_t)lda * 4u + piece * 16u;
    } else if (GATED) {      // per 64 columns of the tile (one wavefront column) 32 gate rows and their 32 up rows
      const int c0 = r0 - BM, n = (c0 / 64) * 32 + (r - BM) % 32;
      base[i] = reinterpret_cast<const char*>(W + ((size_t)n0 + (size_t)((c0 % 64) / 32) * N) * K);
      lane_offset[i] = (uint32_t)min(n, N - 1 - n0) * (uint32_t)K * 4u + piece * 16u;
    } else {
      base[i] = reinterpret_cast<const char*>(W + (size_t)n0 * K);
      lane_offset[i] = (uint32_t)min(r - BM, N - 1 - n0) * (uint32_t)K * 4u + piece * 16u;
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(blm_lds_ptr)&tile[0][0];
  auto fetch = [&](int k0, int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i)
      blm_dma16_to(base[i] + (size_t)k0 * 4, lane_offset[i], lds0 + (uint32_t)(buf * ROWS * GC_BK * 4 + (i * 4 + wave) * 1024));
  };
  // the last, partial step: through registers, zeros behind the end of K (which is a multiple of four)
  auto fetch_part = [&](int k0, int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int r = (i * 4 + wave) * 8 + lane / 8;
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (k0 + ((lane & 7) ^ ((r >> 1) & 7)) * 4 < k_end) v = *reinterpret_cast<const f32x4*>(base[i] + (size_t)k0 * 4 + lane_offset[i]);
      *reinterpret_cast<f32x4*>(&tile[buf][r * GC_BK + (lane & 7) * 4]) = v;
    }
  };

  const int wm = (wave >> 1) * 32 * WM, wn = (wave & 1) * 32 * WN;
  const int li = lane & 31, lk = lane >> 5;
  f32x16 total[WM][WN], acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) total[i][j][v] = acc[i][j][v] = 0.f;

  auto bring = [&](int k0, int buf) {
    if (k0 + GC_BK <= k_end) fetch(k0, buf);
    else if (k0 < k_end) fetch_part(k0, buf);
  };
  auto meet = [&]() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  bring(k_begin, 0);
  meet();
  int buf = 0, in_chunk = 0;
  for (int k0 = k_begin; k0 < k_end; k0 += GC_BK, buf ^= 1) {
    bring(k0 + GC_BK, buf ^ 1);            // its last readers passed the barrier that ended the step before this one
    const float* a_rows = &tile[buf][(wm + li) * GC_BK];
    const float* w_rows = &tile[buf][(BM + wn + li) * GC_BK];
    const int twist = (li >> 1) & 7;       // the rows of a fragment lie 32 apart, so they share it
#pragma unroll
    for (int s = 0; s < GC_BK / 8; ++s) {
      f32x4 a[WM], w[WN];
      const int piece = ((2 * s + lk) ^ twist) * 4;
#pragma unroll
      for (int i = 0; i < WM; ++i) a[i] = *reinterpret_cast<const f32x4*>(a_rows + i * 32 * GC_BK + piece);
#pragma unroll
      for (int j = 0; j < WN; ++j) w[j] = *reinterpret_cast<const f32x4*>(w_rows + j * 32 * GC_BK + piece);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int j = 0; j < WN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][e], w[j][e], acc[i][j], 0, 0, 0);
    }
    in_chunk += GC_BK;
    if (in_chunk == GC_CHUNK || k0 + GC_BK >= k_end) {
      in_chunk = 0;
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            total[i][j][v] += acc[i][j][v];
            acc[i][j][v] = 0.f;
          }
    }
    meet();
  }
  float* out = C + (size_t)blockIdx.y * plane;
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = m0 + wm + i * 32 + 8 * (v >> 2) + 4 * lk + (v & 3);
      if (m >= M) continue;
      if (GATED) {
        const int n = n0 + wn / 2 + li;
        if (n < N) out[(size_t)m * ldc + n] = silu_times(total[i][0][v], total[i][WN - 1][v]);
      } else {
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          const int n = n0 + wn + j * 32 + li;
          if (n < N) out[(size_t)m * ldc + n] = total[i][j][v];
        }
      }
    }
}

// tile: 0 = 128x128, 1 = 128x64, 2 = 64x128, 3 = 64x64 (rows x columns; gated: tiles of 128 columns only, 64 pairs each).
// groups > 1: K in that many groups, C holds a plane of M * N for each (contiguous, ldc = N), which the reader adds up.
extern "C" int blm_gemm_f32(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldc, int gated,
                            int groups, int tile, hipStream_t stream) {
  BLM_REQUIRE(M > 0 && N > 0 && K > 0 && lda >= K && ldc >= N, "gemm_f32: bad sizes M=%d N=%d K=%d lda=%d ldc=%d", M, N, K, lda, ldc);
  BLM_REQUIRE(K % 4 == 0 && lda % 4 == 0 && ((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0,
              "gemm_f32: rows must start at multiples of 16 bytes and hold a multiple of four elements (K=%d lda=%d)", K, lda);
  BLM_REQUIRE(groups >= 1 && groups <= 64 && (groups == 1 || (!gated && ldc == N)), "gemm_f32: bad number of groups %d", groups);
  BLM_REQUIRE(tile >= 0 && tile <= 3 && (!gated || tile == 0 || tile == 2), "gemm_f32: bad tile %d", tile);
  const int bm = tile <= 1 ? 128 : 64, bn = tile == 0 || tile == 2 ? 128 : 64;
  const int m_tiles = (M + bm - 1) / bm, n_tiles = (N + (gated ? bn / 2 : bn) - 1) / (gated ? bn / 2 : bn);
  const long long blocks = (long long)m_tiles * ((n_tiles + 7) / 8 * 8);
  BLM_REQUIRE(blocks < 2147483647LL, "gemm_f32: too many tiles");
  const int k_group = ((K + groups - 1) / groups + GC_BK - 1) / GC_BK * GC_BK;
  dim3 grid((unsigned)blocks, (unsigned)groups), block(256);
#define BLM_GC(WM, WN, G)                                                                                              \
  hipLaunchKernelGGL((gemm_f32_kernel<WM, WN, G>), grid, block, 0, stream, (const float*)A, (const float*)W, (float*)C, \
                     M, N, K, lda, ldc, k_group, (long long)M * N, m_tiles, n_tiles)
  if (gated) {
    if (tile == 0) BLM_GC(2, 2, true);
    else BLM_GC(1, 2, true);
  } else {
    if (tile == 0) BLM_GC(2, 2, false);
    else if (tile == 1) BLM_GC(2, 1, false);
    else if (tile == 2) BLM_GC(1, 2, false);
    else BLM_GC(1, 1, false);
  }
#undef BLM_GC
  BLM_LAUNCH_CHECK("gemm_f32");
  return 0;
}

// ---------------------------------------------------------------------------------------------------------------------
// up to 16 rows: v_mfma_f32_16x16x4_f32 on a copy of the weights packed in the order the instruction wants them (as
// gemv_mfma.hip does for bfloat16; the instruction's lane l holds W[n0 + l % 16][k0 + l / 16], and which elements of K those
// are is free as long as the activations agree, so a lane takes four neighbours):
//     packed[((tile * k_steps + step) * 64 + lane) * 4 + e] = W[tile * 16 + lane % 16][step * 16 + lane / 16 * 4 + e]
// with N padded to a multiple of 16 and K to a multiple of 16 by zeros; every load of a wavefront is one contiguous kilobyte.
// Bound by the weights' bytes.  A block's wavefronts split K (or a group's stretch of it), keep their stretch of the
// activations in registers and walk the block's run of column tiles; the weights come in parts of eight steps, and a
// part's registers are asked for the part after the next as soon as the products that read them are issued.  The partial tiles meet in shared memory.
// Measured (us, 8 rows, [N, K], before: vector multiply-adds that read the activations again for every two columns):
// [2048, 2048] 8.3 -> 6.6 in two groups; [16384, 2048] gated 45 with the pass behind it -> 27.2 (4.9 TB/s); [2048, 8192]
// 28.3 -> 16.0 in four; [128256, 2048] 331 -> 162 (6.5 TB/s); 16 rows (before: 64x64 tiles) 284, 328, 1,270, 751 -> 6.8, 28.6,
// 16.8, 169.  Read from the checkpoint's layout by the 4x4x1 instruction instead (256 contiguous bytes of four
// rows per load, nothing packed): that instruction takes 32 cycles for the 64 weights of a load and four rows, so 16 rows
// took four times the cycles of this one: slower from 5 rows on, equal below.
// ---------------------------------------------------------------------------------------------------------------------
#define GV_MAX_WAVES 8

// KSTEPS: steps of 16 of K per wavefront.  WHOLE: every wavefront of every group has all of them, none partial, and nothing is
// tested on the way (the tests for steps that a wavefront does not have cost 0.25 us: [1000, 520] at 8 rows 4.86 -> 5.11;
// with them a decode step of 8 at the 1B shape took 1,547 us, so 1,533).  gated: a tile's columns are 8 gate rows and their 8 up rows, C = silu(gate) * up.
// ROPE: the columns are query heads, then key heads and value heads; queries and keys turn in adjacent pairs (two neighbouring
// lanes hold a pair's sums), keys and values go to their pages.  In place of a kernel of its own behind the product, 5 us of launch
// and look-ups (8 rows, [3072, 2048]: 8.9 + 5.3 us under the profiler, so 9.9); the rows' sequences and positions are asked for ahead of
// everything, their pages behind the weights.
struct GvRope {
  const int *positions, *token_seq, *block_table;
  const float2* cos_sin;
  float *kcache, *vcache;
  int table_width, page_size, nh, nkv, hd, store;
};

// SCALED: the rows come unscaled (row_scale.h), that many of them to a wavefront.  ONE: every block has one tile.
// The weights come by buffer loads of their tile's bytes: of none behind a block's last tile, where they bring zeros without a trip to memory.
// With a branch around them the compiler counts on the way without them, and every part waits for the next part's loads too.
// Us, eight rows, with the branch, selects of every activation and look-ups of the block's size / so: [3072, 2048] 9.2 / 8.1, [2048, 2048] in two groups
// 6.8 / 6.1, [16384, 2048] gated 27.0 / 26.0, [2048, 8192] in four 16.3 / 15.1; the head [128256, 2048], 31 tiles a block, 163 / 166
// (165.6 / 165.9 with the rest as it is: what it lost is not the loads').
// shape: 2 * wavefronts + gated, and the sums of a row that comes unscaled (the arguments' first fourteen dwords come in registers; a block's size would be a load).
template <int KSTEPS, bool WHOLE, bool ROPE, bool ONE, int SCALED>
__global__ void __launch_bounds__(GV_MAX_WAVES* BLM_WAVE)
    gemv_f32_kernel(const float* __restrict__ A, const float* __restrict__ Wp, int M, int K, int lda, int n_tiles, int k_steps, int shape,
                    int steps_per_group, int tiles_per_block, const float* __restrict__ sums, int N, int ldc, float* __restrict__ C, GvRope rope,
                    float inv_width, float eps) {
  __shared__ float red[GV_MAX_WAVES * 256];
  __shared__ float inv[RS_ROWS];
  RowScaleLoad<SCALED ? SCALED : 1> scale_load;
  __shared__ int pos_of[16], page_of[16];
  int my_pos = 0, my_seq = -1;
  if (ROPE && threadIdx.x < 16) {
    const int m = min((int)threadIdx.x, M - 1);
    my_pos = rope.positions[m];
    my_seq = rope.token_seq[m];
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / BLM_WAVE), lane = threadIdx.x & (BLM_WAVE - 1);
  const int n_waves = (shape >> 1) & 31, gated = shape & 1, n_sums = shape >> RS_SHIFT;
  const int row = lane & 15, kg = lane >> 4;
  const int group_begin = blockIdx.y * steps_per_group, group_end = min(k_steps, group_begin + steps_per_group);
  const int step0 = group_begin + wave * KSTEPS;
  const int kbase = step0 * 16 + kg * 4;
  C += (size_t)blockIdx.y * M * ldc;
  const float* ap = A + (size_t)min(row, M - 1) * lda;   // rows past the last are it once more; their sums go nowhere
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // activations first, then the first tile's weights behind them, all asked for before any is looked at; weights behind the end
  // of the group are some other step's (a step past the matrix is its last), and they and their activations count as zeros
  f32x4 a[KSTEPS];
  if (SCALED) scale_load.ask(sums, n_sums, M, wave, n_waves, lane);
#pragma unroll
  for (int s = 0; s < KSTEPS; ++s) a[s] = *reinterpret_cast<const f32x4*>(ap + min(kbase + s * 16, K - 4));
  const int tile_begin = blockIdx.x * tiles_per_block, tile_end = min(n_tiles, tile_begin + tiles_per_block);
  constexpr int PART = KSTEPS >= 16 ? 8 : 2, PARTS = KSTEPS / PART;      // steps whose weights wait in one set of registers
  const int wfirst = step0 * 1024 + lane * 16;
  auto tile_bytes = [&](int tile, bool there) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)(Wp + (size_t)tile * k_steps * 256), 0, there ? k_steps * 1024 : 0, 0x00027000);
  };
  auto weights = [&](auto bytes, int part, f32x4* w) {
#pragma unroll
    for (int s = 0; s < PART; ++s) w[s] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(bytes, wfirst + (part * PART + s) * 1024, 0, 2));
  };
  f32x4 w[2][PART];
  const auto first = tile_bytes(min(tile_begin, n_tiles - 1), true);
  weights(first, 0, w[0]);
  weights(first, 1, w[1]);
  __builtin_amdgcn_sched_barrier(0);
  if (SCALED) scale_load.finish(n_sums, inv_width, eps, M, wave, n_waves, lane, inv);
  if (ROPE && threadIdx.x < 16) {            // the barrier of the first tile's sum lies between these writes and their readers
    pos_of[threadIdx.x] = my_pos;
    page_of[threadIdx.x] = my_seq < 0 || !rope.store ? -1 : rope.block_table[(size_t)my_seq * rope.table_width + my_pos / rope.page_size];
  }
  if (!WHOLE)
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      const bool keep = (kbase + s * 16 < K) & (step0 + s < group_end);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[s][e] = keep ? a[s][e] : 0.f;
    }
  for (int tile = tile_begin; tile < (ONE ? min(tile_begin + 1, tile_end) : tile_end); ++tile) {
    const auto here = tile_bytes(tile, true), next = tile_bytes(tile + 1, !ONE && tile + 1 < tile_end);
    f32x4 sum[PARTS];
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
      // eight chains: an instruction does not wait for the one before it, and no sum has more than sixteen products in a
      // row before it meets its neighbours (with two chains over all steps the error against 64 bits was twice as large)
      f32x4 acc[8];
#pragma unroll
      for (int x = 0; x < 8; ++x) acc[x] = zero;
      if (!WHOLE && step0 + KSTEPS > group_end)        // zero activations alone would not do: an infinite weight would make them no numbers
#pragma unroll
        for (int s = 0; s < PART; ++s)
          if (step0 + p * PART + s >= group_end) w[p & 1][s] = zero;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < PART; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[(s & 1) * 4 + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[p * PART + s][e], w[p & 1][s][e], acc[(s & 1) * 4 + e], 0, 0, 0);
#pragma unroll
      for (int x = 0; x < 8; ++x) asm volatile("" : "+v"(acc[x]) : : "memory");      // the new loads stay behind the products whose registers they take
      __builtin_amdgcn_sched_barrier(0);
      if (p + 2 < PARTS) weights(here, p + 2, w[p & 1]);
      else if (!ONE) weights(next, p + 2 - PARTS, w[p & 1]);
#pragma unroll
      for (int x = 4; x; x >>= 1)
#pragma unroll
        for (int y = 0; y < x; ++y) acc[y] += acc[y + x];
      sum[p] = acc[0];
    }
#pragma unroll
    for (int x = PARTS / 2; x; x >>= 1)
#pragma unroll
      for (int y = 0; y < x; ++y) sum[y] += sum[y + x];
    // acc[r] belongs to row kg * 4 + r and column tile * 16 + row
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave * 256 + r * 64 + lane] = sum[0][r];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int idx = threadIdx.x; idx < 256; idx += n_waves * BLM_WAVE) {
      const int r = idx >> 6, l2 = idx & 63, col = l2 & 15, m = (l2 >> 4) * 4 + r;
      float s = 0.f, u = 0.f;
      if (!gated) {
        for (int x = 0; x + 1 < n_waves; x += 2) s += red[x * 256 + idx] + red[x * 256 + 256 + idx];
        if (n_waves & 1) s += red[(n_waves - 1) * 256 + idx];
        if (SCALED) s *= inv[min(m, M - 1)];
        const int n = tile * 16 + col;
        if (ROPE) {
          const float other = blm_dpp<BLM_DPP_XOR1>(s);
          if (m >= M || n >= N) continue;
          const int head = n / rope.hd, d = n - head * rope.hd, pos = pos_of[m], page = page_of[m], slot = pos % rope.page_size;
          if (head < rope.nh + rope.nkv) {
            const float2 cs = rope.cos_sin[(size_t)pos * (rope.hd / 2) + d / 2];
            s = d & 1 ? other * cs.y + s * cs.x : s * cs.x - other * cs.y;
          }
          if (head < rope.nh) C[(size_t)m * ldc + n] = s;
          else if (page >= 0 && head < rope.nh + rope.nkv) rope.kcache[(((size_t)page * rope.nkv + (head - rope.nh)) * rope.page_size + slot) * rope.hd + d] = s;
          else if (page >= 0) rope.vcache[(((size_t)page * rope.nkv + (head - rope.nh - rope.nkv)) * rope.hd + d) * rope.page_size + slot] = s;
        } else if (m < M && n < N) {
          C[(size_t)m * ldc + n] = s;
        }
      } else if (col < 8) {
        for (int x = 0; x + 1 < n_waves; x += 2) {
          s += red[x * 256 + idx] + red[x * 256 + 256 + idx];
          u += red[x * 256 + idx + 8] + red[x * 256 + 256 + idx + 8];
        }
        if (n_waves & 1) {
          s += red[(n_waves - 1) * 256 + idx];
          u += red[(n_waves - 1) * 256 + idx + 8];
        }
        if (SCALED) {
          s *= inv[min(m, M - 1)];
          u *= inv[min(m, M - 1)];
        }
        const int n = tile * 8 + col;
        if (m < M && n < N / 2) C[(size_t)m * ldc + n] = silu_times(s, u);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
}

// The longest stretch of K that a group walks for M rows (0: M out of range): 16 steps per wavefront; with 32 the activations
// alone are half of a wavefront's registers and the rest spills ([2048, 8192] in two groups 34 us, in four 16).
extern "C" int blm_gemv_f32_group_limit(int M) { return M >= 1 && M <= 16 ? 16 * 16 * GV_MAX_WAVES : 0; }

// steps of 16 of K per wavefront, wavefronts and blocks per group; a block takes a run of neighbouring column tiles
static void gemv_f32_geometry(int N, int K, int groups, int* ksteps, int* waves, int* blocks) {
  const int n_tiles = (N + 15) / 16, steps = ((K + 15) / 16 + groups - 1) / groups;
  *ksteps = steps <= 4 * GV_MAX_WAVES ? 4 : 16;
  *waves = (steps + *ksteps - 1) / *ksteps;
  const int cap = (*waves > 4 ? 256 : 512) / groups;
  const int most = n_tiles < cap ? n_tiles : cap > 0 ? cap : 1, per_block = (n_tiles + most - 1) / most;
  *blocks = (n_tiles + per_block - 1) / per_block;
}

// Blocks over all groups and wavefronts per block that blm_gemv_f32 launches; 0 if a group's stretch of K is too long.
extern "C" int blm_gemv_f32_geometry(int M, int N, int K, int groups, int* blocks, int* waves) {
  if (M < 1 || M > 16 || N < 1 || K < 4 || groups < 1 || groups > 64) return 0;
  if (((K + 15) / 16 + groups - 1) / groups * 16 > blm_gemv_f32_group_limit(M)) return 0;
  int ksteps, per_group;
  gemv_f32_geometry(N, K, groups, &ksteps, waves, &per_group);
  *blocks = per_group * groups;
  return 1;
}

// Wp: the packed copy of W[N, K], ceil(N / 16) * ceil(K / 16) * 256 floats.  gated: W's rows come in blocks of 8 gate rows and
// their 8 up rows, and C is [M, N / 2].  groups > 1: K in that many groups, a plane of M * N for each (ldc = N), which the
// reader adds up.
static int gv_run(const void* A, const void* Wp, void* C, int M, int N, int K, int lda, int ldc, int gated, int groups, const GvRope* rope,
                  const RowScale* scale, hipStream_t stream) {
  BLM_REQUIRE(M >= 1 && M <= 16 && N > 0 && K > 0 && lda >= K && ldc >= (rope ? rope->nh * rope->hd : gated ? N / 2 : N), "gemv_f32: bad sizes M=%d N=%d K=%d lda=%d ldc=%d", M, N, K, lda, ldc);
  BLM_REQUIRE(K % 4 == 0 && lda % 4 == 0 && ((uintptr_t)A % 16) == 0 && ((uintptr_t)Wp % 16) == 0,
              "gemv_f32: rows must start at multiples of 16 bytes and hold a multiple of four elements (K=%d lda=%d)", K, lda);
  BLM_REQUIRE(groups >= 1 && groups <= 64 && (groups == 1 || (!gated && ldc == N)), "gemv_f32: bad number of groups %d", groups);
  BLM_REQUIRE(!gated || N % 16 == 0, "gemv_f32: a gated matrix needs a multiple of 16 rows, got %d", N);
  const int n_tiles = (N + 15) / 16, k_steps = (K + 15) / 16, steps = (k_steps + groups - 1) / groups;
  BLM_REQUIRE(steps * 16 <= blm_gemv_f32_group_limit(M), "gemv_f32: K=%d in %d group(s) is more than %d per group", K, groups, blm_gemv_f32_group_limit(M));
  int ksteps, waves, blocks;
  gemv_f32_geometry(N, K, groups, &ksteps, &waves, &blocks);
  const int per_block = (n_tiles + blocks - 1) / blocks;
  dim3 grid((unsigned)blocks, (unsigned)groups), block(waves * BLM_WAVE);
#define BLM_GVO(KS, WHOLE, ROPE, ONE, SCALED, SCALE)                                                                    \
  hipLaunchKernelGGL((gemv_f32_kernel<KS, WHOLE, ROPE, ONE, SCALED>), grid, block, 0, stream, (const float*)A, (const float*)Wp, M, K, \
                     lda, n_tiles, k_steps, 2 * waves + (gated ? 1 : 0) + ((SCALE).n << RS_SHIFT), steps, per_block, (SCALE).sums, N, ldc, (float*)C,    \
                     rope ? *rope : GvRope{}, (SCALE).inv_width, (SCALE).eps)
#define BLM_GVS(KS, WHOLE, ROPE, SCALED, SCALE)                                                                         \
  do {                                                                                                                  \
    if (per_block == 1) BLM_GVO(KS, WHOLE, ROPE, true, SCALED, SCALE);                                                  \
    else BLM_GVO(KS, WHOLE, ROPE, false, SCALED, SCALE);                                                                \
  } while (0)
#define BLM_GVR(KS, WHOLE, ROPE)                                                                                        \
  do {                                                                                                                  \
    if (scale == nullptr) BLM_GVS(KS, WHOLE, ROPE, 0, RowScale{});                                                      \
    else if (M <= waves) BLM_GVS(KS, WHOLE, ROPE, 1, *scale);                                                           \
    else BLM_GVS(KS, WHOLE, ROPE, RS_SLOTS, *scale);                                                                    \
  } while (0)
#define BLM_GVF(KS, WHOLE)                                                                                              \
  do {                                                                                                                  \
    if (rope) BLM_GVR(KS, WHOLE, true);                                                                                 \
    else BLM_GVR(KS, WHOLE, false);                                                                                     \
  } while (0)
  const bool whole = K % 16 == 0 && k_steps == groups * steps && steps == waves * ksteps;
  if (ksteps == 4 && whole) BLM_GVF(4, true);
  else if (ksteps == 4) BLM_GVF(4, false);
  else if (whole) BLM_GVF(16, true);
  else BLM_GVF(16, false);
#undef BLM_GVF
#undef BLM_GVR
#undef BLM_GVS
#undef BLM_GVO
  BLM_LAUNCH_CHECK("gemv_f32");
  return 0;
}

extern "C" int blm_gemv_f32(const void* A, const void* Wp, void* C, int M, int N, int K, int lda, int ldc, int gated, int groups,
                            hipStream_t stream) {
  return gv_run(A, Wp, C, M, N, K, lda, ldc, gated, groups, nullptr, nullptr, stream);
}

// The same of up to eight rows that come unscaled: sums [M, n_sums] holds parts of the rows' sums of squares (row_scale.h).
extern "C" int blm_gemv_f32_scaled(const void* A, const void* Wp, void* C, int M, int N, int K, int lda, int ldc, int gated,
                                   const float* sums, int n_sums, float eps, hipStream_t stream) {
  BLM_REQUIRE(row_scale_fits(M, sums, n_sums), "gemv_f32_scaled: M=%d with %d sums a row", M, n_sums);
  const RowScale scale{sums, n_sums, 1.0f / (float)K, eps};
  return gv_run(A, Wp, C, M, N, K, lda, ldc, gated, 1, nullptr, &scale, stream);
}

// The q/k/v projection of up to 16 rows with the rotation (rotary partners are neighbouring columns) and the write of keys and
// values into their pages.  qkv_out [M][ldq]: the queries.
static int gv_rope(const void* A, const void* Wp, void* qkv_out, const int* positions, const int* token_seq,
                   const int* block_table, int table_width, const void* cos_sin, void* kcache, void* vcache, int page_size,
                   int M, int K, int lda, int ldq, int nh, int nkv, int hd, int store, const RowScale* scale, hipStream_t stream) {
  BLM_REQUIRE(nh > 0 && nkv > 0 && hd > 0 && hd % 2 == 0 && page_size > 0 && table_width > 0, "gemv_f32_qkv_rope: bad geometry (head size %d)", hd);
  BLM_REQUIRE(((uintptr_t)cos_sin % 8) == 0, "gemv_f32_qkv_rope: the table of angles must be 8-byte aligned");
  const GvRope rope{positions, token_seq, block_table, (const float2*)cos_sin, (float*)kcache, (float*)vcache, table_width, page_size, nh, nkv, hd, store};
  return gv_run(A, Wp, qkv_out, M, (nh + 2 * nkv) * hd, K, lda, ldq, 0, 1, &rope, scale, stream);
}

extern "C" int blm_gemv_f32_qkv_rope(const void* A, const void* Wp, void* qkv_out, const int* positions, const int* token_seq,
                                     const int* block_table, int table_width, const void* cos_sin, void* kcache, void* vcache, int page_size,
                                     int M, int K, int lda, int ldq, int nh, int nkv, int hd, int store, hipStream_t stream) {
  return gv_rope(A, Wp, qkv_out, positions, token_seq, block_table, table_width, cos_sin, kcache, vcache, page_size, M, K, lda, ldq, nh, nkv, hd,
                 store, nullptr, stream);
}

extern "C" int blm_gemv_f32_qkv_rope_scaled(const void* A, const void* Wp, void* qkv_out, const int* positions, const int* token_seq,
                                            const int* block_table, int table_width, const void* cos_sin, void* kcache, void* vcache, int page_size,
                                            int M, int K, int lda, int ldq, int nh, int nkv, int hd, int store, const float* sums,
                                            int n_sums, float eps, hipStream_t stream) {
  BLM_REQUIRE(row_scale_fits(M, sums, n_sums), "gemv_f32_qkv_rope_scaled: M=%d with %d sums a row", M, n_sums);
  const RowScale scale{sums, n_sums, 1.0f / (float)K, eps};
  return gv_rope(A, Wp, qkv_out, positions, token_seq, block_table, table_width, cos_sin, kcache, vcache, page_size, M, K, lda, ldq, nh, nkv, hd,
                 store, &scale, stream);
}
