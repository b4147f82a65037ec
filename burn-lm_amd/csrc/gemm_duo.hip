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
// with K = 3,072 and 9,681 rows 824 us, now 665 (1.46 PFLOP/s).  Walking 4 or 16 row tiles together instead of 8: equal; 16: 6 % behind.
#include <type_traits>

#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 gd_bf16x8;
typedef __attribute__((ext_vector_type(4))) float gd_f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int gd_u32x4;

#define GD_TILE 256
#define GD_BK 64
#define GD_GROUP 8        // row tiles that are walked together: the 32 tiles of a die at a time are 8 of rows by 4 of columns

__device__ __forceinline__ float gd_silu(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.4426950408889634f));
}
// the tanh form of GELU, z/2 (1 + tanh(a)) with a = sqrt(2/pi) (z + 0.044715 z^3): (1 + tanh(a)) / 2 = sigmoid(2a)
__device__ __forceinline__ float gd_gelu(float x) {
  const float a = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(a * -2.8853900817779268f));
}

#define GD_FENCE() __builtin_amdgcn_sched_barrier(0)
#define GD_BARRIER()                             \
  do {                                           \
    GD_FENCE();                                  \
    asm volatile("s_barrier" ::: "memory");      \
    GD_FENCE();                                  \
  } while (0)
#define GD_WAIT_VM(n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory")
#define GD_WAIT_LDS() __builtin_amdgcn_s_waitcnt(0xC07F)

template <int V>
using GdInt = std::integral_constant<int, V>;

#define GD_REGION (128 * GD_BK * 2)        // bytes: 128 rows of one operand's stage

struct GdTile {
  const char *a, *b;                        // first row of the activations and of the weights, at the group's first k
  int rows, columns;                        // that exist (of the matrix, from the tile's first on)
  uint32_t up;                              // bytes from a gate row to its up row
  int lda, ldw;
};

// byte offsets of a lane's 16 bytes in the loads of one region: 128 rows of 64 k, slot s of row r holds piece s ^ (r / 2 % 8)
__device__ __forceinline__ uint32_t gd_place(int r, int lane) { return (uint32_t)((lane & 7) ^ ((r >> 1) & 7)) * 16u; }
template <int MODE>
__device__ __forceinline__ uint32_t gd_weight_offset(const GdTile& t, int r, int h, int lane) {
  const int n = min(MODE != 0 ? r : r / 32 * 64 + h * 32 + r % 32, t.columns - 1);
  return (uint32_t)n * (uint32_t)t.ldw * 2u + (MODE != 0 && h ? t.up : 0u) + gd_place(r, lane);
}
__device__ __forceinline__ uint32_t gd_row_offset(const GdTile& t, int m, int r, int lane) {
  return (uint32_t)(min(m, t.rows - 1) * t.lda) * 2u + gd_place(r, lane);
}

// acc[i][j]: row i * 16 + l16, columns j * 16 + 4 quad + e of a wavefront's part.  bfloat16: an exchange between neighbouring rows
// of 16 lanes, over two tiles of columns, gives every lane 8 neighbours.
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
      const auto r0 = __builtin_amdgcn_permlane16_swap(f32x2_to_bf16x2_bits(v[0][0], v[0][1]), f32x2_to_bf16x2_bits(v[1][0], v[1][1]), false, false);
      const auto r1 = __builtin_amdgcn_permlane16_swap(f32x2_to_bf16x2_bits(v[0][2], v[0][3]), f32x2_to_bf16x2_bits(v[1][2], v[1][3]), false, false);
      const int n = n0 + (j + (quad & 1)) * 16 + (quad >> 1) * 8;
      if (m < M && n < N) *reinterpret_cast<uint4*>(C + (size_t)m * ldc + n) = make_uint4(r0[0], r1[0], r0[1], r1[1]);
    }
  }
}

// sixteen products: 64 rows and 32 columns of a stage; the loads go out in the middle
template <int TILES, typename Loads>
__device__ __forceinline__ void gd_multiply(gd_f32x4 (&acc)[TILES][4], const gd_u32x4 (&a)[2][4], const gd_u32x4 (&b)[2][2], int ih, int jh, Loads loads) {
  GD_BARRIER();
#pragma unroll
  for (int q = 0; q < 2; ++q) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[ih * 4 + i][jh * 2 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(gd_bf16x8, b[q][j]), __builtin_bit_cast(gd_bf16x8, a[q][i]), acc[ih * 4 + i][jh * 2 + j], 0, 0, 0);
    if (q == 0) {
      GD_FENCE();
      loads();
      GD_FENCE();
    }
  }
  GD_WAIT_LDS();
  GD_BARRIER();
}

template <int TILES>
__device__ __forceinline__ void gd_zero(gd_f32x4 (&acc)[TILES][4]) {
#pragma unroll
  for (int i = 0; i < TILES; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = gd_f32x4{0.f, 0.f, 0.f, 0.f};
}

// A whole tile: a wavefront has 128 rows and 64 columns.
template <int MODE>
__device__ __forceinline__ void gd_whole(gd_f32x4 (&acc)[8][4], const GdTile& t, int stages, unsigned char* lds, int wave, int lane) {
  const int l16 = lane & 15, quad = lane >> 4, wm = wave >> 2, wn = wave & 3;
  uint32_t a_off[2][2], b_off[2][2];                       // [half][load]
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = (wave * 2 + i) * 8 + lane / 8;
      a_off[h][i] = gd_row_offset(t, r / 64 * 128 + h * 64 + r % 64, r, lane);
      b_off[h][i] = gd_weight_offset<MODE>(t, r, h, lane);
    }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(blm_lds_ptr)lds + (uint32_t)wave * 2048u;
  auto fetch_a = [&](int s, int buf, int h) {
    const char* base = t.a + (size_t)s * (GD_BK * 2);
    blm_dma16_to(base, a_off[h][0], lds0 + (buf * 2 + h) * GD_REGION);
    blm_dma16_to(base, a_off[h][1], lds0 + (buf * 2 + h) * GD_REGION + 1024);
  };
  auto fetch_b = [&](int s, int buf, int h) {
    const char* base = t.b + (size_t)s * (GD_BK * 2);
    blm_dma16_to(base, b_off[h][0], lds0 + (4 + buf * 2 + h) * GD_REGION);
    blm_dma16_to(base, b_off[h][1], lds0 + (4 + buf * 2 + h) * GD_REGION + 1024);
  };
  int a_at[2], b_at[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int slot = (4 * q + quad) ^ ((l16 >> 1) & 7);
    a_at[q] = (wm * 64 + l16) * 128 + slot * 16;
    b_at[q] = 4 * GD_REGION + (wn * 32 + l16) * 128 + slot * 16;
  }
  gd_u32x4 a0[2][4], a1[2][4], b0[2][2], b1[2][2];         // [32 of k][16 rows]
  auto read_a = [&](gd_u32x4 (&f)[2][4], int buf, int h, int x) {
    f[x >> 2][x & 3] = *reinterpret_cast<const gd_u32x4*>(lds + a_at[x >> 2] + (buf * 2 + h) * GD_REGION + (x & 3) * 2048);
  };
  auto read_b = [&](gd_u32x4 (&f)[2][2], int buf, int h, int x) {
    f[x >> 1][x & 1] = *reinterpret_cast<const gd_u32x4*>(lds + b_at[x >> 1] + (buf * 2 + h) * GD_REGION + (x & 1) * 2048);
  };
  gd_zero(acc);

#pragma unroll
  for (int s = 0; s < 2; ++s) {
    fetch_a(s, s, 0);
    fetch_b(s, s, 1);
    fetch_a(s, s, 1);
    fetch_b(s, s, 0);
  }
  GD_WAIT_VM(8);
  GD_BARRIER();
#pragma unroll
  for (int x = 0; x < 8; ++x) read_a(a0, 0, 0, x);
#pragma unroll
  for (int x = 0; x < 4; ++x) read_b(b1, 0, 1, x);
  GD_WAIT_LDS();
  GD_BARRIER();
  if (wave >= 4) GD_BARRIER();

  // `left`: stages behind this one that exist (2: two and more)
  auto stage = [&](int s, auto buf_type, auto left_type) {
    constexpr int buf = decltype(buf_type)::value, left = decltype(left_type)::value;
    // first rows, first columns
#pragma unroll
    for (int x = 0; x < 4; ++x) read_b(b0, buf, 0, x);
    read_a(a1, buf, 1, 0);
    read_a(a1, buf, 1, 1);
    gd_multiply(acc, a0, b0, 0, 0, [&] { if (left > 1) fetch_a(s + 2, buf, 0); });
    // first rows, second columns
#pragma unroll
    for (int x = 2; x < 8; ++x) read_a(a1, buf, 1, x);
    if (left > 1) GD_WAIT_VM(8);
    else if (left == 1) GD_WAIT_VM(6);
    gd_multiply(acc, a0, b1, 0, 1, [&] { if (left > 1) fetch_b(s + 2, buf, 1); });
    // second rows, second columns
    if (left > 0)
#pragma unroll
      for (int x = 0; x < 6; ++x) read_a(a0, buf ^ 1, 0, x);
    if (left > 1) GD_WAIT_VM(8);
    else if (left == 1) GD_WAIT_VM(4);
    gd_multiply(acc, a1, b1, 1, 1, [&] { if (left > 1) fetch_a(s + 2, buf, 1); });
    // second rows, first columns
    if (left > 0) {
      read_a(a0, buf ^ 1, 0, 6);
      read_a(a0, buf ^ 1, 0, 7);
#pragma unroll
      for (int x = 0; x < 4; ++x) read_b(b1, buf ^ 1, 1, x);
    }
    if (left > 1) GD_WAIT_VM(6);
    else if (left == 1) GD_WAIT_VM(0);
    gd_multiply(acc, a1, b0, 1, 0, [&] { if (left > 1) fetch_b(s + 2, buf, 0); });
  };
  int s = 0;
  for (; s + 2 < stages; s += 2) {
    stage(s, GdInt<0>{}, GdInt<2>{});
    stage(s + 1, GdInt<1>{}, GdInt<2>{});
  }
  stage(s, GdInt<0>{}, GdInt<1>{});
  stage(s + 1, GdInt<1>{}, GdInt<0>{});
  if (wave < 4) GD_BARRIER();
}

// Half a tile, 128 rows of it: a wavefront has 64 rows and 64 columns.  A stage's fragments are read a stage ahead into a second
// set of registers, and the ring has three stages.  0.57 of a whole tile's time (its reads of shared memory per product are 4 / 3).
template <int MODE>
__device__ __forceinline__ void gd_half(gd_f32x4 (&acc)[4][4], const GdTile& t, int stages, unsigned char* lds, int wave, int lane) {
  const int l16 = lane & 15, quad = lane >> 4, wm = wave >> 2, wn = wave & 3;
  uint32_t off[3][2];                                      // rows, first columns, second columns
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (wave * 2 + i) * 8 + lane / 8;
    off[0][i] = gd_row_offset(t, r, r, lane);
    off[1][i] = gd_weight_offset<MODE>(t, r, 0, lane);
    off[2][i] = gd_weight_offset<MODE>(t, r, 1, lane);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(blm_lds_ptr)lds + (uint32_t)wave * 2048u;
  auto fetch = [&](int s, int slot, int region, int i) {
    blm_dma16_to((region == 0 ? t.a : t.b) + (size_t)s * (GD_BK * 2), off[region][i], lds0 + (uint32_t)((slot * 3 + region) * GD_REGION + i * 1024));
  };
  int a_at[2], b_at[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int slot = (4 * q + quad) ^ ((l16 >> 1) & 7);
    a_at[q] = (wm * 64 + l16) * 128 + slot * 16;
    b_at[q] = GD_REGION + (wn * 32 + l16) * 128 + slot * 16;
  }
  gd_u32x4 a[2][2][4], b0[2][2][2], b1[2][2][2];           // [stage's parity][32 of k][16 rows]
  auto read_a = [&](int set, int slot) {
    const unsigned char* at = lds + slot * (3 * GD_REGION);
#pragma unroll
    for (int x = 0; x < 8; ++x) a[set][x >> 2][x & 3] = *reinterpret_cast<const gd_u32x4*>(at + a_at[x >> 2] + (x & 3) * 2048);
  };
  auto read_b = [&](int set, int slot) {
    const unsigned char* at = lds + slot * (3 * GD_REGION);
#pragma unroll
    for (int x = 0; x < 4; ++x) b0[set][x >> 1][x & 1] = *reinterpret_cast<const gd_u32x4*>(at + b_at[x >> 1] + (x & 1) * 2048);
#pragma unroll
    for (int x = 0; x < 4; ++x) b1[set][x >> 1][x & 1] = *reinterpret_cast<const gd_u32x4*>(at + b_at[x >> 1] + GD_REGION + (x & 1) * 2048);
  };
  gd_zero(acc);

#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int x = 0; x < 6; ++x) fetch(s, s, x >> 1, x & 1);
  GD_WAIT_VM(12);
  GD_BARRIER();
  read_a(0, 0);
  read_b(0, 0);
  GD_WAIT_LDS();
  GD_WAIT_VM(10);
  GD_BARRIER();
  if (wave >= 4) GD_BARRIER();

  // slot: of stage s; `left`: stages behind this one that exist (3: three and more)
  auto stage = [&](int s, int slot, auto set_type, auto left_type) {
    constexpr int set = decltype(set_type)::value, left = decltype(left_type)::value;
    const int next = slot == 2 ? 0 : slot + 1;
    if (left > 0) read_a(set ^ 1, next);
    if (left > 1) GD_WAIT_VM(6);
    else if (left == 1) GD_WAIT_VM(0);
    gd_multiply(acc, a[set], b0[set], 0, 0, [&] {
      if (left > 2) {
        fetch(s + 3, slot, 0, 0);
        fetch(s + 3, slot, 0, 1);
        fetch(s + 3, slot, 1, 0);
      }
    });
    if (left > 0) read_b(set ^ 1, next);
    if (left > 2) GD_WAIT_VM(7);
    else if (left == 2) GD_WAIT_VM(4);
    gd_multiply(acc, a[set], b1[set], 0, 1, [&] {
      if (left > 2) {
        fetch(s + 3, slot, 1, 1);
        fetch(s + 3, slot, 2, 0);
        fetch(s + 3, slot, 2, 1);
      }
    });
    return next;
  };
  int s = 0, slot = 0;
  for (; s + 4 < stages; s += 2) {
    slot = stage(s, slot, GdInt<0>{}, GdInt<3>{});
    slot = stage(s + 1, slot, GdInt<1>{}, GdInt<3>{});
  }
  slot = stage(s, slot, GdInt<0>{}, GdInt<3>{});
  slot = stage(s + 1, slot, GdInt<1>{}, GdInt<2>{});
  slot = stage(s + 2, slot, GdInt<0>{}, GdInt<1>{});
  stage(s + 3, slot, GdInt<1>{}, GdInt<0>{});
  if (wave < 4) GD_BARRIER();
}

// Tiles in the order in which they are walked: [0, whole) as whole ones, the rest of the m_tiles x n_tiles as two halves each, and
// behind them, where `tail`, a row of halves below the last row of tiles.
template <int MODE, typename TC>
__global__ void __launch_bounds__(512, 2)
    gemm_duo_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W, TC* __restrict__ C, int M, int N, int K, int lda, int ldw,
                    int ldc, int m_tiles, int n_tiles, int whole, int k_per_group) {
  constexpr int OUT = MODE != 0 ? GD_TILE / 2 : GD_TILE;   // output columns of a tile
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
  const int m0 = tm * GD_TILE + below, n0 = tn * OUT, k0 = blockIdx.y * k_per_group, stages = min(k_per_group, K - k0) / GD_BK;
  if (m0 >= M) return;                       // a second half that has no rows
  C += (size_t)blockIdx.y * M * ldc;
  GdTile t;
  t.a = reinterpret_cast<const char*>(A + (size_t)m0 * lda + k0);
  t.b = reinterpret_cast<const char*>(W + (size_t)n0 * ldw + k0);
  t.rows = M - m0;
  t.columns = N - n0;
  t.up = (uint32_t)N * (uint32_t)ldw * 2u;
  t.lda = lda;
  t.ldw = ldw;
  const int n = n0 + wn * (MODE != 0 ? 32 : 64);
  if (!half) {
    gd_f32x4 acc[8][4];
    gd_whole<MODE>(acc, t, stages, lds, wave, lane);
    gd_store<MODE, 8, TC>(acc, C, ldc, m0 + wm * 128, M, n, N, l16, quad);
  } else {
    gd_f32x4 acc[4][4];
    gd_half<MODE>(acc, t, stages, lds, wave, lane);
    gd_store<MODE, 4, TC>(acc, C, ldc, m0 + wm * 64, M, n, N, l16, quad);
  }
}

// mode 0: C[M, N] = A W^T, W [N, K].  mode 1: W [2N, K] = [gate rows; up rows], C[M, N] = silu(gate) * up; mode 2: the tanh form of
// GELU in place of silu.  k_groups > 1: C is float [k_groups, M, ldc], a partial product over each group's stretch of K (a multiple
// of 128).  whole: how many of the tiles are run as whole ones, the others as halves.
extern "C" int blm_gemm_duo(const void* A, const void* W, void* C, int c_dtype, int M, int N, int K, int lda, int ldw, int ldc, int mode,
                            int k_groups, int whole, hipStream_t stream) {
  BLM_REQUIRE(M >= 1 && N >= 8 && N % 8 == 0 && K >= 256 && K % 128 == 0, "gemm_duo: sizes M=%d N=%d K=%d not supported", M, N, K);
  BLM_REQUIRE(lda % 8 == 0 && ldw % 8 == 0 && ldc % 8 == 0 && lda >= K && ldw >= K && ldc >= N, "gemm_duo: bad strides lda=%d ldw=%d ldc=%d",
              lda, ldw, ldc);
  BLM_REQUIRE(((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0 && ((uintptr_t)C % 16) == 0, "gemm_duo: operands must be 16-byte aligned");
  BLM_REQUIRE(mode >= 0 && mode <= 2 && (c_dtype == BLM_BF16 || (c_dtype == BLM_F32 && mode == 0)), "gemm_duo: mode %d, dtype %d", mode, c_dtype);
  const int k_per_group = k_groups >= 1 ? ((K + k_groups - 1) / k_groups + 127) / 128 * 128 : 0;
  BLM_REQUIRE(k_groups >= 1 && k_groups <= 64 && (k_groups == 1 || c_dtype == BLM_F32) && K - (k_groups - 1) * k_per_group >= 256,
              "gemm_duo: %d groups of K=%d need 256 each and a float output", k_groups, K);
  BLM_REQUIRE((size_t)256 * lda * 2 < ((size_t)1 << 32) && (size_t)(mode != 0 ? 2 : 1) * N * ldw * 2 < ((size_t)1 << 32),
              "gemm_duo: matrices of 4 GiB and more are not supported (lda=%d, N=%d, ldw=%d)", lda, N, ldw);
  const int columns = mode != 0 ? GD_TILE / 2 : GD_TILE, n_tiles = (N + columns - 1) / columns;
  const bool tail = M % GD_TILE != 0 && M % GD_TILE <= GD_TILE / 2;
  const int m_tiles = tail ? M / GD_TILE : (M + GD_TILE - 1) / GD_TILE;
  BLM_REQUIRE((long long)(m_tiles + 1) * n_tiles < (1LL << 29), "gemm_duo: too many tiles");
  BLM_REQUIRE(whole >= 0 && whole <= m_tiles * n_tiles, "gemm_duo: %d whole tiles of %d", whole, m_tiles * n_tiles);
  const int halves = 2 * (m_tiles * n_tiles - whole) + (tail ? n_tiles : 0);
  const dim3 grid((unsigned)(whole + halves), (unsigned)k_groups), block(512);
#define GD_LAUNCH(MODE, TC)                                                                                                        \
  hipLaunchKernelGGL((gemm_duo_kernel<MODE, TC>), grid, block, 0, stream, (const bf16*)A, (const bf16*)W, (TC*)C, M, N, K, lda, ldw, \
                     ldc, m_tiles, n_tiles, whole, k_per_group)
  if (mode == 1) GD_LAUNCH(1, bf16);
  else if (mode == 2) GD_LAUNCH(2, bf16);
  else if (c_dtype == BLM_F32) GD_LAUNCH(0, float);
  else GD_LAUNCH(0, bf16);
#undef GD_LAUNCH
  BLM_LAUNCH_CHECK("gemm_duo");
  return 0;
}
