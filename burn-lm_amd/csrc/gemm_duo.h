// The 256x256 tile of bfloat16 products and its half, shared by gemm_duo.hip (which says what they are bound by and why they are as
// they are) and moe_grouped.hip.  A block is eight wavefronts of 2 (rows) x 4 (columns); acc[i][j] of a wavefront: row i * 16 + l16,
// columns j * 16 + 4 quad + e of its part.  A whole tile's wavefront has 128 rows and 64 columns, a half's 64 and 64; its columns are
// rows wn * 32 on of the weights' region 0 (j = 0, 1) and of region 1 (j = 2, 3).
#pragma once
#include <type_traits>

#include "common.h"


typedef __attribute__((ext_vector_type(8))) __bf16 gd_bf16x8;
typedef __attribute__((ext_vector_type(4))) float gd_f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int gd_u32x4;

#define GD_TILE 256
#define GD_BK 64
#define GD_GROUP 8        // row tiles that are walked together: the 32 tiles of a die at a time are 8 of rows by 4 of columns

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

#define GD_FIVE_PERCENT 71
#define GD_REGION (128 * GD_BK * 2)        // bytes: 128 rows of one operand's stage

// A tile's operands: `a` and `b` the same in all lanes, at the first k; row(m) and column(r, h) the bytes from there to row m of the
// tile and to row r of the weights' region h.  Staged slot s of row r holds its piece s ^ (r / 2 % 8).
__device__ __forceinline__ uint32_t gd_piece(int r, int lane) { return (uint32_t)((lane & 7) ^ ((r >> 1) & 7)) * 16u; }

// Two tiles of 16 columns of a lane's row, 4 columns of each, as bfloat16: an exchange between neighbouring rows of 16 lanes gives
// every lane 8 neighbours, columns 16 (quad % 2) + 8 (quad / 2) on.
__device__ __forceinline__ uint4 gd_eight(const float (&v)[2][4]) {
  const auto r0 = __builtin_amdgcn_permlane16_swap(f32x2_to_bf16x2_bits(v[0][0], v[0][1]), f32x2_to_bf16x2_bits(v[1][0], v[1][1]), false, false);
  const auto r1 = __builtin_amdgcn_permlane16_swap(f32x2_to_bf16x2_bits(v[0][2], v[0][3]), f32x2_to_bf16x2_bits(v[1][2], v[1][3]), false, false);
  return make_uint4(r0[0], r1[0], r0[1], r1[1]);
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
template <typename Tile>
__device__ __forceinline__ void gd_whole(gd_f32x4 (&acc)[8][4], const Tile& t, int stages, unsigned char* lds, int wave, int lane) {
  const int l16 = lane & 15, quad = lane >> 4, wm = wave >> 2, wn = wave & 3;
  uint32_t a_off[2][2], b_off[2][2];                       // [half][load]
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = (wave * 2 + i) * 8 + lane / 8;
      a_off[h][i] = t.row(r / 64 * 128 + h * 64 + r % 64) + gd_piece(r, lane);
      b_off[h][i] = t.column(r, h) + gd_piece(r, lane);
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

// Part of a tile, 32 TILES rows of it: 128 (a half) or 160 (five eighths).  A wavefront has half of them and 64 columns.  A stage's
// fragments are read a stage ahead into a second set of registers, and the ring has three stages (156 KB for 160 rows, as many as a
// unit's memory and a wavefront's registers hold).  A half takes 0.57 of a whole tile's time (its reads of shared memory per product are
// 4 / 3), five eighths GD_FIVE_PERCENT.
template <int TILES>
struct GdPart {
  static constexpr int ROWS = 32 * TILES, LOADS = (ROWS / 8 + 7) / 8;                 // of the rows, per wavefront and stage
  static constexpr uint32_t A_BYTES = ROWS * GD_BK * 2, STAGE = A_BYTES + 2 * GD_REGION;
};

template <int TILES, typename Tile>
__device__ __forceinline__ void gd_part(gd_f32x4 (&acc)[TILES][4], const Tile& t, int stages, unsigned char* lds, int wave, int lane) {
  using Part = GdPart<TILES>;
  constexpr int NA = Part::LOADS, ALL = NA + 4;
  const int l16 = lane & 15, quad = lane >> 4, wm = wave >> 2, wn = wave & 3;
  // eight rows to a load; beyond 128 rows four loads are left, and wavefronts w and w + 4 bring the same one (each waits for as many)
  auto group = [&](int i) { return i < 2 ? wave * 2 + i : 16 + (wave & 3); };
  uint32_t a_off[NA], b_off[2][2];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int r = group(i) * 8 + lane / 8;
    a_off[i] = t.row(r) + gd_piece(r, lane);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = group(i) * 8 + lane / 8;
    b_off[0][i] = t.column(r, 0) + gd_piece(r, lane);
    b_off[1][i] = t.column(r, 1) + gd_piece(r, lane);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(blm_lds_ptr)lds;
  auto fetch_a = [&](int s, int slot, int i) {
    blm_dma16_to(t.a + (size_t)s * (GD_BK * 2), a_off[i], lds0 + (uint32_t)slot * Part::STAGE + (uint32_t)group(i) * 1024u);
  };
  auto fetch_b = [&](int s, int slot, int h, int i) {
    blm_dma16_to(t.b + (size_t)s * (GD_BK * 2), b_off[h][i], lds0 + (uint32_t)slot * Part::STAGE + Part::A_BYTES + (uint32_t)h * GD_REGION + (uint32_t)group(i) * 1024u);
  };
  int a_at[2], b_at[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int slot = (4 * q + quad) ^ ((l16 >> 1) & 7);
    a_at[q] = (wm * (16 * TILES) + l16) * 128 + slot * 16;
    b_at[q] = Part::A_BYTES + (wn * 32 + l16) * 128 + slot * 16;
  }
  gd_u32x4 a[2][2][TILES], b0[2][2][2], b1[2][2][2];       // [stage's parity][32 of k][16 rows]
  auto read_a = [&](int set, int slot) {
    const unsigned char* at = lds + slot * Part::STAGE;
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int x = 0; x < TILES; ++x) a[set][q][x] = *reinterpret_cast<const gd_u32x4*>(at + a_at[q] + x * 2048);
  };
  auto read_b = [&](int set, int slot) {
    const unsigned char* at = lds + slot * Part::STAGE;
#pragma unroll
    for (int x = 0; x < 4; ++x) b0[set][x >> 1][x & 1] = *reinterpret_cast<const gd_u32x4*>(at + b_at[x >> 1] + (x & 1) * 2048);
#pragma unroll
    for (int x = 0; x < 4; ++x) b1[set][x >> 1][x & 1] = *reinterpret_cast<const gd_u32x4*>(at + b_at[x >> 1] + GD_REGION + (x & 1) * 2048);
  };
  auto multiply = [&](auto set_type, auto side_type, auto loads) {
    constexpr int set = decltype(set_type)::value, side = decltype(side_type)::value;
    GD_BARRIER();
#pragma unroll
    for (int q = 0; q < 2; ++q) {
#pragma unroll
      for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][side * 2 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(gd_bf16x8, side ? b1[set][q][j] : b0[set][q][j]), __builtin_bit_cast(gd_bf16x8, a[set][q][i]), acc[i][side * 2 + j], 0, 0, 0);
      if (q == 0) {
        GD_FENCE();
        loads();
        GD_FENCE();
      }
    }
    GD_WAIT_LDS();
    GD_BARRIER();
  };
  gd_zero(acc);

#pragma unroll
  for (int s = 0; s < 3; ++s) {
#pragma unroll
    for (int i = 0; i < NA; ++i) fetch_a(s, s, i);
#pragma unroll
    for (int x = 0; x < 4; ++x) fetch_b(s, s, x >> 1, x & 1);
  }
  GD_WAIT_VM(2 * ALL);
  GD_BARRIER();
  read_a(0, 0);
  read_b(0, 0);
  GD_WAIT_LDS();
  GD_WAIT_VM(2 * ALL - NA);
  GD_BARRIER();
  if (wave >= 4) GD_BARRIER();

  // slot: of stage s; `left`: stages behind this one that exist (3: three and more).  On entry the next stage's rows are there.
  auto stage = [&](int s, int slot, auto set_type, auto left_type) {
    constexpr int set = decltype(set_type)::value, left = decltype(left_type)::value;
    const int next = slot == 2 ? 0 : slot + 1;
    if (left > 0) read_a(set ^ 1, next);
    if (left > 1) GD_WAIT_VM(ALL);                         // all of the next stage
    else if (left == 1) GD_WAIT_VM(0);
    multiply(set_type, GdInt<0>{}, [&] {
      if (left > 2) {
#pragma unroll
        for (int i = 0; i < NA; ++i) fetch_a(s + 3, slot, i);
        fetch_b(s + 3, slot, 0, 0);
      }
    });
    if (left > 0) read_b(set ^ 1, next);
    if (left > 2) GD_WAIT_VM(ALL + 1);                     // the rows of the stage behind the next
    else if (left == 2) GD_WAIT_VM(4);
    multiply(set_type, GdInt<1>{}, [&] {
      if (left > 2) {
        fetch_b(s + 3, slot, 0, 1);
        fetch_b(s + 3, slot, 1, 0);
        fetch_b(s + 3, slot, 1, 1);
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
