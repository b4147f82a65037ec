// The 32-bit product C[M,N] = A[M,K] * W[N,K]^T of many rows on the bfloat16 matrix instructions, with no less precision than on the
// float ones: a float is the sum of three bfloat16 (hi, mid, lo, rounded to nearest each: 8 + 8 + 8 bits and their signs, the subtractions
// between them exact), a product of two floats the sum of nine exact products, and the three that are left out (mid lo, lo mid, lo lo)
// are below 2^-26 of the whole (floats below 2^-110 have no lo of their own: what is lost of them is below 2^-134).  Six instructions
// of 16 cycles do 16 x 16 x 32, for which the float ones take 256 cycles.  (Floats as sums of three bfloat16: Henry, Tang and Heinecke, "Leveraging
// the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", ARITH 2019.)
//   split_rows : the parts of the rows, in the order of the instruction's fragments
//   gemm_split : the product; the weights, which are not kept a second time, are split on their way from shared memory
// What bounds it: the matrix instructions at the clock that the card's power leaves (1.3 to 1.4 PFLOP/s of them), beside them reads of
// shared memory (a fragment of three parts serves six or twelve instructions), the splitting, 88 vector instructions (104 where a chunk is negated)
// for a stage's 96 matrix ones at 128 x 256, and a chunk's 64 additions.  Every wavefront has all rows of the tile and columns of its own, so that
// no weight is split twice in a block.
// Sums: the matrix instruction adds to its accumulator with what falls off below cut, towards minus infinity: a result of 2,048 products by
// one accumulator is 2.7e-7 off and, the same in all of them, 3e-8 too low, which adds up from layer to layer (logits of the 1B shape
// 3.7e-6 from 64 bits, with the float instructions 2.8e-6).  So a chunk of 128 of K has an accumulator that starts at zero, small products
// first, and joins the total by a rounded addition; and every other chunk is summed with its columns negated and subtracted, so that what is
// cut cancels: 1.7e-7 off (2.17e-7 with the float instructions), 7e-11 too low, and the logits 2.6e-6.  It cancels in pairs, so a group of K with
// an odd number of chunks has its last one in two halves of opposite sign (mean error of normal operands, without / with: K = 128 -8e-9 / 1e-10,
// 640 -4e-9 / -3e-10, 3,072 in 8 groups of three -1.4e-8 / 0; 2-norms 1.52 / 0.97, 1.59 / 1.52, 1.64 / 1.50e-7, the float instructions' 2.0 to 2.1).
// Measured (us, the float instructions' best tile and groups / this, without the parts' pass of 2.7 to 6 us, with K = 8,192 14; weights from memory),
// 1,000 rows: [16384, 2048] gated 502 / 284 (236 TFLOP/s of float products, 1.42 PFLOP/s; cards differ, up to 300), [2048, 8192] 259 / 157, [3072, 2048] 105 / 75, [2048, 2048] 72 / 47;
// 256 rows 137 / 90, 74 / 50, 33 / 26, 24 / 18.  Scoring 1,000 tokens at the 1B shape 16.9 -> 10.8 ms.
// The ring is as deep as the weights' way from memory asks: with the next two stages under way tiles of 64 rows, whose stages are short, took 1.34 us
// a stage for the 64 x 128, with three 0.70 (1.2 and 1.13 for 64 x 256; four and five: as three).
// Tried: columns from global memory straight into registers (120 -> 133 us on 64 blocks), tiles of 256 x 256 (two stages fill the
// shared memory: 334 against 312), two accumulators for small and large products without the rounded additions (5 % faster, 2.7e-7 off),
// the small products' sums added in every step (1.06e-7 off, registers spill).
#include <type_traits>

#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 gs_bf16x8;
typedef __attribute__((ext_vector_type(4))) float gs_f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int gs_u32x4;

#define GS_BK 32
#define GS_FRAGMENT 1024                  // bytes: 16 rows and 32 of K of one part, 16 bytes a lane

__device__ __forceinline__ float gs_low(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float gs_high(uint32_t v) { return __uint_as_float(v & 0xffff0000u); }

__device__ __forceinline__ void gs_split(float x, float y, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = f32x2_to_bf16x2_bits(x, y);
  x -= gs_low(hi);
  y -= gs_high(hi);
  mid = f32x2_to_bf16x2_bits(x, y);
  lo = f32x2_to_bf16x2_bits(x - gs_low(mid), y - gs_high(mid));
}

// A value that has no such parts, or whose first would round to an infinity: hi keeps an infinity or NaN alone, and is cut off otherwise.
__device__ __forceinline__ void gs_split_odd(float x, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  const uint32_t bits = __float_as_uint(x);
  hi = bits >> 16;
  mid = lo = 0u;
  if ((bits & 0x7fffffffu) > 0x7f800000u) hi |= 0x40u;
  else if ((bits & 0x7f800000u) != 0x7f800000u) {
    x -= gs_low(hi);
    mid = f32_to_bf16_bits(x);
    lo = f32_to_bf16_bits(x - gs_low(mid));
  }
}
__device__ __forceinline__ bool gs_odd(float x) { return (__float_as_uint(x) & 0x7fffffffu) >= 0x7f7f8000u; }

__device__ __forceinline__ void gs_split_any(float x, float y, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  if (!(gs_odd(x) || gs_odd(y))) {
    gs_split(x, y, hi, mid, lo);
  } else {
    uint32_t h, m, l;
    gs_split_odd(x, hi, mid, lo);
    gs_split_odd(y, h, m, l);
    hi |= h << 16;
    mid |= m << 16;
    lo |= l << 16;
  }
}

// ---------------------------------------------------------------------------------------------------------------------
// parts of the rows: P [ceil(M / 16)][K / 32][3][64 lanes][8]: lane l holds row l % 16, elements 4 (l / 16) + 0..3 and 16 + 4 (l / 16) + 0..3
// of the 32; rows behind M are zero.
__global__ void __launch_bounds__(256) split_rows_kernel(const float* __restrict__ X, int ldx, uint4* __restrict__ P, int M, int K) {
  const int lane = threadIdx.x & 63, steps = K / GS_BK, per_tile = (steps + 3) / 4, tile = blockIdx.x / per_tile;
  const int ks = (blockIdx.x - tile * per_tile) * 4 + threadIdx.x / 64;
  if (ks >= steps) return;
  const int m = tile * 16 + (lane & 15);
  float4 u = make_float4(0.f, 0.f, 0.f, 0.f), v = u;
  if (m < M) {
    const float* x = X + (size_t)m * ldx + ks * GS_BK + (lane >> 4) * 4;
    u = *reinterpret_cast<const float4*>(x);
    v = *reinterpret_cast<const float4*>(x + 16);
  }
  const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
  uint32_t hi[4], mid[4], lo[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) gs_split_any(x[2 * e], x[2 * e + 1], hi[e], mid[e], lo[e]);
  uint4* p = P + ((size_t)tile * steps + ks) * 192 + lane;
  p[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
  p[64] = make_uint4(mid[0], mid[1], mid[2], mid[3]);
  p[128] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
}

extern "C" int blm_split_rows(const void* X, void* P, int M, int K, int ldx, hipStream_t stream) {
  BLM_REQUIRE(M > 0 && K > 0 && K % GS_BK == 0 && ldx >= K && ldx % 4 == 0, "split_rows: sizes M=%d K=%d ldx=%d not supported", M, K, ldx);
  BLM_REQUIRE(((uintptr_t)X % 16) == 0 && ((uintptr_t)P % 16) == 0, "split_rows: rows and parts must be 16-byte aligned");
  const long long blocks = (long long)((M + 15) / 16) * ((K / GS_BK + 3) / 4);
  BLM_REQUIRE(blocks < 2147483647LL, "split_rows: too many rows");
  hipLaunchKernelGGL(split_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, (const float*)X, ldx, (uint4*)P, M, K);
  BLM_LAUNCH_CHECK("split_rows");
  return 0;
}

__device__ __forceinline__ float gs_silu_times(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// where the first part of row m's column n lies, in the parts of rows of N columns
__device__ __forceinline__ unsigned char* gs_part_of(float* parts, int m, int n, int N) {
  return reinterpret_cast<unsigned char*>(parts) + ((size_t)(m / 16) * (N / GS_BK) + n / GS_BK) * (3 * GS_FRAGMENT) + (m % 16 + n % 16 / 4 * 16) * 16 +
         n % GS_BK / 16 * 8 + n % 4 * 2;
}

// What a weight does to a sum's being a number: zeros, infinities and NaN as they are, all others 2^-100 with their sign (sums of so many rows'
// first parts times these stay finite).
__device__ __forceinline__ uint32_t gs_kind(float x) {
  const uint32_t bits = __float_as_uint(x), top = bits & 0x7fffffffu;
  if (top >= 0x7f800000u) return bits >> 16 | (top > 0x7f800000u ? 0x40u : 0u);
  return top == 0u ? 0u : (bits >> 16 & 0x8000u) | 0x0d80u;
}

template <int V>
using GsInt = std::integral_constant<int, V>;
using GsPlus = std::false_type;
using GsMinus = std::true_type;
__device__ __forceinline__ gs_f32x4 gs_signed(gs_f32x4 v, GsPlus) { return v; }
__device__ __forceinline__ gs_f32x4 gs_signed(gs_f32x4 v, GsMinus) { return -v; }
__device__ __forceinline__ gs_f32x4 gs_signed(gs_f32x4 v, uint32_t mask) { return __builtin_bit_cast(gs_f32x4, __builtin_bit_cast(gs_u32x4, v) ^ mask); }

// MT x 16 rows by 8 x NT x 16 columns, eight wavefronts beside each other: each has all rows and 16 NT columns.  Stages of 32 of K: a ring of
// RING of the rows' parts and one of RING - 1 of each wavefront's own columns.  One barrier a stage, in its middle: behind it the next
// stage's operands are there, the last one of the ring is asked for, and the next columns are split beside the second half's products.
// lane l of a product: row l % 16, columns 4 (l / 16) + 0..3.  W rows past the end are the last one again; nothing stores what comes of them.
// MODE 1, 2: gated (GATED).  2 (PARTS): the results go out as the parts of the rows that the next product reads: a lane's four columns are
// half of its 16 bytes of a fragment.  (Scoring 1,000 tokens at the 1B shape with results and a pass over them / parts: 11.34 / 11.13 ms
// on one card.)
// MODE 3 (ROPE): W is a q/k/v projection with rotary partners in adjacent rows: a lane's four columns are two pairs, which it turns; queries go
// to C, keys and values to their pages.  (us with the parts' pass, product and rotation kernel / this: [3072, 2048] 500 rows 57.9 / 54.7, 1,000 91.2 /
// 84.5, 2,048 158 / 148; [5120, 3072] 500 rows 129 / 111, 1,000 214 / 194.  With a row's look-ups between the stores the gain was half of that.)
struct GsRope {
  const int *positions, *token_seq, *block_table;
  const float2* cos_sin;
  float *kcache, *vcache;      // [pages, nkv, page, hd], [pages, nkv, hd, page]
  int table_width, page_size, nh, nkv, hd, store;
};

// PAIRS: every group of K is an even number of chunks of 128, and a stage's sign is known to the compiler.  Else it is a mask (for all groups:
// 128 x 256 0.5 to 2 % slower; 200 rows of [3072, 3072] in 8 groups of three 32.3 -> 33.2 us).
template <int MT, int NT, int RING, int MODE, bool PAIRS>
__global__ void __launch_bounds__(512, 2)
    gemm_split_kernel(const unsigned char* __restrict__ P, const float* __restrict__ W, float* __restrict__ C, int M, int N, int K, int ldc,
                      int steps_per_group, long long plane, int m_tiles, GsRope rope) {
  constexpr bool GATED = MODE == 1 || MODE == 2, PARTS = MODE == 2, ROPE = MODE == 3;
  static_assert(!GATED || NT == 2, "a gated wavefront has a tile of gate columns and their up columns");
  constexpr int A_LOADS = (3 * MT + 7) / 8, B_LOADS = 2 * NT, LOADS = A_LOADS + B_LOADS;
  constexpr int A_STAGE = MT * 3 * GS_FRAGMENT, B_STAGE = 8 * NT * 2048;
  constexpr int COLUMNS = GATED ? 128 : 128 * NT;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[RING * A_STAGE + (RING - 1) * B_STAGE];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / BLM_WAVE), lane = tid & (BLM_WAVE - 1);
  const int l16 = lane & 15, quad = lane >> 4;
  // neighbouring blocks go to different dies: each die gets a run of the tiles, all rows of a column tile before the next one's
  const int tiles = gridDim.x, die = blockIdx.x & 7, at = die * (tiles >> 3) + min(die, tiles & 7) + (blockIdx.x >> 3);
  const int nt = at / m_tiles, mt = at - nt * m_tiles;
  const int m0 = mt * MT * 16, n0 = nt * COLUMNS, steps_all = K / GS_BK;
  const int s_begin = blockIdx.y * steps_per_group, stages = min(steps_per_group, steps_all - s_begin), last = stages - 1;

  const char* a_base = reinterpret_cast<const char*>(P) + ((size_t)(m0 / 16) * steps_all + s_begin) * (3 * GS_FRAGMENT);
  const char* b_base = reinterpret_cast<const char*>(W + (size_t)n0 * K + (size_t)s_begin * GS_BK);
  const int row_tiles = (M + 15) / 16 - m0 / 16;
  uint32_t a_off[A_LOADS], b_off[B_LOADS], a_to[A_LOADS];
#pragma unroll
  for (int x = 0; x < A_LOADS; ++x) {
    int f = x * 8 + wave;
    if (f >= 3 * MT) f -= 8;              // brings the one before again
    a_off[x] = (uint32_t)min(f / 3, row_tiles - 1) * (uint32_t)steps_all * (3u * GS_FRAGMENT) + (uint32_t)(f % 3) * GS_FRAGMENT + lane * 16u;
    a_to[x] = (uint32_t)f * GS_FRAGMENT;
  }
#pragma unroll
  for (int x = 0; x < B_LOADS; ++x) {
    const int j = x >> 1, r = (x & 1) * 8 + lane / 8, piece = (lane & 7) ^ ((r >> 1) & 7);
    const int n = min(GATED ? wave * 16 + r : wave * 16 * NT + j * 16 + r, N - 1 - n0);
    b_off[x] = ((uint32_t)n + (GATED && j ? (uint32_t)N : 0u)) * (uint32_t)K * 4u + piece * 16u;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(blm_lds_ptr)lds;
  const uint32_t b_to = lds0 + RING * A_STAGE + (uint32_t)wave * (NT * 2048);
  auto fetch = [&](int s, int a_slot, int b_slot) {
    const char *a = a_base + (size_t)s * (3 * GS_FRAGMENT), *b = b_base + (size_t)s * (GS_BK * 4);
#pragma unroll
    for (int x = 0; x < B_LOADS; ++x) blm_dma16_to(b, b_off[x], b_to + (uint32_t)(b_slot * B_STAGE + x * 1024));
#pragma unroll
    for (int x = 0; x < A_LOADS; ++x) blm_dma16_to(a, a_off[x], lds0 + (uint32_t)(a_slot * A_STAGE) + a_to[x]);
  };

  const int b_at = RING * A_STAGE + wave * (NT * 2048) + l16 * 128;
  const int slot0 = (quad ^ ((l16 >> 1) & 7)) * 16, slot1 = ((4 + quad) ^ ((l16 >> 1) & 7)) * 16;
  gs_f32x4 raw[NT][2];
  gs_u32x4 b[2][NT][3];
  auto read_raw = [&](int slot, int j) {
    raw[j][0] = *reinterpret_cast<const gs_f32x4*>(lds + slot * B_STAGE + b_at + j * 2048 + slot0);
    raw[j][1] = *reinterpret_cast<const gs_f32x4*>(lds + slot * B_STAGE + b_at + j * 2048 + slot1);
  };
  // sign: GsPlus, GsMinus or a mask of the sign's bit
  auto split_half = [&](gs_u32x4 (&to)[NT][3], int j, int x, auto sign) {
    uint32_t h[2], m[2], l[2];
    const gs_f32x4 v = gs_signed(raw[j][x], sign);
    gs_split(v[0], v[1], h[0], m[0], l[0]);
    gs_split(v[2], v[3], h[1], m[1], l[1]);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      to[j][0][2 * x + e] = h[e];
      to[j][1][2 * x + e] = m[e];
      to[j][2][2 * x + e] = l[e];
    }
  };
  constexpr int TOGETHER = NT == 1 ? 2 : 1, GROUPS = MT / TOGETHER, HALF = GROUPS > 2 ? GROUPS / 2 : 0;
  constexpr int first[6] = {2, 0, 1, 1, 0, 0}, second[6] = {0, 2, 1, 0, 1, 0};      // small ones first
  gs_u32x4 a[2][TOGETHER][3];
  gs_f32x4 total[MT][NT], t[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) total[i][j] = t[i][j] = gs_f32x4{0.f, 0.f, 0.f, 0.f};
  auto read_a = [&](int set, int slot, int g) {
#pragma unroll
    for (int x = 0; x < TOGETHER; ++x)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        a[set][x][p] = *reinterpret_cast<const gs_u32x4*>(lds + slot * A_STAGE + ((g * TOGETHER + x) * 3 + p) * GS_FRAGMENT + lane * 16);
  };
  auto add = [&](int g, auto sign) {
#pragma unroll
    for (int x = 0; x < TOGETHER; ++x)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        total[g * TOGETHER + x][j] += gs_signed(t[g * TOGETHER + x][j], sign);
        t[g * TOGETHER + x][j] = gs_f32x4{0.f, 0.f, 0.f, 0.f};
      }
  };
  const GsPlus plus;
  const GsMinus minus;
  int a_slot = 0, b_slot = 1;                   // of this stage's rows and of the next one's columns
  // a stage; on entry its first rows' fragments and its columns' parts are in registers
  // (next_sign: that of the next stage's columns, negated where their chunk is subtracted)
  auto stage = [&](int s, auto place_type, auto sign, auto next_sign) __attribute__((always_inline)) {
    constexpr int place = decltype(place_type)::value, now = place & 1, next = now ^ 1;
    const int slot = a_slot, slot1 = slot == RING - 1 ? 0 : slot + 1;
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      const int set = g & 1;
      read_a(set ^ 1, g + 1 < GROUPS ? slot : slot1, g + 1 < GROUPS ? g + 1 : 0);
      if (g == HALF) {
        if (RING > 3 && s + RING - 2 <= last) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((RING - 3) * LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (s + RING - 1 <= last) fetch(s + RING - 1, slot == 0 ? RING - 1 : slot - 1, b_slot == 0 ? RING - 2 : b_slot - 1);
#pragma unroll
        for (int j = 0; j < NT; ++j) read_raw(b_slot, j);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int x = 0; x < TOGETHER; ++x)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            t[g * TOGETHER + x][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gs_bf16x8, b[now][j][first[p]]),
                                                                             __builtin_bit_cast(gs_bf16x8, a[set][x][second[p]]), t[g * TOGETHER + x][j], 0, 0, 0);
      if (place == 3 && g > 0) add(g - 1, sign);
      // the next columns' parts beside the last products
#pragma unroll
      for (int y = 0; y < 2 * NT; ++y)
        if (g - HALF == y * (GROUPS - HALF) / (2 * NT)) split_half(b[next], y >> 1, y & 1, next_sign);
    }
    if (place == 3) add(GROUPS - 1, sign);
    a_slot = slot1;
    b_slot = b_slot == RING - 2 ? 0 : b_slot + 1;
  };
  static_assert(GROUPS % 2 == 0, "the first rows' fragments of every stage lie in the same set");
#pragma unroll
  for (int s = 0; s < RING - 1; ++s)
    if (s <= last) fetch(s, s, s);
  if (RING - 2 <= last) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((RING - 2) * LOADS) : "memory");
  else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    read_raw(0, j);
    split_half(b[0], j, 0, plus);
    split_half(b[0], j, 1, plus);
  }
  read_a(0, 0, 0);
  if constexpr (PAIRS) {
    for (int s = 0; s < stages; s += 8) {
      stage(s, GsInt<0>{}, plus, plus);
      stage(s + 1, GsInt<1>{}, plus, plus);
      stage(s + 2, GsInt<2>{}, plus, plus);
      stage(s + 3, GsInt<3>{}, plus, minus);
      if (s + 4 < stages) {      // (always: without a branch here the compiler mixes both chunks and 128 x 256 spills, 284 -> 387 us)
        stage(s + 4, GsInt<0>{}, minus, minus);
        stage(s + 5, GsInt<1>{}, minus, minus);
        stage(s + 6, GsInt<2>{}, minus, minus);
        stage(s + 7, GsInt<3>{}, minus, plus);
      }
    }
  } else {
    uint32_t sign = 0u;
    const uint32_t flip = 0x80000000u;
    for (int s = 0; s < stages; s += 4) {
      const bool halves = s + 4 == stages && sign == 0u;      // the last one without a second
      stage(s, GsInt<0>{}, sign, sign);
      stage(s + 1, GsInt<1>{}, sign, halves ? flip : sign);
      if (halves) {
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) add(g, plus);
        sign = flip;
      }
      stage(s + 2, GsInt<2>{}, sign, sign);
      stage(s + 3, GsInt<3>{}, sign, sign ^ flip);
      sign ^= flip;
    }
  }

  // Sums that are not numbers.  An operand that is not finite, or rounds to an infinity as a bfloat16, has made NaN of all its products (an infinity
  // less itself, or times a part that is zero); also chunks may have overflowed in opposite directions.  The wavefront asks its rows' first parts and its
  // columns' kinds, by the same instructions, which sums are infinities or NaN whatever the numbers among their operands, and leaves off as soon
  // as all of them are NaN; what is left are sums of finite operands, which the float instructions add up, a tile of rows at a time.
  // (us, 512 rows of [2048, 2048]: clean 127, all rows NaN 134, one NaN or infinity a row or a column 335, a weight a column that rounds to an infinity
  // 900; with every such sum walked by the lane that has it 7,900 in all these cases.  Marked unlikely: in line the code cost a clean prompt 0.9 %.)
  bool any = false;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) any |= total[i][j][e] != total[i][j][e];
  if (__builtin_expect(__any(any), 0)) {
    const float* w[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = GATED ? wave * 16 + l16 : wave * 16 * NT + j * 16 + l16;
      w[j] = W + ((size_t)min(n0 + n, N - 1) + (GATED && j ? (size_t)N : 0)) * K + (size_t)s_begin * GS_BK + quad * 4;
    }
    const char* rows = a_base + lane * 16;
    const size_t row_tile = (size_t)steps_all * (3 * GS_FRAGMENT);
    auto number = [](float x) { return (__float_as_uint(x) & 0x7f800000u) != 0x7f800000u; };
    for (int s = 0; s < stages; ++s) {
      gs_u32x4 kind[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          const gs_f32x4 v = *reinterpret_cast<const gs_f32x4*>(w[j] + s * GS_BK + x * 16);
          kind[j][2 * x] = gs_kind(v[0]) | gs_kind(v[1]) << 16;
          kind[j][2 * x + 1] = gs_kind(v[2]) | gs_kind(v[3]) << 16;
        }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const gs_u32x4 first_part = *reinterpret_cast<const gs_u32x4*>(rows + min(i, row_tiles - 1) * row_tile + (size_t)s * (3 * GS_FRAGMENT));
#pragma unroll
        for (int j = 0; j < NT; ++j)
          t[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gs_bf16x8, kind[j]), __builtin_bit_cast(gs_bf16x8, first_part), t[i][j], 0, 0, 0);
      }
      if (s % 8 == 0) {
        bool open = false;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) open |= total[i][j][e] != total[i][j][e] && t[i][j][e] == t[i][j][e];
        if (!__any(open)) break;
      }
    }
    uint32_t left = 0;           // tiles of rows
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      bool open = false;
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (total[i][j][e] != total[i][j][e]) {
            if (number(t[i][j][e])) open = true;
            else total[i][j][e] = t[i][j][e];
          }
      if (__any(open)) left |= 1u << i;
    }
    for (; left != 0; left &= left - 1) {
      const int tile = __builtin_ctz(left);
      const char* row = rows + min(tile, row_tiles - 1) * row_tile;
      gs_f32x4 sum[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) sum[j] = gs_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
      for (int s = 0; s < stages; ++s) {
        gs_u32x4 part[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) part[p] = *reinterpret_cast<const gs_u32x4*>(row + (size_t)s * (3 * GS_FRAGMENT) + p * GS_FRAGMENT);
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const gs_f32x4 v = *reinterpret_cast<const gs_f32x4*>(w[j] + s * GS_BK + x * 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int at = 2 * x + e / 2;
              const float a = e % 2 ? gs_high(part[0][at]) + (gs_high(part[1][at]) + gs_high(part[2][at]))
                                    : gs_low(part[0][at]) + (gs_low(part[1][at]) + gs_low(part[2][at]));
              sum[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], a, sum[j], 0, 0, 0);
            }
          }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
        if (i == tile)
#pragma unroll
          for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (total[i][j][e] != total[i][j][e] && number(t[i][j][e])) total[i][j][e] = sum[j][e];
    }
  }

  float* out = C + (size_t)blockIdx.y * plane;
  // ROPE: where row m goes (columns of key and value heads of a row without a page go nowhere), and the angles of a lane's two pairs: asked for
  // for all rows at once, since behind the first store every look-up is a trip of its own
  auto page_of = [&](int b, int pos) { return rope.store && b >= 0 ? rope.block_table[(size_t)b * rope.table_width + pos / rope.page_size] : -1; };
  auto angle = [&](int pos, int d) { return rope.cos_sin[(size_t)pos * (rope.hd / 2) + d / 2]; };
  auto turn = [&](float2 cs, float& x, float& y) {
    const float t = x;
    x = t * cs.x - y * cs.y;
    y = t * cs.y + y * cs.x;
  };
  int slots[ROPE ? MT : 1], pages[ROPE ? MT : 1];
  float2 angles[ROPE ? MT : 1][NT][2];
  if constexpr (ROPE) {
    int seqs[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = min(m0 + i * 16 + l16, M - 1);
      slots[i] = rope.positions[m];
      seqs[i] = rope.token_seq[m];
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      pages[i] = page_of(seqs[i], slots[i]);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int d = min(n0 + wave * 16 * NT + j * 16 + quad * 4, N - 4) % rope.hd;
        angles[i][j][0] = angle(slots[i], d);
        angles[i][j][1] = angle(slots[i], d + 2);
      }
      slots[i] %= rope.page_size;
    }
  }
  int slot = 0, page = -1;
  auto value_at = [&](int head, int d) {
    return rope.vcache + (((size_t)page * rope.nkv + (head - rope.nh - rope.nkv)) * rope.hd + d) * rope.page_size + slot;
  };
  auto key_at = [&](int head, int d) { return rope.kcache + (((size_t)page * rope.nkv + (head - rope.nh)) * rope.page_size + slot) * rope.hd + d; };
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + i * 16 + l16;
    if constexpr (ROPE) {
      slot = slots[i];
      page = pages[i];
    }
#pragma unroll
    for (int j = 0; j < (GATED ? 1 : NT); ++j) {
      const int n = n0 + wave * 16 * (GATED ? 1 : NT) + j * 16 + quad * 4;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = GATED ? gs_silu_times(total[i][0][e], total[i][NT - 1][e]) : total[i][j][e];
      if constexpr (ROPE) {
        if (m >= M || n >= N) continue;
        const int head = n / rope.hd, d = n - head * rope.hd;
        if (head < rope.nh + rope.nkv) {
          turn(angles[i][j][0], v[0], v[1]);
          turn(angles[i][j][1], v[2], v[3]);
          if (head < rope.nh) *reinterpret_cast<float4*>(out + (size_t)m * ldc + n) = make_float4(v[0], v[1], v[2], v[3]);
          else if (page >= 0) *reinterpret_cast<float4*>(key_at(head, d)) = make_float4(v[0], v[1], v[2], v[3]);
        } else if (page >= 0) {
          float* to = value_at(head, d);
#pragma unroll
          for (int e = 0; e < 4; ++e) to[e * rope.page_size] = v[e];
        }
      } else if constexpr (PARTS) {
        if (m0 + i * 16 >= M || n >= N) continue;
        uint32_t part[2][3];
#pragma unroll
        for (int e = 0; e < 2; ++e) gs_split_any(m < M ? v[2 * e] : 0.f, m < M ? v[2 * e + 1] : 0.f, part[e][0], part[e][1], part[e][2]);
        unsigned char* to = gs_part_of(C, m, n, N);
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(to + q * GS_FRAGMENT) = make_uint2(part[0][q], part[1][q]);
      } else {
        if (m < M && n < N) *reinterpret_cast<float4*>(out + (size_t)m * ldc + n) = make_float4(v[0], v[1], v[2], v[3]);
      }
    }
  }
}

#define GS_LAUNCH(MT, NT, RING, MODE, PAIRS, rope)                                                                                          \
  hipLaunchKernelGGL((gemm_split_kernel<MT, NT, RING, MODE, PAIRS>), grid, block, 0, stream, (const unsigned char*)P, (const float*)W, (float*)C, \
                     M, N, K, ldc, steps, (long long)M * N, m_tiles, rope)
#define GS_RUN(MT, NT, RING, MODE, rope)                       \
  do {                                                         \
    if (K % 256 == 0 && steps % 8 == 0) GS_LAUNCH(MT, NT, RING, MODE, true, rope); \
    else GS_LAUNCH(MT, NT, RING, MODE, false, rope);           \
  } while (0)

// P: the parts of A [M, K] (split_rows).  rows x columns: a block's tile, 128 or 64 by 256 or 128 (gated: gate and up columns
// together, 256).  gated: 0, 1, or 2 for results that come as parts of rows of N columns, as split_rows makes them.  groups > 1: K in that many groups, C holds a plane of M * N for each (contiguous, ldc = N), which the reader adds up.
extern "C" int blm_gemm_split(const void* P, const void* W, void* C, int M, int N, int K, int ldc, int gated, int groups, int rows,
                              int columns, hipStream_t stream) {
  BLM_REQUIRE(M > 0 && N > 0 && N % 16 == 0 && K > 0 && K % 128 == 0 && ldc >= N && ldc % 4 == 0, "gemm_split: sizes M=%d N=%d K=%d ldc=%d not supported",
              M, N, K, ldc);
  BLM_REQUIRE(((uintptr_t)P % 16) == 0 && ((uintptr_t)W % 16) == 0 && ((uintptr_t)C % 16) == 0, "gemm_split: operands must be 16-byte aligned");
  const int steps = groups >= 1 ? (K / 128 + groups - 1) / groups * 4 : 0;
  BLM_REQUIRE(groups >= 1 && groups <= 64 && (groups == 1 || (!gated && ldc == N)) && (groups - 1) * steps * GS_BK < K, "gemm_split: %d groups of K=%d", groups, K);
  BLM_REQUIRE(gated >= 0 && gated <= 2 && (gated != 2 || (N % GS_BK == 0 && ldc == N)), "gemm_split: gating %d of %d columns", gated, N);
  BLM_REQUIRE(((gated ? N : 0) + 256LL) * K * 4 < (1LL << 32), "gemm_split: gated matrices of 4 GiB and more are not supported (N=%d K=%d)", N, K);
  BLM_REQUIRE((rows == 128 || rows == 64) && (columns == 256 || (columns == 128 && !gated)), "gemm_split: tile %d x %d", rows, columns);
  const int per = gated ? columns / 2 : columns;
  const int m_tiles = (M + rows - 1) / rows, n_tiles = (N + per - 1) / per;
  const long long blocks = (long long)m_tiles * n_tiles;
  BLM_REQUIRE(blocks < 2147483647LL, "gemm_split: too many tiles");
  dim3 grid((unsigned)blocks, (unsigned)groups), block(512);
  if (gated == 2) {
    if (rows == 128) GS_RUN(8, 2, 3, 2, GsRope{});
    else GS_RUN(4, 2, 4, 2, GsRope{});
  } else if (gated) {
    if (rows == 128) GS_RUN(8, 2, 3, 1, GsRope{});
    else GS_RUN(4, 2, 4, 1, GsRope{});
  } else if (columns == 256) {
    if (rows == 128) GS_RUN(8, 2, 3, 0, GsRope{});
    else GS_RUN(4, 2, 4, 0, GsRope{});
  } else {
    if (rows == 128) GS_RUN(8, 1, 3, 0, GsRope{});
    else GS_RUN(4, 1, 4, 0, GsRope{});
  }
  BLM_LAUNCH_CHECK("gemm_split");
  return 0;
}

// The q/k/v projection of many rows with the rotation and the page writes behind it.  Wq: W_qkv [(nh + 2 nkv) * hd, K], rotary partners in adjacent
// rows; qkv_out [M, ldc], of which the first nh * hd columns (the turned queries) are written; store = 0: no keys and values.
extern "C" int blm_gemm_split_qkv_rope(const void* P, const void* Wq, void* qkv_out, const int* positions, const int* token_seq, const int* block_table,
                                       int table_width, const float* cos_sin, void* kcache, void* vcache, int page_size, int M, int K, int ldc, int nh,
                                       int nkv, int hd, int store, int rows, int columns, hipStream_t stream) {
  BLM_REQUIRE(nh > 0 && nkv > 0 && hd > 0 && hd % 4 == 0 && page_size > 0 && table_width > 0, "gemm_split_qkv_rope: bad geometry (head size %d)", hd);
  const int N = (nh + 2 * nkv) * hd;
  BLM_REQUIRE(M > 0 && N % 16 == 0 && K > 0 && K % 128 == 0 && ldc >= nh * hd && ldc % 4 == 0, "gemm_split_qkv_rope: sizes M=%d N=%d K=%d ldc=%d not supported", M, N, K, ldc);
  BLM_REQUIRE(((uintptr_t)P % 16) == 0 && ((uintptr_t)Wq % 16) == 0 && ((uintptr_t)qkv_out % 16) == 0 && ((uintptr_t)kcache % 16) == 0 && ((uintptr_t)vcache % 4) == 0 &&
                  ((uintptr_t)cos_sin % 8) == 0, "gemm_split_qkv_rope: operands must be 16-byte aligned (angles 8-byte)");
  BLM_REQUIRE((rows == 128 || rows == 64) && (columns == 256 || columns == 128), "gemm_split_qkv_rope: tile %d x %d", rows, columns);
  const int m_tiles = (M + rows - 1) / rows, used = store ? N : nh * hd;
  const long long blocks = (long long)m_tiles * ((used + columns - 1) / columns);
  BLM_REQUIRE(blocks < 2147483647LL, "gemm_split_qkv_rope: too many tiles");
  const GsRope rope{positions, token_seq, block_table, (const float2*)cos_sin, (float*)kcache, (float*)vcache,
                    table_width, page_size, nh, nkv, hd, store};
  const void *W = Wq, *C = qkv_out;
  const int steps = K / GS_BK;
  dim3 grid((unsigned)blocks, 1), block(512);
  if (columns == 256) {
    if (rows == 128) GS_RUN(8, 2, 3, 3, rope);
    else GS_RUN(4, 2, 4, 3, rope);
  } else {
    if (rows == 128) GS_RUN(8, 1, 3, 3, rope);
    else GS_RUN(4, 1, 4, 3, rope);
  }
#undef GS_RUN
#undef GS_LAUNCH
  BLM_LAUNCH_CHECK("gemm_split_qkv_rope");
  return 0;
}
