// Latent attention over prompts with keys and values expanded per head (bfloat16).  The absorbed form (latent_attention.hip)
// works on 2 R + Dr lanes per query and row (1,088 at R = 512, Dr = 64) and is the right one for single tokens; a prompt of some
// hundred tokens per sequence pays the expansion of every row it sees once, 2 R (Dn + Dv) operations per row and head, and then
// works on Dn + Dr + Dv lanes (320): a third of the operations at 2,048 tokens.
//   latent_expand : plain keys [page][head][64][Dn] and transposed values [page][head][Dv][64] of the rows in the cache, page
//                   by page, up to each sequence's length; pages are numbered sequence * pages_per_seq + page
//   latent_prompt : attention over them; the turned key part, the same for all heads, comes from the cache rows themselves
// Measured (us a layer, 2,048 tokens, 16 heads, R = 512, Dn = Dv = 128, Dr = 64, before: absorbed with its two products per
// head): window of 1,024 651 -> 61 (expansion 20, attention 41, 370 TFLOP/s of its own work); three prompts of 333 to 1,201
// tokens without a window 564 -> 64.
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 lp_bf16x8;
typedef __attribute__((ext_vector_type(16))) float lp_f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int lp_u32x4;
#define LP_PAGE 64
#define LP_WAVES 4
#define LP_QUERIES 32    // per wavefront

__device__ __forceinline__ lp_f32x16 lp_mfma(lp_u32x4 a, lp_u32x4 b, lp_f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(lp_bf16x8, a), __builtin_bit_cast(lp_bf16x8, b), c, 0, 0, 0);
}

// acc + both numbers of a pair of bf16, one instruction
__device__ __forceinline__ float lp_add_pair(uint32_t pair, float acc) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, 0x3f803f80u), acc, false);
}

__device__ __forceinline__ constexpr int lp_key_of(int row) { return (row & ~12) | ((row & 4) << 1) | ((row & 8) >> 1); }
template <int LANES>     // lanes of a shared-memory row: 32, 64 or 128
__device__ __forceinline__ int lp_twist(int row) { return LANES == 128 ? row & 15 : LANES == 64 ? (row >> 1) & 7 : (row >> 2) & 3; }

// Rows of LANES lanes straight into shared memory by all wavefronts of the block: row r of the tile from src + key(r) * stride.
template <int ROWS, int LANES, bool DEAL>
struct LpRows {
  static constexpr int PIECES = LANES / 8, PER_LOAD = 64 / PIECES, LOADS = ROWS / PER_LOAD / LP_WAVES;
  static_assert(ROWS % (PER_LOAD * LP_WAVES) == 0, "whole loads per wavefront");
  uint32_t offset[LOADS];
  __device__ __forceinline__ void init(int wave, int lane, uint32_t row_bytes) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int r = (i * LP_WAVES + wave) * PER_LOAD + lane / PIECES;
      offset[i] = (uint32_t)(DEAL ? lp_key_of(r) : r) * row_bytes + (uint32_t)(((lane % PIECES) ^ lp_twist<LANES>(r)) * 16);
    }
  }
  __device__ __forceinline__ void fetch(const bf16* src, uint32_t lds, int wave) const {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      blm_dma16_to(reinterpret_cast<const char*>(src), offset[i], lds + (uint32_t)((i * LP_WAVES + wave) * 1024));
  }
};
template <int LANES>
__device__ __forceinline__ lp_u32x4 lp_fragment(const bf16* tile, int row, int piece) {
  return *reinterpret_cast<const lp_u32x4*>(tile + row * LANES + ((piece ^ lp_twist<LANES>(row)) * 8));
}

// ---------------------------------------------------------------------------------------------------------------------
// A block has one page of one sequence and one head; latents and both weights come in steps of 64 elements of R straight into
// one of two buffers of shared memory.  A wavefront has 32 lanes of the keys and 32 of the values (64 lanes: of one of the two).
// A head's blocks are one die's, whose L2 then holds its weights.  With the weights' fragments straight from memory (32 bytes
// of 32 rows an instruction) the kernel took 34 us for 2,048 rows and 16 heads (40 with two pages a block), against 20.
// ---------------------------------------------------------------------------------------------------------------------
#define LP_STEP 64
template <int D>     // lanes of a head's keys and of its values, 64 or 128
__global__ void __launch_bounds__(LP_WAVES* BLM_WAVE)
    latent_expand_kernel(const bf16* __restrict__ kcache, const bf16* __restrict__ w_uk, const bf16* __restrict__ w_uv,
                         bf16* __restrict__ keys, bf16* __restrict__ values, const int* __restrict__ cu_seqlens,
                         const int* __restrict__ lens_after, const int* __restrict__ block_table, int table_width, int pages_per_seq,
                         int H, int R, int Dr, int window) {
  constexpr int LE = LP_PAGE * LP_STEP, WE = D * LP_STEP, STAGE = LE + 2 * WE;
  extern __shared__ __attribute__((aligned(1024))) bf16 lds[];
  const int h = blockIdx.x, page = blockIdx.y, seq = blockIdx.z;
  const int len = lens_after[seq], n_new = cu_seqlens[seq + 1] - cu_seqlens[seq];
  if (n_new <= 0 || page * LP_PAGE >= len) return;
  if (window > 0 && page * LP_PAGE + LP_PAGE - 1 <= len - n_new - window) return;    // the step's first query sees none of it
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / BLM_WAVE), lane = tid & (BLM_WAVE - 1);
  const int c = lane & 31, hb = lane >> 5;
  const bf16* src = kcache + (size_t)__builtin_amdgcn_readfirstlane(block_table[(size_t)seq * table_width + page]) * LP_PAGE * (R + Dr);
  LpRows<LP_PAGE, LP_STEP, false> l_rows;
  LpRows<D, LP_STEP, false> w_rows;
  l_rows.init(wave, lane, (uint32_t)(R + Dr) * 2);
  w_rows.init(wave, lane, (uint32_t)R * 2);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(blm_lds_ptr)lds;
  auto fetch = [&](int k0, int buf) {
    const uint32_t to = lds0 + (uint32_t)(buf * STAGE * 2);
    l_rows.fetch(src + k0, to, wave);
    w_rows.fetch(w_uk + (size_t)h * D * R + k0, to + LE * 2, wave);
    w_rows.fetch(w_uv + (size_t)h * D * R + k0, to + (LE + WE) * 2, wave);
  };
  const int n0 = wave * 32 % D;
  const bool do_keys = D == 128 || wave < 2, do_values = D == 128 || wave >= 2;
  lp_f32x16 k_acc[2], v_acc[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) k_acc[t][v] = v_acc[t][v] = 0.f;
  fetch(0, 0);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  for (int k0 = 0, buf = 0; k0 < R; k0 += LP_STEP, buf ^= 1) {
    if (k0 + LP_STEP < R) fetch(k0 + LP_STEP, buf ^ 1);       // nobody reads that buffer any more
    const bf16* stage = lds + buf * STAGE;
#pragma unroll
    for (int x = 0; x < LP_STEP / 16; ++x) {
      lp_u32x4 lat[2], kw, vw;
#pragma unroll
      for (int t = 0; t < 2; ++t) lat[t] = lp_fragment<LP_STEP>(stage, t * 32 + c, 2 * x + hb);
      if (do_keys) kw = lp_fragment<LP_STEP>(stage + LE, n0 + c, 2 * x + hb);
      if (do_values) vw = lp_fragment<LP_STEP>(stage + LE + WE, n0 + c, 2 * x + hb);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (do_keys) k_acc[t] = lp_mfma(kw, lat[t], k_acc[t]);        // rows: lanes of the head, columns: keys
        if (do_values) v_acc[t] = lp_mfma(lat[t], vw, v_acc[t]);      // rows: keys, columns: lanes of the head
      }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  // Row 8 (v / 4) + 4 hb + v % 4 of a result is four neighbours in one lane: keys are stored lane by lane of the head, values
  // token by token, eight bytes at a time.  Places behind the sequence's end hold whatever a page held before: their values are
  // zeros (a score of theirs is never used, but a probability of zero meets the value).
  const size_t at = ((size_t)(seq * pages_per_seq + page) * H + h) * LP_PAGE * D;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int row = 8 * g + 4 * hb;
      if (do_keys)
        *reinterpret_cast<uint2*>(keys + at + (size_t)(t * 32 + c) * D + n0 + row) =
            make_uint2(f32x2_to_bf16x2_bits(k_acc[t][4 * g], k_acc[t][4 * g + 1]), f32x2_to_bf16x2_bits(k_acc[t][4 * g + 2], k_acc[t][4 * g + 3]));
      if (do_values) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = page * LP_PAGE + t * 32 + row + e < len ? v_acc[t][4 * g + e] : 0.f;
        *reinterpret_cast<uint2*>(values + at + (size_t)(n0 + c) * LP_PAGE + t * 32 + row) = make_uint2(f32x2_to_bf16x2_bits(v[0], v[1]), f32x2_to_bf16x2_bits(v[2], v[3]));
      }
    }
}

// ---------------------------------------------------------------------------------------------------------------------
// Four wavefronts of 32 queries of one head share every page, which comes straight from global memory into one of two buffers
// while the other is worked on.  S^T = K Q^T and O^T = V^T P^T on 32x32x16 products, as in the 32-query attention over plain
// keys: rows of a page's score tiles are keys in an order (bits 2 and 3 of the key's number exchanged) in which the eight
// probabilities that a lane has for one product with the values belong to neighbouring keys.  Shared memory rows are as long as
// in memory, their 16-byte pieces permuted: 16 or 8 pieces a row by the row's number (or half of it) modulo their count.
// A head's blocks follow each other on one die, the longest queries first.
// ---------------------------------------------------------------------------------------------------------------------
template <int D, int DR>
__global__ void __launch_bounds__(LP_WAVES* BLM_WAVE, 2)
    latent_prompt_kernel(const bf16* __restrict__ q, int ld_q, const bf16* __restrict__ q_turned, bf16* __restrict__ out,
                         const int* __restrict__ positions, const int* __restrict__ cu_seqlens, const int* __restrict__ block_table,
                         int table_width, const bf16* __restrict__ kcache, const bf16* __restrict__ keys,
                         const bf16* __restrict__ values, int pages_per_seq, int H, int R, float scale2, int window,
                         const float* __restrict__ sinks) {
  constexpr int KE = LP_PAGE * D, TE = LP_PAGE * DR, STAGE = 2 * KE + TE;     // elements of keys (and values), turned parts, all
  extern __shared__ __attribute__((aligned(1024))) bf16 lds[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / BLM_WAVE), lane = tid & (BLM_WAVE - 1);
  const int c = lane & 31, hb = lane >> 5;
  const int h = blockIdx.x % H, seq = blockIdx.y;
  const int row0 = cu_seqlens[seq], n_q = cu_seqlens[seq + 1] - row0;
  const int first = ((int)gridDim.x / H - 1 - (int)blockIdx.x / H) * LP_WAVES * LP_QUERIES;
  if (first >= n_q) return;
  const int mine = min(first + wave * LP_QUERIES, n_q - 1), nq = min(LP_QUERIES, n_q - mine);   // a wavefront past the end repeats the last query
  const bool active = first + wave * LP_QUERIES < n_q;
  const int row = row0 + mine + min(c, nq - 1);
  const int pos = positions[row], pos_first = positions[row0 + mine], pos_last = positions[row0 + mine + nq - 1];
  const int block_first = positions[row0 + first], block_last = positions[row0 + min(first + LP_WAVES * LP_QUERIES, n_q) - 1];
  const int lo = window > 0 ? max(0, pos - window + 1) : 0, lo_first = window > 0 ? max(0, pos_first - window + 1) : 0;
  const int lo_last = window > 0 ? max(0, pos_last - window + 1) : 0;
  const int page_begin = (window > 0 ? max(0, block_first - window + 1) : 0) / LP_PAGE, page_end = block_last / LP_PAGE + 1;
  const int* pages = block_table + (size_t)seq * table_width;

  lp_u32x4 qf[D / 16 + DR / 16];
  {
    const bf16* plain = q + (size_t)row * ld_q + (size_t)h * (D + DR) + hb * 8;
    const bf16* turned = q_turned + ((size_t)row * H + h) * DR + hb * 8;
#pragma unroll
    for (int s = 0; s < D / 16; ++s) qf[s] = *reinterpret_cast<const lp_u32x4*>(plain + s * 16);
#pragma unroll
    for (int s = 0; s < DR / 16; ++s) qf[D / 16 + s] = *reinterpret_cast<const lp_u32x4*>(turned + s * 16);
  }
  LpRows<LP_PAGE, D, true> k_rows;
  LpRows<D, LP_PAGE, false> v_rows;
  LpRows<LP_PAGE, DR, true> t_rows;
  k_rows.init(wave, lane, D * 2);
  v_rows.init(wave, lane, LP_PAGE * 2);
  t_rows.init(wave, lane, (uint32_t)(R + DR) * 2);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(blm_lds_ptr)lds;
  auto fetch = [&](int page, int buf) {
    const size_t at = ((size_t)(seq * pages_per_seq + page) * H + h) * KE;
    const uint32_t to = lds0 + (uint32_t)(buf * STAGE * 2);
    k_rows.fetch(keys + at, to, wave);
    v_rows.fetch(values + at, to + KE * 2, wave);
    t_rows.fetch(kcache + (size_t)__builtin_amdgcn_readfirstlane(pages[page]) * LP_PAGE * (R + DR) + R, to + KE * 4, wave);
  };
  float m = sinks ? sinks[h] * 1.4426950408889634f : -INFINITY;
  float l = sinks && hb == 0 ? 1.f : 0.f;              // the two lanes of a query add theirs up
  lp_f32x16 o[D / 32];
#pragma unroll
  for (int d = 0; d < D / 32; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[d][v] = 0.f;
  fetch(page_begin, 0);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  for (int page = page_begin; page < page_end; ++page) {
    const bf16* stage = lds + ((page - page_begin) & 1) * STAGE;
    if (page + 1 < page_end) fetch(page + 1, (page + 1 - page_begin) & 1);   // nobody reads that buffer any more
    const int key0 = page * LP_PAGE;
    if (key0 <= pos_last && key0 + LP_PAGE > lo_first) {
      lp_f32x16 s[2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) s[t][v] = 0.f;
#pragma unroll
      for (int x = 0; x < D / 16; ++x)
#pragma unroll
        for (int t = 0; t < 2; ++t) s[t] = lp_mfma(lp_fragment<D>(stage, t * 32 + c, 2 * x + hb), qf[x], s[t]);
#pragma unroll
      for (int x = 0; x < DR / 16; ++x)
#pragma unroll
        for (int t = 0; t < 2; ++t) s[t] = lp_mfma(lp_fragment<DR>(stage + 2 * KE, t * 32 + c, 2 * x + hb), qf[D / 16 + x], s[t]);
      if (key0 + LP_PAGE - 1 > pos_first || key0 < lo_last) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int key = key0 + t * 32 + lp_key_of(8 * (v >> 2) + 4 * hb + (v & 3));
            s[t][v] = key <= pos && key >= lo ? s[t][v] : -INFINITY;
          }
      }
      float top = s[0][0];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) top = blm_max(top, s[t][v]);
      float a, b;
      blm_swap32(top, a, b);
      const float m_new = blm_max(m, blm_max(a, b) * scale2);
      const float base = m_new == -INFINITY ? 0.f : m_new, keep = __builtin_amdgcn_exp2f(m - base);
      // the denominator takes the rounded probabilities that the values meet: their roundings then cancel where the values agree
      float sum = 0.f;
      lp_u32x4 p[4];        // probabilities of the lane's eight keys of each sixteen
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int v = 0; v < 16; v += 2) {
          const float x = __builtin_amdgcn_exp2f(fmaf(s[t][v], scale2, -base)), y = __builtin_amdgcn_exp2f(fmaf(s[t][v + 1], scale2, -base));
          const uint32_t pair = f32x2_to_bf16x2_bits(x, y);
          sum = lp_add_pair(pair, sum);
          p[t * 2 + v / 8][v % 8 / 2] = pair;
        }
      l = l * keep + sum;
      m = m_new;
#pragma unroll
      for (int d = 0; d < D / 32; ++d)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[d][v] *= keep;
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int d = 0; d < D / 32; ++d) o[d] = lp_mfma(lp_fragment<LP_PAGE>(stage + KE, d * 32 + c, 2 * x + hb), p[x], o[d]);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  float a, b;
  blm_swap32(l, a, b);
  if (!active || c >= nq) return;
  const float inv = 1.0f / (a + b);
  bf16* orow = out + ((size_t)row * H + h) * D;
#pragma unroll
  for (int d = 0; d < D / 32; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<uint2*>(orow + d * 32 + 8 * g + 4 * hb) =
          make_uint2(f32x2_to_bf16x2_bits(o[d][4 * g] * inv, o[d][4 * g + 1] * inv), f32x2_to_bf16x2_bits(o[d][4 * g + 2] * inv, o[d][4 * g + 3] * inv));
}

extern "C" int blm_latent_prompt_supported(int R, int Dn, int Dr, int Dv, int page_size) {
  return page_size == LP_PAGE && Dn == Dv && (Dn == 64 || Dn == 128) && (Dr == 32 || Dr == 64) && R > 0 && R % LP_STEP == 0 ? 1 : 0;
}
static size_t lp_prompt_lds(int D, int Dr) { return (size_t)2 * (2 * LP_PAGE * D + LP_PAGE * Dr) * 2; }

// Once per device, outside any stream capture: the kernels use more shared memory than a kernel gets without asking.
extern "C" int blm_latent_prompt_init() {
  const void* kernels[] = {(const void*)latent_expand_kernel<64>, (const void*)latent_expand_kernel<128>, (const void*)latent_prompt_kernel<64, 32>,
                           (const void*)latent_prompt_kernel<64, 64>, (const void*)latent_prompt_kernel<128, 32>, (const void*)latent_prompt_kernel<128, 64>};
  for (const void* k : kernels) {
    const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 81920);
    BLM_REQUIRE(e == hipSuccess, "latent_prompt_init: cannot raise the shared memory limit: %s", hipGetErrorString(e));
  }
  return 0;
}

// keys, values: workspaces of n_seqs * pages_per_seq pages of H * 64 * D elements each; pages_per_seq covers every sequence's
// length and the page table is at least as wide.
extern "C" int blm_latent_prompt(const void* q, int ld_q, const void* q_turned, void* out, const int* positions, const int* cu_seqlens,
                                 const int* lens_after, const int* block_table, int table_width, const void* kcache, const void* w_uk,
                                 const void* w_uv, void* keys, void* values, int pages_per_seq, int n_seqs, int max_new, int H, int R,
                                 int Dn, int Dr, int Dv, float scale, int window, const float* sinks, hipStream_t stream) {
  BLM_REQUIRE(blm_latent_prompt_supported(R, Dn, Dr, Dv, LP_PAGE), "latent_prompt: sizes R=%d Dn=%d Dr=%d Dv=%d not supported", R, Dn, Dr, Dv);
  BLM_REQUIRE(n_seqs > 0 && n_seqs <= 65535 && max_new > 0 && H > 0 && pages_per_seq > 0 && pages_per_seq <= 65535 && pages_per_seq <= table_width,
              "latent_prompt: bad sizes n_seqs=%d max_new=%d H=%d pages=%d of %d", n_seqs, max_new, H, pages_per_seq, table_width);
  BLM_REQUIRE(scale > 0.f && window >= 0, "latent_prompt: the scale must be positive");
  BLM_REQUIRE(ld_q % 8 == 0 && ld_q >= H * (Dn + Dr) && ((uintptr_t)q % 16) == 0 && ((uintptr_t)kcache % 16) == 0 && ((uintptr_t)w_uk % 16) == 0 &&
                  ((uintptr_t)w_uv % 16) == 0, "latent_prompt: rows must start at multiples of 16 bytes");
  const long long blocks = (long long)H * ((max_new + LP_WAVES * LP_QUERIES - 1) / (LP_WAVES * LP_QUERIES));
  BLM_REQUIRE(blocks < 2147483647LL, "latent_prompt: too many queries");
  dim3 block(LP_WAVES * BLM_WAVE), grid1((unsigned)H, (unsigned)pages_per_seq, (unsigned)n_seqs), grid2((unsigned)blocks, (unsigned)n_seqs);
#define BLM_LP(D, DR)                                                                                                      \
  do {                                                                                                                     \
    hipLaunchKernelGGL((latent_expand_kernel<D>), grid1, block, (size_t)2 * (LP_PAGE + 2 * D) * LP_STEP * 2, stream, (const bf16*)kcache, (const bf16*)w_uk, \
                       (const bf16*)w_uv, (bf16*)keys, (bf16*)values, cu_seqlens, lens_after, block_table, table_width, pages_per_seq, H, R, DR, window); \
    BLM_LAUNCH_CHECK("latent_expand");                                                                                     \
    hipLaunchKernelGGL((latent_prompt_kernel<D, DR>), grid2, block, lp_prompt_lds(D, DR), stream, (const bf16*)q, ld_q, (const bf16*)q_turned, \
                       (bf16*)out, positions, cu_seqlens, block_table, table_width, (const bf16*)kcache, (const bf16*)keys, (const bf16*)values, \
                       pages_per_seq, H, R, scale * 1.4426950408889634f, window, sinks);                                   \
    BLM_LAUNCH_CHECK("latent_prompt");                                                                                     \
  } while (0)
  if (Dn == 64 && Dr == 32) BLM_LP(64, 32);
  else if (Dn == 64) BLM_LP(64, 64);
  else if (Dr == 32) BLM_LP(128, 32);
  else BLM_LP(128, 64);
#undef BLM_LP
  return 0;
}
