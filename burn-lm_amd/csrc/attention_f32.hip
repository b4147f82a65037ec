// Float32 attention over the paged cache on the matrix cores' float instruction (v_mfma_f32_16x16x4_f32: float operands,
// products and sums), for head sizes of a multiple of four up to 128 and pages of 64 keys; other sizes take attn_paged.
// Same storage as there: key pages [kv head][token][head_dim], value pages [kv head][head_dim][token].
//
// Scores come as S^T = K Q^T and results as O^T = V^T P^T, so that nothing is transposed on the way: lane l of a product holds
// the scores of query l % 16 with keys 4 (l / 16) + 0..3 of a tile of sixteen, which is just what it has to supply to the
// product with the values, whose fragments are four neighbouring tokens of a value row.  Which four elements of a head an
// instruction takes is free as long as queries and keys agree: a lane takes four neighbours, one 16-byte read for four
// instructions.
//   attn_prefill_f32 : a wavefront has sixteen queries of one head, the four of a block share the pages through shared memory
//   attn_decode_f32  : the sixteen columns are the heads of one group at one token; wavefronts take pages in turn, the last ones in
//                      halves or quarters
#include <type_traits>

#include "attn_merge.h"
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;
#define AF_PAGE 64
#define AF_WAVES 4        // of a block of prompts
#define AF_DECODE_WAVES 8  // of a block of single tokens: two to a SIMD, so that one's loads are under way while the other multiplies

__device__ __forceinline__ f32x4 af_load(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 af_mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ bool af_visible(int key, int pos, int window) { return key <= pos && (window <= 0 || pos - key < window); }

template <int V>
using AfInt = std::integral_constant<int, V>;

// Running softmax of one page: s[t][v] holds the scaled scores of this lane's query (l % 16) with keys 16 t + 4 (l / 16) + v,
// -infinity where the query does not see the key; they become probabilities against the new maximum.  l is this lane's part
// of the sum.  Returns the factor for what was summed before.
template <int TILES = 4>
__device__ __forceinline__ float af_softmax(f32x4* s, float& m, float& l) {
  float top = s[0][0];
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) top = fmaxf(top, s[t][v]);
  const float m_new = fmaxf(m, rows_max(top));
  const float base = m_new == -INFINITY ? 0.f : m_new;       // nothing seen yet: every probability is exp(-inf)
  const float keep = expf(m - base);
  float sum = 0.f;
#pragma unroll
  for (int t = 0; t < TILES; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      s[t][v] = expf(s[t][v] - base);
      sum += s[t][v];
    }
  l = l * keep + sum;
  m = m_new;
  return keep;
}

// One query of one head the plain way, by a whole wavefront: for queries whose result is not finite.  A product on the matrix
// cores multiplies values that the query does not see with a probability of zero, which an infinite value turns into NaN.
__device__ void af_plain_query(const float* __restrict__ qrow, float* __restrict__ out, int pos, const int* __restrict__ pages,
                               const float* __restrict__ kcache, const float* __restrict__ vcache, int nkv, int kvh, int hd,
                               float scale, int window) {
  const int lane = threadIdx.x & (BLM_WAVE - 1), first = window > 0 && pos - window + 1 > 0 ? pos - window + 1 : 0;
  float m = -INFINITY, l = 0.f, acc[2] = {0.f, 0.f};
  for (int j0 = first; j0 <= pos; j0 += BLM_WAVE) {
    const int j = j0 + lane;
    float s = -INFINITY;
    if (j <= pos) {
      const float* k = kcache + (((size_t)pages[j / AF_PAGE] * nkv + kvh) * AF_PAGE + j % AF_PAGE) * hd;
      s = 0.f;
      for (int d = 0; d < hd; ++d) s = fmaf(qrow[d], k[d], s);
      s *= scale;
    }
    const float m_new = fmaxf(m, wave_max(s)), keep = expf(m - m_new), p = j <= pos ? expf(s - m_new) : 0.f;
    l = l * keep + wave_sum(p);
#pragma unroll
    for (int x = 0; x < 2; ++x) acc[x] *= keep;
    for (int y = 0; y < min(BLM_WAVE, pos - j0 + 1); ++y) {
      const float py = __shfl(p, y, BLM_WAVE);
      const float* v = vcache + ((size_t)pages[(j0 + y) / AF_PAGE] * nkv + kvh) * AF_PAGE * hd + (j0 + y) % AF_PAGE;
#pragma unroll
      for (int x = 0; x < 2; ++x)
        if (lane + x * BLM_WAVE < hd) acc[x] = fmaf(py, v[(size_t)(lane + x * BLM_WAVE) * AF_PAGE], acc[x]);
    }
    m = m_new;
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
    if (lane + x * BLM_WAVE < hd) out[lane + x * BLM_WAVE] = acc[x] * (1.0f / l);
}

// The place, from the longest to the shortest, of block `at` of nkv heads' n blocks each; block at + nkv has the next place of its head.  A unit
// starts with the blocks at and at + units, which is units / nkv places further: the second run of that many, whole or not, is turned round, so that the
// longest has the shortest beside it.  What comes later starts as units become free, the longest first.
// (us a layer, every second whole run of 32 turned, which is right for 8 key-value heads alone / this; heads of 64: 2,048 tokens of 16 heads without
// groups 126 / 101, 1,000 of 32 / 32 67.6 / 55.7, of 32 / 4 66 / 54, of 32 / 8 (a second run of 31, which was not turned) 71 / 59.7, 3,000 of 32 / 16
// 402 / 349, of 32 / 8 367 / 350, 2,048 of 32 / 8 186 / 186, of 32 / 4 173 / 174.5; every second run turned: 3,000 of 32 / 8 374, 2,048 of 32 / 4 180.
// Behind another kernel, whose last blocks free the units one by one, 1,000 of 32 / 8 take 56.7 / 55.4.)
__host__ __device__ __forceinline__ int af_place(int at, int n, int nkv, int units) {
  const int place = at / nkv, run = units > nkv ? units / nkv : 1;
  return place >= run && place < 2 * run ? run + min(n, 2 * run) - 1 - place : place;
}

// ---------------------------------------------------------------------------------------------------------------------
// prompts.  A unit is sixteen queries of one head; a block's four wavefronts take neighbouring units of one key-value head
// (the heads of its group at the same queries first), and every page that one of them sees is staged once, through registers
// that hold the next page while this one is worked on.  Rows in shared memory are padded by four floats, so that the sixteen
// rows of a fragment meet every bank.  The longest units start first, those that share a compute unit with them from the shortest up (af_place):
// 32 heads of 64 in 8 groups have 504 blocks for 1,000 tokens, and a unit's two have 17 pages between them, not 2 to 32.
// Measured (us a layer, 32 heads of 64 in 8 groups; before: one wavefront per query and head on the vector units):
// 1,000 tokens 844 -> 96.7; a key-value head's blocks on few dies, no branch for every masked score and every staged piece: 71, and 59.7 in that order (behind the projection 55.4)
// (in the same steps 2,048 tokens 290 -> 186, three sequences of 333 to 1,201 and 24 heads of 128 231 -> 166, 500 tokens 35 -> 28.3, 16 of 300 109 -> 97).
// An exponential by the hardware's power of two and a correction took 4 us less of 1,000 tokens and 20 of 2,048; it was up to 2 ulps off where the
// library's is one, and zero below 2^-126.  Two wavefronts for a unit, one on every other page: 83 -> 90, 500 tokens 35 -> 37.6, but 24 heads of 128
// 121 -> 92.
// ---------------------------------------------------------------------------------------------------------------------
template <int HD, bool FULL>     // HD: the head's lanes rounded up to 32, 64, 96 or 128; FULL: it has all of them
__global__ void __launch_bounds__(AF_WAVES* BLM_WAVE, HD <= 64 ? 3 : 2)
    attn_prefill_f32_kernel(const float* __restrict__ q, int q_row_stride, float* __restrict__ out,
                            const int* __restrict__ positions, const int* __restrict__ cu_seqlens,
                            const int* __restrict__ block_table, int table_width, const float* __restrict__ kcache,
                            const float* __restrict__ vcache, int nh, int nkv, int hd, float scale, int window, int compute_units) {
  constexpr int KP = HD + 4, VP = AF_PAGE + 4, DS = HD / 16, PER = HD * AF_PAGE / 4 / (AF_WAVES * BLM_WAVE);
  __shared__ __attribute__((aligned(16))) float k_page[AF_PAGE * KP];
  __shared__ __attribute__((aligned(16))) float v_page[HD * VP];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / BLM_WAVE), lane = tid & (BLM_WAVE - 1);
  const int c = lane & 15, g = lane >> 4;
  const int seq = blockIdx.z, group = nh / nkv;
  const int row0 = cu_seqlens[seq], n_q = cu_seqlens[seq + 1] - row0;
  const int units = ((n_q + 15) / 16) * group;
  // consecutive blocks go to different dies: a die sees the pages of few key-value heads
  const int at = blockIdx.x + gridDim.x * blockIdx.y, kvh = at % nkv;
  const int unit0 = ((int)gridDim.x - 1 - af_place(at, gridDim.x, nkv, compute_units)) * AF_WAVES;
  if (unit0 >= units) return;
  const int unit = min(unit0 + wave, units - 1);
  const bool active = unit0 + wave < units;
  const int tile = unit / group, head = kvh * group + unit % group;
  const int query = min(tile * 16 + c, n_q - 1), row = row0 + query;
  const int pos = positions[row];
  // pages: of the block (its first unit has the lowest queries), and of this wavefront
  const int block_lo = positions[row0 + unit0 / group * 16], block_hi = positions[row0 + min(min(unit0 + AF_WAVES - 1, units - 1) / group * 16 + 15, n_q - 1)];
  const int wave_lo = positions[row0 + tile * 16], wave_hi = positions[row0 + min(tile * 16 + 15, n_q - 1)];
  const int page_begin = window > 0 && block_lo - window + 1 > 0 ? (block_lo - window + 1) / AF_PAGE : 0;
  const int page_end = block_hi / AF_PAGE + 1;
  const int wave_begin = window > 0 && wave_lo - window + 1 > 0 ? (wave_lo - window + 1) / AF_PAGE : 0, wave_end = wave_hi / AF_PAGE + 1;
  const int* pages = block_table + (size_t)seq * table_width;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

  const float* qrow = q + (size_t)row * q_row_stride + (size_t)head * hd;
  f32x4 qf[DS];
#pragma unroll
  for (int i = 0; i < DS; ++i) qf[i] = i * 16 + g * 4 < hd ? af_load(qrow + i * 16 + g * 4) : zero;
  if (!FULL)     // the lanes that the head does not have count as zeros
    for (int i = tid; i < AF_PAGE * (HD - hd); i += AF_WAVES * BLM_WAVE) k_page[i / (HD - hd) * KP + hd + i % (HD - hd)] = 0.f;

  // a thread's pieces of a page: piece x of the page's hd * 16 pieces of four floats, keys and values alike
  f32x4 ks[PER], vs[PER];
  const int pieces = hd * (AF_PAGE / 4), per_row = hd / 4;
  auto fetch = [&](int page) {
    const size_t base = ((size_t)pages[page] * nkv + kvh) * AF_PAGE * hd;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int x = (FULL ? tid + i * AF_WAVES * BLM_WAVE : min(tid + i * AF_WAVES * BLM_WAVE, pieces - 1)) * 4;
      ks[i] = af_load(kcache + base + x);
      vs[i] = af_load(vcache + base + x);
    }
  };
  auto put = [&](int page) {
    // what lies behind the last key of the block was never written by this sequence: zeros, lest it be no number
    if (page * AF_PAGE + AF_PAGE - 1 > block_hi) {
#pragma unroll
      for (int i = 0; i < PER; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) vs[i][e] = page * AF_PAGE + (tid + i * AF_WAVES * BLM_WAVE) % 16 * 4 + e <= block_hi ? vs[i][e] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int x = tid + i * AF_WAVES * BLM_WAVE;
      if (FULL || x < pieces) {
        const int kr = FULL ? x / (HD / 4) : x / per_row, kx = (x - kr * (FULL ? HD / 4 : per_row)) * 4, vr = x / 16, vx = x % 16 * 4;
        *reinterpret_cast<f32x4*>(&k_page[kr * KP + kx]) = ks[i];
        *reinterpret_cast<f32x4*>(&v_page[vr * VP + vx]) = vs[i];
      }
    }
  };

  float m = -INFINITY, l = 0.f;
  f32x4 o[DS];
#pragma unroll
  for (int d = 0; d < DS; ++d) o[d] = zero;
  fetch(page_begin);
  for (int page = page_begin; page < page_end; ++page) {
    __syncthreads();       // the page before has been read (and, at first, the zeros are written)
    put(page);
    __syncthreads();
    if (page + 1 < page_end) fetch(page + 1);
    if (page < wave_begin || page >= wave_end) continue;
    f32x4 s[4] = {zero, zero, zero, zero};
#pragma unroll
    for (int i = 0; i < DS; ++i) {
      f32x4 kf[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) kf[t] = af_load(&k_page[(t * 16 + c) * KP + i * 16 + g * 4]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < 4; ++t) s[t] = af_mfma(kf[t][e], qf[i][e], s[t]);
    }
    const int key0 = page * AF_PAGE + g * 4;
    const bool whole = page * AF_PAGE + AF_PAGE - 1 <= wave_lo && (window <= 0 || wave_hi - page * AF_PAGE < window);
#pragma unroll
    for (int t = 0; t < 4; ++t) s[t] *= scale;
    if (!whole) {        // a branch for all of them: one for each took as long as the softmax
      const int from = window > 0 ? pos - window : -1;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int key = key0 + t * 16 + v;
          s[t][v] = (key <= pos) & (key > from) ? s[t][v] : -INFINITY;
        }
    }
    const float keep = af_softmax(s, m, l);
#pragma unroll
    for (int d = 0; d < DS; ++d) o[d] *= keep;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      f32x4 vf[DS];
#pragma unroll
      for (int d = 0; d < DS; ++d) vf[d] = af_load(&v_page[(d * 16 + c) * VP + t * 16 + g * 4]);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int d = 0; d < DS; ++d) o[d] = af_mfma(vf[d][e], s[t][e], o[d]);
    }
  }
  if (!active) return;
  const float inv = 1.0f / rows_sum(l);
  bool odd = false;
  float* orow = out + ((size_t)row * nh + head) * hd;
#pragma unroll
  for (int d = 0; d < DS; ++d) {
    o[d] *= inv;
    if (d * 16 + g * 4 < hd) {
#pragma unroll
      for (int v = 0; v < 4; ++v) odd |= !(fabsf(o[d][v]) < INFINITY);
      if (tile * 16 + c < n_q) *reinterpret_cast<f32x4*>(orow + d * 16 + g * 4) = o[d];
    }
  }
  if (__builtin_amdgcn_ballot_w64(odd) == 0) return;
  for (int x = 0; x < min(16, n_q - tile * 16); ++x) {
    const int r = row0 + tile * 16 + x;
    af_plain_query(q + (size_t)r * q_row_stride + (size_t)head * hd, out + ((size_t)r * nh + head) * hd, positions[r], pages, kcache, vcache,
                   nkv, kvh, hd, scale, window);
  }
}

// ---------------------------------------------------------------------------------------------------------------------
// decoding.  A block has one token, one key-value head and up to sixteen heads of its group; its wavefronts take the pages of
// the block's piece of the key range in turn, fragments straight from the pages (a whole page is read by one wavefront only, its
// lines by neighbouring instructions).  The wavefronts' results meet in shared memory; with several pieces per token the blocks
// leave theirs in device-coherent memory, count themselves in, and the last one adds them up (as attn_paged does).
// A page takes a wavefront 128 products, 1.7 us at the matrix cores' rate, behind the fetch of 32 KB; where a last round of whole pages
// would leave half of the wavefronts idle it goes in halves, 32 keys and 128 bytes of each row of values to a wavefront, and where
// three quarters, in quarters: 16 keys, 64 bytes, so that two wavefronts read a line of values each in part.
// Measured (us a layer, 32 heads of 64 in 8 groups, 8 sequences of 400 to 640 keys; before: a wavefront per head, the heads of
// a group each reading the group's keys and values): 43.8 -> 13.3 in three pieces of whole pages; in a graph of its own 11.4, with
// halves 10.5; 8 sequences of 8 pages in four pieces 10.6 -> 9.3 in halves, 8.7 in quarters; 24 heads of 128 15.9 -> 12.4.
// ---------------------------------------------------------------------------------------------------------------------
// FREE: lanes past the head are zeroed behind the loads, which then stand in no branch: behind one the values' loads wait for the keys'.
// Heads of 64 in groups of four, 8 sequences of 1 / 4 / 9 / 18 pages, us, 5.2 / 9.0 / 12.1 / 16.9 without, 4.7 / 8.1 / 11.6 / 16.7 so.  Not
// for heads of up to 48, whose lanes past them are a quarter of the loads and more (16 heads of 48, 40 sequences of 9 / 20 pages 42.1 / 76.6
// without, 44.2 / 80.7 so; of 32, 4 pages 5.9 / 6.0), nor for wide ones, whose values take the keys' registers (128, 9 pages: 17.3 / 20.5).
template <int HD, bool FREE>
__global__ void __launch_bounds__(AF_DECODE_WAVES* BLM_WAVE)
    attn_decode_f32_kernel(const float* __restrict__ q, int q_row_stride, float* __restrict__ out, const int* __restrict__ positions,
                           const int* __restrict__ token_seq, const int* __restrict__ block_table, int table_width,
                           const float* __restrict__ kcache, const float* __restrict__ vcache, int nh, int nkv, int hd, float scale,
                           int window, int n_splits, float* part_o, float* part_ml, int* arrivals) {
  constexpr int DS = HD / 16;
  __shared__ __attribute__((aligned(16))) float all_o[AF_DECODE_WAVES][16][HD + 4];
  __shared__ float all_m[AF_DECODE_WAVES][16], all_l[AF_DECODE_WAVES][16];
  __shared__ int is_last;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / BLM_WAVE), lane = tid & (BLM_WAVE - 1);
  const int c = lane & 15, g = lane >> 4;
  const int token = blockIdx.z, split = blockIdx.x, group = nh / nkv, tiles = (group + 15) / 16;
  const int kvh = blockIdx.y / tiles, head0 = kvh * group + blockIdx.y % tiles * 16, heads = min(16, (kvh + 1) * group - head0);
  const int seq = token_seq[token];
  float* orow = out + ((size_t)token * nh + head0) * hd;
  if (seq < 0) {      // padding: defined output, no cache access
    if (split == 0)
      for (int i = tid; i < heads * hd; i += AF_DECODE_WAVES * BLM_WAVE) orow[i] = 0.f;
    return;
  }
  const int pos = positions[token], first = window > 0 && pos - window + 1 > 0 ? pos - window + 1 : 0;
  const int page_first = first / AF_PAGE, n_pages = pos / AF_PAGE + 1 - page_first;
  const int per_split = (n_pages + n_splits - 1) / n_splits;
  const int page_begin = page_first + split * per_split, page_end = min(page_first + n_pages, page_begin + per_split);
  const int* pages = block_table + (size_t)seq * table_width;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  const float* qrow = q + (size_t)token * q_row_stride + (size_t)(head0 + min(c, heads - 1)) * hd;
  f32x4 qf[DS];
#pragma unroll
  for (int i = 0; i < DS; ++i) qf[i] = FREE ? af_load(qrow + min(i * 16 + g * 4, hd - 4)) : i * 16 + g * 4 < hd ? af_load(qrow + i * 16 + g * 4) : zero;
  if (FREE && hd < HD)
#pragma unroll
    for (int i = 0; i < DS; ++i)
      if (i * 16 + g * 4 >= hd) qf[i] = zero;
  float m = -INFINITY, l = 0.f;
  f32x4 o[DS];
#pragma unroll
  for (int d = 0; d < DS; ++d) o[d] = zero;
  // 16 * TILES keys of a page from tile t0 on
  auto keys = [&](int page, int t0, auto tiles_type) {
    constexpr int TILES = decltype(tiles_type)::value;
    const size_t base = ((size_t)pages[page] * nkv + kvh) * AF_PAGE * hd;
    f32x4 kf[DS][TILES], vf[DS][TILES];
#pragma unroll
    for (int i = 0; i < DS; ++i)
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
        const float* row = kcache + base + (size_t)((t0 + t) * 16 + c) * hd;
        kf[i][t] = FREE ? af_load(row + min(i * 16 + g * 4, hd - 4)) : i * 16 + g * 4 < hd ? af_load(row + i * 16 + g * 4) : zero;
      }
    // wide heads: the values' registers are the keys' once these are multiplied
    if (HD > 64) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; HD <= 64 && d < DS; ++d)
#pragma unroll
      for (int t = 0; t < TILES; ++t) vf[d][t] = af_load(vcache + base + (size_t)min(d * 16 + c, hd - 1) * AF_PAGE + (t0 + t) * 16 + g * 4);
    if (FREE && hd < HD)
#pragma unroll
      for (int i = 0; i < DS; ++i)
#pragma unroll
        for (int t = 0; t < TILES; ++t)
          if (i * 16 + g * 4 >= hd) kf[i][t] = zero;
    f32x4 s[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) s[t] = zero;
#pragma unroll
    for (int i = 0; i < DS; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < TILES; ++t) s[t] = af_mfma(kf[i][t][e], qf[i][e], s[t]);
    if (HD > 64) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < DS; ++d)
#pragma unroll
        for (int t = 0; t < TILES; ++t) vf[d][t] = af_load(vcache + base + (size_t)min(d * 16 + c, hd - 1) * AF_PAGE + (t0 + t) * 16 + g * 4);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int key0 = page * AF_PAGE + t0 * 16 + g * 4;
    bool see[TILES][4];
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        see[t][v] = af_visible(key0 + t * 16 + v, pos, window);
        s[t][v] = see[t][v] ? s[t][v] * scale : -INFINITY;
      }
    const float keep = af_softmax<TILES>(s, m, l);
#pragma unroll
    for (int d = 0; d < DS; ++d) o[d] *= keep;
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int d = 0; d < DS; ++d) o[d] = af_mfma(see[t][e] ? vf[d][t][e] : 0.f, s[t][e], o[d]);   // an unseen value may be anything
  };
  // whole pages, a round of the wavefronts at a time; a last round that would leave half of them idle goes in halves of pages, one
  // that would leave three quarters idle in quarters
  const int left = (page_end - page_begin) % AF_DECODE_WAVES;
  const int whole_end = 2 * left <= AF_DECODE_WAVES ? page_end - max(0, left) : page_end;
  for (int page = page_begin + wave; page < whole_end; page += AF_DECODE_WAVES) keys(page, 0, AfInt<4>{});
  if (4 * left > AF_DECODE_WAVES) {
    const int half = 2 * whole_end + wave;
    if (half < 2 * page_end) keys(half / 2, half % 2 * 2, AfInt<2>{});
  } else {
    const int quarter = 4 * whole_end + wave;
    if (quarter < 4 * page_end) keys(quarter / 4, quarter % 4, AfInt<1>{});
  }
  l = rows_sum(l);
#pragma unroll
  for (int d = 0; d < DS; ++d) *reinterpret_cast<f32x4*>(&all_o[wave][c][d * 16 + g * 4]) = o[d];
  if (g == 0) {
    all_m[wave][c] = m;
    all_l[wave][c] = l;
  }
  __syncthreads();
  const size_t item0 = (size_t)token * nh + head0;
  const auto ex = [](float v) { return expf(v); };
  const auto put = [&](int h, int d, float4 v) {
    float* p = orow + h * hd + d;
    p[0] = v.x;
    p[1] = v.y;
    p[2] = v.z;
    p[3] = v.w;
  };
  ag_block<AF_DECODE_WAVES * BLM_WAVE, AF_DECODE_WAVES>(&all_m[0][0], &all_l[0][0], &all_o[0][0][0], 16 * (HD + 4), HD + 4, heads, hd, ex,
                                                        [&](int h, int d, const AgSum& a) {
    if (n_splits == 1) {
      put(h, d, a.result());
    } else {
      const size_t at = (item0 + h) * n_splits + split;
      ag_leave(a, part_o + at * hd + d, part_ml + at * 2, d == 0);
    }
  });
  if (n_splits == 1) return;
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wavefront's stores have been acknowledged
  __syncthreads();
  if (tid == 0) {
    const int before = __hip_atomic_fetch_add(arrivals + item0, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    is_last = before == n_splits - 1;
    if (is_last) __hip_atomic_store(arrivals + item0, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // zero again for the next launch
  }
  __syncthreads();
  if (!is_last) return;
  ag_merge<AF_DECODE_WAVES * BLM_WAVE>(part_o + item0 * n_splits * hd, part_ml + item0 * n_splits * 2, heads, n_splits, hd, ex,
                                       [&](int h, int d, const AgSum& a) { put(h, d, a.result()); });
}

extern "C" int blm_attn_f32_supported(int hd, int page_size) { return hd >= 4 && hd % 4 == 0 && hd <= 128 && page_size == AF_PAGE ? 1 : 0; }

static int attn_f32_check(const char* name, const void* q, int q_row_stride, const void* k, const void* v, int nh, int nkv, int hd, int table_width, int window) {
  BLM_REQUIRE(nh > 0 && nkv > 0 && nh % nkv == 0 && blm_attn_f32_supported(hd, AF_PAGE), "%s: heads=%d kv_heads=%d head_dim=%d not supported", name, nh, nkv, hd);
  BLM_REQUIRE(q_row_stride >= nh * hd && q_row_stride % 4 == 0 && ((uintptr_t)q % 16) == 0 && ((uintptr_t)k % 16) == 0 && ((uintptr_t)v % 16) == 0,
              "%s: rows and pages must start at multiples of 16 bytes", name);
  BLM_REQUIRE(table_width > 0 && window >= 0, "%s: bad cache geometry", name);
  return 0;
}

extern "C" int blm_attn_prefill_f32_place(int at, int blocks, int nkv, int compute_units) { return af_place(at, blocks, nkv, compute_units); }

extern "C" int blm_attn_prefill_f32(const void* q, int q_row_stride, void* out, const int* positions, const int* cu_seqlens,
                                    const int* block_table, int table_width, const void* kcache, const void* vcache, int n_seqs,
                                    int max_new, int nh, int nkv, int hd, float scale, int window, int compute_units, hipStream_t stream) {
  if (attn_f32_check("attn_prefill_f32", q, q_row_stride, kcache, vcache, nh, nkv, hd, table_width, window)) return 1;
  const long long blocks = ((long long)(max_new + 15) / 16 * (nh / nkv) + AF_WAVES - 1) / AF_WAVES;
  BLM_REQUIRE(n_seqs > 0 && n_seqs <= 65535 && max_new > 0 && nkv <= 65535 && blocks < 2147483647LL && compute_units > 0, "attn_prefill_f32: bad sizes");
  dim3 grid((unsigned)blocks, (unsigned)nkv, (unsigned)n_seqs), block(AF_WAVES * BLM_WAVE);
#define BLM_AFP(HD, FULL)                                                                                                             \
  hipLaunchKernelGGL((attn_prefill_f32_kernel<HD, FULL>), grid, block, 0, stream, (const float*)q, q_row_stride, (float*)out, positions, \
                     cu_seqlens, block_table, table_width, (const float*)kcache, (const float*)vcache, nh, nkv, hd, scale, window, compute_units)
  if (hd == 32) BLM_AFP(32, true);
  else if (hd < 32) BLM_AFP(32, false);
  else if (hd == 64) BLM_AFP(64, true);
  else if (hd < 64) BLM_AFP(64, false);
  else if (hd == 96) BLM_AFP(96, true);
  else if (hd < 96) BLM_AFP(96, false);
  else if (hd == 128) BLM_AFP(128, true);
  else BLM_AFP(128, false);
#undef BLM_AFP
  BLM_LAUNCH_CHECK("attn_prefill_f32");
  return 0;
}

// part_o: T * nh * n_splits * hd floats, part_ml: T * nh * n_splits * 2 floats, arrivals: T * nh ints that are zero before the
// first call (every call leaves them zero again); all three may be null when n_splits is 1.  Calls that share the arrivals
// must not overlap in time.
extern "C" int blm_attn_decode_f32(const void* q, int q_row_stride, void* out, const int* positions, const int* token_seq,
                                   const int* block_table, int table_width, const void* kcache, const void* vcache, int T, int nh,
                                   int nkv, int hd, float scale, int window, int n_splits, float* part_o, float* part_ml,
                                   int* arrivals, hipStream_t stream) {
  if (attn_f32_check("attn_decode_f32", q, q_row_stride, kcache, vcache, nh, nkv, hd, table_width, window)) return 1;
  BLM_REQUIRE(n_splits >= 1 && n_splits <= 65535 && (n_splits == 1 || (part_o && part_ml && arrivals)), "attn_decode_f32: %d splits need their workspace", n_splits);
  const long long y = (long long)nkv * ((nh / nkv + 15) / 16);
  BLM_REQUIRE(((uintptr_t)part_o % 8) == 0 && ((uintptr_t)part_ml % 8) == 0, "attn_decode_f32: the workspace must be 8-byte aligned");
  BLM_REQUIRE(T > 0 && T <= 65535 && y <= 65535, "attn_decode_f32: bad sizes T=%d heads=%d", T, nh);
  dim3 grid((unsigned)n_splits, (unsigned)y, (unsigned)T), block(AF_DECODE_WAVES * BLM_WAVE);
#define BLM_AFD(HD, FREE)                                                                                                 \
  hipLaunchKernelGGL((attn_decode_f32_kernel<HD, FREE>), grid, block, 0, stream, (const float*)q, q_row_stride, (float*)out, positions, \
                     token_seq, block_table, table_width, (const float*)kcache, (const float*)vcache, nh, nkv, hd, scale, window,  \
                     n_splits, part_o, part_ml, arrivals)
  if (hd <= 32) BLM_AFD(32, false);
  else if (hd <= 48) BLM_AFD(64, false);
  else if (hd <= 64) BLM_AFD(64, true);
  else if (hd <= 96) BLM_AFD(96, false);
  else BLM_AFD(128, false);
#undef BLM_AFD
  BLM_LAUNCH_CHECK("attn_decode_f32");
  return 0;
}
