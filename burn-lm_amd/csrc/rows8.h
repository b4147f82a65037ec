// Eight bfloat16 of a row at a time (16-byte accesses), and values turned into pages: what the kernels between a prompt's projections
// and its attention share.
#pragma once
#include "common.h"

__device__ __forceinline__ void r8_unpack(uint4 r, float (&v)[8]) {
  const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __uint_as_float(w[i] << 16);
    v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}
__device__ __forceinline__ void r8_load(const bf16* p, float (&v)[8]) { r8_unpack(*reinterpret_cast<const uint4*>(p), v); }
__device__ __forceinline__ void r8_load(const float* p, float (&v)[8]) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ uint4 r8_pack(const float (&v)[8]) {
  return make_uint4(f32x2_to_bf16x2_bits(v[0], v[1]), f32x2_to_bf16x2_bits(v[2], v[3]), f32x2_to_bf16x2_bits(v[4], v[5]),
                    f32x2_to_bf16x2_bits(v[6], v[7]));
}
__device__ __forceinline__ void r8_store(bf16* p, const float (&v)[8]) { *reinterpret_cast<uint4*>(p) = r8_pack(v); }
__device__ __forceinline__ void r8_store(float* p, const float (&v)[8]) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}

// sum over aligned groups of 1, 2, 4 .. 64 lanes; all lanes of the wavefront active
__device__ __forceinline__ float r8_group_sum(float v, int lanes) {
  if (lanes >= 2) v += blm_dpp<BLM_DPP_XOR1>(v);
  if (lanes >= 4) v += blm_dpp<BLM_DPP_XOR2>(v);
  if (lanes >= 8) v += blm_dpp<BLM_DPP_HALF_MIRROR>(v);
  if (lanes >= 16) v += blm_dpp<BLM_DPP_MIRROR>(v);
  float a, b;
  if (lanes >= 32) { blm_swap16(v, a, b); v = a + b; }
  if (lanes >= 64) { blm_swap32(v, a, b); v = a + b; }
  return v;
}

// lane pairs (cos, sin) of four neighbouring pairs
__device__ __forceinline__ void r8_angles(const float* cs, float (&c)[4], float (&s)[4]) {
  float v[8];
  r8_load(cs, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) c[i] = v[2 * i], s[i] = v[2 * i + 1];
}

// R8_TOKENS tokens' values of one head, `n` lanes from column `col` of the rows on (plus bias), into the transposed pages
// [page][heads][n][page_size]: through shared memory, so that a wavefront's store is a run of neighbouring tokens.  (Token by token
// every store is two bytes of another line, and neighbouring tokens' blocks on other dies write the same lines.)
// r8_turn_rows: lanes [from, to) of the n, which lie at vt[token][lane - from].
#define R8_TOKENS 32
#define R8_VALUE_LDS(n) ((size_t)R8_TOKENS * ((n) + 2) * sizeof(bf16))
__device__ __forceinline__ void r8_turn_rows(const bf16* vt, int stride, int from, int to, int n, int t0, int T, const int* positions, const int* token_seq,
                                             const int* block_table, int table_width, int page_size, bf16* pages, int heads, int head) {
  const int j = threadIdx.x % R8_TOKENS, step = blockDim.x / R8_TOKENS;
  if (t0 + j >= T) return;
  const int seq = token_seq[t0 + j];
  if (seq < 0) return;
  const int pos = positions[t0 + j], page = block_table[(size_t)seq * table_width + pos / page_size];
  if (page < 0) return;
  bf16* dst = pages + ((size_t)page * heads + head) * n * page_size + pos % page_size;
  for (int d = from + threadIdx.x / R8_TOKENS; d < to; d += step) dst[(size_t)d * page_size] = vt[j * stride + d - from];
}
__device__ __forceinline__ void r8_values(const bf16* rows, int ld, int col, const float* bias, int n, int t0, int T, const int* positions,
                                          const int* token_seq, const int* block_table, int table_width, int page_size, bf16* pages,
                                          int heads, int head, bf16* vt) {
  const int stride = n + 2, units = n / 8;
  for (int e = threadIdx.x; e < R8_TOKENS * units; e += blockDim.x) {
    const int j = e / units, d = (e - j * units) * 8;
    if (t0 + j < T) {
      uint4 raw = *reinterpret_cast<const uint4*>(rows + (size_t)(t0 + j) * ld + col + d);
      if (bias) {
        float v[8], b[8];
        r8_unpack(raw, v);
        r8_load(bias + col + d, b);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] += b[i];
        raw = r8_pack(v);
      }
      uint32_t* to = reinterpret_cast<uint32_t*>(vt + j * stride + d);
      to[0] = raw.x; to[1] = raw.y; to[2] = raw.z; to[3] = raw.w;
    }
  }
  __syncthreads();
  r8_turn_rows(vt, stride, 0, n, n, t0, T, positions, token_seq, block_table, table_width, page_size, pages, heads, head);
}
