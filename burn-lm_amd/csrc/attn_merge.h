// Partial results of the pieces that a decode step's attention cuts a sequence into: how a block leaves its own, and how the block that
// is the last of a (token, head tile) to arrive adds them up.  Both go past the dies' caches.
//
// A trip through device-coherent memory is 1 to 1.5 us, so what costs here is the trips in a row.  A thread has four dims of a head (two
// loads of 8 bytes), the maximum and the sum of a piece are one load, and it asks for AG_TRIP pieces at once whatever their number (a branch
// among the loads would wait for what came before it).
// (us, heads / groups x size, pieces; a dim per thread, 32 pieces at once / this: 8 sequences of 1,125 keys 32 / 4 x 128, 5 pieces 16.1 / 11.9,
// 16 / 4 x 128 12.9 / 11.2, 4 of 4,096 24 / 8 x 128, 8 pieces 18.8 / 17.4, 1 of 4,096 13.2 / 11.4; float32, where the pieces came one after the
// other, 8 of 520 32 / 8 x 64, 4 pieces 10.9 / 10.3, 1 of 1,100, 9 pieces 10.3 / 8.2.  Both this and a dim per thread in one kernel, and
// trips of 4, 8 and 16 by the number of pieces: up to 0.5 us more, since a kernel of 8 us has its instructions from memory as well.)
#pragma once
#include "common.h"

#define AG_TRIP 16

__device__ __forceinline__ void ag_store2(float* p, float a, float b) {
  const unsigned long long v = (unsigned long long)__float_as_uint(a) | (unsigned long long)__float_as_uint(b) << 32;
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 ag_load2(const float* p) {
  const unsigned long long v = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return make_float2(__uint_as_float((uint32_t)v), __uint_as_float((uint32_t)(v >> 32)));
}

// four dims of an output: the maximum of the scores so far, the sum of the weights, the weighted sums
struct AgSum {
  float m, l;
  float4 o;
  __device__ __forceinline__ float4 result() const { return make_float4(o.x / l, o.y / l, o.z / l, o.w / l); }
};
// a += what has its maximum, no larger than a's, at m
template <class Exp>
__device__ __forceinline__ void ag_add(AgSum& a, float m, float l, float4 o, Exp ex) {
  const float f = m == a.m ? 1.f : ex(m - a.m);
  a.l += l * f;
  a.o.x += o.x * f;
  a.o.y += o.y * f;
  a.o.z += o.z * f;
  a.o.w += o.w * f;
}

// The wavefronts' results of a block, in shared memory (m, l [WAVES][16]; head h's dims of wavefront w, 16-byte aligned, at o + w * o_wave + h *
// o_head), added up: done(head, dim, sum).  ex: the exponential in the scores' base.
template <int THREADS, int WAVES, class Exp, class Done>
__device__ __forceinline__ void ag_block(const float* m, const float* l, const float* o, int o_wave, int o_head, int heads, int hd, Exp ex, Done done) {
  for (int at = threadIdx.x; at < heads * (hd / 4); at += THREADS) {
    const int h = at / (hd / 4), d = (at - h * (hd / 4)) * 4;
    AgSum a{m[h], 0.f, make_float4(0.f, 0.f, 0.f, 0.f)};
#pragma unroll
    for (int w = 1; w < WAVES; ++w) a.m = fmaxf(a.m, m[w * 16 + h]);
#pragma unroll
    for (int w = 0; w < WAVES; ++w) ag_add(a, m[w * 16 + h], l[w * 16 + h], *reinterpret_cast<const float4*>(o + w * o_wave + h * o_head + d), ex);
    done(h, d, a);
  }
}

// The partial result of a piece: o [hd], of which these are four, and ml [2], both 8-byte aligned.
__device__ __forceinline__ void ag_leave(const AgSum& a, float* o, float* ml, bool first) {
  ag_store2(o, a.o.x, a.o.y);
  ag_store2(o + 2, a.o.z, a.o.w);
  if (first) ag_store2(ml, a.m, a.l);
}

// part_o [heads, n_pieces, hd], part_ml [heads, n_pieces, 2] of the block's heads: done(head, dim, sum).
template <int THREADS, class Exp, class Done>
__device__ __forceinline__ void ag_merge(const float* part_o, const float* part_ml, int heads, int n_pieces, int hd, Exp ex, Done done) {
  for (int at = threadIdx.x; at < heads * (hd / 4); at += THREADS) {
    const int head = at / (hd / 4), d = (at - head * (hd / 4)) * 4;
    const float* o = part_o + (size_t)head * n_pieces * hd + d;
    const float* ml = part_ml + (size_t)head * n_pieces * 2;
    AgSum a{-INFINITY, 0.f, make_float4(0.f, 0.f, 0.f, 0.f)};
    for (int first = 0; first < n_pieces; first += AG_TRIP) {
      float2 s[AG_TRIP], lo[AG_TRIP], hi[AG_TRIP];
#pragma unroll
      for (int i = 0; i < AG_TRIP; ++i) {      // (those behind the last are the last again and add nothing)
        const int p = min(first + i, n_pieces - 1);
        s[i] = ag_load2(ml + (size_t)p * 2);
        lo[i] = ag_load2(o + (size_t)p * hd);
        hi[i] = ag_load2(o + (size_t)p * hd + 2);
      }
      float top = a.m;
#pragma unroll
      for (int i = 0; i < AG_TRIP; ++i) top = fmaxf(top, s[i].x);
      const float keep = a.m == top ? 1.f : ex(a.m - top);
      a = AgSum{top, a.l * keep, make_float4(a.o.x * keep, a.o.y * keep, a.o.z * keep, a.o.w * keep)};
#pragma unroll
      for (int i = 0; i < AG_TRIP; ++i)
        if (first + i < n_pieces) ag_add(a, s[i].x, s[i].y, make_float4(lo[i].x, lo[i].y, hi[i].x, hi[i].y), ex);
    }
    done(head, d, a);
  }
}
