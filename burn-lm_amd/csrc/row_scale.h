// Rows that come unscaled: x = (h + delta) * gamma, with the sums of squares of h + delta beside them, one partial sum for every few
// columns (gemv_join.hip).  A product of such rows is the product of the normed ones once its row is multiplied by
// 1 / sqrt(mean of squares + eps), which its last step does on the float sums.
#pragma once
#include "common.h"

struct RowScale {
  const float* sums;   // [M, n], 16-byte aligned
  int n;               // a multiple of 4, at most RS_SUMS
  float inv_width, eps;
};
// (A kernel takes sums and, in its shape's bits from RS_SHIFT on, n among the first of its arguments, which come in registers: the sums
// are what it asks for first.)
#define RS_SHIFT 8
#define RS_SUMS 256    // what a wavefront reads at once
#define RS_ROWS 8      // most rows
#define RS_SLOTS 8     // and most that a wavefront takes on (blocks of one wavefront)

static inline bool row_scale_fits(int M, const float* sums, int n) {
  return M >= 1 && M <= RS_ROWS && sums != nullptr && ((uintptr_t)sums % 16) == 0 && n >= 4 && n <= RS_SUMS && n % 4 == 0;
}

// A wavefront has every n_waves-th row.  The sums are asked for ahead of everything and added up while the weights come.  SLOTS: rows
// of a wavefront.
template <int SLOTS>
struct RowScaleLoad {
  float4 v[SLOTS];
  __device__ __forceinline__ void ask(const float* sums, int n, int M, int wave, int n_waves, int lane) {
    const float* p = sums + min(lane * 4, n - 4);
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) v[i] = *reinterpret_cast<const float4*>(p + min(wave + i * n_waves, M - 1) * n);
  }
  // inv [M]: the rows' factors; the caller's next barrier makes them visible
  __device__ __forceinline__ void finish(int n, float inv_width, float eps, int M, int wave, int n_waves, int lane, float* inv) {
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      const float s = wave_sum(lane * 4 < n ? (v[i].x + v[i].y) + (v[i].z + v[i].w) : 0.f);
      const int row = wave + i * n_waves;
      if (lane == 0 && row < M) inv[row] = 1.0f / sqrtf(s * inv_width + eps);
    }
  }
};
