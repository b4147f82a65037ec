// Mixture of experts over many rows, every token by its own experts only (bfloat16): the stacked product computes all E experts
// for every token, E / top times what is needed.
//   moe_lists  : for every expert the tokens that chose it, in order, and the place of each among its token's choices
//   moe_gemm 0 : gate and up of an expert's tokens, gathered; silu(gate) * up * weight as bfloat16 rows, expert by expert
//   moe_gemm 1 : the down projection of these rows into float32 planes, one for each place: [top][T][D], which the reader of the
//                feed-forward's result adds up (a token's places that are not taken are zeroed by moe_lists)
// Many rows run on the 256x256 tiles of gemm_duo.h (moe_duo_kernel), few rows and other widths on 256 x 128 tiles (moe_gemm_kernel;
// the rule stands at the launch).  What bounds them: with 512 rows an expert, more or less, the last tile of an expert is a half that is
// nearly empty, and 128 whole tiles and 36 halves are one round on 256 units; the down projection writes 67 MB of planes.
// The 256 x 128 tiles by eight wavefronts share the compute unit's LDS between the direct loads (48 KB a stage), the wavefronts' reads
// (128 KB) and 1,024 cycles of matrix instructions; a stage takes 0.75 us, and the last round of blocks is a quarter of the time.
// Measured within a whole prompt, under the profiler (us, 2,048 tokens, 16 experts of 512 at width 2048, 4 chosen; the stacked products
// and the gating pass / 256 x 128 / 256 x 256): gate/up with gating 122 / 66 / 53, down 77 / 46.5 / 38.2; lists 6.2.
// Tried for 256 x 128: 128 x 128 tiles, two blocks a unit (stages of 32: 70 and 43), the compiler's own order of reads, loads and
// products (72 and 44), four wavefronts of 128 x 64 (83 and 54).
#include "gemm_duo.h"

typedef __attribute__((ext_vector_type(8))) __bf16 mg_bf16x8;
typedef __attribute__((ext_vector_type(16))) float mg_f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int mg_u32x4;
#define MG_BM 256
#define MG_BN 128
#define MG_BK 64
#define MG_WAVES 8
#define MG_MAX_EXPERTS 256

// The same in both tiles, whose products are the same bits: a token's result does not depend on how many there are.  With expf and a
// division: exp2 of x * -log2(e) in float32 is a dozen ulps off at |x| = 16, and of gates from -64
// to -16 one in 10,000 then rounds to another bfloat16.
__device__ __forceinline__ float mg_gated(float g, float up, float weight) { return g / (1.0f + expf(-g)) * up * weight; }

// weights [T][ld]: an expert's weight for a token, zero where it is not chosen.  lists [E][T]: plane rows place * T + token of
// the tokens that chose expert e, with the weight's bits beside them (one trip to memory at the start of a tile); counts [E].  Blocks
// behind the first E zero the plane rows of places that no expert takes.
// N: a table [V][top] of the token ids, top up to N = 4 or 8, names a token's experts instead, each with the weight 1 / top (an id outside it
// chooses none; the id is (*source)[source_rows[t]] where that row number is there and not negative, else ids[t]): a kernel less than with
// the weights made first (N = 0).  What bounds it are trips to memory in a row, so the tokens of four rounds of threads are asked for at once
// (2,048 tokens, 16 experts, 4 of them a token, under the profiler: weights and lists 5.1 + 6.3 us, a round after the other 13.3, so 10.9
// and a launch less), and with many tokens the comparing of a row's entries.  A call with products of width 64, in a graph, us, weights / table: 16 experts,
// 4 a token, 512 / 2,048 / 8,192 tokens 31.4 / 28.1, 36.2 / 32.0, 52.4 / 44.6; 64 experts, 8 a token, 35.8 / 30.0, 46.9 / 36.6, 111.5 / 77.4;
// 16 experts, 8 a token, 8,192 and 16,384 tokens 76.2 / 76.8 and 124.2 / 127.5.  Longer rows, which every expert would read and compare for
// every token, are made weights first (64 experts, 16 a token, 2,048 tokens 50.6 / 115; 128 experts, 64 a token 150 / 1,830).
struct MgTable {
  const int *table, *ids, *source_rows;
  const int* const* source;
  int V;
};
__device__ __forceinline__ const int* mg_table_row(const MgTable& by, int t, int top) {      // null: no expert
  const int r = by.source_rows ? by.source_rows[t] : -1;
  const int id = r >= 0 ? (*by.source)[r] : by.ids[t];
  return (unsigned)id < (unsigned)by.V ? by.table + (size_t)id * top : nullptr;
}
#define MG_AHEAD 4
#define MG_ENTRIES 8      // most of a row: they are held in registers
// the entries of a row, in one or two loads where they allow (places past the row's end repeat its last)
template <int N>
__device__ __forceinline__ void mg_entries(const int* row, int top, bool fours, int (&v)[N]) {
  if (fours) {
#pragma unroll
    for (int k = 0; k < N; k += 4) {
      const int4 a = *reinterpret_cast<const int4*>(row + (k < top ? k : 0));
      v[k] = a.x; v[k + 1] = a.y; v[k + 2] = a.z; v[k + 3] = a.w;
    }
  } else {
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = row[min(k, top - 1)];
  }
}
// whether a row of `top` entries names expert e, and how many experts in front of it (an entry that repeats counts once)
template <int N>
__device__ __forceinline__ bool mg_named(const int (&v)[N], int top, int e, int& place) {
  bool in = false;
  place = 0;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    bool first = k < top;
#pragma unroll
    for (int j = 0; j < k; ++j) first &= v[j] != v[k];
    in |= first && v[k] == e;
    place += first && (unsigned)v[k] < (unsigned)e;
  }
  return in;
}
template <int N>
__global__ void __launch_bounds__(1024)
    moe_lists_kernel(const float* __restrict__ weights, int ld, MgTable by, int T, int E, int top, int2* __restrict__ lists, int* __restrict__ counts,
                     float* __restrict__ planes, int D) {
  __shared__ int wave_sum[16];
  __shared__ int taken[64];
  __shared__ unsigned long long short_of;      // of 64 tokens those with fewer experts than places
  const int tid = threadIdx.x, wave = tid / BLM_WAVE, lane = tid & (BLM_WAVE - 1);
  constexpr bool TABLE = N > 0;
  constexpr int HELD = TABLE ? N : 1;
  const bool fours = top % 4 == 0 && ((uintptr_t)by.table & 15) == 0;
  if ((int)blockIdx.x >= E) {
    const int t0 = ((int)blockIdx.x - E) * 64;
    if (tid < 64) {
      int n = top;
      if constexpr (TABLE) {
        if (t0 + tid < T) {
          const int* row = mg_table_row(by, t0 + tid, top);
          int entries[HELD];
          mg_entries<HELD>(row != nullptr ? row : by.table, top, fours, entries);
          mg_named<HELD>(entries, row != nullptr ? top : 0, E, n);
        }
      } else if (t0 + tid < T) {
        n = 0;
        for (int e = 0; e < E; ++e) n += weights[(size_t)(t0 + tid) * ld + e] != 0.f;
      }
      taken[tid] = n;
      const unsigned long long few = __builtin_amdgcn_ballot_w64(n < top);
      if (tid == 0) short_of = few;
    }
    __syncthreads();
    for (unsigned long long few = short_of; few != 0; few &= few - 1) {
      const int i = __builtin_ctzll(few);
      for (int p = taken[i]; p < top; ++p)
        for (int d = tid; d < D; d += 1024) planes[((size_t)p * T + t0 + i) * D + d] = 0.f;
    }
    return;
  }
  const int e = blockIdx.x;
  int base = 0;
  const int* rows[MG_AHEAD];
  int entries[MG_AHEAD][HELD];
  for (int t0 = 0, ahead = 0; t0 < T; t0 += 1024, ++ahead) {
    const int t = t0 + tid;
    bool in = false;
    int place = 0;
    float weight = 1.0f / (float)top;
    if constexpr (TABLE) {
      if (ahead % MG_AHEAD == 0) {
#pragma unroll
        for (int i = 0; i < MG_AHEAD; ++i) rows[i] = mg_table_row(by, min(t + i * 1024, T - 1), top);
#pragma unroll
        for (int i = 0; i < MG_AHEAD; ++i) mg_entries<HELD>(rows[i] != nullptr ? rows[i] : by.table, top, fours, entries[i]);
      }
      in = mg_named<HELD>(entries[0], rows[0] != nullptr && t < T ? top : 0, e, place);
#pragma unroll
      for (int i = 0; i + 1 < MG_AHEAD; ++i) {
        rows[i] = rows[i + 1];
#pragma unroll
        for (int k = 0; k < HELD; ++k) entries[i][k] = entries[i + 1][k];
      }
    } else {
      const float* row = weights + (size_t)t * ld;
      in = t < T && row[e] != 0.f;
      if (in) {
        weight = row[e];
        for (int x = 0; x < e; ++x) place += row[x] != 0.f;
      }
    }
    in = in && place < top;                 // (weights that are no numbers may be more than top)
    const unsigned long long votes = __builtin_amdgcn_ballot_w64(in);
    if (lane == 0) wave_sum[wave] = __popcll(votes);
    __syncthreads();
    int at = base, all = 0;
    for (int w = 0; w < 16; ++w) {
      if (w < wave) at += wave_sum[w];
      all += wave_sum[w];
    }
    at += __popcll(votes & ((1ull << lane) - 1));
    if (in) lists[(size_t)e * T + at] = make_int2(place * T + t, __float_as_int(weight));
    base += all;
    __syncthreads();
  }
  if (tid == 0) counts[e] = base;
}

// A block has 256 of an expert's rows and 128 columns (MODE 0: 64 gates and their 64 ups); eight wavefronts of 64 x 64, stages
// of 64 along K in three buffers, by direct loads, 16-byte pieces permuted as in gemm_mfma.  Row tiles are counted through the
// experts; which expert and rows a block has it finds from the counts (at most 256 experts: a thread each; read one by one they
// held every block up for ten microseconds and more).  A die (blockIdx % 8) has a stretch of the tiles: neighbouring blocks
// share their rows, the next ones their expert's weights.
template <int MODE>
__global__ void __launch_bounds__(64 * MG_WAVES, 2)
    moe_gemm_kernel(const bf16* __restrict__ A, int lda, const bf16* __restrict__ W, int ldw, const int2* __restrict__ lists, const int* __restrict__ counts, bf16* __restrict__ act, float* __restrict__ planes,
                    int T, int E, int N, int K, int inner, int n_tiles) {
  constexpr int STAGE = (MG_BM + MG_BN) * MG_BK, LOADS = (MG_BM + MG_BN) / 8 / MG_WAVES;
  __shared__ __attribute__((aligned(1024))) bf16 lds[3 * STAGE];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / BLM_WAVE), lane = tid & (BLM_WAVE - 1);
  // a thread for each expert: its tiles and rows, and by a scan those of the experts before it
  __shared__ int sums[2 * MG_WAVES], found[4];
  const int mine = tid < E ? counts[tid] : 0, my_tiles = (mine + MG_BM - 1) / MG_BM;
  int tiles = my_tiles, first = mine;
#pragma unroll
  for (int d = 1; d < BLM_WAVE; d *= 2) {
    const int t = __shfl_up(tiles, d), r = __shfl_up(first, d);
    if (lane >= d) tiles += t, first += r;
  }
  if (lane == BLM_WAVE - 1) sums[wave] = tiles, sums[MG_WAVES + wave] = first;
  __syncthreads();
  int total = 0;
  for (int w = 0; w < MG_WAVES; ++w) {
    if (w < wave) tiles += sums[w], first += sums[MG_WAVES + w];
    total += sums[w];
  }
  const int share = (total * n_tiles + 7) / 8, id = ((int)blockIdx.x & 7) * share + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= share || id >= total * n_tiles) return;
  const int nt = id % n_tiles;
  int tile = id / n_tiles;
  if (tile >= tiles - my_tiles && tile < tiles) found[0] = tid, found[1] = tile - (tiles - my_tiles), found[2] = first - mine, found[3] = mine;
  __syncthreads();
  const int e = __builtin_amdgcn_readfirstlane(found[0]), count = __builtin_amdgcn_readfirstlane(found[3]);
  tile = __builtin_amdgcn_readfirstlane(found[1]);
  first = __builtin_amdgcn_readfirstlane(found[2]);
  const int m0 = tile * MG_BM, rows = min(MG_BM, count - m0);
  const int n0 = nt * (MODE == 0 ? MG_BN / 2 : MG_BN);
  // the tile's rows and their weights (asked for one by one at the end they would cost more than the products)
  __shared__ int list[MG_BM];
  __shared__ float row_weight[MG_BM];
  if (tid < rows) {
    const int2 to = lists[(size_t)e * T + m0 + tid];
    list[tid] = to.x;
    row_weight[tid] = __int_as_float(to.y);
  }
  __syncthreads();

  uint32_t offset[LOADS];
  const char* base[LOADS];                  // the same for a wavefront's lanes (in scalar registers): the eight rows of a load share it
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r0 = (i * MG_WAVES + wave) * 8, r = r0 + lane / 8, piece = (lane & 7) ^ ((r >> 1) & 7);
    if (r0 < MG_BM) {
      const int m = min(r, rows - 1);       // rows past the end are the last one again; nothing stores them
      base[i] = reinterpret_cast<const char*>(MODE == 0 ? A : A + (size_t)(first + m0) * lda);
      offset[i] = (uint32_t)(MODE == 0 ? list[m] % T : m) * (uint32_t)lda * 2u + piece * 16u;
    } else if (MODE == 0) {                 // per 64 columns of the tile 32 gate rows and their 32 up rows
      const int c = r - MG_BM, n = min(n0 + c / 64 * 32 + c % 32, N - 1);
      base[i] = reinterpret_cast<const char*>(W + (size_t)e * N * ldw + (size_t)((r0 - MG_BM) % 64 / 32) * inner * ldw);
      offset[i] = (uint32_t)n * (uint32_t)ldw * 2u + piece * 16u;
    } else {
      base[i] = reinterpret_cast<const char*>(W + (size_t)e * K);
      offset[i] = (uint32_t)min(n0 + r - MG_BM, N - 1) * (uint32_t)ldw * 2u + piece * 16u;
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(blm_lds_ptr)lds;
  auto fetch = [&](int k0, int buf, int i) {
    blm_dma16_to(base[i] + (size_t)k0 * 2, offset[i], lds0 + (uint32_t)(buf * STAGE * 2 + (i * MG_WAVES + wave) * 1024));
  };
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64, c = lane & 31, hb = lane >> 5, twist = (c >> 1) & 7;
  mg_f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  const int stages = K / MG_BK;
  struct Pieces {
    mg_u32x4 a[2][2], w[2][2];
  } left, right;                              // of a stage's first and second 32
  auto read = [&](int buf, int half, Pieces& f, int x, int i, bool of_w) {
    const bf16* at = lds + buf * STAGE + ((of_w ? MG_BM + wn : wm) + i * 32 + c) * MG_BK + ((4 * half + 2 * x + hb) ^ twist) * 8;
    (of_w ? f.w : f.a)[x][i] = *reinterpret_cast<const mg_u32x4*>(at);
  };
  auto multiply = [&](const Pieces& f, int x, int i, int j) {
    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mg_bf16x8, f.a[x][i]), __builtin_bit_cast(mg_bf16x8, f.w[x][j]), acc[i][j], 0, 0, 0);
  };
  // Half a stage: its eight products; in between the next half's eight pieces from the shared memory and half the loads of
  // another stage.
  auto work = [&](const Pieces& now, Pieces& next, int next_buf, int next_half, bool loads, int k0, int to, int first_load, bool live) {
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      if (g < 4) {
        if (live) read(next_buf, next_half, next, g >> 1, g & 1, false);
        if (live) read(next_buf, next_half, next, g >> 1, g & 1, true);
      } else if (loads && g - 4 < LOADS / 2) {
        fetch(k0, to, first_load + g - 4);
      }
      if (live) multiply(now, g >> 2, (g >> 1) & 1, g & 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr int HALF = LOADS / 2;
#pragma unroll
  for (int s = 0; s < 3; ++s)
    if (s < stages)
#pragma unroll
      for (int i = 0; i < (s == 2 ? HALF : LOADS); ++i) fetch(s * MG_BK, s, i);
  if (stages >= 3)
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(LOADS + HALF) : "memory");
  else
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  // A stage's buffer is free once all have its second half in registers (the wait and barrier in the middle): the first loads
  // of the stage three behind it go out in the second half, the others in the next stage's first.  The order is held fast:
  // left to itself the compiler reads first and multiplies then, and issues a stage's loads at a stretch, and the matrix cores
  // idle meanwhile.
  // Wavefronts whose rows are all behind the end only load: a part of a tile leaves the others the LDS (us, 512 tokens of the
  // case above: 30.0 -> 26.9 and 17.0 -> 15.7; 1,000 tokens by 8 of 128 experts of 128 at width 1024: 23.0 -> 19.4 and 34.8 ->
  // 32.7).  Putting the full tiles in front of the parts was slower: an expert's weights are then read twice.
  auto run = [&](auto live_type) {
    constexpr bool live = decltype(live_type)::value;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (live) read(0, 0, left, x, i, false);
        if (live) read(0, 0, left, x, i, true);
      }
    int s = 0, buf = 0, last = 2;               // buffers of stage s and of stage s + 2
    for (; s + 3 < stages; ++s) {
      work(left, right, buf, 1, true, (s + 2) * MG_BK, last, HALF, live);
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LOADS) : "memory");
      last = buf;
      buf = buf == 2 ? 0 : buf + 1;
      work(right, left, buf, 0, true, (s + 3) * MG_BK, last, 0, live);
    }
    if (stages >= 3)
#pragma unroll
      for (int i = HALF; i < LOADS; ++i) fetch((stages - 1) * MG_BK, last, i);
    for (; s < stages; ++s) {
      work(left, right, buf, 1, false, 0, 0, 0, live);
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      buf = buf == 2 ? 0 : buf + 1;
      work(right, left, buf, 0, false, 0, 0, 0, live);      // (behind the last stage: an older one's pieces, not used)
    }
  };
  if (wm < rows)
    run(std::integral_constant<bool, true>{});
  else
    run(std::integral_constant<bool, false>{});
  // acc[i][j][v]: row wm + 32 i + 8 (v / 4) + 4 hb + v % 4, column wn + 32 j + c
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int m = wm + i * 32 + 8 * (v >> 2) + 4 * hb + (v & 3);
      if (MODE == 0) {
        const int n = n0 + wn / 2 + c;
        const float y = mg_gated(acc[i][0][v], acc[i][1][v], row_weight[m]);
        if (m < rows && n < N) act[(size_t)(first + m0 + m) * N + n] = from_float<bf16>(y);
      } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int n = n0 + wn + j * 32 + c;
          if (m < rows && n < N) planes[(size_t)list[m] * N + n] = acc[i][j][v];
        }
      }
    }
}

// The same products in the tiles of gemm_duo.h, 256 rows and 256 columns (MODE 0: 128 gates and their ups).  An expert's rows are
// whole tiles and, where at most 128 are left, a half; or halves all of them, or five eighths, where those come in less time on the `units`.
template <int MODE>
struct MgTile {
  const char *a, *b;
  const int* list;                            // MODE 0: the tokens of the tile's rows
  int rows, n0, N, lda, ldw;
  uint32_t up;
  __device__ __forceinline__ uint32_t row(int m) const {
    m = min(m, rows - 1);
    return (uint32_t)(MODE == 0 ? list[m] : m) * (uint32_t)lda * 2u;
  }
  __device__ __forceinline__ uint32_t column(int r, int h) const {
    const int n = min(n0 + (MODE == 0 ? r : r / 32 * 64 + h * 32 + r % 32), N - 1);
    return (uint32_t)n * (uint32_t)ldw * 2u + (MODE == 0 && h ? up : 0u);
  }
};

template <int MODE, int TILES>
__device__ __forceinline__ void mg_store(const gd_f32x4 (&acc)[TILES][4], bf16* act, float* planes, const int* list, const float* row_weight,
                                         int m0, int rows, int n0, int N, int lane) {
  const int l16 = lane & 15, quad = lane >> 4;
#pragma unroll
  for (int i = 0; i < TILES; ++i) {
    const int m = m0 + i * 16 + l16;
    if (MODE == 0) {
      float v[2][4];
      const float w = row_weight[m];
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[x][e] = mg_gated(acc[i][x][e], acc[i][2 + x][e], w);
      const uint4 eight = gd_eight(v);
      const int n = n0 + (quad & 1) * 16 + (quad >> 1) * 8;
      if (m < rows && n < N) *reinterpret_cast<uint4*>(act + (size_t)m * N + n) = eight;
    } else {
      const int to = list[m];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + j * 16 + quad * 4;
        if (m < rows && n < N) *reinterpret_cast<float4*>(planes + (size_t)to * N + n) = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
      }
    }
  }
}

template <int MODE>
__global__ void __launch_bounds__(512, 2)
    moe_duo_kernel(const bf16* __restrict__ A, int lda, const bf16* __restrict__ W, int ldw, const int2* __restrict__ lists, const int* __restrict__ counts, bf16* __restrict__ act, float* __restrict__ planes,
                   int T, int E, int N, int K, int inner, int n_tiles, int units) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[3 * GdPart<5>::STAGE];
  __shared__ int list[GD_TILE];
  __shared__ float row_weight[GD_TILE];
  __shared__ int sums[5][8], found[4];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / BLM_WAVE), lane = tid & (BLM_WAVE - 1);
  // a thread for each expert: its whole tiles, its half behind them, its halves or five eighths if it has nothing else, its rows; and by
  // a scan those of the experts before it
  const int mine = tid < E ? counts[tid] : 0, over = mine % GD_TILE;
  const int own[5] = {mine / GD_TILE + (over > GD_TILE / 2), over > 0 && over <= GD_TILE / 2, (mine + GD_TILE / 2 - 1) / (GD_TILE / 2),
                      (mine + GdPart<5>::ROWS - 1) / GdPart<5>::ROWS, mine};
  int upto[5], all[5];
#pragma unroll
  for (int x = 0; x < 5; ++x) upto[x] = own[x];
#pragma unroll
  for (int d = 1; d < BLM_WAVE; d *= 2) {
    int before[5];
#pragma unroll
    for (int x = 0; x < 5; ++x) before[x] = __shfl_up(upto[x], d);
#pragma unroll
    for (int x = 0; x < 5; ++x) upto[x] += lane >= d ? before[x] : 0;
  }
  if (lane == BLM_WAVE - 1)
#pragma unroll
    for (int x = 0; x < 5; ++x) sums[x][wave] = upto[x];
  __syncthreads();
#pragma unroll
  for (int x = 0; x < 5; ++x) {
    all[x] = 0;
    for (int w = 0; w < 8; ++w) {
      if (w < wave) upto[x] += sums[x][w];
      all[x] += sums[x][w];
    }
  }
  // rounds in hundredths of a whole tile's time, a half 57 of them, five eighths GD_FIVE_PERCENT (see gemm_duo.hip)
  const int wholes = all[0] * n_tiles, rest = wholes % units, beside = rest ? units - rest : 0;
  const int mixed = wholes / units * 100 + (rest ? 100 : 0) + (max(0, all[1] * n_tiles - beside) + units - 1) / units * 57;
  const int halves = (all[2] * n_tiles + units - 1) / units * 57, fives = (all[3] * n_tiles + units - 1) / units * GD_FIVE_PERCENT;
  // the parts behind the whole tiles: 1: an expert's last rows; 2, 3: all of them, in halves or five eighths
  // (five eighths from K = 1,024 on: what a block does besides its products is the same for a larger and a smaller one, and at K = 512 three
  // rounds' worth of it cost more than the products saved: 2,048 tokens, 16 experts, down projection 38.6 us against 35.0; gate/up, K = 2,048, 42.6 against 51.4.
  // Both products, 130 sizes of 700 to 4,200 tokens, 4 of 16, 2 of 8 or 6 of 64 experts, K of 512 to 4,096, one of the two 1,024 or more: 0.984 of the time without
  // them in the mean, 0.85 (2,152 tokens, 2 of 8 experts of 1,024, width 2,048, 100.2 -> 85.4 us) to 1.04, more than 1.01 at ten sizes.  With them from
  // K = 256 on, 130 sizes with a K of 512 to 896: 0.992 of this rule's time, 0.90 to 1.03: the line could lie lower)
  const int parts = K >= 1024 && fives < min(halves, mixed) ? 3 : halves < mixed ? 2 : 1;
  const int share1 = parts > 1 ? 0 : (wholes + 7) / 8, count2 = all[parts] * n_tiles, share2 = (count2 + 7) / 8;
  int b = blockIdx.x;
  const bool part = b >= share1 * 8;
  if (part) b -= share1 * 8;
  const int share = part ? share2 : share1, id = (b & 7) * share + (b >> 3);       // a die has a stretch of the tiles
  if ((b >> 3) >= share || id >= (part ? count2 : wholes)) return;
  const int nt = id % n_tiles, tile = id / n_tiles;
  const int kind = part ? parts : 0, most = kind == 0 ? GD_TILE : kind == 3 ? GdPart<5>::ROWS : GD_TILE / 2;      // its rows at most
  const int last = kind == 0 ? upto[0] : kind == 1 ? upto[1] : kind == 2 ? upto[2] : upto[3];
  const int has = kind == 0 ? own[0] : kind == 1 ? own[1] : kind == 2 ? own[2] : own[3];
  if (tile < last && tile >= last - has) {
    const int nth = tile - (last - has);
    found[0] = tid;
    found[1] = kind == 1 ? mine / GD_TILE * GD_TILE : nth * most;
    found[2] = upto[4] - mine;
    found[3] = mine;
  }
  __syncthreads();
  const int e = __builtin_amdgcn_readfirstlane(found[0]), m0 = __builtin_amdgcn_readfirstlane(found[1]);
  const int first = __builtin_amdgcn_readfirstlane(found[2]) + m0;
  const int rows = min(most, __builtin_amdgcn_readfirstlane(found[3]) - m0);
  const int n0 = nt * (MODE == 0 ? GD_TILE / 2 : GD_TILE), wm = wave >> 2, wn = wave & 3;
  if (tid < GD_TILE) {
    const int2 to = lists[(size_t)e * T + m0 + min(tid, rows - 1)];
    list[tid] = MODE == 0 ? to.x % T : to.x;
    row_weight[tid] = __int_as_float(to.y);
  }
  __syncthreads();
  MgTile<MODE> t;
  t.a = reinterpret_cast<const char*>(MODE == 0 ? A : A + (size_t)first * lda);
  t.b = reinterpret_cast<const char*>(MODE == 0 ? W + (size_t)e * N * ldw : W + (size_t)e * K);
  t.list = list;
  t.rows = rows;
  t.n0 = n0;
  t.N = N;
  t.lda = lda;
  t.ldw = ldw;
  t.up = (uint32_t)inner * (uint32_t)ldw * 2u;
  const int n = n0 + wn * (MODE == 0 ? 32 : 64);
  if (kind == 0) {
    gd_f32x4 acc[8][4];
    gd_whole(acc, t, K / GD_BK, lds, wave, lane);
    mg_store<MODE, 8>(acc, act + (size_t)first * N, planes, list, row_weight, wm * 128, rows, n, N, lane);
  } else if (kind == 3) {
    gd_f32x4 acc[5][4];
    gd_part<5>(acc, t, K / GD_BK, lds, wave, lane);
    mg_store<MODE, 5>(acc, act + (size_t)first * N, planes, list, row_weight, wm * 80, rows, n, N, lane);
  } else {
    gd_f32x4 acc[4][4];
    gd_part<4>(acc, t, K / GD_BK, lds, wave, lane);
    mg_store<MODE, 4>(acc, act + (size_t)first * N, planes, list, row_weight, wm * 64, rows, n, N, lane);
  }
}

// x [T][ldx], w_gate_up [2 E f][D] (the experts' gates, then their ups), w_down [D][E f], weights [T][ld_weights] float;
// planes [top][T][D] float; lists [E * T] pairs of ints, counts [E] ints and act [T * top][f] are workspaces of the call.  No token has more
// than top weights that are not zero.
// weights null: a table of the token ids chooses (moe_lists; up to MG_ENTRIES experts a token, entries in [0, E)).
extern "C" int blm_moe_grouped(const void* x, int ldx, const void* w_gate_up, const void* w_down, const float* weights, int ld_weights,
                               const int* table, const int* ids, const int* source_rows, const void* source_cell, int V,
                               float* planes, int* lists, int* counts, void* act, int T, int D, int E, int f, int top,
                               int units, hipStream_t stream) {
  BLM_REQUIRE(weights != nullptr || (table != nullptr && ids != nullptr && V > 0 && top <= MG_ENTRIES && (source_rows == nullptr) == (source_cell == nullptr)),
              "moe_grouped: weights, or a table of up to %d experts a token with its token ids", MG_ENTRIES);
  BLM_REQUIRE(T > 0 && E > 0 && E <= MG_MAX_EXPERTS && top > 0 && top <= 64 && top <= E && D % MG_BK == 0 && f % MG_BK == 0 && D > 0 && f > 0,
              "moe_grouped: sizes T=%d D=%d experts=%d of %d, top=%d not supported", T, D, E, f, top);
  BLM_REQUIRE(ldx >= D && ldx % 8 == 0 && (weights == nullptr || ld_weights >= E) && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w_gate_up % 16) == 0 &&
                  ((uintptr_t)w_down % 16) == 0 && ((uintptr_t)act % 16) == 0 && ((uintptr_t)lists % 8) == 0, "moe_grouped: rows must start at multiples of 16 bytes");
  BLM_REQUIRE((long long)T * ldx < (1LL << 31) && (long long)D * E * f < (1LL << 31) && (long long)T * top < (1LL << 31) / 2,
              "moe_grouped: operands of 4 GiB and more");
  const MgTable by{table, ids, source_rows, (const int* const*)source_cell, V};
  const dim3 list_blocks((unsigned)(E + (T + 63) / 64));
#define BLM_ML(N) \
  hipLaunchKernelGGL(moe_lists_kernel<N>, list_blocks, dim3(1024), 0, stream, weights, ld_weights, by, T, E, top, (int2*)lists, counts, planes, D)
  if (weights) BLM_ML(0);
  else if (top <= 4) BLM_ML(4);
  else BLM_ML(MG_ENTRIES);
#undef BLM_ML
  BLM_LAUNCH_CHECK("moe_lists");
  const long long row_tiles = ((long long)T * top + MG_BM - 1) / MG_BM + E;       // every expert's last tile may be part empty
  const long long halves = ((long long)T * top + GD_TILE / 2 - 1) / (GD_TILE / 2) + E;
  BLM_REQUIRE(units > 0 && halves * ((D + 63) / 64 > (f + 63) / 64 ? (D + 63) / 64 : (f + 63) / 64) < 2147483647LL / 64, "moe_grouped: too many tiles");
  // Tiles of 256x256 where K is one of theirs (multiples of 128), a pair of gate and up rows lies within 4 GiB and there is enough of
  // them: gate/up from halves (an expert's last one half full) on two fifths of the units on, down from as many halves as units.
  // Gate/up and down together, 16 experts of 512 at width 2048, 4 chosen, both by the smaller tiles / both by these / as the rule
  // has it, us: 400 tokens 52 / 58 / 52, 512: 55 / 60 / 55, 600: 58 / 58 / 57, 800: 63 / 59 / 59, 1,000: 76 / 69 / 69, 1,500: 72 / 72 / 72,
  // 2,048: 113 / 90 / 90, 8,000: 330 / 261 / 261 (all with the hardware's exp2 in the gating; expf takes either size of tiles 4 more at 2,048).
  const long long about = ((long long)T * top + (GD_TILE / 4) * E) / (GD_TILE / 2);
  const int duo_gates = (f + GD_TILE / 2 - 1) / (GD_TILE / 2), duo_columns = (D + GD_TILE - 1) / GD_TILE;
  if (D % 128 == 0 && D >= 256 && ((long long)E * f + f) * D * 2 < (1LL << 32) && about * duo_gates * 5 >= units * 2LL) {
    const int tiles = duo_gates;
    hipLaunchKernelGGL((moe_duo_kernel<0>), dim3((unsigned)(halves * tiles + 16)), dim3(512), 0, stream, (const bf16*)x, ldx, (const bf16*)w_gate_up, D,
                       (const int2*)lists, counts, (bf16*)act, planes, T, E, f, D, E * f, tiles, units);
  } else {
    const int tiles = (f + MG_BN / 2 - 1) / (MG_BN / 2);
    hipLaunchKernelGGL((moe_gemm_kernel<0>), dim3((unsigned)((row_tiles * tiles + 7) / 8 * 8)), dim3(64 * MG_WAVES), 0, stream, (const bf16*)x, ldx,
                       (const bf16*)w_gate_up, D, (const int2*)lists, counts, (bf16*)act, planes, T, E, f, D, E * f, tiles);
  }
  BLM_LAUNCH_CHECK("moe_grouped gate/up");
  if (f % 128 == 0 && f >= 256 && about * duo_columns >= units) {
    const int tiles = duo_columns;
    hipLaunchKernelGGL((moe_duo_kernel<1>), dim3((unsigned)(halves * tiles + 16)), dim3(512), 0, stream, (const bf16*)act, f, (const bf16*)w_down, E * f,
                       (const int2*)lists, counts, (bf16*)act, planes, T, E, D, f, E * f, tiles, units);
  } else {
    const int tiles = (D + MG_BN - 1) / MG_BN;
    hipLaunchKernelGGL((moe_gemm_kernel<1>), dim3((unsigned)((row_tiles * tiles + 7) / 8 * 8)), dim3(64 * MG_WAVES), 0, stream, (const bf16*)act, f,
                       (const bf16*)w_down, E * f, (const int2*)lists, counts, (bf16*)act, planes, T, E, D, f, E * f, tiles);
  }
  BLM_LAUNCH_CHECK("moe_grouped down");
  return 0;
}
