// Token choice from float logits.
//   argmax : first index of the maximum (lowest index wins ties); a row is searched by 32 blocks.
//   sample : softmax(logits / temperature) in float, nucleus (top-p) cut, inverse-CDF pick at a
//            uniform number u given by the caller, walking the kept tokens in index order; a row
//            is worked on by up to 32 blocks, each pass over it a kernel of its own.
// Nucleus rule: a token is kept while the probability mass of the tokens strictly more likely
// than it is below p; so the token that crosses p is kept, and tokens tied with it are too.
//
// The weight of a token is e = 2^((x - max) * log2(e) / temperature), in (0, 1].  The smallest
// kept weight is found by a radix selection over the bit pattern of e (positive floats order like
// their bits): three passes over the row with histograms of 11, 11 and 8 bits, each bin holding
// the mass of its tokens.  Mass is summed as 64-bit integers (e * 2^32, truncated), so the sums do
// not depend on the order in which the atomics land and the same logits always give the same cut;
// a token lighter than 2^-32 of the heaviest one counts as no mass.  The pick then walks the kept
// tokens in index order: every block owns a contiguous slice of the row, cut into chunks of 1024.
//
// One compute unit reads a row of 128K logits in about 10 us, and the five passes (maximum, three histograms, pick)
// each depend on the one before, so a row is cut into up to 32 slices for as many blocks and every pass is one
// kernel, bound by its trips to memory and its barriers.  What a pass finds for the whole row (the maximum of the
// slices' maxima, the bin of a level) every block of the next one works out for itself from what the blocks left,
// behind its first loads of logits: 1 to 2 us less than blocks that count themselves in, the last of which works it
// out.  Only the pick has such an end: the last of the row's blocks to get there draws the token.  No block ever
// waits for another.  What is asked of all threads (which one has the bin, which are behind the pick) is settled by
// one thread or one ballot: an atomic on one LDS address is done lane by lane.  And loads stand in no branch of a
// lane (SmpRow).
// Blocks of 1,024 threads (see sample_wide_slices) do without two of the passes: the second one lists the weights of
// the first level's bin, a few in a hundred of the row's, and the pick's blocks each take the other two levels from
// the list.  All of it, us, before and now: 64 rows of 128,256 tokens 56.3 and 39.2 (6.3 the maximum, 8.4, 8.5 and
// 15.2 the pick), 64 rows of 32,000 39.5 and 27.9, a row of 128,256 33.3 and 21.9; without the cut 64 rows 25.2 and
// 13.9, a row 18.0 and 9.3.
#include <mutex>

#include "common.h"
#include "no_alloc.h"


// Two stages so that a row of a large vocabulary is searched by many blocks: stage one leaves the
// best (value, index) of each slice of the row, stage two picks among the slices.  Ties go to the
// lower index in both.
#define ARGMAX_SLICES 32

__device__ __forceinline__ void argmax_merge(float& best, int& bi, float ov, int oi) {
  if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
}

__global__ void __launch_bounds__(256)
    argmax_slice_kernel(const float* __restrict__ logits, float* __restrict__ slice_val, int* __restrict__ slice_idx,
                        int V, int ld) {
  __shared__ float sv[4];
  __shared__ int si[4];
  const int row = blockIdx.y, slice = blockIdx.x;
  const int per = (V + ARGMAX_SLICES - 1) / ARGMAX_SLICES;
  const int beg = slice * per, end = min(V, beg + per);
  const float* x = logits + (size_t)row * ld;
  float best = -INFINITY;
  int bi = 0x7fffffff;
  for (int i = beg + threadIdx.x; i < end; i += blockDim.x) argmax_merge(best, bi, x[i], i);
#pragma unroll
  for (int o = BLM_WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, BLM_WAVE);
    const int oi = __shfl_xor(bi, o, BLM_WAVE);
    argmax_merge(best, bi, ov, oi);
  }
  const int lane = threadIdx.x & (BLM_WAVE - 1), w = threadIdx.x / BLM_WAVE;
  if (lane == 0) { sv[w] = best; si[w] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 4; ++k) argmax_merge(best, bi, sv[k], si[k]);
    slice_val[row * ARGMAX_SLICES + slice] = best;
    slice_idx[row * ARGMAX_SLICES + slice] = bi;
  }
}

__global__ void argmax_final_kernel(const float* __restrict__ slice_val, const int* __restrict__ slice_idx,
                                    int* __restrict__ out) {
  const int row = blockIdx.x, lane = threadIdx.x;   // one wavefront per row
  float best = lane < ARGMAX_SLICES ? slice_val[row * ARGMAX_SLICES + lane] : -INFINITY;
  int bi = lane < ARGMAX_SLICES ? slice_idx[row * ARGMAX_SLICES + lane] : 0x7fffffff;
#pragma unroll
  for (int o = BLM_WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, BLM_WAVE);
    const int oi = __shfl_xor(bi, o, BLM_WAVE);
    argmax_merge(best, bi, ov, oi);
  }
  if (lane == 0) out[row] = bi == 0x7fffffff ? 0 : bi;
}

// scratch: R * 32 floats and R * 32 ints
extern "C" int blm_argmax(const float* logits, int* out, int R, int V, int ld, float* slice_val, int* slice_idx,
                          hipStream_t stream) {
  BLM_REQUIRE(R > 0 && R <= 65535 && V > 0 && ld >= V, "argmax: bad sizes R=%d V=%d ld=%d", R, V, ld);
  hipLaunchKernelGGL(argmax_slice_kernel, dim3(ARGMAX_SLICES, R), dim3(256), 0, stream, logits, slice_val, slice_idx, V, ld);
  BLM_LAUNCH_CHECK("argmax_slice");
  hipLaunchKernelGGL(argmax_final_kernel, dim3(R), dim3(BLM_WAVE), 0, stream, slice_val, slice_idx, out);
  BLM_LAUNCH_CHECK("argmax_final");
  return 0;
}

// ---- the same without workspace arguments: see no_alloc.h ------------------------------------
// The array's name is only a stand-in in host code: its address on each device comes from
// hipGetSymbolAddress, asked once per device with that device current, and is what the kernels get.
#define ARGMAX_STATIC_DEVICES 64
static __device__ __align__(256) unsigned char argmax_static_scratch[BLM_ARGMAX_STATIC_MAX_ROWS * ARGMAX_SLICES * 8];
static void* g_argmax_static_ptr[ARGMAX_STATIC_DEVICES];
static std::mutex g_argmax_static_mutex;

static int argmax_static_address(void** ptr) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  BLM_REQUIRE(e == hipSuccess, "argmax_static: hipGetDevice failed: %s", hipGetErrorString(e));
  BLM_REQUIRE(dev >= 0 && dev < ARGMAX_STATIC_DEVICES, "argmax_static: device %d is beyond the %d this library keeps an address for",
              dev, ARGMAX_STATIC_DEVICES);
  std::lock_guard<std::mutex> hold(g_argmax_static_mutex);
  if (g_argmax_static_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(argmax_static_scratch));
    BLM_REQUIRE(e == hipSuccess && p != nullptr, "argmax_static: hipGetSymbolAddress failed on device %d: %s", dev,
                hipGetErrorString(e));
    g_argmax_static_ptr[dev] = p;
  }
  *ptr = g_argmax_static_ptr[dev];
  return 0;
}

extern "C" int blm_static_scratch_init() {
  void* p = nullptr;
  return argmax_static_address(&p);
}

extern "C" int blm_argmax_static(const float* logits, int* out, int R, int V, int ld, hipStream_t stream) {
  BLM_REQUIRE(logits != nullptr && out != nullptr, "argmax_static: logits and out must be given");
  BLM_REQUIRE(R > 0 && V > 0 && ld >= V, "argmax_static: bad sizes R=%d V=%d ld=%d", R, V, ld);
  BLM_REQUIRE(R <= BLM_ARGMAX_STATIC_MAX_ROWS, "argmax_static: %d rows, the library's own scratch array holds %d (use blm_argmax with workspaces)",
              R, BLM_ARGMAX_STATIC_MAX_ROWS);
  void* base = nullptr;
  if (argmax_static_address(&base)) return 1;
  float* slice_val = reinterpret_cast<float*>(base);
  int* slice_idx = reinterpret_cast<int*>(reinterpret_cast<unsigned char*>(base) + (size_t)BLM_ARGMAX_STATIC_MAX_ROWS * ARGMAX_SLICES * 4);
  hipLaunchKernelGGL(argmax_slice_kernel, dim3(ARGMAX_SLICES, R), dim3(256), 0, stream, logits, slice_val, slice_idx, V, ld);
  BLM_LAUNCH_CHECK("argmax_slice");
  hipLaunchKernelGGL(argmax_final_kernel, dim3(R), dim3(BLM_WAVE), 0, stream, slice_val, slice_idx, out);
  BLM_LAUNCH_CHECK("argmax_final");
  return 0;
}

#define SMP_BINS 2048
#define SMP_SLICES 32      // most blocks per row (fewer when there are many rows or few logits)
#define SMP_THREADS 256
#define SMP_CHUNK (SMP_THREADS * 4)   // elements per chunk: four neighbours per thread
#define SMP_WAVES (SMP_THREADS / BLM_WAVE)
#define SMP_ROUND 8         // chunks of a slice whose masses are summed behind one barrier

// behind a level of the selection: the digits found so far, the mass above them and the mass to reach
struct SampleState {
  uint32_t prefix;
  unsigned long long carry, target;
};

__device__ __forceinline__ void smp_store(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float smp_load(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// Whether this block is the last of its row to get here.  What the block wrote before (coherent
// stores, device-wide atomics) has been acknowledged when it counts itself in; the last one sets
// the counter back to zero.  All threads get the answer.
__device__ __forceinline__ bool smp_arrive_last(int* counter, int* flag, int n_slices) {
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  __syncthreads();
  if (threadIdx.x == 0) {
    const int before = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int last = before == n_slices - 1;
    if (last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = last;
  }
  __syncthreads();
  return *flag != 0;
}

// The four elements of thread `tid` in the chunk that starts at element i0 of row x (V elements);
// places past the row's end read as -infinity ("no token").
template <bool VEC>
__device__ __forceinline__ void smp_load4(const float* x, int i0, int V, float xs[4]) {
  if (VEC && i0 + 3 < V) {
    const float4 v = *reinterpret_cast<const float4*>(x + i0);
    xs[0] = v.x; xs[1] = v.y; xs[2] = v.z; xs[3] = v.w;
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) xs[k] = i0 + k < V ? x[i0 + k] : -INFINITY;
  }
}

__device__ __forceinline__ unsigned long long shfl_down_u64(unsigned long long v, int d) {
  const uint32_t lo = __shfl_down((uint32_t)v, d, BLM_WAVE), hi = __shfl_down((uint32_t)(v >> 32), d, BLM_WAVE);
  return ((unsigned long long)hi << 32) | lo;
}

// e * 2^32, truncated, of an e <= 1
__device__ __forceinline__ unsigned long long smp_mass(float e) {
  return e >= 1.0f ? 1ull << 32 : (unsigned long long)(uint32_t)(e * 4294967296.0f);
}

// A row's elements below `end`, to be read in pieces of four.  The loads of several pieces stand in no branch of a lane: with smp_load4,
// whose other side writes the same registers, the compiler has each wait for the one before it, a trip to memory each.
template <bool VEC>
struct SmpRow {
  const float* x;
  int end;
  float rest[3];   // VEC: the elements behind the last whole piece (end % 4 of them)

  __device__ __forceinline__ SmpRow(const float* x, int end) : x(x), end(end) {
#pragma unroll
    for (int k = 0; k < 3; ++k) rest[k] = -INFINITY;
    if (VEC && end & 3)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        if (k < (end & 3)) rest[k] = x[(end & ~3) + k];
  }

  // N pieces, `step` elements apart, this thread's first at i0; `inside`: every thread's pieces end below `end`
  template <int N>
  __device__ __forceinline__ void read(int i0, int step, bool inside, float xs[N][4]) const {
    if (VEC && inside) {
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const float4 v = *reinterpret_cast<const float4*>(x + i0 + u * step);
        xs[u][0] = v.x; xs[u][1] = v.y; xs[u][2] = v.z; xs[u][3] = v.w;
      }
    } else if (VEC) {
      float4 v[N];
#pragma unroll
      for (int u = 0; u < N; ++u) v[u] = *reinterpret_cast<const float4*>(x + max(0, min(i0 + u * step, (end & ~3) - 4)));
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const int i = i0 + u * step;
        const bool whole = i + 3 < end, part = i == (end & ~3);
        xs[u][0] = whole ? v[u].x : part ? rest[0] : -INFINITY;
        xs[u][1] = whole ? v[u].y : part ? rest[1] : -INFINITY;
        xs[u][2] = whole ? v[u].z : part ? rest[2] : -INFINITY;
        xs[u][3] = whole ? v[u].w : -INFINITY;
      }
    } else {
#pragma unroll
      for (int u = 0; u < N; ++u)
#pragma unroll
        for (int k = 0; k < 4; ++k) xs[u][k] = x[min(i0 + u * step + k, end - 1)];
#pragma unroll
      for (int u = 0; u < N; ++u)
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (i0 + u * step + k >= end) xs[u][k] = -INFINITY;
    }
  }
};

// the four times four elements of thread `tid` from element c0 on
template <bool VEC, int THREADS>
__device__ __forceinline__ void smp_load16(const SmpRow<VEC>& x, int c0, int tid, float xs[4][4]) {
  x.template read<4>(c0 + tid * 4, THREADS * 4, c0 + 16 * THREADS <= x.end, xs);
}

// the row's maximum from its slices' (at most SMP_SLICES), to every lane
__device__ __forceinline__ float smp_row_max(const float* part_max, int n_slices) {
  const int lane = threadIdx.x & (BLM_WAVE - 1);
  float m = part_max[min(lane, n_slices - 1)];
#pragma unroll
  for (int o = SMP_SLICES / 2; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, BLM_WAVE));
  return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(m)));
}

// pass 1: the slices' maxima; clears the row's first n_levels histograms for the passes to come
template <bool VEC, int THREADS>
__global__ void __launch_bounds__(THREADS)
    sample_max_kernel(const float* __restrict__ logits, int V, int ld, int slice_len, float* __restrict__ part_max,
                      unsigned long long* __restrict__ hist, int n_rows, int n_levels, const float* __restrict__ uniforms,
                      float* __restrict__ row_uniforms) {
  __shared__ float red[17];
  const int row = blockIdx.y, slice = blockIdx.x, tid = threadIdx.x;
  const float u = slice == 0 ? uniforms[row] : 0.f;   // it may lie in host memory, a longer way than the logits'
  const int begin = slice * slice_len, end = min(V, begin + slice_len);
  const SmpRow<VEC> x(logits + (size_t)row * ld, end);
  float mx = -INFINITY;
  for (int c0 = begin; c0 < end; c0 += 16 * THREADS) {
    float xs[4][4];
    smp_load16<VEC, THREADS>(x, c0, tid, xs);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int k = 0; k < 4; ++k) mx = fmaxf(mx, xs[u][k]);
  }
  for (int b = slice * THREADS + tid; b < n_levels * SMP_BINS; b += gridDim.x * THREADS)
    hist[((size_t)(b / SMP_BINS) * n_rows + row) * SMP_BINS + b % SMP_BINS] = 0ull;
  mx = block_max(mx, red);
  if (tid == 0) part_max[row * SMP_SLICES + slice] = mx;
  if (slice == 0 && tid == 0) row_uniforms[row] = u;
}

template <int THREADS>
struct SmpChoose {
  unsigned long long wave_tot[THREADS / BLM_WAVE], above;
  int found;
};

// The lowest bin above which less than `target` lies, where `carry` lies above all bins; thread t holds the masses m of bins
// [t PER, (t + 1) PER).  `first`: the target is top_p of all mass.  carry becomes what lies above the bin.  All threads get the answer.
template <int THREADS, int PER>
__device__ __forceinline__ uint32_t smp_choose(const unsigned long long (&m)[PER], bool first, float top_p, unsigned long long& carry,
                                               unsigned long long& target, SmpChoose<THREADS>& s) {
  constexpr int WAVES = THREADS / BLM_WAVE;
  const int tid = threadIdx.x, lane = tid & (BLM_WAVE - 1), w = tid / BLM_WAVE;
  unsigned long long tot = 0ull;
#pragma unroll
  for (int j = 0; j < PER; ++j) tot += m[j];
  unsigned long long suf = tot;   // becomes the mass of this thread's bins and of all higher threads' bins
#pragma unroll
  for (int d = 1; d < BLM_WAVE; d <<= 1) {
    const unsigned long long o = shfl_down_u64(suf, d);
    if (lane + d < BLM_WAVE) suf += o;
  }
  if (lane == 0) s.wave_tot[w] = suf;
  __syncthreads();
  unsigned long long total = 0ull;   // the whole mass: what every bin holds
#pragma unroll
  for (int k = 0; k < WAVES; ++k) {
    const unsigned long long t = s.wave_tot[k];
    total += t;
    suf += k > w ? t : 0ull;
  }
  if (first) {
    target = (unsigned long long)((double)top_p * (double)total);
    if (target < 1ull) target = 1ull;
  }
  unsigned long long above = carry + suf - tot;   // above this thread's highest bin
  // the bin is the one that reaches the target; exactly one thread has it (an atomic minimum over all threads that lie above is done
  // lane by lane, 2 us of a pass)
#pragma unroll
  for (int j = PER - 1; j >= 0; --j) {
    if (above < target && (above + m[j] >= target || tid * PER + j == 0)) { s.found = tid * PER + j; s.above = above; }
    above += m[j];
  }
  __syncthreads();
  const int found = s.found;
  carry = s.above;
  __syncthreads();   // the next call may write again
  return (uint32_t)found;
}

// A weight of every lane, added to the bin of its digit if the digits above are `prefix`; the first such lane's once for all that hold the
// same: where a row has many weights in one bin of level 0, few are different, as a rule, and equal ones would queue up at one address.
__device__ __forceinline__ void smp_add(unsigned long long* bins, uint32_t key, uint32_t prefix, int above_bits, int shift, uint32_t mask) {
  const bool in = (key >> above_bits) == prefix;
  const unsigned long long who = __ballot(in);
  if (who == 0) return;
  const int leader = __builtin_ctzll(who);
  const bool same = in && key == (uint32_t)__builtin_amdgcn_readlane(key, leader);
  const int times = __popcll(__ballot(same));
  if (!in || (same && (int)(threadIdx.x & (BLM_WAVE - 1)) != leader)) return;
  const unsigned long long q = smp_mass(__uint_as_float(key)) * (same ? times : 1);
  if (q) atomicAdd(&bins[(key >> shift) & mask], q);
}

// f of all elements, in a loop of four at a time: what few rows run is kept short
template <typename F>
__device__ __forceinline__ void smp_turn(float (&xs)[4][4], F f) {
#pragma unroll 1
  for (int u = 0; u < 4; ++u) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      f(xs[0][k]);
      xs[0][k] = xs[1][k];
      xs[1][k] = xs[2][k];
      xs[2][k] = xs[3][k];
    }
  }
}

// passes 2 to 4: level 0 takes bits 29..19 of the weights' bit patterns, level 1 bits 18..8, level 2 bits 7..0 (e <= 1, so bits 31 and
// 30 are clear).  LIST (level 1): no histogram; the weights with the digits chosen, in any order, and how many.  Where they are more than
// `capacity` (flat logits, few different ones: a bin is a sixteenth of a power of two wide) the slice's histogram stands in the list's place.
template <bool VEC, int LEVEL, bool LIST, int THREADS>
__global__ void __launch_bounds__(THREADS)
    sample_level_kernel(const float* __restrict__ logits, int V, int ld, int slice_len, float k2, float top_p,
                        const float* __restrict__ part_max, SampleState* states, unsigned long long* hist, int n_rows,
                        uint32_t* __restrict__ list, int* __restrict__ counts, int capacity) {
  __shared__ unsigned long long bins[SMP_BINS];
  __shared__ SmpChoose<THREADS> choose;
  __shared__ int listed;
  const int row = blockIdx.y, slice = blockIdx.x, tid = threadIdx.x;
  const int begin = slice * slice_len, end = min(V, begin + slice_len);
  const SmpRow<VEC> x(logits + (size_t)row * ld, end);
  constexpr int shift = LEVEL == 0 ? 19 : (LEVEL == 1 ? 8 : 0);
  constexpr uint32_t mask = LEVEL == 2 ? 0xffu : 0x7ffu;
  constexpr int above_bits = LEVEL == 0 ? 0 : (LEVEL == 1 ? 19 : 8);   // the digits above this level start here
  float xs[4][4];
  smp_load16<VEC, THREADS>(x, begin, tid, xs);
  const float mx = smp_row_max(part_max + row * SMP_SLICES, gridDim.x);
  uint32_t prefix = 0u;
  if (LEVEL > 0) {
    constexpr int PER = SMP_BINS / THREADS;   // a thread looks after eight bins in a row, or two
    unsigned long long m[PER], carry = 0ull, target = 0ull;
#pragma unroll
    for (int j = 0; j < PER; ++j) m[j] = hist[((size_t)(LEVEL - 1) * n_rows + row) * SMP_BINS + tid * PER + j];
    if (LEVEL == 2) {
      prefix = states[row].prefix << 11;
      carry = states[row].carry;
      target = states[row].target;
    }
    prefix |= smp_choose<THREADS, PER>(m, LEVEL == 1, top_p, carry, target, choose);
    if (slice == 0 && tid == 0) states[(size_t)(LEVEL - 1) * n_rows + row] = SampleState{prefix, carry, target};
  }
  if (LIST && tid == 0) listed = 0;
  for (int b = tid; b < SMP_BINS; b += THREADS) bins[b] = 0ull;
  __syncthreads();
  // Level 0: V tokens of weights up to a sixteenth above `light` have less mass than the 1 - top_p of it that lies below the cut (the heaviest
  // alone has 2^32), so no bin that holds one of them can be the cut's: those below `light` count for the whole mass only, in the lowest
  // bin.  Most of a row, as a rule, and a register's add in place of an atomic one each.
  const float light = LEVEL == 0 ? 0.5f * (1.0f - top_p) / (float)V : 0.f;
  uint32_t light_mass = 0u;
  uint32_t* to = LIST ? list + ((size_t)row * gridDim.x + slice) * capacity : nullptr;
  for (int c0 = begin; c0 < end; c0 += 16 * THREADS) {
    if (c0 != begin) smp_load16<VEC, THREADS>(x, c0, tid, xs);
    if (LIST) {
      uint32_t keys[4][4];
      unsigned long long who[4][4];   // the lanes whose element is one, by element
      int n = 0;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float e = __builtin_amdgcn_exp2f((xs[u][k] - mx) * k2);
          keys[u][k] = __float_as_uint(e);
          who[u][k] = __ballot((keys[u][k] >> above_bits) == prefix && e >= 0x1p-32f);
          n += __popcll(who[u][k]);
        }
      if (n == 0) continue;
      int at = 0;   // one place for the wavefront's from all of its elements
      if ((tid & (BLM_WAVE - 1)) == 0) at = atomicAdd(&listed, n);
      at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int place = at + __builtin_amdgcn_mbcnt_hi((uint32_t)(who[u][k] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)who[u][k], 0u));
          if (((who[u][k] >> (tid & (BLM_WAVE - 1))) & 1) && place < capacity) to[place] = keys[u][k];
          at += __popcll(who[u][k]);
        }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float e = __builtin_amdgcn_exp2f((xs[u][k] - mx) * k2);
          const uint32_t key = __float_as_uint(e);
          if (LEVEL == 0) {
            const bool is_light = e < light;
            light_mass += is_light ? (uint32_t)(e * 4294967296.0f) : 0u;
            if (is_light) continue;
          }
          // the digits above this level must be the ones already chosen (none at the first level)
          if (LEVEL == 0 || (key >> above_bits) == prefix) {
            const unsigned long long q = smp_mass(e);
            if (q) atomicAdd(&bins[(key >> shift) & mask], q);
          }
        }
    }
  }
  if (LEVEL == 0) {
#pragma unroll
    for (int o = BLM_WAVE / 2; o > 0; o >>= 1) light_mass += __shfl_xor(light_mass, o, BLM_WAVE);
    if ((tid & (BLM_WAVE - 1)) == 0 && light_mass) atomicAdd(&bins[0], (unsigned long long)light_mass);
  }
  __syncthreads();
  if (LIST) {
    if (tid == 0) counts[row * SMP_SLICES + slice] = listed;
    if (listed <= capacity) return;
    for (int c0 = begin; c0 < end; c0 += 16 * THREADS) {
      smp_load16<VEC, THREADS>(x, c0, tid, xs);
      smp_turn(xs, [&](float v) { smp_add(bins, __float_as_uint(__builtin_amdgcn_exp2f((v - mx) * k2)), prefix, above_bits, shift, mask); });
    }
    __syncthreads();
    for (int b = tid; b < SMP_BINS; b += THREADS) reinterpret_cast<unsigned long long*>(to)[b] = bins[b];
  } else {
    unsigned long long* row_hist = hist + ((size_t)LEVEL * n_rows + row) * SMP_BINS;
    for (int b = tid; b < SMP_BINS; b += THREADS)
      if (bins[b]) __hip_atomic_fetch_add(row_hist + b, bins[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Levels 1 and 2 from the slices' lists of weights in level 0's bin; where a slice had more than its list holds, level 1 from the
// histogram in its place and level 2 from the slice itself.  Returns the smallest kept weight.
// Bound by the instructions of one compute unit on the row's part of a bin, and by what queues up at one bin.  Draws of 128,256 logits, us, 16 and
// 64 rows, blocks of 256 threads with histograms / here, every listed weight by an atomic of its own and flat rows read twice / here: normal
// logits 46.8, 61.4 / 28.0, 41.5 / 28.2, 41.6; rounded to whole numbers (few different weights) 48.3, 67.5 / 55.2, 70.2 / 35.1, 50.5;
// normal by 0.05 49.3, 67.5 / 39.8, 54.3 / 37.1, 51.3, by 0.01 (a bin holds most of the row) 55.0, 78.8 / 69.4, 92.0 / 57.4, 81.1; all the
// same 83.8, 132.6 / 81.9, 108.1 / 80.3, 107.7.  Of 50,021 (addresses of four bytes) 64 rows: 57.1 / 37.1 / 38.3, 58.2 / 48.5 / 49.3, 59.2 /
// 40.3 / 41.6, 64.3 / 72.9 / 64.9, 82.2 / 76.1 / 70.6.
template <bool VEC, int THREADS>
__device__ __forceinline__ uint32_t smp_choose_listed(const float* x, int V, int slice_len, float mx, float k2, SampleState state,
                                                      const uint32_t* list, const int* counts, int n_slices, int capacity,
                                                      unsigned long long* bins, SmpChoose<THREADS>& choose) {
  constexpr int KEPT = 8, PER = SMP_BINS / THREADS;
  const int tid = threadIdx.x, group = THREADS / n_slices, slice = tid / group, first = tid % group;
  const uint32_t* mine = list + (size_t)slice * capacity;
  uint32_t keys[KEPT];   // asked for with their number
#pragma unroll
  for (int i = 0; i < KEPT; ++i) keys[i] = mine[min(first + i * group, capacity - 1)];
  const int lane = tid & (BLM_WAVE - 1), any = counts[min(lane, n_slices - 1)], own = counts[slice];
  const unsigned long long over = __ballot(lane < n_slices && any > capacity);      // the slices without a list
  const int n = own > capacity ? 0 : own;
#pragma unroll
  for (int i = 0; i < KEPT; ++i) keys[i] = first + i * group < n ? keys[i] : 0u;
  uint32_t prefix = state.prefix;
#pragma unroll
  for (int level = 1; level < 3; ++level) {
    const int shift = level == 1 ? 8 : 0, above_bits = level == 1 ? 19 : 8;
    const uint32_t mask = level == 1 ? 0x7ffu : 0xffu;
    for (int b = tid; b <= (int)mask; b += THREADS) bins[b] = 0ull;
    __syncthreads();
    auto add = [&](uint32_t key, int times) {
      if ((key >> above_bits) != prefix) return;
      const unsigned long long q = smp_mass(__uint_as_float(key)) * times;
      if (q) atomicAdd(&bins[(key >> shift) & mask], q);
    };
    // a wavefront's at once where they are one weight, as in rows of few different ones
    auto add_all = [&](const auto& of, int i0) {
      constexpr int N = sizeof(of) / sizeof(of[0]);
      const uint32_t lead = __builtin_amdgcn_readfirstlane(of[0]);
      bool alike = i0 + (N - 1) * group < n;
#pragma unroll
      for (int i = 0; i < N; ++i) alike &= of[i] == lead;
      if (__ballot(!alike) == 0) {
        if (lane == 0) add(lead, N * BLM_WAVE);
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (i0 + i * group < n) add(of[i], 1);
      }
    };
    add_all(keys, first);
    for (int i0 = first + KEPT * group; i0 < n; i0 += 4 * group) {
      uint32_t more[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) more[i] = mine[min(i0 + i * group, capacity - 1)];
      add_all(more, i0);
    }
    if (level == 2 && over) {
      // the logits whose weights may have these digits, to 1e-5 of the exponent (the instruction's error is a hundredth of it)
      const float low = __log2f(__uint_as_float(prefix << 8)), high = __log2f(__uint_as_float((prefix << 8) | 0xffu));
      const float centre = 0.5f * (low + high), reach = prefix ? 0.5f * (high - low) + 1e-5f : INFINITY;
      for (unsigned long long left = over; left; left &= left - 1) {
        const int begin = __builtin_ctzll(left) * slice_len, end = min(V, begin + slice_len);
        const SmpRow<VEC> part(x, end);
        for (int c0 = begin; c0 < end; c0 += 16 * THREADS) {
          float xs[4][4];
          smp_load16<VEC, THREADS>(part, c0, tid, xs);
          smp_turn(xs, [&](float v) {
            const float t = (v - mx) * k2;
            if (__ballot(!(fabsf(t - centre) > reach))) smp_add(bins, __float_as_uint(__builtin_amdgcn_exp2f(t)), prefix, above_bits, shift, mask);
          });
        }
      }
    }
    __syncthreads();
    if (level == 1) {
      unsigned long long m[PER];
#pragma unroll
      for (int j = 0; j < PER; ++j) m[j] = bins[tid * PER + j];
      for (unsigned long long left = over; left; left &= left - 1) {
        const unsigned long long* of = reinterpret_cast<const unsigned long long*>(list + (size_t)__builtin_ctzll(left) * capacity);
#pragma unroll
        for (int j = 0; j < PER; ++j) m[j] += of[tid * PER + j];
      }
      prefix = (prefix << 11) | smp_choose<THREADS, PER>(m, false, 0.f, state.carry, state.target, choose);
    } else {
      unsigned long long m[1] = {tid < 256 ? bins[tid] : 0ull};
      prefix = (prefix << 8) | smp_choose<THREADS, 1>(m, false, 0.f, state.carry, state.target, choose);
    }
  }
  return prefix;
}

// inclusive prefix over the block's first SMP_THREADS threads in thread order, and their total
__device__ __forceinline__ float smp_block_scan(float v, float* wave_sums, float& total) {
  const int lane = threadIdx.x & (BLM_WAVE - 1), w = threadIdx.x / BLM_WAVE;
  float incl = v;
#pragma unroll
  for (int d = 1; d < BLM_WAVE; d <<= 1) {
    const float o = __shfl_up(incl, d, BLM_WAVE);
    if (lane >= d) incl += o;
  }
  __syncthreads();   // wave_sums may still be read from an earlier call
  if (lane == BLM_WAVE - 1) wave_sums[w] = incl;      // (of all wavefronts; those behind the first four are not read)
  __syncthreads();
  float before = 0.f;
  total = 0.f;
  for (int k = 0; k < SMP_WAVES; ++k) {
    if (k == w) before = total;
    total += wave_sums[k];
  }
  return before + incl;
}

// *to becomes the lowest (the highest) thread for which `is` holds, if there is one: one atomic for a wavefront
__device__ __forceinline__ void smp_lowest(int* to, bool is) {
  const unsigned long long who = __ballot(is);
  if ((threadIdx.x & (BLM_WAVE - 1)) == 0 && who) atomicMin(to, (int)threadIdx.x + __builtin_ctzll(who));
}
__device__ __forceinline__ void smp_highest(int* to, bool is) {
  const unsigned long long who = __ballot(is);
  if ((threadIdx.x & (BLM_WAVE - 1)) == 0 && who) atomicMax(to, (int)threadIdx.x + 63 - __builtin_clzll(who));
}

// last pass: the kept mass of every chunk; the last block finds the chunk that holds the pick and
// the token in it.  CUT 0: none, every token with a weight is kept; 1: from the histograms; 2: from the lists.
template <bool VEC, int CUT, int THREADS>
__global__ void __launch_bounds__(THREADS)
    sample_pick_kernel(const float* __restrict__ logits, const float* __restrict__ row_uniforms, int* __restrict__ out, int V,
                       int ld, int slice_len, float k2, const float* __restrict__ part_max, const SampleState* __restrict__ states,
                       const unsigned long long* __restrict__ hist, const uint32_t* __restrict__ list, const int* __restrict__ counts,
                       int capacity, float* chunk_mass, int* counters, int counter_step) {
  __shared__ float red[17];
  constexpr int GROUPS = THREADS / SMP_THREADS, EACH = GROUPS == 1 ? SMP_ROUND : SMP_ROUND / 2, ROUND = EACH * GROUPS;
  __shared__ float wave_sums[THREADS / BLM_WAVE];
  __shared__ float round_sums[ROUND][SMP_WAVES];
  __shared__ int flag, hit, last_with_mass;
  __shared__ SmpChoose<THREADS> choose;
  __shared__ unsigned long long bins[CUT == 2 ? SMP_BINS : 1];
  const int row = blockIdx.y, slice = blockIdx.x, tid = threadIdx.x;
  const float* x = logits + (size_t)row * ld;
  const int begin = slice * slice_len, end = min(V, begin + slice_len);
  const int chunks = slice_len / SMP_CHUNK;            // per slice
  // the chunks of the slice, ROUND at a time, a chunk to SMP_THREADS of the threads: all loads first, one barrier per round
  const int group = tid / SMP_THREADS, part = tid % SMP_THREADS;
  float xs[EACH][4];
  const SmpRow<VEC> slice_row(x, end);
  auto load_round = [&](int c0) {
    slice_row.template read<EACH>(begin + (c0 + group) * SMP_CHUNK + part * 4, GROUPS * SMP_CHUNK, begin + (c0 + ROUND) * SMP_CHUNK <= end, xs);
  };
  load_round(0);
  const float u = row_uniforms[row];
  const float mx = smp_row_max(part_max + row * SMP_SLICES, gridDim.x);
  uint32_t tau = 0u;   // smallest kept weight, as a bit pattern
  if (CUT == 1) {
    SampleState state = states[gridDim.y + row];
    const unsigned long long m[1] = {tid < 256 ? hist[((size_t)2 * gridDim.y + row) * SMP_BINS + tid] : 0ull};
    tau = (state.prefix << 8) | smp_choose<THREADS, 1>(m, false, 0.f, state.carry, state.target, choose);
  }
  if (CUT == 2)
    tau = smp_choose_listed<VEC, THREADS>(x, V, slice_len, mx, k2, states[row], list + (size_t)row * gridDim.x * capacity, counts + row * SMP_SLICES,
                                          gridDim.x, capacity, bins, choose);
  auto kept = [&](float v) {
    const float e = __builtin_amdgcn_exp2f((v - mx) * k2);
    return (__float_as_uint(e) >= tau && e > 0.f) ? e : 0.f;
  };
  float* row_mass = chunk_mass + (size_t)row * gridDim.x * chunks;
  for (int c0 = 0; c0 < chunks; c0 += ROUND) {
    if (c0) load_round(c0);
    __syncthreads();   // round_sums may still be read from the round before
#pragma unroll
    for (int r = 0; r < EACH; ++r) {
      const float s4 = ((kept(xs[r][0]) + kept(xs[r][1])) + kept(xs[r][2])) + kept(xs[r][3]);
      const float ws = wave_sum(s4);
      if ((tid & (BLM_WAVE - 1)) == 0) round_sums[r * GROUPS + group][part / BLM_WAVE] = ws;
    }
    __syncthreads();
    if (tid < ROUND && c0 + tid < chunks) {
      float t = 0.f;
      for (int k = 0; k < SMP_WAVES; ++k) t += round_sums[tid][k];
      smp_store(row_mass + slice * chunks + c0 + tid, t);
    }
  }
  if (!smp_arrive_last(counters + (size_t)row * counter_step, &flag, gridDim.x)) return;

  // the first SMP_THREADS threads have the chunks from here on, and at last the chosen chunk's elements; the others none
  const bool in = tid < SMP_THREADS;
  // chunks in index order: slice by slice; first their total, then the chunk in which u * total falls
  const int n = gridDim.x * chunks;
  if (tid == 0) { hit = 0x7fffffff; last_with_mass = -1; }
  int first_idx = 0x7fffffff, last_idx = -1;   // this thread's lowest chunk that passes u * total, its highest with mass
  float first_front = 0.f, last_front = 0.f;   // and the mass in front of each
  float want;
  if (n <= SMP_THREADS) {
    const float mass = tid < n ? smp_load(row_mass + tid) : 0.f;
    float total;
    const float incl = smp_block_scan(mass, wave_sums, total);
    want = u * total;
    if (mass > 0.f) {
      if (want < incl) { first_idx = tid; first_front = incl - mass; }
      last_idx = tid;
      last_front = incl - mass;
    }
  } else {
    float total = 0.f;
    for (int base = 0; base < n; base += SMP_THREADS) {
      float t;
      smp_block_scan(in && base + tid < n ? smp_load(row_mass + base + tid) : 0.f, wave_sums, t);
      total += t;
    }
    want = u * total;
    float run = 0.f;   // mass in front of this round of chunks
    for (int base = 0; base < n; base += SMP_THREADS) {
      const float mass = in && base + tid < n ? smp_load(row_mass + base + tid) : 0.f;
      float t;
      const float incl = run + smp_block_scan(mass, wave_sums, t);
      if (mass > 0.f) {
        if (want < incl && first_idx == 0x7fffffff) { first_idx = base + tid; first_front = incl - mass; }
        last_idx = base + tid;
        last_front = incl - mass;
      }
      run += t;
    }
  }
  if (n <= SMP_THREADS) {   // a wavefront's lowest and highest are its first and last lane's that have one
    smp_lowest(&hit, first_idx != 0x7fffffff);
    smp_highest(&last_with_mass, last_idx >= 0);
  } else {
    if (first_idx != 0x7fffffff) atomicMin(&hit, first_idx);
    if (last_idx >= 0) atomicMax(&last_with_mass, last_idx);
  }
  __syncthreads();
  const int chunk = hit != 0x7fffffff ? hit : last_with_mass;   // rounding may leave u * total at the upper edge
  if (chunk < 0) {   // no token has a weight: cannot happen (the maximum has weight 1); answer something valid
    if (tid == 0) out[row] = 0;
    return;
  }
  if (first_idx == chunk) red[0] = first_front;
  else if (last_idx == chunk) red[0] = last_front;
  __syncthreads();
  const float front = red[0];   // mass in front of the chosen chunk
  __syncthreads();
  const int cs = chunk / chunks, cc = chunk % chunks;
  const int i0 = cs * slice_len + cc * SMP_CHUNK + tid * 4;
  float es[4];
  smp_load4<VEC>(x, i0, in ? min(V, cs * slice_len + slice_len) : 0, xs[0]);
#pragma unroll
  for (int k = 0; k < 4; ++k) es[k] = kept(xs[0][k]);
  const float s4 = ((es[0] + es[1]) + es[2]) + es[3];
  float t;
  const float incl = front + smp_block_scan(s4, wave_sums, t);
  if (tid == 0) { hit = 0x7fffffff; last_with_mass = -1; }
  __syncthreads();
  smp_lowest(&hit, s4 > 0.f && want < incl);
  smp_highest(&last_with_mass, s4 > 0.f);
  __syncthreads();
  const int owner = hit != 0x7fffffff ? hit : last_with_mass;   // at least one thread has a kept token
  if (tid == owner) {
    float acc = incl - s4;
    int chosen = -1, last = -1;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (es[k] > 0.f) {
        acc += es[k];
        last = i0 + k;
        if (want < acc && chosen < 0) chosen = i0 + k;
      }
    }
    out[row] = chosen >= 0 ? chosen : last;   // rounding may leave want at the thread's upper edge
  }
}

// Blocks per row: a slice's own time falls with their number, the device-wide atomics of all rows' blocks (histograms, the pick's
// arrivals) grow with it and with the rows, so the best number goes with sqrt(V / R): the power of two next to sqrt(V / (16 R)).  Us, for
// 4 / 8 / 16 / 32 blocks, with the nucleus cut: 128,256 logits: 1 row 45.9 / 31.2 / 24.1 / 22.0, 8 rows 46.0 / 31.9 / 25.5 / 23.6, 128 rows
// 72 / 69 / 72 / 80, 512 rows 221 / 231 / 225 / 251; 32,000 logits: 8 rows 25.1 / 22.6 / 23.6 / 24.6, 512 rows 78 / 96 / 115 / 194; without
// it: 128,256 logits: 8 rows 13.8 / 10.6 / 9.3 / 9.6, 64 rows 16.7 / 13.9 / 14.1 / 17.9.  All with a cache line for each row's arrival
// counter: side by side, 1,024 blocks queue up at two lines (64 rows of 128K in 16 blocks, an arrival in every pass, 90.5 us for 79.6).
// With the cut, 16 to 128 rows: blocks of 1,024 threads, one to a compute unit, that ask for 16,384 tokens at once and take two of the
// levels from lists, where a slice has at least three quarters of so many.  Us, 256 threads as above / 1,024 threads in 8 blocks a row up
// to 32 rows, in 4 up to 64, in 2 up to 128: 128,256 logits: 8 rows 23.6 / 25.9, 16 rows 25.7 / 26.0, 24 rows 28.5 / 27.1, 32 rows 29.3 /
// 27.9, 64 rows 43.7 / 39.6, 96 rows 57.1 / 55.1, 128 rows 68.8 / 64.9, 192 rows (2 blocks) 95.2 / 96.1; 50,021 logits: 32 rows 31.5 / 31.3,
// 48 rows 37.1 / 34.9, 64 rows 40.6 / 36.0, 128 rows 59.2 / 47.5; 32,000 logits: 64 rows (4 blocks) 28.1 / 28.8, 128 rows 32.2 / 28.6.
// Without the cut 64 rows of 128,256 logits 13.9 / 15.7.
static int sample_wide_slices(int R, int V, int cut) {      // 0: 256 threads
  const int n = R <= 32 ? 8 : R <= 64 ? 4 : 2;
  return cut && R >= 16 && R <= 128 && V >= n * 12288 ? n : 0;
}
static int sample_slices(int R, int V, int cut) {
  if (const int wide = sample_wide_slices(R, V, cut)) return wide;
  int n = 4;
  while (n < SMP_SLICES && 32LL * n * n * R <= V) n *= 2;
  return n;
}
static int sample_slice_len(int R, int V, int cut) {
  const int n = sample_slices(R, V, cut);
  return ((V + n - 1) / n + SMP_CHUNK - 1) / SMP_CHUNK * SMP_CHUNK;
}

// How many of a slice's weights a list holds: no fewer than its place takes a histogram (SMP_BINS of 64 bits).
static int sample_list_capacity(int slice_len) { return slice_len / 4 > 2 * SMP_BINS ? slice_len / 4 : 2 * SMP_BINS; }
static size_t sample_even(size_t n) { return n + (n & 1); }

// Bytes of scratch that blm_sample needs for R rows of V logits (see there for the layout).
extern "C" long long blm_sample_scratch_bytes(int R, int V) {
  long long chunks = 0;
  for (int cut = 0; cut < 2; ++cut) {
    const long long n = (long long)sample_slices(R, V, cut) * (sample_slice_len(R, V, cut) / SMP_CHUNK);
    chunks = n > chunks ? n : chunks;
  }
  const long long wide = sample_wide_slices(R, V, 1), lists = wide * sample_list_capacity(sample_slice_len(R, V, 1));
  return (long long)R * ((wide ? 1 : 3) * SMP_BINS * 8 + 2 * sizeof(SampleState) + SMP_SLICES * 8 + (1 + chunks + lists) * 4) + 4;
}

// scratch: blm_sample_scratch_bytes(R, V) bytes, 8-byte aligned: the rows' histograms, their states behind two levels, the slices'
// maxima and the lengths of their lists, the rows' uniforms, the chunks' masses, the lists.  counters: R zeroed ints, counter_step apart, left zeroed.
extern "C" int blm_sample(const float* logits, const float* uniforms, int* out, int R, int V, int ld,
                          float temperature, float top_p, void* scratch, int* counters, int counter_step, hipStream_t stream) {
  BLM_REQUIRE(R > 0 && R <= 65535 && V > 0 && ld >= V, "sample: bad sizes R=%d V=%d ld=%d", R, V, ld);
  BLM_REQUIRE(temperature > 0.f, "sample: temperature must be > 0 (got %g); use argmax for 0", (double)temperature);
  BLM_REQUIRE(top_p > 0.f, "sample: top_p must be > 0 (got %g)", (double)top_p);
  BLM_REQUIRE(counter_step >= 1, "sample: counters %d apart", counter_step);
  BLM_REQUIRE(scratch != nullptr && ((uintptr_t)scratch % 8) == 0 && counters != nullptr, "sample: scratch and counters needed");
  const int cut = top_p < 1.0f ? 1 : 0;
  const int slices = sample_slices(R, V, cut), slice_len = sample_slice_len(R, V, cut), capacity = sample_list_capacity(slice_len);
  const bool wide = sample_wide_slices(R, V, cut) != 0;
  const int levels = !cut ? 0 : wide ? 1 : 3;
  unsigned long long* hist = reinterpret_cast<unsigned long long*>(scratch);
  SampleState* states = reinterpret_cast<SampleState*>(hist + (size_t)levels * R * SMP_BINS);
  float* part_max = reinterpret_cast<float*>(states + 2 * (size_t)R);
  int* counts = reinterpret_cast<int*>(part_max + (size_t)R * SMP_SLICES);
  float* row_uniforms = reinterpret_cast<float*>(counts + (size_t)R * SMP_SLICES);
  float* chunk_mass = row_uniforms + R;
  uint32_t* list = reinterpret_cast<uint32_t*>(row_uniforms + sample_even(R + (size_t)R * slices * (slice_len / SMP_CHUNK)));      // 8 bytes aligned
  const float k2 = 1.4426950408889634f / temperature;
  const bool vec = V >= 4 && ld % 4 == 0 && ((uintptr_t)logits % 16) == 0;
  dim3 grid(slices, R), block(wide ? 1024 : SMP_THREADS);
#define SMP_LEVEL(VEC, LEVEL, LIST, THREADS)                                                                              \
  hipLaunchKernelGGL((sample_level_kernel<VEC, LEVEL, LIST, THREADS>), grid, block, 0, stream, logits, V, ld, slice_len, k2, top_p, \
                     part_max, states, hist, R, list, counts, capacity)
#define SMP_PICK(VEC, CUT, THREADS)                                                                                       \
  hipLaunchKernelGGL((sample_pick_kernel<VEC, CUT, THREADS>), grid, block, 0, stream, logits, row_uniforms, out, V, ld, slice_len, k2, \
                     part_max, states, hist, list, counts, capacity, chunk_mass, counters, counter_step)
#define SMP_MAX(VEC, THREADS)                                                                                             \
  hipLaunchKernelGGL((sample_max_kernel<VEC, THREADS>), grid, block, 0, stream, logits, V, ld, slice_len, part_max, hist, R, levels, \
                     uniforms, row_uniforms)
#define SMP_LAUNCH(VEC)                                                                                                   \
  do {                                                                                                                    \
    if (wide) {                                                                                                           \
      SMP_MAX(VEC, 1024);                                                                                                 \
      SMP_LEVEL(VEC, 0, false, 1024);                                                                                     \
      SMP_LEVEL(VEC, 1, true, 1024);                                                                                      \
      SMP_PICK(VEC, 2, 1024);                                                                                             \
    } else if (cut) {                                                                                                     \
      SMP_MAX(VEC, SMP_THREADS);                                                                                          \
      SMP_LEVEL(VEC, 0, false, SMP_THREADS);                                                                              \
      SMP_LEVEL(VEC, 1, false, SMP_THREADS);                                                                              \
      SMP_LEVEL(VEC, 2, false, SMP_THREADS);                                                                              \
      SMP_PICK(VEC, 1, SMP_THREADS);                                                                                      \
    } else {                                                                                                              \
      SMP_MAX(VEC, SMP_THREADS);                                                                                          \
      SMP_PICK(VEC, 0, SMP_THREADS);                                                                                      \
    }                                                                                                                     \
  } while (0)
  if (vec) SMP_LAUNCH(true);
  else SMP_LAUNCH(false);
#undef SMP_LAUNCH
#undef SMP_MAX
#undef SMP_PICK
#undef SMP_LEVEL
  BLM_LAUNCH_CHECK("sample");
  return 0;
}
