// Sets of lattice cells as bitmaps, shared by the density and tree stages: a
// level's cells are the bits of x-major (x, y) rows, each row of z bits
// starting a word, so bit order is the sorted key order and a cell's rank is
// the count of bits before it.  Several levels lie one after another, each
// starting a workgroup's span (BITMAP_BLOCK words), so one launch handles all.
#pragma once
#include "psr_result.h"

namespace psr {

constexpr int BITMAP_MAX_LEVELS = 16;
constexpr int BITMAP_THREADS = 256;
constexpr int BITMAP_ITEMS = 8;
constexpr int BITMAP_BLOCK = BITMAP_THREADS * BITMAP_ITEMS;

// Whether a lattice of `side` cells an axis may be a bitmap: bits take 1/32
// of an int index's memory, so eight times the dense index's cells are
// allowed (2^31 by default, 256 MB).
inline bool bitmap_fits(int64_t side) { return side * side * side <= 8 * dense_index_max_cells(); }

namespace {

// bits lo..hi-1 (of the row) that fall in word w
__device__ __forceinline__ uint32_t word_range(int w, int lo, int hi) {
  const int a = imax(lo - 32 * w, 0), b = imin(hi - 32 * w, 32);
  if (a >= b) return 0u;
  return (b == 32 ? ~0u : (1u << b) - 1u) & ~((1u << a) - 1u);
}

// even bits of v gathered into the low half
__device__ __forceinline__ uint32_t even_bits(uint64_t v) {
  v &= 0x5555555555555555ull;
  v = (v | (v >> 1)) & 0x3333333333333333ull;
  v = (v | (v >> 2)) & 0x0f0f0f0f0f0f0f0full;
  v = (v | (v >> 4)) & 0x00ff00ff00ff00ffull;
  v = (v | (v >> 8)) & 0x0000ffff0000ffffull;
  return (uint32_t)(v | (v >> 16));
}

// Sum over the workgroup's 256 threads and each thread's exclusive prefix.
__device__ __forceinline__ int block_prefix(int v, int* total) {
  __shared__ int wave_sum[BITMAP_THREADS / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
  }
  if (lane == 63) wave_sum[wave] = inc;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int k = 0; k < BITMAP_THREADS / 64; ++k) {
    if (k < wave) before += wave_sum[k];
    all += wave_sum[k];
  }
  *total = all;
  return before + inc - v;
}

__global__ void __launch_bounds__(BITMAP_THREADS) k_bits_count(const uint32_t* __restrict__ bits, int* __restrict__ sums) {
  const uint4* src = (const uint4*)(bits + (size_t)blockIdx.x * BITMAP_BLOCK) + threadIdx.x * (BITMAP_ITEMS / 4);
  int n = 0;
#pragma unroll
  for (int k = 0; k < BITMAP_ITEMS / 4; ++k) {
    const uint4 v = src[k];
    n += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
  }
  int total;
  block_prefix(n, &total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// pre[t] = set bits before word t (all levels), from the blocks' offsets
__global__ void __launch_bounds__(BITMAP_THREADS) k_bits_ranks(const uint32_t* __restrict__ bits, const int* __restrict__ offsets,
                                                             int* __restrict__ pre) {
  const size_t first = (size_t)blockIdx.x * BITMAP_BLOCK + threadIdx.x * BITMAP_ITEMS;
  int c[BITMAP_ITEMS], n = 0;
#pragma unroll
  for (int k = 0; k < BITMAP_ITEMS; ++k) {
    c[k] = n;
    n += __popc(bits[first + k]);
  }
  int total;
  const int p = block_prefix(n, &total) + offsets[blockIdx.x];
#pragma unroll
  for (int k = 0; k < BITMAP_ITEMS; ++k) pre[first + k] = p + c[k];
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == BITMAP_THREADS - 1) pre[first + BITMAP_ITEMS] = p + n;
}

}  // namespace

}  // namespace psr
