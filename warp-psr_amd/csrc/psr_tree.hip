// Stage 4: level-by-level brood tree (src/warp_psr/tree.py:152-201).
//
// Candidate broods of level d are level d-1 cells with coordinates in
// [-2^d, 2^d); they are packed as three (d+1)-bit fields (offset by 2^d), so the
// unique-sort costs ceil((3d+4)/8) radix passes instead of the 60-bit tree key.
// Children of the sorted unique broods are placed at their lexicographic rank
// directly (no second sort).
//
// Up to depth 11 (bitmap_fits) the sets are bitmaps instead, and nothing is
// sorted: see TreeLattice.
#include "psr_bitmap.h"

namespace psr {

namespace {

struct BroodPack {
  int d;
  PSR_HD uint64_t pack(int x, int y, int z) const {
    const int off = 1 << d, b = d + 1;
    return ((uint64_t)(x + off) << (2 * b)) | ((uint64_t)(y + off) << b) | (uint64_t)(z + off);
  }
  PSR_HD uint64_t sentinel() const { return (uint64_t)1 << (3 * (d + 1)); }
  PSR_HD int64_t to_tree_key(uint64_t p) const {
    const int off = 1 << d, b = d + 1;
    const uint64_t m = ((uint64_t)1 << b) - 1;
    return tree_key((int)(p >> (2 * b)) - off, (int)((p >> b) & m) - off, (int)(p & m) - off);
  }
};

PSR_HD bool in_support(int x, int y, int z, int lim) {
  return imin(imin(x, y), z) >= -lim && imax(imax(x, y), z) < lim;
}

// tree.py:41-50 (_seed_broods)
template <class T>
__global__ void k_seed_broods(const int64_t* __restrict__ nkeys, const T* __restrict__ nvals, int64_t count, int d,
                              BroodPack bp, uint64_t* __restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int64_t key = nkeys[i];
  const int nd = key_d(key);
  const T* v = nvals + 3 * i;
  const T w = -T(0);  // the negated fourth record component
  const T len2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + w * w;
  uint64_t packed = bp.sentinel();
  if (nd >= d && double(len2) > 0.0) {
    const int sh = nd - d;
    packed = bp.pack((key_x(key) >> sh) >> 1, (key_y(key) >> sh) >> 1, (key_z(key) >> sh) >> 1);
  }
  out[i] = packed;
}

// tree.py:30-34 (_coarse, lo = -1)
__global__ void k_coarse_broods(int cc, BroodPack bp, uint64_t* __restrict__ out) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cc * cc * cc) return;
  out[i] = bp.pack(i / (cc * cc) - 1, (i / cc) % cc - 1, i % cc - 1);
}

// tree.py:52-64 (_support_broods) for radius 1 (27 per request) or 0
__global__ void k_support_broods(const int64_t* __restrict__ src, int64_t count, int radius, int lim, BroodPack bp,
                                 uint64_t* __restrict__ out) {
  const int width = 2 * radius + 1, w3 = width * width * width;
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= count * w3) return;
  const int64_t i = idx / w3;
  const int j = (int)(idx % w3);
  const int64_t key = src[i];
  const int px = tkey_x(key) >> 1, py = tkey_y(key) >> 1, pz = tkey_z(key) >> 1;
  const int x = px + j / (width * width) - radius, y = py + (j / width) % width - radius, z = pz + j % width - radius;
  out[idx] = in_support(x, y, z, lim) ? bp.pack(x, y, z) : bp.sentinel();
}

__global__ void k_parent_tree_keys(const int64_t* __restrict__ src, int64_t count, BroodPack bp, uint64_t* __restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int64_t key = src[i];
  out[i] = bp.pack(tkey_x(key) >> 1, tkey_y(key) >> 1, tkey_z(key) >> 1);
}

__global__ void k_unpack_unique(const uint64_t* __restrict__ keys, const int* __restrict__ heads, const int* __restrict__ prefix,
                                int64_t n, BroodPack bp, int64_t* __restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && heads[i]) out[prefix[i]] = bp.to_tree_key(keys[i]);
}

// tree.py:78-96: lexicographic rank of each child of the sorted unique broods.
__global__ void k_expand_broods(const int64_t* __restrict__ broods, int64_t nb, int64_t* __restrict__ children) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nb) return;
  const int64_t key = broods[i];
  const int64_t xp = (key >> 40) << 40, xyp = (key >> 20) << 20;
  const int64_t x0 = lower_bound(broods, nb, xp), x1 = lower_bound(broods, nb, xp + ((int64_t)1 << 40));
  const int64_t xy0 = lower_bound(broods, nb, xyp), xy1 = lower_bound(broods, nb, xyp + ((int64_t)1 << 20));
  const int cx = 2 * tkey_x(key), cy = 2 * tkey_y(key), cz = 2 * tkey_z(key);
  for (int k = 0; k < 8; ++k) {
    const int ox = (k >> 2) & 1, oy = (k >> 1) & 1, oz = k & 1;
    // children before this one: all of smaller x runs, then the x half, the
    // smaller y runs inside this x run, the y half, earlier z, then z half
    const int64_t dest = 8 * x0 + 4 * ox * (x1 - x0) + 4 * (xy0 - x0) + 2 * oy * (xy1 - xy0) + 2 * (i - xy0) + oz;
    children[dest] = tree_key(cx + ox, cy + oy, cz + oz);
  }
}

// tree.py:105-123 (basis marks/fill)
__global__ void k_basis_marks(const int64_t* __restrict__ keys, int64_t n, int d, int* __restrict__ marks) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t k = keys[i];
  const int x = tkey_x(k), y = tkey_y(k), z = tkey_z(k);
  const int lim = 1 << d;
  marks[i] = (imin(imin(x, y), z) >= 0 && imax(imax(x, y), z) <= lim) ? 1 : 0;
}

__global__ void k_basis_fill(const int64_t* __restrict__ keys, const int* __restrict__ marks, const int* __restrict__ prefix,
                             int64_t n, int d, int64_t* __restrict__ out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !marks[i]) return;
  const int64_t k = keys[i];
  out[prefix[i]] = basis_key(d, tkey_x(k), tkey_y(k), tkey_z(k));
}

// Sorted unique tree keys of packed candidates (keyed.py:157-178).
DArray<int64_t> unique_packed(DArray<uint64_t>& cand, int64_t total, BroodPack bp, hipStream_t s) {
  DArray<int64_t> out;
  if (!total) return out;
  DArray<int> ids(total, s), heads(total, s), prefix(total, s), cnt(1, s);
  fill_iota(ids.data(), total, s);
  sort_pairs_u64(cand.data(), ids.data(), total, bits_for(bp.sentinel()), s);
  mark_heads_u64(cand.data(), total, bp.sentinel(), heads.data(), s);
  scan_exclusive_i32(heads.data(), prefix.data(), total, cnt.data(), s);
  const int count = read_int(cnt.data(), s);
  out.reset(count, s);
  if (count) {
    hipLaunchKernelGGL(k_unpack_unique, dim3(blocks_for(total, 256)), dim3(256), 0, s, (const uint64_t*)cand.data(),
                       (const int*)heads.data(), (const int*)prefix.data(), total, bp, out.data());
    KERNEL_CHECK();
  }
  return out;
}

// ------------------------------------------------------------ bitmap form
// The broods of every level as bits of a small lattice.  Level d's broods are
// level d - 1 cells from -2 to max(2^(d-1), 1) + 1 on each axis: seeds lie in
// the cube, the coarse box ends one cell outside it, a parent is the floor of
// half a coordinate and a support cell lies within one of that, and
// floor(-2 / 2) - 1 = -2, floor((2^d + 1) / 2) + 1 = 2^(d-1) + 1 (d > 0).  A
// row of z bits starts a word, rows are x-major, so bit order is the sorted
// key order, ranks are population counts, and a level's set follows from the
// finer level's by word operations (halve, dilate) instead of 27 sorted
// candidates per brood.  Sizes: 2.7 MB of words for all levels of depth 9.
//
// The whole tree is two host reads and about 20 launches; with a unique sort
// a level it was some 25 launches and a host read a level (2.45 ms at depth 9
// for 800,000 points, 0.56 ms at depth 4 for 512; 0.37 and 0.10 ms now).
struct TreeLattice {
  int side[BITMAP_MAX_LEVELS + 1];        // cells per axis
  int wz[BITMAP_MAX_LEVELS + 1];          // words per (x, y) row
  uint32_t base[BITMAP_MAX_LEVELS + 1];   // first word of the level
};

PSR_HD int lattice_side(int d) { return (d > 1 ? 1 << (d - 1) : 1) + 4; }

// Halved cells of the finer lattice's rows [x0, x1] x [y0, y1]: bit k of the
// result is set if one of those rows has a cell whose parent is row position
// 32 w - 1 + k (k = 0..33).  A cell at lattice index i has its parent at
// (i >> 1) + 1: both lattices start at -2.
__device__ __forceinline__ uint64_t halved_rows(const uint32_t* __restrict__ fine, int side, int wz, int x0, int x1, int y0, int y1,
                                                int w) {
  uint32_t c0 = 0, c1 = 0, c2 = 0;
  for (int x = imax(x0, 0); x <= imin(x1, side - 1); ++x)
    for (int y = imax(y0, 0); y <= imin(y1, side - 1); ++y) {
      const uint32_t* row = fine + (uint32_t)(x * side + y) * (uint32_t)wz;
      if (w > 0 && 2 * w - 1 < wz) c0 |= row[2 * w - 1];
      if (2 * w < wz) c1 |= row[2 * w];
      if (2 * w + 1 < wz) c2 |= row[2 * w + 1];
    }
  uint64_t v = ((uint64_t)c2 << 32) | c1;
  v |= v >> 1;
  return ((uint64_t)even_bits(v) << 2) | (((c0 >> 30) & 3u) ? 2u : 0u) | (((c0 >> 28) & 3u) ? 1u : 0u);
}

// tree.py:41-50 (_seed_broods) for every level: the first record of each word
// gathers the word's run of records (keys are sorted, z fastest).
template <class T>
__global__ void k_tree_seeds(const int64_t* __restrict__ nkeys, const T* __restrict__ nvals, int64_t count, TreeLattice lat,
                             uint32_t* __restrict__ bits) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int64_t key = nkeys[i];
  // cell z, brood z >> 1, lattice (z >> 1) + 2, word ((z >> 1) + 2) >> 5: z + 4 over 64
  const int64_t run = (key + 4) >> 6;
  if (i > 0 && ((nkeys[i - 1] + 4) >> 6) == run) return;
  uint32_t word = 0;
  for (int64_t j = i; j < count && ((nkeys[j] + 4) >> 6) == run; ++j) {
    const T* v = nvals + 3 * j;
    const T w = -T(0);  // the negated fourth record component
    const T len2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + w * w;
    if (double(len2) > 0.0) word |= 1u << (((key_z(nkeys[j]) >> 1) + 2) & 31);
  }
  if (!word) return;
  const int d = key_d(key), side = lat.side[d], wz = lat.wz[d];
  const int x = (key_x(key) >> 1) + 2, y = (key_y(key) >> 1) + 2, z = (key_z(key) >> 1) + 2;
  atomicOr(&bits[lat.base[d] + (uint32_t)(x * side + y) * (uint32_t)wz + (uint32_t)(z >> 5)], word);
}

// Level d's broods from the finer level's (tree.py:152-201): the seeds
// already there, the coarse box (_coarse, lo = -1), the supports of the
// requests (radius 1, _support_broods) and the parents of the finer broods
// (radius 0; within the supports where the requests are those broods), clipped
// to [-2^d, 2^d).  requests: the finer lattice's bits, null for none.  With
// moved (requests_up from request_src, on this level's lattice) also the next
// level's requests where they move up (tree.py:176-180): their parents.
__global__ void __launch_bounds__(BITMAP_THREADS) k_tree_level(TreeLattice lat, int d, int coarse, const uint32_t* __restrict__ finer,
                                                             const uint32_t* __restrict__ requests, uint32_t* __restrict__ bits,
                                                             const uint32_t* __restrict__ request_src,
                                                             uint32_t* __restrict__ requests_up, uint32_t words) {
  const uint32_t t = blockIdx.x * BITMAP_THREADS + threadIdx.x;
  if (t >= words) return;
  const int side = lat.side[d], wz = lat.wz[d], fside = lat.side[d + 1], fwz = lat.wz[d + 1];
  const int w = (int)(t % (uint32_t)wz), y = (int)((t / (uint32_t)wz) % (uint32_t)side), x = (int)(t / (uint32_t)(wz * side));
  uint32_t out = 0;
  const int lo = imax(2 - (1 << d), 0), hi = imin(2 + (1 << d), side);  // in_support on lattice indices
  if (x >= lo && x < hi && y >= lo && y < hi) {
    if (requests) {
      const uint64_t p = halved_rows(requests, fside, fwz, 2 * x - 4, 2 * x + 1, 2 * y - 4, 2 * y + 1, w);
      out |= (uint32_t)(p | (p >> 1) | (p >> 2));
    }
    if (finer && finer != requests) out |= (uint32_t)(halved_rows(finer, fside, fwz, 2 * x - 2, 2 * x - 1, 2 * y - 2, 2 * y - 1, w) >> 1);
    out &= word_range(w, lo, hi);
  }
  if (coarse && x >= 1 && x <= coarse && y >= 1 && y <= coarse) out |= word_range(w, 1, coarse + 1);
  if (out) bits[t] |= out;
  if (requests_up)
    requests_up[t] = request_src ? (uint32_t)(halved_rows(request_src, fside, fwz, 2 * x - 2, 2 * x - 1, 2 * y - 2, 2 * y - 1, w) >> 1) &
                                       word_range(w, 0, side)
                                 : 0u;
}

// Per level: first workgroup, and the arrays.  Keys of one level fill whole
// workgroups, as words do.
struct TreeArrays {
  int levels;
  int block0[BITMAP_MAX_LEVELS + 1];
  int64_t count[BITMAP_MAX_LEVELS];
  int64_t* tree[BITMAP_MAX_LEVELS];
  int64_t* basis[BITMAP_MAX_LEVELS];
};

// ranks at the levels' first words and the end, for the host
__global__ void k_tree_starts(TreeLattice lat, int levels, const int* __restrict__ pre, uint32_t words, int* __restrict__ out) {
  const int d = threadIdx.x;
  if (d <= levels) out[d] = pre[d < levels ? lat.base[d] : words];
}

__global__ void k_basis_starts(TreeArrays arr, const int* __restrict__ offsets, int* __restrict__ out) {
  const int d = threadIdx.x;
  if (d <= arr.levels) out[d] = offsets[arr.block0[d]];
}

__device__ __forceinline__ int level_of_block(const TreeArrays& a, int block) {
  int d = 0;
  for (int k = 1; k < a.levels; ++k) d = block >= a.block0[k] ? k : d;
  return d;
}

// tree.py:78-96: the children of every brood at their lexicographic rank.
// With ranks at the starts of x planes and (x, y) rows, the children before
// one are: all of smaller planes, then this plane's x half, its smaller rows,
// the row's y half, the row's earlier broods, the z half.
__global__ void __launch_bounds__(BITMAP_THREADS) k_tree_children(TreeLattice lat, TreeArrays arr, const uint32_t* __restrict__ bits,
                                                                const int* __restrict__ pre) {
  const int d = level_of_block(arr, (int)blockIdx.x);
  const int side = lat.side[d], wz = lat.wz[d];
  const uint32_t base = lat.base[d], words = (uint32_t)(side * side) * (uint32_t)wz;
  int64_t* tree = arr.tree[d];
  const int level0 = pre[base];
  for (int k = 0; k < BITMAP_ITEMS; ++k) {
    const uint32_t t = (blockIdx.x - (uint32_t)arr.block0[d]) * BITMAP_BLOCK + k * BITMAP_THREADS + threadIdx.x;
    if (t >= words) return;
    uint32_t b = bits[base + t];
    if (!b) continue;
    const int w = (int)(t % (uint32_t)wz), y = (int)((t / (uint32_t)wz) % (uint32_t)side), x = (int)(t / (uint32_t)(wz * side));
    const uint32_t plane = base + (uint32_t)(x * side) * (uint32_t)wz, row = base + t - (uint32_t)w;
    const int x0 = pre[plane], x1 = pre[plane + (uint32_t)side * (uint32_t)wz], y0 = pre[row], y1 = pre[row + (uint32_t)wz];
    int i = pre[base + t];
    const int64_t at = 8 * (int64_t)(x0 - level0) + 4 * (int64_t)(y0 - x0);
    const int cx = 2 * (x - 2), cy = 2 * (y - 2);
    for (; b; b &= b - 1, ++i) {
      const int cz = 2 * (32 * w + __builtin_ctz(b) - 2);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int ox = c >> 1, oy = c & 1;
        const int64_t dest = at + 4 * (int64_t)ox * (x1 - x0) + 2 * (int64_t)oy * (y1 - y0) + 2 * (int64_t)(i - y0);
        tree[dest] = tree_key(cx + ox, cy + oy, cz);
        tree[dest + 1] = tree_key(cx + ox, cy + oy, cz + 1);
      }
    }
  }
}

// compact_basis (tree.py:126-143) of every level: nodes within [0, 2^d]
__device__ __forceinline__ bool in_basis(int64_t key, int d) {
  const int x = tkey_x(key), y = tkey_y(key), z = tkey_z(key), lim = 1 << d;
  return imin(imin(x, y), z) >= 0 && imax(imax(x, y), z) <= lim;
}

__global__ void __launch_bounds__(BITMAP_THREADS) k_basis_sums(TreeArrays arr, int* __restrict__ sums) {
  const int d = level_of_block(arr, (int)blockIdx.x);
  const int64_t first = (int64_t)((int)blockIdx.x - arr.block0[d]) * BITMAP_BLOCK + threadIdx.x;
  int n = 0;
#pragma unroll
  for (int k = 0; k < BITMAP_ITEMS; ++k) {
    const int64_t i = first + k * BITMAP_THREADS;
    if (i < arr.count[d] && in_basis(arr.tree[d][i], d)) ++n;
  }
  int total;
  block_prefix(n, &total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ void __launch_bounds__(BITMAP_THREADS) k_basis_keys(TreeArrays arr, const int* __restrict__ offsets) {
  const int d = level_of_block(arr, (int)blockIdx.x);
  const int64_t first = (int64_t)((int)blockIdx.x - arr.block0[d]) * BITMAP_BLOCK + threadIdx.x * BITMAP_ITEMS;
  int64_t key[BITMAP_ITEMS];
  int n = 0;
#pragma unroll
  for (int k = 0; k < BITMAP_ITEMS; ++k) {
    key[k] = first + k < arr.count[d] ? arr.tree[d][first + k] : KMAX;
    if (key[k] != KMAX && !in_basis(key[k], d)) key[k] = KMAX;
    if (key[k] != KMAX) ++n;
  }
  int total;
  int64_t at = (int64_t)block_prefix(n, &total) + offsets[blockIdx.x] - offsets[arr.block0[d]];
#pragma unroll
  for (int k = 0; k < BITMAP_ITEMS; ++k)
    if (key[k] != KMAX) arr.basis[d][at++] = basis_key(d, tkey_x(key[k]), tkey_y(key[k]), tkey_z(key[k]));
}

template <class T> void tree_from_bitmaps(Result<T>& r) {
  hipStream_t s = r.s;
  const int depth = r.prm.depth, full = r.prm.full_depth, base = r.prm.base_depth;
  TreeLattice lat{};
  size_t words = 0;
  for (int d = 0; d <= depth + 1 && d <= BITMAP_MAX_LEVELS; ++d) {
    lat.side[d] = lattice_side(d);
    lat.wz[d] = (lat.side[d] + 31) / 32;
    lat.base[d] = (uint32_t)words;
    if (d > depth) break;  // the level past the finest has a shape, no words
    const size_t level = (size_t)lat.side[d] * lat.side[d] * lat.wz[d];
    words += (level + BITMAP_BLOCK - 1) / BITMAP_BLOCK * BITMAP_BLOCK;
  }
  auto level_words = [&](int d) { return (uint32_t)(lat.side[d] * lat.side[d]) * (uint32_t)lat.wz[d]; };
  const int blocks = (int)(words / BITMAP_BLOCK);
  DArray<uint32_t> bits(words, s), moved(base < depth ? words : 0, s);
  bits.zero();
  const int64_t records = r.normal_offsets[depth + 1];
  if (records) {
    hipLaunchKernelGGL(k_tree_seeds<T>, dim3(blocks_for(records, 256)), dim3(256), 0, s, (const int64_t*)r.normal_keys.data(),
                       (const T*)r.normal_vals.data(), records, lat, bits.data());
    KERNEL_CHECK();
  }
  // requests of level d (level-d cells, on level d + 1's lattice): the finer
  // broods above the base level; from there on the parents of the requests
  // before, kept in moved at level d + 1's place
  auto requests_of = [&](int d) -> const uint32_t* {
    if (d >= depth || moved.empty()) return nullptr;
    return (d > base ? bits.data() : moved.data()) + lat.base[d + 1];
  };
  for (int d = depth; d >= 0; --d) {
    const uint32_t* finer = d < depth ? bits.data() + lat.base[d + 1] : nullptr;
    const bool up = d >= 1 && d - 1 <= base && !moved.empty();  // level d - 1's requests live on this lattice
    const int coarse = d <= full ? (d == 0 ? 2 : (1 << (d - 1)) + 2) : 0;
    const uint32_t n = level_words(d);
    hipLaunchKernelGGL(k_tree_level, dim3(blocks_for(n, BITMAP_THREADS)), dim3(BITMAP_THREADS), 0, s, lat, d, coarse, finer, requests_of(d),
                       bits.data() + lat.base[d], requests_of(d), up ? moved.data() + lat.base[d] : (uint32_t*)nullptr, n);
    KERNEL_CHECK();
  }
  // ranks, then one read of the levels' brood counts
  DArray<int> sums(blocks, s), pre(words + 1, s);
  hipLaunchKernelGGL(k_bits_count, dim3(blocks), dim3(BITMAP_THREADS), 0, s, (const uint32_t*)bits.data(), sums.data());
  KERNEL_CHECK();
  scan_exclusive_i32(sums.data(), sums.data(), blocks, nullptr, s);
  hipLaunchKernelGGL(k_bits_ranks, dim3(blocks), dim3(BITMAP_THREADS), 0, s, (const uint32_t*)bits.data(), (const int*)sums.data(),
                     pre.data());
  KERNEL_CHECK();
  TreeArrays arr{};
  arr.levels = depth + 1;
  std::vector<int> first(depth + 2);
  {
    DArray<int> starts(depth + 2, s);
    hipLaunchKernelGGL(k_tree_starts, dim3(1), dim3(64), 0, s, lat, depth + 1, (const int*)pre.data(), (uint32_t)words, starts.data());
    KERNEL_CHECK();
    read_bytes(first.data(), starts.data(), sizeof(int) * (depth + 2), s);
  }
  for (int d = 0; d <= depth; ++d) {
    LevelState<T>& L = r.levels[d];
    arr.block0[d] = (int)(lat.base[d] / BITMAP_BLOCK);
    arr.count[d] = 8 * (int64_t)(first[d + 1] - first[d]);
    L.tree_keys.reset((size_t)arr.count[d], s);
    L.basis_keys.reset((size_t)arr.count[d], s);
    arr.tree[d] = L.tree_keys.data();
    arr.basis[d] = L.basis_keys.data();
  }
  hipLaunchKernelGGL(k_tree_children, dim3(blocks), dim3(BITMAP_THREADS), 0, s, lat, arr, (const uint32_t*)bits.data(),
                     (const int*)pre.data());
  KERNEL_CHECK();
  // basis keys: the same order, filtered
  int key_blocks = 0;
  for (int d = 0; d <= depth; ++d) {
    arr.block0[d] = key_blocks;
    key_blocks += (int)((arr.count[d] + BITMAP_BLOCK - 1) / BITMAP_BLOCK);
  }
  arr.block0[depth + 1] = key_blocks;
  std::vector<int> ends(depth + 2, 0);
  if (key_blocks) {
    DArray<int> basis_sums(key_blocks + 1, s), starts(depth + 2, s);
    hipLaunchKernelGGL(k_basis_sums, dim3(key_blocks), dim3(BITMAP_THREADS), 0, s, arr, basis_sums.data());
    KERNEL_CHECK();
    scan_exclusive_i32(basis_sums.data(), basis_sums.data(), key_blocks, basis_sums.data() + key_blocks, s);
    hipLaunchKernelGGL(k_basis_keys, dim3(key_blocks), dim3(BITMAP_THREADS), 0, s, arr, (const int*)basis_sums.data());
    KERNEL_CHECK();
    hipLaunchKernelGGL(k_basis_starts, dim3(1), dim3(64), 0, s, arr, (const int*)basis_sums.data(), starts.data());
    KERNEL_CHECK();
    read_bytes(ends.data(), starts.data(), sizeof(int) * (depth + 2), s);
  }
  for (int d = 0; d <= depth; ++d) {
    r.levels[d].basis_count = ends[d + 1] - ends[d];
    r.levels[d].basis_keys.shrink((size_t)r.levels[d].basis_count);
  }
}

}  // namespace

template <class T> void stage_tree(Result<T>& r) {
  hipStream_t s = r.s;
  const int depth = r.prm.depth, full = r.prm.full_depth, base = r.prm.base_depth;
  r.levels.resize(depth + 1);
  if (bitmap_fits(lattice_side(depth))) return tree_from_bitmaps(r);
  DArray<int64_t> broods, requests;
  bool have_requests = false;
  // per-level basis counts stay on the device until the loop ends (one read):
  // each level's basis keys are allocated for all 8 * broods candidates
  DArray<int> basis_counts(depth + 1, s);
  basis_counts.zero();
  for (int d = depth; d >= 0; --d) {
    const int64_t r0 = r.normal_offsets[d], r1 = r.normal_offsets[d + 1];
    const int64_t count = r1 - r0;
    // parents = previous broods (level-d cells); kept for this iteration
    DArray<int64_t> parents = std::move(broods);
    BroodPack bp{d};
    if (d > base) {
      requests.reset(parents.size(), s);
      if (parents.size())
        HIP_CHECK(hipMemcpyAsync(requests.data(), parents.data(), parents.size() * sizeof(int64_t), hipMemcpyDeviceToDevice, s));
    } else if (have_requests) {
      // requests move up one level: unique parents (tree.py:176-180)
      const int64_t m = (int64_t)requests.size();
      DArray<uint64_t> rk(m, s);
      BroodPack up{d + 1};  // parents of level-(d+1) cells are level-d cells; pack range of level d+1 broods
      if (m) {
        hipLaunchKernelGGL(k_parent_tree_keys, dim3(blocks_for(m, 256)), dim3(256), 0, s, (const int64_t*)requests.data(), m,
                           up, rk.data());
        KERNEL_CHECK();
      }
      requests = unique_packed(rk, m, up, s);
    } else {
      requests.reset(parents.size(), s);
      if (parents.size())
        HIP_CHECK(hipMemcpyAsync(requests.data(), parents.data(), parents.size() * sizeof(int64_t), hipMemcpyDeviceToDevice, s));
    }
    have_requests = true;
    const int cc = d <= full ? (d == 0 ? 2 : (1 << (d - 1)) + 2) : 0;
    const int64_t nc = (int64_t)cc * cc * cc;
    const int64_t ns = (int64_t)requests.size() * 27;
    const int64_t np = (int64_t)parents.size();
    const int64_t total = count + nc + ns + np;
    DArray<uint64_t> cand(total, s);
    if (count) {
      hipLaunchKernelGGL(k_seed_broods<T>, dim3(blocks_for(count, 256)), dim3(256), 0, s,
                         (const int64_t*)r.normal_keys.data() + r0, (const T*)r.normal_vals.data() + 3 * r0, count, d, bp,
                         cand.data());
      KERNEL_CHECK();
    }
    if (nc) {
      hipLaunchKernelGGL(k_coarse_broods, dim3(blocks_for(nc, 256)), dim3(256), 0, s, cc, bp, cand.data() + count);
      KERNEL_CHECK();
    }
    if (ns) {
      hipLaunchKernelGGL(k_support_broods, dim3(blocks_for(ns, 256)), dim3(256), 0, s, (const int64_t*)requests.data(),
                         (int64_t)requests.size(), 1, 1 << d, bp, cand.data() + count + nc);
      KERNEL_CHECK();
    }
    if (np) {
      hipLaunchKernelGGL(k_support_broods, dim3(blocks_for(np, 256)), dim3(256), 0, s, (const int64_t*)parents.data(), np, 0,
                         1 << d, bp, cand.data() + count + nc + ns);
      KERNEL_CHECK();
    }
    broods = unique_packed(cand, total, bp, s);
    LevelState<T>& L = r.levels[d];
    const int64_t nb = (int64_t)broods.size();
    L.tree_keys.reset(8 * nb, s);
    if (nb) {
      hipLaunchKernelGGL(k_expand_broods, dim3(blocks_for(nb, 256)), dim3(256), 0, s, (const int64_t*)broods.data(), nb,
                         L.tree_keys.data());
      KERNEL_CHECK();
    }
    // compact_basis (tree.py:126-143)
    const int64_t nt = 8 * nb;
    L.basis_keys.reset(nt, s);
    if (nt) {
      DArray<int> marks(nt, s), prefix(nt, s);
      hipLaunchKernelGGL(k_basis_marks, dim3(blocks_for(nt, 256)), dim3(256), 0, s, (const int64_t*)L.tree_keys.data(), nt, d,
                         marks.data());
      KERNEL_CHECK();
      scan_exclusive_i32(marks.data(), prefix.data(), nt, basis_counts.data() + d, s);
      hipLaunchKernelGGL(k_basis_fill, dim3(blocks_for(nt, 256)), dim3(256), 0, s, (const int64_t*)L.tree_keys.data(),
                         (const int*)marks.data(), (const int*)prefix.data(), nt, d, L.basis_keys.data());
      KERNEL_CHECK();
    }
  }
  std::vector<int> counts(depth + 1);
  read_bytes(counts.data(), basis_counts.data(), sizeof(int) * (depth + 1), s);
  for (int d = 0; d <= depth; ++d) {
    r.levels[d].basis_count = counts[d];
    r.levels[d].basis_keys.shrink((size_t)counts[d]);
  }
}

template void stage_tree<float>(Result<float>&);
template void stage_tree<double>(Result<double>&);

}  // namespace psr
