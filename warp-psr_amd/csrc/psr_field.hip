// Stage 6: cumulative coefficients (src/warp_psr/field.py:187-210), the
// reference evaluation (field.py:364-421), the isovalue
// (reconstruction.py:76-138) and the cube/model transforms (transforms.py).
#include "psr_field_index.h"
#include "psr_mesh.h"
#include "../../include/warp_psr_amd_field.h"

#include <cmath>

namespace psr {

namespace {

__global__ void k_field_columns(const int64_t* __restrict__ keys, int64_t n, int* __restrict__ start, int* __restrict__ end) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  auto cell = [&](int64_t k) {
    const int d = key_d(k);
    return column_base(d) + (int64_t)key_x(k) * ((1 << d) + 1) + key_y(k);
  };
  const int64_t c = cell(keys[i]);
  if (i == 0 || cell(keys[i - 1]) != c) start[c] = (int)i;
  if (i == n - 1 || cell(keys[i + 1]) != c) end[c] = (int)(i + 1);
}

template <class T>
__global__ void k_cumulative(FieldIndex f, int d, const T* __restrict__ coef, T* __restrict__ cum) {
  const int64_t i = f.off[d] + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= f.off[d + 1]) return;
  const int64_t key = f.keys[i];
  const int x = key_x(key), y = key_y(key), z = key_z(key);
  T value = T(0);
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b) {  // corners a*4 + b*2 + c in order; one lookup per (x, y) column
      int64_t found[2];
      level_run<2>(f, d - 1, x / 2 + a, y / 2 + b, z / 2, 2, found);
      for (int c = 0; c < 2; ++c) {
        const T h = (T(1) - fabs(T(x) * T(.5) - T(x / 2 + a))) * (T(1) - fabs(T(y) * T(.5) - T(y / 2 + b))) *
                    (T(1) - fabs(T(z) * T(.5) - T(z / 2 + c)));
        if (h > T(0) && found[c] >= 0) value = value + cum[found[c]] * h;
      }
    }
  cum[i] = value + coef[i];
}

template <class T> PSR_HD int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Node words of levels 0..word_depth from the concatenated sorted keys: the
// first key of each word (a key whose predecessor lies in another column or
// below the word's first node) collects the word's keys, at most 32, so no two
// threads write one word.  A shared node can be the first key of both its
// words.  Words without keys keep the cleared value (no bits).
__device__ __forceinline__ void field_word(const int64_t* __restrict__ keys, int64_t n, int word_depth,
                                           NodeWord* __restrict__ words, int64_t i) {
  const int64_t key = keys[i];
  const int d = key_d(key);
  if (d > word_depth) return;
  const int z = key_z(key), wc = word_columns(d), own = word_of(z);
  const int64_t column = key >> 16;
  const int before = i > 0 && (keys[i - 1] >> 16) == column ? key_z(keys[i - 1]) : -1;  // z of the column's key below
  for (int w = z == 31 * own && own > 0 ? own - 1 : own; w <= own && w < wc; ++w) {
    if (before >= 31 * w) continue;
    uint32_t bits = 0;
    for (int64_t j = i; j < n && (keys[j] >> 16) == column && key_z(keys[j]) <= 31 * w + 31; ++j) bits |= 1u << (key_z(keys[j]) - 31 * w);
    words[word_at(d, key_x(key), key_y(key), w)] = NodeWord{bits, (int32_t)i};
  }
}

__global__ void k_field_words(const int64_t* __restrict__ keys, int64_t n, int word_depth, NodeWord* __restrict__ words) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) field_word(keys, n, word_depth, words, i);
}

template <class V> struct LevelArrays {
  const V* a[MAX_LEVELS];
};

// The levels' keys one after another, and the levels' offsets in them.
__global__ void __launch_bounds__(LEVEL_BLOCK) k_concat_keys(LevelBlocks lb, LevelArrays<int64_t> in, int64_t* __restrict__ keys,
                                                             int* __restrict__ offsets) {
  if (blockIdx.x == 0 && (int)threadIdx.x <= lb.levels) offsets[threadIdx.x] = lb.first[threadIdx.x];
  const int d = lb.level_of((int)blockIdx.x), i = lb.row_of((int)blockIdx.x, d, (int)threadIdx.x);
  if (i >= 0) keys[lb.first[d] + i] = in.a[d][i];
}

// The levels' values one after another; a level without an array holds zeros.
template <class T>
__global__ void __launch_bounds__(LEVEL_BLOCK) k_concat_values(LevelBlocks lb, LevelArrays<T> in, T* __restrict__ out) {
  const int d = lb.level_of((int)blockIdx.x), i = lb.row_of((int)blockIdx.x, d, (int)threadIdx.x);
  if (i >= 0) out[lb.first[d] + i] = in.a[d] ? in.a[d][i] : T(0);
}

// One level's eight trilinear corners of a cube point: for each of the four z
// pairs, the index of the first node present (0 if none), which
// of the two are present (two bits each, the lower node's first) and which
// count: present and not left of the point's floor.  A present pair's nodes
// are neighbours in memory.  up: cell + 1 > floor, so the upper corner has
// weight fr, else 1 - fr.  Flags are packed: registers bound the kernel.
template <class T> struct Corners {
  int first[4];
  unsigned flags;  // present: bits 0..7, counts: bits 8..15, up: bits 16..18
  __device__ __forceinline__ unsigned present(int k) const { return (flags >> (2 * k)) & 3u; }
  __device__ __forceinline__ unsigned counts(int k) const { return (flags >> (8 + 2 * k)) & 3u; }
  __device__ __forceinline__ bool up(int a) const { return (flags >> (16 + a)) & 1u; }
};

// field.py:371-393 (add_level), lookups only
template <class T, bool WORDS>
__device__ __forceinline__ void find_corners(const FieldIndex& f, const T* p, int d, Corners<T>& c) {
  const int n = 1 << d;
  int cell[3], base[3];
  c.flags = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const T t = p[a] * T(n);
    cell[a] = clampi<T>((int)ceil(t) - 1, 0, n - 1);
    base[a] = (int)floor(t);
    c.flags |= cell[a] + 1 > base[a] ? 1u << (16 + a) : 0u;
  }
  if constexpr (WORDS) {
    const int w = word_of(cell[2]), bit = cell[2] - 31 * w;
    NodeWord word[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) word[k] = f.words[word_at(d, cell[0] + k / 2, cell[1] + k % 2, w)];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const unsigned present = (word[k].bits >> bit) & 3u;
      c.flags |= present << (2 * k);
      c.first[k] = present ? word[k].first + __popc(word[k].bits & ((1u << bit) - 1u)) : 0;
    }
  } else {
    for (int a = 0; a < 2; ++a)
      for (int b = 0; b < 2; ++b) {
        int64_t found[2];
        level_run<2>(f, d, cell[0] + a, cell[1] + b, cell[2], 2, found);
        c.flags |= ((found[0] >= 0 ? 1u : 0u) | (found[1] >= 0 ? 2u : 0u)) << (2 * (2 * a + b));
        c.first[2 * a + b] = (int)(found[0] >= 0 ? found[0] : found[1] >= 0 ? found[1] : 0);
      }
  }
  // a corner left of the point's floor (a knot owned by the left cell) does not count
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const unsigned right = (cell[2] < base[2] ? 0u : 1u) | (cell[2] + 1 < base[2] ? 0u : 2u);
    if (imin(cell[0] + k / 2 - base[0], cell[1] + k % 2 - base[1]) >= 0) c.flags |= (c.present(k) & right) << (8 + 2 * k);
  }
}

// The pair's two values of a field array, +0 where the node does not count.
// PAIRS: one load of both, for arrays of K + 1 values (the last pair's second
// one is never counted); else two, of present nodes.
template <class T> struct ValuePair;
template <> struct ValuePair<float> { typedef float type __attribute__((ext_vector_type(2), aligned(4))); };
template <> struct ValuePair<double> { typedef double type __attribute__((ext_vector_type(2), aligned(8))); };
template <bool PAIRS, class T>
__device__ __forceinline__ void corner_values(const Corners<T>& c, bool used, const T* __restrict__ src, T* v) {
  using Pair = typename ValuePair<T>::type;
  Pair p[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (PAIRS) {
      p[k] = *(const Pair*)(src + c.first[k]);
    } else {
      p[k].x = c.present(k) ? src[c.first[k]] : T(0);
      p[k].y = c.present(k) == 3u ? src[c.first[k] + 1] : T(0);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const T a = p[k].x, b = p[k].y;
    v[2 * k] = used && (c.counts(k) & 1u) ? a : T(0);
    v[2 * k + 1] = used && (c.counts(k) & 2u) ? ((c.present(k) & 1u) ? b : a) : T(0);
  }
}

// field.py:371-393 (add_level), sums only, corners in order.  An absent
// corner enters as the coefficient +0: its products are zeros of either sign,
// and a sum that starts at +0 is never -0, so adding them changes no bit.
template <class T>
__device__ __forceinline__ void blend_corners(const Corners<T>& c, const T* v, const T* p, int d, T* res) {
  const T n = T(1 << d);
  T h[3][2], sg[3][2];
#pragma unroll
  for (int a = 0; a < 3; ++a) {  // lower corner: node <= floor, upper corner: by `up`
    const T t = p[a] * n, fr = t - T((int)floor(t));
    h[a][0] = T(1) - fr;
    sg[a][0] = T(-1);
    h[a][1] = c.up(a) ? fr : T(1) - fr;
    sg[a][1] = c.up(a) ? T(1) : T(-1);
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int x = k / 4, y = k / 2 % 2, z = k % 2;
    res[0] = res[0] + v[k] * h[0][x] * h[1][y] * h[2][z];
    res[1] = res[1] + v[k] * n * sg[0][x] * h[1][y] * h[2][z];
    res[2] = res[2] + v[k] * n * h[0][x] * sg[1][y] * h[2][z];
    res[3] = res[3] + v[k] * n * h[0][x] * h[1][y] * sg[2][z];
  }
}

// field.py:395-420 (reference evaluation) at a cube point p, nudged off the
// cube's faces here: value and cube-space gradient.  WORDS: every level has
// node words, so the three dependent steps (leaf words, the three blended
// levels' words, their coefficients) each issue all their loads at once; the
// general form searches level by level, a chain of some 40 dependent loads
// (812,000 queries at depth 9 in float64: 561 us; 151 us with words, bound by
// the lines they miss; 156 us where four waves a SIMD are asked for, which
// spills).
template <class T, bool WORDS, bool PAIRS>
__device__ __forceinline__ void field_at(const FieldIndex& f, const T* __restrict__ coef, const T* __restrict__ cum, int depth, T (&p)[3],
                                         T (&res)[4]) {
  int leaf = 0;
  if constexpr (WORDS) {
    // the cell at level d is the finest cell >> (depth - d): scaling by a
    // power of two is exact and ceil(ceil(m) / 2^k) = ceil(m / 2^k)
    const int nf = 1 << depth;
    int cf[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) cf[a] = clampi<T>((int)ceil(p[a] * T(nf)) - 1, 0, nf - 1);
    constexpr int AHEAD = 4;  // levels whose words are loaded together
    bool found = false;
    for (int top = depth; top >= 0 && !found; top -= AHEAD) {
      NodeWord w[AHEAD];
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) {
        const int d = imax(top - k, 0), up = depth - d;
        const int x = cf[0] >> up, y = cf[1] >> up, z = cf[2] >> up;
        w[k] = f.words[word_at(d, x, y, word_of(z))];
      }
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) {
        const int d = imax(top - k, 0);
        const int z = cf[2] >> (depth - d);
        if (!found && ((w[k].bits >> (z - 31 * word_of(z))) & 1u)) { leaf = d; found = true; }
      }
    }
  } else {
    for (int d = depth; d >= 0; --d) {
      const int n = 1 << d;
      const int c0 = clampi<T>((int)ceil(p[0] * T(n)) - 1, 0, n - 1);
      const int c1 = clampi<T>((int)ceil(p[1] * T(n)) - 1, 0, n - 1);
      const int c2 = clampi<T>((int)ceil(p[2] * T(n)) - 1, 0, n - 1);
      int64_t idx;
      level_run<1>(f, d, c0, c1, c2, 1, &idx);
      if (idx >= 0) { leaf = d; break; }
    }
  }
  for (int a = 0; a < 3; ++a) {
    if (p[a] == T(0)) p[a] = T(1e-6);
    else if (p[a] == T(1)) p[a] = T(1.0 - 1e-6);
  }
  const bool lower = leaf > 0, upper = leaf < depth;
  Corners<T> c0, c1, c2;
  find_corners<T, WORDS>(f, p, leaf, c0);
  find_corners<T, WORDS>(f, p, imax(leaf - 1, 0), c1);
  find_corners<T, WORDS>(f, p, imin(leaf + 1, depth), c2);
  T v0[8], v1[8], v2[8];
  corner_values<PAIRS>(c0, true, coef, v0);
  corner_values<PAIRS>(c1, lower, cum, v1);
  corner_values<PAIRS>(c2, upper, coef, v2);
  res[0] = res[1] = res[2] = res[3] = T(0);
  blend_corners(c0, v0, p, leaf, res);
  if (lower) {
    T r2[4] = {T(0), T(0), T(0), T(0)};
    blend_corners(c1, v1, p, leaf - 1, r2);
    for (int a = 0; a < 4; ++a) res[a] = res[a] + r2[a];
  }
  if (upper) {
    T r2[4] = {T(0), T(0), T(0), T(0)};
    blend_corners(c2, v2, p, leaf + 1, r2);
    for (int a = 0; a < 4; ++a) res[a] = res[a] + r2[a];
  }
}

template <class T, bool WORDS>
__global__ void __launch_bounds__(256)
k_evaluate(FieldIndex f, const T* __restrict__ coef, const T* __restrict__ cum, int depth, const T* __restrict__ queries, int64_t m, Affine<T> A, int point_div_mode,
                                                  const T* __restrict__ divisors, T* __restrict__ values, T* __restrict__ grads,
                                                  int* __restrict__ valid) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  T q0 = queries[3 * i], q1 = queries[3 * i + 1], q2 = queries[3 * i + 2];
  if (point_div_mode) {  // reconstruction.py:23-29 (_centroids)
    const T w = divisors[i];
    q0 = q0 / w; q1 = q1 / w; q2 = q2 / w;
  }
  T p[3];
  for (int r = 0; r < 3; ++r) p[r] = A.L[3 * r] * q0 + A.L[3 * r + 1] * q1 + A.L[3 * r + 2] * q2 + A.t[r];
  const bool ok = isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2]) && tmin(tmin(p[0], p[1]), p[2]) >= T(0) &&
                  tmax(tmax(p[0], p[1]), p[2]) <= T(1);
  if (valid) valid[i] = ok ? 1 : 0;
  if (!ok) {
    values[i] = T(NAN);
    if (grads) { grads[3 * i] = T(NAN); grads[3 * i + 1] = T(NAN); grads[3 * i + 2] = T(NAN); }
    return;
  }
  T res[4];
  field_at<T, WORDS, true>(f, coef, cum, depth, p, res);
  values[i] = res[0];
  if (grads)
    for (int c = 0; c < 3; ++c) grads[3 * i + c] = A.L[c] * res[1] + A.L[3 + c] * res[2] + A.L[6 + c] * res[3];
}

// The field less its isovalue at grid nodes (z fastest from plane `start`) or
// at the corners of cells: a mesh's classification and vertices need values
// alone, so no points, gradients or validity go through memory (points,
// evaluation and subtraction of one 17 x 256 x 256 slab: 50 us; 20 us here).
template <bool WORDS>
__global__ void __launch_bounds__(256) k_mesh_values(FieldIndex f, const float* __restrict__ coef, const float* __restrict__ cum,
                                                     int depth, Affine<float> A, MeshGrid g, int start,
                                                     const int* __restrict__ cells, int64_t n, const float* __restrict__ iso,
                                                     float* __restrict__ values) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int x, y, z;
  if (cells) {  // corner order (000,100,110,010,001,101,111,011)
    const int c = (int)(i & 7);
    cell_xyz(g, cells[i >> 3], x, y, z);
    x += ((c + 1) >> 1) & 1;
    y += (c >> 1) & 1;
    z += c >> 2;
  } else {
    const uint32_t t = (uint32_t)i, row = t / (uint32_t)g.nz;
    z = (int)(t - row * (uint32_t)g.nz);
    x = start + (int)(row / (uint32_t)g.ny);
    y = (int)(row % (uint32_t)g.ny);
  }
  float q[3], p[3];
  node_point(g, x, y, z, q);
  for (int r = 0; r < 3; ++r) p[r] = A.L[3 * r] * q[0] + A.L[3 * r + 1] * q[1] + A.L[3 * r + 2] * q[2] + A.t[r];
  const bool ok = isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2]) && tmin(tmin(p[0], p[1]), p[2]) >= 0.0f &&
                  tmax(tmax(p[0], p[1]), p[2]) <= 1.0f;
  float v = NAN;
  if (ok) {
    float res[4];
    field_at<float, WORDS, true>(f, coef, cum, depth, p, res);
    v = res[0];
  }
  values[i] = v - *iso;
}

// field.py:37-75 (evaluation_function): direct summation over all levels of a
// field without cumulative coefficients, as psr_field_detail::direct_levels
// with the cells' words.  Absent corners add +0 products, which change no bit.
template <class T>
__device__ __forceinline__ void direct_at(const FieldIndex& f, const T* __restrict__ coef, int depth, const T* p, T* res) {
  for (int d = 0; d <= depth; ++d) {
    const int n = 1 << d;
    Corners<T> c;
    c.flags = 0;
    int cell[3];
    T fr[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const T t = p[a] * T(n);
      cell[a] = clampi<T>((int)ceil(t) - 1, 0, n - 1);
      fr[a] = t - T(cell[a]);
    }
    const int w = word_of(cell[2]), bit = cell[2] - 31 * w;
    NodeWord word[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) word[k] = f.words[word_at(d, cell[0] + k / 2, cell[1] + k % 2, w)];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const unsigned present = (word[k].bits >> bit) & 3u;
      c.flags |= present << (2 * k) | present << (8 + 2 * k);
      c.first[k] = present ? word[k].first + __popc(word[k].bits & ((1u << bit) - 1u)) : 0;
    }
    T v[8];
    corner_values<false>(c, true, coef, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int o[3] = {k / 4, k / 2 % 2, k % 2};
      T h[3], sg[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        h[a] = o[a] ? fr[a] : T(1) - fr[a];
        sg[a] = o[a] ? T(1) : T(-1);
      }
      res[0] = res[0] + v[k] * h[0] * h[1] * h[2];
      const T cn = v[k] * T(n);
      res[1] = res[1] + cn * (sg[0] * h[1] * h[2]);
      res[2] = res[2] + cn * (h[0] * sg[1] * h[2]);
      res[3] = res[3] + cn * (h[0] * h[1] * sg[2]);
    }
  }
}

// A caller's field through its node words: the bits of psr_evaluate_field,
// whose searches it takes itself where *sorted is 0 (keys that are not
// strictly ascending, or off the grid, have no words).  100,003 queries at
// depth 8 in float64: 130 us by searches, 18 us by words.
template <class T>
__global__ void __launch_bounds__(256) k_level_field(PsrField field, FieldIndex f, const int* __restrict__ sorted,
                                                     const T* __restrict__ queries, int64_t m, T* __restrict__ values,
                                                     T* __restrict__ grads, int* __restrict__ valid) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const T q[3] = {queries[3 * i], queries[3 * i + 1], queries[3 * i + 2]};
  if (!*sorted) {
    T v, g[3];
    const int ok = psr_evaluate_field<T>(field, q, &v, grads ? g : nullptr);
    values[i] = v;
    if (grads) { grads[3 * i] = g[0]; grads[3 * i + 1] = g[1]; grads[3 * i + 2] = g[2]; }
    if (valid) valid[i] = ok;
    return;
  }
  T L[9], t[3], p[3];
  for (int k = 0; k < 9; ++k) L[k] = T(field.linear[k]);
  for (int k = 0; k < 3; ++k) t[k] = T(field.translation[k]);
  for (int r = 0; r < 3; ++r) p[r] = L[3 * r] * q[0] + L[3 * r + 1] * q[1] + L[3 * r + 2] * q[2] + t[r];
  const bool ok = isfinite(p[0]) && isfinite(p[1]) && isfinite(p[2]) && tmin(tmin(p[0], p[1]), p[2]) >= T(0) &&
                  tmax(tmax(p[0], p[1]), p[2]) <= T(1);
  if (valid) valid[i] = ok ? 1 : 0;
  T res[4] = {T(0), T(0), T(0), T(0)};
  if (!ok) {
    values[i] = T(NAN);
    if (grads) { grads[3 * i] = T(NAN); grads[3 * i + 1] = T(NAN); grads[3 * i + 2] = T(NAN); }
    return;
  }
  const T* coef = (const T*)field.coefficients;
  const T* cum = (const T*)field.cumulative;
  if (cum)
    field_at<T, true, false>(f, coef, cum, field.depth, p, res);
  else
    direct_at(f, coef, field.depth, p, res);
  values[i] = res[0];
  if (grads)
    for (int c = 0; c < 3; ++c) grads[3 * i + c] = L[c] * res[1] + L[3 + c] * res[2] + L[6 + c] * res[3];
}

// *sorted stays 1 if the keys ascend strictly and lie on their levels' grids
__global__ void k_keys_sorted(const int64_t* __restrict__ keys, int64_t n, int depth, int* __restrict__ sorted) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t k = keys[i];
  const int d = key_d(k), top = imax(imax(key_x(k), key_y(k)), key_z(k));
  if (k < 0 || d > depth || top > (1 << d) || (i > 0 && keys[i - 1] >= k)) *sorted = 0;
}

__global__ void k_clear_words(NodeWord* __restrict__ words, uint32_t n, int* __restrict__ sorted) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) words[i] = NodeWord{0u, 0};
  if (i == 0) *sorted = 1;
}

// k_field_words over keys that may be off the grid (sorted 0): nothing then
__global__ void k_level_field_words(const int64_t* __restrict__ keys, int64_t n, int depth, const int* __restrict__ sorted,
                                    NodeWord* __restrict__ words) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && *sorted) field_word(keys, n, depth, words, i);
}

// Isovalue: <=1024 aggregates one serial double chain (reconstruction.py:66-83);
// otherwise per-1024 partials: 256 lanes add elements lane+256k (k=0..3) in
// order, then a halving tree; partials combined the same way.
template <class T>
__global__ void __launch_bounds__(256) k_iso_partials(const T* __restrict__ v, const T* __restrict__ w, int64_t G,
                                                      double* __restrict__ tp, double* __restrict__ mp) {
  __shared__ double st[256], sm[256];
  double a = 0.0, m = 0.0;
  for (int k = 0; k < 4; ++k) {
    const int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x + 256 * k;
    if (i < G) { a += double(v[i] * w[i]); m += double(w[i]); }
  }
  st[threadIdx.x] = a;
  sm[threadIdx.x] = m;
  __syncthreads();
  for (int stride = 128; stride > 0; stride >>= 1) {
    if (threadIdx.x < stride) {
      st[threadIdx.x] = st[threadIdx.x] + st[threadIdx.x + stride];
      sm[threadIdx.x] = sm[threadIdx.x] + sm[threadIdx.x + stride];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) { tp[blockIdx.x] = st[0]; mp[blockIdx.x] = sm[0]; }
}

template <class T>
__global__ void __launch_bounds__(256) k_iso_finish(const double* __restrict__ tp, const double* __restrict__ mp, int64_t blocks,
                                                    T* __restrict__ out) {
  __shared__ double st[256], sm[256];
  double a = 0.0, m = 0.0;
  for (int64_t i = threadIdx.x; i < blocks; i += 256) { a += tp[i]; m += mp[i]; }
  st[threadIdx.x] = a;
  sm[threadIdx.x] = m;
  __syncthreads();
  for (int stride = 128; stride > 0; stride >>= 1) {
    if (threadIdx.x < stride) {
      st[threadIdx.x] = st[threadIdx.x] + st[threadIdx.x + stride];
      sm[threadIdx.x] = sm[threadIdx.x] + sm[threadIdx.x + stride];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = T(st[0] / sm[0]);
}

template <class T>
__global__ void k_iso_serial(const T* __restrict__ v, const T* __restrict__ w, int64_t G, T* __restrict__ out) {
  if (threadIdx.x != 0) return;
  double total = 0.0, weight = 0.0;
  for (int64_t i = 0; i < G; ++i) {
    total += double(v[i] * w[i]);
    weight += double(w[i]);
  }
  *out = T(total / weight);
}

}  // namespace

template <class T>
void isovalue_launch(const T* v, const T* w, int64_t G, double* tp, double* mp, T* out, hipStream_t s) {
  if (G <= 1024) {
    hipLaunchKernelGGL(k_iso_serial<T>, dim3(1), dim3(64), 0, s, v, w, G, out);
  } else {
    const int64_t blocks = isovalue_partials(G);
    hipLaunchKernelGGL(k_iso_partials<T>, dim3((unsigned)blocks), dim3(256), 0, s, v, w, G, tp, mp);
    KERNEL_CHECK();
    hipLaunchKernelGGL(k_iso_finish<T>, dim3(1), dim3(256), 0, s, (const double*)tp, (const double*)mp, blocks, out);
  }
  KERNEL_CHECK();
}

template <class T> void compute_isovalue(const T* v, const T* w, int64_t G, T* out, hipStream_t s) {
  const int64_t blocks = G > 1024 ? isovalue_partials(G) : 0;
  DArray<double> tp(blocks, s), mp(blocks, s);
  isovalue_launch(v, w, G, tp.data(), mp.data(), out, s);
}

// The isovalue reduction without allocation, for callers that cannot call
// hipMalloc (HIP graph capture, tight serving loops): the double partials
// live in a file-scope device array, shared by every call on a GPU (calls
// that overlap on one GPU race on it).  Every partial a call reads is written
// by the same call first, so nothing needs clearing.  `scratch` is a
// host-side stand-in for the array in host code; its device address is
// looked up once per device (with that device current) and only that
// address is passed to kernels.
constexpr int ISO_SCRATCH_MAX_DEVICES = 64;
static __device__ __align__(256) double scratch[2 * ISOVALUE_NOALLOC_PARTIALS];

static double* scratch_address(int dev) {
  static std::mutex mu;
  static double* addr[ISO_SCRATCH_MAX_DEVICES] = {};
  if (dev < 0 || dev >= ISO_SCRATCH_MAX_DEVICES) throw PsrError(1, "device index beyond the supported range");
  std::lock_guard<std::mutex> g(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      (void)hipGetLastError();
      throw PsrError(1, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
    }
    addr[dev] = (double*)p;
  }
  return addr[dev];
}

template <class T> void isovalue_noalloc(const T* v, const T* w, int64_t G, T* out, hipStream_t s) {
  if (G > ISOVALUE_NOALLOC_MAX)
    throw PsrError(2, "psr_isovalue_noalloc handles at most " + std::to_string(ISOVALUE_NOALLOC_MAX) +
                          " values (its partial sums live in a fixed device array)");
  int dev = 0;
  HIP_CHECK(hipGetDevice(&dev));
  double* tp = scratch_address(dev);
  isovalue_launch(v, w, G, tp, tp + ISOVALUE_NOALLOC_PARTIALS, out, s);
}

template void isovalue_noalloc<float>(const float*, const float*, int64_t, float*, hipStream_t);
template void isovalue_noalloc<double>(const double*, const double*, int64_t, double*, hipStream_t);
template void isovalue_launch<float>(const float*, const float*, int64_t, double*, double*, float*, hipStream_t);
template void isovalue_launch<double>(const double*, const double*, int64_t, double*, double*, double*, hipStream_t);
template void compute_isovalue<float>(const float*, const float*, int64_t, float*, hipStream_t);
template void compute_isovalue<double>(const double*, const double*, int64_t, double*, hipStream_t);

// transforms.py:13-52 (cofactor inverse in the input precision)
template <class T> static T det3(const T m[3][3]) {
  return m[0][0] * (m[1][1] * m[2][2] - m[1][2] * m[2][1]) - m[0][1] * (m[1][0] * m[2][2] - m[1][2] * m[2][0]) +
         m[0][2] * (m[1][0] * m[2][1] - m[1][1] * m[2][0]);
}
template <class T> static T minor4(const T* m, int row, int col) {
  T out[3][3];
  int rr = 0;
  for (int r = 0; r < 4; ++r) {
    if (r == row) continue;
    int cc = 0;
    for (int c = 0; c < 4; ++c) {
      if (c == col) continue;
      out[rr][cc++] = m[r * 4 + c];
    }
    rr++;
  }
  return det3(out);
}
template <class T> void reference_inverse(const T* m, T* out) {
  T det = T(0);
  for (int c = 0; c < 4; ++c) {
    if (c % 2 == 0) det = det + m[c] * minor4(m, 0, c);
    else det = det - m[c] * minor4(m, 0, c);
  }
  for (int r = 0; r < 4; ++r)
    for (int c = 0; c < 4; ++c) {
      T value = minor4(m, r, c);
      if ((r + c) % 2 != 0) value = -value;
      out[c * 4 + r] = value / det;
    }
}


template <class T>
static void launch_evaluate(const Result<T>& r, const T* queries, int64_t m, const Affine<T>& A, int point_div_mode,
                            const T* divisors, T* values, T* grads, int* valid, hipStream_t s) {
  if (m <= 0) return;
  const int depth = r.prm.depth;
  auto kernel = r.word_depth >= depth ? k_evaluate<T, true> : k_evaluate<T, false>;
  hipLaunchKernelGGL(kernel, dim3(blocks_for(m, 256)), dim3(256), 0, s, field_index(r), (const T*)r.coefficients.data(),
                     (const T*)r.cumulative.data(), depth, queries, m, A, point_div_mode, divisors, values, grads, valid);
  KERNEL_CHECK();
}

void mesh_values(const Result<float>& r, const MeshGrid& g, int start, const int* cells, int64_t n, const float* iso, float* values,
                 hipStream_t s) {
  if (n <= 0) return;
  Affine<float> A;
  for (int i = 0; i < 3; ++i) {
    for (int j = 0; j < 3; ++j) A.L[3 * i + j] = r.model_to_cube[4 * i + j];
    A.t[i] = r.model_to_cube[4 * i + 3];
  }
  auto kernel = r.word_depth >= r.prm.depth ? k_mesh_values<true> : k_mesh_values<false>;
  hipLaunchKernelGGL(kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, field_index(r), (const float*)r.coefficients.data(),
                     (const float*)r.cumulative.data(), r.prm.depth, A, g, start, cells, n, iso, values);
  KERNEL_CHECK();
}

template <class T>
void evaluate_field(const Result<T>& r, const T* queries, int64_t m, const T* linear, const T* translation, T* values, T* grads,
                    int* valid, hipStream_t s) {
  if (m <= 0) return;
  Affine<T> A;
  for (int k = 0; k < 9; ++k) A.L[k] = linear[k];
  for (int k = 0; k < 3; ++k) A.t[k] = translation[k];
  launch_evaluate(r, queries, m, A, 0, (const T*)nullptr, values, grads, valid, s);
}

// Deepest level with node words: the lookup-table limits' dense one (depth 9
// by default; word_base is defined up to there), at most the field's depth.
int node_word_depth(int depth) {
  const int64_t cells = dense_index_max_cells();
  int d = -1;
  for (int e = 0; e <= imin(depth, 9); ++e) {
    const int64_t dim = ((int64_t)1 << e) + 1;
    if (dim * dim * dim > cells) break;
    d = e;
  }
  return d;
}

int64_t level_field_words(int64_t count, int depth) {
  return count <= INT32_MAX && depth >= 0 && node_word_depth(depth) == depth ? (int64_t)word_base(depth + 1) : 0;
}

void build_level_field_words(const int64_t* keys, int64_t count, int depth, NodeWord* words, int* sorted, hipStream_t s) {
  const uint32_t n = word_base(depth + 1);
  hipLaunchKernelGGL(k_clear_words, dim3(blocks_for(n, 256)), dim3(256), 0, s, words, n, sorted);
  KERNEL_CHECK();
  if (!count) return;
  hipLaunchKernelGGL(k_keys_sorted, dim3(blocks_for(count, 256)), dim3(256), 0, s, keys, count, depth, sorted);
  KERNEL_CHECK();
  hipLaunchKernelGGL(k_level_field_words, dim3(blocks_for(count, 256)), dim3(256), 0, s, keys, count, depth, (const int*)sorted,
                     words);
  KERNEL_CHECK();
}

template <class T>
void evaluate_level_field(const PsrField& field, const NodeWord* words, const int* sorted, const T* queries, int64_t m, T* values,
                          T* grads, int* valid, hipStream_t s) {
  FieldIndex f{};
  f.keys = field.keys;
  f.off = field.level_offsets;
  f.words = words;
  f.word_depth = field.depth;
  hipLaunchKernelGGL(k_level_field<T>, dim3(blocks_for(m, 256)), dim3(256), 0, s, field, f, sorted, queries, m, values, grads, valid);
  KERNEL_CHECK();
}
template void evaluate_level_field<float>(const PsrField&, const NodeWord*, const int*, const float*, int64_t, float*, float*, int*,
                                          hipStream_t);
template void evaluate_level_field<double>(const PsrField&, const NodeWord*, const int*, const double*, int64_t, double*, double*,
                                           int*, hipStream_t);

void build_node_words(const int64_t* keys, int64_t n, int word_depth, DArray<NodeWord>& words, hipStream_t s) {
  if (word_depth < 0) return words.free();
  words.reset(word_base(word_depth + 1), s);
  words.zero();
  if (!n) return;
  hipLaunchKernelGGL(k_field_words, dim3(blocks_for(n, 256)), dim3(256), 0, s, keys, n, word_depth, words.data());
  KERNEL_CHECK();
}

template <class T> void index_field(Result<T>& r) {
  hipStream_t s = r.s;
  const int D = r.prm.depth;
  const LevelBlocks lb = level_blocks(r);
  r.level_offsets.assign(lb.first, lb.first + D + 2);
  const int64_t K = r.level_offsets[D + 1];
  r.keys.reset(K, s);
  r.offsets_dev.reset(D + 2, s);
  LevelArrays<int64_t> in;
  for (int d = 0; d <= D; ++d) in.a[d] = r.levels[d].basis_keys.data();
  hipLaunchKernelGGL(k_concat_keys, dim3((unsigned)imax(lb.blocks(), 1)), dim3(LEVEL_BLOCK), 0, s, lb, in, r.keys.data(),
                     r.offsets_dev.data());
  KERNEL_CHECK();
  r.word_depth = K ? node_word_depth(D) : -1;
  build_node_words(r.keys.data(), K, r.word_depth, r.node_words, s);
}

template <class T> void stage_field(Result<T>& r) {
  hipStream_t s = r.s;
  const int D = r.prm.depth;
  r.join_average();
  read_bytes(r.normal_average_host, r.normal_average.data(), sizeof(T) * 3, s);
  r.average_contrib.free();
  const int64_t K = r.level_offsets[D + 1];
  r.coefficients.reset(K + 1, s);  // one value more: corner_values loads pairs
  r.coefficients.shrink(K);
  const LevelBlocks lb = level_blocks(r);
  if (K) {
    LevelArrays<T> in;
    for (int d = 0; d <= D; ++d) in.a[d] = r.levels[d].correction.data();
    hipLaunchKernelGGL(k_concat_values<T>, dim3((unsigned)lb.blocks()), dim3(LEVEL_BLOCK), 0, s, lb, in, r.coefficients.data());
    KERNEL_CHECK();
  }
  // node words are there for the levels within the dense limit (index_field):
  // column tables where deeper levels remain, else searches of the keys
  const bool tables = D <= field_table_max_depth() && K;
  if (tables && r.word_depth < D) {
    const size_t cells = (size_t)column_base(D + 1);
    r.column_start.reset(cells, s);
    r.column_end.reset(cells, s);
    r.column_start.zero();
    r.column_end.zero();
    hipLaunchKernelGGL(k_field_columns, dim3(blocks_for(K, 256)), dim3(256), 0, s, (const int64_t*)r.keys.data(), K,
                       r.column_start.data(), r.column_end.data());
    KERNEL_CHECK();
  } else {
    r.column_start.free();
    r.column_end.free();
  }
  const FieldIndex f = field_index(r);
  r.cumulative.reset(K + 1, s);
  r.cumulative.shrink(K);
  if (K) HIP_CHECK(hipMemcpyAsync(r.cumulative.data(), r.coefficients.data(), sizeof(T) * K, hipMemcpyDeviceToDevice, s));
  for (int d = 1; d <= D; ++d) {
    const int cnt = r.levels[d].basis_count;
    if (!cnt) continue;
    hipLaunchKernelGGL(k_cumulative<T>, dim3(blocks_for(cnt, 256)), dim3(256), 0, s, f, d, (const T*)r.coefficients.data(),
                       r.cumulative.data());
    KERNEL_CHECK();
  }
  // centroid values with the cube-space field (reconstruction.py:295-303)
  const int G = r.G;
  r.centroid_values.reset(G, s);
  Affine<T> I;
  for (int k = 0; k < 9; ++k) I.L[k] = (k % 4 == 0) ? T(1) : T(0);
  for (int k = 0; k < 3; ++k) I.t[k] = T(0);
  launch_evaluate(r, (const T*)r.position_sums.data(), (int64_t)G, I, 1, (const T*)r.weights.data(), r.centroid_values.data(),
                  (T*)nullptr, (int*)nullptr, s);
  DArray<T> iso(1, s);
  compute_isovalue((const T*)r.centroid_values.data(), (const T*)r.weights.data(), (int64_t)G, iso.data(), s);
  read_bytes(&r.iso, iso.data(), sizeof(T), s);
  // transforms.py:54-79 (host scalar work)
  const T sc = r.transform[0];
  const T M[16] = {T(0), sc, T(0), r.transform[1], T(0), T(0), sc, r.transform[2],
                   sc, T(0), T(0), r.transform[3], T(0), T(0), T(0), T(1)};
  reference_inverse(M, r.cube_to_model);
  reference_inverse(r.cube_to_model, r.model_to_cube);
}

template void index_field<float>(Result<float>&);
template void index_field<double>(Result<double>&);
template void stage_field<float>(Result<float>&);
template void stage_field<double>(Result<double>&);
template void evaluate_field<float>(const Result<float>&, const float*, int64_t, const float*, const float*, float*, float*, int*,
                                    hipStream_t);
template void evaluate_field<double>(const Result<double>&, const double*, int64_t, const double*, const double*, double*,
                                     double*, int*, hipStream_t);
template void reference_inverse<float>(const float*, float*);
template void reference_inverse<double>(const double*, double*);

}  // namespace psr
