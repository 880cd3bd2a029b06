// Lookup structure of a concatenated multi-level field (all levels' sorted
// basis keys with per-level offsets, node words and optional (x, y) column
// tables), shared by the field stage and its adjoint.
#pragma once
#include "psr_result.h"
#include "../../include/warp_psr_amd.h"

namespace psr {

// keys of level d occupy [off[d], off[d+1]) of the concatenated sorted keys.
// Levels 0..word_depth have node words (see NodeWord); start/end (optional)
// are the column runs of every level.
struct FieldIndex {
  const int64_t* keys;
  const int* off;  // device, depth+2 entries
  const int* start;
  const int* end;
  const NodeWord* words;
  int word_depth;  // -1: no words
};

// Words of one (x, y) column of level d: word w holds nodes 31 w .. 31 w + 31
// of the column's 2^d + 1, the last one shared with the next word, so the two
// z nodes of a cell always lie in one word.  The words of 4 x 4 columns at one
// w are one 128-byte line, so the four columns of a cell take 1.6 lines on
// average where a column's words in a row took four (812,000 queries at depth
// 9 in float64: 195 -> 151 us; the lines a query misses bound it).
PSR_HD int word_columns(int d) { return d < 5 ? 1 : (1 << (d - 5)) + 1; }  // ceil(2^d / 31), d <= 9
PSR_HD int word_of(int z) { return (int)(((uint32_t)z * 67651u) >> 21); }  // z / 31 for z < 2^15
PSR_HD int word_blocks(int d) { return d < 2 ? 1 : (1 << (d - 2)) + 1; }   // 4-column blocks an axis
// first word of level d, d <= 10: sum over e < d of 16 word_blocks(e)^2 word_columns(e)
// = 16 each for e < 2, (2^e + 4)^2 from there, times 2^e / 32 + 1 from e = 5
PSR_HD uint32_t word_base(int d) {
  const uint32_t p2 = 1u << d, p4 = p2 * p2, p8 = p4 * p2;
  const uint32_t small = 32u + (p4 - 16u) / 3u + 8u * (p2 - 4u) + 16u * ((uint32_t)d - 2u);
  const uint32_t large = 640u + (p8 - 32768u) / 224u + 5u * (p4 - 1024u) / 12u + 17u * (p2 - 32u) / 2u + 16u * ((uint32_t)d - 5u);
  return d < 2 ? 16u * (uint32_t)d : d < 5 ? small : large;
}
PSR_HD uint32_t word_at(int d, int x, int y, int w) {
  const uint32_t nb = (uint32_t)word_blocks(d);
  return word_base(d) + ((((uint32_t)w * nb + (uint32_t)(x >> 2)) * nb + (uint32_t)(y >> 2)) << 4) + (uint32_t)((x & 3) << 2 | (y & 3));
}

// first cell of level d's column table: sum over e < d of (2^e + 1)^2
PSR_HD int64_t column_base(int d) { return (((int64_t)1 << (2 * d)) - 1) / 3 + 2 * (((int64_t)1 << d) - 1) + d; }

// index of the node at `bit` of a word (z - 31 word), or -1
__device__ __forceinline__ int node_in_word(NodeWord w, int bit) {
  const uint32_t m = 1u << bit;
  return (w.bits & m) ? w.first + __popc(w.bits & (m - 1)) : -1;
}

// Absolute indices of keys (d, x, y, z0 + k), k < len (-1 when absent).
template <int MAXLEN>
__device__ __forceinline__ void level_run(const FieldIndex& f, int d, int x, int y, int z0, int len, int64_t* out) {
  if (d <= f.word_depth) {
#pragma unroll
    for (int k = 0; k < MAXLEN; ++k)
      if (k < len) out[k] = -1;
    const int dim = (1 << d) + 1;
    if (x < 0 || y < 0 || x >= dim || y >= dim || z0 < 0 || z0 >= dim) return;
    // node 2^d is the last word's shared one
    int at = imin(word_of(z0), word_columns(d) - 1);
    NodeWord w = f.words[word_at(d, x, y, at)];
#pragma unroll
    for (int k = 0; k < MAXLEN; ++k) {
      const int z = z0 + k;
      if (k >= len || z >= dim) break;
      if (z - 31 * at > 31) w = f.words[word_at(d, x, y, ++at)];
      out[k] = node_in_word(w, z - 31 * at);
    }
    return;
  }
  if (f.start) {
    ColumnTable t;
    t.start = f.start + column_base(d);
    t.end = f.end + column_base(d);
    t.dim = (1 << d) + 1;
    find_run_table<MAXLEN>(f.keys, 0, t, d, x, y, z0, len, out);
    return;
  }
  const int64_t lo = f.off[d];
  find_run<MAXLEN>(f.keys + lo, (int64_t)f.off[d + 1] - lo, d, x, y, z0, len, out);
#pragma unroll
  for (int k = 0; k < MAXLEN; ++k)
    if (k < len && out[k] >= 0) out[k] += lo;
}

// Nodes z0 .. z0 + LEN - 1 (LEN <= 6) of one column: mask has bit k for a
// present node z0 + k, base is the index of the lowest present one.  A column's
// nodes are consecutive in the keys, so node z0 + k has index
// base + popcount(mask below k).
struct NodeSpan {
  int base;
  unsigned mask;
  __device__ __forceinline__ int at(int k) const { return (mask >> k) & 1u ? base + __popc(mask & ((1u << k) - 1u)) : -1; }
};

// x, y and z0 in [0, 2^d]
template <int LEN> __device__ __forceinline__ NodeSpan node_span(const NodeWord* __restrict__ words, int d, int x, int y, int z0) {
  const int wc = word_columns(d), at = imin(word_of(z0), wc - 1), b = z0 - 31 * at;
  const NodeWord w = words[word_at(d, x, y, at)];
  unsigned bits = w.bits >> b;
  int base = w.first + __popc(w.bits & ((1u << b) - 1u));
  if (b + LEN > 32 && at + 1 < wc) {
    const NodeWord v = words[word_at(d, x, y, at + 1)];
    if (!bits) base = v.first;  // the shared node is absent, so v's first node is the next one
    bits |= v.bits << (31 - b);
  }
  return NodeSpan{base, bits & ((1u << LEN) - 1u)};
}

// One level's sorted keys with their lookup: node words (whose indices count
// from `first` keys earlier), else an (x, y) column table, else searches.
struct NodeIndex {
  const int64_t* keys = nullptr;
  int64_t count = 0;
  ColumnTable columns;
  const NodeWord* words = nullptr;
  int first = 0;
};

// Indices within the level of keys (d, x, y, z0 + k), k < LEN; x, y in any
// range, z0 in [0, 2^d].
template <int LEN> __device__ __forceinline__ NodeSpan find_span(const NodeIndex& f, int d, int x, int y, int z0) {
  const int n = 1 << d;
  const bool in = x >= 0 && y >= 0 && x <= n && y <= n;
  if (f.words) {
    // a load at a clamped address, so that several columns' loads go out together
    NodeSpan s = node_span<LEN>(f.words, d, imin(imax(x, 0), n), imin(imax(y, 0), n), z0);
    s.base -= f.first;
    if (!in) s.mask = 0;
    return s;
  }
  NodeSpan s{0, 0u};
  if (!in) return s;
  int64_t found[LEN];
  find_run_table<LEN>(f.keys, f.count, f.columns, d, x, y, z0, LEN, found);
#pragma unroll
  for (int k = LEN - 1; k >= 0; --k)
    if (found[k] >= 0) {
      s.base = (int)found[k];
      s.mask |= 1u << k;
    }
  return s;
}

// Deepest level with node words of keys up to `depth`: the lookup-table limits'
// dense one (depth 9 by default), -1 for none.
int node_word_depth(int depth);
// Node words of levels 0..word_depth of n concatenated sorted keys.
void build_node_words(const int64_t* keys, int64_t n, int word_depth, DArray<NodeWord>& words, hipStream_t s);

// Block-aligned ranges of the levels' rows: every block of a launch over all
// levels' rows belongs to one level, found from its index alone.
constexpr int MAX_LEVELS = 16;  // keys hold 16 bits an axis
constexpr int LEVEL_BLOCK = 256;
struct LevelBlocks {
  int levels = 0;
  int block[MAX_LEVELS + 1];  // first block of each level
  int rows[MAX_LEVELS], first[MAX_LEVELS + 1];
  // level of a block, and its thread's row (-1 beyond the level's rows)
  __device__ __forceinline__ int level_of(int b) const {
    int d = 0;
    while (d + 1 < levels && b >= block[d + 1]) ++d;
    return d;
  }
  __device__ __forceinline__ int row_of(int b, int d, int tid) const {
    const int i = (b - block[d]) * LEVEL_BLOCK + tid;
    return i < rows[d] ? i : -1;
  }
  int blocks() const { return block[levels]; }
};
template <class T> inline LevelBlocks level_blocks(const Result<T>& r) {
  LevelBlocks lb;
  lb.levels = r.prm.depth + 1;
  if (lb.levels > MAX_LEVELS) throw PsrError(1, "too many levels");
  lb.block[0] = lb.first[0] = 0;
  for (int d = 0; d < lb.levels; ++d) {
    lb.rows[d] = r.levels[d].basis_count;
    lb.block[d + 1] = lb.block[d] + (lb.rows[d] + LEVEL_BLOCK - 1) / LEVEL_BLOCK;
    lb.first[d + 1] = lb.first[d] + lb.rows[d];
  }
  return lb;
}

template <class T> inline FieldIndex field_index(const Result<T>& r) {
  FieldIndex f;
  f.words = r.node_words.data();
  f.word_depth = r.word_depth;
  f.keys = r.keys.data();
  f.off = r.offsets_dev.data();
  f.start = r.column_start.empty() ? nullptr : r.column_start.data();
  f.end = r.column_start.empty() ? nullptr : r.column_end.data();
  return f;
}

// A caller's field (LevelField): the number of node words of its levels, 0 if
// it takes none (levels beyond the dense limit), their construction
// (*sorted = 0 for keys that have none) and the evaluation through them.
int64_t level_field_words(int64_t count, int depth);
void build_level_field_words(const int64_t* keys, int64_t count, int depth, NodeWord* words, int* sorted, hipStream_t s);
template <class T>
void evaluate_level_field(const PsrField& field, const NodeWord* words, const int* sorted, const T* queries, int64_t m, T* values,
                          T* grads, int* valid, hipStream_t s);

// model -> cube affine map of queries
template <class T> struct Affine { T L[9]; T t[3]; };

}  // namespace psr
