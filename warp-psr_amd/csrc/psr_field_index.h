// Lookup structure of a concatenated multi-level field (all levels' sorted
// basis keys with per-level offsets, node words and optional (x, y) column
// tables), shared by the field stage and its adjoint.
#pragma once
#include "psr_result.h"

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

// Words of one (x, y) column of level d: 32 nodes each, 2^d + 1 nodes.
PSR_HD int word_columns(int d) { return d < 5 ? 1 : (1 << (d - 5)) + 1; }
// first word of level d: sum over e < d of (2^e + 1)^2 * word_columns(e), d <= 9
PSR_HD uint32_t word_base(int d) {
  const uint32_t p2 = 1u << d, p4 = p2 * p2, p8 = p4 * p2;
  if (d <= 5) return (p4 - 1) / 3 + 2 * (p2 - 1) + d;  // one word a column
  // (2^e + 1)^2 (2^e / 32 + 1) = 8^e / 32 + 17 4^e / 16 + 65 2^e / 32 + 1 summed from e = 5, after 408 words
  return 408u + (p8 - 32768u) / 224u + 17u * (p4 - 1024u) / 48u + 65u * (p2 - 32u) / 32u + (uint32_t)(d - 5);
}

// first cell of level d's column table: sum over e < d of (2^e + 1)^2
PSR_HD int64_t column_base(int d) { return (((int64_t)1 << (2 * d)) - 1) / 3 + 2 * (((int64_t)1 << d) - 1) + d; }

// index of node z in its column's word z >> 5, or -1
__device__ __forceinline__ int node_in_word(NodeWord w, int z) {
  const uint32_t bit = 1u << (z & 31);
  return (w.bits & bit) ? w.first + __popc(w.bits & (bit - 1)) : -1;
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
    const NodeWord* column = f.words + word_base(d) + (uint32_t)(x * dim + y) * (uint32_t)word_columns(d);
    NodeWord w = column[z0 >> 5];
#pragma unroll
    for (int k = 0; k < MAXLEN; ++k) {
      const int z = z0 + k;
      if (k >= len || z >= dim) break;
      if (k && (z & 31) == 0) w = column[z >> 5];
      out[k] = node_in_word(w, z);
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

// model -> cube affine map of queries
template <class T> struct Affine { T L[9]; T t[3]; };

}  // namespace psr
