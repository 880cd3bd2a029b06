// Stages 1-3: sample normalisation and grouping (src/warp_psr/samples.py),
// density and splat depth (src/warp_psr/density.py) and the normal-field
// splat (src/warp_psr/normals.py).
//
// Every keyed reduction is "stable sort by key, then one lane sums its run
// serially" so sums keep the reference order.  Splat records are sorted as
// (packed key, record id) pairs only; the reducing lane recomputes each
// record's value from its id instead of storing and re-reading it.
#include "psr_bitmap.h"
#include "psr_splat.h"

#include <cmath>

namespace psr {

// ------------------------------------------------------------------ samples
template <class T>
__global__ void k_bounds_partial(const T* __restrict__ pts, int64_t n, T* __restrict__ partial, int* __restrict__ bad) {
  __shared__ T sm[6][256];
  __shared__ int sb[256];
  T lo[3], hi[3];
  for (int a = 0; a < 3; ++a) { lo[a] = T(INFINITY); hi[a] = -T(INFINITY); }
  int invalid = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    T p0 = pts[3 * i], p1 = pts[3 * i + 1], p2 = pts[3 * i + 2];
    if (isfinite(p0) && isfinite(p1) && isfinite(p2)) {
      lo[0] = tmin(lo[0], p0); hi[0] = tmax(hi[0], p0);
      lo[1] = tmin(lo[1], p1); hi[1] = tmax(hi[1], p1);
      lo[2] = tmin(lo[2], p2); hi[2] = tmax(hi[2], p2);
    } else {
      invalid++;
    }
  }
  for (int a = 0; a < 3; ++a) { sm[a][threadIdx.x] = lo[a]; sm[a + 3][threadIdx.x] = hi[a]; }
  sb[threadIdx.x] = invalid;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (threadIdx.x < st) {
      for (int a = 0; a < 3; ++a) {
        sm[a][threadIdx.x] = tmin(sm[a][threadIdx.x], sm[a][threadIdx.x + st]);
        sm[a + 3][threadIdx.x] = tmax(sm[a + 3][threadIdx.x], sm[a + 3][threadIdx.x + st]);
      }
      sb[threadIdx.x] += sb[threadIdx.x + st];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    for (int a = 0; a < 6; ++a) partial[blockIdx.x * 6 + a] = sm[a][0];
    bad[blockIdx.x] = sb[0];
  }
}

// One workgroup folds the per-block partials (min/max of finite values are
// order-independent).
template <class T>
__global__ void __launch_bounds__(256) k_bounds_final(const T* __restrict__ partial, const int* __restrict__ bad, int blocks,
                                                      T* __restrict__ out, int* __restrict__ out_bad) {
  __shared__ T sm[6][256];
  __shared__ int sb[256];
  T b[6];
  for (int a = 0; a < 3; ++a) { b[a] = T(INFINITY); b[a + 3] = -T(INFINITY); }
  int invalid = 0;
  for (int k = threadIdx.x; k < blocks; k += 256) {
    for (int a = 0; a < 3; ++a) {
      b[a] = tmin(b[a], partial[k * 6 + a]);
      b[a + 3] = tmax(b[a + 3], partial[k * 6 + a + 3]);
    }
    invalid += bad[k];
  }
  for (int a = 0; a < 6; ++a) sm[a][threadIdx.x] = b[a];
  sb[threadIdx.x] = invalid;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) {
      for (int a = 0; a < 3; ++a) {
        sm[a][threadIdx.x] = tmin(sm[a][threadIdx.x], sm[a][threadIdx.x + st]);
        sm[a + 3][threadIdx.x] = tmax(sm[a + 3][threadIdx.x], sm[a + 3][threadIdx.x + st]);
      }
      sb[threadIdx.x] += sb[threadIdx.x + st];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    for (int a = 0; a < 6; ++a) out[a] = sm[a][0];
    *out_bad = sb[0];
  }
}

template <class T> struct Xform { T t[5]; };

// samples.py:90-134 (_classify); packed leaf key x<<2D | y<<D | z, sentinel 1<<3D
template <class T>
__global__ void k_classify(const T* __restrict__ pts, const T* __restrict__ nrm, int64_t n, Xform<T> tf, int depth,
                           T* __restrict__ q, T* __restrict__ unit, uint64_t* __restrict__ keys, int* __restrict__ order,
                           int* __restrict__ status) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const T* t = tf.t;
  const T inv = t[0];
  T P0 = pts[3 * i], P1 = pts[3 * i + 1], P2 = pts[3 * i + 2];
  T N0 = nrm[3 * i], N1 = nrm[3 * i + 1], N2 = nrm[3 * i + 2];
  T p0 = P1 * inv + t[1], p1 = P2 * inv + t[2], p2 = P0 * inv + t[3];
  T n0 = N1 * t[4], n1 = N2 * t[4], n2 = N0 * t[4];
  T length2 = n0 * n0 + n1 * n1 + n2 * n2;
  q[3 * i] = p0; q[3 * i + 1] = p1; q[3 * i + 2] = p2;
  order[i] = (int)i;
  uint64_t key = (uint64_t)1 << (3 * depth);
  T u0 = T(0), u1 = T(0), u2 = T(0);
  int st = 1;
  const bool ok = length2 > T(0) && isfinite(length2);
  if (ok) st = 2;
  T pmin = wmin(wmin(p0, p1), p2), pmax = wmax(wmax(p0, p1), p2);
  if (ok && pmin >= T(0) && pmax <= T(1)) {
    st = 0;
    T l = sqrt(length2);
    u0 = n0 / l; u1 = n1 / l; u2 = n2 / l;
    const int res = 1 << depth;
    int x = cell_index(p0, res), y = cell_index(p1, res), z = cell_index(p2, res);
    key = ((uint64_t)x << (2 * depth)) | ((uint64_t)y << depth) | (uint64_t)z;
  }
  unit[3 * i] = u0; unit[3 * i + 1] = u1; unit[3 * i + 2] = u2;
  keys[i] = key;
  status[i] = st;
}

// samples.py:149-188 (_groups): serial sums over each run of equal leaf keys.
// A run is [head_pos[g], end): the next head, or for the last group the end
// of its equal keys.
__device__ __forceinline__ int64_t group_end(const uint64_t* __restrict__ keys, const int* __restrict__ head_pos, int g, int G,
                                             int64_t n) {
  if (g + 1 < G) return head_pos[g + 1];
  const uint64_t key = keys[head_pos[g]];
  int64_t lo = head_pos[g], hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (keys[mid] <= key) lo = mid + 1; else hi = mid;
  }
  return lo;
}

template <class T>
__device__ __forceinline__ void group_fields(const uint64_t key, int g, int G, int64_t i, int64_t end, int depth, const int* order,
                                             int64_t* unique, int* first, int* goff) {
  const uint64_t mask = ((uint64_t)1 << depth) - 1;
  unique[g] = basis_key(depth, (int)(key >> (2 * depth)), (int)((key >> depth) & mask), (int)(key & mask));
  first[g] = order[i];
  goff[g] = (int)i;
  if (g == G - 1) goff[G] = (int)end;
}

constexpr int GROUP_SERIAL_MAX = 16;  // longer runs are summed by a wave (k_groups_wide)

template <class T>
__global__ void k_groups(const uint64_t* __restrict__ keys, const int* __restrict__ order, const int* __restrict__ head_pos,
                         int G, int64_t n, int depth, const T* __restrict__ q, const T* __restrict__ unit,
                         int64_t* __restrict__ unique, T* __restrict__ sums, T* __restrict__ nsums, T* __restrict__ weights,
                         int* __restrict__ first, int* __restrict__ goff, int* __restrict__ group_of, int* __restrict__ wide,
                         int* __restrict__ wide_count) {
  int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= G) return;
  const int64_t i = head_pos[g];
  const int64_t end = group_end(keys, head_pos, g, G, n);
  if (end - i > GROUP_SERIAL_MAX) {
    wide[atomicAdd(wide_count, 1)] = g;
    return;
  }
  T p0 = T(0), p1 = T(0), p2 = T(0), s0 = T(0), s1 = T(0), s2 = T(0), w = T(0);
  for (int64_t j = i; j < end; ++j) {
    const int o = order[j];
    p0 = p0 + q[3 * o]; p1 = p1 + q[3 * o + 1]; p2 = p2 + q[3 * o + 2];
    s0 = s0 + unit[3 * o]; s1 = s1 + unit[3 * o + 1]; s2 = s2 + unit[3 * o + 2];
    w = w + T(1);
    group_of[o] = g;
  }
  group_fields<T>(keys[i], g, G, i, end, depth, order, unique, first, goff);
  sums[3 * g] = p0; sums[3 * g + 1] = p1; sums[3 * g + 2] = p2;
  nsums[3 * g] = s0; nsums[3 * g + 1] = s1; nsums[3 * g + 2] = s2;
  weights[g] = w;
}

// Long runs, one wave each: the lanes load 64 members at a time and every
// lane adds them in run order through lane broadcasts, so the sums equal the
// serial ones bit for bit.
template <class T>
__global__ void __launch_bounds__(64) k_groups_wide(const uint64_t* __restrict__ keys, const int* __restrict__ order,
                                                    const int* __restrict__ head_pos, int G, int64_t n, int depth,
                                                    const T* __restrict__ q, const T* __restrict__ unit,
                                                    int64_t* __restrict__ unique, T* __restrict__ sums, T* __restrict__ nsums,
                                                    T* __restrict__ weights, int* __restrict__ first, int* __restrict__ goff,
                                                    int* __restrict__ group_of, const int* __restrict__ wide,
                                                    const int* __restrict__ wide_count) {
  const int lane = threadIdx.x;
  const int count = *wide_count;
  for (int k = blockIdx.x; k < count; k += gridDim.x) {
    const int g = wide[k];
    const int64_t i = head_pos[g];
    const int64_t end = group_end(keys, head_pos, g, G, n);
    T p0 = T(0), p1 = T(0), p2 = T(0), s0 = T(0), s1 = T(0), s2 = T(0), w = T(0);
    for (int64_t base = i; base < end; base += 64) {
      const int64_t j = base + lane;
      T v[6] = {T(0), T(0), T(0), T(0), T(0), T(0)};
      if (j < end) {
        const int o = order[j];
        v[0] = q[3 * o]; v[1] = q[3 * o + 1]; v[2] = q[3 * o + 2];
        v[3] = unit[3 * o]; v[4] = unit[3 * o + 1]; v[5] = unit[3 * o + 2];
        group_of[o] = g;
      }
      const int m = (int)(end - base < 64 ? end - base : 64);
      for (int t = 0; t < m; ++t) {
        p0 = p0 + __shfl(v[0], t, 64); p1 = p1 + __shfl(v[1], t, 64); p2 = p2 + __shfl(v[2], t, 64);
        s0 = s0 + __shfl(v[3], t, 64); s1 = s1 + __shfl(v[4], t, 64); s2 = s2 + __shfl(v[5], t, 64);
        w = w + T(1);
      }
    }
    if (lane == 0) {
      group_fields<T>(keys[i], g, G, i, end, depth, order, unique, first, goff);
      sums[3 * g] = p0; sums[3 * g + 1] = p1; sums[3 * g + 2] = p2;
      nsums[3 * g] = s0; nsums[3 * g + 1] = s1; nsums[3 * g + 2] = s2;
      weights[g] = w;
    }
  }
}

__global__ void k_fill_i32(int* p, int64_t n, int v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

template <class T> void stage_samples(Result<T>& r, const T* pts, const T* nrm) {
  hipStream_t s = r.s;
  const int64_t n = r.n;
  const int depth = r.prm.depth;
  // bounds over finite points (samples.py:34-52)
  const int blocks = (int)std::min<int64_t>(512, std::max<int64_t>(1, (n + 255) / 256));
  DArray<T> partial(6 * blocks, s), bounds(6, s);
  DArray<int> bad(blocks, s), bad_total(1, s);
  hipLaunchKernelGGL(k_bounds_partial<T>, dim3(blocks), dim3(256), 0, s, pts, n, partial.data(), bad.data());
  KERNEL_CHECK();
  hipLaunchKernelGGL(k_bounds_final<T>, dim3(1), dim3(256), 0, s, (const T*)partial.data(), (const int*)bad.data(), blocks,
                     bounds.data(), bad_total.data());
  KERNEL_CHECK();
  struct { T b[6]; int bad; } host;
  read_bytes(host.b, bounds.data(), sizeof(host.b), s);
  read_bytes(&host.bad, bad_total.data(), sizeof(int), s);
  for (int a = 0; a < 6; ++a) r.bounds[a] = host.b[a];
  if (host.bad || compute_transform(r.bounds, r.prm.scale, r.transform))
    throw PsrError(2, "Nonfinite positions or degenerate/overflowing bounding cube");
  Xform<T> tf;
  for (int a = 0; a < 5; ++a) tf.t[a] = r.transform[a];
  // classify + stable sort by leaf key (samples.py:90-134, 269)
  r.q.reset(3 * n, s);
  r.unit_normals.reset(3 * n, s);
  r.input_status.reset(n, s);
  DArray<uint64_t> keys(n, s);
  DArray<int> order(n, s);
  hipLaunchKernelGGL(k_classify<T>, dim3(blocks_for(n, 256)), dim3(256), 0, s, pts, nrm, n, tf, depth, r.q.data(),
                     r.unit_normals.data(), keys.data(), order.data(), r.input_status.data());
  KERNEL_CHECK();
  const uint64_t sentinel = (uint64_t)1 << (3 * depth);
  sort_pairs_u64(keys.data(), order.data(), n, 3 * depth + 1, s);
  // head marks + scan (samples.py:136-147, 270-279)
  DArray<int> heads(n, s), prefix(n, s), total(1, s);
  mark_heads_u64(keys.data(), n, sentinel, heads.data(), s);
  scan_exclusive_i32(heads.data(), prefix.data(), n, total.data(), s);
  const int G = read_int(total.data(), s);
  if (!G) throw PsrError(2, "No accepted samples with finite nonzero normals");
  r.G = G;
  DArray<int> head_pos(G, s);
  compact_heads(heads.data(), prefix.data(), n, head_pos.data(), s);
  r.sample_keys.reset(G, s);
  r.position_sums.reset(3 * G, s);
  r.normal_sums.reset(3 * G, s);
  r.weights.reset(G, s);
  r.first_indices.reset(G, s);
  r.group_offsets.reset(G + 1, s);
  r.input_group.reset(n, s);
  hipLaunchKernelGGL(k_fill_i32, dim3(blocks_for(n, 256)), dim3(256), 0, s, r.input_group.data(), n, -1);
  KERNEL_CHECK();
  DArray<int> wide(G, s), wide_count(1, s);
  wide_count.zero();
  hipLaunchKernelGGL(k_groups<T>, dim3(blocks_for(G, 256)), dim3(256), 0, s, (const uint64_t*)keys.data(),
                     (const int*)order.data(), (const int*)head_pos.data(), G, n, depth, (const T*)r.q.data(),
                     (const T*)r.unit_normals.data(), r.sample_keys.data(), r.position_sums.data(), r.normal_sums.data(),
                     r.weights.data(), r.first_indices.data(), r.group_offsets.data(), r.input_group.data(), wide.data(),
                     wide_count.data());
  KERNEL_CHECK();
  hipLaunchKernelGGL(k_groups_wide<T>, dim3(256), dim3(64), 0, s, (const uint64_t*)keys.data(), (const int*)order.data(),
                     (const int*)head_pos.data(), G, n, depth, (const T*)r.q.data(), (const T*)r.unit_normals.data(),
                     r.sample_keys.data(), r.position_sums.data(), r.normal_sums.data(), r.weights.data(),
                     r.first_indices.data(), r.group_offsets.data(), r.input_group.data(), (const int*)wide.data(),
                     (const int*)wide_count.data());
  KERNEL_CHECK();
  r.input_order = std::move(order);
}

// ------------------------------------------------------------------ density
// density.py:59-72 (_parents) sorted as (parent lexicographic, child octant):
// the reference's Morton-ordered stable sort puts siblings in octant order.
__global__ void k_parent_records(const int64_t* __restrict__ keys, int64_t m, int d, uint64_t* __restrict__ out,
                                 int* __restrict__ ids) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const int64_t k = keys[i];
  const int x = key_x(k), y = key_y(k), z = key_z(k);
  const int pb = d - 1;
  const uint64_t parent = ((uint64_t)(x >> 1) << (2 * pb)) | ((uint64_t)(y >> 1) << pb) | (uint64_t)(z >> 1);
  out[i] = (parent << 3) | (uint64_t)((x & 1) | ((y & 1) << 1) | ((z & 1) << 2));
  ids[i] = (int)i;
}

__global__ void k_parent_heads(const uint64_t* __restrict__ keys, int64_t m, int* __restrict__ heads) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  heads[i] = (i == 0 || (keys[i] >> 3) != (keys[i - 1] >> 3)) ? 1 : 0;
}

template <class T>
__global__ void k_parent_reduce(const uint64_t* __restrict__ keys, const int* __restrict__ ids, const int* __restrict__ head_pos,
                                int count, int64_t m, int pd, const T* __restrict__ vals, int64_t* __restrict__ out_keys,
                                T* __restrict__ out_vals) {
  int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= count) return;
  int64_t j = head_pos[g];
  const uint64_t parent = keys[j] >> 3;
  T a = T(0), b = T(0), c = T(0), w = T(0);
  while (j < m && (keys[j] >> 3) == parent) {
    const T* v = vals + 4 * (int64_t)ids[j];
    a = a + v[0]; b = b + v[1]; c = c + v[2]; w = w + v[3];
    ++j;
  }
  const uint64_t mask = ((uint64_t)1 << pd) - 1;
  out_keys[g] = basis_key(pd, (int)(parent >> (2 * pd)), (int)((parent >> pd) & mask), (int)(parent & mask));
  out_vals[4 * g] = a; out_vals[4 * g + 1] = b; out_vals[4 * g + 2] = c; out_vals[4 * g + 3] = w;
}

template <class T>
__global__ void k_leaf_values(const T* __restrict__ sums, const T* __restrict__ w, int G, T* __restrict__ out) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= G) return;
  out[4 * i] = sums[3 * i]; out[4 * i + 1] = sums[3 * i + 1]; out[4 * i + 2] = sums[3 * i + 2]; out[4 * i + 3] = w[i];
}

// keyed.py:23-38 Morton codes (x is the lowest bit of each triple)
__global__ void k_morton(const int64_t* __restrict__ keys, int64_t m, int depth, uint64_t* __restrict__ codes,
                         int* __restrict__ ids) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  const int64_t k = keys[i];
  const int c[3] = {key_x(k), key_y(k), key_z(k)};
  uint64_t code = 0;
  for (int bit = 0; bit < depth; ++bit)
    for (int a = 0; a < 3; ++a) code |= (uint64_t)((c[a] >> bit) & 1) << (3 * bit + a);
  codes[i] = code;
  ids[i] = (int)i;
}

// density.py:74-106 (_splat), one record: target key and value.
template <class T> struct SplatSource {
  int cx, cy, cz;
  T w;
  Quad bx, by, bz;
};
template <class T> __device__ __forceinline__ SplatSource<T> density_source(const int64_t key, const T* v, int d) {
  SplatSource<T> s;
  s.cx = key_x(key); s.cy = key_y(key); s.cz = key_z(key);
  const int n = 1 << d;
  T p0 = v[0] / v[3], p1 = v[1] / v[3], p2 = v[2] / v[3];
  T h = T(1) / T(n);
  s.bx = quadratic(double((p0 - T(s.cx) * h) / h));
  s.by = quadratic(double((p1 - T(s.cy) * h) / h));
  s.bz = quadratic(double((p2 - T(s.cz) * h) / h));
  s.w = v[3];
  return s;
}

__global__ void k_density_splat_keys(const int64_t* __restrict__ keys, const int* __restrict__ order, int64_t m, int d,
                                     uint64_t* __restrict__ out, int* __restrict__ ids) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= 27 * m) return;
  const int64_t i = idx / 27;
  const int k = (int)(idx % 27);
  const int64_t key = keys[order[i]];
  const int n = 1 << d;
  const int tx = key_x(key) + k / 9 - 1, ty = key_y(key) + k / 3 % 3 - 1, tz = key_z(key) + k % 3 - 1;
  uint64_t packed = (uint64_t)1 << (3 * d);
  if (imin(imin(tx, ty), tz) >= 0 && imax(imax(tx, ty), tz) < n)
    packed = ((uint64_t)tx << (2 * d)) | ((uint64_t)ty << d) | (uint64_t)tz;
  out[idx] = packed;
  ids[idx] = (int)idx;
}

template <class T>
__global__ void k_density_splat_reduce(const uint64_t* __restrict__ keys, const int* __restrict__ ids,
                                       const int* __restrict__ head_pos, int count, int64_t total, int d,
                                       const int64_t* __restrict__ src_keys, const T* __restrict__ src_vals,
                                       const int* __restrict__ order, T scale, int64_t* __restrict__ out_keys,
                                       T* __restrict__ out_vals) {
  int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= count) return;
  int64_t j = head_pos[g];
  const uint64_t key = keys[j];
  T acc = T(0);
  while (j < total && keys[j] == key) {
    const int id = ids[j];
    const int i = id / 27, k = id % 27;
    const int src = order[i];
    SplatSource<T> sp = density_source<T>(src_keys[src], src_vals + 4 * (int64_t)src, d);
    const T weight = sp.w * scale;
    const T val = T(double(weight) * quad_at(sp.bx, k / 9) * quad_at(sp.by, k / 3 % 3) * quad_at(sp.bz, k % 3));
    acc = acc + val;
    ++j;
  }
  const uint64_t mask = ((uint64_t)1 << d) - 1;
  out_keys[g] = basis_key(d, (int)(key >> (2 * d)), (int)((key >> d) & mask), (int)(key & mask));
  out_vals[g] = acc;
}

// density.py:108-150 (density_value at each aggregate centroid)
template <class T>
__global__ void k_density_eval(const int64_t* __restrict__ lkeys, const T* __restrict__ lvals, int64_t lcount, ColumnTable ct,
                               const T* __restrict__ sums, const T* __restrict__ weights, int G, int d, int stride,
                               T* __restrict__ out) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= G) return;
  const T w = weights[i];
  const T p0 = sums[3 * i] / w, p1 = sums[3 * i + 1] / w, p2 = sums[3 * i + 2] / w;
  const int n = 1 << d;
  const int cx = cell_index(p0, n), cy = cell_index(p1, n), cz = cell_index(p2, n);
  const T h = T(1) / T(n);
  const Quad bx = quadratic(double((p0 - T(cx) * h) / h));
  const Quad by = quadratic(double((p1 - T(cy) * h) / h));
  const Quad bz = quadratic(double((p2 - T(cz) * h) / h));
  T value = T(0);
  const int zlo = imax(cz - 1, 0), zhi = imin(cz + 1, n - 1);
  for (int x = 0; x < 3; ++x)
    for (int y = 0; y < 3; ++y) {  // k = 9x + 3y + z, one lookup per (x, y) column
      const int tx = cx + x - 1, ty = cy + y - 1;
      if (tx < 0 || ty < 0 || tx >= n || ty >= n || zlo > zhi) continue;
      int64_t found[3];
      find_run_table<3>(lkeys, lcount, ct, d, tx, ty, zlo, zhi - zlo + 1, found);
      for (int z = 0; z < 3; ++z) {
        const int tz = cz + z - 1;
        if (tz < zlo || tz > zhi) continue;
        const int64_t idx = found[tz - zlo];
        if (idx >= 0) value = value + T(quad_at(bx, x) * quad_at(by, y) * quad_at(bz, z) * double(lvals[idx]));
      }
    }
  out[(int64_t)i * stride + d] = value;
}

// density.py:152-182 (_depths)
template <class T>
__global__ void k_depths(const T* __restrict__ dens, int G, int kd, T target, T* __restrict__ dw) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= G) return;
  const int stride = kd + 1;
  int d = kd;
  T density = dens[(int64_t)i * stride + d];
  T raw;
  if (density >= target) {
    raw = T(double(d) + double(T(det_log(double(density / target)))) / (LN2_D * 2.0));
  } else {
    T fine = density;
    while (density < target && d > 0) {
      fine = density;
      d -= 1;
      density = dens[(int64_t)i * stride + d];
    }
    raw = T(T(d) + T(det_log(double(density / target))) / T(det_log(double(density / fine))));
  }
  const T h = T(1) / T(1 << d);
  dw[2 * i] = raw;
  dw[2 * i + 1] = h * h / density;
}

// density.py:37-50 (_scale), evaluated once on the host.
template <class T> T density_scale_host() {
  T total = T(0);
  const T dx = T(0.1);
  for (int x = 0; x < 10; ++x) {
    T p = dx / T(2) + dx * T(x);
    Quad b = quadratic(double(p));
    T scale = T(1.0 / (b.b0 * b.b0 + b.b1 * b.b1 + b.b2 * b.b2));
    for (int y = 0; y < 10; ++y)
      for (int z = 0; z < 10; ++z) total = total + scale;
  }
  return total / T(1000);
}

// ------------------------------------------------------------ bitmap form
// The aggregates' cells and the density nodes of every level as bitmaps
// (psr_bitmap.h).  Parents are halved words, the nodes of a level its cells
// dilated by one, and every sum is gathered by its receiver in the order the
// sorts gave it: a parent adds its children by octant, a node the aggregates
// around it in Morton order.  One host read sizes everything.  With a sort a
// level (and one of 27 records an aggregate) the stage took 0.33 ms for 512
// points at depth 4 and 1.95 ms for 800,000 at depth 9; 0.13 and 0.42 ms this
// way.
struct CellLattice {
  uint32_t cells[BITMAP_MAX_LEVELS];  // first word of the aggregates' level
  uint32_t nodes[BITMAP_MAX_LEVELS];  // first word of the density nodes' level
};

PSR_HD int cell_words(int d) { return d > 5 ? 1 << (d - 5) : 1; }  // words per (x, y) row of 2^d cells
PSR_HD uint32_t cell_row(int d, int x, int y) { return (((uint32_t)x << d) | (uint32_t)y) * (uint32_t)cell_words(d); }

// the leaf level's bits: the first key of each word gathers the word's run
__global__ void k_cells_mark(const int64_t* __restrict__ keys, int64_t n, int d, uint32_t* __restrict__ bits) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t key = keys[i];
  if (i > 0 && (keys[i - 1] >> 5) == (key >> 5)) return;  // z is the key's lowest field
  uint32_t word = 0;
  for (int64_t j = i; j < n && (keys[j] >> 5) == (key >> 5); ++j) word |= 1u << (int)(keys[j] & 31);
  bits[cell_row(d, key_x(key), key_y(key)) + (uint32_t)(key_z(key) >> 5)] = word;
}

// word t of level d from level d + 1 (density.py:59-72, _parents)
__device__ __forceinline__ uint32_t halved_word(const uint32_t* fine, int d, uint32_t t) {
  const int wz = cell_words(d), fz = cell_words(d + 1);
  const int w = (int)(t % (uint32_t)wz), y = (int)((t / (uint32_t)wz) & ((1u << d) - 1u)), x = (int)((t / (uint32_t)wz) >> d);
  uint32_t c1 = 0, c2 = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t* row = fine + cell_row(d + 1, 2 * x + (k >> 1), 2 * y + (k & 1));
    c1 |= row[2 * w];
    if (2 * w + 1 < fz) c2 |= row[2 * w + 1];
  }
  uint64_t v = ((uint64_t)c2 << 32) | c1;
  return even_bits(v | (v >> 1));
}

__global__ void k_cells_halve(CellLattice lat, int d, uint32_t words, uint32_t* __restrict__ bits) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < words) bits[lat.cells[d] + t] = halved_word(bits + lat.cells[d + 1], d, t);
}

// levels top..0 (at most 1,024 words each) one after another in one workgroup
constexpr int COARSE_CELL_LEVEL = 5;
__global__ void __launch_bounds__(1024) k_cells_coarse(CellLattice lat, int top, uint32_t* bits) {
  for (int d = top; d >= 0; --d) {
    const uint32_t words = (1u << (2 * d)) * (uint32_t)cell_words(d);
    for (uint32_t t = threadIdx.x; t < words; t += 1024) bits[lat.cells[d] + t] = halved_word(bits + lat.cells[d + 1], d, t);
    __syncthreads();
  }
}

// Where a launch over all levels' words or keys finds its level: sets 0..depth
// are the aggregates' levels, the rest the density levels.
template <class T> struct CellArrays {
  int sets;
  int block0[2 * BITMAP_MAX_LEVELS];
  int depth[2 * BITMAP_MAX_LEVELS];
  uint32_t base[2 * BITMAP_MAX_LEVELS];
  int64_t* keys[2 * BITMAP_MAX_LEVELS];
};

template <class A> __device__ __forceinline__ int set_of_block(const A& a, int block) {
  int d = 0;
  for (int k = 1; k < a.sets; ++k) d = block >= a.block0[k] ? k : d;
  return d;
}

// every density level's nodes: the cells within one of an aggregate's
// (density.py:74-106 skips targets outside the grid)
template <class T>
__global__ void __launch_bounds__(BITMAP_THREADS) k_cells_dilate(CellLattice lat, CellArrays<T> arr, int first_set,
                                                                 uint32_t* __restrict__ bits) {
  const int block = (int)blockIdx.x + arr.block0[first_set];
  const int set = set_of_block(arr, block), d = arr.depth[set], n = 1 << d, wz = cell_words(d);
  const uint32_t words = (1u << (2 * d)) * (uint32_t)wz;
  const uint32_t* cells = bits + lat.cells[d];
  for (int k = 0; k < BITMAP_ITEMS; ++k) {
    const uint32_t t = (uint32_t)(block - arr.block0[set]) * BITMAP_BLOCK + k * BITMAP_THREADS + threadIdx.x;
    if (t >= words) return;
    const int w = (int)(t % (uint32_t)wz), y = (int)((t / (uint32_t)wz) & (uint32_t)(n - 1)), x = (int)((t / (uint32_t)wz) >> d);
    uint32_t own = 0, below = 0, above = 0;
    for (int a = imax(x - 1, 0); a <= imin(x + 1, n - 1); ++a)
      for (int b = imax(y - 1, 0); b <= imin(y + 1, n - 1); ++b) {
        const uint32_t* row = cells + cell_row(d, a, b) + w;
        own |= row[0];
        if (w > 0) below |= row[-1];
        if (w + 1 < wz) above |= row[1];
      }
    bits[arr.base[set] + t] = (own | (own << 1) | (own >> 1) | (below >> 31) | (above << 31)) & word_range(w, 0, n);
  }
}

// ranks at the sets' first words and the end, for the host
template <class T>
__global__ void k_cells_starts(CellArrays<T> arr, const int* __restrict__ pre, uint32_t words, int* __restrict__ out) {
  const int k = threadIdx.x;
  if (k <= arr.sets) out[k] = pre[k < arr.sets ? arr.base[k] : words];
}

// all sets' sorted keys
template <class T>
__global__ void __launch_bounds__(BITMAP_THREADS) k_cells_keys(CellArrays<T> arr, const uint32_t* __restrict__ bits,
                                                               const int* __restrict__ pre) {
  const int set = set_of_block(arr, (int)blockIdx.x), d = arr.depth[set], wz = cell_words(d);
  const uint32_t words = (1u << (2 * d)) * (uint32_t)wz, base = arr.base[set];
  for (int k = 0; k < BITMAP_ITEMS; ++k) {
    const uint32_t t = (uint32_t)((int)blockIdx.x - arr.block0[set]) * BITMAP_BLOCK + k * BITMAP_THREADS + threadIdx.x;
    if (t >= words) return;
    uint32_t b = bits[base + t];
    if (!b) continue;
    const int w = (int)(t % (uint32_t)wz), y = (int)((t / (uint32_t)wz) & ((1u << d) - 1u)), x = (int)((t / (uint32_t)wz) >> d);
    int64_t* out = arr.keys[set] + (pre[base + t] - pre[base]);
    for (; b; b &= b - 1) *out++ = basis_key(d, x, y, 32 * w + __builtin_ctz(b));
  }
}

// density.py:228-240: parent g of level d adds its children in octant order
// (x lowest)
template <class T>
__device__ __forceinline__ void parent_sum(int g, int d, const int64_t* keys, const uint32_t* fine_bits, const int* fine_pre,
                                           const T* fine_vals, T* vals) {
  const int64_t key = keys[g];
  const int z = 2 * key_z(key), base = fine_pre[0];
  uint32_t two[4];
  int rank[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {  // row (2x + (k & 1), 2y + (k >> 1)): its cells z, z + 1 lie in one word
    const uint32_t t = cell_row(d + 1, 2 * key_x(key) + (k & 1), 2 * key_y(key) + (k >> 1)) + (uint32_t)(z >> 5);
    const uint32_t b = fine_bits[t];
    two[k] = (b >> (z & 31)) & 3u;
    rank[k] = fine_pre[t] - base + __popc(b & ((1u << (z & 31)) - 1u));
  }
  T v[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll
  for (int o = 0; o < 8; ++o) {
    const int k = o & 3, up = o >> 2;
    if (!((two[k] >> up) & 1u)) continue;
    const T* c = fine_vals + 4 * (int64_t)(rank[k] + (up && (two[k] & 1u) ? 1 : 0));
#pragma unroll
    for (int a = 0; a < 4; ++a) v[a] = v[a] + c[a];
  }
#pragma unroll
  for (int a = 0; a < 4; ++a) vals[4 * (int64_t)g + a] = v[a];
}

template <class T>
__global__ void k_parent_sums(int count, int d, const int64_t* __restrict__ keys, const uint32_t* __restrict__ fine_bits,
                              const int* __restrict__ fine_pre, const T* __restrict__ fine_vals, T* __restrict__ vals) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < count) parent_sum(g, d, keys, fine_bits, fine_pre, fine_vals, vals);
}

template <class T> struct ParentChain {
  int count[COARSE_CELL_LEVEL + 2];
  const int64_t* keys[COARSE_CELL_LEVEL + 2];
  T* vals[COARSE_CELL_LEVEL + 2];
};

template <class T>
__global__ void __launch_bounds__(1024) k_parent_sums_coarse(CellLattice lat, ParentChain<T> c, int top, const uint32_t* bits,
                                                             const int* pre) {
  for (int d = top; d >= 0; --d) {
    for (int g = threadIdx.x; g < c.count[d]; g += 1024)
      parent_sum(g, d, c.keys[d], bits + lat.cells[d + 1], pre + lat.cells[d + 1], (const T*)c.vals[d + 1], c.vals[d]);
    __syncthreads();
  }
}

// Presence of cells z - 1, z, z + 1 of a row (bits 0..2) and the rank of the
// first of them, relative to the level: (rank << 3) | presence.
__device__ __forceinline__ int row_of_three(const uint32_t* bits, const int* pre, uint32_t row, int z, int d) {
  const int z0 = imax(z - 1, 0), w = z0 >> 5, sh = z0 & 31;
  const uint32_t b = bits[row + (uint32_t)w];
  const uint32_t next = w + 1 < cell_words(d) ? bits[row + (uint32_t)w + 1] : 0u;
  const uint32_t win = (uint32_t)((((uint64_t)next << 32) | b) >> sh);
  const int m = z > 0 ? (int)(win & 7u) : (int)((win & 3u) << 1);
  return ((pre[row + (uint32_t)w] - pre[0] + __popc(b & ((1u << sh) - 1u))) << 3) | m;
}

template <class T> struct DensityArrays {
  int sets;  // density levels 0..kd
  int block0[BITMAP_MAX_LEVELS];
  int count[BITMAP_MAX_LEVELS];
  const int64_t* keys[BITMAP_MAX_LEVELS];
  const T* cell_vals[BITMAP_MAX_LEVELS];
  T* vals[BITMAP_MAX_LEVELS];
};

// density.py:74-106, gathered: node t of level d adds the splats of the
// aggregates in the 27 cells around it, in the aggregates' Morton order (the
// stable sort of the splat records by node kept that order).  Three
// neighbouring coordinates t - 1, t, t + 1 have one boundary at a high bit H
// (the carry into t for even t, into t + 1 for odd t) and one at bit 0, so
// two of the cells differ first at the most significant high boundary between
// them, 3 H + axis over the axes, and else at bit 0: the order is the high
// sides with the axes by 3 H + axis, then the low bits z, y, x.
template <class T>
__global__ void __launch_bounds__(256) k_density_gather(CellLattice lat, DensityArrays<T> arr, const uint32_t* __restrict__ bits,
                                                        const int* __restrict__ pre, T scale) {
  __shared__ int rows[9][256];  // row_of_three of the nine (x, y) rows; each thread its own column
  const int d = set_of_block(arr, (int)blockIdx.x), n = 1 << d;
  const int g = ((int)blockIdx.x - arr.block0[d]) * 256 + (int)threadIdx.x;
  if (g >= arr.count[d]) return;
  const int64_t key = arr.keys[d][g];
  const int t[3] = {key_x(key), key_y(key), key_z(key)};
  const uint32_t* cell_bits = bits + lat.cells[d];
  const int* cell_pre = pre + lat.cells[d];
#pragma unroll
  for (int r = 0; r < 9; ++r) {
    const int x = t[0] + r / 3 - 1, y = t[1] + r % 3 - 1;
    rows[r][threadIdx.x] = x >= 0 && y >= 0 && x < n && y < n ? row_of_three(cell_bits, cell_pre, cell_row(d, x, y), t[2], d) : 0;
  }
  int sig[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) sig[a] = 3 * (t[a] == 0 ? 30 : __builtin_ctz((t[a] & 1) ? t[a] + 1 : t[a])) + a;
  // place[a]: the axis's bit in `hi`, 2 for the most significant
  int place[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) place[a] = (sig[a] > sig[(a + 1) % 3] ? 1 : 0) + (sig[a] > sig[(a + 2) % 3] ? 1 : 0);
  const T h = T(1) / T(n);
  const T* vals = arr.cell_vals[d];
  T acc = T(0);
  for (int hi = 0; hi < 8; ++hi)
    for (int low = 0; low < 8; ++low) {
      int off[3];
      bool there = true;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const int side = (hi >> place[a]) & 1, l = (low >> a) & 1;
        // even t: {t - 1 (low bit 1)} | {t, t + 1}; odd t: {t - 1, t} | {t + 1 (low bit 0)}
        const bool odd = t[a] & 1;
        off[a] = odd ? (side ? 1 : l - 1) : (side ? l : -1);
        there = there && (odd ? !(side && l) : (side || l));
      }
      if (!there) continue;
      const int row = rows[(off[0] + 1) * 3 + off[1] + 1][threadIdx.x];
      if (!((row >> (off[2] + 1)) & 1)) continue;
      const T* v = vals + 4 * (int64_t)((row >> 3) + __popc((unsigned)(row & 7) & ((1u << (off[2] + 1)) - 1u)));
      const T w = v[3];
      const int sx = t[0] + off[0], sy = t[1] + off[1], sz = t[2] + off[2];
      const Quad bx = quadratic(double((v[0] / w - T(sx) * h) / h));
      const Quad by = quadratic(double((v[1] / w - T(sy) * h) / h));
      const Quad bz = quadratic(double((v[2] / w - T(sz) * h) / h));
      const T weight = w * scale;
      acc = acc + T(double(weight) * quad_at(bx, 1 - off[0]) * quad_at(by, 1 - off[1]) * quad_at(bz, 1 - off[2]));
    }
  arr.vals[d][g] = acc;
}

// density.py:108-150 (density_value at each aggregate centroid), level
// blockIdx.y, by the node bitmaps
template <class T>
__global__ void __launch_bounds__(256) k_density_at(CellLattice lat, DensityArrays<T> arr, const uint32_t* __restrict__ bits,
                                                    const int* __restrict__ pre, const T* __restrict__ sums,
                                                    const T* __restrict__ weights, int G, T* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, d = blockIdx.y;
  if (i >= G) return;
  const T w = weights[i];
  const T p0 = sums[3 * i] / w, p1 = sums[3 * i + 1] / w, p2 = sums[3 * i + 2] / w;
  const int n = 1 << d;
  const int cx = cell_index(p0, n), cy = cell_index(p1, n), cz = cell_index(p2, n);
  const T h = T(1) / T(n);
  const Quad bx = quadratic(double((p0 - T(cx) * h) / h));
  const Quad by = quadratic(double((p1 - T(cy) * h) / h));
  const Quad bz = quadratic(double((p2 - T(cz) * h) / h));
  const uint32_t* node_bits = bits + lat.nodes[d];
  const int* node_pre = pre + lat.nodes[d];
  const T* lvals = arr.vals[d];
  int row[9];
#pragma unroll
  for (int r = 0; r < 9; ++r) {  // a centroid rounded past the cube's end has cell n: its row of three ends at n - 1
    const int x = cx + r / 3 - 1, y = cy + r % 3 - 1;
    row[r] = x >= 0 && y >= 0 && x < n && y < n && cz <= n ? row_of_three(node_bits, node_pre, cell_row(d, x, y), cz, d) : 0;
  }
  T v[27];
#pragma unroll
  for (int k = 0; k < 27; ++k) {
    const int m = row[k / 3], z = k % 3;
    v[k] = (m >> z) & 1 ? lvals[(m >> 3) + __popc((unsigned)(m & 7) & ((1u << z) - 1u))] : T(0);
  }
  T value = T(0);
#pragma unroll
  for (int k = 0; k < 27; ++k)  // k = 9x + 3y + z
    if ((row[k / 3] >> (k % 3)) & 1)
      value = value + T(quad_at(bx, k / 9) * quad_at(by, k / 3 % 3) * quad_at(bz, k % 3) * double(v[k]));
  out[(int64_t)i * arr.sets + d] = value;
}

template <class T> void density_from_bitmaps(Result<T>& r) {
  hipStream_t s = r.s;
  const int depth = r.prm.depth, kd = r.prm.kernel_depth, G = r.G;
  r.density_scale = density_scale_host<T>();
  r.densities.reset((size_t)G * (kd + 1), s);
  // lattices: the aggregates' levels, then the density levels
  CellLattice lat{};
  CellArrays<T> arr{};
  size_t words = 0;
  auto level_words = [](int d) { return ((size_t)1 << (2 * d)) * (size_t)cell_words(d); };
  auto add_set = [&](int d) {
    arr.base[arr.sets] = (uint32_t)words;
    arr.depth[arr.sets] = d;
    arr.block0[arr.sets++] = (int)(words / BITMAP_BLOCK);
    words += (level_words(d) + BITMAP_BLOCK - 1) / BITMAP_BLOCK * BITMAP_BLOCK;
    return arr.base[arr.sets - 1];
  };
  for (int d = 0; d <= depth; ++d) lat.cells[d] = add_set(d);
  for (int d = 0; d <= kd; ++d) lat.nodes[d] = add_set(d);
  const int blocks = (int)(words / BITMAP_BLOCK), node_set = depth + 1;
  DArray<uint32_t> bits(words, s);
  bits.zero();
  hipLaunchKernelGGL(k_cells_mark, dim3(blocks_for(G, 256)), dim3(256), 0, s, (const int64_t*)r.sample_keys.data(), (int64_t)G, depth,
                     bits.data() + lat.cells[depth]);
  KERNEL_CHECK();
  const int coarse = std::min(depth - 1, COARSE_CELL_LEVEL);
  for (int d = depth - 1; d > coarse; --d) {
    hipLaunchKernelGGL(k_cells_halve, dim3(blocks_for(level_words(d), 256)), dim3(256), 0, s, lat, d, (uint32_t)level_words(d),
                       bits.data());
    KERNEL_CHECK();
  }
  hipLaunchKernelGGL(k_cells_coarse, dim3(1), dim3(1024), 0, s, lat, coarse, bits.data());
  KERNEL_CHECK();
  hipLaunchKernelGGL(k_cells_dilate<T>, dim3(blocks - arr.block0[node_set]), dim3(BITMAP_THREADS), 0, s, lat, arr, node_set, bits.data());
  KERNEL_CHECK();
  DArray<int> sums(blocks, s), pre(words + 1, s), starts(arr.sets + 1, s);
  hipLaunchKernelGGL(k_bits_count, dim3(blocks), dim3(BITMAP_THREADS), 0, s, (const uint32_t*)bits.data(), sums.data());
  KERNEL_CHECK();
  scan_exclusive_i32(sums.data(), sums.data(), blocks, nullptr, s);
  hipLaunchKernelGGL(k_bits_ranks, dim3(blocks), dim3(BITMAP_THREADS), 0, s, (const uint32_t*)bits.data(), (const int*)sums.data(),
                     pre.data());
  KERNEL_CHECK();
  hipLaunchKernelGGL(k_cells_starts<T>, dim3(1), dim3(64), 0, s, arr, (const int*)pre.data(), (uint32_t)words, starts.data());
  KERNEL_CHECK();
  std::vector<int> first(arr.sets + 1);
  read_bytes(first.data(), starts.data(), sizeof(int) * first.size(), s);
  auto count_of = [&](int set) { return first[set + 1] - first[set]; };
  DensityArrays<T> den{};
  den.sets = kd + 1;
  int den_blocks = 0;
  for (int d = 0; d <= depth; ++d) {
    r.levels[d].agg_keys.reset(count_of(d), s);
    r.levels[d].agg_vals.reset(4 * (size_t)count_of(d), s);
    arr.keys[d] = r.levels[d].agg_keys.data();
  }
  for (int d = 0; d <= kd; ++d) {
    LevelState<T>& L = r.levels[d];
    const int count = count_of(node_set + d);
    L.dens_keys.reset(count, s);
    L.dens_vals.reset(count, s);
    arr.keys[node_set + d] = L.dens_keys.data();
    den.block0[d] = den_blocks;
    den_blocks += (int)blocks_for(count, 256);
    den.count[d] = count;
    den.keys[d] = L.dens_keys.data();
    den.cell_vals[d] = L.agg_vals.data();
    den.vals[d] = L.dens_vals.data();
  }
  hipLaunchKernelGGL(k_cells_keys<T>, dim3(blocks), dim3(BITMAP_THREADS), 0, s, arr, (const uint32_t*)bits.data(),
                     (const int*)pre.data());
  KERNEL_CHECK();
  hipLaunchKernelGGL(k_leaf_values<T>, dim3(blocks_for(G, 256)), dim3(256), 0, s, (const T*)r.position_sums.data(),
                     (const T*)r.weights.data(), G, r.levels[depth].agg_vals.data());
  KERNEL_CHECK();
  for (int d = depth - 1; d > coarse; --d) {
    const int count = count_of(d);
    hipLaunchKernelGGL(k_parent_sums<T>, dim3(blocks_for(count, 256)), dim3(256), 0, s, count, d,
                       (const int64_t*)r.levels[d].agg_keys.data(), (const uint32_t*)(bits.data() + lat.cells[d + 1]),
                       (const int*)(pre.data() + lat.cells[d + 1]), (const T*)r.levels[d + 1].agg_vals.data(),
                       r.levels[d].agg_vals.data());
    KERNEL_CHECK();
  }
  ParentChain<T> chain{};
  for (int d = 0; d <= coarse + 1; ++d) {
    chain.count[d] = count_of(d);
    chain.keys[d] = r.levels[d].agg_keys.data();
    chain.vals[d] = r.levels[d].agg_vals.data();
  }
  hipLaunchKernelGGL(k_parent_sums_coarse<T>, dim3(1), dim3(1024), 0, s, lat, chain, coarse, (const uint32_t*)bits.data(),
                     (const int*)pre.data());
  KERNEL_CHECK();
  hipLaunchKernelGGL(k_density_gather<T>, dim3(den_blocks), dim3(256), 0, s, lat, den, (const uint32_t*)bits.data(),
                     (const int*)pre.data(), r.density_scale);
  KERNEL_CHECK();
  hipLaunchKernelGGL(k_density_at<T>, dim3(blocks_for(G, 256), kd + 1), dim3(256), 0, s, lat, den, (const uint32_t*)bits.data(),
                     (const int*)pre.data(), (const T*)r.position_sums.data(), (const T*)r.weights.data(), G, r.densities.data());
  KERNEL_CHECK();
}

template <class T> void density_from_sorts(Result<T>& r);

template <class T> void stage_density(Result<T>& r) {
  hipStream_t s = r.s;
  r.levels.resize(r.prm.depth + 1);
  if (bitmap_fits((int64_t)1 << r.prm.depth)) density_from_bitmaps(r);
  else density_from_sorts(r);
  r.dw.reset(2 * (size_t)r.G, s);
  hipLaunchKernelGGL(k_depths<T>, dim3(blocks_for(r.G, 256)), dim3(256), 0, s, (const T*)r.densities.data(), r.G,
                     r.prm.kernel_depth, T(r.prm.samples_per_node), r.dw.data());
  KERNEL_CHECK();
}

// The same by sorts (levels beyond the bitmap limit).
template <class T> void density_from_sorts(Result<T>& r) {
  hipStream_t s = r.s;
  const int depth = r.prm.depth, kd = r.prm.kernel_depth;
  const int G = r.G;
  LevelState<T>& leaf = r.levels[depth];
  leaf.agg_keys.reset(G, s);
  HIP_CHECK(hipMemcpyAsync(leaf.agg_keys.data(), r.sample_keys.data(), G * sizeof(int64_t), hipMemcpyDeviceToDevice, s));
  leaf.agg_vals.reset(4 * (size_t)G, s);
  hipLaunchKernelGGL(k_leaf_values<T>, dim3(blocks_for(G, 256)), dim3(256), 0, s, (const T*)r.position_sums.data(),
                     (const T*)r.weights.data(), G, leaf.agg_vals.data());
  KERNEL_CHECK();
  // aggregates d -> d-1 (density.py:228-240)
  for (int d = depth; d > 0; --d) {
    LevelState<T>& src = r.levels[d];
    const int64_t m = (int64_t)src.agg_keys.size();
    DArray<uint64_t> keys(m, s);
    DArray<int> ids(m, s), heads(m, s), prefix(m, s), total(1, s);
    hipLaunchKernelGGL(k_parent_records, dim3(blocks_for(m, 256)), dim3(256), 0, s, (const int64_t*)src.agg_keys.data(), m,
                       d, keys.data(), ids.data());
    KERNEL_CHECK();
    sort_pairs_u64(keys.data(), ids.data(), m, 3 * d, s);
    hipLaunchKernelGGL(k_parent_heads, dim3(blocks_for(m, 256)), dim3(256), 0, s, (const uint64_t*)keys.data(), m,
                       heads.data());
    KERNEL_CHECK();
    scan_exclusive_i32(heads.data(), prefix.data(), m, total.data(), s);
    const int count = read_int(total.data(), s);
    DArray<int> head_pos(count, s);
    compact_heads(heads.data(), prefix.data(), m, head_pos.data(), s);
    LevelState<T>& dst = r.levels[d - 1];
    dst.agg_keys.reset(count, s);
    dst.agg_vals.reset(4 * (size_t)count, s);
    hipLaunchKernelGGL(k_parent_reduce<T>, dim3(blocks_for(count, 256)), dim3(256), 0, s, (const uint64_t*)keys.data(),
                       (const int*)ids.data(), (const int*)head_pos.data(), count, m, d - 1, (const T*)src.agg_vals.data(),
                       dst.agg_keys.data(), dst.agg_vals.data());
    KERNEL_CHECK();
  }
  r.density_scale = density_scale_host<T>();
  r.densities.reset((size_t)G * (kd + 1), s);
  // density.py:245-271.  The levels are independent: every level's records
  // are sorted and their heads counted first, the counts come to the host in
  // one read, then each level is reduced and evaluated.
  struct Splat {
    int64_t m = 0, total_records = 0;
    DArray<int> order, rids, heads, prefix;
    DArray<uint64_t> rkeys;
  };
  std::vector<Splat> lv(kd + 1);
  DArray<int> totals(kd + 1, s);
  for (int d = 0; d <= kd; ++d) {
    LevelState<T>& L = r.levels[d];
    Splat& v = lv[d];
    v.m = (int64_t)L.agg_keys.size();
    DArray<uint64_t> codes(v.m, s);
    v.order.reset(v.m, s);
    hipLaunchKernelGGL(k_morton, dim3(blocks_for(v.m, 256)), dim3(256), 0, s, (const int64_t*)L.agg_keys.data(), v.m, d,
                       codes.data(), v.order.data());
    KERNEL_CHECK();
    sort_pairs_u64(codes.data(), v.order.data(), v.m, 3 * d, s);
    v.total_records = 27 * v.m;
    v.rkeys.reset(v.total_records, s);
    v.rids.reset(v.total_records, s);
    v.heads.reset(v.total_records, s);
    v.prefix.reset(v.total_records, s);
    hipLaunchKernelGGL(k_density_splat_keys, dim3(blocks_for(v.total_records, 256)), dim3(256), 0, s,
                       (const int64_t*)L.agg_keys.data(), (const int*)v.order.data(), v.m, d, v.rkeys.data(), v.rids.data());
    KERNEL_CHECK();
    const uint64_t sentinel = (uint64_t)1 << (3 * d);
    sort_pairs_u64(v.rkeys.data(), v.rids.data(), v.total_records, 3 * d + 1, s);
    mark_heads_u64(v.rkeys.data(), v.total_records, sentinel, v.heads.data(), s);
    scan_exclusive_i32(v.heads.data(), v.prefix.data(), v.total_records, totals.data() + d, s);
  }
  std::vector<int> counts(kd + 1);
  read_bytes(counts.data(), totals.data(), sizeof(int) * (kd + 1), s);
  for (int d = 0; d <= kd; ++d) {
    LevelState<T>& L = r.levels[d];
    Splat& v = lv[d];
    const int count = counts[d];
    DArray<int> head_pos(count, s);
    compact_heads(v.heads.data(), v.prefix.data(), v.total_records, head_pos.data(), s);
    L.dens_keys.reset(count, s);
    L.dens_vals.reset(count, s);
    hipLaunchKernelGGL(k_density_splat_reduce<T>, dim3(blocks_for(count, 256)), dim3(256), 0, s,
                       (const uint64_t*)v.rkeys.data(), (const int*)v.rids.data(), (const int*)head_pos.data(), count,
                       v.total_records, d, (const int64_t*)L.agg_keys.data(), (const T*)L.agg_vals.data(),
                       (const int*)v.order.data(), r.density_scale, L.dens_keys.data(), L.dens_vals.data());
    KERNEL_CHECK();
    ColumnIndex columns;
    build_column_index((const int64_t*)L.dens_keys.data(), count, (1 << d) + 1, columns, s);
    hipLaunchKernelGGL(k_density_eval<T>, dim3(blocks_for(G, 256)), dim3(256), 0, s, (const int64_t*)L.dens_keys.data(),
                       (const T*)L.dens_vals.data(), (int64_t)count, columns.view(), (const T*)r.position_sums.data(),
                       (const T*)r.weights.data(), G, d, kd + 1, r.densities.data());
    KERNEL_CHECK();
  }
}

// ------------------------------------------------------------------ normals
__global__ void k_first_keys(const int* __restrict__ first, int G, uint64_t* __restrict__ keys, int* __restrict__ ids) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= G) return;
  keys[i] = (uint64_t)first[i];
  ids[i] = i;
}

template <class T>
__device__ __forceinline__ bool normal_record_valid(int64_t idx, int G, const int* __restrict__ order, const T* __restrict__ sums,
                                                    const T* __restrict__ nsums, const T* __restrict__ weights,
                                                    const T* __restrict__ dw, int minimum, int maximum,
                                                    NormalRecord<T>* rec) {
  if (idx >= 54 * (int64_t)G) return false;
  *rec = normal_record<T>(order[idx / 54], (int)(idx % 54), sums, nsums, weights, dw, minimum, maximum, false);
  return rec->valid;
}

// Valid splat records per 256-record block (normals.py:46-104 skips records
// off the grid and the second depth when the fraction is 1).
template <class T>
__global__ void __launch_bounds__(256) k_normal_splat_count(const int* __restrict__ order, int G, const T* __restrict__ sums,
                                                            const T* __restrict__ nsums, const T* __restrict__ weights,
                                                            const T* __restrict__ dw, int minimum, int maximum,
                                                            int* __restrict__ block_counts) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  NormalRecord<T> rec;
  const bool valid = normal_record_valid(idx, G, order, sums, nsums, weights, dw, minimum, maximum, &rec);
  const int count = __syncthreads_count(valid);
  if (threadIdx.x == 0) block_counts[blockIdx.x] = count;
}

// The valid records, compacted in record order: key top<<3D | x<<2D | y<<D | z,
// the compacted position (the sort payload) and the record's value.
template <class T, class K>
__global__ void __launch_bounds__(256) k_normal_splat_keys(const int* __restrict__ order, int G, const T* __restrict__ sums,
                                                           const T* __restrict__ nsums, const T* __restrict__ weights,
                                                           const T* __restrict__ dw, int minimum, int maximum,
                                                           const int* __restrict__ block_offsets, int64_t capacity,
                                                           K* __restrict__ out, int* __restrict__ ids, T* __restrict__ vals) {
  __shared__ int wave_count[4];
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  NormalRecord<T> rec;
  rec.valid = false;
  if (idx < 54 * (int64_t)G)
    rec = normal_record<T>(order[idx / 54], (int)(idx % 54), sums, nsums, weights, dw, minimum, maximum, true);
  const bool valid = rec.valid;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t ballot = __ballot(valid);
  if (lane == 0) wave_count[wave] = __popcll(ballot);
  __syncthreads();
  if (!valid) return;
  int pos = block_offsets[blockIdx.x] + __popcll(ballot & ((lane == 0) ? 0ull : ((~0ull) >> (64 - lane))));
  for (int w = 0; w < wave; ++w) pos += wave_count[w];
  if (pos >= capacity) return;  // the counting pass saw the same records
  const int D = maximum;
  out[pos] = ((K)rec.top << (3 * D)) | ((K)rec.x << (2 * D)) | ((K)rec.y << D) | (K)rec.z;
  ids[pos] = pos;
  vals[3 * (int64_t)pos] = rec.v0;
  vals[3 * (int64_t)pos + 1] = rec.v1;
  vals[3 * (int64_t)pos + 2] = rec.v2;
}

template <class T, class K>
__global__ void k_normal_splat_reduce(const K* __restrict__ keys, const int* __restrict__ ids, const T* __restrict__ vals,
                                      const int* __restrict__ head_pos, int count, int64_t total, int maximum,
                                      int64_t* __restrict__ out_keys, T* __restrict__ out_vals) {
  int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= count) return;
  int64_t j = head_pos[g];
  const K key = keys[j];
  T a = T(0), b = T(0), c = T(0);
  while (j < total && keys[j] == key) {
    const T* v = vals + 3 * (int64_t)ids[j];
    a = a + v[0]; b = b + v[1]; c = c + v[2];
    ++j;
  }
  const int D = maximum;
  const K mask = ((K)1 << D) - 1;
  out_keys[g] = basis_key((int)(key >> (3 * D)), (int)((key >> (2 * D)) & mask), (int)((key >> D) & mask), (int)(key & mask));
  // normals.py:106-109 (_negative)
  out_vals[3 * g] = -a; out_vals[3 * g + 1] = -b; out_vals[3 * g + 2] = -c;
}

// normals.py:111-163: contributions in first-index order, then one serial
// chain; stored component-major (component c of aggregate i at c * G + i).
template <class T>
__global__ void k_average_contributions(const int* __restrict__ order, int G, const T* __restrict__ nsums,
                                        const T* __restrict__ weights, const T* __restrict__ dw, T* __restrict__ out) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= G) return;
  const int s = order[i];
  const T w = weights[s];
  const T n0 = nsums[3 * s] / w, n1 = nsums[3 * s + 1] / w, n2 = nsums[3 * s + 2] / w;
  T v0 = T(0), v1 = T(0), v2 = T(0);
  if (sqrt(n0 * n0 + n1 * n1 + n2 * n2) > T(0)) {
    v0 = dw[2 * s] * w;
    v1 = dw[2 * s + 1] * w;
    v2 = w;
  }
  out[i] = v0; out[G + i] = v1; out[2 * (int64_t)G + i] = v2;
}

// The three serial chains, each acc = fl(acc + v) in element order, without
// their latency: one add after another takes 7 ns a value (480,000 float64
// aggregates: 3.4 ms, which the operators' assembly and the base solve waited
// for; this form 0.55 ms).
//
// While acc stays in one binade [2^e, 2^(e+1)) it is a whole number S of units
// u = 2^(e-p), and adding v >= 0 is a whole-number addition: v / u rounded to
// the nearest, and halfway cases to the side that leaves S even.  So a value
// is a function of S's parity alone, "add a if S is even, b if odd", and such
// functions compose associatively: a workgroup scans them over a chunk of
// values and every thread knows its S exactly.  The thread in whose values S
// reaches the binade's end adds them to acc one by one in T, and the threads
// after it scan again in the new binade (a chain of n equal values crosses
// log2 n of them).  acc starts at +0, where the first thread with a value
// other than zero adds its own one by one.  Values that are negative or NaN, and
// sums near underflow or not finite, take the whole chunk one by one.
// A skipped contribution is exactly (0,0,0), the identity, as the reference's
// `> 0` test (normals.py:160-163) makes it.
constexpr int AVG_THREADS = 512;
constexpr int AVG_EACH = 8;
constexpr int AVG_CHUNK = AVG_THREADS * AVG_EACH;
constexpr long long AVG_CAP = 1ll << 54;  // sums are only used below 2^53

struct ParityAdd {
  long long even, odd;
};
__device__ __forceinline__ ParityAdd then(ParityAdd l, ParityAdd r) {
  const long long even = l.even + ((l.even & 1) ? r.odd : r.even), odd = l.odd + ((l.odd & 1) ? r.even : r.odd);
  return ParityAdd{even < AVG_CAP ? even : AVG_CAP, odd < AVG_CAP ? odd : AVG_CAP};
}

template <class T>
__global__ void __launch_bounds__(AVG_THREADS) k_average_chains(const T* __restrict__ contrib, int G, T* __restrict__ totals) {
  constexpr int P = sizeof(T) == 8 ? 52 : 23;  // fraction bits
  constexpr int WAVES = AVG_THREADS / 64;
  __shared__ T stage[AVG_CHUNK + AVG_CHUNK / AVG_EACH];  // a value of padding a thread: no bank conflicts
  __shared__ ParityAdd wave_total[WAVES];
  __shared__ int first_cross[WAVES];
  __shared__ T acc;
  __shared__ int bad;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T* __restrict__ src = contrib + (int64_t)blockIdx.x * G;
  T pre[AVG_EACH];
  auto load = [&](int64_t first) {
#pragma unroll
    for (int k = 0; k < AVG_EACH; ++k) {
      const int64_t i = first + k * AVG_THREADS + tid;
      pre[k] = i < G ? src[i] : T(0);
    }
  };
  if (tid == 0) acc = T(0);
  load(0);
  for (int64_t first = 0; first < G; first += AVG_CHUNK) {
    __syncthreads();
    if (tid == 0) bad = 0;
#pragma unroll
    for (int k = 0; k < AVG_EACH; ++k) {
      const int i = k * AVG_THREADS + tid;
      stage[i + i / AVG_EACH] = pre[k];
    }
    __syncthreads();
    if (first + AVG_CHUNK < G) load(first + AVG_CHUNK);
    T v[AVG_EACH];
    bool any = false, wrong = false;
#pragma unroll
    for (int k = 0; k < AVG_EACH; ++k) {
      v[k] = stage[tid * (AVG_EACH + 1) + k];
      any = any || v[k] != T(0);
      wrong = wrong || !(v[k] >= T(0));
    }
    if (wrong) bad = 1;
    __syncthreads();
    for (int from = 0; from < AVG_THREADS;) {  // uniform over the workgroup
      const T a0 = acc;
      if (bad || !(a0 == T(0) || (a0 >= T(1e-30) && a0 <= T(1e30)))) {
        __syncthreads();  // acc is read
        if (tid == 0) {
          T t = a0;
          for (int i = from * AVG_EACH; i < AVG_CHUNK; ++i) t = t + stage[i + i / AVG_EACH];
          acc = t;
        }
        __syncthreads();
        break;
      }
      int e = 0;
      if (a0 != T(0)) e = ilogb(double(a0));
      const double scale = ldexp(1.0, P - e), unit = ldexp(1.0, e - P);
      const long long limit = 1ll << (P + 1), S0 = (long long)(double(a0) * scale);
      ParityAdd own{0, 0};
      if (tid >= from) {
#pragma unroll
        for (int k = 0; k < AVG_EACH; ++k) {
          const double x = fmin(double(v[k]) * scale, double(AVG_CAP)), m = floor(x), f = x - m;
          const long long lo = (long long)m, hi = lo + 1;
          // halfway: to the neighbour that leaves S even
          const ParityAdd one = f == 0.5 ? ParityAdd{(lo & 1) ? hi : lo, (lo & 1) ? lo : hi}
                                         : ParityAdd{f > 0.5 ? hi : lo, f > 0.5 ? hi : lo};
          own = then(own, one);
        }
      }
      ParityAdd scan = own;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const ParityAdd l{__shfl_up(scan.even, o), __shfl_up(scan.odd, o)};
        if (lane >= o) scan = then(l, scan);
      }
      if (lane == 63) wave_total[wave] = scan;
      ParityAdd before{__shfl_up(scan.even, 1), __shfl_up(scan.odd, 1)};
      if (lane == 0) before = ParityAdd{0, 0};
      __syncthreads();
      ParityAdd base{0, 0}, all{0, 0};
      for (int w = 0; w < WAVES; ++w) {
        if (w == wave) base = all;
        all = then(all, wave_total[w]);
      }
      before = then(base, before);
      const long long start = S0 + ((S0 & 1) ? before.odd : before.even);
      const long long end = start + ((start & 1) ? own.odd : own.even);
      const bool cross = tid >= from && (a0 == T(0) ? any : end >= limit);
      const unsigned long long m = __ballot(cross);
      if (lane == 0) first_cross[wave] = m ? wave * 64 + __ffsll(m) - 1 : AVG_THREADS;
      __syncthreads();
      int at = AVG_THREADS;
      for (int w = 0; w < WAVES; ++w) at = min(at, first_cross[w]);
      if (at == AVG_THREADS) {
        if (tid == 0) acc = T(double(S0 + ((S0 & 1) ? all.odd : all.even)) * unit);
      } else if (tid == at) {
        T t = a0 == T(0) ? T(0) : T(double(start) * unit);
#pragma unroll
        for (int k = 0; k < AVG_EACH; ++k) t = t + v[k];
        acc = t;
      }
      from = at + 1;
      __syncthreads();
    }
  }
  __syncthreads();
  if (tid == 0) totals[blockIdx.x] = acc;
}

template <class T> __global__ void k_average_finish(const T* __restrict__ totals, T* __restrict__ out) {
  if (threadIdx.x == 0) {
    const T t0 = totals[0], t1 = totals[1], t2 = totals[2];
    out[0] = out[1] = out[2] = T(0);
    if (t2 > T(0)) {
      out[0] = t0 / t2;
      out[1] = t1 / t2;
      out[2] = t2;
    }
  }
}

__global__ void k_depth_offsets(const int64_t* __restrict__ keys, int64_t n, int count, int* __restrict__ out) {
  int d = blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= count) return;
  out[d] = (int)lower_bound(keys, n, (int64_t)d << 48);
}

// normals.py:46-109: valid splat records compacted, sorted by key (ties in
// record order), reduced per key in that order.
template <class T, class K> void normal_splats(Result<T>& r, int minimum, int maximum, K sentinel) {
  hipStream_t s = r.s;
  const int G = r.G;
  const int64_t records = 54 * (int64_t)G;
  const int blocks = (int)blocks_for(records, 256);
  DArray<int> block_counts(blocks, s), block_offsets(blocks, s), total(1, s);
  hipLaunchKernelGGL(k_normal_splat_count<T>, dim3(blocks), dim3(256), 0, s, (const int*)r.normal_order.data(), G,
                     (const T*)r.position_sums.data(), (const T*)r.normal_sums.data(), (const T*)r.weights.data(),
                     (const T*)r.dw.data(), minimum, maximum, block_counts.data());
  KERNEL_CHECK();
  scan_exclusive_i32(block_counts.data(), block_offsets.data(), blocks, total.data(), s);
  const int64_t valid = read_int(total.data(), s);
  DArray<K> rkeys(valid, s);
  DArray<int> rids(valid, s), heads(valid, s), prefix(valid, s);
  DArray<T> rvals(3 * (size_t)valid, s);
  hipLaunchKernelGGL((k_normal_splat_keys<T, K>), dim3(blocks), dim3(256), 0, s, (const int*)r.normal_order.data(), G,
                     (const T*)r.position_sums.data(), (const T*)r.normal_sums.data(), (const T*)r.weights.data(),
                     (const T*)r.dw.data(), minimum, maximum, (const int*)block_offsets.data(), valid, rkeys.data(),
                     rids.data(), rvals.data());
  KERNEL_CHECK();
  sort_pairs(rkeys.data(), rids.data(), valid, bits_for((uint64_t)sentinel), s);
  mark_heads(rkeys.data(), valid, sentinel, heads.data(), s);
  scan_exclusive_i32(heads.data(), prefix.data(), valid, total.data(), s);
  const int count = valid ? read_int(total.data(), s) : 0;
  DArray<int> head_pos(count, s);
  compact_heads(heads.data(), prefix.data(), valid, head_pos.data(), s);
  r.normal_keys.reset(count, s);
  r.normal_vals.reset(3 * (size_t)count, s);
  if (count) {
    hipLaunchKernelGGL((k_normal_splat_reduce<T, K>), dim3(blocks_for(count, 256)), dim3(256), 0, s,
                       (const K*)rkeys.data(), (const int*)rids.data(), (const T*)rvals.data(), (const int*)head_pos.data(),
                       count, valid, maximum, r.normal_keys.data(), r.normal_vals.data());
    KERNEL_CHECK();
  }
}

template <class T> void stage_normals(Result<T>& r) {
  hipStream_t s = r.s;
  const int G = r.G;
  const int minimum = r.prm.base_depth, maximum = r.prm.depth;
  // order aggregates by first input index (normals.py:190-198)
  {
    DArray<uint64_t> keys(G, s);
    r.normal_order.reset(G, s);
    hipLaunchKernelGGL(k_first_keys, dim3(blocks_for(G, 256)), dim3(256), 0, s, (const int*)r.first_indices.data(), G,
                       keys.data(), r.normal_order.data());
    KERNEL_CHECK();
    sort_pairs_u64(keys.data(), r.normal_order.data(), G, bits_for((uint64_t)r.n), s);
  }
  const uint64_t sentinel = (uint64_t)(maximum + 1) << (3 * maximum);
  if (bits_for(sentinel) <= 32)
    normal_splats<T, uint32_t>(r, minimum, maximum, (uint32_t)sentinel);
  else
    normal_splats<T, uint64_t>(r, minimum, maximum, sentinel);
  // average (normals.py:221-227): contributions here, the serial chain on a
  // side stream (joined before the first use of the average)
  r.average_contrib.reset(3 * (size_t)G, s);
  r.normal_average.reset(3, s);
  r.average_totals.reset(3, s);
  hipLaunchKernelGGL(k_average_contributions<T>, dim3(blocks_for(G, 256)), dim3(256), 0, s,
                     (const int*)r.normal_order.data(), G, (const T*)r.normal_sums.data(), (const T*)r.weights.data(),
                     (const T*)r.dw.data(), r.average_contrib.data());
  KERNEL_CHECK();
  if (!r.side) {
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    r.side = companion_stream(dev, s, 0);
  }
  if (!r.average_done) HIP_CHECK(hipEventCreateWithFlags(&r.average_done, hipEventDisableTiming));
  {
    hipEvent_t ready;
    HIP_CHECK(hipEventCreateWithFlags(&ready, hipEventDisableTiming));
    HIP_CHECK(hipEventRecord(ready, s));
    HIP_CHECK(hipStreamWaitEvent(r.side, ready, 0));
    HIP_CHECK(hipEventDestroy(ready));
  }
  hipLaunchKernelGGL(k_average_chains<T>, dim3(3), dim3(AVG_THREADS), 0, r.side, (const T*)r.average_contrib.data(), G,
                     r.average_totals.data());
  KERNEL_CHECK();
  hipLaunchKernelGGL(k_average_finish<T>, dim3(1), dim3(64), 0, r.side, (const T*)r.average_totals.data(), r.normal_average.data());
  KERNEL_CHECK();
  HIP_CHECK(hipEventRecord(r.average_done, r.side));
  r.average_pending = true;
  // per-depth record offsets (normals.py:17-29, 228-234)
  DArray<int> offsets(maximum + 2, s);
  hipLaunchKernelGGL(k_depth_offsets, dim3(1), dim3(64), 0, s, (const int64_t*)r.normal_keys.data(),
                     (int64_t)r.normal_keys.size(), maximum + 2, offsets.data());
  KERNEL_CHECK();
  r.normal_offsets.resize(maximum + 2);
  read_bytes(r.normal_offsets.data(), offsets.data(), sizeof(int) * (maximum + 2), s);
}

// samples.py:54-88 (_transform), host scalar code shared by the stages
template <class T> int compute_transform(const T* b, double scale, T* t) {
  T width = wmax(b[3] - b[0], wmax(b[4] - b[1], b[5] - b[2])) * T(scale);
  if (!std::isfinite(width) || width <= T(0)) return 1;
  T inv = T(1.0 / double(width));
  t[0] = inv;
  T determinant = inv * (inv * inv);
  t[4] = inv * inv / determinant * T(std::pow(double(determinant), 1.0 / 3.0));
  for (int a = 0; a < 3; ++a) {
    int axis = (a + 1) % 3;
    T origin = (b[axis + 3] + b[axis]) / T(2) - width / T(2);
    t[a + 1] = -origin * inv;
  }
  return 0;
}

#define INSTANTIATE(T)                                                   \
  template void stage_samples<T>(Result<T>&, const T*, const T*);        \
  template void stage_density<T>(Result<T>&);                            \
  template void stage_normals<T>(Result<T>&);                            \
  template int compute_transform<T>(const T*, double, T*);
INSTANTIATE(float)
INSTANTIATE(double)

}  // namespace psr
