// Marching cubes on a uniform model-space grid (meshing.py:150-280): the
// library's case table and the slab-wise extraction state (psr_mesh.hip).
#pragma once
#include "psr_common.h"

#include <cstdint>

namespace psr {

constexpr int MC_MAX_TRIANGLES = 12;

// Triangles of each of the 256 corner-sign cases: count[code] triangles, each
// three cube edges (edges[code][3 t + k]).
struct McTable {
  int8_t count[256];
  int8_t edges[256][3 * MC_MAX_TRIANGLES];
};
const McTable& mc_table();

// A uniform model-space grid: node (x, y, z) at lower + step * node.
struct MeshGrid {
  int nx, ny, nz;
  float lo[3], hi[3], step[3];
};

// meshing.py:37-41 and :88-94 (lower + step * node, clamped to the box),
// rounded after the product and after the sum
__device__ __forceinline__ void node_point(const MeshGrid& g, int x, int y, int z, float* out) {
  const int c[3] = {x, y, z};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float p = g.lo[a] + g.step[a] * float(c[a]);
    out[a] = fminf(fmaxf(p, g.lo[a]), g.hi[a]);
  }
}

__device__ __forceinline__ void cell_xyz(const MeshGrid& g, int cell, int& x, int& y, int& z) {
  const int cy = g.ny - 1, cz = g.nz - 1;
  x = cell / (cy * cz);
  y = (cell / cz) % cy;
  z = cell % cz;
}

template <class T> struct Result;
// A reconstruction's value less *iso (device) at grid nodes [first plane
// start, n nodes, z fastest], or at the eight corners of n / 8 cells: the
// numbers evaluate_field(...) - iso gives at the nodes' points.
void mesh_values(const Result<float>& r, const MeshGrid& g, int start, const int* cells, int64_t n, const float* iso, float* values,
                 hipStream_t s);

struct McState;
McState* mc_create(const int shape[3], const float lower[3], const float upper[3], hipStream_t s);
void mc_free(McState* m);
// nodes of planes [start, start + width] (all y, z): width + 1 planes
int64_t mc_slab_nodes(const McState& m, int start, int width);
void mc_slab_points(McState& m, int start, int width, float* out);
// classify the cells of planes [start, start + width) from the slab's values
void mc_slab_values(McState& m, int start, int width, const float* values);
// the same for every cell of the grid, `slab` planes of cells at a time, from
// a reconstruction's own values
void mc_field_values(McState& m, const Result<float>& r, const float* iso, int slab);
// its values at the selected cells' corners
void mc_field_corners(McState& m, const Result<float>& r, const float* iso, float* values);
// count and list the crossing cells (ascending index); *invalid != 0 when a
// classified value was not finite
int mc_select(McState& m, int* invalid);
void mc_corner_points(McState& m, float* out);
void mc_triangulate(McState& m, const float* corner_values, int* V, int* T);
void mc_copy(const McState& m, float* vertices, int* indices);
void mc_vertex_vjp(const McState& m, const float* corner_values, const float* grad_vertices, float* grad_values);

}  // namespace psr
