// Host-side pieces of the elastic C ABI shared by its translation units: the
// ABI structs turned into the kernels' parameter blocks, and the launchers
// one translation unit per (precision, radius) instantiates.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "../../include/cuwave_amd.h"
#include "elastic.hpp"
#include "elastic_core.hpp"

namespace cwh {
int fail(const std::string &what);
} // namespace cwh

namespace cweh {

using cwh::fail;

inline int hip_status(const char *where) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    fail(std::string(where) + ": " + hipGetErrorString(e));
    return 2;
  }
  return 0;
}

inline int interior_nodes(const cw_elastic_grid &g) {
  int count = 1;
  for (int d = 0; d < g.ndim; ++d)
    count *= g.n[d] - 2;
  return count;
}

// blocks of one thread a node and V lanes
inline int node_blocks(const cw_elastic_grid &g, int V) {
  const int64_t threads = (int64_t)interior_nodes(g) * (g.lanes / V);
  return (int)((threads + cwe::kThreads - 1) / cwe::kThreads);
}

// the nodes of each axis whose stresses no closure, traction face or PML
// memory reaches: [lo, hi), the memories' reach R further in the adjoint
inline void deep_range(const cw_elastic_grid &g, const cw_elastic_layer &p, int d, int *lo,
                       int *hi) {
  const int R = g.order / 2, ext = p.phase ? R : 0;
  const int band = g.closure[0] > g.closure[1] ? g.closure[0] : g.closure[1];
  const int in = band > R ? band : R;
  const int low = p.lo[d] && p.lo[d] + ext > in ? p.lo[d] + ext : in;
  const int high = p.hi[d] && p.hi[d] + ext > in + 1 ? p.hi[d] + ext : in + 1;
  *lo = 1 + low;
  *hi = g.n[d] - 1 - high;
}

// The shape of a 2D core block: lanes a thread and threads, no lanes where the
// pair takes every step. A core block wants 32 columns: the lanes a thread are
// the fewest that give them (fewer lanes leave more waves a SIMD, more columns a
// smaller halo share; 16 lanes at order 4: two lanes a thread 232 us, one 240,
// four 245), two at most from order 6 on (the rings of four spill, and of two
// doubles), and past 16 lanes blocks of 512 threads.
struct CoreShape {
  int vc, nt;
};
inline CoreShape core_shape(const cw_elastic_grid &g) {
  const int size = g.dtype ? 8 : 4;
  const int most = g.order > 4 ? (size == 4 ? 2 : 1) : 16 / size;
  if (g.ndim != 2)
    return {0, 0};
  if (g.lanes <= 8)
    return {1, 256};
  if (g.lanes <= 32)
    return most > 1 ? CoreShape{2, g.lanes == 16 ? 256 : 512} : CoreShape{0, 0};
  return most > 2 ? CoreShape{4, 512} : CoreShape{0, 0};
}

// The box the core steps, false where the pair alone takes the step: where a
// block's columns are under 6 R (a third of its stresses would serve no
// update), where the core holds less than half the nodes (the frame's two
// launches cost what the pair's do), or where a field passes the 4 GiB a 32-bit
// offset reaches.
inline bool core_box(const cw_elastic_grid &g, const cw_elastic_layer &p, const CoreShape &shape,
                     cwe::ElBox *box) {
  if (!shape.vc)
    return false;
  const int R = g.order / 2, per = g.lanes / shape.vc, cols = shape.nt / per;
  if (cols < 6 * R || per > cwe::kHaloPer ||
      (uint64_t)g.np[0] * g.np[1] * g.lanes * (g.dtype ? 8 : 4) >= 1ull << 32)
    return false;
  int lo[2], hi[2];
  for (int d = 0; d < 2; ++d)
    deep_range(g, p, d, &lo[d], &hi[d]);
  box->y0 = lo[0] + R;
  box->y1 = hi[0] - R;
  box->x0 = lo[1] + R;
  box->x1 = hi[1] - R;
  const int64_t h = box->y1 - box->y0, w = box->x1 - box->x0;
  if (h < 4 * R || w < 4 * R || 2 * h * w < (int64_t)interior_nodes(g))
    return false;
  // chunks for 1024 blocks, a third more than the card holds at once where its
  // registers allow three a CU (265 us for 512 blocks, 262 for 1024, at 16 lanes
  // of 1058 x 2114 nodes and order 4), of at least 8 rows (4 and 16 took 23.0
  // and 25 us against 22.5 on 323 x 457)
  const int use = cols - 2 * R;
  box->nx = (int)((w + use - 1) / use);
  const int want = (1024 + box->nx - 1) / box->nx;
  const int chunk = (int)((h + want - 1) / want);
  box->chunk = chunk < 8 ? 8 : chunk;
  box->ny = (int)((h + box->chunk - 1) / box->chunk);
  return true;
}

// the kernels' geometry with the per-axis factors `f` (1 / dx for the
// strains, dt^2 / dx for the update)
template <typename T>
cwe::ElGeom<T> make_elgeom(const cw_elastic_grid &gr, const T *rows, const double *f) {
  cwe::ElGeom<T> g{};
  const int nd = gr.ndim;
  int64_t stride = 1;
  for (int d = 2; d >= 0; --d) {
    g.n[d] = d < nd ? gr.n[d] : 1;
    g.np[d] = d < nd ? gr.np[d] : 1;
  }
  for (int d = nd - 1; d >= 0; --d) {
    g.s[d] = (int)stride;
    stride *= g.np[d];
  }
  for (int d = nd; d < 3; ++d)
    g.s[d] = 0;
  g.nodes = stride;
  g.lanes = gr.lanes;
  g.nbatch = gr.nbatch;
  g.clamped = gr.clamped;
  g.nc = gr.closure[0];
  g.hc = gr.closure[1];
  g.nspan = gr.closure[2];
  g.hspan = gr.closure[3];
  g.interior = interior_nodes(gr);
  for (int k = 0; k < 4; ++k)
    g.sg[k] = (T)gr.stag[k];
  g.lam = (T)gr.lame;
  g.mu = (T)gr.shear;
  for (int d = 0; d < 3; ++d)
    g.f[d] = d < nd ? (T)f[d] : (T)0;
  g.rows = rows;
  return g;
}

template <typename T> cwe::ElLayer<T> make_ellayer(const cw_elastic_layer &l, int ndim) {
  cwe::ElLayer<T> p{};
  for (int d = 0; d < 3; ++d) {
    const bool lined = d < ndim && l.lo[d] + l.hi[d] > 0;
    p.lo[d] = lined ? l.lo[d] : 0;
    p.hi[d] = lined ? l.hi[d] : 0;
    p.aux[d] = lined ? (T *)l.memory[d] : nullptr;
    p.profile[d] = lined ? (const T *)l.profile[d] : nullptr;
  }
  p.phase = l.phase;
  return p;
}

template <typename T, int NDIM, int R>
int elastic_step(const cw_elastic_step_args &a, hipStream_t stream);
template <typename T, int NDIM, int R>
int elastic_gradient(const cw_elastic_gradient_args &a, hipStream_t stream);

} // namespace cweh
