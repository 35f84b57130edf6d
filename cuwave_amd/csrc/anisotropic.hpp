// Device code of the cell-assembled (anisotropic) elastic family for gfx950.
//
// Collocated displacement components on the nodes, the operator assembled
// cell by cell as -B^T C B with C on the cell (cuwave/anisotropic.py:1-12):
// each interior node gathers, from each of the 2^ndim cells it is a corner
// of, the cell's material g times the row of the one-cell stencil K that
// belongs to its corner, applied to the displacements of the cell's corners
// (cuwave/kernels/anisotropic.cu:72-116, 334-365). A cell takes part while
// both of its corners along every axis are interior nodes, so a traction-free
// face is the natural condition of the interior-cell sum and a clamped one a
// zeroed inertia. Order 2 only: one cell reaches one node each way.
//
// Layout as in the other families: per-shot arrays keep the shots
// innermost, (component, *np, lanes); a thread holds V neighbouring lanes of
// one interior node and runs every expression lane by lane in the
// reference's operation order. K sits in device memory, read with uniform
// (scalar) loads: every index into it is a compile-time constant.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace cwa {

using cw::at_bytes;
using cw::LanesOf;
using cw::put_bytes;

// A thread's place in a component, in bytes: 32 bits where a component stays
// under 4 GiB (the batch's elements are under 2^31), so that a neighbour's
// load is a scalar base and this register.
template <int NDIM, typename T>
using Place = std::conditional_t<sizeof(T) == 4 && (NDIM > 1), uint32_t, uint64_t>;

constexpr int kThreads = 256;

template <typename T> struct AnGeom {
  int n[3], s[3];
  int64_t nodes;  // nodes of one component
  int lanes;
  int interior;   // interior nodes, every axis 1 .. n - 2
  cw::Div row;    // interior nodes of the fast axis
  cw::Stripes stripes; // 3D
  T f;            // the update factor dt^2 (the spacing sits in K)
};

template <int NDIM> constexpr int corners() { return 1 << NDIM; }
template <int NDIM> constexpr int nloc() { return corners<NDIM>() * NDIM; }

// the interior node of this thread, the first of its V lanes and its places in
// a node array and in a component
template <int NDIM, typename T> struct AnNode {
  int A[3];
  int64_t idx;
  int lane0;
  Place<NDIM, T> nat, at;
};
template <int NDIM, int V, typename T>
__device__ __forceinline__ bool an_node(const AnGeom<T> &g, AnNode<NDIM, T> &n) {
  using P = Place<NDIM, T>;
  const int per = g.lanes / V;
  const uint32_t t = (uint32_t)cw::xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const uint32_t i = t >> __builtin_ctz(per);
  if (i >= (uint32_t)g.interior)
    return false;
  n.lane0 = (int)(t & (per - 1)) * V;
  if (NDIM == 3) {
    cw::stripe_node(g.stripes, i, n.A);
  } else {
    uint32_t k = i;
    n.A[0] = 1 + (int)(NDIM == 2 ? cw::quot(g.row, i, k) : i);
    if (NDIM == 2)
      n.A[1] = 1 + (int)k;
  }
  int at = 0;
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    at += n.A[d] * g.s[d];
  n.idx = at;
  n.nat = (P)at * (P)sizeof(T);
  n.at = ((P)at * (P)g.lanes + (P)n.lane0) * (P)sizeof(T);
  return true;
}

// the node steps from a node to corner l of the cell whose low corner is the
// node itself moved by `low` (a bit an axis: one node back)
template <int NDIM, typename T>
__device__ __forceinline__ int corner_step(const AnGeom<T> &g, int low, int l) {
  int off = 0;
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    off += (((l >> d) & 1) - ((low >> d) & 1)) * g.s[d];
  return off;
}

// fd_kernel without damping (anisotropic.cu:367-397): the cell-gathered force
// on every component, then u2 = -u0 + 2 u1 + f minv force. The cells run in
// block order (axis 0 fastest, the cell below the node first), then the
// corners of a cell in the same order, then the components.
//
// In 2D its instructions bound it as much as HBM does: the gather is 64 products
// with K a lane (each a rounding of its own, which the order of the reference
// fixes) and the step moves 405 MB at 1026^2 nodes and 16 float lanes. A wave
// off the walls loads the nodes around once (9 in 2D, where a cell after the
// other reads 16) and gathers without a test a cell.
template <typename T, int NDIM, int V>
__global__ void __launch_bounds__(kThreads)
an_step(AnGeom<T> g, const T *__restrict__ K, const T *__restrict__ minv,
        const T *__restrict__ cell, const T *u0, const T *__restrict__ u1, T *u2,
        const T *__restrict__ damping, T dt) {
  using Q = LanesOf<T, V>;
  constexpr int NL = nloc<NDIM>();
  AnNode<NDIM, T> n;
  if (!an_node<NDIM, V>(g, n))
    return;
  const int64_t comp = g.nodes * g.lanes;
  Q force[NDIM];
#pragma unroll
  for (int i = 0; i < NDIM; ++i)
    force[i] = (T)0;
  bool wall = false;
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    wall |= n.A[d] < 2 || n.A[d] > g.n[d] - 3;
  if (NDIM == 2 && !__any(wall)) {
    Q around[3][3][NDIM]; // [axis 0][axis 1]
    T gc[corners<NDIM>()];
#pragma unroll
    for (int c = 0; c < corners<NDIM>(); ++c)
      gc[c] = at_bytes<T>(cell + corner_step<NDIM>(g, corners<NDIM>() - 1 - c, 0), n.nat);
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int j = 0; j < NDIM; ++j)
          around[r][s][j] = at_bytes<Q>(
              u1 + (j * comp + (int64_t)((r - 1) * g.s[0] + (s - 1) * g.s[1]) * g.lanes), n.at);
#pragma unroll
    for (int c = 0; c < corners<NDIM>(); ++c) {
      const int self = corners<NDIM>() - 1 - c; // the node's corner in the cell
#pragma unroll
      for (int l = 0; l < corners<NDIM>(); ++l)
#pragma unroll
        for (int j = 0; j < NDIM; ++j) {
          const Q uj = around[(c & 1) + (l & 1)][((c >> 1) & 1) + ((l >> 1) & 1)][j];
#pragma unroll
          for (int i = 0; i < NDIM; ++i)
            force[i] = force[i] - (gc[c] * K[(self * NDIM + i) * NL + l * NDIM + j]) * uj;
        }
    }
  } else {
#pragma unroll
    for (int c = 0; c < corners<NDIM>(); ++c) {
      bool inside = true;
#pragma unroll
      for (int d = 0; d < NDIM; ++d) {
        const int e = ((c >> d) & 1) - 1; // the cell's low corner, from the node
        inside &= n.A[d] + e >= 1 && n.A[d] + e <= g.n[d] - 3;
      }
      if (!inside)
        continue;
      const int self = corners<NDIM>() - 1 - c; // the node's corner in the cell
      const T gc = at_bytes<T>(cell + corner_step<NDIM>(g, self, 0), n.nat);
#pragma unroll
      for (int l = 0; l < corners<NDIM>(); ++l) {
        const int64_t off = (int64_t)corner_step<NDIM>(g, self, l) * g.lanes;
#pragma unroll
        for (int j = 0; j < NDIM; ++j) {
          const Q uj = at_bytes<Q>(u1 + (j * comp + off), n.at);
#pragma unroll
          for (int i = 0; i < NDIM; ++i)
            force[i] = force[i] - (gc * K[(self * NDIM + i) * NL + l * NDIM + j]) * uj;
        }
      }
    }
  }
  const T mi = at_bytes<T>(minv, n.nat);
  // with a damping field the damped update (anisotropic.cu:380-389), nodal beta
  const T beta = damping ? (T)0.5 * mi * damping[n.idx] * dt : (T)0;
#pragma unroll
  for (int i = 0; i < NDIM; ++i) {
    const Q w0 = at_bytes<Q>(u0 + i * comp, n.at), w1 = at_bytes<Q>(u1 + i * comp, n.at);
    const Q next = damping ? ((T)2 * w1 - w0 * ((T)1 - beta) + g.f * mi * force[i]) / ((T)1 + beta)
                           : -w0 + (T)2 * w1 + (g.f * mi) * force[i];
    put_bytes(u2 + i * comp, n.at, next);
  }
}

// gradient_kernel (anisotropic_sensitivity.cu:111-156): the inertia density of
// the forward triplet against the adjoint l1 at the node, and the stiffness
// density of the cell whose low corner the node is, the one-cell stencil
// paired between l1 and u1; each summed over the lanes into its accumulator
template <typename T, int NDIM, int V>
__global__ void __launch_bounds__(kThreads)
an_gradient(AnGeom<T> g, const T *__restrict__ K, T *__restrict__ g_mass,
            T *__restrict__ g_cell, const T *__restrict__ u0, const T *__restrict__ u1,
            const T *__restrict__ u2, const T *__restrict__ l1, T mass_factor) {
  using Q = LanesOf<T, V>;
  constexpr int NL = nloc<NDIM>();
  AnNode<NDIM, T> n;
  if (!an_node<NDIM, V>(g, n))
    return;
  const int64_t comp = g.nodes * g.lanes;
  Q acc = (T)0;
#pragma unroll
  for (int i = 0; i < NDIM; ++i)
    acc = acc + at_bytes<Q>(l1 + i * comp, n.at) *
                    (at_bytes<Q>(u2 + i * comp, n.at) - (T)2 * at_bytes<Q>(u1 + i * comp, n.at) +
                     at_bytes<Q>(u0 + i * comp, n.at));
  const T mass = cw::shot_sum(mass_factor * acc, g.lanes);
  bool own = true;
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    own &= n.A[d] <= g.n[d] - 3;
  Q bilinear = (T)0;
  if (own) {
#pragma unroll
    for (int l = 0; l < corners<NDIM>(); ++l) {
      const int64_t lo = (int64_t)corner_step<NDIM>(g, 0, l) * g.lanes;
#pragma unroll
      for (int m = 0; m < corners<NDIM>(); ++m) {
        const int64_t mo = (int64_t)corner_step<NDIM>(g, 0, m) * g.lanes;
#pragma unroll
        for (int i = 0; i < NDIM; ++i)
#pragma unroll
          for (int j = 0; j < NDIM; ++j)
            bilinear = bilinear + (at_bytes<Q>(l1 + (i * comp + lo), n.at) *
                                   K[(l * NDIM + i) * NL + m * NDIM + j]) *
                                      at_bytes<Q>(u1 + (j * comp + mo), n.at);
      }
    }
  }
  // every thread of the node takes part in both sums; one writer a node
  const T stiff = cw::shot_sum(bilinear, g.lanes);
  if (n.lane0 == 0) {
    g_mass[n.idx] -= mass;
    if (own)
      g_cell[n.idx] -= stiff;
  }
}

} // namespace cwa
