// Device code of the vector Maxwell family for gfx950.
//
// Maxwell's equations in second-order curl-curl form on the Yee lattice
// (cuwave/maxwell.py:162-260): electric component c sits half a node up axis
// c, the curl of the pair (k, l) half a node up both axes. A step is a pair
// of launches over the interior nodes: the curl launch writes nu W b of each
// pair point of the node into a scratch (b the pair's curl of u1, W its cell
// weight), the update launch gathers the curls into each component's force
// and writes u2 = -u0 + 2 u1 + minv force, with the adjoint's accumulator
// also the inertia density of u1 against the forward v1
// (cuwave/kernels/maxwell.cu:44-275).
//
// The walls read images, never a ghost: a field node past the wall node reads
// its mirror about it, negated across a conductor; a pair point past the
// wall's half point reads its mirror about that, negated across a magnetic
// wall, the opposite parity, so the gather is the curl's exact transpose.
//
// Layout as in the other families: per-shot arrays keep the shots
// innermost, (component, *np, lanes); a thread holds V neighbouring lanes of
// one interior node and runs every expression lane by lane in the
// reference's operation order, so a lane's bits are those of the one-shot
// arithmetic. The densities a node's lanes produce are summed over the lanes
// into one per-point accumulator.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace cwm {

using cw::at_bytes;
using cw::lanes_at;
using cw::LanesOf;
using cw::put_bytes;

// A thread's place in a component, in bytes: 32 bits in float, where a
// component stays under 4 GiB (the batch's elements are under 2^31), so that
// a tap's load is a scalar base and this register.
template <typename T>
using Place = std::conditional_t<sizeof(T) == 4, uint32_t, uint64_t>;

constexpr int kThreads = 256;

// the grid and the operator constants, by value
template <typename T> struct MxGeom {
  int n[3], np[3], s[3];
  int64_t nodes;  // nodes of one component
  int lanes;
  int conductor;  // Conductor faces, bit 2 axis + side
  int interior;   // interior nodes, every axis 1 .. n - 2
  cw::Div row;    // interior nodes of the fast axis
  cw::Stripes stripes; // 3D
  T sg[4];        // full-radius staggered weights, sg[k - 1]
  T nu;           // 1 / permeability
  T f[3];         // per-axis factors: 1 / dx (curl), dt^2 / dx (update)
};

// the curl scratch row of the pair (k, l), k < l: 3 - k - l in 3D
template <int NDIM> __device__ __forceinline__ constexpr int pair_row(int k, int l) {
  return NDIM == 3 ? 3 - k - l : 0;
}

// node b of an axis of N nodes, past the wall node its mirror about it;
// `neg` across a face of `odd` (bit 0 low, bit 1 high)
__device__ __forceinline__ int node_image(int b, int N, int odd, bool &neg) {
  neg = (b < 1 && (odd & 1)) || (b > N - 2 && (odd & 2));
  return b < 1 ? 2 - b : b > N - 2 ? 2 * (N - 2) - b : b;
}

// half point b (half a node up from node b), past the wall's half point its
// mirror about it; `neg` across a face of `odd`
__device__ __forceinline__ int half_image(int b, int N, int odd, bool &neg) {
  neg = (b < 1 && (odd & 1)) || (b > N - 3 && (odd & 2));
  return b < 1 ? 1 - b : b > N - 3 ? 2 * N - 5 - b : b;
}

// the V lanes of point a + j of the line through element e (node a, element
// stride se), through `node_image` or `half_image`
template <bool HALF, typename Q, typename T>
__device__ __forceinline__ Q imaged(const T *__restrict__ u, int64_t e, int64_t se, int a,
                                    int N, int odd, int j) {
  bool neg;
  const int b = HALF ? half_image(a + j, N, odd, neg) : node_image(a + j, N, odd, neg);
  const Q v = lanes_at<Q>(u, e + (int64_t)(b - a) * se);
  return neg ? -v : v;
}

// the interior node of this thread and its place in a node array (`nat`) and
// in a component (`at`), the first of its V lanes
template <typename T> struct MxNode {
  int A[3];
  int64_t idx;
  int lane0;
  Place<T> nat, at;
};
template <int NDIM, int V, typename T>
__device__ __forceinline__ bool mx_node(const MxGeom<T> &g, MxNode<T> &n) {
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
  n.nat = (Place<T>)at * (Place<T>)sizeof(T);
  n.at = ((Place<T>)at * (Place<T>)g.lanes + (Place<T>)n.lane0) * (Place<T>)sizeof(T);
  return true;
}

// the differences j less 1 - j (j = 1 .. R) of the nodes of component `u`
// along an axis of N nodes and `stride` elements: a wave whose nodes' taps all
// stay inside the walls takes them as they lie, one with a node by a wall
// finds each tap's image
template <int R, typename Q, typename T>
__device__ __forceinline__ void node_differences(const T *__restrict__ u, Place<T> at,
                                                 int64_t stride, int a, int N, int odd, Q *d) {
  if (!__any(a < R || a > N - 2 - R)) {
#pragma unroll
    for (int j = 1; j <= R; ++j)
      d[j - 1] = at_bytes<Q>(u + j * stride, at) - at_bytes<Q>(u + (1 - j) * stride, at);
    return;
  }
  const int64_t e = (int64_t)(at / sizeof(T));
#pragma unroll
  for (int j = 1; j <= R; ++j)
    d[j - 1] = imaged<false, Q>(u, e, stride, a, N, odd, j) -
               imaged<false, Q>(u, e, stride, a, N, odd, 1 - j);
}

// the (k, l) curl at the node's pair point (maxwell.cu:49-73): u_k along l
// and u_l along k, nodes 1 - R .. R away, the first term negated
template <int NDIM, int R, typename Q, typename T>
__device__ __forceinline__ Q curl_of(const MxGeom<T> &g, const T *__restrict__ u,
                                     const MxNode<T> &n, int k, int l) {
  const int64_t comp = g.nodes * g.lanes;
  Q dk[R], dl[R];
  node_differences<R>(u + k * comp, n.at, (int64_t)g.s[l] * g.lanes, n.A[l], g.n[l],
                      g.conductor >> (2 * l), dk);
  node_differences<R>(u + l * comp, n.at, (int64_t)g.s[k] * g.lanes, n.A[k], g.n[k],
                      g.conductor >> (2 * k), dl);
  Q b = (T)0;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    b = b - (g.f[l] * g.sg[j]) * dk[j];
    b = b + (g.f[k] * g.sg[j]) * dl[j];
  }
  return b;
}

// curl_kernel (maxwell.cu:209-239): every pair point of the node off the
// staggered ghosts of its two axes, nu times its cell weight (halved on the
// walls of the axis it does not span) times the curl; MAG reads that product
// per pair point from nu_pair (a designed permeability), and GRAD then takes
// the adjoint curl against the forward one off g_nu, summed over the lanes.
// HBM bounds it: at 162^3, order 4, 8 float lanes it moves 858 MB (by the
// counters; 786 algorithmic) in 253 us, 3.4 TB/s.
template <typename T, int NDIM, int R, int V, bool MAG, bool GRAD>
__global__ void __launch_bounds__(kThreads)
mx_curl(MxGeom<T> g, const T *__restrict__ u1, T *__restrict__ h,
        const T *__restrict__ nu_pair, T *__restrict__ g_nu, const T *__restrict__ v1) {
  using Q = LanesOf<T, V>;
  MxNode<T> n;
  if (!mx_node<NDIM, V>(g, n))
    return;
  const int64_t comp = g.nodes * g.lanes;
#pragma unroll
  for (int k = 0; k < NDIM - 1; ++k)
#pragma unroll
    for (int l = k + 1; l < NDIM; ++l) {
      if (n.A[k] > g.n[k] - 3 || n.A[l] > g.n[l] - 3)
        continue;
      T w = (T)1;
#pragma unroll
      for (int d = 0; d < NDIM; ++d)
        if (d != k && d != l && (n.A[d] == 1 || n.A[d] == g.n[d] - 2))
          w *= (T)0.5;
      const Q b = curl_of<NDIM, R, Q>(g, u1, n, k, l);
      const int row = pair_row<NDIM>(k, l);
      if constexpr (GRAD) {
        const T s = cw::shot_sum(b * curl_of<NDIM, R, Q>(g, v1, n, k, l), g.lanes);
        if (n.lane0 == 0)
          g_nu[row * g.nodes + n.idx] -= s;
      }
      if constexpr (MAG)
        put_bytes(h + row * comp, n.at, Q(at_bytes<T>(nu_pair + row * g.nodes, n.nat) * b));
      else
        put_bytes(h + row * comp, n.at, Q((g.nu * w) * b));
    }
}

// the force on component c (maxwell.cu:171-204): the curls of its pairs
// differenced along the other axis, pair points -R .. R - 1 away, halved on
// a wall node of that axis
template <int NDIM, int R, typename Q, typename T>
__device__ __forceinline__ Q force_on(const MxGeom<T> &g, const T *__restrict__ h,
                                      const MxNode<T> &n, int c) {
  Q force = (T)0;
#pragma unroll
  for (int m = 0; m < NDIM; ++m) {
    if (m == c)
      continue;
    const T *hp = h + pair_row<NDIM>(c < m ? c : m, c < m ? m : c) * g.nodes * g.lanes;
    const int64_t sm = (int64_t)g.s[m] * g.lanes;
    const int odd = ~g.conductor >> (2 * m), a = n.A[m], N = g.n[m];
    Q acc = (T)0;
    if (!__any(a < R + 1 || a > N - 2 - R)) { // as node_differences, of half points
#pragma unroll
      for (int j = 1; j <= R; ++j) {
        acc = acc + g.sg[j - 1] * at_bytes<Q>(hp + (j - 1) * sm, n.at);
        acc = acc - g.sg[j - 1] * at_bytes<Q>(hp - j * sm, n.at);
      }
    } else {
      const int64_t e = (int64_t)(n.at / sizeof(T));
#pragma unroll
      for (int j = 1; j <= R; ++j) {
        acc = acc + g.sg[j - 1] * imaged<true, Q>(hp, e, sm, a, N, odd, j - 1);
        acc = acc - g.sg[j - 1] * imaged<true, Q>(hp, e, sm, a, N, odd, -j);
      }
    }
    if (a == 1 || a == N - 2)
      acc = acc * (T)0.5;
    // u_c enters its pair as +d_m u_c for m < c, as -d_m u_c for m > c
    force = force + ((m < c ? (T)1 : (T)-1) * g.f[m]) * acc;
  }
  return force;
}

// fd_kernel (maxwell.cu:242-274): every component of the node off the
// staggered ghost of its own axis; GRAD adds the inertia density of u1
// against the forward v1, summed over the lanes. HBM bounds it: at 162^3,
// order 4, 8 float lanes it moves 1.83 GB (by the counters) in 362 us, 5.1 TB/s
// (the adjoint 2.49 GB in 447, 5.6).
template <typename T, int NDIM, int R, int V, bool GRAD>
__global__ void __launch_bounds__(kThreads)
mx_update(MxGeom<T> g, const T *__restrict__ minv, const T *__restrict__ h, const T *u0,
          const T *__restrict__ u1, T *u2, T *__restrict__ g_mass, const T *__restrict__ v1,
          T mf, const T *__restrict__ damping, T dt) {
  using Q = LanesOf<T, V>;
  MxNode<T> n;
  if (!mx_node<NDIM, V>(g, n))
    return;
#pragma unroll
  for (int c = 0; c < NDIM; ++c) {
    if (n.A[c] > g.n[c] - 3)
      continue;
    const Q force = force_on<NDIM, R, Q>(g, h, n, c);
    const int64_t comp = c * (g.nodes * g.lanes);
    const T mi = at_bytes<T>(minv + c * g.nodes, n.nat);
    const Q w0 = at_bytes<Q>(u0 + comp, n.at), w1 = at_bytes<Q>(u1 + comp, n.at);
    Q next;
    if (damping) {
      // the damped update (maxwell.cu:257-264), damping nodal
      const T beta = (T)0.5 * mi * damping[n.idx] * dt;
      next = ((T)2 * w1 - w0 * ((T)1 - beta) + mi * force) / ((T)1 + beta);
    } else {
      next = -w0 + (T)2 * w1 + mi * force;
    }
    if constexpr (GRAD) {
      const Q v = at_bytes<Q>(v1 + comp, n.at);
      const T sum = cw::shot_sum(mf * v * (next - (T)2 * w1 + w0), g.lanes);
      if (n.lane0 == 0)
        g_mass[c * g.nodes + n.idx] -= sum;
    }
    put_bytes(u2 + comp, n.at, next);
  }
}

} // namespace cwm
