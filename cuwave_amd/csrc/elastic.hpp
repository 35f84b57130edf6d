// Device code of the elastic (staggered displacement) path for gfx950.
//
// Isotropic elasticity on a staggered grid (cuwave/elastic.py:1-10):
// displacement component c sits half a node up axis c, the normal strains on
// the nodes, the shear (k, l) half a node up both axes. A step is a pair of
// launches over the interior nodes: the stress launch forms the strains of
// u1 and writes the stresses (and, in the adjoint pair, the stiffness
// densities), the update launch takes the divergence of the stresses into
// u2 (and the inertia density). A convolutional PML folds into both
// launches through a memory per lined axis. The walls close with the
// staggered summation-by-parts rows of Prochnow et al. 2017, read from a
// table the caller passes.
//
// Layout as in the pressure path: per-shot arrays carry the shots
// innermost, (component, *np, lanes); a thread holds V neighbouring lanes of
// one node and runs every expression lane by lane in the reference's
// operation order (cuwave/kernels/elastic.cu:121-600, 754-853;
// cuwave/kernels/common.cuh:152-298), so a lane's bits are those of the
// one-shot arithmetic. The densities a node's lanes produce are summed over
// the lanes (cw::shot_sum) into one per-node accumulator.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace cwe {

using cw::at_bytes;
using cw::fmat;
using cw::lanes_at;
using cw::lanes_put;
using cw::LanesOf;
using cw::put_bytes;

constexpr int kThreads = 256;

template <typename T> struct Tiny;
template <> struct Tiny<float> {
  static constexpr float value = 1.17549435e-38f;
};
template <> struct Tiny<double> {
  static constexpr double value = 2.2250738585072014e-308;
};

// the grid, the operator and the material constants, by value
template <typename T> struct ElGeom {
  int n[3], np[3], s[3];
  int64_t nodes;          // nodes of one component
  int lanes, nbatch;
  int clamped;            // faces held at zero, bit 2 axis + side
  int nc, hc, nspan, hspan; // closure rows and the points they read
  int interior;           // interior nodes, every axis 1 .. n - 2
  T sg[4];                // full-radius staggered weights, sg[k - 1]
  T lam, mu;              // Lame parameters
  T f[3];                 // per-axis factors: 1 / dx (stress), dt^2 / dx (update)
  const T *rows;          // node closure rows (nc x nspan), then half rows (hc x hspan)
};

// the PML fold: per lined axis (lo + hi > 0) its memory and profile
template <typename T> struct ElLayer {
  T *aux[3];              // (rows, slab, lanes)
  const T *profile[3];    // (4, n[d]): a, b at nodes, then at half points
  int lo[3], hi[3];
  int phase;              // 0 forward; 1 / 2 the adjoint reads block 0 / 2 ndim
};

template <int NDIM>
__device__ __forceinline__ constexpr int stress_row(int c, int e) {
  if (c == e)
    return c;
  const int k = c < e ? c : e, l = c < e ? e : c;
  return NDIM == 3 ? NDIM + 3 - k - l : 2;
}

template <int NDIM> constexpr int nvoigt() { return NDIM + NDIM * (NDIM - 1) / 2; }

template <typename T>
__device__ __forceinline__ bool clamped_face(const ElGeom<T> &g, int d, int side) {
  return (g.clamped >> (2 * d + side)) & 1;
}

// the slab row of node a of an axis (rows lo off the low wall, hi off the
// high one), -1 off the slab; its index in the axis' memory
__device__ __forceinline__ int64_t slab_at(int a, int N, int lo, int hi, bool slow,
                                           int64_t plane, int64_t off) {
  const int row = cw::slab_row(a, N, lo, hi);
  if (row < 0)
    return -1;
  return slow ? (int64_t)row * plane + off : off * (int64_t)(lo + hi) + row;
}

// A thread's place in a component of a field or of the stresses, in bytes: 32
// bits where a component can't pass 4 GiB (the stresses' element count is
// under 2^31), so that a load takes a scalar base and this one register and a
// tap's distance costs no vector instruction.
template <int NDIM, typename T>
using Place = std::conditional_t<NDIM == 3 || (NDIM == 2 && sizeof(T) == 4), uint32_t, uint64_t>;

// A line of points a derivative reads: a field component (or a stress row)
// along an axis, and optionally through the PML memory (the value coef *
// (base + memory) of the reference's Memory accessor,
// cuwave/kernels/common.cuh:421-437).
template <typename T, typename Off> struct Line {
  const T *p;        // field or stresses (the same for every thread)
  Off off;           // the thread's place in a component
  int64_t comp, step; // elements between components, and a step of the axis
  int lanes;
  int e;             // the axis
  bool stress;       // rows by stress_row(k, e)
  bool memory;
  const T *aux;      // offset to the thread's first lane
  const T *profile;
  int64_t size, plane, slab;
  int row0, a, lo, hi, N;
  bool own_half, slow;
};

// through the PML memory: the value `base` read j points away
template <typename Q, typename T, typename Off>
__device__ __forceinline__ Q through_memory(const Line<T, Off> &L, int k, int j, const Q &base) {
  const int at = L.a + j;
  const int64_t i = slab_at(at, L.N, L.lo, L.hi, L.slow, L.plane, L.slab);
  if (i < 0)
    return Q((T)0);
  const bool half = (k == L.e) == L.own_half;
  const T coef = L.profile[(half ? 2 * L.N : 0) + at];
  return coef * (base + lanes_at<Q>(L.aux, ((int64_t)(L.row0 + k) * L.size + i) * L.lanes));
}

// the point j steps away, j the same for every thread ...
template <int NDIM, typename Q, typename T, typename Off>
__device__ __forceinline__ Q line_at(const Line<T, Off> &L, int k, int j) {
  const int row = L.stress ? stress_row<NDIM>(k, L.e) : k;
  const Q base = at_bytes<Q>(L.p + (row * L.comp + j * L.step), L.off);
  return L.memory ? through_memory(L, k, j, base) : base;
}
// ... and j the thread's own
template <int NDIM, typename Q, typename T, typename Off>
__device__ __forceinline__ Q line_var(const Line<T, Off> &L, int k, int j) {
  const int row = L.stress ? stress_row<NDIM>(k, L.e) : k;
  const Q base = at_bytes<Q>(L.p + row * L.comp,
                             L.off + (Off)j * (Off)(L.step * (int64_t)sizeof(T)));
  return L.memory ? through_memory(L, k, j, base) : base;
}

template <typename T, typename Off>
__device__ __forceinline__ Line<T, Off> field_line(const T *p, Off off, const ElGeom<T> &g,
                                                   int d) {
  Line<T, Off> L{};
  L.p = p;
  L.off = off;
  L.comp = g.nodes * g.lanes;
  L.step = (int64_t)g.s[d] * g.lanes;
  L.lanes = g.lanes;
  L.e = d;
  return L;
}

// ------------------------------------------- staggered SBP derivatives
// closure rows off a wall (cuwave/kernels/common.cuh:214-242): the row's span
// is read four points at a time (past its end the last point again, the term
// dropped), so that a wall node waits on memory once for four points and not
// once for each
template <int NDIM, typename Q, typename T, typename At>
__device__ __forceinline__ Q closure_row(const T *row, int span, bool low, At at) {
  Q acc((T)0);
  for (int m0 = 0; m0 < span; m0 += 4) {
    T w[4];
    Q v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + i < span ? m0 + i : span - 1;
      w[i] = row[m];
      v[i] = at(m);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Q term = w[i] * v[i];
      acc = m0 + i >= span ? acc : low ? acc + term : acc - term;
    }
  }
  return acc;
}

template <int NDIM, typename Q, typename T, typename Off>
__device__ Q node_rows(const ElGeom<T> &g, const Line<T, Off> &L, int k, int lo, int hi) {
  const bool low = lo < g.nc;
  return closure_row<NDIM, Q>(g.rows + (low ? lo : hi) * g.nspan, g.nspan, low, [&](int m) {
    return line_var<NDIM, Q>(L, k, low ? m - lo : hi - 1 - m);
  });
}

template <int NDIM, typename Q, typename T, typename Off>
__device__ Q half_rows(const ElGeom<T> &g, const Line<T, Off> &L, int k, int lo, int hi) {
  const bool low = lo < g.hc;
  return closure_row<NDIM, Q>(g.rows + g.nc * g.nspan + (low ? lo : hi) * g.hspan, g.hspan, low,
                              [&](int m) {
                                return line_var<NDIM, Q>(L, k, low ? m - lo : hi + 1 - m);
                              });
}

// the stencils away from the walls, at a node (h = 0, of half-point values)
// or at a half point (h = 1, of nodal ones)
template <int NDIM, int R, typename Q, typename T, typename Off>
__device__ __forceinline__ Q inner_derivative(const ElGeom<T> &g, const Line<T, Off> &L, int k,
                                              int h) {
  Q acc((T)0);
#pragma unroll
  for (int q = 1; q <= R; ++q)
    acc += g.sg[q - 1] * (line_at<NDIM, Q>(L, k, q - 1 + h) - line_at<NDIM, Q>(L, k, h - q));
  return acc;
}
template <int NDIM, int R, typename Q, typename T, typename Off>
__device__ __forceinline__ Q inner_divergence(const ElGeom<T> &g, const Line<T, Off> &L, int k,
                                              int h) {
  Q acc((T)0);
#pragma unroll
  for (int q = 1; q <= R; ++q) {
    acc += g.sg[q - 1] * line_at<NDIM, Q>(L, k, q - 1 + h);
    acc -= g.sg[q - 1] * line_at<NDIM, Q>(L, k, h - q);
  }
  return acc;
}

// whether a wall of axis e is near: whether a derivative or divergence along
// it may be a closure row, or one that is not there
template <typename T>
__device__ __forceinline__ bool near_wall(const ElGeom<T> &g, int a, int e) {
  const int rows = g.nc > g.hc ? g.nc : g.hc, band = rows > 1 ? rows : 1;
  return a - 1 < band || g.n[e] - 3 - a < band;
}

// d/dx at node a of a half-point field (common.cuh:247-258)
template <int NDIM, int R, typename Q, typename T, typename Off>
__device__ __forceinline__ Q node_derivative(const ElGeom<T> &g, const Line<T, Off> &L, int k, int a,
                                             int N) {
  const int lo = a - 1, hi = N - 2 - a;
  if (lo < g.nc || hi < g.nc)
    return node_rows<NDIM, Q>(g, L, k, lo, hi);
  return inner_derivative<NDIM, R, Q>(g, L, k, 0);
}

// d/dx at half point a of a nodal field (common.cuh:261-271)
template <int NDIM, int R, typename Q, typename T, typename Off>
__device__ __forceinline__ Q half_derivative(const ElGeom<T> &g, const Line<T, Off> &L, int k, int a,
                                             int N) {
  const int lo = a - 1, hi = N - 3 - a;
  if (lo < g.hc || hi < g.hc)
    return half_rows<NDIM, Q>(g, L, k, lo, hi);
  return inner_derivative<NDIM, R, Q>(g, L, k, 1);
}

// the divergence of a nodal stress at half point a (common.cuh:276-288)
template <int NDIM, int R, typename Q, typename T, typename Off>
__device__ __forceinline__ Q node_divergence(const ElGeom<T> &g, const Line<T, Off> &L, int k, int a,
                                             int N) {
  const int lo = a - 1, hi = N - 3 - a;
  if (lo < g.hc || hi < g.hc)
    return half_rows<NDIM, Q>(g, L, k, lo, hi);
  return inner_divergence<NDIM, R, Q>(g, L, k, 1);
}

// the divergence of a half-point stress at node a (common.cuh:292-304)
template <int NDIM, int R, typename Q, typename T, typename Off>
__device__ __forceinline__ Q half_divergence(const ElGeom<T> &g, const Line<T, Off> &L, int k, int a,
                                             int N) {
  const int lo = a - 1, hi = N - 2 - a;
  if (lo < g.nc || hi < g.nc)
    return node_rows<NDIM, Q>(g, L, k, lo, hi);
  return inner_divergence<NDIM, R, Q>(g, L, k, 0);
}

// -------------------------------------------------- strains and stresses
template <int NDIM, typename T>
__device__ __forceinline__ bool traction_zero(const ElGeom<T> &g, const int *A, int d) {
  return (A[d] == 1 && !clamped_face(g, d, 0)) || (A[d] == g.n[d] - 2 && !clamped_face(g, d, 1));
}

template <int NDIM, typename T>
__device__ __forceinline__ int zeroed_axes(const ElGeom<T> &g, const int *A) {
  int zeroed = 0;
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    if (traction_zero<NDIM>(g, A, d))
      zeroed |= 1 << d;
  return zeroed;
}

// the derivative of u_k along axis e at its strain point, zero where there is
// none (a traction wall's normal strain, a shear point past the last);
// strain_term (elastic.cu:417-431) is f[e] times it
template <int NDIM, int R, typename Q, typename T, typename L>
__device__ __forceinline__ Q strain_derivative(const ElGeom<T> &g, const L &line, int k, int e,
                                               const int *A) {
  if (k == e) {
    if (traction_zero<NDIM>(g, A, e))
      return Q((T)0);
    return node_derivative<NDIM, R, Q>(g, line, e, A[e], g.n[e]);
  }
  if (A[k] > g.n[k] - 3 || A[e] > g.n[e] - 3)
    return Q((T)0);
  return half_derivative<NDIM, R, Q>(g, line, k, A[e], g.n[e]);
}

// every derivative of u, D[k][e] = d u_k / d x_e: an axis with no wall near
// takes its NDIM derivatives in one branch, so that the thread waits on memory
// once for their taps and not once for each derivative. Latency bounds the
// pair (a third of the instructions issued that could be): with the updates'
// divergences and the layers' memories taken likewise, an update of 107 x 120 x
// 131 with two shots went from 150 to 101 us and 136 to 91 registers, the
// stresses of the same step from 116 to 98 us.
template <int NDIM, int R, typename Q, typename T, typename Off>
__device__ __forceinline__ void derivatives(const ElGeom<T> &g, const T *u, Off off, const int *A,
                                            Q (*D)[NDIM]) {
#pragma unroll
  for (int e = 0; e < NDIM; ++e) {
    const auto line = field_line(u, off, g, e);
    if (near_wall(g, A[e], e)) {
#pragma unroll
      for (int k = 0; k < NDIM; ++k)
        D[k][e] = strain_derivative<NDIM, R, Q>(g, line, k, e, A);
    } else {
#pragma unroll
      for (int k = 0; k < NDIM; ++k)
        D[k][e] = inner_derivative<NDIM, R, Q>(g, line, k, k != e);
#pragma unroll
      for (int k = 0; k < NDIM; ++k)
        if (k != e && A[k] > g.n[k] - 3)
          D[k][e] = Q((T)0);
    }
  }
}

// the normal strains of u at a node, zero on a traction wall (elastic.cu:121-141)
template <int NDIM, int R, typename Q, typename T, typename Off>
__device__ __forceinline__ int normal_strains(const ElGeom<T> &g, const T *u, Off off,
                                              const int *A, Q *eps) {
  int zeroed = 0;
#pragma unroll
  for (int d = 0; d < NDIM; ++d) {
    if (traction_zero<NDIM>(g, A, d)) {
      eps[d] = Q((T)0);
      zeroed |= 1 << d;
    } else {
      eps[d] = g.f[d] * node_derivative<NDIM, R, Q>(g, field_line(u, off, g, d), d, A[d], g.n[d]);
    }
  }
  return zeroed;
}

// the Lame parameter condensed over the traction-free axes (elastic.cu:145-154)
template <int NDIM, typename T>
__device__ __forceinline__ T condensed_lame(const ElGeom<T> &g, int zeroed) {
  T lam = g.lam;
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    if ((zeroed >> d) & 1)
      lam = (T)2.f * lam * g.mu / (lam + (T)2.f * g.mu);
  return lam;
}

// the engineering shear strain (k, l) at its point (elastic.cu:159-170)
template <int NDIM, int R, typename Q, typename T, typename Off>
__device__ __forceinline__ Q shear_strain(const ElGeom<T> &g, const T *u, Off off, int k, int l,
                                          const int *A) {
  const Q dk = half_derivative<NDIM, R, Q>(g, field_line(u, off, g, k), l, A[k], g.n[k]);
  const Q dl = half_derivative<NDIM, R, Q>(g, field_line(u, off, g, l), k, A[l], g.n[l]);
  return fmat(g.f[k], dk, g.f[l] * dl);
}

template <typename T>
__device__ __forceinline__ bool shear_point(const ElGeom<T> &g, int k, int l, const int *A) {
  return A[k] <= g.n[k] - 3 && A[l] <= g.n[l] - 3;
}

// every strain of u from its derivatives D[k][e] = d u_k / d x_e
// (elastic.cu:216-233)
template <int NDIM, typename Q, typename T>
__device__ __forceinline__ void strains_of(const ElGeom<T> &g, const Q (*D)[NDIM], const int *A,
                                           Q *eps) {
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    eps[d] = traction_zero<NDIM>(g, A, d) ? Q((T)0) : g.f[d] * D[d][d];
#pragma unroll
  for (int k = 0; k < NDIM - 1; ++k)
#pragma unroll
    for (int l = k + 1; l < NDIM; ++l)
      eps[stress_row<NDIM>(k, l)] =
          shear_point(g, k, l, A) ? fmat(g.f[k], D[l][k], g.f[l] * D[k][l]) : Q((T)0);
}

// the stresses of the strains (elastic.cu:236-263); the shear gamma of the
// pair points comes prepared (`shear`: the node's pair rows of prep)
template <int NDIM, typename Q, typename T>
__device__ __forceinline__ void stress_of(const ElGeom<T> &g, const Q *eps, int zeroed, T gn,
                                          const T *shear, const int *A, Q *sig) {
  const T lam = condensed_lame<NDIM>(g, zeroed);
  Q tr((T)0);
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    tr += eps[d];
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    sig[d] = ((zeroed >> d) & 1) ? Q((T)0) : gn * ((T)2.f * g.mu * eps[d] + lam * tr);
#pragma unroll
  for (int k = 0; k < NDIM - 1; ++k)
#pragma unroll
    for (int l = k + 1; l < NDIM; ++l) {
      const int v = stress_row<NDIM>(k, l);
      sig[v] = shear_point(g, k, l, A) ? shear[v - NDIM] * g.mu * eps[v] : Q((T)0);
    }
}

// the divergence of the stresses of component c along axis e at its point;
// divergence_term (elastic.cu:434-442) is f[e] times it
template <int NDIM, int R, typename Q, typename T, typename L>
__device__ __forceinline__ Q stress_divergence(const ElGeom<T> &g, const L &line, int c, int e,
                                               int row, const int *A) {
  if (c == e)
    return node_divergence<NDIM, R, Q>(g, line, c, A[c], g.n[c]);
  return half_divergence<NDIM, R, Q>(g, line, row, A[e], g.n[e]);
}

// the normal-strain energy form of two strain sets (elastic.cu:339-351)
template <int NDIM, typename Q, typename T>
__device__ __forceinline__ Q normal_form(const ElGeom<T> &g, const Q *ea, const Q *eb, int zeroed) {
  const T lam = condensed_lame<NDIM>(g, zeroed);
  Q tra((T)0), trb((T)0), dot((T)0);
#pragma unroll
  for (int d = 0; d < NDIM; ++d) {
    tra += ea[d];
    trb += eb[d];
    dot += ea[d] * eb[d];
  }
  return (T)2.f * g.mu * dot + lam * tra * trb;
}

// ------------------------------------------------------------ the pml fold
template <int NDIM, typename T>
__device__ __forceinline__ bool in_slab(const ElGeom<T> &g, int a, int e, int lo, int hi, int ext) {
  return (lo && a - 1 < lo + ext) || (hi && g.n[e] - 2 - a < hi + ext);
}

template <int NDIM, typename T>
__device__ __forceinline__ void slab_geometry(const ElGeom<T> &g, int e, int lo, int hi,
                                              const int *A, int64_t *plane, int64_t *size,
                                              int64_t *off) {
  int64_t p = 1, o = 0;
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    if (d != e) {
      p *= g.np[d];
      o = o * g.np[d] + A[d];
    }
  *plane = p;
  *size = p * (int64_t)(lo + hi);
  *off = o;
}

// the stresses of the memory strains t of axis e (elastic.cu:445-467)
template <int NDIM, typename Q, typename T>
__device__ __forceinline__ void add_stress(const ElGeom<T> &g, Q *sig, T gn, const T *shear,
                                           int e, const Q *t, const int *A) {
  const int zeroed = zeroed_axes<NDIM>(g, A);
  if (!((zeroed >> e) & 1)) {
    const T lam = condensed_lame<NDIM>(g, zeroed);
    const Q gg = gn * t[e];
#pragma unroll
    for (int d = 0; d < NDIM; ++d)
      if (!((zeroed >> d) & 1))
        sig[d] += gg * ((d == e ? (T)2.f * g.mu : (T)0) + lam);
  }
#pragma unroll
  for (int k = 0; k < NDIM; ++k)
    if (k != e && A[k] <= g.n[k] - 3 && A[e] <= g.n[e] - 3) {
      const int v = stress_row<NDIM>(k, e);
      sig[v] += shear[v - NDIM] * g.mu * t[k];
    }
}

// the strain memory of axis e (elastic.cu:486-528), D[k] = d u_k / d x_e
template <int NDIM, int R, int V, int e, typename T, typename Off>
__device__ __forceinline__ void stress_memory(const ElGeom<T> &g, const ElLayer<T> &P, const T *u,
                                              const LanesOf<T, V> (*D)[NDIM], T gn,
                                              const T *shear, Off place, int lane0, const int *A,
                                              LanesOf<T, V> *sig) {
  using Q = LanesOf<T, V>;
  const int a = A[e], lo = P.lo[e], hi = P.hi[e];
  if (!(lo + hi) || !in_slab<NDIM>(g, a, e, lo, hi, P.phase ? R : 0))
    return;
  int64_t plane, size, off;
  slab_geometry<NDIM>(g, e, lo, hi, A, &plane, &size, &off);
  const int N = g.n[e];
  const T *prof = P.profile[e];
  Q q[3];
  if (P.phase) {
    Line<T, Off> h = field_line(u, place, g, e);
    h.memory = true;
    h.aux = P.aux[e] + lane0;
    h.profile = prof;
    h.size = size;
    h.plane = plane;
    h.slab = off;
    h.row0 = NDIM;
    h.a = a;
    h.lo = lo;
    h.hi = hi;
    h.N = N;
    h.own_half = true;
    h.slow = e < NDIM - 1;
#pragma unroll
    for (int k = 0; k < NDIM; ++k)
      q[k] = g.f[e] * strain_derivative<NDIM, R, Q>(g, h, k, e, A);
  } else {
    const int64_t t = slab_at(a, N, lo, hi, e < NDIM - 1, plane, off);
    T *aux = P.aux[e] + lane0;
    // the rows read before any is written: one wait for all
    const T pn = prof[N + a], dn = prof[a], ph = prof[3 * N + a], dh = prof[2 * N + a];
    Q m[NDIM];
#pragma unroll
    for (int k = 0; k < NDIM; ++k)
      m[k] = lanes_at<Q>(aux, ((int64_t)k * size + t) * g.lanes);
#pragma unroll
    for (int k = 0; k < NDIM; ++k) {
      q[k] = (k == e ? pn : ph) * m[k] + (k == e ? dn : dh) * (g.f[e] * D[k][e]);
      lanes_put(aux, ((int64_t)k * size + t) * g.lanes, q[k]);
    }
  }
  add_stress<NDIM>(g, sig, gn, shear, e, q, A);
}

// the divergence memories of axis e (elastic.cu:532-573) into the components'
// updates, D[c] the divergences of the axis; `on`: the components that have
// their point here
template <int NDIM, int R, int V, int e, typename T, typename Off>
__device__ __forceinline__ void force_memory(const ElGeom<T> &g, const ElLayer<T> &P,
                                             const T *sigma, const LanesOf<T, V> (*D)[NDIM],
                                             const LanesOf<T, V> *w1, const T *mi, const bool *on,
                                             Off place, int lane0, const int *A,
                                             LanesOf<T, V> *next) {
  using Q = LanesOf<T, V>;
  const int a = A[e], lo = P.lo[e], hi = P.hi[e];
  if (!(lo + hi))
    return;
  if (!in_slab<NDIM>(g, a, e, lo, hi, P.phase ? R : 0)) {
#pragma unroll
    for (int c = 0; c < NDIM; ++c)
      next[c] += mi[c] * Q((T)0);
    return;
  }
  int64_t plane, size, off;
  slab_geometry<NDIM>(g, e, lo, hi, A, &plane, &size, &off);
  const int N = g.n[e];
  const bool slow = e < NDIM - 1;
  const int64_t t = slab_at(a, N, lo, hi, slow, plane, off);
  const T *prof = P.profile[e];
  T *aux = P.aux[e] + lane0;
  if (P.phase) {
    Line<T, Off> k = field_line(sigma, place, g, e);
    k.stress = true;
    k.memory = true;
    k.aux = aux;
    k.profile = prof;
    k.size = size;
    k.plane = plane;
    k.slab = off;
    k.row0 = P.phase == 1 ? 0 : 2 * NDIM;
    k.a = a;
    k.lo = lo;
    k.hi = hi;
    k.N = N;
    k.own_half = false;
    k.slow = slow;
#pragma unroll
    for (int c = 0; c < NDIM; ++c) {
      if (!on[c])
        continue;
      next[c] += mi[c] * (g.f[e] * stress_divergence<NDIM, R, Q>(g, k, c, e, c, A));
      if (t >= 0) {
        const int at = (c == e ? 3 * N : N) + a;
        const int64_t z = ((int64_t)(NDIM + c) * size + t) * g.lanes;
        lanes_put(aux, z, prof[at] * (lanes_at<Q>(aux, z) + w1[c]));
      }
    }
    return;
  }
  // the rows read before any is written: one wait for all
  const T pn = prof[N + a], dn = prof[a], ph = prof[3 * N + a], dh = prof[2 * N + a];
  Q m[NDIM];
#pragma unroll
  for (int c = 0; c < NDIM; ++c)
    m[c] = lanes_at<Q>(aux, ((int64_t)(NDIM + c) * size + t) * g.lanes);
#pragma unroll
  for (int c = 0; c < NDIM; ++c) {
    if (!on[c])
      continue;
    m[c] = (c == e ? ph : pn) * m[c] + (c == e ? dh : dn) * Q(g.f[e] * D[c][e]);
    lanes_put(aux, ((int64_t)(NDIM + c) * size + t) * g.lanes, m[c]);
    next[c] += mi[c] * m[c];
  }
}

// the adjoint's strain memory settled into its other block (elastic.cu:577-595)
template <int NDIM, int V, typename T>
__device__ __forceinline__ void settle_memory(const ElGeom<T> &g, const ElLayer<T> &P,
                                              const T *sigma, int64_t idx, int lane0, int e,
                                              const int *A) {
  using Q = LanesOf<T, V>;
  const int a = A[e], lo = P.lo[e], hi = P.hi[e];
  if (!in_slab<NDIM>(g, a, e, lo, hi, 0))
    return;
  int64_t plane, size, off;
  slab_geometry<NDIM>(g, e, lo, hi, A, &plane, &size, &off);
  const int N = g.n[e];
  const int64_t t = slab_at(a, N, lo, hi, e < NDIM - 1, plane, off);
  const int from = P.phase == 1 ? 0 : 2 * NDIM, to = 2 * NDIM - from;
  const T *prof = P.profile[e];
  T *aux = P.aux[e] + lane0;
#pragma unroll
  for (int k = 0; k < NDIM; ++k) {
    const int at = (k == e ? 0 : 2 * N) + a;
    const Q s = lanes_at<Q>(sigma, ((int64_t)stress_row<NDIM>(k, e) * g.nodes + idx) * g.lanes);
    lanes_put(aux, ((int64_t)(to + k) * size + t) * g.lanes,
              prof[N + at] * (lanes_at<Q>(aux, ((int64_t)(from + k) * size + t) * g.lanes) + s));
  }
}

// ---------------------------------------------------------------- kernels
// thread -> (interior node, first lane): a node's lanes / V threads are
// neighbours in the wave; false past the last node (whole node groups).
// Blocks go to the XCDs in contiguous runs of nodes (cw::xcd_tile), so the
// rows a block's taps read along the slow axes were fetched into the same
// XCD's L2 by the blocks before it.
template <int NDIM, int V, typename T>
__device__ __forceinline__ bool node_of(const ElGeom<T> &g, int *A, int64_t *idx, int *lane0) {
  // threads are under 2^31: 32-bit arithmetic, the lanes a power of two
  const int per = g.lanes / V, shift = __builtin_ctz(per);
  const uint32_t t = (uint32_t)cw::xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  const uint32_t i = t >> shift;
  if (i >= (uint32_t)g.interior)
    return false;
  *lane0 = (int)(t & (per - 1)) * V;
  uint32_t rest = i;
#pragma unroll
  for (int d = NDIM - 1; d >= 0; --d) {
    const uint32_t w = g.n[d] - 2;
    A[d] = 1 + (int)(d ? rest % w : rest);
    rest /= w;
  }
  int64_t at = 0;
#pragma unroll
  for (int d = 0; d < NDIM; ++d)
    at += (int64_t)A[d] * g.s[d];
  *idx = at;
  return true;
}

// the thread's place in a component
template <int NDIM, typename T>
__device__ __forceinline__ Place<NDIM, T> place_of(const ElGeom<T> &g, int64_t idx, int lane0) {
  return ((Place<NDIM, T>)idx * (Place<NDIM, T>)g.lanes + (Place<NDIM, T>)lane0) *
         (Place<NDIM, T>)sizeof(T);
}

// the per-node sum over the shots of a density, taken off accumulator `acc`
template <typename T, int V>
__device__ __forceinline__ void take_off(T *acc, int64_t at, const LanesOf<T, V> &x, int lanes,
                                         int lane0) {
  const T sum = cw::shot_sum(x, lanes);
  if (lane0 == 0)
    acc[at] -= sum;
}

// the prepared material of each interior node: the inverse inertia of each
// component point (elastic.cu:200-211), then the shear gamma of each pair
// point (elastic.cu:189-197). The reference's CPU fallback (the oracle's
// IEEE path) forms the pair's reciprocals in double precision, `fmax` being
// the C library's double function there, and rounds the sum to T after each
// term; the float build does the same so its bits match.
template <typename T, int NDIM>
__global__ void __launch_bounds__(kThreads)
el_prepare(ElGeom<T> g, const T *__restrict__ gamma, T rho, T *__restrict__ prep) {
  int A[3];
  int64_t idx;
  int lane0;
  ElGeom<T> one = g;
  one.lanes = 1;
  if (!node_of<NDIM, 1>(one, A, &idx, &lane0))
    return;
  const T tiny = Tiny<T>::value;
#pragma unroll
  for (int c = 0; c < NDIM; ++c) {
    bool held = false;
#pragma unroll
    for (int d = 0; d < NDIM; ++d)
      if (d != c && ((A[d] == 1 && clamped_face(g, d, 0)) ||
                     (A[d] == g.n[d] - 2 && clamped_face(g, d, 1))))
        held = true;
    T minv = (T)0;
    if (A[c] <= g.n[c] - 2) {
      const T mean = (T)0.5 * (gamma[idx] + gamma[idx + g.s[c]]);
      minv = held ? (T)0 : (T)1 / fmax(rho * mean, tiny);
    }
    prep[(int64_t)c * g.nodes + idx] = minv;
  }
#pragma unroll
  for (int k = 0; k < NDIM - 1; ++k)
#pragma unroll
    for (int l = k + 1; l < NDIM; ++l) {
      const int v = stress_row<NDIM>(k, l);
      T out = (T)0;
      if (shear_point(g, k, l, A)) {
        const int64_t at[4] = {idx, idx + g.s[l], idx + g.s[k], idx + g.s[k] + g.s[l]};
        T sum = (T)(1.0 / fmax((double)gamma[at[0]], (double)tiny));
#pragma unroll
        for (int i = 1; i < 4; ++i)
          sum = (T)((double)sum + 1.0 / fmax((double)gamma[at[i]], (double)tiny));
        out = (T)4 / sum;
      }
      prep[(int64_t)v * g.nodes + idx] = out;
    }
}

// stress_kernel (elastic.cu:756-795): the stresses of u1 into sigma, the PML
// fold, and in the adjoint pair (GRAD) the stiffness densities of u1 against
// the forward field v1 (stiffness_density, elastic.cu:356-383)
template <typename T, int NDIM, int R, int V, bool GRAD>
__device__ __forceinline__ void
stress_node(const ElGeom<T> &g, const ElLayer<T> &P, const T *__restrict__ gamma,
            const T *__restrict__ prep, const T *__restrict__ u1, T *__restrict__ sigma,
            T *__restrict__ g_normal, T *__restrict__ g_shear, const T *__restrict__ v1,
            const int *A, int64_t idx, int lane0) {
  using Q = LanesOf<T, V>;
  constexpr int NV = nvoigt<NDIM>();
  const auto place = place_of<NDIM>(g, idx, lane0);
  const T gn = gamma[idx];
  T shear[NV > NDIM ? NV - NDIM : 1]; // read at every node: used where the pair has its point
#pragma unroll
  for (int v = 0; v < NV - NDIM; ++v)
    shear[v] = prep[(NDIM + v) * g.nodes + idx];
  // each derivative once: the strains and the forward's memory both read it
  Q D[NDIM][NDIM];
  derivatives<NDIM, R, Q>(g, u1, place, A, D);
  Q eps[NV], sig[NV];
  const int zeroed = zeroed_axes<NDIM>(g, A);
  strains_of<NDIM>(g, D, A, eps);
  if constexpr (GRAD) {
    Q eu[NDIM];
    const int z2 = normal_strains<NDIM, R, Q>(g, v1, place, A, eu);
    take_off<T, V>(g_normal, idx, normal_form<NDIM, Q>(g, eps, eu, z2), g.lanes, lane0);
#pragma unroll
    for (int k = 0; k < NDIM - 1; ++k)
#pragma unroll
      for (int l = k + 1; l < NDIM; ++l) {
        if (!shear_point(g, k, l, A))
          continue;
        const int w = stress_row<NDIM>(k, l);
        const Q d = g.mu * eps[w] * shear_strain<NDIM, R, Q>(g, v1, place, k, l, A);
        take_off<T, V>(g_shear, (int64_t)(w - NDIM) * g.nodes + idx, d, g.lanes, lane0);
      }
  }
  stress_of<NDIM, Q>(g, eps, zeroed, gn, shear, A, sig);
  // the axis a constant of each: so large a loop is left rolled at the long
  // stencils, and its arrays go to scratch memory
  stress_memory<NDIM, R, V, 0>(g, P, u1, D, gn, shear, place, lane0, A, sig);
  if constexpr (NDIM > 1)
    stress_memory<NDIM, R, V, 1>(g, P, u1, D, gn, shear, place, lane0, A, sig);
  if constexpr (NDIM > 2)
    stress_memory<NDIM, R, V, 2>(g, P, u1, D, gn, shear, place, lane0, A, sig);
#pragma unroll
  for (int w = 0; w < NV; ++w)
    put_bytes(sigma + w * (g.nodes * g.lanes), place, sig[w]);
}

template <typename T, int NDIM, int R, int V, bool GRAD>
__global__ void __launch_bounds__(kThreads)
el_stress(ElGeom<T> g, ElLayer<T> P, const T *__restrict__ gamma, const T *__restrict__ prep,
          const T *__restrict__ u1, T *__restrict__ sigma, T *__restrict__ g_normal,
          T *__restrict__ g_shear, const T *__restrict__ v1) {
  int A[3];
  int64_t idx;
  int lane0;
  if (node_of<NDIM, V>(g, A, &idx, &lane0))
    stress_node<T, NDIM, R, V, GRAD>(g, P, gamma, prep, u1, sigma, g_normal, g_shear, v1, A, idx,
                                     lane0);
}

// fd_kernel (elastic.cu:798-853): u2 from u0, u1 and the stresses, the PML
// fold, and in the adjoint pair the inertia density against v1; u2 may be u0
template <typename T, int NDIM, int R, int V, bool GRAD>
__device__ __forceinline__ void
update_node(const ElGeom<T> &g, const ElLayer<T> &P, const T *__restrict__ prep, const T *sigma,
            const T *u0, const T *__restrict__ u1, T *u2, T *__restrict__ g_mass,
            const T *__restrict__ v1, T mf, const int *A, int64_t idx, int lane0) {
  using Q = LanesOf<T, V>;
  const auto place = place_of<NDIM>(g, idx, lane0);
  // the node's own values (of every component: an update that has no point
  // here is dropped), then the divergence of component c along axis e, once:
  // the force (nodal_force, elastic.cu:281-303) and the forward's memory read
  // it. As in `derivatives`, an axis with no wall near takes its divergences
  // in one branch.
  bool on[NDIM];
  T mi[NDIM];
  Q w0[NDIM], w1[NDIM], D[NDIM][NDIM], next[NDIM];
#pragma unroll
  for (int c = 0; c < NDIM; ++c) {
    const int64_t comp = c * (g.nodes * g.lanes);
    on[c] = A[c] <= g.n[c] - 3;
    mi[c] = prep[(int64_t)c * g.nodes + idx];
    w0[c] = at_bytes<Q>(u0 + comp, place);
    w1[c] = at_bytes<Q>(u1 + comp, place);
  }
#pragma unroll
  for (int e = 0; e < NDIM; ++e) {
    const auto line = field_line(sigma, place, g, e);
    if (near_wall(g, A[e], e)) {
#pragma unroll
      for (int c = 0; c < NDIM; ++c)
        D[c][e] = on[c] ? stress_divergence<NDIM, R, Q>(g, line, c, e, stress_row<NDIM>(c, e), A)
                        : Q((T)0);
    } else {
#pragma unroll
      for (int c = 0; c < NDIM; ++c)
        D[c][e] = inner_divergence<NDIM, R, Q>(g, line, stress_row<NDIM>(c, e), c == e);
    }
  }
#pragma unroll
  for (int c = 0; c < NDIM; ++c) {
    Q force = g.f[c] * D[c][c];
#pragma unroll
    for (int l = 0; l < NDIM; ++l)
      if (l != c)
        force = fmat(g.f[l], D[c][l], force);
    next[c] = -w0[c] + (T)2.f * w1[c] + mi[c] * force;
  }
  // the axis a constant of each, as in stress_node
  force_memory<NDIM, R, V, 0>(g, P, sigma, D, w1, mi, on, place, lane0, A, next);
  if constexpr (NDIM > 1)
    force_memory<NDIM, R, V, 1>(g, P, sigma, D, w1, mi, on, place, lane0, A, next);
  if constexpr (NDIM > 2)
    force_memory<NDIM, R, V, 2>(g, P, sigma, D, w1, mi, on, place, lane0, A, next);
#pragma unroll
  for (int c = 0; c < NDIM; ++c) {
    if (!on[c])
      continue;
    const int64_t comp = c * (g.nodes * g.lanes);
    if constexpr (GRAD) {
      const Q v = at_bytes<Q>(v1 + comp, place);
      take_off<T, V>(g_mass, (int64_t)c * g.nodes + idx,
                     mf * v * (next[c] - (T)2.f * w1[c] + w0[c]), g.lanes, lane0);
    }
    put_bytes(u2 + comp, place, next[c]);
  }
  if (P.phase) {
#pragma unroll
    for (int e = 0; e < NDIM; ++e)
      if (P.lo[e] + P.hi[e])
        settle_memory<NDIM, V>(g, P, sigma + lane0, idx, lane0, e, A);
  }
}

template <typename T, int NDIM, int R, int V, bool GRAD>
__global__ void __launch_bounds__(kThreads)
el_update(ElGeom<T> g, ElLayer<T> P, const T *__restrict__ prep, const T *sigma, const T *u0,
          const T *__restrict__ u1, T *u2, T *__restrict__ g_mass, const T *__restrict__ v1, T mf) {
  int A[3];
  int64_t idx;
  int lane0;
  if (node_of<NDIM, V>(g, A, &idx, &lane0))
    update_node<T, NDIM, R, V, GRAD>(g, P, prep, sigma, u0, u1, u2, g_mass, v1, mf, A, idx,
                                     lane0);
}

// gradient_kernel (elastic_sensitivity.cu:115-158): both densities of the
// forward triplet u0, u1, u2 against the adjoint l1; g.f holds 1 / dx
template <typename T, int NDIM, int R, int V>
__global__ void __launch_bounds__(kThreads)
el_gradient(ElGeom<T> g, T *__restrict__ g_mass, T *__restrict__ g_normal,
            T *__restrict__ g_shear, const T *__restrict__ u0, const T *__restrict__ u1,
            const T *__restrict__ u2, const T *__restrict__ l1, T mf) {
  using Q = LanesOf<T, V>;
  int A[3];
  int64_t idx;
  int lane0;
  if (!node_of<NDIM, V>(g, A, &idx, &lane0))
    return;
#pragma unroll
  for (int c = 0; c < NDIM; ++c) {
    if (A[c] > g.n[c] - 3)
      continue;
    const int64_t n = (int64_t)c * g.nodes + idx;
    const int64_t at = n * g.lanes + lane0;
    const Q l = lanes_at<Q>(l1, at);
    const Q w0 = lanes_at<Q>(u0, at), w1 = lanes_at<Q>(u1, at), w2 = lanes_at<Q>(u2, at);
    take_off<T, V>(g_mass, n, mf * l * (w2 - (T)2.f * w1 + w0), g.lanes, lane0);
  }
  const auto place = place_of<NDIM>(g, idx, lane0);
  Q eu[NDIM], el[NDIM];
  const int zeroed = normal_strains<NDIM, R, Q>(g, u1, place, A, eu);
  normal_strains<NDIM, R, Q>(g, l1, place, A, el);
  take_off<T, V>(g_normal, idx, normal_form<NDIM, Q>(g, el, eu, zeroed), g.lanes, lane0);
#pragma unroll
  for (int k = 0; k < NDIM - 1; ++k)
#pragma unroll
    for (int l = k + 1; l < NDIM; ++l) {
      if (!shear_point(g, k, l, A))
        continue;
      const int w = stress_row<NDIM>(k, l);
      const Q d = g.mu * shear_strain<NDIM, R, Q>(g, l1, place, k, l, A) *
                  shear_strain<NDIM, R, Q>(g, u1, place, k, l, A);
      take_off<T, V>(g_shear, (int64_t)(w - NDIM) * g.nodes + idx, d, g.lanes, lane0);
    }
}

// --------------------------------------------------------------- points
// entry e of a point list reads or writes element lin[e] * lanes + b of a
// field for shot lane b (every lane when shot[e] < 0, else lane shot[e]) and
// element row * rs + col[e] * cs + b * ss of a table
struct ElPoints {
  const int32_t *starts; // (runs + 1) CSR: the entries of a run share one node
  const int32_t *lin, *shot, *col;
  int32_t runs;
  int64_t rs, cs, ss;
};

// kind 0: u += weight * table (injection, a run's entries in order);
// 1: table = u (record); 2: u = table (strip replay); 3: the adjoint
// injection, u += weight * table and g_mass += -mf u1 weight * table, lane
// after lane (cuwave/kernels/common.cuh:456-503)
template <typename T>
__global__ void __launch_bounds__(kThreads)
el_points(ElPoints p, int kind, int lanes, int nbatch, int64_t row, T *__restrict__ u,
          T *__restrict__ table, const T *__restrict__ weight, T *__restrict__ g_mass,
          const T *__restrict__ u1, T mf) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (kind == 3) {
    if (t >= p.runs)
      return;
    for (int e = p.starts[t]; e < p.starts[t + 1]; ++e) {
      const int64_t n = p.lin[e];
      for (int b = 0; b < nbatch; ++b) {
        if (p.shot[e] >= 0 && p.shot[e] != b)
          continue;
        const T load = weight[e] * table[row * p.rs + p.col[e] * p.cs + b * p.ss];
        u[n * lanes + b] += load;
        g_mass[n] += -mf * u1[n * lanes + b] * load;
      }
    }
    return;
  }
  const int64_t run = t / lanes;
  const int b = (int)(t % lanes);
  if (run >= p.runs || b >= nbatch)
    return;
  for (int e = p.starts[run]; e < p.starts[run + 1]; ++e) {
    if (p.shot[e] >= 0 && p.shot[e] != b)
      continue;
    const int64_t n = (int64_t)p.lin[e] * lanes + b;
    const int64_t m = row * p.rs + p.col[e] * p.cs + b * p.ss;
    if (kind == 0)
      u[n] += weight[e] * table[m];
    else if (kind == 1)
      table[m] = u[n];
    else
      u[n] = table[m];
  }
}

} // namespace cwe
