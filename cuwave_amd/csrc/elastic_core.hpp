// The core of a 2D elastic step: stresses and update fused, for the nodes no
// wall closure, traction face or PML memory reaches.
//
// The pair writes every stress to memory and reads it back about four times
// over (it stays in L2, but 8 of the 14 passes over memory a step makes are
// the stresses'). Here a block marches down the slow axis with the stresses in
// registers and LDS: a step of the core reads u^(t-1) and u^(t-2) once and
// writes u^t once, which is what bounds it.
//
// A thread is one column and V shot lanes. Marching row by row it keeps the
// displacement rows its slow-axis derivatives read and the stress rows its
// slow-axis divergences read in register rings of 2 R + 2 rows, the march
// unrolled by as many so that no value moves (the moves were a quarter of the
// instructions: 352 us a step against 263). Iteration r stages displacement
// row r and stress rows r - R (all of them known) in LDS, one barrier, then
// forms stress row r from its neighbours' displacements and update row r - R
// from its neighbours' stresses: one barrier a row, two LDS buffers in turn. A
// row's loads are issued while the row before computes. A block's C columns of
// stresses serve C - 2 R columns of update, and a chunk of rows costs 2 R rows
// of stresses more.
//
// Measured at 1058 x 2114 nodes, order 4, 16 float lanes, the frame's part
// included: 271 us a step (595 by the pair alone), the core's launch 232 us
// for the 860 MB it cannot do without; 323 x 457 at 4 lanes 24 us (35).
//
// The frame around the core (walls, closures, PML slabs and the reach of their
// memories) runs the pair's own code over its nodes only: its stresses in the
// core's launch, after the core's blocks, its update in a second launch.
//
// The arithmetic is the pair's deep path term by term in the same order, so a
// node's bits do not depend on which of the two stepped it.
#pragma once

#include "elastic.hpp"

namespace cwe {

// the core's update rectangle, rows [y0, y1) x columns [x0, x1), cut into nx
// block columns and ny chunks of `chunk` rows
struct ElBox {
  int y0, y1, x0, x1;
  int chunk, nx, ny;
};

// interior nodes outside a hole, rows [y0, y1) x columns [x0, x1)
struct ElFrame {
  int y0, y1, x0, x1;
  int nodes;
};

// node i of the frame: the rows above the hole, the rows below, then the
// hole's rows left and right of it
template <typename T>
__device__ __forceinline__ void frame_node(const ElGeom<T> &g, const ElFrame &f, int i, int *A) {
  const int w = g.n[1] - 2;
  const int above = (f.y0 - 1) * w, below = (g.n[0] - 1 - f.y1) * w;
  if (i < above) {
    A[0] = 1 + i / w;
    A[1] = 1 + i % w;
  } else if (i < above + below) {
    A[0] = f.y1 + (i - above) / w;
    A[1] = 1 + (i - above) % w;
  } else {
    const int left = f.x0 - 1, side = left + g.n[1] - 1 - f.x1;
    const int k = (i - above - below) % side;
    A[0] = f.y0 + (i - above - below) / side;
    A[1] = k < left ? 1 + k : f.x1 + k - left;
  }
}

// the frame node and first lane of thread `t`, false past the last
template <int V, typename T>
__device__ __forceinline__ bool frame_thread(const ElGeom<T> &g, const ElFrame &f, uint32_t t,
                                             int *A, int64_t *idx, int *lane0) {
  const int per = g.lanes / V, i = (int)(t >> __builtin_ctz(per));
  if (i >= f.nodes)
    return false;
  *lane0 = (int)(t & (per - 1)) * V;
  frame_node(g, f, i, A);
  *idx = (int64_t)A[0] * g.s[0] + A[1];
  return true;
}

// LDS of a core block of NT threads: two buffers of two displacement rows
// with R columns of halo either side (up to kHaloPer threads a column) and two
// stress rows, at compile-time offsets
constexpr int kHaloPer = 16;
template <int R, int NT> struct CoreRows {
  static constexpr int wide = NT + 2 * R * kHaloPer; // a displacement row
  static constexpr int buffer = 2 * wide + 2 * NT;
  static constexpr int bytes(int q_bytes) { return 2 * buffer * q_bytes; }
};

// block `item` of the core; g holds the strain factors, fu0 and fu1 the
// update's
template <typename T, int R, int V, int NT>
__device__ __forceinline__ void el_core_block(const ElGeom<T> &g, const T fu0, const T fu1,
                                              const ElBox &box, const T *__restrict__ gamma,
                                              const T *__restrict__ prep, const T *u0,
                                              const T *__restrict__ u1, T *u2, int item,
                                              char *lds) {
  using Q = LanesOf<T, V>;
  using S = CoreRows<R, NT>;
  constexpr uint32_t QB = sizeof(Q);
  constexpr int P = 2 * R + 2; // rows a ring holds: those in use and the one arriving
  const int per = g.lanes / V, cols = NT / per;
  const int h = (int)threadIdx.x, c = h / per, l = h % per;
  const int kx = item % box.nx, ky = item / box.nx;
  const int ya = box.y0 + ky * box.chunk, yb = min(ya + box.chunk, box.y1);
  const int xs = box.x0 - R + kx * (cols - 2 * R); // the block's first stress column
  const int x = xs + c;
  const bool mine = c >= R && c < cols - R && x < box.x1; // this column is updated
  const int last = g.np[1] - 1;
  const int xc = min(x, last); // columns past the box load in range, unused
  // byte offsets of this thread's column in a row of a field and of a node array
  const uint32_t row = (uint32_t)g.s[0] * per * QB, nrow = (uint32_t)g.s[0] * sizeof(T);
  const uint32_t col = ((uint32_t)xc * per + l) * QB, ncol = (uint32_t)xc * sizeof(T);
  const int64_t comp = g.nodes * g.lanes;
  const T *ua = u1, *ub = u1 + comp;            // the components of u^(t-1)
  const T *wa = u0, *wb = u0 + comp;            // of u^(t-2)
  T *na = u2, *nb = u2 + comp;                  // of u^t
  const T *ma = prep, *mb = prep + g.nodes, *sh = prep + 2 * g.nodes;
  // the halo column this thread stages: entry h of 2 R x per
  const bool halo = h < 2 * R * per;
  const int hc = h / per; // 0 .. R - 1 left of the block, R .. 2 R - 1 right
  const int hx = min(max(hc < R ? xs - R + hc : xs + cols + hc - R, 0), last);
  const uint32_t hcol = ((uint32_t)hx * per + l) * QB;
  Q *base = reinterpret_cast<Q *>(lds);
  const int hme = hc < R ? h : NT + h; // a right halo column: (hc - R) past the block's last
  // this thread's place in a displacement row and its neighbours' (-R .. R
  // columns away), in a stress row R per entries less
  Q *at[2 * R + 1];
#pragma unroll
  for (int j = 0; j <= 2 * R; ++j)
    at[j] = base + h + j * per;
  Q *back[R + 1]; // 0 .. R columns left in a stress row
#pragma unroll
  for (int j = 0; j <= R; ++j)
    back[j] = base + h - j * per;
  struct Ahead {
    Q ha, hb, wa, wb;
    T gn, sh, ma, mb;
  };
  Ahead ahead[2];
  // rings by row: displacement rows r - R .. r + R and the arriving one, stress
  // rows r - 2 R .. r
  Q qa[P], qb[P], s00[P], s01[P], s11[P];
  const int ra = ya - R, rb = yb + R; // stress rows [ra, rb)
#pragma unroll
  for (int i = 0; i < P; ++i) {
    s00[i] = Q((T)0);
    s01[i] = Q((T)0);
    s11[i] = Q((T)0);
  }
  // row ra + K sits in ring place (K + R) % P
#pragma unroll
  for (int i = 0; i < 2 * R - 1; ++i)
    qa[i] = at_bytes<Q>(ua, (uint32_t)(ra - R + i) * row + col);
#pragma unroll
  for (int i = 0; i < 2 * R; ++i)
    qb[i] = at_bytes<Q>(ub, (uint32_t)(ra - R + i) * row + col);
  // what iteration r reads: the rings' next rows, the halo of row r, the
  // material of row r and the update's own values of row r - R
  auto fetch = [&](int r, Q &na_, Q &nb_, Ahead &f) {
    const uint32_t o = (uint32_t)r * row, on = (uint32_t)r * nrow + ncol;
    na_ = at_bytes<Q>(ua, o + (uint32_t)(R - 1) * row + col);
    nb_ = at_bytes<Q>(ub, o + (uint32_t)R * row + col);
    if (halo) {
      f.ha = at_bytes<Q>(ua, o + hcol);
      f.hb = at_bytes<Q>(ub, o + hcol);
    }
    f.gn = at_bytes<T>(gamma, on);
    f.sh = at_bytes<T>(sh, on);
    if (mine && r - R >= ya) {
      f.wa = at_bytes<Q>(wa, o - R * row + col);
      f.wb = at_bytes<Q>(wb, o - R * row + col);
      f.ma = at_bytes<T>(ma, on - R * nrow);
      f.mb = at_bytes<T>(mb, on - R * nrow);
    }
  };
  fetch(ra, qa[2 * R - 1], qb[2 * R], ahead[0]);
  for (int r0 = ra; r0 < rb; r0 += P) {
#pragma unroll
    for (int K = 0; K < P; ++K) {
      const int r = r0 + K;
      if (r >= rb)
        break;
      // ring places of the rows j away from r (displacements, stresses)
#define CW_ROW(j) ((K + R + (j) + 2 * P) % P)
      constexpr int la = 0, lb = S::wide, l11 = 2 * S::wide, l01 = 2 * S::wide + NT;
      const int buf = (K & 1) * S::buffer;
      const Ahead &f = ahead[K & 1];
      at[R][buf + la] = qa[CW_ROW(0)];
      at[R][buf + lb] = qb[CW_ROW(0)];
      if (halo) {
        base[buf + la + hme] = f.ha;
        base[buf + lb + hme] = f.hb;
      }
      // row r - R of the stresses, formed by the iterations before
      at[0][buf + l11] = s11[CW_ROW(-R)];
      at[0][buf + l01] = s01[CW_ROW(-R)];
      __syncthreads();
      if (r + 1 < rb)
        fetch(r + 1, qa[CW_ROW(R)], qb[CW_ROW(R + 1)], ahead[(K + 1) & 1]);
      // stress row r (strain_point, stress_of)
      Q d0((T)0), d1((T)0), dk((T)0), dl((T)0);
#pragma unroll
      for (int q = 1; q <= R; ++q) {
        d0 += g.sg[q - 1] * (qa[CW_ROW(q - 1)] - qa[CW_ROW(-q)]);
        d1 += g.sg[q - 1] * (at[R + q - 1][buf + lb] - at[R - q][buf + lb]);
        dk += g.sg[q - 1] * (qb[CW_ROW(q)] - qb[CW_ROW(1 - q)]);
        dl += g.sg[q - 1] * (at[R + q][buf + la] - at[R + 1 - q][buf + la]);
      }
      const Q e0 = g.f[0] * d0, e1 = g.f[1] * d1;
      const Q e01 = fmat(g.f[0], dk, g.f[1] * dl);
      Q tr((T)0);
      tr += e0;
      tr += e1;
      s00[CW_ROW(0)] = f.gn * ((T)2.f * g.mu * e0 + g.lam * tr);
      s11[CW_ROW(0)] = f.gn * ((T)2.f * g.mu * e1 + g.lam * tr);
      s01[CW_ROW(0)] = f.sh * g.mu * e01;
      // update row r - R (nodal_force, el_update); neighbours in a stress row
      // are `at` less its R columns of halo
      if (mine && r - R >= ya) {
        Q da((T)0), ha((T)0), db((T)0), hb((T)0);
#pragma unroll
        for (int q = 1; q <= R; ++q) {
          da += g.sg[q - 1] * s00[CW_ROW(q - R)];
          da -= g.sg[q - 1] * s00[CW_ROW(1 - q - R)];
          ha += g.sg[q - 1] * at[q - 1][buf + l01];
          ha -= g.sg[q - 1] * back[q][buf + l01];
          db += g.sg[q - 1] * at[q][buf + l11];
          db -= g.sg[q - 1] * back[q - 1][buf + l11];
          hb += g.sg[q - 1] * s01[CW_ROW(q - 1 - R)];
          hb -= g.sg[q - 1] * s01[CW_ROW(-q - R)];
        }
        const Q fa = fmat(fu1, ha, fu0 * da);
        const Q fb = fmat(fu0, hb, fu1 * db);
        const uint32_t o = (uint32_t)(r - R) * row + col;
        put_bytes(na, o, -f.wa + (T)2.f * qa[CW_ROW(-R)] + f.ma * fa);
        put_bytes(nb, o, -f.wb + (T)2.f * qb[CW_ROW(-R)] + f.mb * fb);
      }
#undef CW_ROW
    }
  }
}

// the core's blocks, then the stresses of the frame
template <typename T, int R, int V, int VC, int NT>
__global__ void __launch_bounds__(NT)
el_core(ElGeom<T> g, T fu0, T fu1, ElBox box, ElFrame frame, ElLayer<T> P,
        const T *__restrict__ gamma, const T *__restrict__ prep, const T *u0,
        const T *__restrict__ u1, T *u2, T *__restrict__ sigma) {
  extern __shared__ __align__(16) char lds[];
  const int blocks = box.nx * box.ny;
  if ((int)blockIdx.x < blocks) {
    el_core_block<T, R, VC, NT>(g, fu0, fu1, box, gamma, prep, u0, u1, u2,
                               cw::xcd_tile(blockIdx.x, blocks), lds);
    return;
  }
  int A[3];
  int64_t idx;
  int lane0;
  const int b = cw::xcd_tile((int)blockIdx.x - blocks, (int)gridDim.x - blocks);
  if (frame_thread<V>(g, frame, (uint32_t)b * NT + threadIdx.x, A, &idx, &lane0))
    stress_node<T, 2, R, V, false>(g, P, gamma, prep, u1, sigma, (T *)nullptr, (T *)nullptr,
                                   (const T *)nullptr, A, idx, lane0);
}

// the frame's update
template <typename T, int R, int V>
__global__ void __launch_bounds__(kThreads)
el_frame_update(ElGeom<T> g, ElFrame frame, ElLayer<T> P, const T *__restrict__ prep,
                const T *sigma, const T *u0, const T *__restrict__ u1, T *u2) {
  int A[3];
  int64_t idx;
  int lane0;
  if (frame_thread<V>(g, frame,
                      (uint32_t)cw::xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x, A,
                      &idx, &lane0))
    update_node<T, 2, R, V, false>(g, P, prep, sigma, u0, u1, u2, (T *)nullptr,
                                   (const T *)nullptr, (T)0, A, idx, lane0);
}

} // namespace cwe
