// dcl_step2d.hpp -- one 2D level-set update (SL step, then the 9-point
// curvature of the new phi) of a tile, in one pass: the dense 2D step and the
// 2D batch.
//
// A block of 64 x 4 threads works an area of 64 x 4 R nodes, R rows per
// thread.  phi0 over the area plus a halo of 3 nodes and the velocity faces
// over it plus 1 node below and 2 above are staged in LDS with coalesced
// loads; the 16 (4) stencil values, the node's faces and the RK2 midpoint's
// corners come from there (a node whose stencil leaves the halo, a departure
// of 2 cells or more, gathers from memory).  The new phi of the area goes to
// LDS too, and the curvature of the nodes inside its outer layer is taken
// from there; those 62 x (4 R - 2) nodes are the tile's output, the outer
// layer being worked by the neighbouring tiles too, with the same bits.  So
// phi is written once and not read back.  phi and kappa have the bits of the
// separate SL and curvature kernels.
//
// With R = 4 a tile may also be wide: all 64 columns are its output, and the
// column to either side is worked after them (32 nodes, one more round of one
// wave; departures of a cell or more from these gather).  A wide tile takes
// 7/6 of a narrow one's time, so it is the better one where it saves a column
// of tiles of at most six, windows 64, 128, 192, 256 or 320 nodes wide above
// all: 64 cells of 128 x 128 in FP32 19.2 us a step narrow, 15.5 wide.
//
// What it replaces read every stencil value with its own gather (about 20
// vector loads per node, the texture path's limit) and phi again for the
// curvature: 256 FP64 cells of edges 64 to 512 (1.9e7 nodes), tricubic RK2,
// 406 -> 251 us per step (1.8 -> 3.0 TB/s of the 40 bytes per node); a 128 x
// 128 step replayed from a graph 4.7 -> 3.2 us, one launch instead of two.
// The FP64 tile (R = 4) takes 40.6 KB of LDS and 113 registers, four blocks
// per CU by either; the arithmetic is about 60% of its time.
#pragma once

#include "dcl_curv.hpp"
#include "dcl_sl.hpp"

namespace dcl {

constexpr int S2_TX = 64, S2_TY = 4, S2_H = 3;  // threads of a block, phi0's halo

template <int R>
struct Step2 {
  static constexpr bool WIDE = R == 4;                  // has wide tiles
  static constexpr int AY = S2_TY * R;                  // area rows
  static constexpr int AX = S2_TX + (WIDE ? 2 : 0);     // pitch of the new phi
  static constexpr int OX = S2_TX - 2, OY = AY - 2;     // a narrow tile's output nodes
  static constexpr int PX = S2_TX + 2 * S2_H, PY = AY + 2 * S2_H;
  static constexpr int VX = S2_TX + 3, VY = AY + 3;     // u ends a row earlier
  static constexpr int NT = S2_TX * S2_TY;
};
template <typename T, int R>
struct Step2Lds {
  T phi[Step2<R>::PX * Step2<R>::PY];
  T u[Step2<R>::VX * (Step2<R>::VY - 1)], v[Step2<R>::VX * Step2<R>::VY];
  T out[Step2<R>::AY * Step2<R>::AX];
};
// columns of a tile of a window this wide
__host__ __device__ inline int step2d_cols(int nx, int rows) {
  const bool wide = rows == 4 && 7 * ((nx + S2_TX - 1) / S2_TX) < 6 * ((nx + S2_TX - 3) / (S2_TX - 2));
  return wide ? S2_TX : S2_TX - 2;
}
inline int64_t step2d_tiles(int nx, int ny, int rows) {
  const int cols = step2d_cols(nx, rows), oy = S2_TY * rows - 2;
  return (int64_t)((nx + cols - 1) / cols) * ((ny + oy - 1) / oy);
}

// Rows per thread, from the tiles there are with 4 and with 2: more rows stage
// and recompute fewer halo values per node, fewer finish a small window sooner.
// The lines lie where they cross, at 2.5 and 1.5 blocks per CU.  us per FP64
// tricubic RK2 step with 1 / 2 / 4 rows, one window n x n: 128 3.2 / 4.3 /
// 8.9, 256 4.2 / 4.5 / 6.4, 384 5.7 / 5.6 / 6.6, 512 8.1 / 6.9 / 8.5, 768 15.5
// / 13.0 / 11.7, 1024 23.0 / 18.8 / 17.8; a batch of 128 x 128 cells: one 3.9 /
// 5.2 / 8.2, 4 5.2 / 6.3 / 8.7, 8 7.4 / 6.9 / 8.8, 16 11.4 / 9.4 / 11.2, 32
// 19.7 / 15.6 / 14.2, 64 35.3 / 28.4 / 20.7.  FP32 and the trilinear scheme
// cross at about the same sizes.
inline int step2d_rows(int64_t tiles4, int64_t tiles2, int cus) {
  return 2 * tiles4 >= (int64_t)5 * cus ? 4 : 2 * tiles2 >= (int64_t)3 * cus ? 2 : 1;
}

// LDS reads through pointers of their own address space: where a branch reads
// the same values from memory instead, the compiler would otherwise make one
// flat load of the two
template <typename T>
using lds_cptr = const __attribute__((address_space(3))) T*;

// the SL value of interior node (i, j) of a window whose velocity has the
// same window; (x0, y0) the area's first node
template <typename T, int INTERP, int BT, int R>
__device__ __forceinline__ T step2d_node(const T* __restrict__ phi0, const T* __restrict__ vel, const SLP& P,
                                         const Step2Lds<T, R>& S, int x0, int y0, int i, int j) {
  typedef Step2<R> G;
  const int nx = P.w.nx, ny = P.w.ny;
  const double Xd[2] = {(double)(P.w.px + i), (double)(P.w.py + j)};
  const int vo = (j - y0 + 1) * G::VX + (i - x0 + 1);
  T V[2];
  V[0] = vmid(S.u[vo], S.u[vo + 1]);
  V[1] = vmid(S.v[vo], S.v[vo + G::VX]);
  if (BT == DCL_RK2) {
    const double Xm[2] = {Xd[0] - (double)V[0] * P.ch[0], Xd[1] - (double)V[1] * P.ch[1]};
    int b0[3], b1[3];
    T f0[3], f1[3];
    mac_split<T, 2>(P.v, Xm, b0, b1, f0, f1);
    // b0 <= b1 <= b0 + 1 along each axis
    const int lx = b0[0] - (x0 - 1), ly = b0[1] - (y0 - 1);
    const bool in = lx >= 0 && b1[0] - (x0 - 1) <= G::VX - 2 && ly >= 0 && ly <= G::VY - 3 &&
                    b1[1] - (y0 - 1) <= G::VY - 2;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int ix = c == 0 ? b1[0] : b0[0], iy = c == 1 ? b1[1] : b0[1];
      const T x1 = c == 0 ? f1[0] : f0[0], y1 = c == 1 ? f1[1] : f0[1];
      T a00, a10, a01, a11;
      if (in) {
        const lds_cptr<T> q = (lds_cptr<T>)(c == 0 ? S.u : S.v) + (iy - (y0 - 1)) * G::VX + (ix - (x0 - 1));
        a00 = q[0], a10 = q[1], a01 = q[G::VX], a11 = q[G::VX + 1];
      } else {
        const T* q = vel + (iy * nx + ix) * P.v.dof + P.v.udof + c * P.v.cs;
        const int sx = P.v.dof, sy = nx * P.v.dof;
        a00 = q[0], a10 = q[sx], a01 = q[sy], a11 = q[sy + sx];
      }
      V[c] = vlerp(vlerp(a00, a10, x1), vlerp(a01, a11, x1), y1);
    }
  }
  const double X = Xd[0] - (double)V[0] * P.c[0], Y = Xd[1] - (double)V[1] * P.c[1];
  double fx, fy;
  constexpr int NP = INTERP == DCL_CUBIC ? 4 : 2;
  int bx, by;
  if (INTERP == DCL_CUBIC) {
    bx = cub_split(X, P.w.px, nx, fx) - 1;
    by = cub_split(Y, P.w.py, ny, fy) - 1;
  } else {
    bx = lin_split(X, P.w.px, nx, fx);
    by = lin_split(Y, P.w.py, ny, fy);
  }
  const int lx = bx - (x0 - S2_H), ly = by - (y0 - S2_H);
  const bool in = (unsigned)lx <= (unsigned)(G::PX - NP) && (unsigned)ly <= (unsigned)(G::PY - NP);
  T rows[NP][NP];
  if (in) {
#pragma unroll
    for (int b = 0; b < NP; ++b)
#pragma unroll
      for (int a = 0; a < NP; ++a) rows[b][a] = ((lds_cptr<T>)S.phi)[(ly + b) * G::PX + lx + a];
  } else {
#pragma unroll
    for (int b = 0; b < NP; ++b)
#pragma unroll
      for (int a = 0; a < NP; ++a) rows[b][a] = phi0[(by + b) * nx + bx + a];
  }
  if constexpr (INTERP == DCL_CUBIC) {
    T wx[4], wy[4];
    cr_weights<T>((T)fx, wx);
    cr_weights<T>((T)fy, wy);
    T sum = T(0);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      T sx = T(0);
#pragma unroll
      for (int a = 0; a < 4; ++a) sx = fma(wx[a], rows[b][a], sx);
      sum = fma(wy[b], sx, sum);
    }
    return sum;
  } else {
    return bilinear_sum2d<T>(rows[0], rows[1], fx, fy);
  }
}

// one tile: output nodes (ox .. ox + cols - 1, oy .. oy + OY - 1), cols as
// step2d_cols says, clipped to the window; kappa may be NULL (phi only).  Every thread of the block calls it; it ends on a barrier.
template <typename T, int INTERP, int BT, int R>
__device__ __forceinline__ void step2d_tile(const T* __restrict__ phi0, T* __restrict__ phi, T* __restrict__ kappa,
                                            const T* __restrict__ vel, const SLP& P, T dx, T dy, const Curv2R<T>& cr, int ox,
                                            int oy, int cols, Step2Lds<T, R>& S) {
  typedef Step2<R> G;
  const int nx = P.w.nx, ny = P.w.ny;
  const bool wide = G::WIDE && cols == S2_TX;
  const int x0 = wide ? ox : ox - 1, y0 = oy - 1;
  const int tid = threadIdx.x + S2_TX * threadIdx.y;
  constexpr int NP = (G::PX * G::PY + G::NT - 1) / G::NT, NV = (G::VX * G::VY + G::NT - 1) / G::NT;
  T pv[NP], vv[NV][2];
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    const int e = min(tid + q * G::NT, G::PX * G::PY - 1);
    const int by = e / G::PX, bx = e - by * G::PX;
    pv[q] = phi0[clampi(y0 - S2_H + by, 0, ny - 1) * nx + clampi(x0 - S2_H + bx, 0, nx - 1)];
  }
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const int e = min(tid + q * G::NT, G::VX * G::VY - 1);
    const int by = e / G::VX, bx = e - by * G::VX;
    const T* p = vel + (clampi(y0 - 1 + by, 0, ny - 1) * nx + clampi(x0 - 1 + bx, 0, nx - 1)) * P.v.dof + P.v.udof;
    vv[q][0] = p[0];
    vv[q][1] = p[P.v.cs];
  }
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    const int e = tid + q * G::NT;
    if (e < G::PX * G::PY) S.phi[e] = pv[q];
  }
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    const int e = tid + q * G::NT;
    if (e < G::VX * (G::VY - 1)) S.u[e] = vv[q][0];
    if (e < G::VX * G::VY) S.v[e] = vv[q][1];
  }
  __syncthreads();
  constexpr int C0 = G::WIDE ? 1 : 0;  // of the new phi: the column before the area
  auto work = [&](int i, int j, int col, int row) {
    T v = S.phi[(row + S2_H) * G::PX + col + S2_H];
    if (i >= 2 && i <= nx - 3 && j >= 2 && j <= ny - 3)
      v = step2d_node<T, INTERP, BT, R>(phi0, vel, P, S, x0, y0, i, j);
    S.out[row * G::AX + col + C0] = v;
  };
  const int i = x0 + (int)threadIdx.x;
#pragma unroll 1
  for (int row = threadIdx.y; row < G::AY; row += S2_TY) work(i, y0 + row, threadIdx.x, row);
  if (G::WIDE && wide && tid < 2 * G::AY) {
    const int col = tid < G::AY ? -1 : S2_TX, row = tid % G::AY;
    work(x0 + col, y0 + row, col, row);
  }
  __syncthreads();
  if (i < nx && (wide || (threadIdx.x >= 1 && threadIdx.x <= G::OX))) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = threadIdx.y + S2_TY * r, j = y0 + row;
      if (row < 1 || row > G::OY || j >= ny) continue;
      const lds_cptr<T> p = (lds_cptr<T>)S.out + row * G::AX + threadIdx.x + C0;
      phi[j * nx + i] = p[0];
      if (!kappa) continue;
      T k = T(0);
      if (i >= 1 && i <= nx - 2 && j >= 1 && j <= ny - 2) k = curv2d_recip_at<T>(p, G::AX, dx, dy, cr);
      kappa[j * nx + i] = k;
    }
  }
  __syncthreads();
}

}  // namespace dcl
