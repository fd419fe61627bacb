// Matrix-free Helmholtz stencil, damped Jacobi, grid transfers, casts and the
// dense coarsest-level solve.  All HBM-bound streaming kernels.
//
// Operator (src/GetHelmholtz.jl:33-50, src/PlainNodalLaplacian.jl:18-46):
//   (A x)_p = sum_d (2 x_p - x~_{p-e_d} - x~_{p+e_d}) / h_d^2 + d_p x_p
// with mirror ghosts (BC=2) or ghost = self (BC=1) on every face, and the
// per-node complex diagonal d_p = -w^2 m_p (1 - i g_p / Re w) + Sommerfeld
// terms (+ i s w^2 m_p for a shifted operator).
//
// Launch shape: 256 threads over consecutive positions of a row (2-D) or of
// a plane or a band of rows (3-D), numbered across the grid so no lane idles at a
// ragged row end; each thread marches a run of rows/planes along the slowest axis
// keeping the previous/current/next values in registers.  In-plane neighbours come
// from the caches (small blocks) or from the neighbouring lanes.  The XCD-aware
// block order groups right-hand sides that share the diagonal in L2.
#include "hh_kernels.h"

#include <algorithm>

namespace hh {

template <typename TD>
__device__ __forceinline__ cx<TD> node_diag(const cx<TD>* __restrict__ d, const double* __restrict__ m,
                                            cx<double> sfac, int64_t p) {
  cx<TD> dv = d[p];
  if (m) {
    double mv = m[p];
    dv.re += (TD)(sfac.re * mv);
    dv.im += (TD)(sfac.im * mv);
  }
  return dv;
}

// What a mode makes of A x at one node; M_JACOBI: x + F (b - A x) with the level's
// precomputed damped-Jacobi factor F = wj (d + diag of the Laplacian)^-1 when fj is
// given, else wj (b - A x) / Dtot
template <typename TO, typename TD, int MODE>
__device__ __forceinline__ cx<TO> finish(cx<TD> xc, cx<TD> Ax, cx<TO> bo, cx<TD> Dtot, TD wj, bool has_f, cx<TD> f) {
  if (MODE == M_APPLY) return cvt<TD, TO>(Ax);
  const cx<TD> r = cvt<TO, TD>(bo) - Ax;
  if (MODE == M_RESID) return cvt<TD, TO>(r);
  return cvt<TD, TO>(xc + (has_f ? cmul_fma(f, r) : wj * cmul_fma(r, cinv(Dtot))));
}

// Small blocks (x in L2): one thread per (column position, run of `rows`
// rows/planes), the positions of a row (2-D) or of a plane (3-D) numbered
// consecutively across the whole grid so no lane idles at a ragged row end; each
// thread marches its run along the slowest axis keeping the previous/current/next
// values in registers and reads its in-plane neighbours from the caches.
template <typename TI, typename TO, typename TD, int MODE>
__global__ __launch_bounds__(256) void k_stencil2d(Grid g, const cx<TI>* __restrict__ x,
                                                   const cx<TO>* __restrict__ b, cx<TO>* __restrict__ y,
                                                   const cx<TD>* __restrict__ d, const double* __restrict__ m,
                                                   cx<double> sfac, TD wj, int rows, TileMap tm,
                                                   const int* __restrict__ skip, const cx<TD>* __restrict__ fj) {
  int bx, by, rhs;
  tile_of(tm, bx, by, rhs);
  if (skip && skip[rhs]) return;
  const int n1 = g.n1, n2 = g.n2;
  const unsigned item = (unsigned)bx * 256u + threadIdx.x, band = item / (unsigned)n1;
  const int i = (int)(item - band * (unsigned)n1);
  const int j0 = (int)band * rows;
  if (j0 >= n2) return;
  const int j1 = min(j0 + rows, n2);
  const int64_t off = (int64_t)rhs * g.N;
  const cx<TI>* xr = x + off;
  const cx<TO>* bo = MODE == M_APPLY ? nullptr : b + off;
  cx<TO>* yo = y + off;
  const int il = lo_nb(i, g.bc), ir = hi_nb(i, n1, g.bc);
  const TD ih1 = (TD)g.ih1, ih2 = (TD)g.ih2;
  const TD ldx = (TD)(g.ih1 * lap_diag1(i, n1, g.bc));
  cx<TD> xm = cvt<TI, TD>(xr[(int64_t)lo_nb(j0, g.bc) * n1 + i]);
  cx<TD> xc = cvt<TI, TD>(xr[(int64_t)j0 * n1 + i]);
  for (int j = j0; j < j1; ++j) {
    const int64_t row = (int64_t)j * n1;
    const int jp = hi_nb(j, n2, g.bc);
    cx<TD> xp = cvt<TI, TD>(xr[(int64_t)jp * n1 + i]);
    cx<TD> xl = cvt<TI, TD>(xr[row + il]);
    cx<TD> xrr = cvt<TI, TD>(xr[row + ir]);
    const int64_t p = row + i;
    cx<TD> dv = node_diag<TD>(d, m, sfac, p);
    cx<TD> Ax = apply5(xc, xl, xrr, xm, xp, ih1, ih2, dv);
    cx<TD> Dtot = dv;
    if (MODE == M_JACOBI && !fj) {
      Dtot.re += ldx + (TD)(g.ih2 * lap_diag1(j, n2, g.bc));
    }
    yo[p] = finish<TO, TD, MODE>(xc, Ax, MODE == M_APPLY ? mk<TO>(0, 0) : bo[p], Dtot, wj, fj != nullptr,
                                 MODE == M_JACOBI && fj ? fj[p] : mk<TD>(0, 0));
    xm = xc;
    xc = xp;
  }
}

template <typename TI, typename TO, typename TD, int MODE>
__global__ __launch_bounds__(256) void k_stencil3d(Grid g, const cx<TI>* __restrict__ x,
                                                   const cx<TO>* __restrict__ b, cx<TO>* __restrict__ y,
                                                   const cx<TD>* __restrict__ d, const double* __restrict__ m,
                                                   cx<double> sfac, TD wj, int rows, TileMap tm,
                                                   const int* __restrict__ skip, const cx<TD>* __restrict__ fj) {
  int bx, by, rhs;
  tile_of(tm, bx, by, rhs);
  if (skip && skip[rhs]) return;
  const int n1 = g.n1, n2 = g.n2, n3 = g.n3;
  const unsigned item = (unsigned)bx * 256u + threadIdx.x, jj = item / (unsigned)n1;
  const int i = (int)(item - jj * (unsigned)n1), j = (int)jj;
  const int k0 = by * rows;
  if (j >= n2 || k0 >= n3) return;
  const int k1 = min(k0 + rows, n3);
  const int64_t plane = (int64_t)n1 * n2;
  const int64_t off = (int64_t)rhs * g.N;
  const cx<TI>* xr = x + off;
  const cx<TO>* bo = MODE == M_APPLY ? nullptr : b + off;
  cx<TO>* yo = y + off;
  const int il = lo_nb(i, g.bc), ir = hi_nb(i, n1, g.bc);
  const int jl = lo_nb(j, g.bc), jr = hi_nb(j, n2, g.bc);
  const TD ih1 = (TD)g.ih1, ih2 = (TD)g.ih2, ih3 = (TD)g.ih3;
  const TD ldxy = (TD)(g.ih1 * lap_diag1(i, n1, g.bc) + g.ih2 * lap_diag1(j, n2, g.bc));
  const int64_t col = (int64_t)j * n1 + i;
  const int64_t c1l = (int64_t)j * n1 + il, c1r = (int64_t)j * n1 + ir;
  const int64_t c2l = (int64_t)jl * n1 + i, c2r = (int64_t)jr * n1 + i;
  cx<TD> xm = cvt<TI, TD>(xr[(int64_t)lo_nb(k0, g.bc) * plane + col]);
  cx<TD> xc = cvt<TI, TD>(xr[(int64_t)k0 * plane + col]);
  for (int k = k0; k < k1; ++k) {
    const int64_t pl = (int64_t)k * plane;
    const int kp = hi_nb(k, n3, g.bc);
    cx<TD> xp = cvt<TI, TD>(xr[(int64_t)kp * plane + col]);
    cx<TD> x1l = cvt<TI, TD>(xr[pl + c1l]);
    cx<TD> x1r = cvt<TI, TD>(xr[pl + c1r]);
    cx<TD> x2l = cvt<TI, TD>(xr[pl + c2l]);
    cx<TD> x2r = cvt<TI, TD>(xr[pl + c2r]);
    const int64_t p = pl + col;
    cx<TD> dv = node_diag<TD>(d, m, sfac, p);
    cx<TD> Ax = apply7(xc, x1l, x1r, x2l, x2r, xm, xp, ih1, ih2, ih3, dv);
    cx<TD> Dtot = dv;
    if (MODE == M_JACOBI && !fj) {
      Dtot.re += ldxy + (TD)(g.ih3 * lap_diag1(k, n3, g.bc));
    }
    yo[p] = finish<TO, TD, MODE>(xc, Ax, MODE == M_APPLY ? mk<TO>(0, 0) : bo[p], Dtot, wj, fj != nullptr,
                                 MODE == M_JACOBI && fj ? fj[p] : mk<TD>(0, 0));
    xm = xc;
    xc = xp;
  }
}

// neighbour lanes' values: lane l gets lane l - 1's (l + 1's), lane 0 (63) its own e
__device__ __forceinline__ float lane_below(float v, float e) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(e), __float_as_int(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_above(float v, float e) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(e), __float_as_int(v), 0x130, 0xf, 0xf, false));
}
__device__ __forceinline__ double lane_below(double v, double e) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(__double2hiint(e), __double2hiint(v), 0x138, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(__double2loint(e), __double2loint(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ double lane_above(double v, double e) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(__double2hiint(e), __double2hiint(v), 0x130, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(__double2loint(e), __double2loint(v), 0x130, 0xf, 0xf, false));
}

// x neighbours of a thread's node from the wavefront's own values: lane l holds
// position l of 64 consecutive ones, so the node to the left (right) is in lane
// l - 1 (l + 1) unless the row ends there (mirror or self ghost) or the
// wavefront does (lanes 0 and 63: one value read at `at`).
struct XEdge {
  int at;  // position in the row that lane 0 / 63 reads beside its own, -1: none
  bool first, last, mirror;
  __device__ __forceinline__ void init(int i, int n1, int bc) {
    const int lane = threadIdx.x & 63;
    first = i == 0;
    last = i == n1 - 1;
    mirror = bc == 2;
    at = lane == 0 && !first ? i - 1 : (lane == 63 && !last ? i + 1 : -1);
  }
  template <typename T>
  __device__ __forceinline__ void neighbours(cx<T> c, cx<T> e, cx<T>& l, cx<T>& r) const {
    const cx<T> lo = mk<T>(lane_below(c.re, e.re), lane_below(c.im, e.im));
    const cx<T> hi = mk<T>(lane_above(c.re, e.re), lane_above(c.im, e.im));
    l = first ? (mirror ? hi : c) : lo;
    r = last ? (mirror ? lo : c) : hi;
  }
};

// Larger blocks: the gathering kernels above load five (2-D: three) values of x a node
// and read a plane's neighbours a step after the plane itself, when part of it has left
// L1 and L2: 193 x 193 x 97 x 32 complex64 took 55.7 million L2 requests and read 2.03 GB
// for 0.93 (663 us).  Here every value that a thread needs is loaded once, a step ahead,
// and kept: the x neighbours come from the neighbouring lanes' registers, in 3-D a thread
// owns RY rows of a column and reads them and the row on either side.  39.1 million
// requests, 520 us, 3.6 TB/s of x and y; 1.92 GB are still read, since the rows between
// two bands and the planes between two runs mostly miss L2 (1025 x 513 x 64 complex64:
// 0.58 -> 0.47 GB for 0.27, 157 -> 125-150 us).
// 2-D: one thread per (column position, run of `rows` rows) numbered as above.
template <typename TI, typename TO, typename TD, int MODE>
__global__ __launch_bounds__(256) void k_march2d(Grid g, const cx<TI>* __restrict__ x,
                                                   const cx<TO>* __restrict__ b, cx<TO>* __restrict__ y,
                                                   const cx<TD>* __restrict__ d, const double* __restrict__ m,
                                                   cx<double> sfac, TD wj, int rows, TileMap tm,
                                                   const int* __restrict__ skip, const cx<TD>* __restrict__ fj) {
  int bx, by, rhs;
  tile_of(tm, bx, by, rhs);
  if (skip && skip[rhs]) return;
  const int n1 = g.n1, n2 = g.n2;
  const unsigned item = (unsigned)bx * 256u + threadIdx.x, band = item / (unsigned)n1;
  const int i = (int)(item - band * (unsigned)n1);
  // lanes past the last band walk the last row and store nothing (their
  // neighbours in the wavefront read their registers)
  const bool own = (int64_t)band * rows < n2;
  const int j0 = own ? (int)band * rows : n2 - 1;
  const int64_t off = (int64_t)rhs * g.N;
  const cx<TI>* xr = x + off;
  const cx<TO>* bo = MODE == M_APPLY ? nullptr : b + off;
  cx<TO>* yo = y + off;
  XEdge ed;
  ed.init(i, n1, g.bc);
  const TD ih1 = (TD)g.ih1, ih2 = (TD)g.ih2;
  const TD ldx = (TD)(g.ih1 * lap_diag1(i, n1, g.bc));
  const cx<TI> zi = mk<TI>(0, 0);
  cx<TI> xm = xr[(int64_t)lo_nb(j0, g.bc) * n1 + i];
  cx<TI> xc = xr[(int64_t)j0 * n1 + i];
  cx<TI> ec = ed.at >= 0 ? xr[(int64_t)j0 * n1 + ed.at] : zi;
  for (int s = 0; s < rows; ++s) {
    const int j = min(j0 + s, n2 - 1);
    const int64_t row = (int64_t)j * n1, up = (int64_t)hi_nb(j, n2, g.bc) * n1;
    const int64_t p = row + i;
    const cx<TI> xp = xr[up + i];
    const cx<TI> ep = ed.at >= 0 ? xr[up + ed.at] : zi;
    const cx<TD> dv = node_diag<TD>(d, m, sfac, p);
    const cx<TO> bv = MODE == M_APPLY ? mk<TO>(0, 0) : bo[p];
    const cx<TD> fv = MODE == M_JACOBI && fj ? fj[p] : mk<TD>(0, 0);
    cx<TI> xl, xrr;
    ed.neighbours(xc, ec, xl, xrr);
    const cx<TD> c = cvt<TI, TD>(xc);
    const cx<TD> Ax = apply5(c, cvt<TI, TD>(xl), cvt<TI, TD>(xrr), cvt<TI, TD>(xm), cvt<TI, TD>(xp), ih1, ih2, dv);
    cx<TD> Dtot = dv;
    if (MODE == M_JACOBI && !fj) Dtot.re += ldx + (TD)(g.ih2 * lap_diag1(j, n2, g.bc));
    if (own && j0 + s < n2) yo[p] = finish<TO, TD, MODE>(c, Ax, bv, Dtot, wj, fj != nullptr, fv);
    xm = xc;
    xc = xp;
    ec = ep;
  }
}

// 3-D: a thread owns RY nodes of one in-plane column, rows j0 .. j0 + RY - 1, over a
// run of `rows` planes; the columns of a band of RY rows are numbered consecutively
// over the bands.
template <typename TI, typename TO, typename TD, int MODE, int RY>
__global__ __launch_bounds__(256) void k_march3d(Grid g, const cx<TI>* __restrict__ x,
                                                   const cx<TO>* __restrict__ b, cx<TO>* __restrict__ y,
                                                   const cx<TD>* __restrict__ d, const double* __restrict__ m,
                                                   cx<double> sfac, TD wj, int rows, TileMap tm,
                                                   const int* __restrict__ skip, const cx<TD>* __restrict__ fj) {
  int bx, by, rhs;
  tile_of(tm, bx, by, rhs);
  if (skip && skip[rhs]) return;
  const int n1 = g.n1, n2 = g.n2, n3 = g.n3;
  const unsigned item = (unsigned)bx * 256u + threadIdx.x, band = item / (unsigned)n1;
  const int i = (int)(item - band * (unsigned)n1);
  const int k0 = by * rows;
  const int k1 = min(k0 + rows, n3);
  // lanes past the last band walk the last row and store nothing
  const int j0 = min((int)band * RY, n2 - 1);
  const bool own = (int64_t)band * RY < n2;
  const int64_t plane = (int64_t)n1 * n2;
  const int64_t off = (int64_t)rhs * g.N;
  const cx<TI>* xr = x + off;
  const cx<TO>* bo = MODE == M_APPLY ? nullptr : b + off;
  cx<TO>* yo = y + off;
  XEdge ed;
  ed.init(i, n1, g.bc);
  const TD ih1 = (TD)g.ih1, ih2 = (TD)g.ih2, ih3 = (TD)g.ih3;
  const TD ldx = (TD)(g.ih1 * lap_diag1(i, n1, g.bc));
  // rows j0 - 1 .. j0 + RY with their ghosts (a row past the ghost row is never used)
  int rw[RY + 2];
#pragma unroll
  for (int r = 0; r < RY + 2; ++r) {
    const int t = j0 + r - 1;
    rw[r] = (t < 0 ? lo_nb(0, g.bc) : (t < n2 ? t : (t == n2 ? hi_nb(n2 - 1, n2, g.bc) : n2 - 1))) * n1;
  }
  const cx<TI> zi = mk<TI>(0, 0);
  cx<TI> xm[RY], xc[RY + 2], ec[RY];
#pragma unroll
  for (int r = 0; r < RY; ++r) {
    xm[r] = xr[(int64_t)lo_nb(k0, g.bc) * plane + rw[r + 1] + i];
    ec[r] = ed.at >= 0 ? xr[(int64_t)k0 * plane + rw[r + 1] + ed.at] : zi;
  }
#pragma unroll
  for (int r = 0; r < RY + 2; ++r) xc[r] = xr[(int64_t)k0 * plane + rw[r] + i];
  for (int k = k0; k < k1; ++k) {
    const int64_t pl = (int64_t)k * plane;
    const cx<TI>* xu = xr + (int64_t)hi_nb(k, n3, g.bc) * plane;
    cx<TI> xp[RY + 2], ep[RY];
    cx<TD> dv[RY], fv[RY];
    cx<TO> bv[RY];
#pragma unroll
    for (int r = 0; r < RY; ++r) {
      const int64_t p = pl + rw[r + 1] + i;
      xp[r + 1] = xu[rw[r + 1] + i];
      dv[r] = node_diag<TD>(d, m, sfac, p);
      bv[r] = MODE == M_APPLY ? mk<TO>(0, 0) : bo[p];
      fv[r] = MODE == M_JACOBI && fj ? fj[p] : mk<TD>(0, 0);
    }
    xp[0] = xp[RY + 1] = zi;
#pragma unroll
    for (int r = 0; r < RY; ++r) ep[r] = zi;
    if (k + 1 < k1) {  // the next step's in-plane neighbours
      xp[0] = xu[rw[0] + i];
      xp[RY + 1] = xu[rw[RY + 1] + i];
      if (ed.at >= 0)
#pragma unroll
        for (int r = 0; r < RY; ++r) ep[r] = xu[rw[r + 1] + ed.at];
    }
#pragma unroll
    for (int r = 0; r < RY; ++r) {
      cx<TI> xl, xrr;
      ed.neighbours(xc[r + 1], ec[r], xl, xrr);
      const cx<TD> c = cvt<TI, TD>(xc[r + 1]);
      const cx<TD> Ax = apply7(c, cvt<TI, TD>(xl), cvt<TI, TD>(xrr), cvt<TI, TD>(xc[r]), cvt<TI, TD>(xc[r + 2]),
                               cvt<TI, TD>(xm[r]), cvt<TI, TD>(xp[r + 1]), ih1, ih2, ih3, dv[r]);
      cx<TD> Dtot = dv[r];
      if (MODE == M_JACOBI && !fj)
        Dtot.re += (TD)(ldx + (TD)(g.ih2 * lap_diag1(j0 + r, n2, g.bc))) + (TD)(g.ih3 * lap_diag1(k, n3, g.bc));
      if (own && j0 + r < n2)
        yo[pl + rw[r + 1] + i] = finish<TO, TD, MODE>(c, Ax, bv[r], Dtot, wj, fj != nullptr, fv[r]);
    }
#pragma unroll
    for (int r = 0; r < RY; ++r) {
      xm[r] = xc[r + 1];
      ec[r] = ep[r];
    }
#pragma unroll
    for (int r = 0; r < RY + 2; ++r) xc[r] = xp[r];
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_jacobi0(Grid g, const cx<T>* __restrict__ b, cx<T>* __restrict__ x,
                                                 const cx<T>* __restrict__ f, const int* __restrict__ skip) {
  const int rhs = blockIdx.y;
  if (skip && skip[rhs]) return;
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= g.N) return;
  const int64_t o = (int64_t)rhs * g.N + p;
  x[o] = cmul_fma(f[p], b[o]);
}

// Full weighting with mirror ghosts, fine residual -> coarse right-hand side.
template <typename T>
__global__ __launch_bounds__(256) void k_restrict(Grid gf, Grid gc, const cx<T>* __restrict__ rf,
                                                  cx<T>* __restrict__ bc, const int* __restrict__ skip) {
  const int rhs = blockIdx.y;
  if (skip && skip[rhs]) return;
  const int64_t pc = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (pc >= gc.N) return;
  int I, J, K;
  node_coords(gc, pc, I, J, K);
  const cx<T>* r = rf + (int64_t)rhs * gf.N;
  const T w[3] = {(T)0.25, (T)0.5, (T)0.25};
  cx<T> acc = mk<T>(0, 0);
  const int kk = gf.dim == 3 ? 3 : 1;
  for (int c = 0; c < kk; ++c) {
    int fk = 0;
    T wk = (T)1;
    if (gf.dim == 3) {
      int f = 2 * K + c - 1;
      fk = f < 0 ? 1 : (f >= gf.n3 ? gf.n3 - 2 : f);
      wk = w[c];
    }
    for (int bb = 0; bb < 3; ++bb) {
      int f2 = 2 * J + bb - 1;
      int fj = f2 < 0 ? 1 : (f2 >= gf.n2 ? gf.n2 - 2 : f2);
      for (int a = 0; a < 3; ++a) {
        int f1 = 2 * I + a - 1;
        int fi = f1 < 0 ? 1 : (f1 >= gf.n1 ? gf.n1 - 2 : f1);
        acc = acc + (wk * w[bb] * w[a]) * r[((int64_t)fk * gf.n2 + fj) * gf.n1 + fi];
      }
    }
  }
  bc[(int64_t)rhs * gc.N + pc] = acc;
}

// 3-D full weighting marching along z: a thread owns one coarse (I, J) column
// over a run of coarse planes; the in-plane 9-point weighted sum s_f of each
// fine plane f at (I, J) is formed once and the coarse value is
// s_{2K-1} / 4 + s_{2K} / 2 + s_{2K+1} / 4 (mirror ghosts on every axis).
template <typename T>
__global__ __launch_bounds__(256) void k_restrict3(Grid gf, Grid gc, int rows, TileMap tm,
                                                   const cx<T>* __restrict__ rf, cx<T>* __restrict__ bc,
                                                   const int* __restrict__ skip) {
  int bx, by, rhs;
  tile_of(tm, bx, by, rhs);
  if (skip && skip[rhs]) return;
  const unsigned item = (unsigned)bx * 256u + threadIdx.x, JJ = item / (unsigned)gc.n1;
  const int I = (int)(item - JJ * (unsigned)gc.n1), J = (int)JJ;
  const int K0 = by * rows;
  if (J >= gc.n2 || K0 >= gc.n3) return;
  const int K1 = min(K0 + rows, gc.n3);
  const cx<T>* r = rf + (int64_t)rhs * gf.N;
  cx<T>* out = bc + (int64_t)rhs * gc.N;
  const T w[3] = {(T)0.25, (T)0.5, (T)0.25};
  int64_t cols[3][3];
  for (int bb = 0; bb < 3; ++bb) {
    const int f2 = 2 * J + bb - 1;
    const int fj = f2 < 0 ? 1 : (f2 >= gf.n2 ? gf.n2 - 2 : f2);
    for (int aa = 0; aa < 3; ++aa) {
      const int f1 = 2 * I + aa - 1;
      const int fi = f1 < 0 ? 1 : (f1 >= gf.n1 ? gf.n1 - 2 : f1);
      cols[bb][aa] = (int64_t)fj * gf.n1 + fi;
    }
  }
  const int64_t plane = (int64_t)gf.n1 * gf.n2;
  auto plane_sum = [&](int f) {
    const int fk = f < 0 ? 1 : (f >= gf.n3 ? gf.n3 - 2 : f);
    const cx<T>* rp = r + (int64_t)fk * plane;
    cx<T> acc = mk<T>(0, 0);
    for (int bb = 0; bb < 3; ++bb)
      for (int aa = 0; aa < 3; ++aa) acc = acc + (w[bb] * w[aa]) * rp[cols[bb][aa]];
    return acc;
  };
  const int64_t ccol = (int64_t)J * gc.n1 + I, cplane = (int64_t)gc.n1 * gc.n2;
  cx<T> sm = plane_sum(2 * K0 - 1);
  for (int K = K0; K < K1; ++K) {
    const cx<T> s0 = plane_sum(2 * K), sp = plane_sum(2 * K + 1);
    out[(int64_t)K * cplane + ccol] = w[0] * sm + w[1] * s0 + w[2] * sp;
    sm = sp;
  }
}

// Same full weighting on a real nodal coefficient field (m, gamma).
__global__ __launch_bounds__(256) void k_restrict_real(Grid gf, Grid gc, const double* __restrict__ f,
                                                       double* __restrict__ c) {
  const int64_t pc = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (pc >= gc.N) return;
  const int I = (int)(pc % gc.n1);
  const int64_t q = pc / gc.n1;
  const int J = (int)(q % gc.n2);
  const int K = (int)(q / gc.n2);
  const double w[3] = {0.25, 0.5, 0.25};
  double acc = 0.0;
  const int kk = gf.dim == 3 ? 3 : 1;
  for (int cc = 0; cc < kk; ++cc) {
    int fk = 0;
    double wk = 1.0;
    if (gf.dim == 3) {
      int fz = 2 * K + cc - 1;
      fk = fz < 0 ? 1 : (fz >= gf.n3 ? gf.n3 - 2 : fz);
      wk = w[cc];
    }
    for (int bb = 0; bb < 3; ++bb) {
      int f2 = 2 * J + bb - 1;
      int fj = f2 < 0 ? 1 : (f2 >= gf.n2 ? gf.n2 - 2 : f2);
      for (int a = 0; a < 3; ++a) {
        int f1 = 2 * I + a - 1;
        int fi = f1 < 0 ? 1 : (f1 >= gf.n1 ? gf.n1 - 2 : f1);
        acc += wk * w[bb] * w[a] * f[((int64_t)fk * gf.n2 + fj) * gf.n1 + fi];
      }
    }
  }
  c[pc] = acc;
}

// Bi/tri-linear nodal prolongation of the coarse correction, added in place.
template <typename T>
__global__ __launch_bounds__(256) void k_prolong_add(Grid gf, Grid gc, const cx<T>* __restrict__ xc,
                                                     cx<T>* __restrict__ xf, const int* __restrict__ skip) {
  const int rhs = blockIdx.y;
  if (skip && skip[rhs]) return;
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= gf.N) return;
  int i, j, k;
  node_coords(gf, p, i, j, k);
  const cx<T>* c = xc + (int64_t)rhs * gc.N;
  const int i0 = i >> 1, j0 = j >> 1, k0 = k >> 1;
  const int i1 = (i & 1) ? i0 + 1 : i0, j1 = (j & 1) ? j0 + 1 : j0, k1 = (k & 1) ? k0 + 1 : k0;
  const T wi = (i & 1) ? (T)0.5 : (T)1, wj = (j & 1) ? (T)0.5 : (T)1, wk = (k & 1) ? (T)0.5 : (T)1;
  const int64_t P1 = gc.n1, P2 = (int64_t)gc.n1 * gc.n2;
  cx<T> acc = mk<T>(0, 0);
  const int ik[2] = {i0, i1}, jk[2] = {j0, j1}, kk[2] = {k0, k1};
  const int ni = (i & 1) ? 2 : 1, nj = (j & 1) ? 2 : 1, nk = (k & 1) ? 2 : 1;
  for (int c3 = 0; c3 < nk; ++c3)
    for (int c2 = 0; c2 < nj; ++c2)
      for (int c1 = 0; c1 < ni; ++c1) acc = acc + (wi * wj * wk) * c[kk[c3] * P2 + jk[c2] * P1 + ik[c1]];
  const int64_t o = (int64_t)rhs * gf.N + p;
  xf[o] = xf[o] + acc;
}

// 3-D prolongation marching along z: a thread owns one fine (i, j) column
// over a run of fine planes starting at an even plane.  The in-plane bilinear
// value of each coarse plane K at (i, j) is formed once (weights 1 or 1/2 per
// axis) and reused: fine plane 2K adds c_K, fine plane 2K + 1 adds
// (c_K + c_{K+1}) / 2.
template <typename T>
__global__ __launch_bounds__(256) void k_prolong_add3(Grid gf, Grid gc, int rows, TileMap tm,
                                                      const cx<T>* __restrict__ xc, cx<T>* __restrict__ xf,
                                                      const int* __restrict__ skip) {
  int bx, by, rhs;
  tile_of(tm, bx, by, rhs);
  if (skip && skip[rhs]) return;
  const int n1 = gf.n1, n2 = gf.n2;
  const unsigned item = (unsigned)bx * 256u + threadIdx.x, jj = item / (unsigned)n1;
  const int i = (int)(item - jj * (unsigned)n1), j = (int)jj;
  const int k0 = by * rows;
  if (j >= n2 || k0 >= gf.n3) return;
  const int k1 = min(k0 + rows, gf.n3);
  const cx<T>* c = xc + (int64_t)rhs * gc.N;
  cx<T>* x = xf + (int64_t)rhs * gf.N;
  const int i0 = i >> 1, j0 = j >> 1;
  const int i1 = (i & 1) ? i0 + 1 : i0, j1 = (j & 1) ? j0 + 1 : j0;
  const T wi = (i & 1) ? (T)0.5 : (T)1, wj = (j & 1) ? (T)0.5 : (T)1;
  const int64_t P1 = gc.n1, P2 = (int64_t)gc.n1 * gc.n2;
  const int64_t a00 = j0 * P1 + i0, a01 = j0 * P1 + i1, a10 = j1 * P1 + i0, a11 = j1 * P1 + i1;
  const bool two_i = (i & 1) != 0, two_j = (j & 1) != 0;
  auto plane_val = [&](int K) {
    const cx<T>* cp = c + (int64_t)K * P2;
    cx<T> acc = (wi * wj) * cp[a00];
    if (two_i) acc = acc + (wi * wj) * cp[a01];
    if (two_j) {
      acc = acc + (wi * wj) * cp[a10];
      if (two_i) acc = acc + (wi * wj) * cp[a11];
    }
    return acc;
  };
  const int64_t plane = (int64_t)n1 * n2, col = (int64_t)j * n1 + i;
  cx<T> cK = plane_val(k0 >> 1);
  for (int k = k0; k < k1; ++k) {
    cx<T> e;
    if (k & 1) {
      const cx<T> cK1 = plane_val((k >> 1) + 1);
      e = (T)0.5 * (cK + cK1);
      cK = cK1;
    } else {
      e = cK;
    }
    const int64_t o = (int64_t)k * plane + col;
    x[o] = x[o] + e;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_zero(cx<T>* __restrict__ a, int64_t n) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p < n) a[p] = mk<T>(0, 0);
}

template <typename A, typename B>
__global__ __launch_bounds__(256) void k_cast(const cx<A>* __restrict__ a, cx<B>* __restrict__ b, int64_t n) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p < n) b[p] = cvt<A, B>(a[p]);
}

// Nodal diagonal d = -w^2 m (1 - i g/Re w) + i Re(w) sqrt(m) sum_faces 2/h_d
// (src/GetHelmholtz.jl:41-47, 222-247; Sommerfeld rows always use BC = 2).
// complex diagonal -(w^2) m (1 - i gamma / Re w) + Sommerfeld at node p, in double
__device__ __forceinline__ void diag_at(const Grid& g, const double* __restrict__ m, const double* __restrict__ gam,
                                        double wre, double wim, int neumann_top, int sommerfeld, double h1, double h2,
                                        double h3, int64_t p, double& dr, double& di) {
  const double mv = m[p], gv = gam[p];
  const double w2r = wre * wre - wim * wim, w2i = 2.0 * wre * wim;
  // -(w^2) * m * (1 - i g / wre)
  const double ar = 1.0, ai = -gv / wre;
  dr = -(w2r * ar - w2i * ai) * mv;
  di = -(w2r * ai + w2i * ar) * mv;
  if (sommerfeld) {
    const int i = (int)(p % g.n1);
    const int64_t q = p / g.n1;
    const int j = (int)(q % g.n2);
    const int k = (int)(q / g.n2);
    double s = 0.0;
    if (i == 0) s += 2.0 / h1;
    if (i == g.n1 - 1) s += 2.0 / h1;
    if (g.dim == 2) {
      if (j == 0 && !neumann_top) s += 2.0 / h2;
      if (j == g.n2 - 1) s += 2.0 / h2;
    } else {
      if (j == 0) s += 2.0 / h2;
      if (j == g.n2 - 1) s += 2.0 / h2;
      if (k == 0 && !neumann_top) s += 2.0 / h3;
      if (k == g.n3 - 1) s += 2.0 / h3;
    }
    di += wre * s * sqrt(mv);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_diag(Grid g, const double* __restrict__ m, const double* __restrict__ gam,
                                              double wre, double wim, int neumann_top, int sommerfeld,
                                              double h1, double h2, double h3, cx<T>* __restrict__ d) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= g.N) return;
  double dr, di;
  diag_at(g, m, gam, wre, wim, neumann_top, sommerfeld, h1, h2, h3, p, dr, di);
  d[p] = mk<T>((T)dr, (T)di);
}

// damped-Jacobi factor relax * (d + Laplacian diagonal)^-1 per node, in double,
// rounded once to T
template <typename T>
__global__ __launch_bounds__(256) void k_jacobi_factor(Grid g, const double* __restrict__ m,
                                                       const double* __restrict__ gam, double wre, double wim,
                                                       int neumann_top, int sommerfeld, double h1, double h2,
                                                       double h3, double relax, cx<T>* __restrict__ f) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= g.N) return;
  double dr, di;
  diag_at(g, m, gam, wre, wim, neumann_top, sommerfeld, h1, h2, h3, p, dr, di);
  const int i = (int)(p % g.n1);
  const int64_t q = p / g.n1;
  const int j = (int)(q % g.n2);
  const int k = (int)(q / g.n2);
  dr += lap_diag1(i, g.n1, g.bc) * g.ih1 + lap_diag1(j, g.n2, g.bc) * g.ih2;
  if (g.dim == 3) dr += lap_diag1(k, g.n3, g.bc) * g.ih3;
  const double s = relax / (dr * dr + di * di);
  f[p] = mk<T>((T)(dr * s), (T)(-di * s));
}

__global__ __launch_bounds__(256) void k_add_const(double* __restrict__ a, double c, int64_t n) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p < n) a[p] += c;
}

// ---- coarsest level: apply of the dense inverse (hh_dense.hip) ----
// x_b = Ainv r_b in complex128 for every right-hand side.  Bound by reading the
// inverse from the Infinity Cache or HBM and r from L2.  A block takes RT rows and DR
// right-hand sides; its 256 threads stride the columns of the row-major inverse
// (coalesced), each keeps RT x DR partial sums, and wave shuffles and one exchange
// through LDS combine them, in the same order of additions for every RT and DR.  The
// four wavefronts split the columns, so a value of r serves RT rows from one load; with a
// row to a wavefront r came from L2 DR times for each value of the inverse (2145 nodes
// x 4 RHS: 22 us for 73 MB, now 15.6).  UN column steps are loaded before the first is used.
// acc + a r in explicit fmas: every tile gives the same bits
__device__ __forceinline__ cx<double> cmac(cx<double> acc, cx<double> a, cx<double> r) {
  return mk<double>(fma(-a.im, r.im, fma(a.re, r.re, acc.re)), fma(a.im, r.re, fma(a.re, r.im, acc.im)));
}

template <int RT, int DR, int UN>
__global__ __launch_bounds__(256) void k_dense_apply(const cx<double>* __restrict__ Arow, int n, int nrhs,
                                                     const cx<double>* __restrict__ r, cx<double>* __restrict__ x,
                                                     const int* __restrict__ skip) {
  constexpr int M = 2 * RT * DR;
  __shared__ double sums[4][M];
  const int lane = threadIdx.x & 63, wid = (int)(threadIdx.x >> 6);
  const int i0 = (int)blockIdx.x * RT;
  const int rhs0 = blockIdx.y * DR;
  const int nr = min(DR, nrhs - rhs0);
  if (skip) {
    int done = 1;
#pragma unroll
    for (int k = 0; k < DR; ++k) done &= skip[rhs0 + min(k, nr - 1)] != 0;
    if (done) return;
  }
  const cx<double>* row[RT];
#pragma unroll
  for (int a = 0; a < RT; ++a) row[a] = Arow + (int64_t)min(i0 + a, n - 1) * n;
  const cx<double>* rc[DR];
#pragma unroll
  for (int k = 0; k < DR; ++k) rc[k] = r + (int64_t)(rhs0 + min(k, nr - 1)) * n;
  cx<double> acc[RT][DR];
#pragma unroll
  for (int a = 0; a < RT; ++a)
#pragma unroll
    for (int k = 0; k < DR; ++k) acc[a][k] = mk<double>(0.0, 0.0);
  for (int j = threadIdx.x; j < n; j += 256 * UN) {
    cx<double> av[UN][RT];
    cx<double> rv[UN][DR];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int ju = min(j + 256 * u, n - 1);  // a column past the last one: its values times 0
#pragma unroll
      for (int a = 0; a < RT; ++a) av[u][a] = row[a][ju];
#pragma unroll
      for (int k = 0; k < DR; ++k) rv[u][k] = rc[k][ju];
    }
#pragma unroll
    for (int u = 0; u < UN; ++u)
#pragma unroll
      for (int k = 0; k < DR; ++k) {
        const cx<double> rk = j + 256 * u < n ? rv[u][k] : mk<double>(0.0, 0.0);
#pragma unroll
        for (int a = 0; a < RT; ++a) acc[a][k] = cmac(acc[a][k], av[u][a], rk);
      }
  }
  double v[M];
#pragma unroll
  for (int a = 0; a < RT; ++a)
#pragma unroll
    for (int k = 0; k < DR; ++k) {
      v[2 * (a * DR + k)] = acc[a][k].re;
      v[2 * (a * DR + k) + 1] = acc[a][k].im;
    }
  WaveSums<M, 32>::run(v, lane, 0, M, [&](int q, double s) { sums[wid][q] = s; });
  __syncthreads();
  const int q = threadIdx.x;
  if (q >= M) return;
  const int a = (q >> 1) / DR, k = (q >> 1) % DR;
  if (i0 + a >= n || k >= nr || (skip && skip[rhs0 + k])) return;
  ((double*)x)[2 * ((int64_t)(rhs0 + k) * n + i0 + a) + (q & 1)] =
      ((sums[0][q] + sums[1][q]) + sums[2][q]) + sums[3][q];
}

// ---- coarsest apply on MFMA (complex64 preconditioner) ----
// The complex product x = A^-1 r is one real GEMM with the real-ified matrix
// A_R (2n x 2n; entry (i, j) of A^-1 becomes [[re, -im], [im, re]] at rows
// 2i, 2i+1 and columns 2j, 2j+1) and r read as a real 2n x nrhs matrix, which
// the interleaved complex64 block already is.  K runs in groups of 16; within
// group g, step u (0..3) of v_mfma_f32_16x16x4_f32 gives lane l the column
// k = 16g + 4(l/16) + u (a permutation of the group, the same for A and r), so
// a lane reads its four A entries as one packed float4 and its four r entries
// as another.  A_R is packed once, in fp32: block (R, g), lane l
// holds row 16R + l % 16, columns 16g + 4(l/16) + 0..3 (zero beyond 2n).
__global__ __launch_bounds__(256) void k_pack_inv_mfma(const cx<double>* __restrict__ Arow, int n, int ng, int nrb,
                                                       float4* __restrict__ P) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (int64_t)nrb * ng * 64) return;
  const int lane = (int)(t & 63);
  const int64_t blk = t >> 6;
  const int g = (int)(blk % ng), R = (int)(blk / ng);
  const int row = R * 16 + (lane & 15), col0 = g * 16 + 4 * (lane >> 4);
  float v[4];
  for (int u = 0; u < 4; ++u) {
    const int col = col0 + u;
    v[u] = 0.f;
    if (row < 2 * n && col < 2 * n) {
      const cx<double> e = Arow[(int64_t)(row >> 1) * n + (col >> 1)];
      const int ra = row & 1, cb = col & 1;
      v[u] = (float)(ra == cb ? e.re : (ra == 0 ? -e.im : e.im));
    }
  }
  P[t] = make_float4(v[0], v[1], v[2], v[3]);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// one block per 16 x 16 tile of the real-ified result (16 real rows, 16 RHS);
// its four wavefronts take every fourth K-group and their partial tiles are
// summed through LDS in a fixed order (deterministic).  Bound by the address unit: a B
// operand is 16 columns apart for 16 lanes, so it is one 16-byte load of four k and not
// two of 8 (561 nodes x 256 RHS 34.8 -> 17.0 us, 2145 x 256 391 -> 195, 97 TFLOP/s, 1183 x
// 32 28.4 -> 20.4 and with two K-groups in flight 13.1; gfx950 takes 16-byte loads at
// 8-byte alignment).
template <int UN>
__global__ __launch_bounds__(256) void k_dense_apply_mfma(const float4* __restrict__ P, int n2, int ng, int nrhs,
                                                          const float* __restrict__ r, float* __restrict__ x,
                                                          const int* __restrict__ skip) {
  __shared__ f32x4 part[3][64];
  const int lane = threadIdx.x & 63, wv = (int)(threadIdx.x >> 6);
  const int R = blockIdx.x, C = blockIdx.y;
  int live = 0;
  for (int q = 0; q < 16; ++q) {
    const int cq = C * 16 + q;
    live |= cq < nrhs && !(skip && skip[cq]);
  }
  if (!live) return;  // whole block: every RHS of the tile is done
  const int col = C * 16 + (lane & 15);
  const bool colok = col < nrhs;
  const int kl = lane >> 4;
  const float4* __restrict__ Pb = P + (int64_t)R * ng * 64 + lane;
  // n2 is even, so every column starts 8-byte aligned
  typedef float f32x4u __attribute__((ext_vector_type(4), aligned(8)));
  const float* __restrict__ rc = r + (int64_t)(colok ? col : 0) * n2;
  f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
  int g = wv;
  if constexpr (UN > 1)  // whole groups, UN of them in flight; then what is left one by one
    for (const int whole = n2 / 16; g + 4 * (UN - 1) < whole; g += 4 * UN) {
      float4 av[UN];
      f32x4u b[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        av[u] = Pb[(int64_t)(g + 4 * u) * 64];
        b[u] = *(const f32x4u*)(rc + (g + 4 * u) * 16 + 4 * kl);
      }
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u].x, b[u].x, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u].y, b[u].y, acc1, 0, 0, 0);
        acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u].z, b[u].z, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u].w, b[u].w, acc1, 0, 0, 0);
      }
    }
  for (; g < ng; g += 4) {
    const float4 av = Pb[(int64_t)g * 64];
    const int k = g * 16 + 4 * kl;
    f32x4u b = {0.f, 0.f, 0.f, 0.f};
    if (colok && k + 4 <= n2) {
      b = *(const f32x4u*)(rc + k);
    } else if (colok && k < n2) {  // the last group of 2n = 2 mod 4
      b.x = rc[k];
      b.y = rc[k + 1];
    }
    acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av.x, b.x, acc0, 0, 0, 0);
    acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(av.y, b.y, acc1, 0, 0, 0);
    acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av.z, b.z, acc0, 0, 0, 0);
    acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(av.w, b.w, acc1, 0, 0, 0);
  }
  const f32x4 acc = acc0 + acc1;
  if (wv > 0) part[wv - 1][lane] = acc;
  __syncthreads();
  if (wv != 0) return;
  const f32x4 sum = ((acc + part[0][lane]) + part[1][lane]) + part[2][lane];
  if (colok && !(skip && skip[col])) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = R * 16 + 4 * kl + i;
      if (row < n2) x[(int64_t)col * n2 + row] = sum[i];
    }
  }
}

// ---------------------------------------------------------------- launchers
void pack_inv_mfma(const cx<double>* Ainv, int64_t n, float* P, hipStream_t s) {
  const int n2 = (int)(2 * n), ng = (n2 + 15) / 16, nrb = (n2 + 15) / 16;
  const int64_t total = (int64_t)nrb * ng * 64;
  hipLaunchKernelGGL(k_pack_inv_mfma, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, Ainv, (int)n, ng, nrb,
                     (float4*)P);
}
int64_t pack_inv_mfma_size(int64_t n) {
  const int64_t b = (2 * n + 15) / 16;
  return b * b * 64 * 4;
}
void launch_dense_apply_mfma(const float* P, int64_t n, int nrhs, const cx<float>* r, cx<float>* x, const int* skip,
                             hipStream_t s) {
  const int n2 = (int)(2 * n), ng = (n2 + 15) / 16, nrb = (n2 + 15) / 16;
  dim3 grid((unsigned)nrb, (unsigned)((nrhs + 15) / 16));
  // two K-groups in flight where the blocks are too few to hide a load's latency (one / two,
  // us: 561 nodes x 48 RHS, 213 blocks 10.4 / 7.0; 1183 x 64, 592 blocks 22.8 / 20.1; 2145 x
  // 48, 807 blocks 46.5 / 46.8; 561 x 256, 1136 blocks 16.4 / 17.5)
  if ((int64_t)grid.x * grid.y < 800)
    hipLaunchKernelGGL(k_dense_apply_mfma<2>, grid, dim3(256), 0, s, (const float4*)P, n2, ng, nrhs, (const float*)r,
                       (float*)x, skip);
  else
    hipLaunchKernelGGL(k_dense_apply_mfma<1>, grid, dim3(256), 0, s, (const float4*)P, n2, ng, nrhs, (const float*)r,
                       (float*)x, skip);
}
// Runs along the slowest axis for `cols` wavefronts per run: enough wavefronts to fill
// 256 CUs, runs of about 16 (of nearly equal length) otherwise.
static inline int pick_rows(int len, int64_t cols) {
  int runs = std::max(1, (len + 8) / 16);
  while (3 * runs <= len && cols * runs < 8192) runs *= 2;
  return (len + runs - 1) / runs;
}

// x blocks up to 16 MB lie in the L2s, where re-reading the neighbours is cheaper than
// the marches' longer start: us a call on an x of its own each time, gathered / marched,
// 129 x 129 x 1 complex128 19.3 / 20.6, 61 x 50 x 33 x 8 complex64 23.4 / 26.3, 1025 x 513
// x 2 complex128 (16 MB) 26.5 / 27.5.  From there on the marches gain: 97 x 97 x 49 x 3
// complex128 (21 MB) 31.6 / 30.8, x 8 complex64 (28 MB) 42.8 / 41.7, 150 x 171 x 101 x 3
// complex128 105 / 88, 1025 x 513 x 64 complex64 171 / 149, 193 x 193 x 97 x 12 complex128
// 510 / 387, x 32 complex64 680 / 535.  RY: complex128 2 / 4 rows 37 / 41 us (101 x 83 x
// 57 x 8), complex64 566 / 528 us (193 x 193 x 97 x 32).
// y goes through the caches.  Stored past them the call is faster only on 96-256 MB of x
// that the last call left in the Infinity Cache (97 x 97 x 49 x 55 complex64 152 -> 117
// us; an x of its own each time 153 / 154), and the kernel that reads y next pays for it
// (call and a product of y, through / past: 513 x 257 x 64 complex64 85 / 103 us, x 32
// complex128 82 / 91, 97 x 97 x 49 x 142 complex64 699 / 743; call and a scaling of y, an x
// of its own each time: from 0.5% faster to 7% slower past them, 2% slower in the mean).
template <typename TI, typename TO, typename TD, int MODE>
void launch_stencil(const Grid& g, int nrhs, const cx<TI>* x, const cx<TO>* b, cx<TO>* y, const cx<TD>* d,
                    const double* m, cx<double> sfac, double wj, const int* skip, hipStream_t s, int rows_override,
                    const cx<TD>* fj) {
  const bool d3 = g.dim == 3;
  const int len = d3 ? g.n3 : g.n2;
  const int64_t xbytes = (int64_t)sizeof(cx<TI>) * g.N * nrhs;
  if (xbytes <= (16 << 20)) {
    const int64_t cols = ((int64_t)g.n1 * (d3 ? g.n2 : 1) + 63) / 64 * nrhs;
    int rows = 16;
    while (rows > 2 && cols * ((len + rows - 1) / rows) < 8192) rows >>= 1;
    if (rows_override > 0) rows = rows_override;
    const int runs = (len + rows - 1) / rows;
    const int64_t items = (int64_t)g.n1 * (d3 ? g.n2 : runs);
    const TileMap tm = make_tile_map((int)((items + 255) / 256), d3 ? runs : 1, nrhs);
    if (d3)
      hipLaunchKernelGGL((k_stencil3d<TI, TO, TD, MODE>), dim3(tm.T), dim3(256), 0, s, g, x, b, y, d, m, sfac,
                         (TD)wj, rows, tm, skip, fj);
    else
      hipLaunchKernelGGL((k_stencil2d<TI, TO, TD, MODE>), dim3(tm.T), dim3(256), 0, s, g, x, b, y, d, m, sfac,
                         (TD)wj, rows, tm, skip, fj);
    return;
  }
  constexpr int RY = sizeof(TI) == 4 ? 4 : 2;
  const int64_t bands = d3 ? (g.n2 + RY - 1) / RY : 1;
  const int rows = rows_override > 0 ? rows_override : pick_rows(len, ((int64_t)g.n1 * bands + 63) / 64 * nrhs);
  const int runs = (len + rows - 1) / rows;
  const int64_t items = (int64_t)g.n1 * (d3 ? bands : runs);
  const TileMap tm = make_tile_map((int)((items + 255) / 256), d3 ? runs : 1, nrhs);
  if (d3)
    hipLaunchKernelGGL((k_march3d<TI, TO, TD, MODE, RY>), dim3(tm.T), dim3(256), 0, s, g, x, b, y, d, m, sfac, (TD)wj,
                       rows, tm, skip, fj);
  else
    hipLaunchKernelGGL((k_march2d<TI, TO, TD, MODE>), dim3(tm.T), dim3(256), 0, s, g, x, b, y, d, m, sfac, (TD)wj,
                       rows, tm, skip, fj);
}

template void launch_stencil<double, double, double, M_APPLY>(const Grid&, int, const cx<double>*,
                                                               const cx<double>*, cx<double>*,
                                                               const cx<double>*, const double*, cx<double>,
                                                               double, const int*, hipStream_t, int,
                                                              const cx<double>*);
template void launch_stencil<double, double, double, M_RESID>(const Grid&, int, const cx<double>*,
                                                               const cx<double>*, cx<double>*,
                                                               const cx<double>*, const double*, cx<double>,
                                                               double, const int*, hipStream_t, int,
                                                              const cx<double>*);
template void launch_stencil<double, double, double, M_JACOBI>(const Grid&, int, const cx<double>*,
                                                                const cx<double>*, cx<double>*,
                                                                const cx<double>*, const double*, cx<double>,
                                                                double, const int*, hipStream_t, int,
                                                              const cx<double>*);
template void launch_stencil<float, float, float, M_APPLY>(const Grid&, int, const cx<float>*, const cx<float>*,
                                                            cx<float>*, const cx<float>*, const double*,
                                                            cx<double>, double, const int*, hipStream_t, int,
                                                              const cx<float>*);
template void launch_stencil<float, float, float, M_RESID>(const Grid&, int, const cx<float>*, const cx<float>*,
                                                            cx<float>*, const cx<float>*, const double*,
                                                            cx<double>, double, const int*, hipStream_t, int,
                                                              const cx<float>*);
template void launch_stencil<float, float, float, M_JACOBI>(const Grid&, int, const cx<float>*, const cx<float>*,
                                                             cx<float>*, const cx<float>*, const double*,
                                                             cx<double>, double, const int*, hipStream_t, int,
                                                              const cx<float>*);
template void launch_stencil<float, double, double, M_APPLY>(const Grid&, int, const cx<float>*,
                                                              const cx<double>*, cx<double>*,
                                                              const cx<double>*, const double*, cx<double>,
                                                              double, const int*, hipStream_t, int,
                                                              const cx<double>*);

template <typename T>
void launch_jacobi0(const Grid& g, int nrhs, const cx<T>* b, cx<T>* x, const cx<T>* f, const int* skip,
                    hipStream_t s) {
  dim3 grid((unsigned)((g.N + 255) / 256), nrhs);
  hipLaunchKernelGGL((k_jacobi0<T>), grid, dim3(256), 0, s, g, b, x, f, skip);
}
template void launch_jacobi0<double>(const Grid&, int, const cx<double>*, cx<double>*, const cx<double>*,
                                     const int*, hipStream_t);
template void launch_jacobi0<float>(const Grid&, int, const cx<float>*, cx<float>*, const cx<float>*, const int*,
                                    hipStream_t);

template <typename T>
void launch_restrict(const Grid& gf, const Grid& gc, int nrhs, const cx<T>* rf, cx<T>* bc, const int* skip,
                     hipStream_t s) {
  if (gf.dim == 3) {
    const int rows = 4;
    const int64_t items = (int64_t)gc.n1 * gc.n2;
    const TileMap tm = make_tile_map((int)((items + 255) / 256), (gc.n3 + rows - 1) / rows, nrhs);
    hipLaunchKernelGGL((k_restrict3<T>), dim3(tm.T), dim3(256), 0, s, gf, gc, rows, tm, rf, bc, skip);
    return;
  }
  dim3 grid((unsigned)((gc.N + 255) / 256), nrhs);
  hipLaunchKernelGGL((k_restrict<T>), grid, dim3(256), 0, s, gf, gc, rf, bc, skip);
}
template void launch_restrict<double>(const Grid&, const Grid&, int, const cx<double>*, cx<double>*, const int*,
                                      hipStream_t);
template void launch_restrict<float>(const Grid&, const Grid&, int, const cx<float>*, cx<float>*, const int*,
                                     hipStream_t);

void launch_restrict_real(const Grid& gf, const Grid& gc, const double* f, double* c, hipStream_t s) {
  hipLaunchKernelGGL(k_restrict_real, dim3((unsigned)((gc.N + 255) / 256)), dim3(256), 0, s, gf, gc, f, c);
}

template <typename T>
void launch_prolong_add(const Grid& gf, const Grid& gc, int nrhs, const cx<T>* xc, cx<T>* xf, const int* skip,
                        hipStream_t s) {
  if (gf.dim == 3) {
    const int rows = 8;  // even: every run starts on a fine plane that coincides with a coarse one
    const int64_t items = (int64_t)gf.n1 * gf.n2;
    const TileMap tm = make_tile_map((int)((items + 255) / 256), (gf.n3 + rows - 1) / rows, nrhs);
    hipLaunchKernelGGL((k_prolong_add3<T>), dim3(tm.T), dim3(256), 0, s, gf, gc, rows, tm, xc, xf, skip);
    return;
  }
  dim3 grid((unsigned)((gf.N + 255) / 256), nrhs);
  hipLaunchKernelGGL((k_prolong_add<T>), grid, dim3(256), 0, s, gf, gc, xc, xf, skip);
}
template void launch_prolong_add<double>(const Grid&, const Grid&, int, const cx<double>*, cx<double>*,
                                         const int*, hipStream_t);
template void launch_prolong_add<float>(const Grid&, const Grid&, int, const cx<float>*, cx<float>*, const int*,
                                        hipStream_t);

template <typename T>
void launch_zero(cx<T>* a, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL((k_zero<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, n);
}
template void launch_zero<double>(cx<double>*, int64_t, hipStream_t);
template void launch_zero<float>(cx<float>*, int64_t, hipStream_t);

template <typename A, typename B>
void launch_cast(const cx<A>* a, cx<B>* b, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL((k_cast<A, B>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, b, n);
}
template void launch_cast<double, float>(const cx<double>*, cx<float>*, int64_t, hipStream_t);
template void launch_cast<float, double>(const cx<float>*, cx<double>*, int64_t, hipStream_t);

template <typename T>
void launch_diag(const Grid& g, const double* m, const double* gam, double wre, double wim, int neumann_top,
                 int sommerfeld, const double h[3], cx<T>* d, hipStream_t s) {
  hipLaunchKernelGGL((k_diag<T>), dim3((unsigned)((g.N + 255) / 256)), dim3(256), 0, s, g, m, gam, wre, wim,
                     neumann_top, sommerfeld, h[0], h[1], h[2], d);
}
template void launch_diag<double>(const Grid&, const double*, const double*, double, double, int, int,
                                  const double*, cx<double>*, hipStream_t);
template void launch_diag<float>(const Grid&, const double*, const double*, double, double, int, int,
                                 const double*, cx<float>*, hipStream_t);

template <typename T>
void launch_jacobi_factor(const Grid& g, const double* m, const double* gam, double wre, double wim, int neumann_top,
                          int sommerfeld, const double* h, double relax, cx<T>* f, hipStream_t s) {
  hipLaunchKernelGGL((k_jacobi_factor<T>), dim3((unsigned)((g.N + 255) / 256)), dim3(256), 0, s, g, m, gam, wre, wim,
                     neumann_top, sommerfeld, h[0], h[1], h[2], relax, f);
}
template void launch_jacobi_factor<double>(const Grid&, const double*, const double*, double, double, int, int,
                                           const double*, double, cx<double>*, hipStream_t);
template void launch_jacobi_factor<float>(const Grid&, const double*, const double*, double, double, int, int,
                                          const double*, double, cx<float>*, hipStream_t);

void launch_add_const(double* a, double c, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_add_const, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, c, n);
}

template <int RT, int DR, int UN>
static void dense_apply_go(const cx<double>* Ainv, int n, int nrhs, const cx<double>* r, cx<double>* x,
                           const int* skip, hipStream_t s) {
  dim3 grid((unsigned)((n + RT - 1) / RT), (unsigned)((nrhs + DR - 1) / DR));
  hipLaunchKernelGGL((k_dense_apply<RT, DR, UN>), grid, dim3(256), 0, s, Ainv, n, nrhs, r, x, skip);
}

// Rows x right-hand sides per block.  Kernel times on MI355X in us, one-row (4 x 4)
// wavefronts of before / now: 561 nodes 1 RHS 3.2 / 3.2, 4 RHS 5.1 / 4.5, 8 RHS 6.6 / 5.4;
// 1183 nodes 1 RHS 5.6 / 4.4, 2 RHS 7.4 / 5.7, 4 RHS 10.0 / 6.7, 8 RHS 13.1 / 9.4;
// 2145 nodes 1 RHS 14.6 / 13.1, 2 RHS 16.2 / 13.9, 4 RHS 21.9 / 15.6, 8 RHS 35.2 / 22.7.
// More rows a block lose the small ones their blocks (561 nodes 4 RHS with 4 rows 5.3).
// An inverse that the L2s hold is cheap to read again, r is not cheaper: tiles of 8 RHS
// win beyond about 1600 nodes (1183 nodes x 8 RHS, 4 / 8 a tile: 9.4 / 11.1 us; 2145: 26.0 /
// 22.7).  Past the Infinity Cache (n > 4096) the inverse comes from HBM, and four rows with
// more columns in flight keep it busiest: 6305 nodes with the call 1 RHS 131 / 120 us,
// 2 RHS 132 / 125, 4 RHS 147 / 140, 8 RHS 269 / 254.
void launch_dense_apply(const cx<double>* Ainv, int64_t n, int nrhs, const cx<double>* r, cx<double>* x,
                        const int* skip, hipStream_t s) {
  if (n > 4096) {
    if (nrhs == 1)
      dense_apply_go<2, 1, 4>(Ainv, (int)n, nrhs, r, x, skip, s);
    else if (nrhs == 2)
      dense_apply_go<4, 2, 4>(Ainv, (int)n, nrhs, r, x, skip, s);
    else
      dense_apply_go<4, 4, 4>(Ainv, (int)n, nrhs, r, x, skip, s);
  } else if (nrhs == 1) {
    dense_apply_go<2, 1, 1>(Ainv, (int)n, nrhs, r, x, skip, s);
  } else if (nrhs == 2) {
    dense_apply_go<2, 2, 2>(Ainv, (int)n, nrhs, r, x, skip, s);
  } else if (nrhs <= 4 || n <= 1600) {
    dense_apply_go<2, 4, 1>(Ainv, (int)n, nrhs, r, x, skip, s);
  } else {
    dense_apply_go<2, 8, 1>(Ainv, (int)n, nrhs, r, x, skip, s);
  }
}

}  // namespace hh
