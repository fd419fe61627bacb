// The spread ("high-order") Helmholtz operator of GetHelmholtzOperatorHO
// (src/GetHelmholtz.jl:54-72, src/PlainNodalLaplacian.jl:54-141), matrix-free:
//
//   H x = Lap x + M (d o x),   d = -w^2 m (1 - i gamma / Re w) + Sommerfeld
//
// 2-D (beta scalar):   Lap = A2 (x) L1 + L2 (x) A1,   M = (avb2 (x) I + I (x) avb1) / 2
// 3-D (b_l, b_m):      Lap = sum over axes q of L_q applied along q to P_q x,
//                      P_q = b_l I + (1 - b_l)/2 (av along the two other axes),
//                      M = (avb1 + avb2 + avb3) / 3 along each axis
//
// with, per axis of n nodes, the tridiagonals (row i, column i + a):
//   L   = ddxCN' ddxCN / h^2-scaled: natural-Neumann second difference
//   av  = av3term(n, 1/2), avb = av3term(n, b_m), A = (1 - b_l) av + b_l I.
// The separable forms follow from G' Gs with G, Gs kron products of ddxCN and
// av3term.
//
// Every one of these tridiagonals is its interior row with the value outside
// the grid replaced by the edge node's own (ghost = self): L's end row is
// f_0 - f_1, av3term's end entry 1/2 + alpha/2 is alpha plus the off-diagonal.  So
// with indices clamped to the grid H has constant coefficients, one per class
// of neighbours (centre, +-e_q, +-e_q +- e_o), and splits into planes: with
//   w_k = c0 x + a1 sx + a2 sy + e12 sxy + bm dx + t (dx's four neighbours)
//   u_k = a3 x + e13 sx + e23 sy + t dx        (sx, sy, sxy: neighbour sums in
// plane k, dx = d x), y_k = w_k + u_{k-1} + u_{k+1}: a march along the last axis
// reads each plane once.  Rows take the place of planes in 2-D.
//
// Lap and M are symmetric (sums of kron products of symmetric tridiagonals), so
// the transpose is H^T x = Lap x + d o (M x): with TR the mass sums take x and
// the diagonal at the row's own node multiplies them.  Adjoint solves use it:
// H^H x = b <=> H^T conj(x) = conj(b).  The arithmetic is float64.
#include <algorithm>

#include "hh_kernels.h"

namespace hh {

namespace {

// coefficients of the neighbour classes (2-D: axis 3 unused, axis 2 the marched one)
struct HoC {
  double c0, a1, a2, a3, e12, e13, e23;  // Laplacian
  double bm, t;                          // mass: centre, neighbour
};

HoC ho_coef(const Grid& g, double bl, double bm) {
  HoC c{};
  const double p0 = bl + 0.5 * (1.0 - bl);  // centre weight of A (2-D) and of P (3-D)
  if (g.dim == 2) {
    const double p1 = 0.25 * (1.0 - bl);
    c.c0 = 2.0 * (g.ih1 + g.ih2) * p0;
    c.a1 = 2.0 * g.ih2 * p1 - g.ih1 * p0;
    c.a2 = 2.0 * g.ih1 * p1 - g.ih2 * p0;
    c.e12 = -(g.ih1 + g.ih2) * p1;
    c.t = 0.25 * (1.0 - bm);
  } else {
    const double p1 = 0.125 * (1.0 - bl);
    c.c0 = 2.0 * (g.ih1 + g.ih2 + g.ih3) * p0;
    c.a1 = 2.0 * (g.ih2 + g.ih3) * p1 - g.ih1 * p0;
    c.a2 = 2.0 * (g.ih1 + g.ih3) * p1 - g.ih2 * p0;
    c.a3 = 2.0 * (g.ih1 + g.ih2) * p1 - g.ih3 * p0;
    c.e12 = -(g.ih1 + g.ih2) * p1;
    c.e13 = -(g.ih1 + g.ih3) * p1;
    c.e23 = -(g.ih2 + g.ih3) * p1;
    c.t = (1.0 - bm) / 6.0;
  }
  c.bm = bm;
  return c;
}

template <typename TI>
__device__ __forceinline__ cx<double> ld(const cx<TI>* __restrict__ x, int64_t p) {
  const cx<TI> v = x[p];
  return mk<double>((double)v.re, (double)v.im);
}
// acc + c v
__device__ __forceinline__ cx<double> axpy(double c, cx<double> v, cx<double> acc) {
  return mk<double>(fma(c, v.re, acc.re), fma(c, v.im, acc.im));
}
__device__ __forceinline__ int clampi(int i, int n) { return i < 0 ? 0 : (i >= n ? n - 1 : i); }

// y = H x (+ sfac m x) or b - H x at one node from lap (the Laplacian's sum,
// with the mass term where !TR), mass (TR: the mass sum), x and d there
template <int MODE, bool TR>
__device__ __forceinline__ cx<double> ho_out(cx<double> lap, cx<double> mass, cx<double> x, cx<double> dv,
                                             const cx<double>* __restrict__ b, const double* __restrict__ m,
                                             cx<double> sfac, int64_t p) {
  cx<double> v = TR ? lap + dv * mass : lap;
  if (m) v = v + (m[p] * sfac) * x;
  return MODE == M_RESID ? b[p] - v : v;
}

// ---- 3-D: a 32 x 16 tile (30 x 14 owned, one position per thread) marched along
// z over a run of planes; x and d x of the current plane in LDS, double buffered,
// one barrier per plane.  The kernel it replaces took one thread per node and
// gathered 19 neighbours and 7 diagonals per axis, with the coefficients formed per
// node: 176 us a call for 101 x 83 x 57 nodes x 8 RHS (complex128) on MI355X, this
// one 56 us; 193 x 193 x 97 x 2 374 / 85 us, 65 x 65 x 33 x 1 22 / 21 us (the call
// itself takes about 10).  Bound by the planes' load latency and barriers: the
// 130 MB of the first case take 28 us at the copy rate.
constexpr int HO_W = 32, HO_R = 16, HO_NT = HO_W * HO_R;

template <typename TI, int MODE, bool TR>
__global__ __launch_bounds__(HO_NT) void k_ho3(TileMap tm, int ytiles, int zrun, Grid g, HoC c,
                                               const cx<TI>* __restrict__ x, const cx<double>* __restrict__ b,
                                               cx<double>* __restrict__ y, const cx<double>* __restrict__ d,
                                               const double* __restrict__ m, cx<double> sfac,
                                               const int* __restrict__ skip) {
  __shared__ cx<double> xs[2][HO_NT], ds[TR ? 1 : 2][TR ? 1 : HO_NT];
  int xt, yz, rhs;
  tile_of(tm, xt, yz, rhs);
  if (skip && skip[rhs]) return;
  const int z0 = (yz / ytiles) * zrun, z1 = min(g.n3, z0 + zrun);
  const int lane = threadIdx.x & (HO_W - 1), row = threadIdx.x / HO_W, q = threadIdx.x;
  const int gx = xt * (HO_W - 2) - 1 + lane, gy = (yz % ytiles) * (HO_R - 2) - 1 + row;
  const bool own = lane >= 1 && lane < HO_W - 1 && row >= 1 && row < HO_R - 1 && gx < g.n1 && gy < g.n2;
  const int64_t plane = (int64_t)g.n1 * g.n2, off = (int64_t)rhs * g.N;
  const int po = clampi(gy, g.n2) * g.n1 + clampi(gx, g.n1);
  const cx<TI>* __restrict__ xr = x + off + po;
  const cx<double>* __restrict__ dp = d + po;
  const cx<double> zero = mk<double>(0.0, 0.0);
  // planes z - 1 and z - 2: w, u, their mass parts (TR), x and d at this node
  cx<double> w1 = zero, u1 = zero, u2 = zero, wm1 = zero, um1 = zero, um2 = zero, x1 = zero, d1 = zero;
  cx<double> xn = ld(xr, (int64_t)clampi(z0 - 1, g.n3) * plane), dn = dp[(int64_t)clampi(z0 - 1, g.n3) * plane];
  for (int z = z0 - 1; z <= z1; ++z) {
    const cx<double> xv = xn, dv = dn;
    const int s = z & 1;
    xs[s][q] = xv;
    const cx<double> mv = TR ? xv : dv * xv;
    if (!TR) ds[s][q] = mv;
    if (z < z1) {
      const int64_t pz = (int64_t)clampi(z + 1, g.n3) * plane;
      xn = ld(xr, pz);
      dn = dp[pz];
    }
    __syncthreads();
    if (own) {
      const cx<double>* xl = xs[s] + q;
      const cx<double>* ml = TR ? xl : ds[TR ? 0 : s] + (TR ? 0 : q);
      const cx<double> sx = xl[-1] + xl[1], sy = xl[-HO_W] + xl[HO_W];
      const cx<double> sxy = (xl[-HO_W - 1] + xl[-HO_W + 1]) + (xl[HO_W - 1] + xl[HO_W + 1]);
      const cx<double> sm = TR ? sx + sy : (ml[-1] + ml[1]) + (ml[-HO_W] + ml[HO_W]);
      cx<double> w = axpy(c.e12, sxy, axpy(c.a2, sy, axpy(c.a1, sx, c.c0 * xv)));
      cx<double> u = axpy(c.e23, sy, axpy(c.e13, sx, c.a3 * xv));
      const cx<double> wm = axpy(c.t, sm, c.bm * mv), um = c.t * mv;
      if (!TR) {
        w = w + wm;
        u = u + um;
      }
      if (z > z0) {
        const int64_t p = (int64_t)(z - 1) * plane + po;
        y[off + p] = ho_out<MODE, TR>(w1 + (u2 + u), TR ? wm1 + (um2 + um) : zero, x1, d1, b ? b + off : nullptr, m,
                                      sfac, p);
      }
      u2 = u1;
      u1 = u;
      w1 = w;
      if (TR) {
        um2 = um1;
        um1 = um;
        wm1 = wm;
        d1 = dv;
      }
      x1 = xv;
    }
  }
}

// ---- 2-D: one thread per column and run of rows, the row's neighbours from
// L1; two rows of partial sums in registers (a call at 1025 x 513 nodes x 32
// RHS: 306 us with the nine-point gather, 160 us; 1039 x 164 x 7: 35, 25 us)
template <typename TI, int MODE, bool TR>
__global__ __launch_bounds__(256) void k_ho2(TileMap tm, int rows, Grid g, HoC c, const cx<TI>* __restrict__ x,
                                             const cx<double>* __restrict__ b, cx<double>* __restrict__ y,
                                             const cx<double>* __restrict__ d, const double* __restrict__ m,
                                             cx<double> sfac, const int* __restrict__ skip) {
  int bx, by, rhs;
  tile_of(tm, bx, by, rhs);
  if (skip && skip[rhs]) return;
  const unsigned item = (unsigned)bx * 256u + threadIdx.x, band = item / (unsigned)g.n1;
  const int i = (int)(item - band * (unsigned)g.n1), j0 = (int)band * rows;
  if (j0 >= g.n2) return;
  const int j1 = min(j0 + rows, g.n2);
  const int il = i > 0 ? i - 1 : 0, ir = i < g.n1 - 1 ? i + 1 : i;
  const int64_t off = (int64_t)rhs * g.N;
  const cx<TI>* __restrict__ xr = x + off;
  const cx<double> zero = mk<double>(0.0, 0.0);
  cx<double> w1 = zero, u1 = zero, u2 = zero, wm1 = zero, um1 = zero, um2 = zero, x1 = zero, d1 = zero;
  for (int j = j0 - 1; j <= j1; ++j) {
    const int64_t r = (int64_t)clampi(j, g.n2) * g.n1;
    const cx<double> xv = ld(xr, r + i), xl = ld(xr, r + il), xq = ld(xr, r + ir), dv = d[r + i];
    const cx<double> sx = xl + xq;
    const cx<double> mv = TR ? xv : dv * xv, sm = TR ? sx : d[r + il] * xl + d[r + ir] * xq;
    cx<double> w = axpy(c.a1, sx, c.c0 * xv), u = axpy(c.e12, sx, c.a2 * xv);
    const cx<double> wm = axpy(c.t, sm, c.bm * mv), um = c.t * mv;
    if (!TR) {
      w = w + wm;
      u = u + um;
    }
    if (j > j0) {
      const int64_t p = (int64_t)(j - 1) * g.n1 + i;
      y[off + p] = ho_out<MODE, TR>(w1 + (u2 + u), TR ? wm1 + (um2 + um) : zero, x1, d1, b ? b + off : nullptr, m,
                                    sfac, p);
    }
    u2 = u1;
    u1 = u;
    w1 = w;
    um2 = um1;
    um1 = um;
    wm1 = wm;
    x1 = xv;
    d1 = dv;
  }
}

template <typename TI, int MODE, bool TR>
void ho_go(const Grid& g, const HoC& c, int nrhs, const cx<TI>* x, const cx<double>* b, cx<double>* y,
           const cx<double>* d, const double* m, cx<double> sfac, const int* skip, hipStream_t s) {
  if (g.dim == 2) {
    // runs of up to 16 rows (two rows are read twice per run) while 8192 wavefronts
    // remain; below 2048 (eight per CU) down to single rows, whose loads need not
    // wait for a march
    const int64_t cols = ((int64_t)g.n1 + 63) / 64 * nrhs;
    auto waves = [&](int r) { return cols * ((g.n2 + r - 1) / r); };
    int rows = 16;
    while (rows > 4 && waves(rows) < 8192) rows >>= 1;
    while (rows > 1 && waves(rows) < 2048) rows >>= 1;
    const int64_t items = (int64_t)g.n1 * ((g.n2 + rows - 1) / rows);
    const TileMap tm = make_tile_map((int)((items + 255) / 256), 1, nrhs);
    hipLaunchKernelGGL((k_ho2<TI, MODE, TR>), dim3(tm.T), dim3(256), 0, s, tm, rows, g, c, x, b, y, d, m, sfac, skip);
    return;
  }
  const int xtiles = (g.n1 + HO_W - 3) / (HO_W - 2), ytiles = (g.n2 + HO_R - 3) / (HO_R - 2);
  // z-runs of up to 48 planes, down to 8 (two planes are formed twice per run) while
  // there are fewer than 1024 blocks (four per CU)
  const int64_t per_run = (int64_t)xtiles * ytiles * nrhs;
  const int want = (int)std::min<int64_t>((1024 + per_run - 1) / per_run, std::max(1, g.n3 / 8));
  const int runs = std::max((g.n3 + 47) / 48, want), zrun = (g.n3 + runs - 1) / runs;
  const TileMap tm = make_tile_map(xtiles, ytiles * ((g.n3 + zrun - 1) / zrun), nrhs);
  hipLaunchKernelGGL((k_ho3<TI, MODE, TR>), dim3(tm.T), dim3(HO_NT), 0, s, tm, ytiles, zrun, g, c, x, b, y, d, m, sfac,
                     skip);
}

}  // namespace

template <typename TI, int MODE>
void launch_ho_stencil(const Grid& g, double bl, double bm, int nrhs, const cx<TI>* x, const cx<double>* b,
                       cx<double>* y, const cx<double>* d, const double* m, cx<double> sfac, const int* skip,
                       hipStream_t s, int tr) {
  const HoC c = ho_coef(g, bl, bm);
  if (tr)
    ho_go<TI, MODE, true>(g, c, nrhs, x, b, y, d, m, sfac, skip, s);
  else
    ho_go<TI, MODE, false>(g, c, nrhs, x, b, y, d, m, sfac, skip, s);
}
template void launch_ho_stencil<double, M_APPLY>(const Grid&, double, double, int, const cx<double>*,
                                                 const cx<double>*, cx<double>*, const cx<double>*, const double*,
                                                 cx<double>, const int*, hipStream_t, int);
template void launch_ho_stencil<float, M_APPLY>(const Grid&, double, double, int, const cx<float>*,
                                                const cx<double>*, cx<double>*, const cx<double>*, const double*,
                                                cx<double>, const int*, hipStream_t, int);
template void launch_ho_stencil<double, M_RESID>(const Grid&, double, double, int, const cx<double>*,
                                                 const cx<double>*, cx<double>*, const cx<double>*, const double*,
                                                 cx<double>, const int*, hipStream_t, int);

}  // namespace hh
