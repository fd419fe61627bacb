// Dense coarsest level: assembly of the shifted operator and its explicit
// complex128 inverse by blocked Gauss-Jordan elimination with partial pivoting.
//
// In-place elimination on the column-major n x n matrix M.  Eliminating a set
// K of columns replaces the matrix by
//   M_KK' = M_KK^-1, M_IK' = -M_IK M_KK^-1, M_KJ' = M_KK^-1 M_KJ,
//   M_IJ' = M_IJ - M_IK M_KK^-1 M_KJ            (I, J outside K, rows pivoted),
// so once the columns K themselves are done ("panel", n x |K|) every other
// column J needs M_J' = (M_J with rows K zeroed) + panel * M_KJ.  Two kernels:
//   k_gj_panel   one workgroup holds all n rows of up to NBI columns in
//                registers and eliminates them one after the other (pivot
//                search over the rows not yet used, two barriers a column);
//   k_gj_update  a block owns whole columns J: it applies the panel's row
//                exchanges to them and adds panel * M_KJ.
// Panels of NBI columns are grouped NB = 32 to a block: inside a block only
// the block's own columns are updated (rank NBI), the rest of the matrix once
// per block (rank 32).  The rank-1 form it replaces (four launches and one
// pass over n x 1.5 n values per column) was bound by launches for n ~ 500 and
// by those passes for n ~ 2000; this one is bound by the panels' serial chain
// (15-16 us per panel of 8, 6 or 4 columns) and, for n > 2000, by the rank-32
// updates as well.  Set-up time of a solver on MI355X (hierarchy included),
// rank-1 form / this one: 561 nodes 7.0 / 2.0 ms, 1183 nodes 23.5 / 7.0 ms,
// 2145 nodes 62 / 17 ms, 8385 nodes 2943 / 371 ms.
//
// The operator is banded in its node order (offsets up to bw = n1, in 3-D n1 n2), and
// rows not yet used keep at most bw columns to their left and 2 bw to their right.  Up to
// bw = 224 the elimination uses that (gj_band): a block's pivots lie in a window of
// 32 + bw rows that one workgroup eliminates at once (k_gj_window: 32 columns in
// 44-58 us instead of eight panels and updates in 160; bound by its barriers and LDS
// reads, 1.4-1.8 us a column), the rows used before take one small product (k_gj_rows),
// and the rank-32 update stops at column ke + 2 bw.  Panel form / this one: 1183 nodes
// (13 x 13 x 7) 6.7 / 4.5 ms, 2145 nodes 16.8 / 8.1 ms, 3201 nodes 32 / 15 ms, 8385
// nodes 371 / 116 ms; 561 nodes 1.9 / 1.8 ms.  The node order is the grid's own, so a 2-D
// grid of n1 > 224 takes the panels although its other axis may be short.
#include <algorithm>

#include "hh_kernels.h"

namespace hh {

namespace {

// entries of a net row exchange: rows pos[e] receive the rows src[e]
constexpr int GJ_NB = 32;            // columns per block
constexpr int GJ_LIST = 2 * GJ_NB;   // rows a block's exchanges can touch
struct GjPerm {
  int cnt;
  int pos[GJ_LIST], src[GJ_LIST];
};

__global__ __launch_bounds__(256) void k_dense_assemble(Grid g, const cx<double>* __restrict__ d,
                                                        cx<double>* __restrict__ M) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t n = g.N;
  if (p >= n) return;
  int i, j, k;
  node_coords(g, p, i, j, k);
  const int64_t P1 = g.n1, P2 = (int64_t)g.n1 * g.n2;
  // row p of A: sum_d ih_d (2 x_p - x_lo - x_hi) + d_p x_p
  const double diag = 2.0 * (g.ih1 + g.ih2 + (g.dim == 3 ? g.ih3 : 0.0));
  M[p + p * n] = mk<double>(diag + d[p].re, d[p].im);
  int64_t nb[6];
  double cf[6];
  int cnt = 0;
  nb[cnt] = (int64_t)k * P2 + j * P1 + lo_nb(i, g.bc); cf[cnt++] = g.ih1;
  nb[cnt] = (int64_t)k * P2 + j * P1 + hi_nb(i, g.n1, g.bc); cf[cnt++] = g.ih1;
  nb[cnt] = (int64_t)k * P2 + lo_nb(j, g.bc) * P1 + i; cf[cnt++] = g.ih2;
  nb[cnt] = (int64_t)k * P2 + hi_nb(j, g.n2, g.bc) * P1 + i; cf[cnt++] = g.ih2;
  if (g.dim == 3) {
    nb[cnt] = (int64_t)lo_nb(k, g.bc) * P2 + j * P1 + i; cf[cnt++] = g.ih3;
    nb[cnt] = (int64_t)hi_nb(k, g.n3, g.bc) * P2 + j * P1 + i; cf[cnt++] = g.ih3;
  }
  for (int c = 0; c < cnt; ++c) M[p + nb[c] * n].re -= cf[c];
}

// net exchange of the swaps (k0 + s, pivot s), s < cnt <= GJ_NB, formed by one
// wavefront: lane s holds pivot s in pv, lane e entry e of the list (lanes
// 0..cnt-1 the rows k0 + e)
__device__ __forceinline__ void gj_net(int k0, int cnt, int pv, GjPerm* out) {
  const int lane = threadIdx.x & 63;
  int pos = lane < cnt ? k0 + lane : -1, src = pos;
  int used = cnt;
  for (int s = 0; s < cnt; ++s) {
    const int b = __builtin_amdgcn_readlane(pv, s);
    const unsigned long long at = __ballot(pos == b);
    int lb;
    if (at) {
      lb = __ffsll((unsigned long long)at) - 1;
    } else {
      lb = used++;
      if (lane == lb) pos = src = b;
    }
    const int sa = __builtin_amdgcn_readlane(src, s), sb = __builtin_amdgcn_readlane(src, lb);
    if (lane == s) src = sb;
    if (lane == lb) src = sa;
  }
  if (lane < used) {
    out->pos[lane] = pos;
    out->src[lane] = src;
  }
  if (lane == 0) out->cnt = used;
}

// maximum of v over the wavefront by DPP moves, valid in lane 63
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long dpp_max(unsigned long long v) {
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)v, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(v >> 32), CTRL, ROWS, 0xf, false);
  const unsigned long long o = ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo;
  return o > v ? o : v;
}
__device__ __forceinline__ unsigned long long wave_max(unsigned long long v) {
  v = dpp_max<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v = dpp_max<0x112, 0xf>(v);
  v = dpp_max<0x114, 0xf>(v);
  v = dpp_max<0x118, 0xf>(v);
  v = dpp_max<0x142, 0xa>(v);  // row_bcast:15 into rows 1, 3
  return dpp_max<0x143, 0xc>(v);  // row_bcast:31 into rows 2, 3
}

// Panel of columns k0 .. k0 + w - 1 (w <= W), all n rows in registers: thread
// t holds rows t, t + T, ..., R of them (T = blockDim.x).  piv[s]: pivot row of
// column kb + s of the block the panel belongs to; pin: the panel's exchange,
// pout (with the block's last panel, else null): the whole block's exchange.
// A pivot is found as the maximum of one 64-bit key per row, |a|^2 with its 14
// lowest bits (up to 3.6e-12 of it, n < 2^14) replaced by the reversed row number: one
// DPP reduction and one LDS atomic per wavefront (a 4-column panel of 2145 rows:
// 20 us with value and row reduced by shuffles, 15 us so).
template <int W, int R>
__global__ __launch_bounds__(1024) void k_gj_panel(cx<double>* __restrict__ M, int n, int k0, int w, int kb,
                                                   int* __restrict__ piv, GjPerm* __restrict__ pin,
                                                   GjPerm* __restrict__ pout) {
  __shared__ unsigned long long key[W];
  __shared__ cx<double> rowp[W], rowk[W];
  __shared__ int pvs[W];
  const int t = threadIdx.x, T = blockDim.x, lane = t & 63;
  if (t < W) key[t] = 0ull;
  // wavefront 0: the block's earlier pivots, lane s that of column kb + s
  const int pv0 = t < k0 - kb ? piv[t] : 0;
  cx<double> a[R][W];
#pragma unroll
  for (int c = 0; c < W; ++c) {
    const cx<double>* __restrict__ col = M + (int64_t)(k0 + min(c, w - 1)) * n;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const unsigned row = (unsigned)(t + r * T);
      a[r][c] = row < (unsigned)n ? col[row] : mk<double>(0.0, 0.0);
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < W; ++c) {
    if (c >= w) break;
    const int k = k0 + c;
    // pivot: largest |a| in rows k .. n-1, the first of equal ones
    unsigned long long best = 0ull;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = t + r * T;
      const unsigned long long v =
          ((unsigned long long)__double_as_longlong(cabs2(a[r][c])) & ~16383ull) | (unsigned)(16383 - row);
      if (row >= k && row < n && v > best) best = v;
    }
    best = wave_max(best);
    if (lane == 63) atomicMax(&key[c], best);
    __syncthreads();
    const int p = 16383 - (int)(key[c] & 16383ull);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = t + r * T;
      if (row == p)
#pragma unroll
        for (int q = 0; q < W; ++q) rowp[q] = a[r][q];
      if (row == k)
#pragma unroll
        for (int q = 0; q < W; ++q) rowk[q] = a[r][q];
    }
    if (t == 0) pvs[c] = p;
    __syncthreads();
    // row k takes the pivot row times 1 / pivot, the row the pivot came from the old row k
    const cx<double> inv = cinv(rowp[c]);
    cx<double> f[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = t + r * T;
      f[r] = row == p ? rowk[c] : a[r][c];
      a[r][c] = row == k ? inv : mk<double>(0.0, 0.0) - f[r] * inv;
    }
#pragma unroll
    for (int q = 0; q < W; ++q) {
      if (q == c) continue;
      const cx<double> pq = rowp[q] * inv, kq = rowk[q];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int row = t + r * T;
        const cx<double> v = row == p ? kq : a[r][q];
        a[r][q] = row == k ? pq : v - f[r] * pq;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < W; ++c) {
    if (c >= w) break;
    cx<double>* __restrict__ col = M + (int64_t)(k0 + c) * n;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const unsigned row = (unsigned)(t + r * T);
      if (row < (unsigned)n) col[row] = a[r][c];
    }
  }
  if (t < 64) {
    const int done = k0 - kb;
    const int pv = lane >= done && lane < done + w ? pvs[lane - done] : pv0;
    if (lane >= done && lane < done + w) piv[lane] = pv;
    gj_net(k0, w, __shfl(pv, min(lane + done, 63), 64), pin);
    if (pout) gj_net(kb, done + w, pv, pout);
  }
}

// Block of columns kb .. kb + w - 1 (w <= 32) of a banded matrix: with node offsets of at
// most bw, the rows not yet used that reach into the block lie in the window kb .. kb +
// wr - 1, wr = 32 + bw at most, so the pivots are found and eliminated there: one
// workgroup, four threads a row with eight columns each in registers.  The window's
// rows get the panel's values, rows kb .. kb + w - 1 among them M_KK^-1; the rows used
// before follow in k_gj_rows, all others are zero.  Same pivots as k_gj_panel's.
__global__ __launch_bounds__(1024) void k_gj_window(cx<double>* __restrict__ M, int n, int kb, int w, int wr,
                                                    GjPerm* __restrict__ pout) {
  __shared__ unsigned long long key[GJ_NB];
  __shared__ cx<double> rowp[GJ_NB], rowk[GJ_NB], pinv;
  __shared__ int pvs[GJ_NB];
  const int t = threadIdx.x, lane = t & 63, row = t >> 2, grp = t & 3;
  const bool in = row < wr;
  if (t < GJ_NB) key[t] = 0ull;
  cx<double> a[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int c = grp * 8 + q;
    a[q] = in && c < w ? M[(int64_t)(kb + c) * n + kb + row] : mk<double>(0.0, 0.0);
  }
  __syncthreads();
  for (int g = 0; g < 4; ++g) {
#pragma unroll
    for (int q0 = 0; q0 < 8; ++q0) {
      const int c = 8 * g + q0;
      if (c >= w) break;
      unsigned long long best = 0ull;
      if (grp == g && row >= c && in)
        best = ((unsigned long long)__double_as_longlong(cabs2(a[q0])) & ~16383ull) | (unsigned)(16383 - (kb + row));
      best = wave_max(best);
      if (lane == 63) atomicMax(&key[c], best);
      // this row's value in column c, held by the group's thread g
      const int from = (lane & ~3) | g;
      const cx<double> own = mk<double>(__shfl(a[q0].re, from, 64), __shfl(a[q0].im, from, 64));
      const cx<double> rec = cinv(a[q0]);  // ready, off the chain, should this be the pivot
      __syncthreads();
      const int p = 16383 - (int)(key[c] & 16383ull) - kb;
      if (row == p)
#pragma unroll
        for (int q = 0; q < 8; ++q) rowp[grp * 8 + q] = a[q];
      if (row == p && grp == g) pinv = rec;
      if (row == c)
#pragma unroll
        for (int q = 0; q < 8; ++q) rowk[grp * 8 + q] = a[q];
      if (t == 0) pvs[c] = kb + p;
      __syncthreads();
      const cx<double> inv = pinv;
      cx<double> f = own;
      if (row == p) {  // (one wavefront's branch: the others leave LDS alone)
        f = rowk[c];
#pragma unroll
        for (int q = 0; q < 8; ++q) a[q] = rowk[grp * 8 + q];
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const cx<double> pq = rowp[grp * 8 + q] * inv;
        a[q] = row == c ? pq : a[q] - f * pq;
      }
      if (grp == g) a[q0] = row == c ? inv : mk<double>(0.0, 0.0) - f * inv;
    }
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int c = grp * 8 + q;
    if (in && c < w) M[(int64_t)(kb + c) * n + kb + row] = a[q];
  }
  if (t < 64) gj_net(kb, w, lane < w ? pvs[lane] : 0, pout);
}

// Rows used before the block: M_IK' = -M_IK M_KK^-1, a block of 256 threads 64 rows,
// eight columns a thread, M_KK^-1 (rows kb .. of the panel) in LDS.
__global__ __launch_bounds__(256) void k_gj_rows(cx<double>* __restrict__ M, int n, int kb, int w) {
  __shared__ cx<double> B[GJ_NB][GJ_NB];
  const int t = threadIdx.x, grp = t >> 6;
  for (int e = t; e < GJ_NB * GJ_NB; e += 256) {
    const int l = e % GJ_NB, c = e / GJ_NB;
    B[l][c] = l < w && c < w ? M[(int64_t)(kb + c) * n + kb + l] : mk<double>(0.0, 0.0);
  }
  const int i = blockIdx.x * 64 + (t & 63), r = min(i, kb - 1);
  __syncthreads();
  cx<double> acc[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) acc[q] = mk<double>(0.0, 0.0);
#pragma unroll 8
  for (int l = 0; l < GJ_NB; ++l) {
    const cx<double> v = M[(int64_t)(kb + min(l, w - 1)) * n + r];  // (past the last: times a zero row)
#pragma unroll
    for (int q = 0; q < 8; ++q) acc[q] = acc[q] - v * B[l][grp * 8 + q];
  }
  __syncthreads();  // every thread of a row has read it
  if (i >= kb) return;
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (grp * 8 + q < w) M[(int64_t)(kb + grp * 8 + q) * n + i] = acc[q];
}

// Columns J of [s0, s1) outside the eliminated columns [k0, k0 + kw), CB whole
// columns per block: the exchange, then M_J = (M_J, rows K zero) + panel M_KJ in the
// first nr rows (the panel is zero below).
template <int KM, int CB, int NT>
__global__ __launch_bounds__(NT) void k_gj_update(cx<double>* __restrict__ M, int n, int nr, int k0, int kw, int s0,
                                                   int s1, const GjPerm* __restrict__ pp) {
  __shared__ cx<double> Rk[KM][CB];
  __shared__ cx<double> V[2 * KM][CB];
  const int t = threadIdx.x;
  const int q0 = s0 + blockIdx.x * CB;  // position among the columns of [s0, s1) without K
  const int cnt = pp->cnt, total = s1 - kw;
  for (int e = t; e < cnt * CB; e += NT) {
    const int c = e % CB, l = e / CB, q = q0 + c;
    if (q < total) V[l][c] = M[pp->src[l] + (int64_t)(q < k0 ? q : q + kw) * n];
  }
  __syncthreads();
  for (int e = t; e < cnt * CB; e += NT) {
    const int c = e % CB, l = e / CB, q = q0 + c;
    if (q >= total) continue;
    const int pos = pp->pos[l];
    if (pos >= k0 && pos < k0 + kw)
      Rk[pos - k0][c] = V[l][c];
    else
      M[pos + (int64_t)(q < k0 ? q : q + kw) * n] = V[l][c];
  }
  if (kw < KM)
    for (int e = t; e < (KM - kw) * CB; e += NT) Rk[kw + e / CB][e % CB] = mk<double>(0.0, 0.0);
  __syncthreads();
  cx<double>* col[CB];
#pragma unroll
  for (int c = 0; c < CB; ++c) {
    const int q = min(q0 + c, total - 1);
    col[c] = M + (int64_t)(q < k0 ? q : q + kw) * n;
  }
  const cx<double>* __restrict__ P = M + (int64_t)k0 * n;
  // two rows at a time: an M_KJ value read from LDS serves both
  for (int r0 = t; r0 < nr; r0 += 2 * NT) {
    const int r[2] = {r0, min(r0 + NT, nr - 1)};
    cx<double> acc[2][CB];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < CB; ++c)
        acc[h][c] = r[h] >= k0 && r[h] < k0 + kw ? mk<double>(0.0, 0.0) : col[c][r[h]];
#pragma unroll 4
    for (int j = 0; j < KM; ++j) {
      // (past the last column: a zero row of M_KJ, the panel read again at its last column)
      const cx<double>* __restrict__ pc = P + (int64_t)min(j, kw - 1) * n;
      const cx<double> p0 = pc[r[0]], p1 = pc[r[1]];
#pragma unroll
      for (int c = 0; c < CB; ++c) {
        const cx<double> q = Rk[j][c];
        acc[0][c] = acc[0][c] + p0 * q;
        acc[1][c] = acc[1][c] + p1 * q;
      }
    }
#pragma unroll
    for (int c = 0; c < CB; ++c)
      if (q0 + c < total) {
        col[c][r[0]] = acc[0][c];
        if (r0 + NT < nr) col[c][r[1]] = acc[1][c];
      }
  }
}

// Row order after all exchanges, one wavefront: pi[j] = row of A at row j of
// P A, the blocks' exchange lists applied in turn to an array in LDS
__global__ __launch_bounds__(64) void k_gj_order(int n, int nlist, const GjPerm* __restrict__ lists,
                                                 int* __restrict__ pi) {
  extern __shared__ int ord[];
  const int lane = threadIdx.x;
  for (int q = lane; q < n; q += 64) ord[q] = q;
  int cnt = lists[0].cnt, pos = lists[0].pos[lane], src = lists[0].src[lane];
  __syncthreads();
  for (int l = 0; l < nlist; ++l) {
    const GjPerm* nx = lists + min(l + 1, nlist - 1);
    const int ncnt = nx->cnt, npos = nx->pos[lane], nsrc = nx->src[lane];
    const int v = lane < cnt ? ord[src] : 0;
    __syncthreads();
    if (lane < cnt) ord[pos] = v;
    __syncthreads();
    cnt = ncnt, pos = npos, src = nsrc;
  }
  for (int q = lane; q < n; q += 64) pi[q] = ord[q];
}

// M holds (P A)^-1 column-major with row j of P A the row pi[j] of A:
// A^-1 row-major, out[i n + pi[j]] = M[i + j n], through 32 x 32 LDS tiles
__global__ __launch_bounds__(256) void k_inv_rows(const cx<double>* __restrict__ M, int n, const int* __restrict__ pi,
                                                  cx<double>* __restrict__ out) {
  __shared__ cx<double> tile[32][33];
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
  const int i0 = blockIdx.x * 32, j0 = blockIdx.y * 32;
  for (int q = y; q < 32; q += 8)
    if (i0 + x < n && j0 + q < n) tile[q][x] = M[(i0 + x) + (int64_t)(j0 + q) * n];
  __syncthreads();
  for (int q = y; q < 32; q += 8)
    if (i0 + q < n && j0 + x < n) out[(int64_t)(i0 + q) * n + pi[j0 + x]] = tile[x][q];
}

// work space of one inversion (device): row order, pivots of a block, the
// current panel's exchange, the exchanges of every block
struct GjWork {
  int* pi;
  int* piv;
  GjPerm* inner;
  GjPerm* blocks;
};

// up to 768 nodes the whole matrix is 9 MB: rank-W updates of all of it cost
// less than the extra launches of the blocked form
bool gj_blocked(int n) { return n > 768; }

template <int W, int R>
void gj_run(cx<double>* M, int n, const GjWork& wk, hipStream_t s) {
  const int T = std::min(1024, (n + 63) / 64 * 64);
  const bool blocked = gj_blocked(n);
  const int NB = blocked ? GJ_NB : W;
  int nlist = 0;
  for (int kb = 0; kb < n; kb += NB, ++nlist) {
    const int ke = std::min(n, kb + NB);
    GjPerm* blk = wk.blocks + nlist;
    for (int k0 = kb; k0 < ke; k0 += W) {
      const int w = std::min(W, ke - k0);
      hipLaunchKernelGGL((k_gj_panel<W, R>), dim3(1), dim3(T), 0, s, M, n, k0, w, kb, wk.piv,
                         blocked ? wk.inner : blk, blocked && k0 + w == ke ? blk : nullptr);
      if (!blocked) {
        if (n > w)
          hipLaunchKernelGGL((k_gj_update<W, 2, 256>), dim3((n - w + 1) / 2), dim3(256), 0, s, M, n, n, k0, w, 0, n, blk);
      } else if (ke - kb > w) {  // the block's other columns
        hipLaunchKernelGGL((k_gj_update<W, 1, 1024>), dim3(ke - kb - w), dim3(1024), 0, s, M, n, n, k0, w, kb, ke,
                           wk.inner);
      }
    }
    if (blocked && n > ke - kb)
      hipLaunchKernelGGL((k_gj_update<GJ_NB, 4, 256>), dim3((n - (ke - kb) + 3) / 4), dim3(256), 0, s, M, n, n, kb,
                         ke - kb, 0, n, blk);
  }
  hipLaunchKernelGGL(k_gj_order, dim3(1), dim3(64), sizeof(int) * n, s, n, nlist, wk.blocks, wk.pi);
}

// The banded elimination: per 32 columns one window, the rows used before and a rank-32
// update of the columns that the rows in use reach (ke + 2 bw).
constexpr int GJ_WINDOW = 256;  // rows of a window: 1024 threads
void gj_band(cx<double>* M, int n, int bw, const GjWork& wk, hipStream_t s) {
  int nlist = 0;
  for (int kb = 0; kb < n; kb += GJ_NB, ++nlist) {
    const int w = std::min(GJ_NB, n - kb), wr = std::min(n - kb, GJ_NB + bw);
    const int nr = kb + wr, s1 = std::min(n, kb + w + 2 * bw);
    hipLaunchKernelGGL(k_gj_window, dim3(1), dim3((4 * wr + 63) / 64 * 64), 0, s, M, n, kb, w, wr, wk.blocks + nlist);
    if (kb > 0) hipLaunchKernelGGL(k_gj_rows, dim3((kb + 63) / 64), dim3(256), 0, s, M, n, kb, w);
    if (s1 > w)
      hipLaunchKernelGGL((k_gj_update<GJ_NB, 4, 256>), dim3((s1 - w + 3) / 4), dim3(256), 0, s, M, n, nr, kb, w, 0, s1,
                         wk.blocks + nlist);
  }
  hipLaunchKernelGGL(k_gj_order, dim3(1), dim3(64), sizeof(int) * n, s, n, nlist, wk.blocks, wk.pi);
}

constexpr size_t gj_ints(int64_t n) { return ((size_t)(n + GJ_NB) + 3) / 4 * 4; }

}  // namespace

// bytes of the work space launch_dense_inverse takes (one exchange list per two columns at most)
size_t dense_inverse_work_bytes(int64_t n) {
  return sizeof(int) * gj_ints(n) + sizeof(GjPerm) * (1 + (size_t)(n + 1) / 2);
}

void launch_dense_inverse(const Grid& g, const cx<double>* d, cx<double>* M2, void* work, hipStream_t s) {
  const int n = (int)g.N;
  cx<double>* M = M2 + (int64_t)n * n;
  GjWork wk;
  wk.pi = (int*)work;
  wk.piv = wk.pi + n;
  wk.inner = (GjPerm*)(wk.pi + gj_ints(n));
  wk.blocks = wk.inner + 1;
  launch_zero<double>(M, (int64_t)n * n, s);
  hipLaunchKernelGGL(k_dense_assemble, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g, d, M);
  const int64_t bw = (int64_t)g.n1 * (g.dim == 3 ? g.n2 : 1);  // largest node offset of a row
  // columns per panel so that a thread's rows fit its 128 registers
  if (bw + GJ_NB <= GJ_WINDOW)
    gj_band(M, n, (int)bw, wk, s);
  else if (n <= 1024)
    gj_run<8, 1>(M, n, wk, s);
  else if (n <= 2048)
    gj_run<6, 2>(M, n, wk, s);
  else if (n <= 4096)
    gj_run<4, 4>(M, n, wk, s);
  else if (n <= 8192)
    gj_run<2, 8>(M, n, wk, s);
  else
    gj_run<1, 10>(M, n, wk, s);
  hipLaunchKernelGGL(k_inv_rows, dim3((n + 31) / 32, (n + 31) / 32), dim3(256), 0, s, M, n, wk.pi, M2);
}

}  // namespace hh
