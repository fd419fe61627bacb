// GMRES-accelerated damped-Jacobi smoothing ("Jac-GMRES", a relaxType of
// Multigrid.jl that test/ShiftedLaplacianTest.jl:137-142 runs with the
// K-cycle), batched over right-hand sides: s steps of GMRES on A x = b from
// the current x, right-preconditioned by the level's damped-Jacobi factor F:
//
//   r0 = b - A x, beta = ||r0||, v0 = r0 / beta
//   step i:  w = A (F v_i);  classical Gram-Schmidt twice against v_0..v_i
//            (h = V^H w, w -= V h, twice), h_{i+1,i} = ||w||, v_{i+1} = w / ||w||
//   y = argmin || beta e1 - Hbar y ||  (Givens QR per RHS)
//   x <- x + F (V y)
//
// so x minimises ||b - A x|| over x0 + F K_s(A F, r0).  The stored vectors are
// unnormalised: u_0 = r0, u_{i+1} = the orthogonalised A F u_i, v_i = s_i u_i with
// s_i = 1 / ||u_i||; the scales enter the coefficients only.  Vectors stay in the
// level's precision; inner products, the Hessenberg matrix and y are
// complex128, and every reduction runs in a fixed order.
//
// A step is three launches: the product with the partial sums of u_k^H w, the
// first projection with those of the second, the second with those of ||w||^2;
// each block reduces the previous launch's partial sums itself (at most 256 per
// sum).  The levels this runs on are small, so a smoothing costs its launches:
// one kernel per operation (F v, A u, dots, reduction, update, scaling) took 27 for
// two steps, with the dots on one block per 4096 nodes (8.9 us each); now eight.
// K-cycle solve of 257 x 129 x 4 RHS in complex128 (3 levels; 89 to 95 iterations by
// the medium) on MI355X: 83 ms with the separate kernels, 41 ms.
#include "hh_kernels.h"

#include <algorithm>

namespace hh {

namespace {

constexpr int GM_NB = GM_MAX_STEPS + 1;  // basis vectors
constexpr int GM_PK = GM_NB + 1;         // partial-sum slots per chunk: dots, then ||w||^2
constexpr int GM_CH = 256;               // chunks at most

// node chunks per RHS: one node per thread up to 65536 nodes (by the grid alone,
// so a block of RHS gives the bits of single ones)
int gm_chunks(int64_t N) { return (int)std::max<int64_t>(1, std::min<int64_t>(GM_CH, (N + 255) / 256)); }

template <typename T>
__device__ __forceinline__ cx<double> up(cx<T> v) {
  return mk<double>((double)v.re, (double)v.im);
}

__device__ __forceinline__ double gsum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

// The operands of one smoothing call as its kernels see them.  Partial sums of
// launch n are written to half n & 1 of part while the other half is read:
// part[((half * GM_CH + c) * GM_PK + k) * nrhs + b], slot GM_NB the squared norm.
template <typename T>
struct GmK {
  Grid g;
  int nrhs, nch;
  const cx<T>* u0;   // u_0 (b itself when the call starts from x = 0)
  cx<T>* V;          // u_k = V + k stride, k >= 1
  const cx<T>* d;
  const cx<T>* f;
  cx<double>* part;
  cx<double>* H;     // [b][GM_NB][GM_MAX_STEPS]
  double* sc;        // [k][b] 1 / ||u_k||
  double* beta;
  const int* skip;
  __device__ __forceinline__ const cx<T>* u(int k) const { return k == 0 ? u0 : V + (int64_t)k * g.N * nrhs; }
  __device__ __forceinline__ cx<double>* slot(int half, int c, int k, int b) const {
    return part + ((int64_t)(half * GM_CH + c) * GM_PK + k) * nrhs + b;
  }
};

__device__ __forceinline__ void chunk(int64_t N, int nch, int c, int64_t* p0, int64_t* p1) {
  const int64_t L = (N + nch - 1) / nch;
  *p0 = (int64_t)c * L;
  *p1 = min(N, *p0 + L);
}

// block sums of acc[0..nv) and nn into this chunk's slots
template <typename T>
__device__ __forceinline__ void gm_store(const GmK<T>& k, int half, int c, int b, int nv, const cx<double> (&acc)[GM_NB],
                                         double nn) {
  constexpr int M = 2 * GM_NB + 1;
  __shared__ double sums[4][M];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, q = threadIdx.x;
  double v[M];
#pragma unroll
  for (int i = 0; i < GM_NB; ++i) v[2 * i] = acc[i].re, v[2 * i + 1] = acc[i].im;
  v[M - 1] = nn;
  WaveSums<M, 32>::run(v, lane, 0, M, [&](int j, double s) { sums[wid][j] = s; });
  __syncthreads();
  if (q >= M) return;
  const double s = ((sums[0][q] + sums[1][q]) + sums[2][q]) + sums[3][q];
  if (q == M - 1)
    *k.slot(half, c, GM_NB, b) = mk<double>(s, 0.0);
  else if (q < 2 * nv)
    ((double*)k.slot(half, c, q >> 1, b))[q & 1] = s;
}

// A z at node p (5/7-point operator, the ghosts' values by index), z given by
// its node values; apply5/apply7 fix the order of operations
template <typename T, int DIM, typename F>
__device__ __forceinline__ cx<T> gm_stencil(const Grid& g, int64_t p, cx<T> dv, F&& z) {
  int i, j, kz;
  node_coords(g, p, i, j, kz);
  const int64_t n1 = g.n1, plane = n1 * g.n2, pl = DIM == 3 ? (int64_t)kz * plane : 0, row = pl + (int64_t)j * n1;
  const cx<T> c = z(p), l1 = z(row + lo_nb(i, g.bc)), r1 = z(row + hi_nb(i, g.n1, g.bc));
  const cx<T> l2 = z(pl + (int64_t)lo_nb(j, g.bc) * n1 + i), r2 = z(pl + (int64_t)hi_nb(j, g.n2, g.bc) * n1 + i);
  if (DIM == 2) return apply5(c, l1, r1, l2, r2, (T)g.ih1, (T)g.ih2, dv);
  const int64_t col = (int64_t)j * n1 + i;
  return apply7(c, l1, r1, l2, r2, z((int64_t)lo_nb(kz, g.bc) * plane + col), z((int64_t)hi_nb(kz, g.n3, g.bc) * plane + col),
                (T)g.ih1, (T)g.ih2, (T)g.ih3, dv);
}

// sum over chunks of slot i (one wavefront; every lane gets it)
template <typename T>
__device__ __forceinline__ cx<double> gm_total(const GmK<T>& k, int half, int i, int b) {
  const int lane = threadIdx.x & 63;
  cx<double> v[GM_CH / 64];
#pragma unroll
  for (int q = 0; q < GM_CH / 64; ++q) v[q] = lane + 64 * q < k.nch ? *k.slot(half, lane + 64 * q, i, b) : mk<double>(0.0, 0.0);
  double re = 0.0, im = 0.0;
#pragma unroll
  for (int q = 0; q < GM_CH / 64; ++q) re += v[q].re, im += v[q].im;
  return mk<double>(__shfl(gsum(re), 0, 64), __shfl(gsum(im), 0, 64));
}

// wavefront 0 of chunk 0: the norm of u_i from half's squared norm; s_i, and beta
// (i = 0) or H[i][i - 1] = s_{i-1} ||u_i||
template <typename T>
__device__ __forceinline__ void gm_norm(const GmK<T>& k, int half, int i, int b) {
  const double nn = gm_total(k, half, GM_NB, b).re;
  if (threadIdx.x != 0) return;
  const double nr = nn > 0.0 ? sqrt(nn) : 0.0;
  k.sc[i * k.nrhs + b] = nr > 0.0 ? 1.0 / nr : 0.0;
  if (i == 0)
    k.beta[b] = nr;
  else
    k.H[((int64_t)b * GM_NB + i) * GM_MAX_STEPS + i - 1] = mk<double>(k.sc[(i - 1) * k.nrhs + b] * nr, 0.0);
}

}  // namespace

// r0 = b - A x into u_0 (WRITE; otherwise u_0 is b and only its norm is formed)
template <typename T, bool WRITE, int DIM>
__global__ __launch_bounds__(256) void k_gm_start(GmK<T> k, const cx<T>* __restrict__ x, const cx<T>* __restrict__ b0,
                                                  cx<T>* __restrict__ r0, int half) {
  const int c = blockIdx.x, b = blockIdx.y;
  if (k.skip && k.skip[b]) return;
  const Grid& g = k.g;
  int64_t p0, p1;
  chunk(g.N, k.nch, c, &p0, &p1);
  const int64_t base = (int64_t)b * g.N;
  cx<double> acc[GM_NB];
#pragma unroll
  for (int q = 0; q < GM_NB; ++q) acc[q] = mk<double>(0.0, 0.0);
  double nn = 0.0;
  for (int64_t p = p0 + threadIdx.x; p < p1; p += 256) {
    cx<T> r = b0[base + p];
    if (WRITE) {
      const cx<T>* __restrict__ xb = x + base;
      r = r - gm_stencil<T, DIM>(g, p, k.d[p], [&](int64_t q) { return xb[q]; });
      r0[base + p] = r;
    }
    nn += cabs2(up(r));
  }
  gm_store(k, half, c, b, 0, acc, nn);
}

// w = A (F u_i) into u_{i+1}, partial sums of u_q^H w (q <= i); chunk 0 also closes
// the norm of u_i (half ^ 1)
template <typename T, int DIM>
__global__ __launch_bounds__(256) void k_gm_product(GmK<T> k, int i, int half) {
  const int c = blockIdx.x, b = blockIdx.y;
  if (k.skip && k.skip[b]) return;
  if (c == 0 && threadIdx.x < 64) gm_norm(k, half ^ 1, i, b);
  const Grid& g = k.g;
  int64_t p0, p1;
  chunk(g.N, k.nch, c, &p0, &p1);
  const int64_t base = (int64_t)b * g.N;
  const cx<T>* __restrict__ ui = k.u(i) + base;
  const cx<T>* __restrict__ f = k.f;
  cx<T>* __restrict__ w = k.V + (int64_t)(i + 1) * g.N * k.nrhs + base;
  cx<double> acc[GM_NB];
#pragma unroll
  for (int q = 0; q < GM_NB; ++q) acc[q] = mk<double>(0.0, 0.0);
  for (int64_t p = p0 + threadIdx.x; p < p1; p += 256) {
    const cx<T> v = gm_stencil<T, DIM>(g, p, k.d[p], [&](int64_t q) { return f[q] * ui[q]; });
    w[p] = v;
#pragma unroll
    for (int q = 0; q < GM_NB; ++q)
      if (q <= i) acc[q] = acc[q] + cmulc(up(k.u(q)[base + p]), up(v));
  }
  gm_store(k, half, c, b, i + 1, acc, 0.0);
}

// w -= sum_q c_q u_q with c_q = s_q^2 u_q^H w (q <= i) from half ^ 1; pass 1 leaves the
// partial sums of the second projection, pass 2 those of ||w||^2.  Chunk 0 adds
// s_q s_i u_q^H w to H[q][i].
template <typename T>
__global__ __launch_bounds__(256) void k_gm_project(GmK<T> k, int i, int pass, int half) {
  const int c = blockIdx.x, b = blockIdx.y;
  if (k.skip && k.skip[b]) return;
  __shared__ cx<double> cf[GM_NB];
  const int wid = threadIdx.x >> 6;
  for (int q = wid; q <= i; q += 4) {
    const cx<double> t = gm_total(k, half ^ 1, q, b);
    if ((threadIdx.x & 63) == 0) {
      const double sq = k.sc[q * k.nrhs + b];
      cf[q] = (sq * sq) * t;
      if (c == 0) {
        const cx<double> h = (sq * k.sc[i * k.nrhs + b]) * t;
        cx<double>& e = k.H[((int64_t)b * GM_NB + q) * GM_MAX_STEPS + i];
        e = pass == 1 ? h : e + h;
      }
    }
  }
  __syncthreads();
  const int64_t N = k.g.N, base = (int64_t)b * N;
  int64_t p0, p1;
  chunk(N, k.nch, c, &p0, &p1);
  cx<T>* __restrict__ w = k.V + (int64_t)(i + 1) * N * k.nrhs + base;
  cx<double> acc[GM_NB];
#pragma unroll
  for (int q = 0; q < GM_NB; ++q) acc[q] = mk<double>(0.0, 0.0);
  double nn = 0.0;
  for (int64_t p = p0 + threadIdx.x; p < p1; p += 256) {
    cx<double> v = up(w[p]);
    cx<T> uq[GM_NB];
#pragma unroll
    for (int q = 0; q < GM_NB; ++q)
      if (q <= i) uq[q] = k.u(q)[base + p];
#pragma unroll
    for (int q = 0; q < GM_NB; ++q)
      if (q <= i) v = v - cf[q] * up(uq[q]);
    const cx<T> o = mk<T>((T)v.re, (T)v.im);
    w[p] = o;
    if (pass == 1) {
#pragma unroll
      for (int q = 0; q < GM_NB; ++q)
        if (q <= i) acc[q] = acc[q] + cmulc(up(uq[q]), up(o));
    } else {
      nn += cabs2(up(o));
    }
  }
  gm_store(k, half, c, b, pass == 1 ? i + 1 : 0, acc, nn);
}

// y = argmin || beta e1 - Hbar y || over the leading columns whose
// subdiagonal stays nonzero (an exact Krylov direction ends the space), by
// Givens rotations; every block solves it again, one thread on LDS (R: Hbar,
// g: scratch), the last norm from half ^ 1.  Then x (+)= F o (sum_i y_i s_i u_i)
// over the first s basis vectors; assign = 1 writes instead of adding
// (smoothing from x = 0).
template <typename T>
__global__ __launch_bounds__(256) void k_gm_finish(GmK<T> k, int s, cx<T>* __restrict__ x, int assign, int half) {
  const int c = blockIdx.x, b = blockIdx.y;
  if (k.skip && k.skip[b]) return;
  __shared__ cx<double> R[GM_NB][GM_MAX_STEPS], g[GM_NB], y[GM_MAX_STEPS];
  __shared__ double sc[GM_NB];
  const int t = threadIdx.x;
  if (t >= 64) {  // (wavefront 0 forms the last row's entry)
    for (int e = t - 64; e < s * s; e += 192) R[e / s][e % s] = k.H[((int64_t)b * GM_NB + e / s) * GM_MAX_STEPS + e % s];
    if (t - 64 < s) {
      sc[t - 64] = k.sc[(t - 64) * k.nrhs + b];
      R[s][t - 64] = mk<double>(0.0, 0.0);
      g[t - 64 + 1] = mk<double>(0.0, 0.0);
      y[t - 64] = mk<double>(0.0, 0.0);
    }
  }
  double last = 0.0;
  if (t < 64) {
    const double nn = gm_total(k, half ^ 1, GM_NB, b).re;
    last = nn > 0.0 ? sqrt(nn) : 0.0;
  }
  __syncthreads();
  if (t == 0) {
    const double be = k.beta[b];
    R[s][s - 1] = mk<double>(sc[s - 1] * last, 0.0);
    // entries below the subdiagonal hold no Hessenberg values
    for (int i = 0; i < s; ++i)
      for (int q = i + 2; q <= s; ++q) R[q][i] = mk<double>(0.0, 0.0);
    g[0] = mk<double>(be, 0.0);
    int kk = s;  // columns in use
    for (int i = 0; i < s; ++i)
      if (!(cabs2(R[i + 1][i]) > 0.0)) {
        kk = i + 1;
        break;
      }
    if (be > 0.0) {
      for (int i = 0; i < kk; ++i) {
        // rotation zeroing R[i+1][i] against R[i][i]
        const cx<double> a = R[i][i], cc = R[i + 1][i];
        const double na = sqrt(cabs2(a)), nc = sqrt(cabs2(cc));
        if (!(nc > 0.0)) continue;
        const double r = sqrt(na * na + nc * nc);
        // [cs  sn; -conj(sn) cs] with cs real: cs = |a| / r, sn = (a / |a|) conj(c) / r
        const double cs = na / r;
        const cx<double> ph = na > 0.0 ? mk<double>(a.re / na, a.im / na) : mk<double>(1.0, 0.0);
        const cx<double> sn = ph * mk<double>(cc.re / r, -cc.im / r);
        for (int j = i; j < kk; ++j) {
          const cx<double> t0 = R[i][j], t1 = R[i + 1][j];
          R[i][j] = cs * t0 + sn * t1;
          R[i + 1][j] = cs * t1 - mk<double>(sn.re, -sn.im) * t0;
        }
        const cx<double> g0 = g[i], g1 = g[i + 1];
        g[i] = cs * g0 + sn * g1;
        g[i + 1] = cs * g1 - mk<double>(sn.re, -sn.im) * g0;
      }
      for (int i = kk - 1; i >= 0; --i) {
        cx<double> v = g[i];
        for (int j = i + 1; j < kk; ++j) v = v - R[i][j] * y[j];
        y[i] = cabs2(R[i][i]) > 0.0 ? v * cinv(R[i][i]) : mk<double>(0.0, 0.0);
      }
    }
    for (int i = 0; i < s; ++i) y[i] = sc[i] * y[i];
  }
  __syncthreads();
  const int64_t N = k.g.N, base = (int64_t)b * N;
  int64_t p0, p1;
  chunk(N, k.nch, c, &p0, &p1);
  for (int64_t p = p0 + t; p < p1; p += 256) {
    cx<double> acc = mk<double>(0.0, 0.0);
    for (int i = 0; i < s; ++i) acc = acc + y[i] * up(k.u(i)[base + p]);
    const cx<double> e = up(k.f[p]) * acc;
    const cx<double> xn = assign ? e : up(x[base + p]) + e;
    x[base + p] = mk<T>((T)xn.re, (T)xn.im);
  }
}

size_t gm_part_elems(int nrhs) { return (size_t)2 * GM_CH * GM_PK * nrhs; }

template <typename T>
void gm_smooth(const GmArgs<T>& a, int steps, hipStream_t st) {
  if (steps <= 0) return;
  GmK<T> k;
  k.g = a.g;
  k.nrhs = a.nrhs;
  k.nch = gm_chunks(a.g.N);
  k.u0 = a.zero_x ? a.b : a.V;
  k.V = a.V;
  k.d = a.d;
  k.f = a.f;
  k.part = a.part;
  k.H = a.H;
  k.sc = a.sc;
  k.beta = a.beta;
  k.skip = a.skip;
  const dim3 cg(k.nch, a.nrhs), tb(256);
  const bool d3 = a.g.dim == 3;
  int half = 0;
  if (a.zero_x)
    hipLaunchKernelGGL((k_gm_start<T, false, 2>), cg, tb, 0, st, k, a.x, a.b, a.V, half);
  else if (d3)
    hipLaunchKernelGGL((k_gm_start<T, true, 3>), cg, tb, 0, st, k, a.x, a.b, a.V, half);
  else
    hipLaunchKernelGGL((k_gm_start<T, true, 2>), cg, tb, 0, st, k, a.x, a.b, a.V, half);
  for (int i = 0; i < steps; ++i) {
    half ^= 1;
    if (d3)
      hipLaunchKernelGGL((k_gm_product<T, 3>), cg, tb, 0, st, k, i, half);
    else
      hipLaunchKernelGGL((k_gm_product<T, 2>), cg, tb, 0, st, k, i, half);
    for (int pass = 1; pass <= 2; ++pass) {
      half ^= 1;
      hipLaunchKernelGGL((k_gm_project<T>), cg, tb, 0, st, k, i, pass, half);
    }
  }
  half ^= 1;
  hipLaunchKernelGGL((k_gm_finish<T>), cg, tb, 0, st, k, steps, a.x, a.zero_x ? 1 : 0, half);
}

template void gm_smooth<float>(const GmArgs<float>&, int, hipStream_t);
template void gm_smooth<double>(const GmArgs<double>&, int, hipStream_t);

}  // namespace hh
