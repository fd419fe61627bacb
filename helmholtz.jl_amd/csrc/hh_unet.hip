// U-Net coarse-grid correction: BF16 activations/weights with FP32
// accumulation on MFMA (v_mfma_f32_16x16x16_bf16), hand-written forward,
// backward and Adam.
//
// Layout: activations NHWC with the pixel index x-fastest (p = i + nx*j, the
// solver's nodal order) and channels contiguous (multiples of 16).
// 3x3 convolution = implicit GEMM: out[p][co] = sum_{tap,ci} W[tap][co][ci]
// in[p + off(tap)][ci] (zero padding), a tile of pixels per block with its inputs
// in LDS.  Backward-data is the same kernel on the output gradient with W transposed and taps flipped; the
// weight gradient is a split-K MFMA over pixels with per-chunk partials summed
// in a fixed order (deterministic).  Down-sampling is nodal full weighting
// ([1 2 1]/4 per axis, stride 2, zero padding) and up-sampling nodal
// bilinear interpolation; their adjoints are each other up to a factor 4.
#include <cmath>
#include <cstring>
#include <stdexcept>
#include <string>

#include "hh_unet.h"

namespace hh {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __host__ __forceinline__ bf16 f2bf(float f) {
  unsigned u = __builtin_bit_cast(unsigned, f);
  u = u + 0x7fffu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__device__ __host__ __forceinline__ float bf2f(bf16 h) {
  unsigned u = ((unsigned)h) << 16;
  return __builtin_bit_cast(float, u);
}

struct ConvSpec {
  int ci, co, level;
};
// encoder 16/32/64, bottleneck 64, decoder with skip concatenations
static const ConvSpec kSpec[UNET_NCONV] = {{16, 16, 0},  {16, 16, 0},  {16, 32, 1}, {32, 32, 1}, {32, 64, 2},
                                           {64, 64, 2},  {64, 64, 3},  {64, 64, 3}, {128, 64, 2}, {64, 64, 2},
                                           {96, 32, 1},  {32, 32, 1},  {48, 16, 0}, {16, 16, 0}};

int64_t unet_param_count() {
  int64_t n = 0;
  for (int l = 0; l < UNET_NCONV; ++l) n += 9 * kSpec[l].co * kSpec[l].ci + kSpec[l].co;
  return n + 2 * 16 + 2;
}

static void ck(hipError_t e, const char* w) {
  if (e != hipSuccess) throw std::runtime_error(std::string(w) + ": " + hipGetErrorString(e));
}
template <typename T>
static T* dmal(size_t n) {
  void* p = nullptr;
  if (hipMalloc(&p, (n ? n : 1) * sizeof(T)) != hipSuccess) {
    (void)hipGetLastError();
    throw std::runtime_error("hipMalloc failed in U-Net workspace");
  }
  return (T*)p;
}

// ------------------------------------------------------------------ kernels
// The channels of an activation: [0, ca) in a, [ca, ca + cb) in b (the up-sampled
// and the skip part of a decoder layer's input; b is unused for one block)
struct Src {
  const bf16* a;
  const bf16* b;
  int ca, cb;
};
struct Dst {
  bf16* a;
  bf16* b;
  int ca, cb;
};

// A block computes a tile of tw x th pixels x wc NCO 16 output channels (channel
// block blockIdx.z): its four wavefronts are 4 / wc groups of pixels (G times the
// 16 pixels of an MFMA operand each, counted along the tile's rows) times wc
// groups of NCO channel blocks.  The tile's inputs with their one-pixel ring, all
// channels, are staged in LDS once (16-byte loads, zero outside the image; 16
// bytes of padding per pixel: the 16 pixels of an operand hit distinct banks), so
// that the nine taps read LDS.  The weights come in operand order (512 contiguous
// bytes per operand) and three (tap, 16-channel) steps ahead.  With the weights as
// the MFMA's rows a lane ends with four channels of one pixel: 8-byte stores.  A
// gradient leaves with the producing layer's ReLU mask applied where `mask` is
// that layer's output.
// The products' order (taps, then channel blocks, one accumulator per output) is
// that of the kernel before, which loaded pixels nine times over from L1 with a
// bounds test each and masked, joined and split activations in passes of their
// own.  One loss and gradient for 16 images of 129 x 129 on MI355X: the 27
// convolutions 690 us and those passes 197 us there, 325 us here in all, 125 TFLOP/s:
// the level-0 layers are bound by activations (12 us a
// launch against 4 us at the copy rate), the small levels by the chain of LDS
// reads and products of their one or two wavefronts per SIMD.
template <int NCO, int G>
__global__ __launch_bounds__(256) void k_conv3x3(Src in, const bf16* __restrict__ w, const float* __restrict__ bias,
                                                 Dst out, const bf16* __restrict__ mask, int nx, int ny, int relu,
                                                 int wc, int tw, int th, int xtiles) {
  extern __shared__ __align__(16) bf16 tile[];
  __shared__ int pix[256];
  const int cin = in.ca + in.cb, nb = (out.ca + out.cb) / 16;
  const int64_t ipx = (int64_t)blockIdx.y * nx * ny;  // the image's first pixel
  const int x0 = (int)(blockIdx.x % (unsigned)xtiles) * tw, y0 = (int)(blockIdx.x / (unsigned)xtiles) * th;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kq = (lane >> 4) * 4;
  const int cob0 = ((int)blockIdx.z * wc + wv % wc) * NCO, grp0 = (wv / wc) * G;
  const int ld = cin + 8, nch = cin / 8, sw = tw + 2;
  // output pixel of each of the tile's pixels (-1: none)
  if ((int)threadIdx.x < 64 * G / wc) {
    const int ly = (int)threadIdx.x / tw, lx = (int)threadIdx.x - ly * tw;
    pix[threadIdx.x] = ly < th && x0 + lx < nx && y0 + ly < ny ? (y0 + ly) * nx + x0 + lx : -1;
  }
  const int items = sw * (th + 2) * nch;
  for (int e0 = threadIdx.x; e0 < items; e0 += 1024) {
    uint4 v[4];
    int d[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = e0 + 256 * u;
      const int px = e / nch, ch = (e - px * nch) * 8, ly = px / sw, lx = px - ly * sw;
      const int gx = x0 - 1 + lx, gy = y0 - 1 + ly;
      d[u] = e < items ? px * ld + ch : -1;
      v[u] = make_uint4(0u, 0u, 0u, 0u);
      if (e < items && gx >= 0 && gx < nx && gy >= 0 && gy < ny) {
        const int64_t q = ipx + (int64_t)gy * nx + gx;
        v[u] = *(const uint4*)(ch < in.ca ? in.a + q * in.ca + ch : in.b + q * in.cb + (ch - in.ca));
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (d[u] >= 0) *(uint4*)(tile + d[u]) = v[u];
  }
  f4 acc[G][NCO];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int c = 0; c < NCO; ++c) acc[g][c] = f4{0.f, 0.f, 0.f, 0.f};
  const int steps = 9 * (cin / 16);
  const bf16* wl = w + ((int64_t)cob0 * 64 + lane) * 4;
  const int64_t wstep = (int64_t)nb * 256;
  s4 a[3][NCO];
#pragma unroll
  for (int u = 0; u < 3; ++u)
#pragma unroll
    for (int c = 0; c < NCO; ++c) a[u][c] = *(const s4*)(wl + u * wstep + c * 256);
  const bf16* tl[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int p = (grp0 + g) * 16 + m, ly = p / tw;
    tl[g] = tile + (ly < th ? ly * sw + p - ly * tw : 0) * ld + kq;
  }
  __syncthreads();
  int cb = 0, dx = 0, row = 0;
  for (int s = 0; s < steps; s += 3) {
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const int o = row + dx * ld + cb;
      s4 b[G];
#pragma unroll
      for (int g = 0; g < G; ++g) b[g] = *(const s4*)(tl[g] + o);
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int c = 0; c < NCO; ++c)
          acc[g][c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[u][c], b[g], acc[g][c], 0, 0, 0);
      // (the last steps load their own operands again)
      const int nx3 = s + u + 3 < steps ? s + u + 3 : s + u;
#pragma unroll
      for (int c = 0; c < NCO; ++c) a[u][c] = *(const s4*)(wl + nx3 * wstep + c * 256);
      cb += 16;
      if (cb == cin) {
        cb = 0;
        if (++dx == 3) {
          dx = 0;
          row += sw * ld;
        }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < NCO; ++c) {
    const int co = (cob0 + c) * 16 + kq;
    const bool first = co < out.ca;
    bf16* ob = first ? out.a + co : out.b + (co - out.ca);
    const int st = first ? out.ca : out.cb;
    const float4 bi = bias ? *(const float4*)(bias + co) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int p = pix[(grp0 + g) * 16 + m];
      if (p < 0) continue;
      float v[4] = {acc[g][c][0] + bi.x, acc[g][c][1] + bi.y, acc[g][c][2] + bi.z, acc[g][c][3] + bi.w};
      s4 r;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (relu) v[i] = v[i] > 0.f ? v[i] : 0.f;
        r[i] = (short)f2bf(v[i]);
      }
      const int64_t q = (ipx + p) * st;
      if (mask) {
        const s4 y = *(const s4*)(mask + q + co);
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = bf2f((bf16)y[i]) > 0.f ? r[i] : (short)0;
      }
      *(s4*)(ob + q) = r;
    }
  }
}

// Weight and bias gradients of a 3x3 layer as one MFMA GEMM per tap over
// pixels: dW[tap][co][ci] = sum_q dpre[q][co] in[q + off(tap)][ci] and
// db[co] = sum_q dpre[q][co].  A block takes the pixel range [q0, q0 + per) of
// the flattened (image, pixel) index and one 16-channel block of ci (grid.y),
// for all 9 taps and all output channels.  Each chunk of 64 pixels is staged
// once in LDS with 16-byte global loads, transposed so that the MFMA's
// reduction index (pixels) is contiguous: sA[co][px] = dpre, and the
// im2col of the input sB[tap][ci][px] (zero outside the image); a thread
// loads 4 pixels x 8 channels and stores each channel's 4 pixels as one
// 8-byte piece (a quarter of the LDS stores of one 2-byte store per value).  Every
// operand of v_mfma_f32_16x16x16bf16 (lane: 4 consecutive pixels of one
// channel) is then one aligned 8-byte LDS read; rows are padded to 68
// entries so the 16 lanes of a group hit distinct banks.  The 9 NCO tiles of
// 16x16 outputs are spread over the 4 wavefronts; partial sums per block are
// reduced in a fixed order afterwards (deterministic).
constexpr int WG_PX = 64;         // pixels per staged chunk
constexpr int WG_LD = WG_PX + 4;  // padded LDS row (136 B: 8-byte aligned pieces)

// Four pixels' 8 channels (v[i]: pixel i, channels 0..7, two per word) into
// the transposed tile: channel k's four pixels as one 8-byte store at
// dst + k WG_LD (dst 8-byte aligned)
__device__ __forceinline__ void store_px4(bf16* dst, const uint4 (&v)[4]) {
  const unsigned w[4][4] = {{v[0].x, v[0].y, v[0].z, v[0].w}, {v[1].x, v[1].y, v[1].z, v[1].w},
                            {v[2].x, v[2].y, v[2].z, v[2].w}, {v[3].x, v[3].y, v[3].z, v[3].w}};
#pragma unroll
  for (int h = 0; h < 4; ++h) {  // word h: channels 2h (low half) and 2h + 1 (high half)
    uint2 lo, hi;
    lo.x = (w[0][h] & 0xffffu) | (w[1][h] << 16);
    lo.y = (w[2][h] & 0xffffu) | (w[3][h] << 16);
    hi.x = (w[0][h] >> 16) | (w[1][h] & 0xffff0000u);
    hi.y = (w[2][h] >> 16) | (w[3][h] & 0xffff0000u);
    *(uint2*)(dst + (2 * h) * WG_LD) = lo;
    *(uint2*)(dst + (2 * h + 1) * WG_LD) = hi;
  }
}
template <int NCO>
__global__ __launch_bounds__(256) void k_conv_wgrad(const bf16* __restrict__ dpre, Src src, int nx, int ny,
                                                   int64_t total, int64_t per, float* __restrict__ part) {
  constexpr int COUT = 16 * NCO;
  constexpr int NTILE = 9 * NCO;
  constexpr int TPW = (NTILE + 3) / 4;
  constexpr int BPX = WG_PX * COUT / 256;
  __shared__ __align__(16) bf16 sA[COUT * WG_LD];
  __shared__ __align__(16) bf16 sB[9 * 16 * WG_LD];
  __shared__ int sbase[WG_PX], si[WG_PX], sj[WG_PX];
  const int cib = blockIdx.y, cin = src.ca + src.cb;
  const bf16* __restrict__ in = cib * 16 < src.ca ? src.a + cib * 16 : src.b + (cib * 16 - src.ca);
  const int ild = cib * 16 < src.ca ? src.ca : src.cb;  // the block's 16 channels at in + pixel ild
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kq = (lane >> 4) * 4;
  const int npix = nx * ny;
  const int64_t qb0 = (int64_t)blockIdx.x * per;
  const int64_t qb1 = qb0 + per < total ? qb0 + per : total;
  f4 acc[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
  float bsum = 0.f;
  for (int64_t q0 = qb0; q0 < qb1; q0 += WG_PX) {
    __syncthreads();  // the previous chunk's operands are consumed
    if (threadIdx.x < WG_PX) {
      const int64_t q = q0 + threadIdx.x;
      if (q < qb1) {
        const int64_t img = q / npix;
        const int p = (int)(q - img * npix);
        sbase[threadIdx.x] = (int)img;
        si[threadIdx.x] = p % nx;
        sj[threadIdx.x] = p / nx;
      } else {
        sbase[threadIdx.x] = -1;
      }
    }
    // dpre: 64 pixels x COUT channels; an item is 4 pixels x 8 channels (four
    // 16-byte loads), stored as one 8-byte row piece per channel
    for (int e = threadIdx.x; e < (WG_PX / 4) * (COUT / 8); e += 256) {
      const int px4 = e / (COUT / 8), c8 = (e % (COUT / 8)) * 8;
      uint4 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t q = q0 + 4 * px4 + i;
        v[i] = q < qb1 ? *(const uint4*)(dpre + q * COUT + c8) : make_uint4(0u, 0u, 0u, 0u);
      }
      store_px4(sA + c8 * WG_LD + 4 * px4, v);
    }
    __syncthreads();  // pixel coordinates
    // im2col of the input for this ci block: tap t, 4 pixels x 8 channels per item
    for (int e = threadIdx.x; e < 9 * (WG_PX / 4) * 2; e += 256) {
      const int t = e / ((WG_PX / 4) * 2), r = e % ((WG_PX / 4) * 2);
      const int px4 = r >> 1, c8 = (r & 1) * 8;
      uint4 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int px = 4 * px4 + i;
        v[i] = make_uint4(0u, 0u, 0u, 0u);
        const int img = sbase[px];
        if (img >= 0) {
          const int ii = si[px] + t % 3 - 1, jj = sj[px] + t / 3 - 1;
          if (ii >= 0 && ii < nx && jj >= 0 && jj < ny)
            v[i] = *(const uint4*)(in + ((int64_t)img * npix + (int64_t)jj * nx + ii) * ild + c8);
        }
      }
      store_px4(sB + (t * 16 + c8) * WG_LD + 4 * px4, v);
    }
    __syncthreads();
    // bias gradient (ci block 0 only): a thread sums BPX pixels of a channel.  One thread
    // per channel over all 64 held up the chunk's other wavefronts (27.2 us a launch of
    // 16 channels x 266k pixels, 26.1 so).
    if (cib == 0) {
      const bf16* q = sA + (threadIdx.x % COUT) * WG_LD + (threadIdx.x / COUT) * BPX;
#pragma unroll
      for (int px = 0; px < BPX; px += 4) {
        const s4 v = *(const s4*)(q + px);
#pragma unroll
        for (int i = 0; i < 4; ++i) bsum += bf2f((bf16)v[i]);
      }
    }
#pragma unroll
    for (int k0 = 0; k0 < WG_PX; k0 += 16) {
#pragma unroll
      for (int ti = 0; ti < TPW; ++ti) {
        const int tile = wv + 4 * ti;
        if (tile < NTILE) {
          const int t = tile / NCO, cob = tile % NCO;
          const s4 a = *(const s4*)(sA + (cob * 16 + m) * WG_LD + k0 + kq);
          const s4 b = *(const s4*)(sB + (t * 16 + m) * WG_LD + k0 + kq);
          acc[ti] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[ti], 0, 0, 0);
        }
      }
    }
  }
  // partials part[block][9 COUT cin + COUT]: the weights [tap][co][ci] (C row =
  // co, column = ci), then the bias [co] — the layer's own parameter layout,
  // so one reduction sums both
  const int64_t nw = 9LL * COUT * cin;
  float* out = part + (int64_t)blockIdx.x * (nw + COUT);
#pragma unroll
  for (int ti = 0; ti < TPW; ++ti) {
    const int tile = wv + 4 * ti;
    if (tile < NTILE) {
      const int t = tile / NCO, cob = tile % NCO;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        out[((int64_t)t * COUT + cob * 16 + kq + i) * cin + cib * 16 + m] = acc[ti][i];
    }
  }
  if (cib == 0) {
    float* sb = (float*)sA;  // the pixel groups' sums, added in order
    __syncthreads();
    sb[threadIdx.x] = bsum;
    __syncthreads();
    if (threadIdx.x < COUT) {
      float b = 0.f;
#pragma unroll
      for (int h = 0; h < 256 / COUT; ++h) b += sb[h * COUT + threadIdx.x];
      out[nw + threadIdx.x] = b;
    }
  }
}

// out[k] = sum_c part[c][k] in a fixed order: a block takes 16 outputs, its
// 16 thread rows sum the partials c = row, row + 16, ... and the first row adds
// the 16 row sums in order.  Bound by the latency of a thread's row of loads, so eight are
// in flight at a time (833 partials of 2320 values: 17.1 us one by one, 5.7 so; the
// training batch's fifteen launches 165 and 110 us).
__global__ __launch_bounds__(256) void k_sum_parts(const float* __restrict__ part, int nparts, int64_t n,
                                                   float* __restrict__ out) {
  __shared__ float sh[16][17];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int64_t k = (int64_t)blockIdx.x * 16 + tx;
  float acc = 0.f;
  if (k < n)
    for (int c = ty; c < nparts; c += 128) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = c + 16 * u < nparts ? part[(int64_t)(c + 16 * u) * n + k] : 0.f;
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += v[u];
    }
  sh[ty][tx] = acc;
  __syncthreads();
  if (ty == 0 && k < n) {
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) s += sh[r][tx];
    out[k] = s;
  }
}

// Eight channels of a pixel as floats, and back (rounded)
__device__ __forceinline__ void ld8(const bf16* p, float (&v)[8]) {
  const uint4 u = *(const uint4*)p;
  const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    v[2 * h] = __builtin_bit_cast(float, w[h] << 16);
    v[2 * h + 1] = __builtin_bit_cast(float, w[h] & 0xffff0000u);
  }
}
__device__ __forceinline__ void st8(bf16* p, const float (&v)[8], const bf16* __restrict__ mask) {
  float y[8];
  if (mask) ld8(mask, y);
  unsigned w[4];
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const unsigned lo = !mask || y[2 * h] > 0.f ? f2bf(v[2 * h]) : 0u;
    const unsigned hi = !mask || y[2 * h + 1] > 0.f ? f2bf(v[2 * h + 1]) : 0u;
    w[h] = lo | (hi << 16);
  }
  *(uint4*)p = make_uint4(w[0], w[1], w[2], w[3]);
}

// Nodal full weighting, stride 2, zero padding: out = scale * R in, with the ReLU
// mask of `mask` (that layer's output, or null).  A thread takes eight channels of
// a pixel (16-byte accesses, one index decomposition for the eight: the training
// batch's six launches 36 us, one value per thread 60 us; k_up's 38 and 127 us);
// blockIdx.y is the image.
__global__ __launch_bounds__(256) void k_down(const bf16* __restrict__ in, int C, int nx, int ny, bf16* __restrict__ out,
                                              int ncx, int ncy, float scale, const bf16* __restrict__ mask) {
  const unsigned k = blockIdx.x * 256 + threadIdx.x;
  const unsigned c8 = C / 8, nc = (unsigned)ncx * ncy, q = k / c8;
  if (q >= nc) return;
  const int c = (int)(k - q * c8) * 8;
  const int J = (int)(q / (unsigned)ncx), I = (int)q - J * ncx;
  const bf16* ib = in + (int64_t)blockIdx.y * nx * ny * C + c;
  const float wgt[3] = {0.25f, 0.5f, 0.25f};
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = -1; b <= 1; ++b) {
    const int j = 2 * J + b;
    if (j < 0 || j >= ny) continue;
#pragma unroll
    for (int a = -1; a <= 1; ++a) {
      const int i = 2 * I + a;
      if (i < 0 || i >= nx) continue;
      float v[8];
      ld8(ib + ((int64_t)j * nx + i) * C, v);
#pragma unroll
      for (int h = 0; h < 8; ++h) s[h] += wgt[a + 1] * wgt[b + 1] * v[h];
    }
  }
#pragma unroll
  for (int h = 0; h < 8; ++h) s[h] *= scale;
  const int64_t o = ((int64_t)blockIdx.y * nc + q) * C + c;
  st8(out + o, s, mask ? mask + o : nullptr);
}

// Nodal bilinear prolongation: out (+)= scale * P in, masked and split over threads
// as k_down
__global__ __launch_bounds__(256) void k_up(const bf16* __restrict__ in, int C, int ncx, int ncy, bf16* __restrict__ out,
                                            int nx, int ny, float scale, int accumulate,
                                            const bf16* __restrict__ mask) {
  const unsigned k = blockIdx.x * 256 + threadIdx.x;
  const unsigned c8 = C / 8, nf = (unsigned)nx * ny, q = k / c8;
  if (q >= nf) return;
  const int c = (int)(k - q * c8) * 8;
  const int j = (int)(q / (unsigned)nx), i = (int)q - j * nx;
  const int i0 = i >> 1, j0 = j >> 1;
  const bf16* ib = in + (int64_t)blockIdx.y * ncx * ncy * C + c;
  auto at = [&](int a, int b, float (&v)[8]) {
    if (a < ncx && b < ncy) {
      ld8(ib + ((int64_t)b * ncx + a) * C, v);
    } else {
#pragma unroll
      for (int h = 0; h < 8; ++h) v[h] = 0.f;
    }
  };
  float s[8], v[8];
  at(i0, j0, s);
  if (i & 1) {
    at(i0 + 1, j0, v);
#pragma unroll
    for (int h = 0; h < 8; ++h) s[h] += v[h];
  }
  if (j & 1) {
    at(i0, j0 + 1, v);
#pragma unroll
    for (int h = 0; h < 8; ++h) s[h] += v[h];
    if (i & 1) {
      at(i0 + 1, j0 + 1, v);
#pragma unroll
      for (int h = 0; h < 8; ++h) s[h] += v[h];
    }
  }
  const float f = ((i & 1) ? 0.5f : 1.f) * ((j & 1) ? 0.5f : 1.f);
  const int64_t o = ((int64_t)blockIdx.y * nf + q) * C + c;
#pragma unroll
  for (int h = 0; h < 8; ++h) s[h] = f * s[h] * scale;
  if (accumulate) {
    ld8(out + o, v);
#pragma unroll
    for (int h = 0; h < 8; ++h) s[h] += v[h];
  }
  st8(out + o, s, mask ? mask + o : nullptr);
}

// 1x1 head: y[p][o] = hb[o] + sum_c hw[o][c] x[p][c], 16 -> 2, fp32 out
__global__ __launch_bounds__(256) void k_head_fwd(const bf16* __restrict__ x, const float* __restrict__ hw,
                                                  const float* __restrict__ hb, float* __restrict__ y, int64_t npix) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= npix) return;
  float y0 = hb[0], y1 = hb[1];
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    const float v = bf2f(x[p * 16 + c]);
    y0 += hw[c] * v;
    y1 += hw[16 + c] * v;
  }
  y[2 * p] = y0;
  y[2 * p + 1] = y1;
}

// dx = hw^T dy (bf16) with x's own ReLU mask (x is a layer's output); per-block partial sums of dhw (2x16) and dhb (2).
// Bound by its one pass over x and dx: 16-byte accesses and a block per 512 pixels (266k
// pixels: 64 blocks with 2-byte accesses 67 us, 505 blocks so 14.7).
__global__ __launch_bounds__(256) void k_head_bwd(const bf16* __restrict__ x, const float* __restrict__ hw,
                                                  const float* __restrict__ dy, bf16* __restrict__ dx, int64_t npix,
                                                  int64_t chunk, float* __restrict__ part) {
  __shared__ float sh[34][64];
  const int64_t q0 = (int64_t)blockIdx.x * chunk;
  const int64_t q1 = q0 + chunk < npix ? q0 + chunk : npix;
  float acc[34];
#pragma unroll
  for (int k = 0; k < 34; ++k) acc[k] = 0.f;
  for (int64_t p = q0 + threadIdx.x; p < q1; p += 256) {
    const float2 dp = ((const float2*)dy)[p];
    const float d0 = dp.x, d1 = dp.y;
    float v[16], g[16];
    ld8(x + p * 16, *(float(*)[8])v);
    ld8(x + p * 16 + 8, *(float(*)[8])(v + 8));
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      acc[c] += d0 * v[c];
      acc[16 + c] += d1 * v[c];
      g[c] = v[c] > 0.f ? hw[c] * d0 + hw[16 + c] * d1 : 0.f;
    }
    st8(dx + p * 16, *(const float(*)[8])g, nullptr);
    st8(dx + p * 16 + 8, *(const float(*)[8])(g + 8), nullptr);
    acc[32] += d0;
    acc[33] += d1;
  }
  // reduce 256 threads -> 1 (fixed order): wave shuffles then LDS
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < 34; ++k) {
    float v = acc[k];
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if (lane == 0) sh[k][wv] = v;
  }
  __syncthreads();
  if (threadIdx.x < 34) {
    const int k = threadIdx.x;
    part[(int64_t)blockIdx.x * 34 + k] = sh[k][0] + sh[k][1] + sh[k][2] + sh[k][3];
  }
}

__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ y, const float* __restrict__ t,
                                             float* __restrict__ dy, float* __restrict__ parts, int64_t n, float inv_n) {
  __shared__ float sh[4];
  float s = 0.f;
  for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (int64_t)gridDim.x * 256) {
    const float d = y[k] - t[k];
    dy[k] = 2.f * d * inv_n;
    s += d * d;
  }
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) parts[blockIdx.x] = (sh[0] + sh[1] + sh[2] + sh[3]) * inv_n;
}

__global__ __launch_bounds__(256) void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                                              float* __restrict__ v, int64_t n, float lr, float b1, float b2, float eps,
                                              float c1, float c2) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  const float gk = g[k];
  const float mk = b1 * m[k] + (1.f - b1) * gk;
  const float vk = b2 * v[k] + (1.f - b2) * gk * gk;
  m[k] = mk;
  v[k] = vk;
  w[k] -= lr * (mk / c1) / (sqrtf(vk / c2) + eps);
}

// bf16 copies in operand order: 16 x 16 blocks [tap][k / 16][m / 16] of 64 lanes x 4
// values, lane (m % 16) + 16 ((k % 16) / 4), value k % 4.  wb: m = co, k = ci; wt:
// m = ci, k = co, taps flipped.
__global__ __launch_bounds__(256) void k_wcopy(const float* __restrict__ w, bf16* __restrict__ wb, bf16* __restrict__ wt,
                                               int co, int ci) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t n = 9LL * co * ci;
  if (k >= n) return;
  const int c_i = (int)(k % ci);
  const int64_t r = k / ci;
  const int c_o = (int)(r % co);
  const int tap = (int)(r / co);
  auto at = [](int t, int kk, int nk, int m, int nm) {
    return ((((int64_t)t * (nk / 16) + kk / 16) * (nm / 16) + m / 16) * 64 + m % 16 + 16 * (kk % 16 / 4)) * 4 + kk % 4;
  };
  const bf16 v = f2bf(w[k]);
  wb[at(tap, c_i, ci, c_o, co)] = v;
  wt[at(8 - tap, c_o, co, c_i, ci)] = v;
}

__device__ __forceinline__ uint64_t mix64(uint64_t x) {
  x ^= x >> 33;
  x *= 0xff51afd7ed558ccdULL;
  x ^= x >> 33;
  x *= 0xc4ceb9fe1a85ec53ULL;
  x ^= x >> 33;
  return x;
}
// normal(0, std) from a counter-based hash (Box-Muller)
__global__ __launch_bounds__(256) void k_randn(float* __restrict__ w, int64_t n, float stdv, uint64_t seed) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k >= n) return;
  const uint64_t h1 = mix64(seed * 0x9e3779b97f4a7c15ULL + 2 * (uint64_t)k + 1);
  const uint64_t h2 = mix64(h1 ^ 0x632be59bd9b4e019ULL);
  const float u1 = ((h1 >> 40) + 1.f) / 16777217.f, u2 = (h2 >> 40) / 16777216.f;
  w[k] = stdv * sqrtf(-2.f * logf(u1)) * cosf(6.28318530718f * u2);
}

// network input: [Re r, Im r] / rms(r), k^2 h^2, gamma / Re w, zeros
__global__ __launch_bounds__(256) void k_rms(const cx<float>* __restrict__ r, int64_t N, float* __restrict__ scale,
                                             const int* __restrict__ skip) {
  __shared__ float sh[4];
  const int img = blockIdx.x;
  if (skip && skip[img]) return;
  const cx<float>* rb = r + (int64_t)img * N;
  float s = 0.f;
  for (int64_t p = threadIdx.x; p < N; p += 256) s += cabs2(rb[p]);
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    const float t = sqrtf((sh[0] + sh[1] + sh[2] + sh[3]) / (float)N);
    scale[img] = t > 0.f ? t : 1.f;
  }
}

__global__ __launch_bounds__(256) void k_prep(const cx<float>* __restrict__ r, int64_t N, const float* __restrict__ kh2,
                                              const float* __restrict__ gw, const float* __restrict__ scale,
                                              bf16* __restrict__ x, const int* __restrict__ skip, int nimg) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k >= N * nimg) return;
  const int64_t img = k / N;
  const int64_t p = k - img * N;
  bf16* xo = x + k * UNET_CIN;
  if (skip && skip[img]) {
    for (int c = 0; c < UNET_CIN; ++c) xo[c] = 0;
    return;
  }
  const float is = 1.f / scale[img];
  const cx<float> v = r[k];
  xo[0] = f2bf(v.re * is);
  xo[1] = f2bf(v.im * is);
  xo[2] = f2bf(kh2[p]);
  xo[3] = f2bf(gw[p]);
#pragma unroll
  for (int c = 4; c < UNET_CIN; ++c) xo[c] = 0;
}

__global__ __launch_bounds__(256) void k_post(const float* __restrict__ y, int64_t N, const float* __restrict__ scale,
                                              float h2, cx<float>* __restrict__ e, const int* __restrict__ skip,
                                              int nimg) {
  const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (k >= N * nimg) return;
  const int64_t img = k / N;
  if (skip && skip[img]) return;
  const float s = scale[img] * h2;
  e[k] = mk<float>(s * y[2 * k], s * y[2 * k + 1]);
}

// ------------------------------------------------------------------ host side
static inline unsigned nblk(int64_t n) { return (unsigned)((n + 255) / 256); }

enum Act {
  A_A0, A_S0, A_D1, A_A1, A_S1, A_D2, A_A2, A_S2, A_D3, A_A3, A_B3, A_U2, A_C2, A_A4, A_B4, A_U1, A_C1, A_A5, A_B5,
  A_U0, A_C0, A_A6, A_B6, A_NUM
};
static const int kActLevel[A_NUM] = {0, 0, 1, 1, 1, 2, 2, 2, 3, 3, 3, 2, 2, 2, 2, 1, 1, 1, 1, 0, 0, 0, 0};
static const int kActC[A_NUM] = {16, 16, 16, 32, 32, 32, 64, 64, 64, 64, 64, 64, 128, 64, 64, 64, 96, 32, 32, 32, 48, 16, 16};
// conv layer l: input activation, output activation (-1 input = network input)
static const int kIn[UNET_NCONV] = {-1, A_A0, A_D1, A_A1, A_D2, A_A2, A_D3, A_A3, A_C2, A_A4, A_C1, A_A5, A_C0, A_A6};
static const int kOut[UNET_NCONV] = {A_A0, A_S0, A_A1, A_S1, A_A2, A_S2, A_A3, A_B3, A_A4, A_B4, A_A5, A_B5, A_A6, A_B6};

struct Dims {
  int nx[4], ny[4];
  int64_t T[4];
};
static Dims dims_of(int nimg, int nx, int ny) {
  Dims d;
  d.nx[0] = nx;
  d.ny[0] = ny;
  for (int l = 1; l < 4; ++l) {
    d.nx[l] = (d.nx[l - 1] + 1) / 2;
    d.ny[l] = (d.ny[l - 1] + 1) / 2;
  }
  for (int l = 0; l < 4; ++l) d.T[l] = (int64_t)nimg * d.nx[l] * d.ny[l];
  return d;
}

void UNetWork::release() {
  for (void* p : bufs)
    if (p) (void)hipFree(p);
  bufs.clear();
  if (scratch) (void)hipFree(scratch);
  scratch = nullptr;
  scratch_n = 0;
  nimg = nx = ny = 0;
}

// buffers: [0, A_NUM) activations, [A_NUM, 2 A_NUM) gradients (none for the decoder
// inputs A_C*, which are read and written as their two parts).  Reallocated when
// the shape grows; a smaller batch of the same grid reuses them (launches index
// with their own nimg).
static bool is_joined(int a) { return a == A_C0 || a == A_C1 || a == A_C2; }
static void ensure_ws(UNetWork& ws, int nimg, int nx, int ny) {
  if (ws.nx == nx && ws.ny == ny && nimg <= ws.nimg && !ws.bufs.empty()) return;
  for (void* p : ws.bufs)
    if (p) (void)hipFree(p);
  ws.bufs.assign(2 * A_NUM, nullptr);
  ws.nimg = ws.nx = ws.ny = 0;
  Dims d = dims_of(nimg, nx, ny);
  for (int a = 0; a < A_NUM; ++a) {
    if (is_joined(a)) continue;
    ws.bufs[a] = dmal<bf16>((size_t)d.T[kActLevel[a]] * kActC[a]);
    ws.bufs[A_NUM + a] = dmal<bf16>((size_t)d.T[kActLevel[a]] * kActC[a]);
  }
  ws.nimg = nimg;
  ws.nx = nx;
  ws.ny = ny;
}

static bf16* act(UNetWork& ws, int a) { return (bf16*)ws.bufs[a]; }
static bf16* grd(UNetWork& ws, int a) { return (bf16*)ws.bufs[A_NUM + a]; }

// the two parts of a decoder layer's input: up-sampled, skip
static void parts_of(int a, int* up, int* skip) {
  *up = a == A_C0 ? A_U0 : a == A_C1 ? A_U1 : A_U2;
  *skip = a == A_C0 ? A_S0 : a == A_C1 ? A_S1 : A_S2;
}
static Src src_of(UNetWork& ws, int a, const bf16* x) {
  if (a < 0) return {x, nullptr, UNET_CIN, 0};
  if (!is_joined(a)) return {act(ws, a), nullptr, kActC[a], 0};
  int u, k;
  parts_of(a, &u, &k);
  return {act(ws, u), act(ws, k), kActC[u], kActC[k]};
}
static Dst grad_of(UNetWork& ws, int a) {
  if (!is_joined(a)) return {grd(ws, a), nullptr, kActC[a], 0};
  int u, k;
  parts_of(a, &u, &k);
  return {grd(ws, u), grd(ws, k), kActC[u], kActC[k]};
}
static bool is_conv_out(int a) {
  for (int o : kOut)
    if (o == a) return true;
  return false;
}

// Shape of a convolution launch: G pixel groups and NCO channel blocks per
// wavefront, wc channel groups per block, tiles of tw x th pixels
struct ConvShape {
  int nco, g, wc, tw, th, xt, yt;
  size_t lds;
};
constexpr size_t CONV_LDS = 63 << 10;  // the largest tile (64 KiB less the pixel table)
// Tile of at most P pixels: the width (the image's, split evenly) for which the
// MFMAs, work done for the tile's unused slots included, and the staged pixels
// come to the least; false if no tile fits the LDS
static bool conv_tile(ConvShape* c, int P, int cin, int nx, int ny) {
  double best = 0;
  c->lds = 0;
  for (int w = 4; w <= 32; ++w) {
    const int xt = (nx + w - 1) / w, tw = (nx + xt - 1) / xt;
    int th = P / tw < ny ? P / tw : ny;
    if (th < 1) continue;
    const int yt = (ny + th - 1) / th;
    th = (ny + yt - 1) / yt;
    const int staged = (tw + 2) * (th + 2);
    const size_t lds = sizeof(bf16) * staged * (size_t)(cin + 8);
    const double cost = (double)xt * yt * (2 * P + staged);
    if (lds <= CONV_LDS && (c->lds == 0 || cost < best)) {
      best = cost;
      c->tw = tw;
      c->th = th;
      c->xt = xt;
      c->yt = yt;
      c->lds = lds;
    }
  }
  return c->lds != 0;
}
// The fewest operand loads per MFMA (1 / NCO + 1 / G) that still leave 2048
// wavefronts (two per SIMD), or the most wavefronts.  Channel groups share a
// block's tile as long as it keeps 64 pixels.
static ConvShape conv_shape(int cin, int cout, int nimg, int nx, int ny) {
  const int nb = cout / 16;
  ConvShape best{};
  double load = 0;
  for (int nco : {4, 3, 2, 1})
    for (int g : {4, 2, 1}) {
      if (nb % nco) continue;
      ConvShape c{};
      c.nco = nco;
      c.g = g;
      c.wc = g;
      while (nb / nco % c.wc) c.wc /= 2;
      if (!conv_tile(&c, 64 * g / c.wc, cin, nx, ny)) continue;
      const double waves = 4.0 * c.xt * c.yt * nimg * (nb / (nco * c.wc));
      const double l = 1.0 / nco + 1.0 / g;
      if (best.nco == 0 || (waves >= 2048 ? l < load - 1e-9 : load > 2.0)) {
        best = c;
        load = waves >= 2048 ? l : 3.0;
      }
    }
  return best;
}

static void conv_launch(Src in, const bf16* w, const float* bias, Dst out, const bf16* mask, int nimg, int nx, int ny,
                        int relu, hipStream_t s) {
  const int cin = in.ca + in.cb, cout = out.ca + out.cb;
  if (in.ca % 16 || in.cb % 16 || out.ca % 16 || out.cb % 16 || cin <= 0 || cout <= 0)
    throw std::runtime_error("unsupported channel count");
  const ConvShape c = conv_shape(cin, cout, nimg, nx, ny);
  const dim3 grid((unsigned)(c.xt * c.yt), (unsigned)nimg, (unsigned)(cout / 16 / (c.nco * c.wc)));
#define HH_CONV(N, G)                                                                                                  \
  case 8 * N + G:                                                                                                      \
    hipLaunchKernelGGL((k_conv3x3<N, G>), grid, dim3(256), c.lds, s, in, w, bias, out, mask, nx, ny, relu, c.wc, c.tw, \
                       c.th, c.xt);                                                                                    \
    break;
  switch (8 * c.nco + c.g) {
    HH_CONV(1, 1) HH_CONV(1, 2) HH_CONV(1, 4)
    HH_CONV(2, 1) HH_CONV(2, 2) HH_CONV(2, 4)
    HH_CONV(3, 1) HH_CONV(3, 2) HH_CONV(3, 4)
    HH_CONV(4, 1) HH_CONV(4, 2) HH_CONV(4, 4)
    default: throw std::runtime_error("unsupported channel count");
  }
#undef HH_CONV
}

// R and P between level lf and lf + 1 (k_down, k_up)
static void down_launch(const Dims& d, int nimg, const bf16* in, bf16* out, int C, int lf, float scale,
                        const bf16* mask, hipStream_t s) {
  const int64_t n = (int64_t)d.nx[lf + 1] * d.ny[lf + 1] * (C / 8);
  hipLaunchKernelGGL(k_down, dim3(nblk(n), (unsigned)nimg), dim3(256), 0, s, in, C, d.nx[lf], d.ny[lf], out,
                     d.nx[lf + 1], d.ny[lf + 1], scale, mask);
}
static void up_launch(const Dims& d, int nimg, const bf16* in, bf16* out, int C, int lf, float scale, int accumulate,
                      const bf16* mask, hipStream_t s) {
  const int64_t n = (int64_t)d.nx[lf] * d.ny[lf] * (C / 8);
  hipLaunchKernelGGL(k_up, dim3(nblk(n), (unsigned)nimg), dim3(256), 0, s, in, C, d.nx[lf + 1], d.ny[lf + 1], out,
                     d.nx[lf], d.ny[lf], scale, accumulate, mask);
}

void unet_sync_bf16(UNet& net) {
  for (int l = 0; l < UNET_NCONV; ++l) {
    const int64_t n = 9LL * kSpec[l].co * kSpec[l].ci;
    hipLaunchKernelGGL(k_wcopy, dim3(nblk(n)), dim3(256), 0, net.stream, net.w[l], net.wb[l], net.wt[l], kSpec[l].co,
                       kSpec[l].ci);
  }
}

void unet_init(UNet& net, uint64_t seed, hipStream_t s) {
  net.stream = s;
  net.nparam = unet_param_count();
  net.flat = dmal<float>(net.nparam);
  net.grad = dmal<float>(net.nparam);
  net.adam_m = dmal<float>(net.nparam);
  net.adam_v = dmal<float>(net.nparam);
  ck(hipMemsetAsync(net.flat, 0, sizeof(float) * net.nparam, s), "memset");
  ck(hipMemsetAsync(net.grad, 0, sizeof(float) * net.nparam, s), "memset");
  ck(hipMemsetAsync(net.adam_m, 0, sizeof(float) * net.nparam, s), "memset");
  ck(hipMemsetAsync(net.adam_v, 0, sizeof(float) * net.nparam, s), "memset");
  int64_t off = 0;
  for (int l = 0; l < UNET_NCONV; ++l) {
    const int64_t nw = 9LL * kSpec[l].co * kSpec[l].ci;
    net.w[l] = net.flat + off;
    off += nw;
    net.b[l] = net.flat + off;
    off += kSpec[l].co;
    const int fan_in = 9 * (l == 0 ? UNET_FEATS : kSpec[l].ci);
    hipLaunchKernelGGL(k_randn, dim3(nblk(nw)), dim3(256), 0, s, net.w[l], nw, sqrtf(2.f / fan_in),
                       seed * 131 + l);
    net.wb[l] = dmal<bf16>(nw);
    net.wt[l] = dmal<bf16>(nw);
  }
  net.hw = net.flat + off;
  off += 32;
  net.hb = net.flat + off;
  hipLaunchKernelGGL(k_randn, dim3(1), dim3(256), 0, s, net.hw, (int64_t)32, 0.25f, seed * 131 + 99);
  net.adam_t = 0;
  unet_sync_bf16(net);
  ck(hipGetLastError(), "unet_init");
}

void unet_free(UNet& net) {
  for (int l = 0; l < UNET_NCONV; ++l) {
    if (net.wb[l]) (void)hipFree(net.wb[l]);
    if (net.wt[l]) (void)hipFree(net.wt[l]);
  }
  for (float* p : {net.flat, net.grad, net.adam_m, net.adam_v})
    if (p) (void)hipFree(p);
  net = UNet{};
}

void unet_forward(const UNet& net, UNetWork& ws, hipStream_t s, int nimg, int nx, int ny, const bf16* x, float* y) {
  ensure_ws(ws, nimg, nx, ny);
  Dims d = dims_of(nimg, nx, ny);
  auto conv = [&](int l) {
    const int lv = kSpec[l].level;
    conv_launch(src_of(ws, kIn[l], x), net.wb[l], net.b[l], {act(ws, kOut[l]), nullptr, kSpec[l].co, 0}, nullptr, nimg,
                d.nx[lv], d.ny[lv], 1, s);
  };
  auto down = [&](int a_in, int a_out, int lf) {
    down_launch(d, nimg, act(ws, a_in), act(ws, a_out), kActC[a_in], lf, 1.f, nullptr, s);
  };
  auto up = [&](int a_in, int a_out, int lc) {
    up_launch(d, nimg, act(ws, a_in), act(ws, a_out), kActC[a_in], lc - 1, 1.f, 0, nullptr, s);
  };
  conv(0); conv(1); down(A_S0, A_D1, 0);
  conv(2); conv(3); down(A_S1, A_D2, 1);
  conv(4); conv(5); down(A_S2, A_D3, 2);
  conv(6); conv(7);
  up(A_B3, A_U2, 3);
  conv(8); conv(9);
  up(A_B4, A_U1, 2);
  conv(10); conv(11);
  up(A_B5, A_U0, 1);
  conv(12); conv(13);
  hipLaunchKernelGGL(k_head_fwd, dim3(nblk(d.T[0])), dim3(256), 0, s, act(ws, A_B6), net.hw, net.hb, y, d.T[0]);
}

static int64_t pick_chunks(int64_t total, int64_t* chunk) {
  int64_t nch = total / 512;
  if (nch < 1) nch = 1;
  if (nch > 512) nch = 512;
  int64_t c = (total + nch - 1) / nch;
  c = (c + 15) / 16 * 16;
  *chunk = c;
  return (total + c - 1) / c;
}

// Pixel blocks of the weight-gradient GEMM: a block walks its chunks of WG_PX
// pixels one after another (stage, barrier, MFMA), so few long blocks leave
// the kernel bound by that chain (about 60 us per launch whatever the layer's
// size when every block took at least 16 chunks).  Blocks of WG_MINCH chunks,
// at most WG_MAXBLK of them (past that the partials' reduction costs more
// than the shorter chains save) and as many as the partials' scratch holds for
// the layer (np weights and biases per block).
constexpr int64_t WG_MINCH = 2;
constexpr int64_t WG_MAXBLK = 1024;
constexpr int64_t WG_SCRATCH = 64LL << 20;  // floats of weight-gradient partials
static int64_t pick_wgrad_blocks(int64_t total, int64_t np, int64_t* per) {
  int64_t nb = (total + WG_MINCH * WG_PX - 1) / (WG_MINCH * WG_PX);
  if (nb > WG_MAXBLK) nb = WG_MAXBLK;
  const int64_t cap = WG_SCRATCH / np;
  if (nb > cap) nb = cap;
  if (nb < 1) nb = 1;
  int64_t p = (total + nb - 1) / nb;
  p = (p + WG_PX - 1) / WG_PX * WG_PX;
  *per = p;
  return (total + p - 1) / p;
}

static void ensure_scratch(UNetWork& ws, int64_t n) {
  if (ws.scratch_n >= n) return;
  if (ws.scratch) (void)hipFree(ws.scratch);
  ws.scratch = nullptr;
  ws.scratch_n = 0;
  ws.scratch = dmal<float>(n);
  ws.scratch_n = n;
}

void unet_backward(UNet& net, UNetWork& ws, hipStream_t s, int nimg, int nx, int ny, const bf16* x, const float* dy) {
  Dims d = dims_of(nimg, nx, ny);
  // scratch: weight- and bias-gradient partials (WG_SCRATCH floats), or head
  // partials
  ensure_scratch(ws, WG_SCRATCH);
  const int64_t head_off = unet_param_count() - 34;
  // head
  {
    int64_t chunk;
    const int64_t nch = pick_chunks(d.T[0], &chunk);
    hipLaunchKernelGGL(k_head_bwd, dim3((unsigned)nch), dim3(256), 0, s, act(ws, A_B6), net.hw, dy, grd(ws, A_B6),
                       d.T[0], chunk, ws.scratch);
    hipLaunchKernelGGL(k_sum_parts, dim3(3), dim3(256), 0, s, ws.scratch, (int)nch, (int64_t)34, net.grad + head_off);
  }
  int64_t off[UNET_NCONV];
  {
    int64_t o = 0;
    for (int l = 0; l < UNET_NCONV; ++l) {
      off[l] = o;
      o += 9LL * kSpec[l].co * kSpec[l].ci + kSpec[l].co;
    }
  }
  // conv layer backward: the gradient before the ReLU (each pass that completes the
  // gradient of a layer's output masks it) -> dW, db, g(in)
  auto conv_b = [&](int l, bool need_din) {
    const ConvSpec& c = kSpec[l];
    const int lv = c.level;
    const int64_t T = d.T[lv];
    const bf16* dpre = grd(ws, kOut[l]);
    const Src in = src_of(ws, kIn[l], x);
    int64_t per;
    const int64_t np = 9LL * c.co * c.ci + c.co;  // the layer's weights and bias
    const int64_t nb = pick_wgrad_blocks(T, np, &per);
    float* pw = ws.scratch;
    const dim3 g((unsigned)nb, (unsigned)(c.ci / 16));
    switch (c.co / 16) {
      case 1: hipLaunchKernelGGL(k_conv_wgrad<1>, g, dim3(256), 0, s, dpre, in, d.nx[lv], d.ny[lv], T, per, pw); break;
      case 2: hipLaunchKernelGGL(k_conv_wgrad<2>, g, dim3(256), 0, s, dpre, in, d.nx[lv], d.ny[lv], T, per, pw); break;
      case 4: hipLaunchKernelGGL(k_conv_wgrad<4>, g, dim3(256), 0, s, dpre, in, d.nx[lv], d.ny[lv], T, per, pw); break;
      default: throw std::runtime_error("unsupported output channel count");
    }
    hipLaunchKernelGGL(k_sum_parts, dim3((unsigned)((np + 15) / 16)), dim3(256), 0, s, pw, (int)nb, np,
                       net.grad + off[l]);
    if (need_din)
      conv_launch({dpre, nullptr, c.co, 0}, net.wt[l], nullptr, grad_of(ws, kIn[l]),
                  is_conv_out(kIn[l]) ? act(ws, kIn[l]) : nullptr, nimg, d.nx[lv], d.ny[lv], 0, s);
  };
  // g(b) = P^T g(u) = 4 R g(u)
  auto up_b = [&](int au, int ab, int lc) {
    down_launch(d, nimg, grd(ws, au), grd(ws, ab), kActC[au], lc - 1, 4.f, act(ws, ab), s);
  };
  // g(s) += R^T g(d) = P g(d) / 4
  auto down_b = [&](int ad, int as, int lf) {
    up_launch(d, nimg, grd(ws, ad), grd(ws, as), kActC[ad], lf, 0.25f, 1, act(ws, as), s);
  };
  conv_b(13, true); conv_b(12, true);
  up_b(A_U0, A_B5, 1);
  conv_b(11, true); conv_b(10, true);
  up_b(A_U1, A_B4, 2);
  conv_b(9, true); conv_b(8, true);
  up_b(A_U2, A_B3, 3);
  conv_b(7, true); conv_b(6, true);
  down_b(A_D3, A_S2, 2);
  conv_b(5, true); conv_b(4, true);
  down_b(A_D2, A_S1, 1);
  conv_b(3, true); conv_b(2, true);
  down_b(A_D1, A_S0, 0);
  conv_b(1, true); conv_b(0, false);
}

void unet_adam(UNet& net, float lr, float b1, float b2, float eps) {
  net.adam_t += 1;
  const float c1 = 1.f - powf(b1, (float)net.adam_t), c2 = 1.f - powf(b2, (float)net.adam_t);
  hipLaunchKernelGGL(k_adam, dim3(nblk(net.nparam)), dim3(256), 0, net.stream, net.flat, net.grad, net.adam_m,
                     net.adam_v, net.nparam, lr, b1, b2, eps, c1, c2);
  unet_sync_bf16(net);
}

void unet_prep_input(int nimg, int64_t N, const cx<float>* r, const float* kh2, const float* gw, bf16* x16,
                     float* scale, const int* skip, hipStream_t s) {
  hipLaunchKernelGGL(k_rms, dim3(nimg), dim3(256), 0, s, r, N, scale, skip);
  hipLaunchKernelGGL(k_prep, dim3(nblk(N * nimg)), dim3(256), 0, s, r, N, kh2, gw, scale, x16, skip, nimg);
}

void unet_post_output(int nimg, int64_t N, const float* y, const float* scale, float h2, cx<float>* e, const int* skip,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_post, dim3(nblk(N * nimg)), dim3(256), 0, s, y, N, scale, h2, e, skip, nimg);
}

void unet_mse(int64_t n, const float* y, const float* t, float* dy, float* loss_parts, int nparts, hipStream_t s) {
  hipLaunchKernelGGL(k_mse, dim3(nparts), dim3(256), 0, s, y, t, dy, loss_parts, n, 1.f / (float)n);
}

}  // namespace hh
