// Kernels of the learned warm start (a small U-Net): BF16 GEMM on the
// matrix cores with FP32 accumulation, 3x3 convolutions and their gradients,
// pooling, upsampling, ReLU, bias reductions, MSE and Adam.
//
// Activations are FP32 in [C][N][H][W] order (channel planes over the whole
// batch).  The network's layers run k_conv3, k_conv3_dgrad and k_conv3_wgrad; the
// primitives fhs_nn_im2col3, fhs_nn_col2im3 and fhs_nn_gemm compose the same
// convolution:
//   forward      out[co][q]  = sum_k W[co][k] col[k][q] (+ bias, ReLU)
//   grad input   dcol[k][q]  = sum_co W[co][k] dout[co][q]  -> col2im gather
//   grad weight  dW[co][k]   = sum_q dout[co][q] col[k][q]
// with k = ci*9 + ky*3 + kx and q = (n, y, x).  Operands are rounded to BF16
// when staged in LDS; v_mfma_f32_16x16x16_bf16 accumulates in FP32.
#include <algorithm>
#include <cmath>

#include "common.hpp"

namespace fhs {
namespace {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned short to_bf16(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);   // round to nearest even
  return (unsigned short)(u >> 16);
}

constexpr int GT = 64;     // C tile edge
constexpr int GK = 16;     // k step (one MFMA depth)
constexpr int GTHREADS = 256;

// C (M x N, row-major ldc) = alpha op(A) op(B) + beta C (+ bias[m]) (ReLU)
// op(A)[m][k] = ta ? A[k*lda + m] : A[m*lda + k]; op(B)[k][n] = tb ? B[n*ldb + k] : B[k*ldb + n]
// Split-K: workgroup z sums k in [z*kchunk, (z+1)*kchunk) and, when part is
// given, stores alpha * (its partial product) to part[z][M][N]; k_gemm_reduce
// then adds the partials in z order (deterministic), beta C, bias and ReLU.
__global__ __launch_bounds__(GTHREADS) void k_gemm_bf16(int M, int N, int K, const float* __restrict__ A,
                                                        int lda, int ta, const float* __restrict__ B, int ldb,
                                                        int tb, float* __restrict__ Cm, int ldc, float alpha,
                                                        float beta, const float* __restrict__ bias, int relu,
                                                        int kchunk, float* __restrict__ part) {
  __shared__ unsigned short As[GT][GK + 4];
  __shared__ unsigned short Bs[GK][GT + 4];
  const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
  const int kb = blockIdx.z * kchunk, ke = min(K, kb + kchunk);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;   // wave sub-tile origin
  v4f acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  for (int k0 = kb; k0 < ke; k0 += GK) {
    for (int t = threadIdx.x; t < GT * GK; t += GTHREADS) {
      // A tile: GT rows x GK cols
      int r, c;
      if (ta) { r = t % GT; c = t / GT; } else { c = t % GK; r = t / GK; }
      const int m = m0 + r, k = k0 + c;
      float v = 0.f;
      if (m < M && k < ke) v = ta ? A[(size_t)k * lda + m] : A[(size_t)m * lda + k];
      As[r][c] = to_bf16(v);
    }
    for (int t = threadIdx.x; t < GT * GK; t += GTHREADS) {
      int r, c;   // r = k, c = n
      if (tb) { r = t % GK; c = t / GK; } else { c = t % GT; r = t / GT; }
      const int k = k0 + r, n = n0 + c;
      float v = 0.f;
      if (n < N && k < ke) v = tb ? B[(size_t)n * ldb + k] : B[(size_t)k * ldb + n];
      Bs[r][c] = to_bf16(v);
    }
    __syncthreads();
    // lane l: A fragment rows l%16, k 4*(l/16)..+3 ; B fragment k 4*(l/16)..+3, col l%16
    const int fr = lane & 15, fk = 4 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      v4s a;
      a[0] = (short)As[wm + 16 * i + fr][fk + 0];
      a[1] = (short)As[wm + 16 * i + fr][fk + 1];
      a[2] = (short)As[wm + 16 * i + fr][fk + 2];
      a[3] = (short)As[wm + 16 * i + fr][fk + 3];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        v4s b;
        b[0] = (short)Bs[fk + 0][wn + 16 * j + fr];
        b[1] = (short)Bs[fk + 1][wn + 16 * j + fr];
        b[2] = (short)Bs[fk + 2][wn + 16 * j + fr];
        b[3] = (short)Bs[fk + 3][wn + 16 * j + fr];
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[i][j], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // D[4*(lane/16) + r][lane%16]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
        const int n = n0 + wn + 16 * j + (lane & 15);
        if (m < M && n < N) {
          float v = alpha * acc[i][j][r];
          if (part) {
            part[((size_t)blockIdx.z * M + m) * N + n] = v;
            continue;
          }
          if (beta != 0.f) v += beta * Cm[(size_t)m * ldc + n];
          if (bias) v += bias[m];
          if (relu) v = fmaxf(v, 0.f);
          Cm[(size_t)m * ldc + n] = v;
        }
      }
}

__global__ void k_gemm_reduce(int M, int N, int splits, const float* __restrict__ part, float* __restrict__ Cm,
                              int ldc, float beta, const float* __restrict__ bias, int relu) {
  const int64_t total = (int64_t)M * N;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int m = (int)(i / N), n = (int)(i % N);
    float v = 0.f;
    for (int z = 0; z < splits; ++z) v += part[(size_t)z * total + i];
    if (beta != 0.f) v += beta * Cm[(size_t)m * ldc + n];
    if (bias) v += bias[m];
    if (relu) v = fmaxf(v, 0.f);
    Cm[(size_t)m * ldc + n] = v;
  }
}

// ---- 3x3 convolution without im2col ----------------------------------------
// The layers' own kernels: the gathered columns of a 3x3 convolution (9 FP32
// copies of the input) are never stored.  Operands are rounded to BF16 as they
// are staged in LDS and accumulated in FP32 by the same instruction, in the same
// order, as im2col + k_gemm_bf16 (+ k_col2im3) would: activations and gradients are
// the same bits.  (Any other order of the FP32
// sums flips a few BF16 roundings, and after four layers the network's roundings
// are all different ones.)
// A training step of the 16/32/64/128 network on four 8 x 256 x 256 tiles took
// 10.75 ms through im2col and GEMM (its weight gradients 160 us a layer, on a K of
// up to 262144 pixels read column by column) and takes 2.01: 18 to 35 us a layer
// forward, 39 to 54 for its weights, 15 to 63 for its input.  Staging and latency bound
// the kernels (the products alone are 69 us a step at a large GEMM's rate).

constexpr int CV_W = 32;          // output columns of a workgroup
constexpr int CV_R = CV_W + 2;    // staged columns, with the halo
constexpr int CV_C = 16;          // channels staged at a time: 9 k steps of 16

// The stage of both kernels, in registers until the previous one is consumed: a
// thread takes a pixel of the tile with its halo in CV_C channels.  Every load is
// unconditional (clamped address, value selected afterwards), so they are all in
// flight together while the matrix cores work on the stage before.
template <int RW, bool MASK>
struct ConvTile {
  static constexpr int PIX = (4 * RW + 2) * CV_R, LOADS = (PIX + GTHREADS - 1) / GTHREADS;
  float f[LOADS][CV_C], k[MASK ? LOADS : 1][CV_C];
  size_t at[LOADS];
  bool ok[LOADS];
  __device__ __forceinline__ void place(int x0, int y0, int H, int W, size_t plane) {
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
      const int p = threadIdx.x + u * GTHREADS;
      const int iy = y0 + p / CV_R - 1, ix = x0 + p % CV_R - 1;
      ok[u] = p < PIX && iy >= 0 && iy < H && ix >= 0 && ix < W;
      at[u] = plane + (ok[u] ? (size_t)iy * W + ix : 0);
    }
  }
  __device__ __forceinline__ void load(const float* in, const float* mask, int c0, int ci_n, size_t Q) {
#pragma unroll
    for (int u = 0; u < LOADS; ++u)
#pragma unroll
      for (int c = 0; c < CV_C; ++c) {
        const size_t a = min(c0 + c, ci_n - 1) * Q + at[u];
        f[u][c] = in[a];
        if (MASK) k[u][c] = mask[a];
      }
  }
  // the ReLU's gradient passes unless its output is <= 0
  __device__ __forceinline__ unsigned short value(int u, int c, int c0, int ci_n) const {
    const bool on = ok[u] && c0 + c < ci_n && !(MASK && k[MASK ? u : 0][c] <= 0.f);
    return on ? to_bf16(f[u][c]) : (unsigned short)0;
  }
};

// out[o][q] = sum_k W[o][k] in[k / 9][q + tap k % 9] + bias[o] (ReLU) for a tile of
// 4 RW x CV_W pixels (wave w makes rows RW w ..) and 16 MT output channels.  A lane's
// four consecutive k are four taps of at most two channels: it gathers them one by
// one from channel planes in LDS, at offsets that repeat every 16 channels (144 k).
template <int RW, int MT>
__global__ __launch_bounds__(GTHREADS) void k_conv3(const float* __restrict__ in, int ci_n, int NB, int H, int W,
                                                    const float* __restrict__ wt, int co_n,
                                                    const float* __restrict__ bias, int relu,
                                                    float* __restrict__ out) {
  using Tile = ConvTile<RW, false>;
  constexpr int KC = 9 * CV_C, WL = 16 * MT * KC / GTHREADS;
  __shared__ unsigned short xs[CV_C * Tile::PIX];
  __shared__ __align__(16) unsigned short ws[16 * MT * KC];
  const int tw = (W + CV_W - 1) / CV_W, th = (H + 4 * RW - 1) / (4 * RW);
  const int x0 = (blockIdx.x % tw) * CV_W, y0 = (blockIdx.x / tw % th) * 4 * RW, n = blockIdx.x / (tw * th);
  const int o0 = blockIdx.y * 16 * MT;
  const size_t Q = (size_t)NB * H * W, plane = (size_t)n * H * W;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
  Tile tile;
  float wv[WL];
  auto load = [&](int c0) {
    tile.load(in, nullptr, c0, ci_n, Q);
#pragma unroll
    for (int u = 0; u < WL; ++u) {
      const int e = threadIdx.x + u * GTHREADS, o = min(o0 + e / KC, co_n - 1), k = min(9 * c0 + e % KC, 9 * ci_n - 1);
      wv[u] = wt[(size_t)o * 9 * ci_n + k];
    }
  };
  int off[9][4];
#pragma unroll
  for (int s = 0; s < 9; ++s)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = 16 * s + 4 * g + j, t = k % 9;
      off[s][j] = k / 9 * Tile::PIX + (RW * wave + t / 3) * CV_R + t % 3 + li;
    }
  v4f acc[MT][2 * RW];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < 2 * RW; ++t) acc[m][t] = (v4f){0.f, 0.f, 0.f, 0.f};
  tile.place(x0, y0, H, W, plane);
  load(0);
  for (int c0 = 0; c0 < ci_n; c0 += CV_C) {
    if (c0) __syncthreads();
#pragma unroll
    for (int u = 0; u < Tile::LOADS; ++u) {
      const int p = threadIdx.x + u * GTHREADS;
      if (p < Tile::PIX)
#pragma unroll
        for (int c = 0; c < CV_C; ++c) xs[c * Tile::PIX + p] = tile.value(u, c, c0, ci_n);
    }
#pragma unroll
    for (int u = 0; u < WL; ++u) {
      const int e = threadIdx.x + u * GTHREADS;
      ws[e] = o0 + e / KC < co_n && 9 * c0 + e % KC < 9 * ci_n ? to_bf16(wv[u]) : (unsigned short)0;
    }
    __syncthreads();
    if (c0 + CV_C < ci_n) load(c0 + CV_C);
#pragma unroll
    for (int s = 0; s < 9; ++s) {
      if (9 * c0 + 16 * s >= 9 * ci_n) break;
      v4s a[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m] = *reinterpret_cast<const v4s*>(&ws[(16 * m + li) * KC + 16 * s + 4 * g]);
#pragma unroll
      for (int t = 0; t < 2 * RW; ++t) {
        v4s b;
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = (short)xs[off[s][j] + (t >> 1) * CV_R + (t & 1) * 16];
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[m], b, acc[m][t], 0, 0, 0);
      }
    }
  }
  // lane (pixel li, g) holds output channels 4 g .. 4 g + 3
#pragma unroll
  for (int t = 0; t < 2 * RW; ++t) {
    const int y = y0 + RW * wave + (t >> 1), x = x0 + (t & 1) * 16 + li;
    if (y < H && x < W) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int o = o0 + 16 * m + 4 * g + r;
          if (o < co_n) {
            float v = acc[m][t][r];
            if (bias) v += bias[o];
            if (relu) v = fmaxf(v, 0.f);
            out[o * Q + plane + (size_t)y * W + x] = v;
          }
        }
    }
  }
}

// Gradient with respect to the layer's input:
//   gin[i][q] = sum_t (sum_o W[o][i][t] g[o][q - t]),
// g = gout where the layer's output passed the ReLU (mask; MASK false: everywhere),
// for 4 x CV_W pixels and 16 input channels.  The nine taps keep a sum of their
// own over all output channels and are added at the end, t ascending and without
// those outside of the image.  A lane's four consecutive k are four channels of a
// pixel, one 8-byte read of pixel-major LDS.  (Two rows a wave: 144 sums a lane and one wave a
// SIMD, 92 us instead of 63 for 32 channels of 256 x 256 x 4.)
template <bool MASK>
__global__ __launch_bounds__(GTHREADS) void k_conv3_dgrad(const float* __restrict__ gout, int co_n, int NB, int H,
                                                          int W, const float* __restrict__ wt, int ci_n,
                                                          const float* __restrict__ mask, float* __restrict__ gin) {
  using Tile = ConvTile<1, MASK>;
  typedef unsigned short us8 __attribute__((ext_vector_type(8)));
  constexpr int KI = 9 * 16, WL = CV_C * KI / GTHREADS;
  __shared__ __align__(16) unsigned short gs[Tile::PIX * CV_C];
  __shared__ __align__(16) unsigned short ws[9 * 16 * CV_C];      // [tap][input channel][output channel]
  const int tw = (W + CV_W - 1) / CV_W, th = (H + 3) / 4;
  const int x0 = (blockIdx.x % tw) * CV_W, y0 = (blockIdx.x / tw % th) * 4, n = blockIdx.x / (tw * th);
  const int i0 = blockIdx.y * 16;
  const size_t Q = (size_t)NB * H * W, plane = (size_t)n * H * W;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
  Tile tile;
  float wv[WL];
  auto load = [&](int c0) {
    tile.load(gout, mask, c0, co_n, Q);
#pragma unroll
    for (int u = 0; u < WL; ++u) {
      const int e = threadIdx.x + u * GTHREADS, o = min(c0 + e / KI, co_n - 1), k = min(9 * i0 + e % KI, 9 * ci_n - 1);
      wv[u] = wt[(size_t)o * 9 * ci_n + k];
    }
  };
  v4f acc[9][2];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int p = 0; p < 2; ++p) acc[t][p] = (v4f){0.f, 0.f, 0.f, 0.f};
  tile.place(x0, y0, H, W, plane);
  load(0);
  for (int c0 = 0; c0 < co_n; c0 += CV_C) {
    if (c0) __syncthreads();
#pragma unroll
    for (int u = 0; u < Tile::LOADS; ++u) {
      const int p = threadIdx.x + u * GTHREADS;
      if (p < Tile::PIX)
#pragma unroll
        for (int c = 0; c < CV_C; c += 8) {
          us8 v;
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = tile.value(u, c + j, c0, co_n);
          *reinterpret_cast<us8*>(&gs[p * CV_C + c]) = v;
        }
    }
#pragma unroll
    for (int u = 0; u < WL; ++u) {
      const int e = threadIdx.x + u * GTHREADS, k = e % KI;
      const bool on = c0 + e / KI < co_n && 9 * i0 + k < 9 * ci_n;
      ws[(k % 9 * 16 + k / 9) * CV_C + e / KI] = on ? to_bf16(wv[u]) : (unsigned short)0;
    }
    __syncthreads();
    if (c0 + CV_C < co_n) load(c0 + CV_C);
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const v4s a = *reinterpret_cast<const v4s*>(&ws[(t * 16 + li) * CV_C + 4 * g]);
      const int p0 = (wave + 2 - t / 3) * CV_R + 2 - t % 3 + li;     // pixel q - t
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const v4s b = *reinterpret_cast<const v4s*>(&gs[(p0 + p * 16) * CV_C + 4 * g]);
        acc[t][p] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[t][p], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int y = y0 + wave, x = x0 + p * 16 + li;
    if (y < H && x < W) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = i0 + 4 * g + r;
        float v = 0.f;
#pragma unroll
        for (int t = 0; t < 9; ++t) {
          const int yy = y + 1 - t / 3, xx = x + 1 - t % 3;
          if (yy >= 0 && yy < H && xx >= 0 && xx < W) v += acc[t][p][r];
        }
        if (i < ci_n) gin[i * Q + plane + (size_t)y * W + x] = v;
      }
    }
  }
}

// Weight and bias gradients of the layer:
//   dW[o][i][t] = sum_q gy[o][q] x[i][q + t],  db[o] = sum_q gy[o][q],
// gy taken unless mask <= 0 (MASK false: everywhere).  A workgroup sums 16 output by
// 16 input channels over the kchunk pixels of its z, 16 a matrix instruction, as
// k_gemm_bf16 does; wave w makes the taps of kernel row w.  CW_ST pixels are staged
// at a time: a lane takes four in a row, shifts them along x between lanes and
// stores them once per tap, so every read of the loop is 8 aligned bytes.  Partial
// sums go to part and are added in z order by k_conv3_reduce.  db is summed in FP64
// from the unrounded gradient.
constexpr int CW_ST = 128, CW_S = CW_ST + 8, CW_THREADS = 192;

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// four values of a plane of Q at q: in one load where the whole stage lies inside
__device__ __forceinline__ v4f load_four(const float* __restrict__ p, int64_t q, int64_t Q, bool inside) {
  v4f f;
  if (inside) {
    f = *reinterpret_cast<const f4u*>(p + q);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] = p[min(max(q + j, (int64_t)0), Q - 1)];
  }
  return f;
}

template <bool MASK>
__global__ __launch_bounds__(CW_THREADS) void k_conv3_wgrad(const float* __restrict__ x, int ci_n, int NB, int H, int W,
                                                            const float* __restrict__ gy, int co_n,
                                                            const float* __restrict__ mask, int kchunk,
                                                            float* __restrict__ part, double* __restrict__ bpart) {
  __shared__ __align__(16) unsigned short gs[16 * CW_S];
  __shared__ __align__(16) unsigned short xs[9 * 16 * CW_S];
  constexpr int GL = (16 * CW_ST / 4 + CW_THREADS - 1) / CW_THREADS;
  const int64_t Q = (int64_t)NB * H * W;
  const int64_t kb = (int64_t)blockIdx.z * kchunk, ke = min(Q, kb + kchunk);
  const int o0 = blockIdx.x * 16, i0 = blockIdx.y * 16;
  const int lane = threadIdx.x & 63, ky = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
  const int half = lane >> 5, p4 = 4 * (lane & 31);
  const bool first = (lane & 31) == 0, last = (lane & 31) == 31;
  unsigned short* xw = xs + ky * 3 * 16 * CW_S;
  v4f xv[8], gv[GL], kv[MASK ? GL : 1];
  float xe[8];
  auto load = [&](int64_t q0) {
    const int64_t s0 = q0 + (int64_t)(ky - 1) * W;
    const bool xin = s0 >= 0 && s0 + CW_ST <= Q, gin = q0 + CW_ST <= Q;
    const int64_t edge = min(max(s0 + p4 + (first ? -1 : 4), (int64_t)0), Q - 1);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float* p = x + min(i0 + 2 * c + half, ci_n - 1) * Q;
      xv[c] = load_four(p, s0 + p4, Q, xin);
      xe[c] = p[edge];
    }
#pragma unroll
    for (int u = 0; u < GL; ++u) {
      const int e = threadIdx.x + u * CW_THREADS;
      const int64_t at = min(o0 + e / (CW_ST / 4), co_n - 1) * Q, q = q0 + e % (CW_ST / 4) * 4;
      gv[u] = load_four(gy + at, q, Q, gin);
      if (MASK) kv[u] = load_four(mask + at, q, Q, gin);
    }
  };
  v4f acc[3];
#pragma unroll
  for (int t = 0; t < 3; ++t) acc[t] = (v4f){0.f, 0.f, 0.f, 0.f};
  double bs[GL];
#pragma unroll
  for (int u = 0; u < GL; ++u) bs[u] = 0.0;
  load(kb);
  for (int64_t q0 = kb; q0 < ke; q0 += CW_ST) {
    if (q0 > kb) __syncthreads();
    bool on[3][4];      // the pixel's column of the tap lies in the image
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned q = (unsigned)(q0 + p4 + j), row = q / W, c = q - row * W;
      const int y = (int)(row % H) + ky - 1;
      on[1][j] = q0 + p4 + j < ke && y >= 0 && y < H;
      on[0][j] = on[1][j] && c > 0;
      on[2][j] = on[1][j] && c + 1 < (unsigned)W;
    }
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const bool ch = i0 + 2 * c + half < ci_n;
      float f[6];
#pragma unroll
      for (int j = 0; j < 4; ++j) f[1 + j] = xv[c][j];
      const float l = __shfl_up(f[4], 1), r = __shfl_down(f[1], 1);
      f[0] = first ? xe[c] : l;
      f[5] = last ? xe[c] : r;
      unsigned short h[6];
#pragma unroll
      for (int j = 0; j < 6; ++j) h[j] = to_bf16(f[j]);
#pragma unroll
      for (int kx = 0; kx < 3; ++kx) {
        v4s v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = ch && on[kx][j] ? (short)h[j + kx] : (short)0;
        *reinterpret_cast<v4s*>(&xw[(kx * 16 + 2 * c + half) * CW_S + p4]) = v;
      }
    }
#pragma unroll
    for (int u = 0; u < GL; ++u) {
      const int e = threadIdx.x + u * CW_THREADS, o = e / (CW_ST / 4), p = e % (CW_ST / 4) * 4;
      if (o < 16) {
        v4s v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bool ok = o0 + o < co_n && q0 + p + j < ke && !(MASK && kv[MASK ? u : 0][j] <= 0.f);
          const float f = ok ? gv[u][j] : 0.f;
          bs[u] += f;
          v[j] = (short)to_bf16(f);
        }
        *reinterpret_cast<v4s*>(&gs[o * CW_S + p]) = v;
      }
    }
    __syncthreads();
    if (q0 + CW_ST < ke) load(q0 + CW_ST);
#pragma unroll
    for (int s = 0; s < CW_ST / 16; ++s) {
      if (q0 + 16 * s >= ke) break;
      const v4s a = *reinterpret_cast<const v4s*>(&gs[li * CW_S + 16 * s + 4 * g]);
#pragma unroll
      for (int kx = 0; kx < 3; ++kx) {
        const v4s b = *reinterpret_cast<const v4s*>(&xw[(kx * 16 + li) * CW_S + 16 * s + 4 * g]);
        acc[kx] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[kx], 0, 0, 0);
      }
    }
  }
  float* out = part + (size_t)blockIdx.z * co_n * ci_n * 9;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int o = o0 + 4 * g + r, i = i0 + li;
    if (o < co_n && i < ci_n) {
#pragma unroll
      for (int kx = 0; kx < 3; ++kx) out[((size_t)o * ci_n + i) * 9 + 3 * ky + kx] = acc[kx][r];
    }
  }
  if (blockIdx.y == 0) {
#pragma unroll
    for (int u = 0; u < GL; ++u) {
      const int o = (threadIdx.x + u * CW_THREADS) / (CW_ST / 4);
      double s = bs[u];
      for (int d = 16; d; d >>= 1) s += __shfl_xor(s, d);
      if (first && o < 16 && o0 + o < co_n) bpart[(size_t)blockIdx.z * co_n + o0 + o] = s;
    }
  }
}

// dW[e] += sum_z part[z][e] in z order, db[o] += sum_z bpart[z][o].  A workgroup adds
// 32 weights, whose partials it first brings to LDS with all its threads, or one bias.
constexpr int CR_E = 32, CR_Z = 128;
__global__ __launch_bounds__(GTHREADS) void k_conv3_reduce(int nw, int nz, const float* __restrict__ part,
                                                           float* __restrict__ dw, int co_n,
                                                           const double* __restrict__ bpart, float* __restrict__ db) {
  __shared__ float sh[CR_Z][CR_E];
  __shared__ double bsh[4];
  const int wb = (nw + CR_E - 1) / CR_E;
  if ((int)blockIdx.x >= wb) {
    const int o = blockIdx.x - wb;
    double s[1] = {0.0};
    for (int z = threadIdx.x; z < nz; z += GTHREADS) s[0] += bpart[(size_t)z * co_n + o];
    block_sum<1>(s, bsh);
    if (threadIdx.x == 0) db[o] += (float)s[0];
    return;
  }
  const int c = threadIdx.x % CR_E, zr = threadIdx.x / CR_E, e = blockIdx.x * CR_E + c;
  float v = 0.f;
  for (int z0 = 0; z0 < nz; z0 += CR_Z) {
    if (z0) __syncthreads();
    const int zn = min(CR_Z, nz - z0);
#pragma unroll
    for (int k = 0; k < CR_Z; k += GTHREADS / CR_E)
      if (zr + k < zn) sh[zr + k][c] = part[(size_t)(z0 + zr + k) * nw + min(e, nw - 1)];
    __syncthreads();
    if (zr == 0)
#pragma unroll 8
      for (int z = 0; z < zn; ++z) v += sh[z][c];
  }
  if (zr == 0 && e < nw) dw[e] += v;
}

// col[ci*9 + ky*3 + kx][n, y, x] = in[ci][n][y + ky - 1][x + kx - 1]
__global__ void k_im2col3(const float* __restrict__ in, int C, int NB, int H, int W, float* __restrict__ col) {
  const int64_t Q = (int64_t)NB * H * W;
  const int64_t total = (int64_t)C * 9 * Q;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t q = i % Q;
    const int64_t kk = i / Q;
    const int ci = (int)(kk / 9), r = (int)(kk % 9), ky = r / 3, kx = r % 3;
    const int x = (int)(q % W), y = (int)((q / W) % H), n = (int)(q / ((int64_t)W * H));
    const int yy = y + ky - 1, xx = x + kx - 1;
    float v = 0.f;
    if (yy >= 0 && yy < H && xx >= 0 && xx < W) v = in[(((int64_t)ci * NB + n) * H + yy) * W + xx];
    col[i] = v;
  }
}

// din[ci][n][y][x] = sum_{ky,kx} dcol[ci*9 + ky*3 + kx][n, y - ky + 1, x - kx + 1]
__global__ void k_col2im3(const float* __restrict__ dcol, int C, int NB, int H, int W, float* __restrict__ din) {
  const int64_t Q = (int64_t)NB * H * W;
  const int64_t total = (int64_t)C * Q;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t q = i % Q;
    const int ci = (int)(i / Q);
    const int x = (int)(q % W), y = (int)((q / W) % H), n = (int)(q / ((int64_t)W * H));
    float s = 0.f;
    for (int ky = 0; ky < 3; ++ky) {
      const int yy = y - ky + 1;
      if (yy < 0 || yy >= H) continue;
      for (int kx = 0; kx < 3; ++kx) {
        const int xx = x - kx + 1;
        if (xx < 0 || xx >= W) continue;
        s += dcol[((int64_t)ci * 9 + ky * 3 + kx) * Q + ((int64_t)n * H + yy) * W + xx];
      }
    }
    din[i] = s;
  }
}

__global__ void k_relu_bwd(const float* __restrict__ y, float* __restrict__ g, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    if (y[i] <= 0.f) g[i] = 0.f;
}

// 2x2 max pooling over [C*NB] planes of H x W (H, W even)
__global__ void k_maxpool2(const float* __restrict__ in, int64_t planes, int H, int W, float* __restrict__ out) {
  const int Ho = H / 2, Wo = W / 2;
  const int64_t total = planes * Ho * Wo;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int x = (int)(i % Wo), y = (int)((i / Wo) % Ho);
    const int64_t p = i / ((int64_t)Wo * Ho);
    const float* b = in + (p * H + 2 * y) * W + 2 * x;
    out[i] = fmaxf(fmaxf(b[0], b[1]), fmaxf(b[W], b[W + 1]));
  }
}

// gradient goes to the first maximal element of each window
__global__ void k_maxpool2_bwd(const float* __restrict__ in, const float* __restrict__ gout, int64_t planes, int H,
                               int W, float* __restrict__ gin) {
  const int Ho = H / 2, Wo = W / 2;
  const int64_t total = planes * Ho * Wo;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int x = (int)(i % Wo), y = (int)((i / Wo) % Ho);
    const int64_t p = i / ((int64_t)Wo * Ho);
    const int64_t o = (p * H + 2 * y) * W + 2 * x;
    const float v[4] = {in[o], in[o + 1], in[o + W], in[o + W + 1]};
    int a = 0;
    for (int t = 1; t < 4; ++t)
      if (v[t] > v[a]) a = t;
    const float g = gout[i];
    gin[o] = a == 0 ? g : 0.f;
    gin[o + 1] = a == 1 ? g : 0.f;
    gin[o + W] = a == 2 ? g : 0.f;
    gin[o + W + 1] = a == 3 ? g : 0.f;
  }
}

// nearest 2x upsampling of [planes] H x W -> 2H x 2W, and its adjoint
__global__ void k_upsample2(const float* __restrict__ in, int64_t planes, int H, int W, float* __restrict__ out) {
  const int64_t total = planes * 4 * H * W;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int x = (int)(i % (2 * W)), y = (int)((i / (2 * W)) % (2 * H));
    const int64_t p = i / ((int64_t)4 * H * W);
    out[i] = in[(p * H + y / 2) * W + x / 2];
  }
}

__global__ void k_upsample2_bwd(const float* __restrict__ gout, int64_t planes, int H, int W,
                                float* __restrict__ gin) {
  const int64_t total = planes * H * W;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int x = (int)(i % W), y = (int)((i / W) % H);
    const int64_t p = i / ((int64_t)H * W);
    const float* g = gout + (p * 2 * H + 2 * y) * (2 * W) + 2 * x;
    gin[i] = g[0] + g[1] + g[2 * W] + g[2 * W + 1];
  }
}

// db[c] = sum_q g[c][q]  (one workgroup per channel, FP64 accumulation)
__global__ __launch_bounds__(256) void k_bias_grad(const float* __restrict__ g, int64_t Q, float* __restrict__ db) {
  __shared__ double sh[4];
  double s[1] = {0.0};
  const float* gc = g + (int64_t)blockIdx.x * Q;
  for (int64_t i = threadIdx.x; i < Q; i += blockDim.x) s[0] += gc[i];
  block_sum<1>(s, sh);
  if (threadIdx.x == 0) db[blockIdx.x] = (float)s[0];
}

// loss partials: sum (p - t)^2 ; grad = scale (p - t)
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ p, const float* __restrict__ t, int64_t n,
                                             float scale, float* __restrict__ grad, double* __restrict__ part) {
  __shared__ double sh[4];
  double s[1] = {0.0};
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float d = p[i] - t[i];
    s[0] += (double)d * d;
    if (grad) grad[i] = scale * d;
  }
  block_sum<1>(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, int64_t n, float lr, float b1, float b2, float eps, float c1, float c2) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

unsigned egrid(int64_t n) {
  const int64_t b = (n + 255) / 256;
  return (unsigned)(b < 8192 ? (b < 1 ? 1 : b) : 8192);
}

// k per workgroup: a long K over few output tiles (the weight gradient) is split
// across workgroups so that the chip fills, partials reduced in a fixed order
int gemm_kchunk(int M, int N, int64_t K) {
  const int64_t tiles = (int64_t)cdiv(N, GT) * cdiv(M, GT);
  int splits = 1;
  if (tiles < 1024 && K >= 4 * 1024) {
    splits = (int)std::min<int64_t>(cdiv(K, 1024), std::max<int64_t>(1, 2048 / tiles));
    splits = std::min(splits, 1024);
  }
  return (int)((cdiv(K, splits) + GK - 1) / GK * GK);
}

}  // namespace
}  // namespace fhs

using namespace fhs;

extern "C" {

int fhs_nn_gemm(fhs_ctx* ctx, int M, int N, int K, const float* A, int lda, int trans_a, const float* B,
                int ldb, int trans_b, float* C, int ldc, float alpha, float beta, const float* bias, int relu) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(M > 0 && N > 0 && K > 0 && A && B && C, "nn_gemm: bad argument");
    Scope sc(ctx, "nn_gemm");
    const int kchunk = gemm_kchunk(M, N, K), splits = (int)cdiv(K, kchunk);
    float* part = nullptr;
    if (splits > 1)
      part = (float*)ctx->ws.get("nn_gemm_split", (size_t)splits * M * N * sizeof(float));
    k_gemm_bf16<<<dim3(cdiv(N, GT), cdiv(M, GT), splits), GTHREADS, 0, ctx->stream>>>(
        M, N, K, A, lda, trans_a, B, ldb, trans_b, C, ldc, alpha, beta, bias, relu, kchunk, part);
    check_launch();
    if (splits > 1) {
      k_gemm_reduce<<<egrid((int64_t)M * N), 256, 0, ctx->stream>>>(M, N, splits, part, C, ldc, beta, bias, relu);
      check_launch();
    }
  });
}

int fhs_nn_conv3x3(fhs_ctx* ctx, const float* in, int cin, int NB, int H, int W, const float* w, int cout,
                   const float* bias, int relu, float* out) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(in && w && out && cin > 0 && cout > 0 && NB > 0 && H > 0 && W > 0, "nn_conv3x3: bad argument");
    Scope sc(ctx, "nn_conv3x3");
    // Two rows a wave and two groups of 16 output channels, which share the input
    // tile, where that still leaves two workgroups a CU (32 -> 32 channels, us, one row
    // and group, two rows, both: 512 such workgroups 35, 33, 26, 256 of them 18, 16.5,
    // 19, 64 of them 8.7, 12, 18.5; 16 -> 16 channels, rows: 512 13.7, 12.3, 256 8.9, 9.6)
    const bool rows2 = cdiv(W, CV_W) * cdiv(H, 8) * NB * cdiv(cout, 32) >= 512;
    const bool two = cout > 16 && rows2;
    const unsigned tiles = cdiv(W, CV_W) * cdiv(H, rows2 ? 8 : 4) * NB;
    auto run = [&](auto kern) {
      kern<<<dim3(tiles, cdiv(cout, two ? 32 : 16)), GTHREADS, 0, ctx->stream>>>(in, cin, NB, H, W, w, cout, bias, relu,
                                                                               out);
      check_launch();
    };
    if (two)
      run(k_conv3<2, 2>);
    else
      rows2 ? run(k_conv3<2, 1>) : run(k_conv3<1, 1>);
  });
}

int fhs_nn_conv3x3_backward(fhs_ctx* ctx, const float* in, int cin, int NB, int H, int W, const float* w, int cout,
                            const float* out_relu, const float* gout, float* dw, float* db, float* gin) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(in && w && gout && dw && db && cin > 0 && cout > 0 && NB > 0 && H > 0 && W > 0,
              "nn_conv3x3_backward: bad argument");
    {
      Scope sc(ctx, "nn_conv3x3_wgrad");
      const int64_t Q = (int64_t)NB * H * W;
      const int kchunk = gemm_kchunk(cout, 9 * cin, Q), nw = cout * cin * 9;
      const unsigned nz = cdiv(Q, kchunk);
      float* part = (float*)ctx->ws.get("nn_conv_dw", (size_t)nz * nw * sizeof(float));
      double* bpart = (double*)ctx->ws.get("nn_conv_db", (size_t)nz * cout * sizeof(double));
      auto run = [&](auto kern) {
        kern<<<dim3(cdiv(cout, 16), cdiv(cin, 16), nz), CW_THREADS, 0, ctx->stream>>>(in, cin, NB, H, W, gout, cout,
                                                                                     out_relu, kchunk, part, bpart);
        check_launch();
      };
      out_relu ? run(k_conv3_wgrad<true>) : run(k_conv3_wgrad<false>);
      k_conv3_reduce<<<cdiv(nw, CR_E) + cout, GTHREADS, 0, ctx->stream>>>(nw, (int)nz, part, dw, cout, bpart, db);
      check_launch();
    }
    if (gin) {
      Scope sc(ctx, "nn_conv3x3_dgrad");
      auto run = [&](auto kern) {
        kern<<<dim3(cdiv(W, CV_W) * cdiv(H, 4) * NB, cdiv(cin, 16)), GTHREADS, 0, ctx->stream>>>(
            gout, cout, NB, H, W, w, cin, out_relu, gin);
        check_launch();
      };
      out_relu ? run(k_conv3_dgrad<true>) : run(k_conv3_dgrad<false>);
    }
  });
}

int fhs_nn_im2col3(fhs_ctx* ctx, const float* in, int C, int NB, int H, int W, float* col) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    k_im2col3<<<egrid((int64_t)C * 9 * NB * H * W), 256, 0, ctx->stream>>>(in, C, NB, H, W, col);
    check_launch();
  });
}

int fhs_nn_col2im3(fhs_ctx* ctx, const float* dcol, int C, int NB, int H, int W, float* din) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    k_col2im3<<<egrid((int64_t)C * NB * H * W), 256, 0, ctx->stream>>>(dcol, C, NB, H, W, din);
    check_launch();
  });
}

int fhs_nn_relu_bwd(fhs_ctx* ctx, const float* y, float* g, int64_t n) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    k_relu_bwd<<<egrid(n), 256, 0, ctx->stream>>>(y, g, n);
    check_launch();
  });
}

int fhs_nn_maxpool2(fhs_ctx* ctx, const float* in, int64_t planes, int H, int W, float* out) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(H % 2 == 0 && W % 2 == 0, "nn_maxpool2: even sizes");
    k_maxpool2<<<egrid(planes * H * W / 4), 256, 0, ctx->stream>>>(in, planes, H, W, out);
    check_launch();
  });
}

int fhs_nn_maxpool2_bwd(fhs_ctx* ctx, const float* in, const float* gout, int64_t planes, int H, int W,
                        float* gin) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    k_maxpool2_bwd<<<egrid(planes * H * W / 4), 256, 0, ctx->stream>>>(in, gout, planes, H, W, gin);
    check_launch();
  });
}

int fhs_nn_upsample2(fhs_ctx* ctx, const float* in, int64_t planes, int H, int W, float* out) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    k_upsample2<<<egrid(planes * H * W * 4), 256, 0, ctx->stream>>>(in, planes, H, W, out);
    check_launch();
  });
}

int fhs_nn_upsample2_bwd(fhs_ctx* ctx, const float* gout, int64_t planes, int H, int W, float* gin) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    k_upsample2_bwd<<<egrid(planes * H * W), 256, 0, ctx->stream>>>(gout, planes, H, W, gin);
    check_launch();
  });
}

int fhs_nn_bias_grad(fhs_ctx* ctx, const float* g, int C, int64_t Q, float* db) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    k_bias_grad<<<C, 256, 0, ctx->stream>>>(g, Q, db);
    check_launch();
  });
}

int fhs_nn_mse(fhs_ctx* ctx, const float* pred, const float* target, int64_t n, float grad_scale, float* grad,
               double* loss) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    const unsigned G = egrid(n) < 1024 ? egrid(n) : 1024;
    double* part = (double*)ctx->ws.get("nn_mse_part", G * sizeof(double));
    k_mse<<<G, 256, 0, ctx->stream>>>(pred, target, n, grad_scale, grad, part);
    check_launch();
    std::vector<double> h(G);
    FHS_HIP(hipMemcpyAsync(h.data(), part, G * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    FHS_HIP(hipStreamSynchronize(ctx->stream));
    double s = 0.0;
    for (double v : h) s += v;
    if (loss) *loss = s;
  });
}

int fhs_nn_adam(fhs_ctx* ctx, float* w, const float* g, float* m, float* v, int64_t n, float lr, float beta1,
                float beta2, float eps, int step) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(step >= 1, "nn_adam: step >= 1");
    const float c1 = 1.f - std::pow(beta1, (float)step), c2 = 1.f - std::pow(beta2, (float)step);
    k_adam<<<egrid(n), 256, 0, ctx->stream>>>(w, g, m, v, n, lr, beta1, beta2, eps, c1, c2);
    check_launch();
  });
}

}  // extern "C"
