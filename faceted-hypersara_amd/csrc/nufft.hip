// Oversampled scaled 2-D FFT of the NUFFT: A = fft2(pad(sn .* x)) and its
// adjoint, batched over channels.
//
// The grid is Kty x Ktx (column-major, y contiguous); the image Ny x Nx sits
// in its top-left corner.  The image is real, so two of its columns make one
// complex y transform, and the adjoint needs the rows ky <= Kty / 2 of the grid's
// Hermitian part only.  Each transform is two passes through HBM:
//   forward : (1) y-pass: one workgroup per two image columns a, b: scale by sn
//                 and 1/2, zero pad to Kty, FFT of a + i b -> Z (Kty x Nx / 2);
//             (2) x-pass: one workgroup per B consecutive grid rows: the columns'
//                 rows from Z[ky] and Z[-ky], FFT of length Ktx -> Fx.
//   adjoint (adj_half; a small launch transforms all rows and single columns):
//             (1') x-pass: the real part of the image comes from the Hermitian
//                 part g[ky][kx] + conj g[-ky][-kx]; inverse FFT of its rows
//                 ky <= Kty / 2, first Nx outputs -> U (half of Kty, x Nx);
//             (2') y-pass of U[a] + i U[b]: real and imaginary part are the two
//                 columns, keep Ny outputs, * sn / 2 * scale.
// Against one transform per column and per row, us of (1) (2) (1') (2'): 16 grids of
// 1024^2 30 48 51 25 -> 20 51 42 18, 8 of 2048^2 61 119 132 52 -> 36 116 97 35, 4 of
// 4096^2 141 414 323 122 -> 79 377 277 77; the bytes of the full grid bound the x-passes.
// (Rows ky <= Kty / 2 in (2) too, each writing its mirror: 56 and 158 us at 1024 and
// 2048, since mirrored row groups are never aligned and write parts of lines.)
// Two columns, or rows, in one transform take each other's rounding, and half of a
// Hermitian grid is no longer averaged with the other half.  Error against FP64, one
// column a transform -> pairs: forward 1.55e-7 -> 1.59e-7, adjoint of a general grid
// 1.63e-7 -> 1.68e-7, of a Hermitian one 0.96e-7 -> 1.10e-7 (512 x 512 images).
// The y-passes use a register-resident radix-16 Stockham FFT whose first
// stage reads the column from global memory and whose last stage writes it
// (two LDS round trips at 4096 points).  The x-passes read and write B
// consecutive complex values per grid column (B = 16 -> 128-byte segments,
// B = 8 -> 64, B = 4 -> 32), keep the B transforms interleaved in LDS
// (s[i*B + b]) so that consecutive lanes touch consecutive LDS words, and
// run radix-4 Stockham stages in LDS (one radix-2 stage when log2 n is
// odd): measured faster than the register form for these strided passes.
// Twiddles come from an FP64-computed table exp(-2 pi i k/n).
#include <cmath>
#include <string>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "nufft.hpp"

namespace fhs {
namespace {

constexpr int ilog2(int n) { return n <= 1 ? 0 : 1 + ilog2(n >> 1); }

// ---- LDS radix-4 Stockham FFT (the x-passes) --------------------------------
template <int N, int B, int NT, bool INV>
__device__ __forceinline__ void fft_lds(float2* s, const float2* tw) {
  const int tid = threadIdx.x;
  constexpr int LOG = ilog2(N);
  int Ns = 1;
  if constexpr (LOG & 1) {
    constexpr int NB = (B * N / 2 + NT - 1) / NT;
    float2 v[NB][2];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int u = tid + q * NT;
      if (u < B * N / 2) {
        const int b = u % B, j = u / B;
        v[q][0] = s[j * B + b];
        v[q][1] = s[(j + N / 2) * B + b];
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int u = tid + q * NT;
      if (u < B * N / 2) {
        const int b = u % B, j = u / B;
        s[(2 * j) * B + b] = cadd(v[q][0], v[q][1]);
        s[(2 * j + 1) * B + b] = csub(v[q][0], v[q][1]);
      }
    }
    __syncthreads();
    Ns = 2;
  }
#pragma unroll 1
  for (; Ns < N; Ns *= 4) {
    constexpr int NB = (B * N / 4 + NT - 1) / NT;
    const int tstride = N / (4 * Ns);
    float2 v[NB][4];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int u = tid + q * NT;
      if (u < B * N / 4) {
        const int b = u % B, j = u / B;
        const int k = j & (Ns - 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[q][r] = s[(j + r * (N / 4)) * B + b];
        if (k) {
#pragma unroll
          for (int r = 1; r < 4; ++r) {
            float2 w = tw[r * k * tstride];
            if (INV) w.y = -w.y;
            v[q][r] = cmul(v[q][r], w);
          }
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const int u = tid + q * NT;
      if (u < B * N / 4) {
        const int b = u % B, j = u / B;
        const int k = j & (Ns - 1);
        const float2 a0 = cadd(v[q][0], v[q][2]);
        const float2 a1 = csub(v[q][0], v[q][2]);
        const float2 a2 = cadd(v[q][1], v[q][3]);
        const float2 d = csub(v[q][1], v[q][3]);
        // forward: (v1 - v3) * (-i); inverse: * (+i)
        const float2 a3 = INV ? make_float2(-d.y, d.x) : make_float2(d.y, -d.x);
        const int base = (j / Ns) * Ns * 4 + k;
        s[(base)*B + b] = cadd(a0, a2);
        s[(base + Ns) * B + b] = cadd(a1, a3);
        s[(base + 2 * Ns) * B + b] = csub(a0, a2);
        s[(base + 3 * Ns) * B + b] = csub(a1, a3);
      }
    }
    __syncthreads();
  }
}

// The radix-4 stages read twiddles tw[r k tstride] < 3N/4.  They are staged
// in LDS once per workgroup (read behind the data loads' barrier) instead of
// a cache round trip in every stage.  The y-passes (one column, N x 8 bytes
// of LDS) always stage them; the x-passes up to N = 2048 only, since at
// N = 4096 the table would halve their occupancy.
template <int N>
constexpr int TW_LDS = (N < 4 || N > 2048) ? 1 : 3 * N / 4;
template <int N, int NT, int TWN>
__device__ __forceinline__ const float2* stage_twiddles(const float2* __restrict__ tw, float2* tws) {
  if constexpr (TWN == 1) return tw;
  for (int i = threadIdx.x; i < TWN; i += NT) tws[i] = tw[i];
  return tws;
}

// ---- register-resident Stockham FFT ----------------------------------------
// A length-N transform (N a power of two) is done in stages of radix R = 16
// (then one smaller radix for what remains: 2048 = 16 16 8).  A stage of
// sub-transform size NS takes butterfly j (0 <= j < N/R) with k = j mod NS:
//   v[r] = in[j + r N/R] * W_N^(r k N/(NS R)),  r < R,   (no twiddle at NS = 1)
//   v <- DFT_R(v),  out[(j / NS) NS R + k + r NS] = v[r],
// with W_N = exp(-2 pi i / N) (conjugated for the inverse).  Each thread keeps
// its butterfly's R values in registers; the first stage reads its inputs
// from global memory and the last writes its outputs there (first stage:
// n = j + r N/R; last stage: n = j + r N/R as well, since NS R = N), so a
// 4096-point transform makes two LDS round trips (three barriers) instead
// of the six of radix 4.  B transforms of a workgroup are interleaved in LDS
// (slot n B + b), with one pad slot per 16 rows so that the stride-R writes
// of the early stages do not all fall in one bank.
// cos / sin of 2 pi k / 16, k = 0..7
__device__ constexpr float kC16[8] = {1.f, 0.923879532511287f, 0.707106781186548f, 0.382683432365090f,
                                      0.f, -0.382683432365090f, -0.707106781186548f, -0.923879532511287f};
__device__ constexpr float kS16[8] = {0.f, 0.382683432365090f, 0.707106781186548f, 0.923879532511287f,
                                      1.f, 0.923879532511287f, 0.707106781186548f, 0.382683432365090f};

// in-place DFT of R = 1, 2, 4, 8 or 16 registers (radix-2 decimation in time)
template <int R, bool INV>
__device__ __forceinline__ void dft_reg(float2* v) {
  if constexpr (R == 2) {
    const float2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R > 2) {
    float2 e[R / 2], o[R / 2];
#pragma unroll
    for (int i = 0; i < R / 2; ++i) {
      e[i] = v[2 * i];
      o[i] = v[2 * i + 1];
    }
    dft_reg<R / 2, INV>(e);
    dft_reg<R / 2, INV>(o);
#pragma unroll
    for (int k = 0; k < R / 2; ++k) {
      const int q = k * (16 / R);   // W_R^k = W_16^q
      float2 t;
      if (q == 0) {
        t = o[k];
      } else if (q == 4) {          // -i forward, +i inverse
        t = INV ? make_float2(-o[k].y, o[k].x) : make_float2(o[k].y, -o[k].x);
      } else {
        const float2 w = make_float2(kC16[q], INV ? kS16[q] : -kS16[q]);
        t = cmul(o[k], w);
      }
      v[k] = cadd(e[k], t);
      v[k + R / 2] = csub(e[k], t);
    }
  }
}

__host__ __device__ constexpr int fft_pad(int n) { return n + (n >> 4); }

template <int N, int B>
constexpr int fft_lds_slots() { return fft_pad(N) * B + B; }

template <int N>
constexpr int fft_radix(int ns) { return N / ns >= 16 ? 16 : N / ns; }

// one stage; load(q, r, b, n) / store(q, r, b, n, v) serve the first / last
// stage (q: the thread's butterfly slot, r: its value index)
template <int N, int R, int NS, int B, int NT, bool INV, bool FIRST, bool LAST, class Load, class Store>
__device__ __forceinline__ void fft_stage(float2* s, const float2* __restrict__ tw, int tws, Load& load,
                                          Store& store) {
  constexpr int NBF = B * N / R;
  constexpr int PER = (NBF + NT - 1) / NT;
  constexpr int TS = N / (NS * R);
  float2 v[PER][R];
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int u = threadIdx.x + q * NT;
    if (u < NBF) {
      const int b = u % B, j = u / B;
      const int k = j & (NS - 1);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int n = j + r * (N / R);
        v[q][r] = FIRST ? load(q, r, b, n) : s[fft_pad(n) * B + b];
      }
      if (NS > 1 && k) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          float2 w = tw[(r * k * TS) * tws];
          if (INV) w.y = -w.y;
          v[q][r] = cmul(v[q][r], w);
        }
      }
      dft_reg<R, INV>(v[q]);
    }
  }
  if constexpr (!FIRST && !LAST) __syncthreads();   // in place: every read of the stage before its writes
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int u = threadIdx.x + q * NT;
    if (u < NBF) {
      const int b = u % B, j = u / B;
      const int k = j & (NS - 1);
      const int base = (j / NS) * NS * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int n = base + r * NS;
        if constexpr (LAST)
          store(q, r, b, n, v[q][r]);
        else
          s[fft_pad(n) * B + b] = v[q][r];
      }
    }
  }
  if constexpr (!LAST) __syncthreads();
}

template <int N, int NS, int B, int NT, bool INV, bool FIRST, class Load, class Store>
__device__ __forceinline__ void fft_stages(float2* s, const float2* __restrict__ tw, int tws, Load& load,
                                           Store& store) {
  constexpr int R = fft_radix<N>(NS);
  constexpr bool LAST = NS * R == N;
  fft_stage<N, R, NS, B, NT, INV, FIRST, LAST>(s, tw, tws, load, store);
  if constexpr (!LAST) fft_stages<N, NS * R, B, NT, INV, false>(s, tw, tws, load, store);
}

// B transforms of length N: inputs from load, outputs to store.  tw is the
// twiddle table exp(-2 pi i m / (N tws)) read at stride tws (tws = 2 for the
// half-length transforms of the split x-passes).  s: fft_lds_slots<N, B>()
// complex values of LDS.  Must be called by all NT threads (it has barriers).
template <int N, int B, int NT, bool INV, class Load, class Store>
__device__ __forceinline__ void fft_reg(float2* s, const float2* __restrict__ tw, int tws, Load& load,
                                        Store& store) {
  fft_stages<N, 1, B, NT, INV, true>(s, tw, tws, load, store);
}

// threads of a workgroup running B transforms of length n: one radix-16
// butterfly each (at least one wave, at most 1024)
template <int n, int B>
constexpr int fft_threads() { return B * n / 16 < 64 ? 64 : (B * n / 16 > 1024 ? 1024 : B * n / 16); }

// grid rows per x-pass workgroup: 16 up to N = 512, 8 at N = 1024 (two
// workgroups per CU), 4 from N = 2048 (64 KB of rows plus the twiddles, two
// workgroups per CU; 128 KB and one per CU at N = 4096, where 2 rows, 16-byte
// segments, measured slower).  Segments below 128 bytes are merged in one
// XCD's L2 (xpass_row0).
template <int N>
constexpr int b_strided() { return N >= 2048 ? 4 : (N >= 1024 ? 8 : 16); }
template <int N, int B>
constexpr int nt_strided() {
  return B * N / 4 > 1024 ? 1024 : (B * N / 4 < 64 ? 64 : B * N / 4);
}

// x-pass workgroup -> first of its B grid rows.  Workgroups are dispatched to the 8
// XCDs round-robin (linear id mod 8; gridDim.x is a multiple of 8, so blockIdx.x mod
// 8).  Forward: when B rows are fewer than a 128-byte line (G = 16 / B workgroups
// share each line of every grid column), workgroups b, b + 8, ..., b + 8 (G - 1)
// take G adjacent row groups, so the line is put together in one XCD's L2.
template <int B>
__device__ __forceinline__ int xpass_row0() {
  constexpr int G = 16 / B;
  const int b = blockIdx.x;
  if constexpr (G == 1) {
    return b * B;
  } else {
    if (gridDim.x % (8 * G)) return b * B;
    return ((b / (8 * G)) * (8 * G) + (b % 8) * G + (b / 8) % G) * B;
  }
}
// Runtime lengths and the adjoint, whose groups read their mirror too, which is not
// aligned: an XCD takes a contiguous eighth of the rows in turn, so that the lines two
// groups share meet in one L2 (adjoint x-pass, groups in launch order -> this, us: 16
// grids of 1024^2 64 -> 45, of 2048^2 417 -> 229, 4 of 1000 x 1440 49 -> 31).
__device__ __forceinline__ int xpass_eighth_row0(int B) {
  return ((blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8) * B;
}
inline unsigned xpass_eighth_grid(int rows, int B) { return (cdiv(rows, B) + 7) / 8 * 8; }

// ---- rows of a real image's transform ---------------------------------------
// An adjoint x-pass of the fixed sizes runs rows 0 .. half_rows(Kty) - 1: with Kty even
// rows 0 and Kty / 2, both Hermitian in kx (real outputs), share slot 0 as real and
// imaginary part, so that Kty / 2 transforms fill the grid exactly.
__host__ __device__ inline int half_rows(int Kty) { return Kty % 2 ? Kty / 2 + 1 : Kty / 2; }
// stride of a column of U (rows 0 .. Kty / 2), whole 128-byte lines
__host__ __device__ inline int half_stride(int Kty) { return (Kty / 2 + 1 + 15) / 16 * 16; }

// Row ky of columns 2 p and 2 p + 1 from z = Z[p][ky], m = Z[p][-ky] (1/2 is in Z)
__device__ __forceinline__ void split_pair(float2 z, float2 m, float2& a, float2& b) {
  a = make_float2(z.x + m.x, z.y - m.y);
  b = make_float2(z.y + m.y, m.x - z.x);
}

// The rows of an adjoint x-pass thread: its own, its mirror, and the second row of the
// shared slot.  A thread beyond the last row idles on row 0.
struct HalfRow {
  int ky, mirror, second;
  bool valid, shared;
  __device__ __forceinline__ HalfRow(int k, int Kty) {
    valid = k < half_rows(Kty);
    ky = valid ? k : 0;
    mirror = ky ? Kty - ky : 0;
    shared = ky == 0 && Kty % 2 == 0;
    second = Kty / 2;
  }
};

// an adjoint x-pass output: the shared slot holds row 0 and row Kty / 2, both real
__device__ __forceinline__ void adj_store(float2* __restrict__ col, const HalfRow& row, float2 u) {
  col[row.ky] = row.shared ? make_float2(u.x, 0.f) : u;
  if (row.shared) col[row.second] = make_float2(u.y, 0.f);
}

// twice the Hermitian part of the grid at (ky, kx)
__device__ __forceinline__ float2 hermitian(float2 v, float2 m) { return make_float2(v.x + m.x, v.y - m.y); }

// threads of a y-pass workgroup of an N-point grid
template <int N>
constexpr int nt_y() { return fft_threads<N, 1>(); }

// (1) forward y-pass: one workgroup per two image columns, scaled by sn, zero
// padded to N = Kty
template <int N>
__global__ __launch_bounds__(nt_y<N>()) void k_fwd_y(const float* __restrict__ x,
                                                              const float* __restrict__ sy,
                                                              const float* __restrict__ sx, int Ny, int Nx,
                                                              const float2* __restrict__ tw,
                                                              float2* __restrict__ Z) {
  constexpr int NT = fft_threads<N, 1>();
  __shared__ float2 s[fft_lds_slots<N, 1>()];
  const int ix = 2 * blockIdx.x, l = blockIdx.y, two = ix + 1 < Nx;
  const float* __restrict__ xa = x + ((size_t)l * Nx + ix) * Ny;
  const float* __restrict__ xb = xa + (two ? Ny : 0);
  const float sa = 0.5f * sx[ix], sb = two ? 0.5f * sx[ix + 1] : 0.f;
  float2* __restrict__ out = Z + ((size_t)l * gridDim.x + blockIdx.x) * N;
  auto load = [&](int, int, int, int n) {
    return n < Ny ? make_float2(xa[n] * sy[n] * sa, two ? xb[n] * sy[n] * sb : 0.f) : make_float2(0.f, 0.f);
  };
  auto store = [&](int, int, int, int n, float2 v) { out[n] = v; };
  fft_reg<N, 1, NT, false>(s, tw, 1, load, store);
}

// (2) forward x-pass: N = Ktx.  A thread's LDS slots are two neighbouring columns of
// one row: slots(j) = ((2 p) B + b, (2 p + 1) B + b) for pair p B + b = threadIdx.x + j NT.
template <int N, int B>
__global__ __launch_bounds__((nt_strided<N, B>())) void k_fwd_x(const float2* __restrict__ Z, int Kty,
                                                          int Nx, const float2* __restrict__ tw,
                                                          float2* __restrict__ Fx) {
  constexpr int NT = nt_strided<N, B>();
  static_assert(NT % B == 0 && N * B / 2 % NT == 0, "a thread keeps its row");
  __shared__ float2 s[N * B];
  __shared__ float2 tws[TW_LDS<N>];
  const int b = threadIdx.x % B, p0 = threadIdx.x / B, l = blockIdx.y, row = xpass_row0<B>() + b;
  const bool valid = row < Kty;
  const int ky = valid ? row : 0, mk = ky ? Kty - ky : 0;
  const float2* twp = stage_twiddles<N, NT, TW_LDS<N>>(tw, tws);
  const float2* Zl = Z + (size_t)l * ((Nx + 1) / 2) * Kty;
  constexpr int PER = N * B / 2 / NT;   // every load issued before the first LDS store
  float2 z[PER], m[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int p = p0 + j * (NT / B);
    const bool in = 2 * p < Nx;
    z[j] = in ? Zl[(size_t)p * Kty + ky] : make_float2(0.f, 0.f);
    m[j] = in ? Zl[(size_t)p * Kty + mk] : make_float2(0.f, 0.f);
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int p = p0 + j * (NT / B);
    float2 a, c;
    split_pair(z[j], m[j], a, c);
    s[2 * p * B + b] = a;
    s[(2 * p + 1) * B + b] = 2 * p + 1 < Nx ? c : make_float2(0.f, 0.f);
  }
  __syncthreads();
  fft_lds<N, B, NT, false>(s, twp);
  float2* F = Fx + (size_t)l * N * Kty;
  for (int t = threadIdx.x; t < N * B; t += NT) {
    if (valid) F[(size_t)(t / B) * Kty + ky] = s[t];
  }
}

// The first row of an adjoint x-pass workgroup, its thread's row and where the outputs
// go: HALF as above, or one of all Kty rows of a launch too small to gain from half of
// them (adj_half).
template <int B, bool HALF>
__device__ __forceinline__ int adj_row0() { return HALF ? xpass_eighth_row0(B) : xpass_row0<B>(); }

template <bool HALF>
__device__ __forceinline__ HalfRow adj_row(int k, int Kty) {
  HalfRow row(HALF ? k : 0, Kty);
  if (!HALF) {
    row.valid = k < Kty;
    row.ky = row.valid ? k : 0;
  }
  return row;
}

template <bool HALF>
__host__ __device__ inline int adj_stride(int Kty) { return HALF ? half_stride(Kty) : Kty; }

template <bool HALF>
__device__ __forceinline__ void adj_put(float2* __restrict__ col, const HalfRow& row, float2 u) {
  if (HALF)
    adj_store(col, row, u);
  else
    col[row.ky] = u;
}

// inputs of an adjoint x-pass thread: its values at columns STEP (PER of them, NT / B
// apart) + odd, every load issued before the first is used
template <int N, int B, int NT, int PER, int STEP, bool HALF>
__device__ __forceinline__ void adj_load(const float2* __restrict__ gl, int Kty, const HalfRow& row, int odd, float2* v) {
  float2 m[HALF ? PER : 1];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int k = STEP * ((threadIdx.x + j * NT) / B) + odd;
    v[j] = gl[(size_t)k * Kty + row.ky];
    if constexpr (HALF) m[j] = gl[(size_t)((N - k) % N) * Kty + row.mirror];
  }
  if constexpr (HALF) {
#pragma unroll
    for (int j = 0; j < PER; ++j) v[j] = hermitian(v[j], m[j]);
    if (row.shared)
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        const int k = STEP * ((threadIdx.x + j * NT) / B) + odd;
        const float2 h = hermitian(gl[(size_t)k * Kty + row.second], gl[(size_t)((N - k) % N) * Kty + row.second]);
        v[j] = make_float2(v[j].x - h.y, v[j].y + h.x);
      }
  }
}

// (1') adjoint x-pass: N = Ktx, keep the first Nx outputs
// (64 registers of a half's 8 values and their mirrors, for two workgroups of 1024 threads on a CU)
template <int N, int B, bool HALF>
__global__ __launch_bounds__((nt_strided<N, B>()), N * B <= 8192 ? 8 : 4) void k_adj_x(const float2* __restrict__ g, int Kty,
                                                          int Nx, const float2* __restrict__ tw,
                                                          float2* __restrict__ U) {
  constexpr int NT = nt_strided<N, B>();
  __shared__ float2 s[N * B];
  __shared__ float2 tws[TW_LDS<N>];
  const int l = blockIdx.y, ky0 = adj_row0<B, HALF>();
  if (HALF && ky0 >= half_rows(Kty)) return;
  const HalfRow row = adj_row<HALF>(ky0 + threadIdx.x % B, Kty);
  const float2* twp = stage_twiddles<N, NT, TW_LDS<N>>(tw, tws);
  constexpr int PER = N * B / NT;
  float2 v[PER];
  adj_load<N, B, NT, PER, 1, HALF>(g + (size_t)l * N * Kty, Kty, row, 0, v);
#pragma unroll
  for (int j = 0; j < PER; ++j) s[threadIdx.x + j * NT] = v[j];
  __syncthreads();
  fft_lds<N, B, NT, true>(s, twp);
  const int hs = adj_stride<HALF>(Kty);
  float2* Ul = U + (size_t)l * Nx * hs;
  if (row.valid)
    for (int t = threadIdx.x; t < Nx * B; t += NT) adj_put<HALF>(Ul + (size_t)(t / B) * hs, row, s[t]);
}

// Split x-passes for N >= X_SPLIT_MIN when the image holds at most half the
// grid columns (Nx <= N / 2, true of every 2x-oversampled grid).  With
// H = N / 2 and W = exp(-2 pi i / N):
//   forward : only x[0 .. H) is non-zero, so
//             X[2m] = FFT_H(x)[m],  X[2m + 1] = FFT_H(W^n x[n])[m];
//   adjoint : only y[0 .. H) is kept, so
//             y[n] = IFFT_H(g[2m])[n] + conj(W^n) IFFT_H(g[2m + 1])[n].
// The two H-point transforms run one after the other in the same H x B
// rows of LDS (64 KB at N = 4096 instead of 128 KB: two workgroups per CU),
// the H-point twiddles being every other entry of the N-point table.
// 64 registers, for those two workgroups of 1024 threads: a few spilled values cost less
// than one workgroup a CU (adjoint 332 -> 277 us, 4 grids of 4096^2).
constexpr int X_SPLIT_MIN = 4096;

template <int N, int B>
__global__ __launch_bounds__((nt_strided<N, B>()), B == 8 ? 4 : 8) void k_fwd_x_split(const float2* __restrict__ Z, int Kty,
                                                                int Nx, const float2* __restrict__ tw,
                                                                float2* __restrict__ Fx) {
  constexpr int H = N / 2;
  constexpr int NT = nt_strided<N, B>();
  static_assert(H * B / 2 % NT == 0 && NT % B == 0, "split x-pass: whole rows per thread");
  __shared__ float2 s[H * B];
  __shared__ float2 tws[3 * H / 4];
  const int b = threadIdx.x % B, p0 = threadIdx.x / B, l = blockIdx.y, row = xpass_row0<B>() + b;
  const bool valid = row < Kty;
  const int ky = valid ? row : 0, mk = ky ? Kty - ky : 0;
  for (int i = threadIdx.x; i < 3 * H / 4; i += NT) tws[i] = tw[2 * i];
  const float2* Zl = Z + (size_t)l * ((Nx + 1) / 2) * Kty;
  constexpr int PER = H * B / 2 / NT;
  float2 v[PER], w[PER];          // columns 2 p and 2 p + 1
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int p = p0 + j * (NT / B);
    const bool in = 2 * p < Nx;
    v[j] = in ? Zl[(size_t)p * Kty + ky] : make_float2(0.f, 0.f);
    w[j] = in ? Zl[(size_t)p * Kty + mk] : make_float2(0.f, 0.f);
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int p = p0 + j * (NT / B);
    float2 a, c;
    split_pair(v[j], w[j], a, c);
    v[j] = a;
    w[j] = 2 * p + 1 < Nx ? c : make_float2(0.f, 0.f);
    s[2 * p * B + b] = v[j];
    s[(2 * p + 1) * B + b] = w[j];
  }
  __syncthreads();
  fft_lds<H, B, NT, false>(s, tws);
  float2* F = Fx + (size_t)l * N * Kty;
#pragma unroll
  for (int j = 0; j < PER; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = 2 * (p0 + j * (NT / B)) + i;
      if (valid) F[(size_t)(2 * k) * Kty + ky] = s[k * B + b];
    }
  // each thread read back, and now overwrites, only its own LDS slots
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int k = 2 * (p0 + j * (NT / B));
    s[k * B + b] = cmul(v[j], tw[k]);
    s[(k + 1) * B + b] = cmul(w[j], tw[k + 1]);
  }
  __syncthreads();
  fft_lds<H, B, NT, false>(s, tws);
#pragma unroll
  for (int j = 0; j < PER; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = 2 * (p0 + j * (NT / B)) + i;
      if (valid) F[(size_t)(2 * k + 1) * Kty + ky] = s[k * B + b];
    }
}

template <int N, int B, bool HALF>
__global__ __launch_bounds__((nt_strided<N, B>()), B == 8 || !HALF ? 4 : 8) void k_adj_x_split(const float2* __restrict__ g, int Kty,
                                                                int Nx, const float2* __restrict__ tw,
                                                                float2* __restrict__ U) {
  constexpr int H = N / 2;
  constexpr int NT = nt_strided<N, B>();
  static_assert(H * B % NT == 0 && NT % B == 0, "split x-pass: whole rows per thread");
  __shared__ float2 s[H * B];
  __shared__ float2 tws[3 * H / 4];
  const int l = blockIdx.y, ky0 = adj_row0<B, HALF>();
  if (HALF && ky0 >= half_rows(Kty)) return;
  const HalfRow row = adj_row<HALF>(ky0 + threadIdx.x % B, Kty);
  for (int i = threadIdx.x; i < 3 * H / 4; i += NT) tws[i] = tw[2 * i];
  const float2* gl = g + (size_t)l * N * Kty;
  constexpr int PER = H * B / NT;
  float2 v[PER], e[PER];
  adj_load<N, B, NT, PER, 2, HALF>(gl, Kty, row, 0, v);
#pragma unroll
  for (int j = 0; j < PER; ++j) s[threadIdx.x + j * NT] = v[j];
  if (!HALF) adj_load<N, B, NT, PER, 2, HALF>(gl, Kty, row, 1, v);
  __syncthreads();
  fft_lds<H, B, NT, true>(s, tws);
  if (HALF) adj_load<N, B, NT, PER, 2, HALF>(gl, Kty, row, 1, v);
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int t = threadIdx.x + j * NT;
    e[j] = s[t];
    s[t] = v[j];
  }
  __syncthreads();
  fft_lds<H, B, NT, true>(s, tws);
  const int hs = adj_stride<HALF>(Kty);
  float2* Ul = U + (size_t)l * Nx * hs;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int t = threadIdx.x + j * NT, n = t / B;
    if (n < Nx && row.valid) {
      float2 w = tw[n];
      w.y = -w.y;
      adj_put<HALF>(Ul + (size_t)n * hs, row, cadd(e[j], cmul(s[t], w)));
    }
  }
}

// element n of U[a] + i U[b], both Hermitian with rows 0 .. N / 2 stored
__device__ __forceinline__ float2 join_pair(const float2* __restrict__ ua, const float2* __restrict__ ub, int N, int n) {
  const bool mirror = 2 * n > N;
  const int k = mirror ? N - n : n;
  const float2 a = ua[k], c = ub ? ub[k] : make_float2(0.f, 0.f);
  return mirror ? make_float2(a.x + c.y, c.x - a.y) : make_float2(a.x - c.y, a.y + c.x);
}

// (2') adjoint y-pass: N = Kty, two columns (HALF; else one, whole), keep Ny outputs,
// scale
template <int N, bool HALF>
__global__ __launch_bounds__(nt_y<N>()) void k_adj_y(const float2* __restrict__ U,
                                                              const float* __restrict__ sy,
                                                              const float* __restrict__ sx, int Ny, int Nx,
                                                              const float2* __restrict__ tw,
                                                              const float* __restrict__ scale,
                                                              float* __restrict__ out) {
  constexpr int NT = fft_threads<N, 1>();
  __shared__ float2 s[fft_lds_slots<N, 1>()];
  const int ix = (HALF ? 2 : 1) * blockIdx.x, l = blockIdx.y, hs = HALF ? half_stride(N) : N;
  const bool two = HALF && ix + 1 < Nx;
  const float2* __restrict__ ua = U + ((size_t)l * Nx + ix) * hs;
  const float2* __restrict__ ub = two ? ua + hs : nullptr;
  const float sc = (HALF ? 0.5f : 1.f) * (scale ? scale[l] : 1.f), sa = sc * sx[ix], sb = two ? sc * sx[ix + 1] : 0.f;
  float* __restrict__ o = out + ((size_t)l * Nx + ix) * Ny;
  auto load = [&](int, int, int, int n) { return HALF ? join_pair(ua, ub, N, n) : ua[n]; };
  auto store = [&](int, int, int, int n, float2 v) {
    if (n < Ny) {
      o[n] = sa * sy[n] * v.x;
      if (two) o[Ny + n] = sb * sy[n] * v.y;
    }
  };
  fft_reg<N, 1, NT, true>(s, tw, 1, load, store);
}

template <template <int> class K, class... Args>
void dispatch_pow2(int n, Args&&... args) {
  switch (n) {
#define FHS_CASE(v) \
  case v:           \
    K<v>::run(args...); \
    break;
    FHS_CASE(16) FHS_CASE(32) FHS_CASE(64) FHS_CASE(128) FHS_CASE(256) FHS_CASE(512)
    FHS_CASE(1024) FHS_CASE(2048) FHS_CASE(4096)
#undef FHS_CASE
    default:
      throw Error(FHS_ERR_UNSUPPORTED, "nufft: grid size must be a power of two in [16, 4096]");
  }
}

template <int N>
struct RunFwdY {
  static void run(hipStream_t st, int Nx, int L, const float* x, const fhs_nufft* p, float2* T) {
    k_fwd_y<N><<<dim3((Nx + 1) / 2, L), nt_y<N>(), 0, st>>>(x, p->sy, p->sx, p->Ny, p->Nx, p->twy, T);
  }
};
// Rows per x-pass workgroup: the default of a launch that fills the chip first, then
// the other candidates (those whose rows fit in LDS).
template <int N, bool SPLIT>
struct XRows {
  static constexpr int n = N >= 4096 ? (SPLIT ? 3 : 2) : N >= 256 ? 3 : 1;
  static constexpr int at(int i) {
    if (N >= 4096) return i == 0 ? 4 : i == 1 ? 2 : 8;
    if (N == 2048) return i == 0 ? 4 : i == 1 ? 2 : 8;
    if (N == 1024) return i == 0 ? 8 : i == 1 ? 4 : 16;
    if (N >= 256) return i == 0 ? 16 : i == 1 ? 8 : 4;
    return 16;
  }
};
constexpr int X_FULL = 256;   // workgroups that occupy every CU
// The rows of a launch without tuning: fewer than the default while CUs would stay
// idle (forward x-pass of one image, default rows -> these, us: 256 x 256 8.7 -> 5.2,
// 512 x 512 12.2 -> 8.8, 128 x 1024 12.2 -> 9.8).
template <int N, bool SPLIT>
int x_rows(int rows, int L) {
  using R = XRows<N, SPLIT>;
  int best = 0;
  for (int i = 1; i < R::n && (int64_t)cdiv(rows, R::at(best)) * L < X_FULL; ++i)
    if (R::at(i) < R::at(best)) best = i;
  return best;
}

inline bool is_pow2_grid(int n) { return n >= 16 && n <= 4096 && (n & (n - 1)) == 0; }

// Half of the rows and two columns a transform in the adjoint, where that is the
// faster form.  A launch that does not fill the chip is a chain of latencies, which
// mirrored rows and a second column lengthen.  And the mirrored rows are not aligned,
// so that every XCD's eighth of the rows costs a line more in each grid column,
// which the saved y-pass makes up for on tall grids, on wide ones only if tall enough
// and many.  All rows against half, us: 256 x 256 images 9.4, 15.6 (16 of them 23.7,
// 22.3), 512 x 512 13.7, 17.1 (4: 25.4, 25.0; 16: 67, 58), 1024 x 1024 x 4 84, 70;
// wide ones, 512 x 1024 x 4 45, 48 (16: 168, 142), 512 x 2048 x 4 85, 99 (16: 342,
// 326), 1024 x 2048 x 4 190, 159, 64 x 2048 x 16 62, 81.
inline bool adj_half(const fhs_nufft* p, int L) {
  if (!is_pow2_grid(p->Kty) || !is_pow2_grid(p->Ktx)) return true;
  const int B = p->Ktx >= 2048 ? 4 : p->Ktx >= 1024 ? 8 : 16;
  const int64_t groups = (int64_t)cdiv(half_rows(p->Kty), B) * L;
  return p->Kty >= p->Ktx ? groups >= X_FULL : groups >= 4 * X_FULL && p->Kty >= 1024;
}

template <int N, bool SPLIT, class F>
void with_rows(int i, F&& f) {
  using R = XRows<N, SPLIT>;
  switch (i) {
    case 0: f(std::integral_constant<int, R::at(0)>{}); break;
    case 1: if constexpr (R::n > 1) f(std::integral_constant<int, R::at(1)>{}); break;
    default: if constexpr (R::n > 2) f(std::integral_constant<int, R::at(2)>{}); break;
  }
}

template <int N, bool SPLIT>
const char* const* xrow_labels() {
  static const std::string lab[3] = {std::to_string(XRows<N, SPLIT>::at(0)) + " rows",
                                     std::to_string(XRows<N, SPLIT>::at(1)) + " rows",
                                     std::to_string(XRows<N, SPLIT>::at(2)) + " rows"};
  static const char* const p[3] = {lab[0].c_str(), lab[1].c_str(), lab[2].c_str()};
  return p;
}

inline std::string xpass_key(const char* k, int N, int Kty, int Nx, int L) {
  return std::string(k) + "/N" + std::to_string(N) + "xKty" + std::to_string(Kty) + "xNx" + std::to_string(Nx) +
         "xL" + std::to_string(L);
}

template <int N>
struct RunFwdX {
  static void run(fhs_ctx* ctx, int Kty, int L, const float2* T, const fhs_nufft* p, float2* F) {
    const bool split = N >= X_SPLIT_MIN && 2 * p->Nx <= N;
    auto go = [&](auto split_c) {
      constexpr bool SP = decltype(split_c)::value;
      tune_launch(ctx, xpass_key("fft_fwd_x", N, Kty, p->Nx, L), XRows<N, SP>::n, x_rows<N, SP>(Kty, L), xrow_labels<N, SP>(),
                  [&](int c) {
                    with_rows<N, SP>(c, [&](auto b_c) {
                      constexpr int B = decltype(b_c)::value;
                      if constexpr (SP)
                        k_fwd_x_split<N, B><<<dim3(cdiv(Kty, B), L), nt_strided<N, B>(), 0, ctx->stream>>>(T, Kty, p->Nx,
                                                                                                    p->twx, F);
                      else
                        k_fwd_x<N, B><<<dim3(cdiv(Kty, B), L), nt_strided<N, B>(), 0, ctx->stream>>>(T, Kty, p->Nx,
                                                                                              p->twx, F);
                      check_launch();
                    });
                  });
    };
    if constexpr (N >= X_SPLIT_MIN) {
      if (split) {
        go(std::true_type{});
        return;
      }
    }
    go(std::false_type{});
  }
};
template <int N>
struct RunAdjX {
  static void run(fhs_ctx* ctx, int Kty, int L, const float2* g, const fhs_nufft* p, float2* T) {
    const bool split = N >= X_SPLIT_MIN && 2 * p->Nx <= N;
    auto go = [&](auto split_c, auto half_c) {
      constexpr bool SP = decltype(split_c)::value, HALF = decltype(half_c)::value;
      const int rows = HALF ? half_rows(Kty) : Kty;
      tune_launch(ctx, xpass_key("fft_adj_x", N, Kty, p->Nx, L), XRows<N, SP>::n, x_rows<N, SP>(rows, L), xrow_labels<N, SP>(),
                  [&](int c) {
                    with_rows<N, SP>(c, [&](auto b_c) {
                      constexpr int B = decltype(b_c)::value;
                      const dim3 grid(HALF ? xpass_eighth_grid(rows, B) : cdiv(rows, B), L);
                      if constexpr (SP)
                        k_adj_x_split<N, B, HALF><<<grid, nt_strided<N, B>(), 0, ctx->stream>>>(g, Kty, p->Nx, p->twx, T);
                      else
                        k_adj_x<N, B, HALF><<<grid, nt_strided<N, B>(), 0, ctx->stream>>>(g, Kty, p->Nx, p->twx, T);
                      check_launch();
                    });
                  });
    };
    auto form = [&](auto split_c) { adj_half(p, L) ? go(split_c, std::true_type{}) : go(split_c, std::false_type{}); };
    if constexpr (N >= X_SPLIT_MIN) {
      if (split) {
        form(std::true_type{});
        return;
      }
    }
    form(std::false_type{});
  }
};
template <int N>
struct RunAdjY {
  static void run(hipStream_t st, int Nx, int L, const float2* T, const fhs_nufft* p,
                  const float* scale, float* out) {
    if (adj_half(p, L))
      k_adj_y<N, true><<<dim3((Nx + 1) / 2, L), nt_y<N>(), 0, st>>>(T, p->sy, p->sx, p->Ny, p->Nx, p->twy, scale, out);
    else
      k_adj_y<N, false><<<dim3(Nx, L), nt_y<N>(), 0, st>>>(T, p->sy, p->sx, p->Ny, p->Nx, p->twy, scale, out);
  }
};

float2* twiddles(int n) {
  std::vector<float2> h(n);
  for (int k = 0; k < n; ++k) {
    const double a = -2.0 * M_PI * (double)k / (double)n;
    h[k] = make_float2((float)std::cos(a), (float)std::sin(a));
  }
  float2* d = nullptr;
  FHS_HIP(hipMalloc(&d, n * sizeof(float2)));
  FHS_HIP(hipMemcpy(d, h.data(), n * sizeof(float2), hipMemcpyHostToDevice));
  return d;
}

// ---- grids that are not powers of two: runtime-length mixed radix ---------
// Grid sizes N = 2^a 3^b 5^c (an oversampled 2560-pixel axis is 5120 =
// 16 16 4 5) run the same register Stockham stages with the length known at
// run time: radix 16 while N/NS divides by 16, then the remaining power of
// two, then radix 5 and 3 stages (dft3 / dft5 below).  Each thread holds up
// to ceil(PT / R) butterflies of a radix-R stage; the x-passes use the same
// core on B rows per workgroup (no split form).
__device__ __forceinline__ int fft_radix_rt(int rem) {
  if (rem % 16 == 0) return 16;
  const int p2 = rem & -rem;
  if (p2 > 1) return p2;
  return rem % 5 == 0 ? 5 : 3;
}

template <bool INV>
__device__ __forceinline__ float2 mul_i(float2 z, float s) {   // z * (-i s) forward, z * (+i s) inverse
  return INV ? make_float2(-z.y * s, z.x * s) : make_float2(z.y * s, -z.x * s);
}

template <bool INV>
__device__ __forceinline__ void dft3(float2* x) {
  const float c = -0.5f, s = 0.866025403784438647f;   // cos, sin of 2 pi / 3
  const float2 t1 = cadd(x[1], x[2]);
  const float2 t2 = mul_i<INV>(csub(x[1], x[2]), s);
  const float2 u = make_float2(x[0].x + c * t1.x, x[0].y + c * t1.y);
  x[0] = cadd(x[0], t1);
  x[1] = cadd(u, t2);
  x[2] = csub(u, t2);
}

template <bool INV>
__device__ __forceinline__ void dft5(float2* x) {
  const float c1 = 0.309016994374947424f, s1 = 0.951056516295153572f;    // 2 pi / 5
  const float c2 = -0.809016994374947424f, s2 = 0.587785252292473129f;   // 4 pi / 5
  const float2 a1 = cadd(x[1], x[4]), b1 = csub(x[1], x[4]);
  const float2 a2 = cadd(x[2], x[3]), b2 = csub(x[2], x[3]);
  const float2 u1 = make_float2(x[0].x + c1 * a1.x + c2 * a2.x, x[0].y + c1 * a1.y + c2 * a2.y);
  const float2 u2 = make_float2(x[0].x + c2 * a1.x + c1 * a2.x, x[0].y + c2 * a1.y + c1 * a2.y);
  const float2 t1 = mul_i<INV>(make_float2(s1 * b1.x + s2 * b2.x, s1 * b1.y + s2 * b2.y), 1.f);
  const float2 t2 = mul_i<INV>(make_float2(s2 * b1.x - s1 * b2.x, s2 * b1.y - s1 * b2.y), 1.f);
  x[0] = cadd(x[0], cadd(a1, a2));
  x[1] = cadd(u1, t1);
  x[2] = cadd(u2, t2);
  x[3] = csub(u2, t2);
  x[4] = csub(u1, t1);
}

template <int R, bool INV>
__device__ __forceinline__ void dft_any(float2* v) {
  if constexpr (R == 3)
    dft3<INV>(v);
  else if constexpr (R == 5)
    dft5<INV>(v);
  else
    dft_reg<R, INV>(v);
}

template <int PT, int R, bool INV, class Load, class Store>
__device__ __forceinline__ void fft_stage_rt(float2* s, const float2* __restrict__ tw, int N, int NS, int B, int NT,
                                             bool first, bool last, Load& load, Store& store) {
  constexpr int PMAX = (PT + R - 1) / R;   // butterflies per thread (NT >= B N / PT)
  const int NBF = B * N / R;
  const int TS = N / (NS * R);
  // The thread's index is opaque to the compiler in each half of a stage: the addresses of
  // the first loads and last stores of all six radices do not change from stage to
  // stage, and were kept in registers, 1040 to 2180 bytes of them spilled in every lane
  // (now none, in 58 registers).
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  float2 v[PMAX][R];
#pragma unroll
  for (int q = 0; q < PMAX; ++q) {
    const int u = tid + q * NT;
    if (u < NBF) {
      const int b = u % B, j = u / B;
      const int k = j % NS;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int n = j + r * (N / R);
        v[q][r] = first ? load(q, r, b, n) : s[fft_pad(n) * B + b];
      }
      if (k) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          float2 w = tw[r * k * TS];
          if (INV) w.y = -w.y;
          v[q][r] = cmul(v[q][r], w);
        }
      }
      dft_any<R, INV>(v[q]);
    }
  }
  if (!first && !last) __syncthreads();
  asm volatile("" : "+v"(tid));
#pragma unroll
  for (int q = 0; q < PMAX; ++q) {
    const int u = tid + q * NT;
    if (u < NBF) {
      const int b = u % B, j = u / B;
      const int k = j % NS;
      const int base = (j / NS) * NS * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int n = base + r * NS;
        if (last)
          store(q, r, b, n, v[q][r]);
        else
          s[fft_pad(n) * B + b] = v[q][r];
      }
    }
  }
  if (!last) __syncthreads();
}

template <int PT, bool INV, class Load, class Store>
__device__ __forceinline__ void fft_rt(float2* s, const float2* __restrict__ tw, int N, int B, int NT, Load& load, Store& store) {
  int ns = 1;
  bool first = true;
  while (ns < N) {
    const int R = fft_radix_rt(N / ns);
    const bool last = ns * R == N;
    switch (R) {
      case 16: fft_stage_rt<PT, 16, INV>(s, tw, N, ns, B, NT, first, last, load, store); break;
      case 8: fft_stage_rt<PT, 8, INV>(s, tw, N, ns, B, NT, first, last, load, store); break;
      case 4: fft_stage_rt<PT, 4, INV>(s, tw, N, ns, B, NT, first, last, load, store); break;
      case 2: fft_stage_rt<PT, 2, INV>(s, tw, N, ns, B, NT, first, last, load, store); break;
      case 5: fft_stage_rt<PT, 5, INV>(s, tw, N, ns, B, NT, first, last, load, store); break;
      default: fft_stage_rt<PT, 3, INV>(s, tw, N, ns, B, NT, first, last, load, store); break;
    }
    ns *= R;
    first = false;
  }
}

// Values per thread of a runtime-length workgroup of B transforms, its threads and LDS
// bytes.  As few values as 1024 threads allow: the stages are a chain of
// latencies, which more threads shorten (one 1000 x 1440 grid, 16 values -> 4, us:
// x-passes 26 -> 21 and 25 -> 20; 128 pairs of 2000-point columns 16 -> 12 and 19 -> 12).
inline int fft_rt_values(int N, int B) { return B * N <= 4096 ? 4 : B * N <= 8192 ? 8 : 16; }
inline int fft_rt_threads(int N, int B) {
  const int t = (int)cdiv(B * N, fft_rt_values(N, B));
  return std::max(64, (t + 63) / 64 * 64);
}
inline size_t fft_rt_lds(int N, int B) { return ((size_t)fft_pad(N) * B + B) * sizeof(float2); }
template <class F>
void with_values(int v, F&& f) {
  if (v == 4)
    f(std::integral_constant<int, 4>{});
  else if (v == 8)
    f(std::integral_constant<int, 8>{});
  else
    f(std::integral_constant<int, 16>{});
}
// rows per runtime x-pass workgroup: 4, 2 or 1, with one radix-16 butterfly per
// thread (B N <= 16384) and the rows in LDS, fewer while CUs would stay idle.
inline int fft_rt_rows(int N, int rows, int L) {
  for (int B : {4, 2})
    if (B * N <= 16384 && fft_rt_lds(N, B) <= 150 * 1024 && (int64_t)cdiv(rows, B) * L >= 256) return B;
  return 1;
}

template <int PT>
__global__ __launch_bounds__(1024) void k_fwd_y_rt(const float* __restrict__ x, const float* __restrict__ sy,
                                                   const float* __restrict__ sx, int Ny, int Nx, int N,
                                                   const float2* __restrict__ tw, float2* __restrict__ Z) {
  extern __shared__ __align__(16) float2 s_rt[];
  const int ix = 2 * blockIdx.x, l = blockIdx.y, two = ix + 1 < Nx;
  const float* __restrict__ xa = x + ((size_t)l * Nx + ix) * Ny;
  const float* __restrict__ xb = xa + (two ? Ny : 0);
  const float sa = 0.5f * sx[ix], sb = two ? 0.5f * sx[ix + 1] : 0.f;
  float2* __restrict__ out = Z + ((size_t)l * gridDim.x + blockIdx.x) * N;
  auto load = [&](int, int, int, int n) {
    return n < Ny ? make_float2(xa[n] * sy[n] * sa, two ? xb[n] * sy[n] * sb : 0.f) : make_float2(0.f, 0.f);
  };
  auto store = [&](int, int, int, int n, float2 v) { out[n] = v; };
  fft_rt<PT, false>(s_rt, tw, N, 1, blockDim.x, load, store);
}

template <int PT>
__global__ __launch_bounds__(1024) void k_adj_y_rt(const float2* __restrict__ U, const float* __restrict__ sy,
                                                   const float* __restrict__ sx, int Ny, int Nx, int N,
                                                   const float2* __restrict__ tw, const float* __restrict__ scale,
                                                   float* __restrict__ out) {
  extern __shared__ __align__(16) float2 s_rt[];
  const int ix = 2 * blockIdx.x, l = blockIdx.y, hs = half_stride(N);
  const bool two = ix + 1 < Nx;
  const float2* __restrict__ ua = U + ((size_t)l * Nx + ix) * hs;
  const float2* __restrict__ ub = two ? ua + hs : nullptr;
  const float sc = 0.5f * (scale ? scale[l] : 1.f), sa = sc * sx[ix], sb = two ? sc * sx[ix + 1] : 0.f;
  float* __restrict__ o = out + ((size_t)l * Nx + ix) * Ny;
  auto load = [&](int, int, int, int n) { return join_pair(ua, ub, N, n); };
  auto store = [&](int, int, int, int n, float2 v) {
    if (n < Ny) {
      o[n] = sa * sy[n] * v.x;
      if (two) o[Ny + n] = sb * sy[n] * v.y;
    }
  };
  fft_rt<PT, true>(s_rt, tw, N, 1, blockDim.x, load, store);
}

template <int PT>
__global__ __launch_bounds__(1024) void k_fwd_x_rt(const float2* __restrict__ Z, int Kty, int Nx, int N, int B,
                                                   const float2* __restrict__ tw, float2* __restrict__ Fx) {
  extern __shared__ __align__(16) float2 s_rt[];
  const int ky0 = xpass_eighth_row0(B), l = blockIdx.y;
  if (2 * ky0 > Kty) return;
  const float2* __restrict__ Zl = Z + (size_t)l * ((Nx + 1) / 2) * Kty;
  float2* __restrict__ F = Fx + (size_t)l * N * Kty;
  auto load = [&](int, int, int b, int n) {
    const int ky = ky0 + b;
    if (n >= Nx || 2 * ky > Kty) return make_float2(0.f, 0.f);
    const float2* __restrict__ zp = Zl + (size_t)(n >> 1) * Kty;
    float2 a, c;
    split_pair(zp[ky], zp[ky ? Kty - ky : 0], a, c);
    return n & 1 ? c : a;
  };
  auto store = [&](int, int, int b, int n, float2 v) {
    const int ky = ky0 + b;
    if (2 * ky > Kty) return;
    F[(size_t)n * Kty + ky] = v;
    if (ky && 2 * ky < Kty) F[(size_t)(n ? N - n : 0) * Kty + Kty - ky] = make_float2(v.x, -v.y);
  };
  fft_rt<PT, false>(s_rt, tw, N, B, blockDim.x, load, store);
}

template <int PT>
__global__ __launch_bounds__(1024) void k_adj_x_rt(const float2* __restrict__ g, int Kty, int Nx, int N, int B,
                                                   const float2* __restrict__ tw, float2* __restrict__ U) {
  extern __shared__ __align__(16) float2 s_rt[];
  const int ky0 = xpass_eighth_row0(B), l = blockIdx.y, hs = half_stride(Kty);
  if (2 * ky0 > Kty) return;
  const float2* __restrict__ gl = g + (size_t)l * N * Kty;
  float2* __restrict__ Ul = U + (size_t)l * Nx * hs;
  auto load = [&](int, int, int b, int n) {
    const int ky = ky0 + b;
    if (2 * ky > Kty) return make_float2(0.f, 0.f);
    return hermitian(gl[(size_t)n * Kty + ky], gl[(size_t)(n ? N - n : 0) * Kty + (ky ? Kty - ky : 0)]);
  };
  auto store = [&](int, int, int b, int n, float2 v) {
    const int ky = ky0 + b;
    if (n < Nx && 2 * ky <= Kty) Ul[(size_t)n * hs + ky] = v;
  };
  fft_rt<PT, true>(s_rt, tw, N, B, blockDim.x, load, store);
}

void fwd_y_any(fhs_ctx* ctx, const fhs_nufft* p, int L, const float* x, float2* T) {
  if (is_pow2_grid(p->Kty)) {
    dispatch_pow2<RunFwdY>(p->Kty, ctx->stream, p->Nx, L, x, p, T);
    return;
  }
  const size_t lds = fft_rt_lds(p->Kty, 1);
  with_values(fft_rt_values(p->Kty, 1), [&](auto v) {
    constexpr int PT = decltype(v)::value;
    allow_dynamic_lds((const void*)k_fwd_y_rt<PT>, lds);
    k_fwd_y_rt<PT><<<dim3((p->Nx + 1) / 2, L), fft_rt_threads(p->Kty, 1), lds, ctx->stream>>>(
        x, p->sy, p->sx, p->Ny, p->Nx, p->Kty, p->twy, T);
  });
}

void adj_y_any(fhs_ctx* ctx, const fhs_nufft* p, int L, const float2* T, const float* scale, float* out) {
  if (is_pow2_grid(p->Kty)) {
    dispatch_pow2<RunAdjY>(p->Kty, ctx->stream, p->Nx, L, T, p, scale, out);
    return;
  }
  const size_t lds = fft_rt_lds(p->Kty, 1);
  with_values(fft_rt_values(p->Kty, 1), [&](auto v) {
    constexpr int PT = decltype(v)::value;
    allow_dynamic_lds((const void*)k_adj_y_rt<PT>, lds);
    k_adj_y_rt<PT><<<dim3((p->Nx + 1) / 2, L), fft_rt_threads(p->Kty, 1), lds, ctx->stream>>>(
        T, p->sy, p->sx, p->Ny, p->Nx, p->Kty, p->twy, scale, out);
  });
}

void fwd_x_any(fhs_ctx* ctx, const fhs_nufft* p, int L, const float2* T, float2* F) {
  if (is_pow2_grid(p->Ktx)) {
    dispatch_pow2<RunFwdX>(p->Ktx, ctx, p->Kty, L, T, p, F);
    return;
  }
  const int B = fft_rt_rows(p->Ktx, p->Kty / 2 + 1, L);
  const size_t lds = fft_rt_lds(p->Ktx, B);
  with_values(fft_rt_values(p->Ktx, B), [&](auto v) {
    constexpr int PT = decltype(v)::value;
    allow_dynamic_lds((const void*)k_fwd_x_rt<PT>, lds);
    k_fwd_x_rt<PT><<<dim3(xpass_eighth_grid(p->Kty / 2 + 1, B), L), fft_rt_threads(p->Ktx, B), lds, ctx->stream>>>(
        T, p->Kty, p->Nx, p->Ktx, B, p->twx, F);
  });
}

void adj_x_any(fhs_ctx* ctx, const fhs_nufft* p, int L, const float2* g, float2* T) {
  if (is_pow2_grid(p->Ktx)) {
    dispatch_pow2<RunAdjX>(p->Ktx, ctx, p->Kty, L, g, p, T);
    return;
  }
  const int B = fft_rt_rows(p->Ktx, p->Kty / 2 + 1, L);
  const size_t lds = fft_rt_lds(p->Ktx, B);
  with_values(fft_rt_values(p->Ktx, B), [&](auto v) {
    constexpr int PT = decltype(v)::value;
    allow_dynamic_lds((const void*)k_adj_x_rt<PT>, lds);
    k_adj_x_rt<PT><<<dim3(xpass_eighth_grid(p->Kty / 2 + 1, B), L), fft_rt_threads(p->Ktx, B), lds, ctx->stream>>>(
        g, p->Kty, p->Nx, p->Ktx, B, p->twx, T);
  });
}

// Z of the forward, U of the adjoint transform, in either of its forms
float2* nufft_workspace(fhs_ctx* ctx, const fhs_nufft* p, int L) {
  const size_t z = (size_t)((p->Nx + 1) / 2) * p->Kty;
  const size_t u = (size_t)p->Nx * (adj_half(p, L) ? half_stride(p->Kty) : p->Kty);
  return (float2*)ctx->ws.get("nufft_T", L * std::max(z, u) * sizeof(float2));
}

}  // namespace

// Used by the fused data-fidelity step.
void nufft_forward(fhs_ctx* ctx, const fhs_nufft* p, const float* x, int L, float2* Fx) {
  float2* T = nufft_workspace(ctx, p, L);
  {
    Scope sc(ctx, "fft_fwd_y");
    fwd_y_any(ctx, p, L, x, T);
    check_launch();
  }
  {
    Scope sc(ctx, "fft_fwd_x");
    fwd_x_any(ctx, p, L, (const float2*)T, Fx);
    check_launch();
  }
}

void nufft_adjoint(fhs_ctx* ctx, const fhs_nufft* p, const float2* g, int L, const float* scale_dev,
                   float* out) {
  float2* T = nufft_workspace(ctx, p, L);
  {
    Scope sc(ctx, "fft_adj_x");
    adj_x_any(ctx, p, L, g, T);
    check_launch();
  }
  {
    Scope sc(ctx, "fft_adj_y");
    adj_y_any(ctx, p, L, (const float2*)T, scale_dev, out);
    check_launch();
  }
}

}  // namespace fhs

using namespace fhs;

extern "C" {

int fhs_nufft_create_host(fhs_ctx* ctx, int Ny, int Nx, int Kty, int Ktx, const double* sy,
                          const double* sx, fhs_nufft** out) {
  if (!ctx || !out) return FHS_ERR_ARG;
  *out = nullptr;
  return guard(ctx, [&] {
    auto smooth = [](int n) {   // 2^a 3^b 5^c in [16, 8192]
      if (n < 16 || n > 8192) return false;
      for (int f : {2, 3, 5})
        while (n % f == 0) n /= f;
      return n == 1;
    };
    FHS_CHECK(smooth(Kty) && smooth(Ktx), "nufft_create: Kty, Ktx must be of the form 2^a 3^b 5^c in [16, 8192]");
    FHS_CHECK(Ny >= 1 && Nx >= 1 && Ny <= Kty && Nx <= Ktx, "nufft_create: image larger than grid");
    FHS_HIP(hipSetDevice(ctx->device));
    fhs_nufft* p = new fhs_nufft();
    p->device = ctx->device;
    p->Ny = Ny;
    p->Nx = Nx;
    p->Kty = Kty;
    p->Ktx = Ktx;
    std::vector<float> hy(sy, sy + Ny), hx(sx, sx + Nx);
    FHS_HIP(hipMalloc(&p->sy, Ny * sizeof(float)));
    FHS_HIP(hipMalloc(&p->sx, Nx * sizeof(float)));
    FHS_HIP(hipMemcpy(p->sy, hy.data(), Ny * sizeof(float), hipMemcpyHostToDevice));
    FHS_HIP(hipMemcpy(p->sx, hx.data(), Nx * sizeof(float), hipMemcpyHostToDevice));
    p->twy = twiddles(Kty);
    p->twx = twiddles(Ktx);
    *out = p;
  });
}

int fhs_nufft_info(const fhs_nufft* p, int* Ny, int* Nx, int* Kty, int* Ktx) {
  if (!p) return FHS_ERR_ARG;
  if (Ny) *Ny = p->Ny;
  if (Nx) *Nx = p->Nx;
  if (Kty) *Kty = p->Kty;
  if (Ktx) *Ktx = p->Ktx;
  return FHS_OK;
}

int fhs_nufft_destroy(fhs_nufft* p) {
  if (!p) return FHS_OK;
  (void)hipSetDevice(p->device);
  (void)hipFree(p->sy);
  (void)hipFree(p->sx);
  (void)hipFree(p->twy);
  (void)hipFree(p->twx);
  delete p;
  return FHS_OK;
}

int fhs_apply_scaled_fourier_transform(fhs_ctx* ctx, const fhs_nufft* p, const float* x, int L,
                                       void* Fx) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(p && x && Fx && L >= 1 && L <= 65535, "apply_scaled_fourier_transform: bad argument");
    nufft_forward(ctx, p, x, L, (float2*)Fx);
  });
}

int fhs_apply_scaled_fourier_adjoint(fhs_ctx* ctx, const fhs_nufft* p, const void* g, int L,
                                     const float* scale, float* out) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(p && g && out && L >= 1 && L <= 65535, "apply_scaled_fourier_adjoint: bad argument");
    float* sd = nullptr;
    if (scale) {
      sd = (float*)ctx->ws.get("nufft_scale", L * sizeof(float));
      FHS_HIP(hipMemcpyAsync(sd, scale, L * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
    }
    nufft_adjoint(ctx, p, (const float2*)g, L, sd, out);
  });
}

}  // extern "C"
