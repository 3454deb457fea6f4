// SARA dictionary on the GPU: Psit (analysis) and Psi (synthesis, exact
// adjoint) of db1..db8 + Dirac with 'zpd' extension, batched over bases and
// channels, and the weighted l21 dual step.
//
// Coefficient vector of one channel (length s, MATLAB wavedec2 order per
// basis, bases in order, Dirac last), each basis scaled by 1/sqrt(P):
//   [ A_J H_J V_J D_J H_{J-1} ... D_1 ]_db1 ... [ ... ]_dbK [ x(:) ]_dirac
// One zpd analysis step along an axis with reconstruction filter f (length
// lf): out[k] = sum_j f[j] in[2k + 2 - lf + j], n_out = floor((n + lf - 1)/2).
// a = lo_y lo_x, h = hi_y lo_x, v = lo_y hi_x, d = hi_y hi_x (y = rows).
//
// Both directions run one wave per tile on registers and LDS of its own (see
// k_analysis and k_synthesis); the l21 step is part of the analysis.
#include <algorithm>
#include <cmath>
#include <memory>

#include "common.hpp"
#include "kernels.hpp"

namespace fhs {

constexpr int WMAX_BASES = 8;
constexpr int WMAX_LEVELS = 6;
constexpr int WMAX_LF = 16;

struct SaraGeom {
  int Ny, Nx, nlevel, nb, dirac;
  float norm;                            // 1/sqrt(P)
  int lf[WMAX_BASES];
  int ny[WMAX_BASES][WMAX_LEVELS + 1];   // level shapes, [0] = image
  int nx[WMAX_BASES][WMAX_LEVELS + 1];
  int64_t boff[WMAX_BASES + 1];          // basis offsets in a channel vector; boff[nb] = dirac
  int64_t aoff[WMAX_BASES];              // A_J offset inside basis (= 0)
  int64_t doff[WMAX_BASES][WMAX_LEVELS + 1];  // offset of H_k (V, D follow) inside basis
  int64_t scr[WMAX_BASES][WMAX_LEVELS + 1];   // scratch offset of approx level k (per channel)
  int64_t scr_per_chan;
  int64_t s;                             // coefficients per channel
  float lo[WMAX_BASES][WMAX_LF];         // reconstruction low-pass; high-pass (-1)^j lo[lf - 1 - j]
};

// What a launch on one level reads of it, by value: a launch or a captured graph
// then needs the dictionary no more.  A workgroup's share is the few fields in
// front and the 120 bytes of its basis, two or three lines of the arguments: as
// fast as a copy in device memory (dual step of 128 x 128 67 us, 1024 x 1024 x 16
// 925 against 940), where the whole geometry by value, 2 KB with every field of a
// basis in another line, took 1.2 us more a launch (73 us).
struct SaraLevel {
  int lf;                 // taps
  int ny, nx, py, px;     // shapes of levels k and k - 1
  int64_t hoff;           // H_k (V_k, D_k follow) in a channel's coefficients
  int64_t aoff;           // A_J
  int64_t fine, coarse;   // scratch offsets of the approximations of levels k - 1 and k
  float lo[WMAX_LF];
};
struct SaraArgs {
  int Ny, Nx, nlevel, nb, dirac, k;
  float norm;
  int64_t s, scr_per_chan, dstart;
  SaraLevel b[WMAX_BASES];
};

SaraArgs level_args(const SaraGeom& G, int k) {
  SaraArgs A{};
  A.Ny = G.Ny;
  A.Nx = G.Nx;
  A.nlevel = G.nlevel;
  A.nb = G.nb;
  A.dirac = G.dirac;
  A.k = k;
  A.norm = G.norm;
  A.s = G.s;
  A.scr_per_chan = G.scr_per_chan;
  A.dstart = G.boff[G.nb];
  for (int b = 0; b < G.nb; ++b) {
    SaraLevel& B = A.b[b];
    B.lf = G.lf[b];
    B.ny = G.ny[b][k];
    B.nx = G.nx[b][k];
    B.py = G.ny[b][k - 1];
    B.px = G.nx[b][k - 1];
    B.hoff = G.boff[b] + G.doff[b][k];
    B.aoff = G.boff[b] + G.aoff[b];
    B.fine = G.scr[b][k - 1];
    B.coarse = G.scr[b][k];
    for (int j = 0; j < B.lf; ++j) B.lo[j] = G.lo[b][j];
  }
  return A;
}

}  // namespace fhs

struct fhs_sara {
  fhs::SaraGeom g{};
  fhs::SaraArgs level[fhs::WMAX_LEVELS + 1];   // [k], k = 1 .. nlevel
};

namespace fhs {
namespace {

// ---- analysis -----------------------------------------------------------------
// One wave transforms one tile of AT_Y x AT_X outputs of a level, basis and
// channel.  Its input window has at most 2 AT_Y + 14 = 126 rows: lane r reads the
// 2 AT_X + lf - 2 values of rows r and r + 64 along x straight from memory, 64
// consecutive floats a load, so the x filter runs on registers (an earlier form
// staged the window in LDS and read every tap of every output from there).  The
// two x-filtered halves turn through LDS of the wave's own, even and odd rows
// apart, and lane ky filters along y; its accesses to v1 are again 56
// consecutive floats.  A workgroup's waves hold the channels of one tile, so the
// norms of the l21 step over the channels close inside it: analysis, threshold
// and dual update read and write v1 once, not twice.  One channel a wave, and one
// column address per array with the columns as lane offsets: four channels a wave
// and an address per column spilled 200 scalar registers into lanes, which
// doubled the instructions (level 1 of 16 channels of 1024 x 1024: 508 us, 411 us
// in this form).  What bounds it there: 1024-thread workgroups of 80 registers, one
// on a CU, whose load and filter phases do not overlap.
constexpr int AT_Y = 56, AT_X = 4;
constexpr int AT_LD = 96;                 // LDS stride of the 63 rows of a parity: even and odd rows in other banks
constexpr int AT_PAIR = 2;                // columns in the turning tile at a time
constexpr int AT_LH = 4 * AT_PAIR * AT_LD;   // floats of a wave's turning tile
constexpr int AN_CHANNELS = 16;           // waves of a workgroup at most

// hi[j] = (-1)^j lo[lf - 1 - j]: one set of taps in scalar registers serves both
// filters
template <int LF>
struct Taps {
  float f[LF];
  __device__ __forceinline__ float lo(int j) const { return f[j]; }
  __device__ __forceinline__ float hi(int j) const { return j & 1 ? -f[LF - 1 - j] : f[LF - 1 - j]; }
};
template <int LF>
__device__ __forceinline__ Taps<LF> load_taps(const SaraLevel& G) {
  Taps<LF> t;
#pragma unroll
  for (int j = 0; j < LF; ++j) t.f[j] = G.lo[j];
  return t;
}
// element `off` bytes behind a wave-uniform base
__device__ __forceinline__ float& at_bytes(float* base, unsigned off) {
  return *reinterpret_cast<float*>(reinterpret_cast<char*>(base) + off);
}
__device__ __forceinline__ float at_bytes(const float* base, unsigned off) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + off);
}

// what becomes of the coefficients c
enum AnMode {
  AN_ADD = 0,      // v1 += c
  AN_SET = 1,      // v1 = c
  AN_L21 = 2,      // r = v1 + c over the channels, v1 = r - max(|r| - beta w, 0) / (|r| + eps) r
  AN_WEIGHT = 3,   // wout = beta / (beta + |c|)
  AN_NORM = 4      // part[workgroup] = sum of |c|
};

struct AnArgs {
  const float* x;        // image cube, the input of level 1
  float* scr;            // A_1 .. A_{J-1} of the bases and channels
  float* v1;
  const float* w;
  double beta;
  float* wout;
  double* part;
  int L;
};

// the l21 factor of a coefficient with norm sqrt(ss): v1 = r - f r
__device__ __forceinline__ float l21_factor(double ss, double t) {
  const double l2 = sqrt(ss);
  return (float)(fmax(l2 - t, 0.0) / (l2 + 2.220446049250313e-16));
}

template <int LF, int MODE, bool LAST>
__device__ __forceinline__ void an_tile(const SaraArgs& G, const SaraLevel& B, const AnArgs& A, int ky0, int kx0, float* lds) {
  constexpr int NS = LAST ? 4 : 3;        // subbands kept as coefficients: h, v, d (and a)
  constexpr int NQ = NS * AT_X;           // coefficients per lane
  constexpr int WW = 2 * AT_X + LF - 2;   // window columns
  constexpr bool NORMS = MODE >= AN_L21;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave = channel
  const int l = NORMS ? wv : (int)(blockIdx.y * (blockDim.x >> 6)) + wv;
  if (!NORMS && l >= A.L) return;
  const int k = G.k, iny = B.py, inx = B.px, ny = B.ny, nx = B.nx;
  const int64_t sz = (int64_t)ny * nx;
  const Taps<LF> T = load_taps<LF>(B);
  const bool live = lane < AT_Y && ky0 + lane < ny;
  const int ncol = min(AT_X, nx - kx0);
  // offsets of the kept subbands in a channel vector, of the tile, of this lane
  const int64_t hoff = B.hoff, toff = ky0 + (int64_t)ny * kx0;
  auto soff = [&](int s) { return s == 3 ? B.aoff : hoff + s * sz; };
  const unsigned loff = (unsigned)lane * sizeof(float), cstep = (unsigned)ny * sizeof(float);
  float* v1 = A.v1 + (int64_t)l * G.s + toff;
  // r: old coefficients, then plus the new ones (r[3]: the approximation, a coefficient
  // only at the last level)
  float r[4][AT_X];
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int q = 0; q < AT_X; ++q) r[s][q] = 0.f;
  if ((MODE == AN_ADD || MODE == AN_L21) && live) {
#pragma unroll
    for (int q = 0; q < AT_X; ++q)
      if (q < ncol) {
#pragma unroll
        for (int s = 0; s < NS; ++s) r[s][q] = at_bytes(v1 + soff(s), loff + q * cstep);
      }
  }
  float wc = 1.f;   // the threshold weight of the coefficient this thread finishes below
  auto coef = [&](int e, int64_t& c) {
    const int i = e >> 6, ln = e & 63, s = i / AT_X, q = i % AT_X;
    c = soff(s) + toff + (int64_t)ny * q + ln;
    return q < ncol && ln < AT_Y && ky0 + ln < ny;
  };
  if (MODE == AN_L21 && A.w) {
    int64_t c;
    if (threadIdx.x < NQ * 64 && coef(threadIdx.x, c)) wc = A.w[c];
  }
  // x filter of rows lane and lane + 64
  float lw[2][AT_X], hg[2][AT_X];
  {
    const int wy0 = 2 * ky0 + 2 - LF, wx0 = 2 * kx0 + 2 - LF;
    const float* img = (k == 1 ? A.x + (int64_t)l * iny * inx : A.scr + (int64_t)l * G.scr_per_chan + B.fine) +
                       (int64_t)iny * wx0;
    const float scale = k == 1 ? G.norm : 1.f;
    const bool inside = wx0 >= 0 && wx0 + WW <= inx;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int row = lane + 64 * hh, wy = wy0 + row;
      const unsigned off = (unsigned)wy * sizeof(float), step = (unsigned)iny * sizeof(float);
      float win[WW];
#pragma unroll
      for (int c = 0; c < WW; ++c) win[c] = 0.f;
      if (wy >= 0 && wy < iny && row < 2 * AT_Y + LF - 2) {
        if (inside) {
#pragma unroll
          for (int c = 0; c < WW; ++c) win[c] = at_bytes(img, off + c * step);
        } else {
#pragma unroll
          for (int c = 0; c < WW; ++c)
            if (wx0 + c >= 0 && wx0 + c < inx) win[c] = at_bytes(img, off + c * step);
        }
      }
#pragma unroll
      for (int q = 0; q < AT_X; ++q) {
        float sl = 0.f, sh = 0.f;
#pragma unroll
        for (int j = 0; j < LF; ++j) {
          sl += T.lo(j) * win[2 * q + j];
          sh += T.hi(j) * win[2 * q + j];
        }
        lw[hh][q] = sl * scale;
        hg[hh][q] = sh * scale;
      }
    }
  }
  // y filter, AT_PAIR columns at a time: output ky0 + lane from rows 2 lane .. 2 lane + LF - 1
  float* lh = lds + wv * AT_LH;
  float* dst = lh + (lane & 1) * AT_LD + (lane >> 1);   // row lane; row lane + 64 is 32 further
  const float* src = lh + min(lane, AT_Y - 1);
#pragma unroll
  for (int q0 = 0; q0 < AT_X; q0 += AT_PAIR) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < AT_PAIR; ++q)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        dst[(4 * q) * AT_LD + 32 * hh] = lw[hh][q0 + q];
        dst[(4 * q + 2) * AT_LD + 32 * hh] = hg[hh][q0 + q];
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < AT_PAIR; ++q) {
      float a = 0.f, h = 0.f, v = 0.f, d = 0.f;
#pragma unroll
      for (int j = 0; j < LF; ++j) {
        const float xl = src[(4 * q + (j & 1)) * AT_LD + j / 2], xh = src[(4 * q + 2 + (j & 1)) * AT_LD + j / 2];
        a += T.lo(j) * xl;
        h += T.hi(j) * xl;
        v += T.lo(j) * xh;
        d += T.hi(j) * xh;
      }
      r[0][q0 + q] += h;
      r[1][q0 + q] += v;
      r[2][q0 + q] += d;
      r[3][q0 + q] += a;
      // the sums are made here: sunk into the masked stores below, they would keep every
      // tap's input in registers (and spill)
#pragma unroll
      for (int s = 0; s < 4; ++s) asm volatile("" : "+v"(r[s][q0 + q]));
    }
  }
  if (!LAST && live) {
    float* ak = A.scr + (int64_t)l * G.scr_per_chan + B.coarse + toff;
#pragma unroll
    for (int q = 0; q < AT_X; ++q)
      if (q < ncol) at_bytes(ak, loff + q * cstep) = r[3][q];
  }
  auto put = [&](auto value) {
    if (live) {
#pragma unroll
      for (int q = 0; q < AT_X; ++q)
        if (q < ncol) {
#pragma unroll
          for (int s = 0; s < NS; ++s) at_bytes(v1 + soff(s), loff + q * cstep) = value(s, q);
        }
    }
  };
  if constexpr (!NORMS) {
    put([&](int s, int q) { return r[s][q]; });
  } else {
    // the channels' values meet in LDS (the turning tiles are done with once every
    // wave has arrived); thread t finishes coefficients t, t + blockDim, ...
    const int nw = blockDim.x >> 6;
    float* vals = lds;                       // [channel][coefficient][lane]
    float* fac = lds + nw * NQ * 64;
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int q = 0; q < AT_X; ++q) vals[(wv * NQ + s * AT_X + q) * 64 + lane] = r[s][q];
    __syncthreads();
    double tot[1] = {0.0};
    for (int e = threadIdx.x; e < NQ * 64; e += blockDim.x) {
      int64_t c;
      if (!coef(e, c)) continue;
      if (MODE == AN_L21 && A.w && e >= (int)blockDim.x) wc = A.w[c];
      double sq = 0.0;
      for (int u = 0; u < nw; ++u) {
        const double t = vals[u * NQ * 64 + e];
        sq += t * t;
      }
      if constexpr (MODE == AN_L21) fac[e] = l21_factor(sq, A.beta * (double)wc);
      if constexpr (MODE == AN_WEIGHT) A.wout[c] = (float)(A.beta / (A.beta + sqrt(sq)));
      if constexpr (MODE == AN_NORM) tot[0] += sqrt(sq);
    }
    if constexpr (MODE == AN_NORM) {
      __syncthreads();
      block_sum<1>(tot, reinterpret_cast<double*>(lds));
      if (threadIdx.x == 0) A.part[blockIdx.x] = tot[0];
    }
    if constexpr (MODE == AN_L21) {
      __syncthreads();
      put([&](int s, int q) { return r[s][q] - fac[(s * AT_X + q) * 64 + lane] * r[s][q]; });
    }
  }
}

// Workgroup -> (tile, basis).  The XCDs take contiguous runs of tiles (y
// fastest), each tile's bases one after the other, so the image window the
// bases share and the lines two tiles of a column share meet in one L2.
template <int MODE, bool LAST>
__global__ __launch_bounds__(64 * AN_CHANNELS) void k_analysis(SaraArgs G, AnArgs A, int ty, int tx) {
  extern __shared__ __align__(16) float an_lds[];
  const int per = (ty * tx + 7) / 8, s = blockIdx.x / 8;
  const int tile = (int)(blockIdx.x % 8) * per + s / G.nb, b = s % G.nb;
  const int ky0 = (tile % ty) * AT_Y, kx0 = (tile / ty) * AT_X;
  if (s / G.nb >= per || ky0 >= G.b[b].ny || kx0 >= G.b[b].nx) {
    if (MODE == AN_NORM && threadIdx.x == 0) A.part[blockIdx.x] = 0.0;
    return;
  }
  switch (G.b[b].lf) {   // db1 .. db8: 2, 4, ..., 16 taps
    case 2: an_tile<2, MODE, LAST>(G, G.b[b], A, ky0, kx0, an_lds); break;
    case 4: an_tile<4, MODE, LAST>(G, G.b[b], A, ky0, kx0, an_lds); break;
    case 6: an_tile<6, MODE, LAST>(G, G.b[b], A, ky0, kx0, an_lds); break;
    case 8: an_tile<8, MODE, LAST>(G, G.b[b], A, ky0, kx0, an_lds); break;
    case 10: an_tile<10, MODE, LAST>(G, G.b[b], A, ky0, kx0, an_lds); break;
    case 12: an_tile<12, MODE, LAST>(G, G.b[b], A, ky0, kx0, an_lds); break;
    case 14: an_tile<14, MODE, LAST>(G, G.b[b], A, ky0, kx0, an_lds); break;
    default: an_tile<16, MODE, LAST>(G, G.b[b], A, ky0, kx0, an_lds); break;
  }
}

// The Dirac block: r_l = v1_l + x_l / sqrt(P) (v1 absent in AN_WEIGHT, AN_NORM and
// AN_SET), then as the modes say, for the 16 channels from 16 blockIdx.y.  VEC consecutive pixels per thread with wide
// accesses when the block is 16-byte aligned in every channel.
template <int MODE, int VEC>
__global__ __launch_bounds__(256) void k_dirac(SaraGeom G, const float* __restrict__ x, float* __restrict__ v1, int L,
                                               const float* __restrict__ w, double beta, float* __restrict__ wout,
                                               double* __restrict__ part) {
  struct alignas(4 * VEC) Vec {
    float v[VEC];
  };
  constexpr bool KEEP = MODE == AN_ADD || MODE == AN_L21;
  __shared__ double sh[256 / 64];
  const int64_t N = (int64_t)G.Ny * G.Nx, d0 = G.boff[G.nb];
  x += (int64_t)blockIdx.y * AN_CHANNELS * N;
  if (KEEP || MODE == AN_SET) v1 += (int64_t)blockIdx.y * AN_CHANNELS * G.s;
  L = min(L - (int)blockIdx.y * AN_CHANNELS, AN_CHANNELS);
  double tot[1] = {0.0};
  for (int64_t p = VEC * (blockIdx.x * (int64_t)blockDim.x + threadIdx.x); p < N;
       p += VEC * (int64_t)gridDim.x * blockDim.x) {
    constexpr int LREG = AN_CHANNELS;   // channels kept in registers between the norm and the update
    Vec r[LREG];
    double ss[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) ss[j] = 0.0;
#pragma unroll
    for (int l = 0; l < LREG; ++l)
      if (l < L) {
        r[l] = *reinterpret_cast<const Vec*>(x + (int64_t)l * N + p);
        Vec old;
        if (KEEP) old = *reinterpret_cast<const Vec*>(v1 + (int64_t)l * G.s + d0 + p);
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
          r[l].v[j] = KEEP ? old.v[j] + r[l].v[j] * G.norm : r[l].v[j] * G.norm;
          ss[j] += (double)r[l].v[j] * r[l].v[j];
        }
      }
    float f[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      f[j] = 0.f;
      if (MODE == AN_L21) f[j] = l21_factor(ss[j], beta * (w ? (double)w[d0 + p + j] : 1.0));
      if (MODE == AN_WEIGHT) wout[d0 + p + j] = (float)(beta / (beta + sqrt(ss[j])));
      if (MODE == AN_NORM) tot[0] += sqrt(ss[j]);
    }
    if (MODE <= AN_L21) {
#pragma unroll
      for (int l = 0; l < LREG; ++l)
        if (l < L) {
#pragma unroll
          for (int j = 0; j < VEC; ++j)
            if (MODE == AN_L21) r[l].v[j] -= f[j] * r[l].v[j];
          *reinterpret_cast<Vec*>(v1 + (int64_t)l * G.s + d0 + p) = r[l];
        }
    }
  }
  if (MODE == AN_NORM) {
    block_sum<1>(tot, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = tot[0];
  }
}

// ---- synthesis -------------------------------------------------------------
// One wave makes one tile of ST_Y x ST_X pixels of the finer level from the four
// subbands of level k.  Output i takes the lf / 2 coefficients floor(i / 2) + m with
// filter tap (i & 1) + lf - 2 - 2 m, so both pixels of a parity pair share their
// coefficients.  Lane r holds coefficient row r of the tile (at most 56 + 7) and
// reads the 3 + lf / 2 columns of each subband straight from memory, 64 consecutive
// floats a load; the x filter runs on those registers (finest level of 16 channels
// of 1024 x 1024: 410 us staged, 201 us).  The two half-filtered images turn through LDS of the wave's own and lane (ix, g) filters along y the
// 14 rows 14 g .. 14 g + 13 of column ix, keeping the sum over the bases in
// registers at the finest level (the image is written once).  No barrier: an
// earlier form staged 32 x 32 tiles in LDS, whose column segments of 18 to 25
// coefficients used half of the lines they touched.
constexpr int ST_Y = 112, ST_X = 8;
constexpr int ST_WAVES = 4;                       // tiles per workgroup
constexpr int ST_PER = ST_Y * ST_X / 64;          // pixels per lane
constexpr int ST_LD = 66;
// A tile's bases run one after the other; below this many tiles x channels the chip
// is not full and the four waves of a workgroup share a tile's bases instead (whole
// synthesis, tiles' bases in sequence -> split, us: 96 tiles 35 -> 24, 768 36 -> 27, 1280
// 45 -> 37, 1920 48 -> 43; beyond the line 2560 tiles 51 -> 47, 3840 64 -> 62, 5120 75 -> 76).
constexpr int64_t SYN_SPLIT_BELOW = 2048;

struct SynIn {
  const float* a;   // approx of level k (column-major ny x nx)
  const float* h;   // H_k, V_k = h + sz, D_k = h + 2 sz
  int ny, nx;
};

template <int LF>
__device__ __forceinline__ void syn_tile(const SaraLevel& B, const SynIn& in, int iy0, int ix0, float* pq,
                                         float* acc) {
  constexpr int NC = ST_X / 2 + LF / 2 - 1;
  const int lane = threadIdx.x & 63;
  const Taps<LF> T = load_taps<LF>(B);
  const int cy = iy0 / 2 + lane, cx0 = ix0 / 2;
  const int64_t sz = (int64_t)in.ny * in.nx, toff = (int64_t)in.ny * cx0;
  const float *ba = in.a + toff, *bh = in.h + toff, *bv = bh + sz, *bd = bv + sz;
  const unsigned off = (unsigned)cy * sizeof(float), step = (unsigned)in.ny * sizeof(float);
  float a[NC], h[NC], v[NC], d[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) a[c] = h[c] = v[c] = d[c] = 0.f;
  if (cy < in.ny && lane < ST_Y / 2 + LF / 2 - 1) {
    if (cx0 + NC <= in.nx) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        a[c] = at_bytes(ba, off + c * step);
        h[c] = at_bytes(bh, off + c * step);
        v[c] = at_bytes(bv, off + c * step);
        d[c] = at_bytes(bd, off + c * step);
      }
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (cx0 + c < in.nx) {
          a[c] = at_bytes(ba, off + c * step);
          h[c] = at_bytes(bh, off + c * step);
          v[c] = at_bytes(bv, off + c * step);
          d[c] = at_bytes(bd, off + c * step);
        }
    }
  }
  // x filter: P = lo a + hi v (low along y), Q = lo h + hi d (high along y)
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int u = 0; u < ST_X / 2; ++u) {
    float pe = 0.f, po = 0.f, qe = 0.f, qo = 0.f;
#pragma unroll
    for (int m = 0; m < LF / 2; ++m) {
      const int je = LF - 2 - 2 * m, jo = je + 1;
      pe += T.lo(je) * a[u + m] + T.hi(je) * v[u + m];
      po += T.lo(jo) * a[u + m] + T.hi(jo) * v[u + m];
      qe += T.lo(je) * h[u + m] + T.hi(je) * d[u + m];
      qo += T.lo(jo) * h[u + m] + T.hi(jo) * d[u + m];
    }
    pq[(2 * u) * ST_LD + lane] = pe;
    pq[(2 * u + 1) * ST_LD + lane] = po;
    pq[(ST_X + 2 * u) * ST_LD + lane] = qe;
    pq[(ST_X + 2 * u + 1) * ST_LD + lane] = qo;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  // y filter: the lane's 7 parity pairs
  const int ix = lane & 7, g = lane >> 3;
  constexpr int NR = ST_PER / 2 + LF / 2 - 1;
  const float* P = pq + ix * ST_LD + (ST_PER / 2) * g;
  const float* Q = P + ST_X * ST_LD;
  float pr[NR], qr[NR];
#pragma unroll
  for (int t = 0; t < NR; ++t) {
    pr[t] = P[t];
    qr[t] = Q[t];
  }
#pragma unroll
  for (int u = 0; u < ST_PER / 2; ++u) {
    float e = 0.f, o = 0.f;
#pragma unroll
    for (int m = 0; m < LF / 2; ++m) {
      const int je = LF - 2 - 2 * m, jo = je + 1;
      e += T.lo(je) * pr[u + m] + T.hi(je) * qr[u + m];
      o += T.lo(jo) * pr[u + m] + T.hi(jo) * qr[u + m];
    }
    acc[2 * u] += e;
    acc[2 * u + 1] += o;
  }
}

__device__ __forceinline__ void syn_basis(const SaraLevel& B, const SynIn& in, int iy0, int ix0, float* pq,
                                          float* acc) {
  switch (B.lf) {
    case 2: syn_tile<2>(B, in, iy0, ix0, pq, acc); break;
    case 4: syn_tile<4>(B, in, iy0, ix0, pq, acc); break;
    case 6: syn_tile<6>(B, in, iy0, ix0, pq, acc); break;
    case 8: syn_tile<8>(B, in, iy0, ix0, pq, acc); break;
    case 10: syn_tile<10>(B, in, iy0, ix0, pq, acc); break;
    case 12: syn_tile<12>(B, in, iy0, ix0, pq, acc); break;
    case 14: syn_tile<14>(B, in, iy0, ix0, pq, acc); break;
    default: syn_tile<16>(B, in, iy0, ix0, pq, acc); break;
  }
}

// One level.  FINEST: out = scale * (sum over the bases + Dirac) / sqrt(P), grid over
// (tiles, channels); otherwise A_{k-1} of one basis, grid over (tiles, bases,
// channels).  SPLIT (few tiles): the four waves of a workgroup share one tile of
// the finest level, each taking a pair of bases with the same number of taps in
// all, and add their sums in wave order.
template <bool FINEST, bool SPLIT>
__global__ __launch_bounds__(64 * ST_WAVES) void k_synthesis(SaraArgs G, int ty, int tx, int nz,
                                                             const float* __restrict__ v1, float* __restrict__ scr,
                                                             float scale, float* __restrict__ out) {
  __shared__ float lds[ST_WAVES][2 * ST_X * ST_LD];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int txg = SPLIT ? tx : (tx + ST_WAVES - 1) / ST_WAVES;
  // XCDs take contiguous runs of workgroups, x fastest: neighbours in x share columns
  const int total = ty * txg * nz, per = (total + 7) / 8;
  const int s = blockIdx.x / 8, id = (int)(blockIdx.x % 8) * per + s;
  if (s >= per || id >= total) return;
  const int z = id / (ty * txg), t = id % (ty * txg);
  const int iy0 = (t / txg) * ST_Y, ix0 = (SPLIT ? t % txg : (t % txg) * ST_WAVES + wv) * ST_X;
  const int b0 = FINEST ? 0 : z % G.nb, l = FINEST ? z : z / G.nb;
  const int py = FINEST ? G.Ny : G.b[b0].py, px = FINEST ? G.Nx : G.b[b0].px;
  if (!SPLIT && (iy0 >= py || ix0 >= px)) return;
  const float* v1l = v1 + (int64_t)l * G.s;
  float* sc = scr + (int64_t)l * G.scr_per_chan;
  float* pq = lds[wv];
  float acc[ST_PER];
#pragma unroll
  for (int q = 0; q < ST_PER; ++q) acc[q] = 0.f;
  auto one = [&](int b) {
    SynIn in;
    const SaraLevel& B = G.b[b];
    in.a = G.k == G.nlevel ? v1l + B.aoff : sc + B.coarse;
    in.h = v1l + B.hoff;
    in.ny = B.ny;
    in.nx = B.nx;
    syn_basis(B, in, iy0, ix0, pq, acc);
  };
  if constexpr (!FINEST) {
    one(b0);
  } else if constexpr (SPLIT) {
    for (int b = wv; b < G.nb; b += 2 * ST_WAVES) {
      one(b);
      const int c = b - wv + 2 * ST_WAVES - 1 - wv;
      if (c < G.nb) one(c);
    }
  } else {
    for (int b = 0; b < G.nb; ++b) one(b);
  }
  // through LDS into whole columns of ST_Y pixels
  __builtin_amdgcn_wave_barrier();
  {
    float* o = pq + (lane & 7) * ST_Y + ST_PER * (lane >> 3);
#pragma unroll
    for (int q = 0; q < ST_PER; ++q) o[q] = acc[q];
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  float* dst = FINEST ? out + (int64_t)l * G.Ny * G.Nx : sc + G.b[b0].fine;
  const float* dir = v1l + G.dstart;
  auto store = [&](int e, float v) {
    const int iy = iy0 + e % ST_Y, ix = ix0 + e / ST_Y;
    if (iy >= py || ix >= px) return;
    const int64_t p = iy + (int64_t)py * ix;
    if (FINEST) {
      v *= G.norm;
      if (G.dirac) v += dir[p] * G.norm;
      v *= scale;
    }
    dst[p] = v;
  };
  if constexpr (SPLIT) {
    __syncthreads();
    for (int e = threadIdx.x; e < ST_Y * ST_X; e += 64 * ST_WAVES)
      store(e, ((lds[0][e] + lds[1][e]) + lds[2][e]) + lds[3][e]);
  } else {
#pragma unroll
    for (int q = 0; q < ST_PER; ++q) store(q * 64 + lane, pq[q * 64 + lane]);
  }
}

// The Dirac basis alone: no tiles (8 images of 512 x 512, dual step 17.3 -> 10.5 us).
template <int VEC>
__global__ __launch_bounds__(256) void k_dirac_synthesis(SaraGeom G, const float* __restrict__ v1, float scale,
                                                         float* __restrict__ out) {
  struct alignas(4 * VEC) Vec {
    float v[VEC];
  };
  const int64_t N = (int64_t)G.Ny * G.Nx;
  v1 += blockIdx.y * G.s;
  out += blockIdx.y * N;
  for (int64_t p = VEC * (blockIdx.x * (int64_t)blockDim.x + threadIdx.x); p < N;
       p += VEC * (int64_t)gridDim.x * blockDim.x) {
    Vec r = *reinterpret_cast<const Vec*>(v1 + p);
#pragma unroll
    for (int j = 0; j < VEC; ++j) r.v[j] = r.v[j] * G.norm * scale;
    *reinterpret_cast<Vec*>(out + p) = r;
  }
}

// ---- more than 16 channels ---------------------------------------------------
// The modes over the channels from stored coefficients, Dirac block included (mode 0:
// l21 step, 1: sum of the norms, 2: weights).
__global__ __launch_bounds__(256) void k_l21(int64_t s, float* __restrict__ v1, int L,
                                             const float* __restrict__ w, double beta, int mode,
                                             float* __restrict__ wout, double* __restrict__ partial) {
  __shared__ double sh[256 / 64];
  double tot[1] = {0.0};
  for (int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; c < s;
       c += (int64_t)gridDim.x * blockDim.x) {
    constexpr int LREG = 16;   // channels kept in registers between the norm and the update
    float rv[LREG];
    double ss = 0.0;
#pragma unroll
    for (int l = 0; l < LREG; ++l) {
      if (l < L) {
        const float r = v1[(int64_t)l * s + c];
        rv[l] = r;
        ss += (double)r * r;
      }
    }
    for (int l = LREG; l < L; ++l) {
      const float r = v1[(int64_t)l * s + c];
      ss += (double)r * r;
    }
    const double l2 = sqrt(ss);
    if (mode == 1) {
      tot[0] += l2;
      continue;
    }
    if (mode == 2) {   // reweighting: w = upsilon / (upsilon + l2), beta = upsilon
      wout[c] = (float)(beta / (beta + l2));
      continue;
    }
    const double t = beta * (w ? (double)w[c] : 1.0);
    const float f = (float)(fmax(l2 - t, 0.0) / (l2 + 2.220446049250313e-16));
#pragma unroll
    for (int l = 0; l < LREG; ++l)
      if (l < L) v1[(int64_t)l * s + c] = rv[l] - f * rv[l];
    for (int l = LREG; l < L; ++l) {
      const float r = v1[(int64_t)l * s + c];
      v1[(int64_t)l * s + c] = r - f * r;
    }
  }
  if (mode == 1) {
    block_sum<1>(tot, sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot[0];
  }
}

__global__ void k_sum_l(const double* __restrict__ partial, int n, double* out) {
  __shared__ double sh[4];
  double s[1] = {0.0};
  for (int i = threadIdx.x; i < n; i += blockDim.x) s[0] += partial[i];
  block_sum<1>(s, sh);
  if (threadIdx.x == 0) *out = s[0];
}

unsigned analysis_grid(const SaraGeom& G, int k, int& ty, int& tx) {
  int ny = 0, nx = 0;
  for (int b = 0; b < G.nb; ++b) {
    ny = std::max(ny, G.ny[b][k]);
    nx = std::max(nx, G.nx[b][k]);
  }
  ty = (int)cdiv(ny, AT_Y);
  tx = (int)cdiv(nx, AT_X);
  return 8 * cdiv((long long)ty * tx, 8) * G.nb;
}

template <int MODE>
void launch_analysis(fhs_ctx* ctx, const fhs_sara* S, int k, const AnArgs& A, unsigned grid, int ty, int tx) {
  // Waves of a workgroup: all channels, or equal shares of more than AN_CHANNELS,
  // whose groups share a launch (a chain of launches per 16 channels took 186 us for
  // the analysis of 128 x 128 x 64, 70 so, and 137 -> 106 at 512 x 512 x 17).
  const unsigned groups = cdiv(A.L, AN_CHANNELS), waves = cdiv(A.L, groups);
  // LDS: the turning tiles, or every channel's coefficients and the factors
  const bool last = k == S->g.nlevel;
  const size_t nq = (last ? 4 : 3) * AT_X * 64;
  const size_t lds = std::max<size_t>(waves * AT_LH, MODE >= AN_L21 ? (waves + 1) * nq : 0) * sizeof(float);
  auto go = [&](auto kern) {
    allow_dynamic_lds((const void*)kern, lds);
    kern<<<dim3(grid, groups), 64 * waves, lds, ctx->stream>>>(S->level[k], A, ty, tx);
    check_launch();
  };
  last ? go(k_analysis<MODE, true>) : go(k_analysis<MODE, false>);
}

// All levels and the Dirac block in one mode; at most AN_CHANNELS channels for the
// modes over the channels.  Returns the number of workgroup sums (AN_NORM).
template <int MODE>
unsigned sara_analyse(fhs_ctx* ctx, const fhs_sara* S, const float* x, int L, float* v1, const float* w, double beta,
                      float* wout, double* part) {
  const SaraGeom& G = S->g;
  float* scr = (float*)ctx->ws.get("sara_scratch", std::max<int64_t>(1, G.scr_per_chan * L) * sizeof(float));
  const int64_t N = (int64_t)G.Ny * G.Nx;
  unsigned nsum = 0;
  AnArgs A;
  A.L = L;
  A.x = x;
  A.scr = scr;
  A.v1 = v1;
  A.w = w;
  A.beta = beta;
  A.wout = wout;
  for (int k = 1; k <= G.nlevel && G.nb > 0; ++k) {
    int ty, tx;
    const unsigned grid = analysis_grid(G, k, ty, tx);
    A.part = part ? part + nsum : nullptr;
    launch_analysis<MODE>(ctx, S, k, A, grid, ty, tx);
    nsum += grid;
  }
  if (G.dirac) {
    const bool vec = N % 4 == 0 && (uintptr_t)x % 16 == 0 &&
                     (MODE > AN_L21 || (G.s % 4 == 0 && G.boff[G.nb] % 4 == 0 && (uintptr_t)v1 % 16 == 0));
    const unsigned grid = std::min<unsigned>(2048, cdiv(vec ? N / 4 : N, 256));
    (vec ? k_dirac<MODE, 4> : k_dirac<MODE, 1>)<<<dim3(grid, cdiv(L, AN_CHANNELS)), 256, 0, ctx->stream>>>(
        G, x, v1, L, w, beta, wout, part ? part + nsum : nullptr);
    check_launch();
    nsum += grid;
  }
  return nsum;
}

}  // namespace

// out = scale * Psi(v1) (wavelets + Dirac)
void sara_synthesis(fhs_ctx* ctx, const fhs_sara* S, const float* v1, int L, float scale, float* out) {
  const SaraGeom& G = S->g;
  float* scr = (float*)ctx->ws.get("sara_scratch", std::max<int64_t>(1, G.scr_per_chan * L) * sizeof(float));
  Scope sc(ctx, "wavelet_synthesis");
  if (G.nb == 0) {   // G.s = Ny Nx
    const bool vec = G.s % 4 == 0 && ((uintptr_t)v1 | (uintptr_t)out) % 16 == 0;
    (vec ? k_dirac_synthesis<4> : k_dirac_synthesis<1>)<<<dim3(std::min<unsigned>(2048, cdiv(vec ? G.s / 4 : G.s, 256)), L),
                                                         256, 0, ctx->stream>>>(G, v1, scale, out);
    check_launch();
    return;
  }
  auto grid = [](int ty, int txg, int z) { return dim3(8 * cdiv((long long)ty * txg * z, 8), 1, 1); };
  for (int k = G.nlevel; k >= 2; --k) {
    int py = 0, px = 0;
    for (int b = 0; b < G.nb; ++b) {
      py = std::max(py, G.ny[b][k - 1]);
      px = std::max(px, G.nx[b][k - 1]);
    }
    const int ty = (int)cdiv(py, ST_Y), tx = (int)cdiv(px, ST_X);
    k_synthesis<false, false><<<grid(ty, (int)cdiv(tx, ST_WAVES), G.nb * L), 64 * ST_WAVES, 0, ctx->stream>>>(
        S->level[k], ty, tx, G.nb * L, v1, scr, scale, out);
    check_launch();
  }
  const int ty = (int)cdiv(G.Ny, ST_Y), tx = (int)cdiv(G.Nx, ST_X);
  if ((int64_t)ty * tx * L < SYN_SPLIT_BELOW)
    k_synthesis<true, true><<<grid(ty, tx, L), 64 * ST_WAVES, 0, ctx->stream>>>(S->level[1], ty, tx, L, v1, scr, scale,
                                                                                       out);
  else
    k_synthesis<true, false><<<grid(ty, (int)cdiv(tx, ST_WAVES), L), 64 * ST_WAVES, 0, ctx->stream>>>(
        S->level[1], ty, tx, L, v1, scr, scale, out);
  check_launch();
}

// v1 <- l21 dual step of (v1 + Psit(xhat)); g1 = sigma1 * Psi(v1)
void sara_dual_step(fhs_ctx* ctx, const fhs_sara* S, float* v1, const float* xhat, int L,
                    const float* w, double beta, float sigma1, float* g1) {
  const SaraGeom& G = S->g;
  {
    Scope sc(ctx, "wavelet_l21");
    if (L <= AN_CHANNELS) {
      sara_analyse<AN_L21>(ctx, S, xhat, L, v1, w, beta, nullptr, nullptr);
    } else {
      sara_analyse<AN_ADD>(ctx, S, xhat, L, v1, nullptr, 0.0, nullptr, nullptr);
      k_l21<<<std::min<unsigned>(2048, cdiv(G.s, 256)), 256, 0, ctx->stream>>>(G.s, v1, L, w, beta, 0, nullptr, nullptr);
      check_launch();
    }
  }
  sara_synthesis(ctx, S, v1, L, sigma1, g1);
}

int64_t sara_ncoefs(const fhs_sara* S) { return S->g.s; }

}  // namespace fhs

using namespace fhs;

extern "C" {

int fhs_sara_create_host(fhs_ctx* ctx, int Ny, int Nx, int nlevel, int nbases,
                         const int* filter_len, const double* lo_r, int with_dirac, fhs_sara** out) {
  if (!ctx || !out) return FHS_ERR_ARG;
  *out = nullptr;
  return guard(ctx, [&] {
    FHS_CHECK(Ny >= 1 && Nx >= 1, "sara_create: bad image size");
    FHS_CHECK(nlevel >= 1 && nlevel <= WMAX_LEVELS, "sara_create: nlevel must be in [1, 6]");
    FHS_CHECK(nbases >= 0 && nbases <= WMAX_BASES, "sara_create: at most 8 wavelet bases");
    FHS_CHECK(nbases + (with_dirac ? 1 : 0) >= 1, "sara_create: empty dictionary");
    auto S = std::make_unique<fhs_sara>();
    SaraGeom& G = S->g;
    G.Ny = Ny;
    G.Nx = Nx;
    G.nlevel = nlevel;
    G.nb = nbases;
    G.dirac = with_dirac ? 1 : 0;
    G.norm = (float)(1.0 / std::sqrt((double)(nbases + G.dirac)));
    int64_t off = 0, soff = 0;
    const double* f = lo_r;
    for (int b = 0; b < nbases; ++b) {
      const int lf = filter_len[b];
      FHS_CHECK(lf >= 2 && lf <= WMAX_LF && lf % 2 == 0, "sara_create: filter length must be even in [2, 16]");
      G.lf[b] = lf;
      for (int j = 0; j < lf; ++j) {
        G.lo[b][j] = (float)f[j];
      }
      f += lf;
      G.ny[b][0] = Ny;
      G.nx[b][0] = Nx;
      for (int k = 1; k <= nlevel; ++k) {
        G.ny[b][k] = (G.ny[b][k - 1] + lf - 1) / 2;
        G.nx[b][k] = (G.nx[b][k - 1] + lf - 1) / 2;
      }
      // scratch: approx levels 1..nlevel-1 (analysis), also reused by synthesis
      for (int k = 1; k < nlevel; ++k) {
        G.scr[b][k] = soff;
        soff += (int64_t)G.ny[b][k] * G.nx[b][k];
      }
      G.boff[b] = off;
      G.aoff[b] = 0;
      int64_t p = (int64_t)G.ny[b][nlevel] * G.nx[b][nlevel];
      for (int k = nlevel; k >= 1; --k) {
        G.doff[b][k] = p;
        p += 3 * (int64_t)G.ny[b][k] * G.nx[b][k];
      }
      off += p;
    }
    G.boff[nbases] = off;
    G.s = off + (G.dirac ? (int64_t)Ny * Nx : 0);
    G.scr_per_chan = soff;
    for (int k = 1; k <= nlevel; ++k) S->level[k] = level_args(G, k);
    *out = S.release();
  });
}

int fhs_sara_destroy(fhs_sara* S) {
  delete S;
  return FHS_OK;
}

int fhs_sara_info(const fhs_sara* S, int64_t* n_coefs) {
  if (!S) return FHS_ERR_ARG;
  if (n_coefs) *n_coefs = S->g.s;
  return FHS_OK;
}

int fhs_sara_analysis(fhs_ctx* ctx, const fhs_sara* S, const float* x, int L, float* coefs,
                      int accumulate) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(S && x && coefs && L >= 1 && L * std::max(1, S->g.nb) <= 65535, "sara_analysis: bad argument");
    Scope sc(ctx, "wavelet_analysis");
    if (accumulate)
      sara_analyse<AN_ADD>(ctx, S, x, L, coefs, nullptr, 0.0, nullptr, nullptr);
    else
      sara_analyse<AN_SET>(ctx, S, x, L, coefs, nullptr, 0.0, nullptr, nullptr);
  });
}

int fhs_sara_synthesis(fhs_ctx* ctx, const fhs_sara* S, const float* coefs, int L, float scale,
                       float* out) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(S && coefs && out && L >= 1 && L * std::max(1, S->g.nb) <= 65535, "sara_synthesis: bad argument");
    sara_synthesis(ctx, S, coefs, L, scale, out);
  });
}

int fhs_update_dual_sparsity(fhs_ctx* ctx, const fhs_sara* S, float* v1, const float* xhat, int L,
                             const float* weights1, double beta1, float sigma1, float* g1) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(S && v1 && xhat && g1 && L >= 1 && L * std::max(1, S->g.nb) <= 65535, "update_dual_sparsity: bad argument");
    sara_dual_step(ctx, S, v1, xhat, L, weights1, beta1, sigma1, g1);
  });
}

int fhs_sara_update_weights(fhs_ctx* ctx, const fhs_sara* S, const float* x, int L, double upsilon,
                            float* weights1) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(S && x && weights1 && L >= 1 && L * std::max(1, S->g.nb) <= 65535,
              "sara_update_weights: bad argument");
    const SaraGeom& G = S->g;
    if (L <= AN_CHANNELS) {   // the coefficients are never stored
      sara_analyse<AN_WEIGHT>(ctx, S, x, L, nullptr, nullptr, upsilon, weights1, nullptr);
      return;
    }
    float* c = (float*)ctx->ws.get("sara_prior_coefs", (size_t)G.s * L * sizeof(float));
    sara_analyse<AN_SET>(ctx, S, x, L, c, nullptr, 0.0, nullptr, nullptr);
    k_l21<<<std::min<unsigned>(2048, cdiv(G.s, 256)), 256, 0, ctx->stream>>>(G.s, c, L, nullptr, upsilon, 2, weights1,
                                                                             nullptr);
    check_launch();
  });
}

int fhs_compute_sara_prior(fhs_ctx* ctx, const fhs_sara* S, const float* x, int L, double* out) {
  if (!ctx) return FHS_ERR_ARG;
  return guard(ctx, [&] {
    FHS_CHECK(S && x && out && L >= 1 && L * std::max(1, S->g.nb) <= 65535, "compute_sara_prior: bad argument");
    const SaraGeom& G = S->g;
    unsigned n = 2048;   // workgroup sums
    for (int k = 1; k <= G.nlevel && G.nb > 0; ++k) {
      int ty, tx;
      n += analysis_grid(G, k, ty, tx);
    }
    double* part = (double*)ctx->ws.get("sara_prior_partial", (n + 1) * sizeof(double));
    unsigned nsum = 0;
    if (L <= AN_CHANNELS) {
      nsum = sara_analyse<AN_NORM>(ctx, S, x, L, nullptr, nullptr, 0.0, nullptr, part);
    } else {
      float* c = (float*)ctx->ws.get("sara_prior_coefs", (size_t)G.s * L * sizeof(float));
      sara_analyse<AN_SET>(ctx, S, x, L, c, nullptr, 0.0, nullptr, nullptr);
      nsum = std::min<unsigned>(2048, cdiv(G.s, 256));
      k_l21<<<nsum, 256, 0, ctx->stream>>>(G.s, c, L, nullptr, 0.0, 1, nullptr, part);
      check_launch();
    }
    k_sum_l<<<1, 256, 0, ctx->stream>>>(part, (int)nsum, part + n);
    check_launch();
    FHS_HIP(hipMemcpyAsync(out, part + n, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    FHS_HIP(hipStreamSynchronize(ctx->stream));
  });
}

}  // extern "C"
