// Device-resident interpolation matrix G of one channel.
//
// Forward (degridding, y = G Fx) reads G transposed: value j of row m sits at
// vals[j*M + m], so the 64 lanes of a wavefront (64 consecutive rows) load
// 64 consecutive complex values per tap (one 512-byte coalesced load).
// Two row formats share that value layout:
//   ELL    : explicit column per tap (cols[j*M + m]), any sparsity pattern;
//   WINDOW : one anchor per row; tap j = jx*Ky + jy reads grid point
//            ((ky0 + jy) mod Kty, (kx0 + jx) mod Ktx) - the dense min-max
//            window, no column indices (8 B per nonzero instead of 12).
//   SEP    : the min-max interpolator of a 2-D NUFFT is the Kronecker
//            product of two 1-D interpolators, G[m, (jy, jx)] =
//            cy[m][jy] cx[m][jx]: a row stores Ky + Kx complex values plus
//            its anchor, row-major in one 128-byte line (cy in slots 0-7, cx
//            in slots 8-15, zero padded) instead of 392 B for 7 x 7 taps, so
//            any gather order costs one line per row.  The CSC of the adjoint
//            (small grids) stores only (row << 6 | tap) per nonzero (4 B).
// Adjoint (gridding, Fx = G' y) is computed per grid point, each output
// owned by one thread (no atomics, deterministic summation order): from a
// CSC copy (colptr / rows / values) in general, by tile gridding for the
// separable layout on grids of whole 32 x 32 tiles.
#pragma once

#include <hip/hip_fp16.h>

#include <type_traits>

#include "common.hpp"

namespace fhs {

enum GLayout { G_ELL = 0, G_WINDOW = 1, G_SEP = 2 };
constexpr int SEP_KMAX = 16;  // max taps per axis of the separable layout
// A separable row holds 2 kmax complex slots (cy in 0..kmax-1, cx in
// kmax..2 kmax-1, zero padded), kmax = 8 (128-byte rows, windows of up to
// 8 taps: the min-max interpolator) or 16 (256-byte rows: w-projected rows).
inline int sep_kmax_for(int Ky, int Kx) { return (Ky <= 8 && Kx <= 8) ? 8 : 16; }

struct GDev {
  int layout;
  int M, K;
  int Kty, Ktx, Ky, Kx;
  int ncols;
  const int* cols;      // ELL: [K][M]
  const int* anchor;    // WINDOW: [M]
  const float2* vals;   // ELL / WINDOW: [K][M]; SEP: [M][2 kmax] (__half2 slots if half)
  int kmax;             // SEP: complex slots per axis in a row (8 or 16)
  int half;             // SEP on a tiled grid: rows stored as FP16 (re, im) pairs, 4 B a slot
  const int* colptr;    // [ncols + 1]
  const int* csc_rows;  // [nnz]
  const float2* csc_vals;
  const int* ucol;      // adjoint work units: unit u = columns [ucol[u], ucol[u+1])
  int nunits;
  const unsigned* csc_pk;  // SEP: (row << 6) | (jx*Ky + jy) per nonzero
  // SEP on a tiled grid: adjoint by patches (no CSC; nunits = workgroups of 4 jobs)
  int tiled, tiles_y, tiles_x;
  // rows listed under every 16 x 16 patch of the grid their window touches:
  // {row, window origin relative to the patch as two signed bytes (y, x << 8)},
  // rows ascending inside a patch
  const int2* pent;
  // one wave's work each, longest first: {patch, first entry, entries, slot};
  // slot -1 writes the patch, slot >= 0 writes partial[slot] (a patch split over
  // several jobs, summed in slot order by the reduce pass), slot -2 zeroes the
  // empty patches empty[first .. first + entries)
  const int4* jobs;
  int njobs, patches_y;
  const int* empty;
  const int4* red;         // {patch, first slot, slot count} of the split patches
  int nred;
  float2* partial;         // [slots][PATCH * PATCH]
  // forward by tile: rows grouped by the tile of their anchor (ascending row
  // order inside a tile), work items {tile, begin, end, 0} of <= FWD_ITEM rows
  const int* prim_rows;
  const int4* fitems;
  int nfitems;
  // holographic form (square, rows = columns = grid points): the full
  // Hermitian stencil G'G of each active mode i, stencil[o * nact + i] for the
  // (2Ky-1) x (2Kx-1) neighbourhood offsets o = (dy + Ky-1) + (2Ky-1)(dx + Kx-1),
  // and act[p] = i for the active grid points (-1 elsewhere)
  const float2* stencil;
  const int* act;
  int nact;
};

// one FP16 slot (re, im), as stored in a 32-bit word, in FP32
__device__ __forceinline__ float2 h2f(unsigned u) {
  __half2 h;
  __builtin_memcpy(&h, &u, 4);
  return __half22float2(h);
}

// the 2 KM complex slots of separable row m (KM 16-byte loads, KM / 2 for
// FP16 rows); KM = g.kmax
template <int KM>
__device__ __forceinline__ void sep_load(const GDev& g, int m, float2* cy, float2* cx) {
  if (g.half) {
    const uint4* q = reinterpret_cast<const uint4*>(reinterpret_cast<const __half2*>(g.vals) + (size_t)m * (2 * KM));
#pragma unroll
    for (int i = 0; i < KM / 4; ++i) {
      const uint4 a = q[i], b = q[KM / 4 + i];
      cy[4 * i] = h2f(a.x);
      cy[4 * i + 1] = h2f(a.y);
      cy[4 * i + 2] = h2f(a.z);
      cy[4 * i + 3] = h2f(a.w);
      cx[4 * i] = h2f(b.x);
      cx[4 * i + 1] = h2f(b.y);
      cx[4 * i + 2] = h2f(b.z);
      cx[4 * i + 3] = h2f(b.w);
    }
    return;
  }
  const float4* p = reinterpret_cast<const float4*>(g.vals + (size_t)m * (2 * KM));
#pragma unroll
  for (int i = 0; i < KM / 2; ++i) {
    const float4 a = p[i], b = p[KM / 2 + i];
    cy[2 * i] = make_float2(a.x, a.y);
    cy[2 * i + 1] = make_float2(a.z, a.w);
    cx[2 * i] = make_float2(b.x, b.y);
    cx[2 * i + 1] = make_float2(b.z, b.w);
  }
}

// value and row of CSC entry e
__device__ __forceinline__ void g_csc_entry(const GDev& g, int e, float2& v, int& r) {
  if (g.layout == G_SEP) {
    const unsigned pk = g.csc_pk[e];
    r = (int)(pk >> 6);
    const int tap = (int)(pk & 63u), jx = tap / g.Ky, jy = tap - jx * g.Ky;
    v = cmul(g.vals[(size_t)r * 2 * g.kmax + jy], g.vals[(size_t)r * 2 * g.kmax + g.kmax + jx]);
  } else {
    v = g.csc_vals[e];
    r = g.csc_rows[e];
  }
}

// Adjoint work units: contiguous column ranges holding about ADJ_ENTRIES
// nonzeros (and at most ADJ_COLS columns), so every workgroup streams the
// same amount of CSC data whatever the uv density.
constexpr int ADJ_THREADS = 256;
constexpr int ADJ_ENTRIES = 2048;
constexpr int ADJ_COLS = 2048;
constexpr int ADJ_LDS = 4096;

// sum over taps j of row m: G[m, c_j] * f(c_j)
template <class F>
__device__ __forceinline__ float2 g_row_apply(const GDev& g, int m, F&& f) {
  float2 acc = make_float2(0.f, 0.f);
  if (g.layout == G_ELL) {
    for (int j = 0; j < g.K; ++j) {
      const int c = g.cols[(size_t)j * g.M + m];
      const float2 v = g.vals[(size_t)j * g.M + m];
      const float2 x = f(c);
      acc.x += v.x * x.x - v.y * x.y;
      acc.y += v.x * x.y + v.y * x.x;
    }
  } else if (g.layout == G_SEP && g.kmax > 8) {
    const int a = g.anchor[m];
    const int ky0 = a % g.Kty, kx0 = a / g.Kty;
    const float2* row = g.vals + (size_t)m * 2 * g.kmax;
    for (int jx = 0; jx < g.Kx; ++jx) {
      int kx = kx0 + jx;
      if (kx >= g.Ktx) kx -= g.Ktx;
      const int colbase = kx * g.Kty;
      float2 s = make_float2(0.f, 0.f);
      for (int jy = 0; jy < g.Ky; ++jy) {
        int ky = ky0 + jy;
        if (ky >= g.Kty) ky -= g.Kty;
        const float2 x = f(colbase + ky), c = row[jy];
        s.x += c.x * x.x - c.y * x.y;
        s.y += c.x * x.y + c.y * x.x;
      }
      const float2 c = row[g.kmax + jx];
      acc.x += c.x * s.x - c.y * s.y;
      acc.y += c.x * s.y + c.y * s.x;
    }
  } else if (g.layout == G_SEP) {
    const int a = g.anchor[m];
    const int ky0 = a % g.Kty, kx0 = a / g.Kty;
    float2 cy[8], cx[8];
    sep_load<8>(g, m, cy, cx);
#pragma unroll
    for (int jx = 0; jx < 8; ++jx) {   // fully unrolled: cy / cx stay in registers
      if (jx < g.Kx) {
        int kx = kx0 + jx;
        if (kx >= g.Ktx) kx -= g.Ktx;
        const int colbase = kx * g.Kty;
        float2 s = make_float2(0.f, 0.f);
#pragma unroll
        for (int jy = 0; jy < 8; ++jy) {
          if (jy < g.Ky) {
            int ky = ky0 + jy;
            if (ky >= g.Kty) ky -= g.Kty;
            const float2 x = f(colbase + ky);
            s.x += cy[jy].x * x.x - cy[jy].y * x.y;
            s.y += cy[jy].x * x.y + cy[jy].y * x.x;
          }
        }
        const float2 c = cx[jx];
        acc.x += c.x * s.x - c.y * s.y;
        acc.y += c.x * s.y + c.y * s.x;
      }
    }
  } else {
    const int a = g.anchor[m];
    const int ky0 = a % g.Kty, kx0 = a / g.Kty;
    int j = 0;
    for (int jx = 0; jx < g.Kx; ++jx) {
      int kx = kx0 + jx;
      if (kx >= g.Ktx) kx -= g.Ktx;
      const int colbase = kx * g.Kty;
      for (int jy = 0; jy < g.Ky; ++jy, ++j) {
        int ky = ky0 + jy;
        if (ky >= g.Kty) ky -= g.Kty;
        const float2 v = g.vals[(size_t)j * g.M + m];
        const float2 x = f(colbase + ky);
        acc.x += v.x * x.x - v.y * x.y;
        acc.y += v.x * x.y + v.y * x.x;
      }
    }
  }
  return acc;
}

__device__ __forceinline__ float2 g_row_dot(const GDev& g, int m, const float2* __restrict__ Fx) {
  return g_row_apply(g, m, [&](int c) { return Fx[c]; });
}

// sum over rows r of column k: conj(G[r,k]) * w(r)
template <class W>
__device__ __forceinline__ float2 g_col_dot(const GDev& g, int k, W&& w) {
  float2 acc = make_float2(0.f, 0.f);
  const int e0 = g.colptr[k], e1 = g.colptr[k + 1];
  for (int e = e0; e < e1; ++e) {
    float2 v;
    int r;
    g_csc_entry(g, e, v, r);
    const float2 y = w(r);
    acc.x += v.x * y.x + v.y * y.y;
    acc.y += v.x * y.y - v.y * y.x;
  }
  return acc;
}

// One adjoint work unit: the unit's CSC entries are loaded coalesced (lane
// t takes entries t, t+256, ...), their products conj(G) w(row) staged in
// LDS, then each thread sums whole columns from LDS and writes them: every
// output column belongs to exactly one unit (no atomics).  extra(c) is added
// to column c (the G w term of the Hermitian DR form).
template <class W, class X>
__device__ __forceinline__ void g_adjoint_unit(const GDev& g, int u, W&& w, X&& extra,
                                               float2* __restrict__ out, float2* prod) {
  const int c0 = g.ucol[u], c1 = g.ucol[u + 1];
  const int e0 = g.colptr[c0], n = g.colptr[c1] - e0;
  if (n <= ADJ_LDS) {
    for (int e = threadIdx.x; e < n; e += ADJ_THREADS) {
      float2 v;
      int r;
      g_csc_entry(g, e0 + e, v, r);
      const float2 y = w(r);
      prod[e] = make_float2(v.x * y.x + v.y * y.y, v.x * y.y - v.y * y.x);
    }
    __syncthreads();
    for (int c = c0 + threadIdx.x; c < c1; c += ADJ_THREADS) {
      const int a = g.colptr[c] - e0, b = g.colptr[c + 1] - e0;
      float2 s = make_float2(0.f, 0.f);
      for (int e = a; e < b; ++e) s = cadd(s, prod[e]);
      out[c] = cadd(s, extra(c));
    }
  } else {   // a column longer than the LDS stage: direct gather
    for (int c = c0 + threadIdx.x; c < c1; c += ADJ_THREADS) out[c] = cadd(g_col_dot(g, c, w), extra(c));
  }
}

// Gridding adjoint of the separable layout, on the matrix cores.
//
// The grid is cut into 16 x 16 patches, and at creation every row is listed
// under each patch its Ky x Kx window touches (1.9 for a 7 x 7 window on
// average, 3.5 for 15 x 15), with its window origin (dy, dx) relative to the
// patch.  Restricted to a patch the adjoint is a sum of rank-1 updates,
//   out[y][x] = sum_rows conj(cy[y - dy]) * (w(row) conj(cx[x - dx])),
// a GEMM whose inner dimension runs over the listed rows.  One wave owns one
// patch and accumulates v_mfma_f32_16x16x4f32 in FP32, two complex rows per
// instruction pair: lane (i, k) supplies re / im (k even / odd) of row k / 2 of
// the pair.  The wave stages its rows in LDS of its own, 16 at a time, so there
// is no barrier and no compaction.  A lane outside a row's window reads the
// zero slot behind the row (its slot index is clamped).
//
// A zero times a non-finite value would still spread NaN over the patch, so
// a patch with a non-finite sum is summed again tap by tap (patch_exact):
// only the points a row's window covers see its value.
//
// Every output point is written once, by one lane, after a fixed-order sum: no
// atomics, deterministic.  The uv density varies by orders of magnitude (empty
// corners, a dense centre), so a patch's list is cut into jobs of at most
// PATCH_JOB rows whose partial patches a second pass adds in a fixed order, and
// empty patches are zeroed in groups.  Jobs are sorted by length, so the four
// waves of a workgroup end together.  256 rows a job: the partial patches add an
// eighth to the row bytes of a dense patch, and a channel of 65k rows still
// fills the GPU (SARA 256 x 256: 18 us against 54 us for the earlier gather by
// 32 x 32 tiles in LDS).  2.6M 7 x 7 rows on 16 grids of 1024 x 1024: 172 us
// against 268 us for the gather; 1.6M 15 x 15 rows on 4 grids of 4096 x 4096:
// 318 us, 112 us of it the time to write the grids at the rate of a large copy.
constexpr int PATCH = 16;
constexpr int PATCH_JOB = 256;                       // listed rows per job
constexpr int PATCH_EMPTY_GROUP = 8;                 // empty patches zeroed per job
// The forward stages windows of 32 x 32 tiles.
constexpr int TILE_Y = 32, TILE_X = 32;
constexpr int FWD_ITEM = 1024;                       // rows per forward work item
template <int KM>
constexpr int fwd_win() { return (TILE_Y + KM - 1) * (TILE_X + KM - 1); }   // forward window (complex)

inline bool tile_grid_ok(int Kty, int Ktx, int Ky, int Kx) {
  return Kty % TILE_Y == 0 && Ktx % TILE_X == 0 && Kty >= TILE_Y + Ky - 1 && Ktx >= TILE_X + Kx - 1;
}

typedef float mfma_f4 __attribute__((ext_vector_type(4)));

// Pointers that a kernel reads from memory (the members of GDev) are generic
// to the compiler, whose flat loads wait on the LDS counter too; these casts
// say that they point to global memory.
#define FHS_GLOBAL __attribute__((address_space(1)))
typedef float vec2f __attribute__((ext_vector_type(2)));
typedef int vec2i __attribute__((ext_vector_type(2)));
typedef unsigned vec4u __attribute__((ext_vector_type(4)));
typedef float vec4f __attribute__((ext_vector_type(4)));
typedef float vec4f_a8 __attribute__((ext_vector_type(4), aligned(8)));   // a caller's complex array is 8-byte aligned
template <class T>
__device__ __forceinline__ const FHS_GLOBAL T* as_global(const void* p) {
  return (const FHS_GLOBAL T*)p;
}

// value of lane P of this lane's row of 16 (one DPP move, no LDS).  Used in sums
// only: folded into a subtraction (v_subrev_u32_dpp) it was read from the
// other operand.
template <int P>
__device__ __forceinline__ int row_bcast(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x150 + P, 0xf, 0xf, true);   // row_newbcast:P
}

// Rows of a patch staged at a time by its wave, in LDS of its own: cy of each
// slot, and conj(cx) w as the two B operands of re / im (k even: q.re, q.im;
// k odd: q.im, -q.re), with a zero slot behind each row.
constexpr int PR = 16;
template <int KM>
struct PatchStage {
  float4 b[PR][KM + 1];
  float2 a[PR][KM + 1];
};

// Sums the n listed rows of one job: lane (j, g) gets rows 4g .. 4g + 3
// of column j.
// Chunks of PR rows: the row lines come in as 16-byte words (a load of 64
// scattered slots takes 16 address cycles, three per pair of rows), the next
// chunk's while this one is multiplied and its entries a chunk earlier.  Lane
// (i, k) holds the entry of row 2 (i mod 8) + k / 2, so pair p reads its window
// origins from lane p of its 16 lanes.
template <int KM, bool HALF, bool LAM>
__device__ __forceinline__ void patch_mfma(const GDev& g, const int2* __restrict__ entries, int n,
                                              const float2* __restrict__ wv, const float* __restrict__ lamv,
                                              PatchStage<KM>& st, mfma_f4& cre, mfma_f4& cim) {
  constexpr int ROWB = 2 * KM * (HALF ? 4 : 8);   // bytes of a row
  constexpr int LPR = ROWB / 16, RPI = 64 / LPR;  // lanes per row, rows per load
  constexpr int NI = PR / RPI;                    // loads per chunk
  constexpr int SPL = HALF ? 4 : 2;               // slots per lane
  const int lane = threadIdx.x & 63;
  const int li = lane & 15, part = (lane >> 4) & 1, half = lane >> 5;
  const int mine = 2 * (li & 7) + half;
  const int sub = lane % LPR, rl = lane / LPR, s0 = (sub % (LPR / 2)) * SPL;
  const bool isb = sub >= LPR / 2;
  const FHS_GLOBAL char* rows = as_global<char>(g.vals);
  const FHS_GLOBAL vec2f* w = as_global<vec2f>(wv);
  const FHS_GLOBAL float* lam = as_global<float>(lamv);
  const FHS_GLOBAL vec2i* ent = as_global<vec2i>(entries);
  if (lane < PR) {
    st.a[lane][KM] = make_float2(0.f, 0.f);
    st.b[lane][KM] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // lanes past the end repeat the first row with its window out of reach
  const int first = ent[0].x;
  auto entry = [&](int c) {
    vec2i e = {first, 0xc0c0};   // (dy, dx) = (-64, -64)
    if (c + mine < n) e = ent[c + mine];
    return e;
  };
  vec4u raw[NI];
  vec2f v[NI];
  float lm[NI];
  auto fetch = [&](int row) {
#pragma unroll
    for (int t = 0; t < NI; ++t) {
      const int rr = t * RPI + rl;
      const int r = __shfl(row, (rr >> 1) + 32 * (rr & 1), 64);
      raw[t] = *(const FHS_GLOBAL vec4u*)(rows + (size_t)(unsigned)r * ROWB + sub * 16);
      v[t] = w[r];
      if constexpr (LAM) lm[t] = lam[r];
    }
  };
  auto stage = [&] {
#pragma unroll
    for (int t = 0; t < NI; ++t) {
      const int rr = t * RPI + rl;
      float2 c[SPL];
      if constexpr (HALF) {
#pragma unroll
        for (int j = 0; j < SPL; ++j) c[j] = h2f(raw[t][j]);
      } else {
#pragma unroll
        for (int j = 0; j < SPL; ++j) c[j] = make_float2(__uint_as_float(raw[t][2 * j]), __uint_as_float(raw[t][2 * j + 1]));
      }
      if (isb) {
        float2 x = make_float2(v[t].x, v[t].y);
        if constexpr (LAM) x = cscale(x, lm[t]);
#pragma unroll
        for (int j = 0; j < SPL; ++j) {
          const float qx = c[j].x * x.x + c[j].y * x.y, qy = c[j].x * x.y - c[j].y * x.x;
          st.b[rr][s0 + j] = make_float4(qx, qy, qy, -qx);
        }
      } else {
#pragma unroll
        for (int j = 0; j < SPL; ++j) st.a[rr][s0 + j] = c[j];
      }
    }
  };
  const float* sa = &st.a[half][0].x + part;
  const float2* sb = reinterpret_cast<const float2*>(&st.b[half][0]) + part;
  // re += cy.x q.re + cy.y q.im, im += cy.x q.im - cy.y q.re
  auto pair = [&](auto pc, int ndy, int ndx) {
    constexpr int P = decltype(pc)::value;
    const unsigned sy = min((unsigned)(li + row_bcast<P>(ndy)), (unsigned)KM);
    const unsigned sx = min((unsigned)(li + row_bcast<P>(ndx)), (unsigned)KM);
    const float a = sa[2 * (P * 2 * (KM + 1) + sy)];
    const float2 b = sb[2 * (P * 2 * (KM + 1) + sx)];
    cre = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b.x, cre, 0, 0, 0);
    cim = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b.y, cim, 0, 0, 0);
  };
  vec2i cur = entry(0), nxt = entry(PR);
  fetch(cur.x);
  for (int c = 0; c < n; c += PR) {
    __builtin_amdgcn_wave_barrier();
    stage();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int ndy = -(int)(signed char)(cur.y & 0xff), ndx = -(int)(signed char)((cur.y >> 8) & 0xff);
    const int rem = n - c;
    if (rem > PR) {
      cur = nxt;
      fetch(cur.x);
      nxt = entry(c + 2 * PR);
    }
    pair(std::integral_constant<int, 0>{}, ndy, ndx);
    pair(std::integral_constant<int, 1>{}, ndy, ndx);
    if (rem <= 4) break;
    pair(std::integral_constant<int, 2>{}, ndy, ndx);
    pair(std::integral_constant<int, 3>{}, ndy, ndx);
    if (rem <= 8) break;
    pair(std::integral_constant<int, 4>{}, ndy, ndx);
    pair(std::integral_constant<int, 5>{}, ndy, ndx);
    if (rem <= 12) break;
    pair(std::integral_constant<int, 6>{}, ndy, ndx);
    pair(std::integral_constant<int, 7>{}, ndy, ndx);
    static_assert(PR == 16, "eight pairs a chunk");
  }
}

// The same sums tap by tap (the lane's four points, rows in list order).  Called,
// not inlined, so it takes the members it needs by value: a reference to a matrix
// that is a kernel argument would copy the whole of it, 240 bytes, to scratch in
// every lane (500k rows of 15 x 15 taps on a 4096 x 4096 grid: 230 us, 100 without;
// 1M of 7 x 7 on 2048 x 2048: 111 and 64).
struct PatchSums {
  mfma_f4 re, im;
};
template <int KM, class W>
__device__ __noinline__ PatchSums patch_exact(const float2* __restrict__ vals, int half, int Ky, int Kx,
                                              const int2* __restrict__ ent, int n, W w) {
  const int lane = threadIdx.x & 63, li = lane & 15, y0 = 4 * (lane >> 4);
  auto slot = [&](int r, int j) {
    const size_t i = (size_t)r * (2 * KM) + j;
    return half ? h2f(reinterpret_cast<const unsigned*>(vals)[i]) : vals[i];
  };
  mfma_f4 cre = {0.f, 0.f, 0.f, 0.f}, cim = cre;
  for (int e = 0; e < n; ++e) {
    const int r = ent[e].x, pk = ent[e].y;
    const int dy = (int)(signed char)(pk & 0xff), dx = (int)(signed char)((pk >> 8) & 0xff);
    const int jx = li - dx;
    if ((unsigned)jx >= (unsigned)Kx) continue;
    const float2 v = w(r), c = slot(r, KM + jx);
    const float2 q = make_float2(c.x * v.x + c.y * v.y, c.x * v.y - c.y * v.x);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int jy = y0 + i - dy;
      if ((unsigned)jy < (unsigned)Ky) {
        const float2 a = slot(r, jy);
        cre[i] += a.x * q.x + a.y * q.y;
        cim[i] += a.x * q.y - a.y * q.x;
      }
    }
  }
  return {cre, cim};
}

// Four jobs, one per wave.
template <int KM, bool LAM>
__device__ __forceinline__ void g_adjoint_patches(const GDev& g, int unit, const float2* __restrict__ w,
                                                  const float* __restrict__ lam, float2* __restrict__ out) {
  __shared__ PatchStage<KM> stages[ADJ_THREADS / 64];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = unit * (ADJ_THREADS / 64) + wv;
  if (j >= g.njobs) return;
  const int4 job = g.jobs[j];
  const int patch = __builtin_amdgcn_readfirstlane(job.x), e0 = __builtin_amdgcn_readfirstlane(job.y);
  const int n = __builtin_amdgcn_readfirstlane(job.z), slot = __builtin_amdgcn_readfirstlane(job.w);
  // a patch leaves as 16-byte words, 8 lanes to a column of 16 points, so whole
  // 128-byte lines are written
  auto put = [&](float2* o, size_t stride, vec4f v0, vec4f v1) {
    FHS_GLOBAL char* q = (FHS_GLOBAL char*)(o + (lane >> 3) * stride + 2 * (lane & 7));
    *(FHS_GLOBAL vec4f_a8*)q = v0;
    *(FHS_GLOBAL vec4f_a8*)(q + 8 * stride * sizeof(float2)) = v1;
  };
  auto at = [&](int p) {
    const int py = p % g.patches_y, px = p / g.patches_y;
    return out + (size_t)(px * PATCH) * g.Kty + py * PATCH;
  };
  if (slot == -2) {
    const vec4f zero = {0.f, 0.f, 0.f, 0.f};
    for (int e = e0; e < e0 + n; ++e) put(at(g.empty[e]), g.Kty, zero, zero);
    return;
  }
  mfma_f4 cre = {0.f, 0.f, 0.f, 0.f}, cim = cre;
  const int2* __restrict__ ent = g.pent + e0;
  if (g.half)
    patch_mfma<KM, true, LAM>(g, ent, n, w, lam, stages[wv], cre, cim);
  else
    patch_mfma<KM, false, LAM>(g, ent, n, w, lam, stages[wv], cre, cim);
  bool bad = false;
#pragma unroll
  for (int r = 0; r < 4; ++r) bad = bad || !isfinite(cre[r]) || !isfinite(cim[r]);
  if (__any(bad)) {
    auto wr = [=](int r) { return LAM ? cscale(w[r], lam[r]) : w[r]; };
    const PatchSums e = patch_exact<KM>(g.vals, g.half, g.Ky, g.Kx, ent, n, wr);
    cre = e.re;
    cim = e.im;
  }
  // lane (i, k) holds points 4k .. 4k + 3 of column i: transposed through LDS
  static_assert(sizeof(PatchStage<KM>) >= PATCH * PATCH * sizeof(float2), "a patch fits the stage");
  vec4f* t = reinterpret_cast<vec4f*>(&stages[wv]);
  __builtin_amdgcn_wave_barrier();
  t[(lane & 15) * 8 + 2 * (lane >> 4)] = vec4f{cre[0], cim[0], cre[1], cim[1]};
  t[(lane & 15) * 8 + 2 * (lane >> 4) + 1] = vec4f{cre[2], cim[2], cre[3], cim[3]};
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (slot >= 0)
    put(g.partial + (size_t)slot * (PATCH * PATCH), PATCH, t[lane], t[lane + 64]);
  else
    put(at(patch), g.Kty, t[lane], t[lane + 64]);
}

// sum of the partial patches of split patch r, in slot order (one point per thread)
__device__ __forceinline__ void g_adjoint_reduce(const GDev& g, int r, float2* __restrict__ out) {
  static_assert(ADJ_THREADS == PATCH * PATCH, "one point per thread");
  const int4 rd = g.red[r];
  const int py = rd.x % g.patches_y, px = rd.x / g.patches_y, p = threadIdx.x;
  const float2* part = g.partial + (size_t)rd.y * (PATCH * PATCH) + p;
  float2 a = make_float2(0.f, 0.f);
  for (int j = 0; j < rd.z; ++j) a = cadd(a, part[(size_t)j * (PATCH * PATCH)]);
  out[(size_t)(px * PATCH + p / PATCH) * g.Kty + py * PATCH + p % PATCH] = a;
}

// Forward (degridding) of one work item: the (TILE_Y + Ky - 1) x (TILE_X +
// Kx - 1) grid window of the tile is staged in LDS once (all loads issued
// before the stores), then every row of the item reads its Ky x Kx taps from
// LDS instead of gathering them through the caches.  emit(r, G Fx) stores
// row r's value.
template <int KM, class P, class E>
__device__ __forceinline__ void g_forward_tile(const GDev& g, int item, const float2* __restrict__ Fx,
                                               float2* win, P&& pre, E&& emit) {
  const int4 it = g.fitems[item];
  const int t = it.x;
  const int ty0 = (t % g.tiles_y) * TILE_Y, tx0 = (t / g.tiles_y) * TILE_X;
  const int wy = TILE_Y + g.Ky - 1, wx = TILE_X + g.Kx - 1, nw = wy * wx;
  constexpr int PER = (fwd_win<KM>() + ADJ_THREADS - 1) / ADJ_THREADS;
  float2 v[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = threadIdx.x + i * ADJ_THREADS;
    v[i] = make_float2(0.f, 0.f);
    if (e < nw) {
      int ky = ty0 + e % wy, kx = tx0 + e / wy;
      if (ky >= g.Kty) ky -= g.Kty;
      if (kx >= g.Ktx) kx -= g.Ktx;
      v[i] = Fx[(size_t)kx * g.Kty + ky];
    }
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = threadIdx.x + i * ADJ_THREADS;
    if (e < nw) win[e] = v[i];
  }
  __syncthreads();
  int k = it.y + threadIdx.x;
  int rn = k < it.z ? g.prim_rows[k] : 0;
  for (; k < it.z; k += ADJ_THREADS) {
    const int r = rn;   // the next row index is loaded one step ahead
    if (k + ADJ_THREADS < it.z) rn = g.prim_rows[k + ADJ_THREADS];
    const auto pf = pre(r);   // the caller's per-row loads, issued before the arithmetic
    const int a = g.anchor[r];
    const int ly = a % g.Kty - ty0, lx = a / g.Kty - tx0;
    float2 cy[KM], cx[KM];
    sep_load<KM>(g, r, cy, cx);
    float2 acc = make_float2(0.f, 0.f);
#pragma unroll
    for (int jx = 0; jx < KM; ++jx) {
      if (jx < g.Kx) {
        const float2* col = win + (lx + jx) * wy + ly;
        float2 s = make_float2(0.f, 0.f);
#pragma unroll
        for (int jy = 0; jy < KM; ++jy) {
          if (jy < g.Ky) {
            const float2 x = col[jy];
            s.x += cy[jy].x * x.x - cy[jy].y * x.y;
            s.y += cy[jy].x * x.y + cy[jy].y * x.x;
          }
        }
        const float2 c = cx[jx];
        acc.x += c.x * s.x - c.y * s.y;
        acc.y += c.x * s.y + c.y * s.x;
      }
    }
    emit(r, acc, pf);
  }
}

// host construction helpers (gmat.hip)
std::vector<int> adjoint_units(const std::vector<int>& colptr);
void sep_csc(int64_t M, const int32_t* anchor, int Kty, int Ktx, int Ky, int Kx, std::vector<int>& colptr,
             std::vector<unsigned>& pk);

}  // namespace fhs

struct fhs_gmat {
  int device = 0;
  fhs::GDev d{};
  int64_t M = 0, ncols = 0, nnz = 0;
  int64_t n_modes = 0;   // holographic form: active Fourier modes (0 for a measurement G)
  void* mem[14] = {};
};
