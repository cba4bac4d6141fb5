// gfx950 kernel of ONE step of an LSTM layer with its input projection: a recurrent decoder's call, once per output label.
#pragma once

#include <hip/hip_runtime.h>

#include "lstm2_kernels.h"

namespace rtn {

struct LstmStepParams {
  const void* x;     // [B,in] AT
  const void* h;     // [B,n] AT
  const float* c;    // [B,n]
  const void* ff;    // [4n,in] AT, gate blocks cell-in, input, forget, output
  const void* rec;   // [n,4n] AT
  const void* bias;  // [4n] AT or null
  void* y;           // [B,n] AT
  void* h_out;       // [B,n] AT: the same values, in an array of their own
  float* c_out;      // [B,n]
  int B, in_dim, n;
  int by_fragments;  // 1: rows of x, h and ff are whole fragments, cells come in whole workgroups, every array is below 2 GB
};

// A step reads every weight once and uses it for a handful of rows: it is bound by bringing (in + n) * 4n weights on chip
// (n = 1024, in = 512 in bf16: 12.6 MB, which stay in the L2s from step to step) and by the latency of a launch.  So: one
// launch, no packing of the weights, no workspace.
//
// A workgroup of 8 wavefronts owns 8 cells = two MFMA tiles of 16 gate columns (row i of tile m: gate i % 4 of cell
// 2 (i / 4) + m, so that a lane of the result holds the four gates of one (cell, row) pair) and 16 * NT rows; the
// macro steps of the contraction, those of x and of h counted through, are dealt to the wavefronts, which sum their
// partial tiles through LDS.  8 cells: 128 workgroups at n = 1024 -- with 16 the CU's address unit would be as busy (a
// load of rec touches 16 pieces of 16 rows either way) and half of the CUs idle.  ff lies along the contraction and its
// rows are fragments as they are; rec lies across it: a lane loads a pair of neighbouring cells from every row of its
// fragment and deals the halves to the two tiles.  Workgroups of neighbouring cells go to one XCD, whose L2 then serves
// the 128-byte lines that 8 of them share.
// Measured (bf16, B = 12, in = 512, n = 1024): mask, projection, packing of W, the recurrent kernel and the final output were
// five launches of 38 us together, and 123 us per call; as one launch 11.2 us per call while rec was asked for behind the products of x and
// the cell state and the bias behind those of h -- three latencies in a row --, 9.9 now that all of them leave at once (n = 2048, in = 1024 27.5 / 25.2, 40 rows
// 12.6 / 11.2, float32 16.3 / 15.2; smaller calls are the host's 9.3).  What is left is the way of 12.6 MB through the address units, 16 pieces of 16 bytes
// per load of rec.  (Every 64 rows read all weights:
// where that is much, the caller takes a GEMM and the recurrent kernels, see lstm_step in the binding.)
constexpr int kStepThreads = 512, kStepWaves = kStepThreads / 64, kStepCells = 8;

template <typename AT>
struct CellPair;  // two neighbouring cells of one row of rec, and the fragments that KE rows of them make
template <>
struct CellPair<__bf16> {
  typedef unsigned T;
  typedef unsigned __attribute__((aligned(2))) T_any;
  static __device__ __forceinline__ T make(__bf16 a, __bf16 b) {
    return (unsigned)__builtin_bit_cast(unsigned short, a) | ((unsigned)__builtin_bit_cast(unsigned short, b) << 16);
  }
  static __device__ __forceinline__ void fragments(const T (&v)[8], i32x4& f0, i32x4& f1) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      f0[w] = (int)((v[2 * w] & 0xFFFFu) | (v[2 * w + 1] << 16));
      f1[w] = (int)((v[2 * w] >> 16) | (v[2 * w + 1] & 0xFFFF0000u));
    }
  }
};
template <>
struct CellPair<float> {
  typedef unsigned long long T;
  typedef unsigned long long __attribute__((aligned(4))) T_any;
  static __device__ __forceinline__ T make(float a, float b) {
    return (T)__builtin_bit_cast(unsigned, a) | ((T)__builtin_bit_cast(unsigned, b) << 32);
  }
  static __device__ __forceinline__ void fragments(const T (&v)[4], i32x4& f0, i32x4& f1) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      f0[w] = (int)(unsigned)v[w];
      f1[w] = (int)(unsigned)(v[w] >> 32);
    }
  }
};

// KE elements of a row from column k on, zeros from column `width` on.
template <typename AT>
__device__ __forceinline__ i32x4 step_fragment(const AT* row, int k, int width) {
  constexpr int KE = Elem<AT>::KE;
  if (k + KE <= width) return __builtin_bit_cast(i32x4, *(const u32x4_any*)(row + k));
  struct { AT v[KE]; } f;
#pragma unroll
  for (int e = 0; e < KE; ++e) f.v[e] = k + e < width ? row[k + e] : (AT)0.f;
  return __builtin_bit_cast(i32x4, f);
}

template <typename AT, int NT>
__global__ __launch_bounds__(kStepThreads) void k_lstm_step(const LstmStepParams p) {
  static_assert(2 * NT <= kStepWaves, "a wavefront per tile in the last part");
  using E = Elem<AT>;
  constexpr int KE = E::KE, KM = E::KM;
  __shared__ f32x4 red[kStepWaves][2 * NT][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int per_xcd = (int)gridDim.x / 8;
  const int r = ((int)blockIdx.x % 8) * per_xcd + (int)blockIdx.x / 8;  // (the grid is a multiple of 8: ids go round-robin to the XCDs)
  const int n = p.n, cell0 = r * kStepCells, b0 = (int)blockIdx.y * 16 * NT;
  if (cell0 >= n) return;
  const int i = lane & 15, kg = lane >> 4, gate = i & 3, cp = cell0 + 2 * (i >> 2);  // this lane's row of the two A tiles: gate of cells cp, cp + 1
  const int Sx = (p.in_dim + KM - 1) / KM, S = Sx + (n + KM - 1) / KM;
  // What the last part needs besides the sums, asked for now: a thread of wavefront `tile` finishes one (cell, row) pair.
  const int ft = min(wave, 2 * NT - 1), fb = b0 + 16 * (ft % NT) + i, fcell = cell0 + 2 * kg + ft / NT;
  const bool finishes = wave < 2 * NT && fb < p.B && fcell < n;
  const size_t fat = finishes ? (size_t)fb * n + fcell : 0;
  AT bias[4];
  float c_before = 0.f;
  if (finishes) {
    c_before = p.c[fat];
#pragma unroll
    for (int k = 0; k < 4; ++k) bias[k] = p.bias ? ((const AT*)p.bias)[(size_t)k * n + fcell] : (AT)0.f;
  }
  const AT* rc = (const AT*)p.rec + (size_t)gate * n + cp;
  typedef CellPair<AT> CP;
  const bool whole = cell0 + kStepCells <= n;
  f32x4 acc[2][NT];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[m][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int U = NT == 1 ? 4 : 2;  // macro steps whose loads are in flight together
  // the first macro step of h of this wavefront
  const int qh0 = wave + kStepWaves * ((max(0, Sx - wave) + kStepWaves - 1) / kStepWaves);
  if (p.by_fragments) {
    // Whole fragments and pairs only, and arrays that 32 bits address: every load is a buffer load whose offset is out of range where there
    // is nothing (0 comes back), and the first loads of rec leave together with those of x's weights.
    constexpr int ES = (int)sizeof(AT);
    const unsigned row_rec = 4u * n * ES;
    __amdgpu_buffer_rsrc_t rs_ff = __builtin_amdgcn_make_buffer_rsrc((void*)p.ff, 0, 4u * n * p.in_dim * ES, kBufFlags);
    __amdgpu_buffer_rsrc_t rs_rec = __builtin_amdgcn_make_buffer_rsrc((void*)p.rec, 0, n * row_rec, kBufFlags);
    __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, (unsigned)p.B * p.in_dim * ES, kBufFlags);
    __amdgpu_buffer_rsrc_t rs_h = __builtin_amdgcn_make_buffer_rsrc((void*)p.h, 0, (unsigned)p.B * n * ES, kBufFlags);
    auto frag = [](__amdgpu_buffer_rsrc_t rs, unsigned off) { return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0)); };
    unsigned off_a[2], off_x[NT], off_h[NT];
#pragma unroll
    for (int m = 0; m < 2; ++m) off_a[m] = (unsigned)((gate * n + cp + m) * p.in_dim + KE * kg) * ES;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int row = min(b0 + 16 * nt + i, p.B - 1);
      off_x[nt] = (unsigned)(row * p.in_dim + KE * kg) * ES;
      off_h[nt] = (unsigned)(row * n + KE * kg) * ES;
    }
    const unsigned off_r = (unsigned)(KE * kg) * row_rec + (unsigned)(gate * n + cp) * ES;
    i32x4 xa[U][2], xb[U][NT], hb[U][NT];
    typename CP::T hv[U][KE];
    auto load_x = [&](int q) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = KM * (q + kStepWaves * u);
        const bool there = k + KE * kg < p.in_dim;
#pragma unroll
        for (int m = 0; m < 2; ++m) xa[u][m] = frag(rs_ff, there ? off_a[m] + k * ES : 0x80000000u);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) xb[u][nt] = frag(rs_x, there ? off_x[nt] + k * ES : 0x80000000u);
      }
    };
    auto load_h = [&](int q) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = KM * (q - Sx + kStepWaves * u);
        const bool there = k + KE * kg < n;
        const unsigned at = there ? off_r + k * row_rec : 0x80000000u;
#pragma unroll
        for (int e = 0; e < KE; ++e) {
          if constexpr (ES == 2)
            hv[u][e] = __builtin_amdgcn_raw_buffer_load_b32(rs_rec, at, e * row_rec, 0);
          else
            hv[u][e] = __builtin_bit_cast(typename CP::T, __builtin_amdgcn_raw_buffer_load_b64(rs_rec, at, e * row_rec, 0));
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) hb[u][nt] = frag(rs_h, there ? off_h[nt] + k * ES : 0x80000000u);
      }
    };
    load_x(wave);
    load_h(qh0);
    for (int q = wave;;) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) acc[m][nt] = E::mma(xa[u][m], xb[u][nt], acc[m][nt]);
      if ((q += kStepWaves * U) >= Sx) break;
      load_x(q);
    }
    for (int q = qh0;;) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        i32x4 a[2];
        CP::fragments(hv[u], a[0], a[1]);
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) acc[m][nt] = E::mma(a[m], hb[u][nt], acc[m][nt]);
      }
      if ((q += kStepWaves * U) >= S) break;
      load_h(q);
    }
  } else {
  // rows of A beyond the width are any valid row (their results are dropped), so are rows of B beyond the batch
  const AT* fa[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) fa[m] = (const AT*)p.ff + ((size_t)gate * n + min(cp + m, n - 1)) * p.in_dim;
  const AT *xb[NT], *hb[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const size_t row = (size_t)min(b0 + 16 * nt + i, p.B - 1);
    xb[nt] = (const AT*)p.x + row * p.in_dim;
    hb[nt] = (const AT*)p.h + row * n;
  }
  int q = wave;
  for (; q < Sx; q += kStepWaves * U) {
    i32x4 a[U][2], b[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = KM * (q + kStepWaves * u) + KE * kg;  // (from in_dim on: zeros)
#pragma unroll
      for (int m = 0; m < 2; ++m) a[u][m] = step_fragment(fa[m], k, p.in_dim);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) b[u][nt] = step_fragment(xb[nt], k, p.in_dim);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[m][nt] = E::mma(a[u][m], b[u][nt], acc[m][nt]);
  }
  for (q = qh0; q < S; q += kStepWaves * U) {
    typename CP::T v[U][KE];
    i32x4 b[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = KM * (q - Sx + kStepWaves * u) + KE * kg;
#pragma unroll
      for (int e = 0; e < KE; ++e) {
        v[u][e] = 0;
        if (k + e < n) {
          const AT* src = rc + (size_t)(k + e) * 4 * n;
          if (whole)
            v[u][e] = *(const typename CP::T_any*)src;
          else if (cp < n)
            v[u][e] = CP::make(src[0], cp + 1 < n ? src[1] : (AT)0.f);
        }
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) b[u][nt] = step_fragment(hb[nt], k, n);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      i32x4 a[2];
      CP::fragments(v[u], a[0], a[1]);
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[m][nt] = E::mma(a[m], b[u][nt], acc[m][nt]);
    }
  }
  }
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) red[wave][m * NT + nt][lane] = acc[m][nt];
  __syncthreads();
  if (finishes) {
    f32x4 g = red[0][ft][lane];
#pragma unroll
    for (int w = 1; w < kStepWaves; ++w) g += red[w][ft][lane];
    if (p.bias) {
#pragma unroll
      for (int k = 0; k < 4; ++k) g[k] += (float)bias[k];
    }
    const float c = c_before * Act<AT>::sigmoid(g[2]) + Act<AT>::tanh(g[0]) * Act<AT>::sigmoid(g[1]);
    const float y = Act<AT>::tanh(c) * Act<AT>::sigmoid(g[3]);
    p.c_out[fat] = c;
    E::store(p.y, fat, y);
    E::store(p.h_out, fat, y);
  }
}

}  // namespace rtn
