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
// five launches of 38 us together, and 123 us per call; one launch of 8.9 us and 16.3 us per call now.  (Every 64 rows read all weights:
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
  const AT* rc = (const AT*)p.rec + (size_t)gate * n + cp;
  f32x4 acc[2][NT];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[m][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int U = NT == 1 ? 4 : 2;  // macro steps whose loads are in flight together
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
  // the first macro step of h of this wavefront (x's last turn may have gone past Sx by whole turns of the unrolled loop)
  q = wave + kStepWaves * ((max(0, Sx - wave) + kStepWaves - 1) / kStepWaves);
  typedef CellPair<AT> CP;
  const bool whole = cell0 + kStepCells <= n;
  for (; q < S; q += kStepWaves * U) {
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
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) red[wave][m * NT + nt][lane] = acc[m][nt];
  __syncthreads();
  for (int t = tid; t < 2 * NT * 64; t += kStepThreads) {
    const int tile = t >> 6, l = t & 63;
    f32x4 g = red[0][tile][l];
#pragma unroll
    for (int w = 1; w < kStepWaves; ++w) g += red[w][tile][l];
    const int b = b0 + 16 * (tile % NT) + (l & 15), cell = cell0 + 2 * (l >> 4) + tile / NT;
    if (b >= p.B || cell >= n) continue;
    if (p.bias) {
#pragma unroll
      for (int k = 0; k < 4; ++k) g[k] += E::load(p.bias, (size_t)k * n + cell);
    }
    const size_t at = (size_t)b * n + cell;
    const float c = p.c[at] * Act<AT>::sigmoid(g[2]) + Act<AT>::tanh(g[0]) * Act<AT>::sigmoid(g[1]);
    const float y = Act<AT>::tanh(c) * Act<AT>::sigmoid(g[3]);
    p.c_out[at] = c;
    E::store(p.y, at, y);
    E::store(p.h_out, at, y);
  }
}

}  // namespace rtn
