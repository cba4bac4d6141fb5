// gfx950 kernels of the weight gradients: C = A^T B with few columns and very many rows.
#pragma once

#include <hip/hip_runtime.h>

#include "lstm2_kernels.h"

namespace rtn {

// ---------------------------------------------------------------------------------------------------------------
// DW[n,4n] = sum over frames and sequences of Y[row]^T DX[row], plus y0^T dx0: the matrices are [T B, n] and [T B, 4n].  For small
// layers the product has a few tiles of output and ten thousands of rows, and a library product that gives a workgroup a tile leaves
// most of the chip idle.  Here the rows are dealt to slices, a workgroup takes 64 x 64 of the output of one slice, and a second
// kernel adds the slices' results; y0^T dx0 is one slice more.  (The gradient of the input's weights, DX^T source, is such a product too.)
//
// A and B are used as they lie: v_mfma_f32_16x16x4 takes ONE k per lane group, so lane (kg, i) needs row k + kg at column i, and with
// four neighbouring columns per lane one load of 16 bytes (8 in bf16, widened: the products are exact) is the operand of four tiles, whose columns are then
// 4 apart: tile t has columns 4 i + t.  Four rows are 2 loads for 16 MFMAs of 32 clocks, no LDS, no transposition.  The four wavefronts take
// every fourth four rows and add their tiles through LDS.  A slice's workgroups are on one XCD (slice = id % slices), whose L2 they share.
// Bound by the float32 matrix rate from n = 256 on (26 GFLOP at n = 256, T B = 49 750: 202 ... 255 us, the matrix cores busy for 95 % of it; the library's
// best rate, 152 TFLOP/s, would be 172), below by the two launches.
// Measured (gradient op with the recurrence, us, library / this): float32 n = 128, T = 300, B = 100 804 / 437, n = 256 937 / 662; bf16 n = 64 422 / 333,
// n = 128 474 / 399, T = 20, B = 4 61 / 40.  Largest error against float64, of the largest element, for n = 64 ... 384 and 80 ... 50 000 rows: float32 7e-7 ...
// 31e-7 / 1.3e-7 ... 8.3e-7, bf16 inputs 0.9e-7 ... 16e-7 / 0.9e-7 ... 4.1e-7.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kWeightTile = 64;       // columns of A and of B per workgroup
constexpr int kWeightAhead = 4;       // steps of 16 rows whose loads are in flight together
constexpr int kMaxWeightCalls = 2;
constexpr unsigned kNoColumn = 0x80000000u;  // an offset that stays out of range while rows are stepped over (those of a slice end below 2^30)
struct WeightGradCall {
  const void *a[2], *b[2];            // [rows][m], [rows][n]: the long product's and the other's
  long long rows[2], lda[2], ldb[2];  // elements from one row to the next
  float* part;                        // [parts][m][n]
  void* out;                          // [m][n]
  int add;                            // k_weight_last: out = part + A^T B
};
struct WeightGradArgs {
  int m, n;                           // m: a multiple of 4
  int slices;                         // of the long product
  int parts;                          // slices, and one more for the other product
  long long slice_rows;
  WeightGradCall call[kMaxWeightCalls];
};

// Four neighbouring elements, as one load brings them.
template <typename AT>
struct FourOf {
  typedef std::conditional_t<sizeof(AT) == 4, u32x4, u32x2> T;
  static __device__ __forceinline__ T load(__amdgpu_buffer_rsrc_t rs, unsigned at) {
    if constexpr (sizeof(AT) == 4)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0));
    else
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rs, at, 0, 0));
  }
  static __device__ __forceinline__ float get(T v, int k) {
    if constexpr (sizeof(AT) == 4)
      return __builtin_bit_cast(float, (unsigned)v[k]);
    else
      return __builtin_bit_cast(float, k & 1 ? v[k >> 1] & 0xFFFF0000u : v[k >> 1] << 16);
  }
};

// ANY: n, and the distance between the rows of B, need not be multiples of 4: B comes in and the result goes out by element.
template <typename AT, bool ANY>
__global__ __launch_bounds__(kWgThreads) void k_weight_grad(const WeightGradArgs args) {
  constexpr int ES = (int)sizeof(AT);
  typedef typename FourOf<AT>::T Quad4;
  __shared__ f32x4 red[kWaves][16][64];
  const WeightGradCall& q = args.call[blockIdx.y];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), kg = lane >> 4, i = lane & 15;
  const int tiles_m = (args.m + kWeightTile - 1) / kWeightTile, tiles = tiles_m * ((args.n + kWeightTile - 1) / kWeightTile);
  const bool other = (int)blockIdx.x >= tiles * args.slices;
  const int which = other ? 1 : 0, slice = other ? 0 : (int)blockIdx.x % args.slices, tile = other ? (int)blockIdx.x - tiles * args.slices : (int)blockIdx.x / args.slices;
  const int m0 = kWeightTile * (tile % tiles_m), n0 = kWeightTile * (tile / tiles_m);
  const long long first = other ? 0 : slice * args.slice_rows;
  const int rows = (int)max(0LL, min(other ? q.rows[1] : args.slice_rows, q.rows[which] - first));
  const unsigned pitch_a = (unsigned)(q.lda[which] * ES), pitch_b = (unsigned)(q.ldb[which] * ES);
  // (rows behind the slice lie behind the buffer, and so do lanes whose columns do not exist: zeros come back)
  __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)q.a[which] + first * q.lda[which] * ES, 0, rows > 0 ? (rows - 1) * pitch_a + args.m * ES : 0u, kBufFlags);
  __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)q.b[which] + first * q.ldb[which] * ES, 0, rows > 0 ? (rows - 1) * pitch_b + args.n * ES : 0u, kBufFlags);
  unsigned at_each[ANY ? 4 : 1];
  if constexpr (ANY) {
#pragma unroll
    for (int k = 0; k < 4; ++k) at_each[k] = n0 + 4 * i + k < args.n ? (4 * wave + kg) * pitch_b + (n0 + 4 * i + k) * ES : kNoColumn;
  }
  unsigned at_a = m0 + 4 * i < args.m ? (4 * wave + kg) * pitch_a + (m0 + 4 * i) * ES : kNoColumn, at_b = n0 + 4 * i < args.n ? (4 * wave + kg) * pitch_b + (n0 + 4 * i) * ES : kNoColumn;
  const unsigned step_a = 4 * kWaves * pitch_a, step_b = 4 * kWaves * pitch_b;
  f32x4 acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  Quad4 va[2][kWeightAhead], vb[2][ANY ? 1 : kWeightAhead];
  u32x4 each[2][ANY ? kWeightAhead : 1];  // (as the loads bring them)
  auto fetch = [&](auto set_tag) {
    constexpr int S = decltype(set_tag)::value;
#pragma unroll
    for (int u = 0; u < kWeightAhead; ++u) {
      va[S][u] = FourOf<AT>::load(ra, at_a);
      if constexpr (ANY) {
        unsigned v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if constexpr (ES == 4)
            v[k] = __builtin_amdgcn_raw_buffer_load_b32(rb, at_each[k], 0, 0);
          else
            v[k] = __builtin_amdgcn_raw_buffer_load_b16(rb, at_each[k], 0, 0);
          at_each[k] += step_b;
        }
        each[S][u] = u32x4{v[0], v[1], v[2], v[3]};
      } else {
        vb[S][u] = FourOf<AT>::load(rb, at_b);
        at_b += step_b;
      }
      at_a += step_a;
    }
  };
  auto multiply = [&](auto set_tag) {
    constexpr int S = decltype(set_tag)::value;
#pragma unroll
    for (int u = 0; u < kWeightAhead; ++u)
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          float right;
          if constexpr (ANY)
            right = __builtin_bit_cast(float, ES == 4 ? (unsigned)each[S][u][b] : (unsigned)each[S][u][b] << 16);
          else
            right = FourOf<AT>::get(vb[S][u], b);
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(FourOf<AT>::get(va[S][u], a), right, acc[a][b], 0, 0, 0);
        }
  };
  constexpr int kRows = 4 * kWaves * kWeightAhead;
  // entry 4 a + r of a lane: row 4 (4 kg + r) + a of the tile, columns 4 i ... 4 i + 3
  auto row_of = [&](int entry) { return m0 + 4 * (4 * kg + (entry & 3)) + (entry >> 2); };
  const int col = n0 + 4 * i;
  fetch(IntTag<0>{});
  for (int r = 0; r < rows; r += 2 * kRows) {
    fetch(IntTag<1>{});
    multiply(IntTag<0>{});
    fetch(IntTag<0>{});
    multiply(IntTag<1>{});
  }
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][4 * a + r][lane] = f32x4{acc[a][0][r], acc[a][1][r], acc[a][2][r], acc[a][3][r]};
  __syncthreads();
  float* out = q.part + (size_t)(other ? args.slices : slice) * args.m * args.n;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int entry = 4 * wave + e, row = row_of(entry);
    const f32x4 sum = ((red[0][entry][lane] + red[1][entry][lane]) + red[2][entry][lane]) + red[3][entry][lane];
    if constexpr (ANY) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (row < args.m && col + k < args.n) out[(size_t)row * args.n + col + k] = sum[k];
    } else {
      if (row < args.m && col < args.n) *(f32x4*)(out + (size_t)row * args.n + col) = sum;
    }
  }
}

// out = A^T B of few rows (a[0], b[0]), plus what is in part if the call says so: the last frame's share y0^T dx0 of a wide layer's gradient, whose
// long product is the library's, and the conversion to the parameter's type, in one pass over DW for all directions.  Every wavefront has a tile of
// 32 x 64 of its own, asks for what is there first, multiplies meanwhile (operands as above, two neighbouring columns of A per lane) and writes 16 bytes
// (8 in bf16) per lane, 256 (128) of a row together.  Bound by that pass (101 MB at bf16 n = 2048: 20 us) and the float32 matrix rate (14 us at 64
// rows); 33.5 us, with tiles of 64 x 64 and half the wavefronts 40, with a tile per workgroup, its rows dealt to the wavefronts and added
// through LDS, 47; library product and conversion 45.  Both directions of float32 n = 500, 40 rows: 8.4 us, 11.1, 8.1 and 14.6.
template <typename AT, typename OT>
__global__ __launch_bounds__(kWgThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_weight_last(const WeightGradArgs args) {
  constexpr int ES = (int)sizeof(AT);
  typedef typename FourOf<AT>::T Quad4;
  typedef std::conditional_t<ES == 4, u32x2, unsigned> Pair;
  const WeightGradCall& q = args.call[blockIdx.y];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), kg = lane >> 4, i = lane & 15;
  const int tiles_n = (args.n + kWeightTile - 1) / kWeightTile, tile = (int)blockIdx.x * kWaves + wave;
  const int m0 = 32 * (tile / tiles_n), n0 = kWeightTile * (tile % tiles_n);
  if (m0 >= args.m) return;
  const int rows = (int)q.rows[0], col = n0 + 4 * i;
  auto row_of = [&](int a, int r) { return m0 + 2 * (4 * kg + r) + a; };
  f32x4 before[2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      before[a][r] = q.add && row_of(a, r) < args.m && col < args.n ? *(const f32x4*)(q.part + (size_t)row_of(a, r) * args.n + col) : f32x4{0.f, 0.f, 0.f, 0.f};
  const unsigned pitch_a = (unsigned)(q.lda[0] * ES), pitch_b = (unsigned)(q.ldb[0] * ES);
  __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)q.a[0], 0, rows > 0 ? (rows - 1) * pitch_a + args.m * ES : 0u, kBufFlags);
  __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void*)q.b[0], 0, rows > 0 ? (rows - 1) * pitch_b + args.n * ES : 0u, kBufFlags);
  unsigned at_a = m0 + 2 * i < args.m ? kg * pitch_a + (m0 + 2 * i) * ES : kNoColumn, at_b = col < args.n ? kg * pitch_b + col * ES : kNoColumn;
  auto left = [](Pair v, int k) {
    if constexpr (ES == 4)
      return __builtin_bit_cast(float, (unsigned)v[k]);
    else
      return __builtin_bit_cast(float, k ? v & 0xFFFF0000u : v << 16);
  };
  f32x4 acc[2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  Pair va[2][kWeightAhead];
  Quad4 vb[2][kWeightAhead];
  auto fetch = [&](auto set_tag) {
    constexpr int S = decltype(set_tag)::value;
#pragma unroll
    for (int u = 0; u < kWeightAhead; ++u) {
      if constexpr (ES == 4)
        va[S][u] = __builtin_bit_cast(Pair, __builtin_amdgcn_raw_buffer_load_b64(ra, at_a, 0, 0));
      else
        va[S][u] = __builtin_amdgcn_raw_buffer_load_b32(ra, at_a, 0, 0);
      vb[S][u] = FourOf<AT>::load(rb, at_b);
      at_a += 4 * pitch_a;
      at_b += 4 * pitch_b;
    }
  };
  auto multiply = [&](auto set_tag) {
    constexpr int S = decltype(set_tag)::value;
#pragma unroll
    for (int u = 0; u < kWeightAhead; ++u)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(left(va[S][u], a), FourOf<AT>::get(vb[S][u], b), acc[a][b], 0, 0, 0);
  };
  constexpr int kRows = 4 * kWeightAhead;
  fetch(IntTag<0>{});
  for (int r = 0; r < rows; r += 2 * kRows) {
    fetch(IntTag<1>{});
    multiply(IntTag<0>{});
    fetch(IntTag<0>{});
    if (r + kRows < rows) multiply(IntTag<1>{});
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (row_of(a, r) >= args.m || col >= args.n) continue;
      const f32x4 all = before[a][r] + f32x4{acc[a][0][r], acc[a][1][r], acc[a][2][r], acc[a][3][r]};
      typedef OT Four __attribute__((ext_vector_type(4)));
      *(Four*)((OT*)q.out + (size_t)row_of(a, r) * args.n + col) = __builtin_convertvector(all, Four);
    }
}

// out := the sum of the parts, four elements per lane; the wavefronts take every fourth part.
template <typename OT>
__global__ __launch_bounds__(kWgThreads) void k_weight_grad_sum(const WeightGradArgs args) {
  __shared__ f32x4 red[kWaves][64];
  const WeightGradCall& q = args.call[blockIdx.y];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const long long quads = (long long)args.m * args.n / 4, at = blockIdx.x * 64LL + lane;
  f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
  if (at < quads)
#pragma unroll 8
    for (int s = wave; s < args.parts; s += kWaves) sum += ((const f32x4*)q.part)[s * quads + at];
  red[wave][lane] = sum;
  __syncthreads();
  if (wave == 0 && at < quads) {
    const f32x4 all = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
    if constexpr (sizeof(OT) == 4) {
      ((f32x4*)q.out)[at] = all;
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) Elem<OT>::store(q.out, 4 * at + k, all[k]);
    }
  }
}

}  // namespace rtn
