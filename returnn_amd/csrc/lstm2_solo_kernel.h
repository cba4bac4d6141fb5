// gfx950 kernel of the forward recurrence for layers whose recurrent weights fit the registers of ONE compute unit.
#pragma once

#include <hip/hip_runtime.h>

#include "lstm2_kernels.h"

namespace rtn {

// ---------------------------------------------------------------------------------------------
// A step of a small layer (n = 64 in float32: 64 KB of weights, 0.2 us of MFMAs on one CU) is shorter than one hand-over
// between workgroups (0.4 us and more), so nothing is handed over: a workgroup takes its batch rows through all steps by
// itself, W in its registers, h in LDS, one barrier per step.  Workgroups know nothing of each other: no packing of W, no
// ring, no waits, any number of them.
//
// Such a step is one chain (h from LDS, the product, the gates, h to LDS, a barrier) and its length is instructions issued,
// so while there are CUs to spare a workgroup has ONE row (k_lstm2_solo_row) and a lane one gate of a cell instead of four: a fourth of the
// product and two fifths of the non-linearities; up to four rows share one (k_lstm2_solo) where CUs run short.
//
// A wavefront owns 16 cells, all four gates of them, and the whole contraction; the lane that ends up with a (row, cell)
// pair has its four gates.  4 rows per workgroup: one pair per lane, and more rows would lengthen the pointwise part, which
// is half of the step, while B / 4 workgroups find a CU each up to 1024 rows.  One row: lane 4 c + q has gate q of cell c.
//  * float32: v_mfma_f32_4x4x1 -- 16 blocks of 4 rows x 4 columns; A (h) of block k is broadcast to all of them, so that one
//    instruction takes 4 rows x 64 gate columns x one k in 8 clocks (a 16x16x4 tile spends three quarters of its 32 clocks on
//    rows that do not exist).  The results lie gate by gate in the lanes of a quad and are transposed there.  One row: a multiply-add of
//    4 clocks for the 64 columns of one k.
//  * bf16: v_mfma_f32_16x16x32 on tiles of 4 cells, four tiles in ONE accumulator: tile t's B operand has the four rows
//    in columns 4 t ... 4 t + 3 and zeros elsewhere (one row: in all four of them).
// The order of additions per element is that of the other kernels (their four wavefronts' shares of k are four
// accumulators here), so the results are theirs bit for bit.
// Measured, us per step (T = 300, 4 rows; four rows per workgroup / one): float32 n = 32 0.64 / 0.44, n = 64 0.74 / 0.51; bf16 n = 32 0.41 / 0.29,
// n = 64 0.62 / 0.38, n = 96 0.71 / 0.60, n = 128 0.87 / 0.73.  float32 against k_lstm2_regw: n = 96 1.07 / 0.88, n = 128 1.06 / 1.01, with 256 rows
// 1.37 / 0.91 and 1.39 / 1.07.  One call with T = 32, B = 4, n = 64: 45 us with packing (5.3) and k_lstm2_regw (36.5), 27 with four rows per workgroup, 20 with one.
// All of these with library functions in the float32 gates; one row without: n = 32 0.36, 64 0.45, 96 0.84, 128 0.99, the call 18.2 us; with one exponential and one
// reciprocal for whichever gate a lane has: 0.34, 0.43, 0.81, 0.96 and 17.5.  (h as one read of all macro steps' elements per lane: 0.35, 0.44, 0.81, 0.95 and 17.8.)
// ---------------------------------------------------------------------------------------------
constexpr int kSoloRows = 4;
constexpr int kSoloCells = 16;  // cells per wavefront
constexpr int kSoloAhead = 4;   // sets of gate inputs: the loads of a step's are issued three steps before it

// S: macro steps of the contraction, which with it gives the width: wavefronts = S (float32) or 2 S (bf16).
template <typename AT>
constexpr int solo_waves(int S) { return S * Elem<AT>::KM / kSoloCells; }

// k = 0 ... 15 of macro steps 4 j ... 4 j + 3, in the order in which a 16x16x4 MFMA of fragments of 4 takes them (0, 4, 8, 12,
// 1, 5, ...); the four macro steps go to four accumulators, which hides the MFMA's latency.
template <int S, int J, int... I>
__device__ __forceinline__ void solo_mfma_f32(const float (&h)[S], const float (&w)[16 * S], f32x4 (&acc)[4], std::integer_sequence<int, I...>) {
  (([&] {
     constexpr int k = (I >> 2) + 4 * (I & 3);
#pragma unroll
     for (int v = 0; v < 4; ++v)
       if (4 * J + v < S) acc[v] = mfma_4x4x1<k>(h[4 * J + v < S ? 4 * J + v : 0], w[16 * (4 * J + v < S ? 4 * J + v : 0) + k], acc[v]);
   }()),
   ...);
}
template <int S, int... J>
__device__ __forceinline__ void solo_mfma_f32_all(const float (&h)[S], const float (&w)[16 * S], f32x4 (&acc)[4], std::integer_sequence<int, J...>) {
  (solo_mfma_f32<S, J>(h, w, acc, std::make_integer_sequence<int, 16>{}), ...);
}

// W of this wavefront's cells.  float32: a lane's column is gate lane % 4 of cell lane / 4, one register per k.  bf16: row
// i = lane % 16 of tile t is gate i % 4 of cell 4 (i / 4) + t: a lane loads four neighbouring cells at once.  (What lies
// beyond the width is loaded from inside and replaced by zeros: no branches between the loads.)
// CLAMP: cells beyond the width are copies of one inside (solo_cell).
template <typename AT, int S, bool CLAMP>
__device__ __forceinline__ void solo_weights(const void* W, int nc, int wave, int lane, float (&wf)[sizeof(AT) == 4 ? 16 * S : 1], i32x4 (&wb)[sizeof(AT) == 4 ? 1 : 4][sizeof(AT) == 4 ? 1 : S]) {
  constexpr int KM = Elem<AT>::KM;
  if constexpr (sizeof(AT) == 4) {
    const int wcell = kSoloCells * wave + (lane >> 2);
    const float* src = (const float*)W + (size_t)(lane & 3) * nc + min(wcell, nc - 1);
#pragma unroll
    for (int k = 0; k < 16 * S; ++k) wf[k] = src[(size_t)min(k, nc - 1) * 4 * nc];
#pragma unroll
    for (int k = 0; k < 16 * S; ++k) wf[k] = k < nc && (CLAMP || wcell < nc) ? wf[k] : 0.f;
  } else {
    const int i = lane & 15, kg = lane >> 4, wcell = kSoloCells * wave + 4 * (i >> 2);
    typedef unsigned long long u64_any __attribute__((aligned(2)));
    const unsigned short* src = (const unsigned short*)W + (size_t)(i & 3) * nc;
    const bool whole = nc % 4 == 0;  // (no lane's four cells are cut)
#pragma unroll
    for (int s = 0; s < S; ++s) {
      unsigned long long v[8];
      if (whole) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = *(const u64_any*)(src + (size_t)min(KM * s + 8 * kg + e, nc - 1) * 4 * nc + min(wcell, nc - 4));
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = KM * s + 8 * kg + e < nc && (CLAMP || wcell < nc) ? v[e] : 0;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int k = KM * s + 8 * kg + e;
          v[e] = 0;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const unsigned long long x = src[(size_t)min(k, nc - 1) * 4 * nc + min(wcell + c, nc - 1)];
            v[e] |= (k < nc && (CLAMP || wcell + c < nc) ? x : 0) << (16 * c);
          }
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int w = 0; w < 4; ++w)
          wb[t][s][w] = (int)(((unsigned)(v[2 * w] >> (16 * t)) & 0xFFFFu) | ((unsigned)(v[2 * w + 1] >> (16 * t)) << 16));
    }
  }
}

// bf16: the accumulator of tile t's product with macro step i of h.  A column's products are all in one tile, so with one or two macro
// steps a step's tiles can have accumulators of their own: the others' are zero there and the sum over the four is the same.
template <int S>
constexpr int solo_acc(int t, int i) { return S == 1 ? t : S == 2 ? 2 * i + (t & 1) : i & 3; }

// One row per workgroup.  float32: the row against a lane's column of W, a multiply-add for every k; lane k of every 16 holds
// element k of a macro step of h, and the instruction itself broadcasts it to the 16 (row_newbcast).  The order of additions is that of the
// MFMAs.  In assembly, since the compiler makes two instructions of a multiply-add of a lane's broadcast; one block, since a lane
// operand must not be read in the two instructions after a vector instruction that wrote it: the wait is in front of the first.
#define RTN_FMA(v, k) "v_fmac_f32_dpp %[a" #v "], %[h" #v "], %[w" #v "_" #k "] row_newbcast:" #k " row_mask:0xf bank_mask:0xf\n\t"
#define RTN_FMA2(k) RTN_FMA(0, k) RTN_FMA(1, k)
#define RTN_FMA4(k) RTN_FMA2(k) RTN_FMA(2, k) RTN_FMA(3, k)
#define RTN_FMAS(m) m(0) m(4) m(8) m(12) m(1) m(5) m(9) m(13) m(2) m(6) m(10) m(14) m(3) m(7) m(11) m(15)
#define RTN_W1(v, k) [w##v##_##k] "v"(w[16 * v + k])
#define RTN_W(v) RTN_W1(v, 0), RTN_W1(v, 1), RTN_W1(v, 2), RTN_W1(v, 3), RTN_W1(v, 4), RTN_W1(v, 5), RTN_W1(v, 6), RTN_W1(v, 7), RTN_W1(v, 8), \
    RTN_W1(v, 9), RTN_W1(v, 10), RTN_W1(v, 11), RTN_W1(v, 12), RTN_W1(v, 13), RTN_W1(v, 14), RTN_W1(v, 15)
__device__ __forceinline__ void solo_fma2(const float* h, const float* w, float (&acc)[4]) {
  asm("s_nop 1\n\t" RTN_FMAS(RTN_FMA2) : [a0] "+&v"(acc[0]), [a1] "+&v"(acc[1]) : [h0] "v"(h[0]), [h1] "v"(h[1]), RTN_W(0), RTN_W(1));
}
__device__ __forceinline__ void solo_fma4(const float* h, const float* w, float (&acc)[4]) {
  asm("s_nop 1\n\t" RTN_FMAS(RTN_FMA4)
      : [a0] "+&v"(acc[0]), [a1] "+&v"(acc[1]), [a2] "+&v"(acc[2]), [a3] "+&v"(acc[3])
      : [h0] "v"(h[0]), [h1] "v"(h[1]), [h2] "v"(h[2]), [h3] "v"(h[3]), RTN_W(0), RTN_W(1), RTN_W(2), RTN_W(3));
}
#undef RTN_FMA
#undef RTN_FMA2
#undef RTN_FMA4
#undef RTN_FMAS
#undef RTN_W1
#undef RTN_W
template <int S>
__device__ __forceinline__ void solo_fma_all(const float (&h)[S], const float (&w)[16 * S], float (&acc)[4]) {
  static_assert(S % 2 == 0, "blocks of two and four macro steps");
#pragma unroll
  for (int i = 0; i + 4 <= S; i += 4) solo_fma4(h + i, w + 16 * i, acc);
  if constexpr (S % 4 == 2) solo_fma2(h + S - 2, w + 16 * (S - 2), acc);
}
// The cell whose weights solo_weights<CLAMP> gives to a cell beyond the width.
template <typename AT>
__device__ __forceinline__ int solo_cell(int cell, int nc) { return cell < nc ? cell : sizeof(AT) == 2 && nc % 4 == 0 ? nc - 4 + (cell & 3) : nc - 1; }
// Lane Q of a quad, to all four.
template <int Q>
__device__ __forceinline__ float quad_lane(float v) { return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x55 * Q, 0xF, 0xF, true)); }
// The non-linearity of a lane's gate: tanh of the first, sigmoid of the others.
template <typename AT>
__device__ __forceinline__ float solo_gate(float x, bool first) {
  if constexpr (sizeof(AT) == 4) {
    const float e = exp_f32(first ? tanh_exponent(x) : sigmoid_exponent(x)), d = 1.f + e, q = reciprocal_f32(d);  // (one of each for both)
    const float t = tanh_of(x, q), s = sigmoid_of(x, e, d, q);
    return first ? t : s;
  } else {  // Act<__bf16>'s two with one exponential and one reciprocal
    const float r = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f((first ? -2.8853900817779268f : -1.4426950408889634f) * x));
    return first ? __builtin_fmaf(2.f, r, -1.f) : r;
  }
}

// (Two wavefronts per SIMD allowed for, which none of the builds needs more registers than: the compiler then keeps the
// accumulators in the vector registers the pointwise part reads them from.)
template <typename AT, int S>
__global__ __launch_bounds__(64 * solo_waves<AT>(S)) __attribute__((amdgpu_waves_per_eu(2))) void k_lstm2_solo(const Lstm2Multi multi) {
  using E = Elem<AT>;
  constexpr int KM = E::KM, ES = (int)sizeof(AT);
  constexpr bool F32 = ES == 4;
  const Lstm2Params p = multi.p[blockIdx.y];
  __shared__ __align__(16) unsigned char hbuf[2][S * KM * kSoloRows * ES];  // h, one buffer per parity of the step

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nc = p.nc, nsteps = p.nsteps;
  const int b_base = (int)blockIdx.x * kSoloRows, rows = min(kSoloRows, p.B - b_base);
  const long long bn = (long long)p.B * nc;
  if (blockIdx.x == 0 && tid < 64) p.status[tid] = status_word(tid, p.abort_word, p.abort_id);

  // The pair of this lane.
  const int row = lane & 3, cell = kSoloCells * wave + (F32 ? lane >> 2 : 4 * (lane >> 4) + ((lane >> 2) & 3));
  const bool valid = row < rows && cell < nc;
  const unsigned h_put = F32 ? (unsigned)((cell * kSoloRows + row) * 4) : (unsigned)(((cell / 8) * kSoloRows + row) * 16 + (cell % 8) * 2);
  float c_state = 0.f, h_prev = 0.f;
  if (valid) {
    const long long bc = (long long)(b_base + row) * nc + cell;
    c_state = p.c0[bc];
    h_prev = E::load(p.y0, bc);
  }
  *(AT*)(hbuf[0] + h_put) = (AT)h_prev;  // (rows and cells that do not exist stay 0)

  // The op's streams, as buffer accesses without a branch: pairs and frames that do not exist have offsets beyond any frame.
  const long long brow = b_base + row;
  const unsigned x_at = valid ? (unsigned)((brow * p.ldX + cell) * ES) : kOobOffset, h_at = valid ? (unsigned)((brow * 4 * nc + cell) * ES) : kOobOffset,
                 y_at = valid ? (unsigned)((brow * p.ldY + cell) * ES) : kOobOffset, c_at = valid ? (unsigned)((brow * nc + cell) * 4) : kOobOffset,
                 m_at = row < rows ? (unsigned)(brow * 4) : kOobOffset;
  const unsigned frame_x = (unsigned)((size_t)p.B * p.ldX * ES), frame_h = (unsigned)((size_t)p.B * 4 * nc * ES), frame_y = (unsigned)((size_t)p.B * p.ldY * ES),
                 frame_c = (unsigned)(bn * 4), frame_m = (unsigned)(p.B * 4), gate = (unsigned)(nc * ES);
  auto frame = [&](const void* base, int s, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((unsigned char*)base + frame_of(p, s) * (long long)bytes, 0, bytes, kBufFlags);
  };
  AT xin[kSoloAhead][4];
  float msk[kSoloAhead];
  auto fetch = [&](int s, auto slot_tag) {
    constexpr int K = decltype(slot_tag)::value;
    const bool there = s < nsteps;
    const int f = there ? s : 0;  // (a frame that exists: only the offsets decide)
    __amdgpu_buffer_rsrc_t xr = frame(p.X, f, frame_x), mr = frame(p.mask, f, frame_m);
    const unsigned at = there ? x_at : kOobOffset;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if constexpr (F32)
        xin[K][q] = __builtin_bit_cast(AT, __builtin_amdgcn_raw_buffer_load_b32(xr, at, q * gate, 0));
      else
        xin[K][q] = __builtin_bit_cast(AT, __builtin_amdgcn_raw_buffer_load_b16(xr, at, q * gate, 0));
    }
    msk[K] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(mr, there ? m_at : kOobOffset, 0, 0));
  };
  AT a_out[4], y_out = (AT)0.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) a_out[q] = (AT)0.f;
  auto put = [&](int s) {
    const bool there = s >= 0;
    const int f = there ? s : 0;
    __amdgpu_buffer_rsrc_t hr = frame(p.H, f, frame_h), yr = frame(p.Y, f, frame_y), cr = frame(p.C, f, frame_c);
    auto store = [&](AT v, __amdgpu_buffer_rsrc_t rs, unsigned off, unsigned block) {
      if constexpr (F32)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rs, off, block, 0);
      else
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), rs, off, block, 0);
    };
#pragma unroll
    for (int q = 0; q < 4; ++q) store(a_out[q], hr, there ? h_at : kOobOffset, q * gate);
    store(y_out, yr, there ? y_at : kOobOffset, 0);
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, c_state), cr, there ? c_at : kOobOffset, 0, 0);
  };

  fetch(0, IntTag<0>{});
  fetch(1, IntTag<1>{});
  fetch(2, IntTag<2>{});
  float wf[F32 ? 16 * S : 1];
  i32x4 wb[F32 ? 1 : 4][F32 ? 1 : S];
  solo_weights<AT, S, false>(p.W, nc, wave, lane, wf, wb);

  auto step = [&](int s, auto slot_tag) {
    constexpr int K = decltype(slot_tag)::value;
    const unsigned char* hb = hbuf[K & 1];
    f32x4 acc[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (F32) {
      float h[S];
#pragma unroll
      for (int i = 0; i < S; ++i) h[i] = *(const float*)(hb + i * 256 + lane * 4);
      put(s - 1);  // (these two in the shadow of the LDS reads and of the MFMAs)
      fetch(s + kSoloAhead - 1, IntTag<(K + kSoloAhead - 1) % kSoloAhead>{});
      solo_mfma_f32_all<S>(h, wf, acc, std::make_integer_sequence<int, (S + 3) / 4>{});
    } else {
      i32x4 h[S];
#pragma unroll
      for (int i = 0; i < S; ++i) h[i] = *(const i32x4*)(hb + (((4 * i + (lane >> 4)) * kSoloRows) + (lane & 3)) * 16);
      put(s - 1);
      fetch(s + kSoloAhead - 1, IntTag<(K + kSoloAhead - 1) % kSoloAhead>{});
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int keep = ((lane >> 2) & 3) == t ? -1 : 0;
#pragma unroll
        for (int i = 0; i < S; ++i) {
          const i32x4 b = i32x4{h[i][0] & keep, h[i][1] & keep, h[i][2] & keep, h[i][3] & keep};
          const int a = solo_acc<S>(t, i);
          acc[a] = E::mma(wb[t][i], b, acc[a]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < (F32 ? 16 * S : 4 * S); ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                // an MFMA ...
      __builtin_amdgcn_sched_group_barrier(0x076, F32 ? 1 : 3, 0);  // ... and what fits behind it of everything else but LDS
    }
    f32x4 g = acc[0];
#pragma unroll
    for (int v = 1; v < 4; ++v) g += acc[v];
    if constexpr (F32) g = quad_transpose(g, lane);
    const float m = msk[K];
    const float a0 = Act<AT>::tanh(g[0] + (float)xin[K][0]);
    const float a1 = Act<AT>::sigmoid(g[1] + (float)xin[K][1]);
    const float a2 = Act<AT>::sigmoid(g[2] + (float)xin[K][2]);
    const float a3 = Act<AT>::sigmoid(g[3] + (float)xin[K][3]);
    const float pc = c_state;
    const float c = (pc * a2 + a0 * a1) * m + pc * (1.f - m);
    const float y = E::round(Act<AT>::tanh(c) * a3 * m);
    const float hn = (p.op_flags & kOpNoCarry) ? y : E::round(y + h_prev * (1.f - m));
    *(AT*)(hbuf[(K & 1) ^ 1] + h_put) = (AT)(valid ? hn : 0.f);
    c_state = c;
    h_prev = hn;
    y_out = (AT)y;
    a_out[0] = (AT)((p.op_flags & kOpH0IsCell) ? c : a0);
    a_out[1] = (AT)a1; a_out[2] = (AT)a2; a_out[3] = (AT)a3;
    __syncthreads();
  };
  __syncthreads();
  for (int s = 0; s < nsteps; s += kSoloAhead) {
    step(s, IntTag<0>{});
    if (s + 1 >= nsteps) break;
    step(s + 1, IntTag<1>{});
    if (s + 2 >= nsteps) break;
    step(s + 2, IntTag<2>{});
    if (s + 3 >= nsteps) break;
    step(s + 3, IntTag<3>{});
  }
  put(nsteps - 1);
  if (valid) {
    const long long bc = brow * nc + cell;
    p.d[bc] = c_state;
    if (p.hN) E::store(p.hN, bc, h_prev);
  }
}

// One row per workgroup (see the top).
template <typename AT, int S>
__global__ __launch_bounds__(64 * solo_waves<AT>(S)) __attribute__((amdgpu_waves_per_eu(2))) void k_lstm2_solo_row(const Lstm2Multi multi) {
  using E = Elem<AT>;
  constexpr int KM = E::KM, ES = (int)sizeof(AT);
  constexpr bool F32 = ES == 4;
  const Lstm2Params p = multi.p[blockIdx.y];
  __shared__ __align__(16) AT hbuf[2][S * KM];  // h, one buffer per parity of the step

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nc = p.nc, nsteps = p.nsteps;
  const long long row = blockIdx.x, bn = (long long)p.B * nc;
  if (blockIdx.x == 0 && tid < 64) p.status[tid] = status_word(tid, p.abort_word, p.abort_id);

  // This lane's gate of its quad's cell.  Cells beyond the width are copies of one inside, with its weights, inputs and state, and store the
  // same values to the same places: without a branch around the stores, behind which the compiler would have to take them for not issued
  // and wait for the input of this step as if it had been asked for a step ago.
  const int slot = kSoloCells * wave + (lane >> 2), cell = solo_cell<AT>(slot, nc), mine = lane & 3;
  const bool valid = slot < nc;
  float c_state = p.c0[row * nc + cell], h_prev = E::load(p.y0, row * nc + cell);
  hbuf[0][slot] = (AT)(valid ? h_prev : 0.f);

  // The op's streams.  Scalar pointers that go from frame to frame and the lane's constant offset: two scalar additions per stream and
  // step (buffer descriptors, as in the kernel above, took ten, and here no MFMAs hide them).  A step that does not exist reads the last
  // one's input.
  unsigned gate_at = (unsigned)(mine * nc + cell) * ES, y_at = (unsigned)cell * ES, c_at = (unsigned)cell * 4;
  const long long stride_x = (long long)p.step * p.B * p.ldX * ES, stride_m = (long long)p.step * p.B * 4, stride_h = (long long)p.step * bn * 4 * ES,
                  stride_y = (long long)p.step * p.B * p.ldY * ES, stride_c = (long long)p.step * bn * 4;
  const long long first_row = (long long)p.first * p.B + row;
  const unsigned char *in_x = (const unsigned char*)p.X + first_row * p.ldX * ES, *in_m = (const unsigned char*)(p.mask + first_row);
  unsigned char *out_h = (unsigned char*)p.H + first_row * 4 * nc * ES, *out_y = (unsigned char*)p.Y + first_row * p.ldY * ES, *out_c = (unsigned char*)(p.C + first_row * nc);
  AT xin[kSoloAhead];
  float msk[kSoloAhead];
  int more = nsteps - 1;  // frames behind the one that is fetched next
  auto fetch = [&](auto slot_tag) {
    constexpr int K = decltype(slot_tag)::value;
    asm volatile("" : "+v"(gate_at));
    xin[K] = *(const AT*)(in_x + gate_at);
    msk[K] = *(const float*)in_m;
    in_x += more > 0 ? stride_x : 0;
    in_m += more > 0 ? stride_m : 0;
    --more;
  };
  AT a_out = (AT)0.f, y_out = (AT)0.f;
  auto put = [&]() {  // the step before's outputs (the quad's lanes store the same y and c)
    asm volatile("" : "+v"(gate_at), "+v"(y_at), "+v"(c_at));  // (32 bits wide up to the access: the pointer stays scalar)
    *(AT*)(out_h + gate_at) = a_out;
    *(AT*)(out_y + y_at) = y_out;
    *(float*)(out_c + c_at) = c_state;
    out_h += stride_h;
    out_y += stride_y;
    out_c += stride_c;
  };

  fetch(IntTag<0>{});
  fetch(IntTag<1>{});
  fetch(IntTag<2>{});
  float wf[F32 ? 16 * S : 1];
  i32x4 wb[F32 ? 1 : 4][F32 ? 1 : S];
  solo_weights<AT, S, true>(p.W, nc, wave, lane, wf, wb);

  auto step = [&](int s, auto slot_tag) {
    constexpr int K = decltype(slot_tag)::value;
    const AT* hb = hbuf[K & 1];
    float g;
    if constexpr (F32) {
      float h[S], dot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < S; ++i) h[i] = hb[16 * i + (lane & 15)];
      __builtin_amdgcn_sched_barrier(0);
      if (s > 0) put();  // (these two while the LDS reads are under way)
      fetch(IntTag<(K + kSoloAhead - 1) % kSoloAhead>{});
      solo_fma_all<S>(h, wf, dot);
      g = ((dot[0] + dot[1]) + dot[2]) + dot[3];
    } else {
      f32x4 acc[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[v] = f32x4{0.f, 0.f, 0.f, 0.f};
      i32x4 h[S];
#pragma unroll
      for (int i = 0; i < S; ++i) h[i] = *(const i32x4*)(hb + 32 * i + 8 * (lane >> 4));
      __builtin_amdgcn_sched_barrier(0);
      if (s > 0) put();
      fetch(IntTag<(K + kSoloAhead - 1) % kSoloAhead>{});
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int keep = ((lane >> 2) & 3) == t ? -1 : 0;
#pragma unroll
        for (int i = 0; i < S; ++i) {
          const i32x4 b = i32x4{h[i][0] & keep, h[i][1] & keep, h[i][2] & keep, h[i][3] & keep};
          const int a = solo_acc<S>(t, i);
          acc[a] = E::mma(wb[t][i], b, acc[a]);
        }
      }
#pragma unroll
      for (int i = 0; i < 4 * S; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x076, 3, 0);
      }
      const f32x4 sum = ((acc[0] + acc[1]) + acc[2]) + acc[3];
      // the quad's four lanes have the same four gates: each takes its own
      const float lo = mine & 1 ? sum[1] : sum[0], hi = mine & 1 ? sum[3] : sum[2];
      g = mine & 2 ? hi : lo;
    }
    const float own = solo_gate<AT>(g + (float)xin[K], mine == 0);
    const float a0 = quad_lane<0>(own), a1 = quad_lane<1>(own), a2 = quad_lane<2>(own), a3 = quad_lane<3>(own);
    const float m = msk[K];
    const float pc = c_state;
    const float c = (pc * a2 + a0 * a1) * m + pc * (1.f - m);
    const float y = E::round(Act<AT>::tanh(c) * a3 * m);
    const float hn = (p.op_flags & kOpNoCarry) ? y : E::round(y + h_prev * (1.f - m));
    hbuf[(K & 1) ^ 1][slot] = (AT)(valid ? hn : 0.f);  // (four times the same)
    c_state = c;
    h_prev = hn;
    y_out = (AT)y;
    a_out = (AT)(mine == 0 && (p.op_flags & kOpH0IsCell) ? c : own);
    __syncthreads();
  };
  __syncthreads();
  for (int s = 0; s < nsteps; s += kSoloAhead) {
    step(s, IntTag<0>{});
    if (s + 1 >= nsteps) break;
    step(s + 1, IntTag<1>{});
    if (s + 2 >= nsteps) break;
    step(s + 2, IntTag<2>{});
    if (s + 3 >= nsteps) break;
    step(s + 3, IntTag<3>{});
  }
  put();
  if (valid && mine == 0) {
    p.d[row * nc + cell] = c_state;
    if (p.hN) E::store(p.hN, row * nc + cell, h_prev);
  }
}

}  // namespace rtn
