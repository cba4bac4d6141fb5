// gfx950 kernel of the forward recurrence for layers whose recurrent weights fit the registers of ONE compute unit.
#pragma once

#include <hip/hip_runtime.h>

#include "lstm2_kernels.h"

namespace rtn {

// ---------------------------------------------------------------------------------------------
// A step of a small layer (n = 64 in float32: 64 KB of weights, 0.2 us of MFMAs on one CU) is shorter than one hand-over
// between workgroups (0.4 us and more), so nothing is handed over: a workgroup takes 4 batch rows through all steps by
// itself, W in its registers, h in LDS, one barrier per step.  Workgroups know nothing of each other: no packing of W, no
// ring, no waits, any number of them.
//
// A wavefront owns 16 cells, all four gates of them, and the whole contraction; the lane that ends up with a (row, cell)
// pair has its four gates.  4 rows per workgroup: one pair per lane, and more rows would lengthen the pointwise part, which
// is half of the step, while B / 4 workgroups find a CU each up to 1024 rows.
//  * float32: v_mfma_f32_4x4x1 -- 16 blocks of 4 rows x 4 columns; A (h) of block k is broadcast to all of them, so that one
//    instruction takes 4 rows x 64 gate columns x one k in 8 clocks (a 16x16x4 tile spends three quarters of its 32 clocks on
//    rows that do not exist).  The results lie gate by gate in the lanes of a quad and are transposed there.
//  * bf16: v_mfma_f32_16x16x32 on tiles of 4 cells, four tiles in ONE accumulator: tile t's B operand has the four rows
//    in columns 4 t ... 4 t + 3 and zeros elsewhere.
// The order of additions per element is that of the other kernels (their four wavefronts' shares of k are four
// accumulators here), so the results are theirs bit for bit.
// Measured (float32, T = 32, B = 4, n = 64): one call 27 us; 45 us with packing (5.3) and k_lstm2_regw (36.5).
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
  // W of this wavefront's cells.  float32: a lane's column is gate lane % 4 of cell lane / 4, one register per k.  bf16: row
  // i = lane % 16 of tile t is gate i % 4 of cell 4 (i / 4) + t: a lane loads four neighbouring cells at once.  (What lies
  // beyond the width is loaded from inside and replaced by zeros: no branches between the loads.)
  float wf[F32 ? 16 * S : 1];
  i32x4 wb[F32 ? 1 : 4][F32 ? 1 : S];
  if constexpr (F32) {
    const int wcell = kSoloCells * wave + (lane >> 2);
    const float* src = (const float*)p.W + (size_t)(lane & 3) * nc + min(wcell, nc - 1);
#pragma unroll
    for (int k = 0; k < 16 * S; ++k) wf[k] = src[(size_t)min(k, nc - 1) * 4 * nc];
#pragma unroll
    for (int k = 0; k < 16 * S; ++k) wf[k] = k < nc && wcell < nc ? wf[k] : 0.f;
  } else {
    const int i = lane & 15, kg = lane >> 4, wcell = kSoloCells * wave + 4 * (i >> 2);
    typedef unsigned long long u64_any __attribute__((aligned(2)));
    const unsigned short* src = (const unsigned short*)p.W + (size_t)(i & 3) * nc;
    const bool whole = nc % 4 == 0;  // (no lane's four cells are cut)
#pragma unroll
    for (int s = 0; s < S; ++s) {
      unsigned long long v[8];
      if (whole) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = *(const u64_any*)(src + (size_t)min(KM * s + 8 * kg + e, nc - 1) * 4 * nc + min(wcell, nc - 4));
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = KM * s + 8 * kg + e < nc && wcell < nc ? v[e] : 0;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int k = KM * s + 8 * kg + e;
          v[e] = 0;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const unsigned long long x = src[(size_t)min(k, nc - 1) * 4 * nc + min(wcell + c, nc - 1)];
            v[e] |= (k < nc && wcell + c < nc ? x : 0) << (16 * c);
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
          acc[i & 3] = E::mma(wb[t][i], b, acc[i & 3]);
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

}  // namespace rtn
