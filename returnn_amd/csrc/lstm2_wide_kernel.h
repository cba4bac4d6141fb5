// gfx950 persistent kernel of the forward recurrence for layers so wide that the recurrent weights take the registers AND
// the LDS of the whole device.
#pragma once

#include <hip/hip_runtime.h>

#include "lstm2_kernels.h"

namespace rtn {

// ---------------------------------------------------------------------------------------------
// W of n = 4096 in bf16 is 128 MB: 512 KB for each of the 256 CUs, which have 512 KB of registers and 160 KB of LDS.
// Launches per step read W from memory 200 times instead (22.6 us per step at 6 TB/s); here it is read once.
//
// One batch group of up to 16 * NT rows per launch, on all workgroups: workgroup r owns MT tiles of 4 cells, wavefront w
// of it the macro steps w, w + 4, ... of k: KS fragments per tile, all but the last LF of the MT * KS in registers, those in
// LDS.  The arithmetic and its order per element are those of k_lstm2_mfma and k_lstm2_regw.
//
// What such a step is made of is the exchange: every CU needs all n x rows values of h (128 KB at n = 4096), 32 MB per step
// over the device, which the memory side delivers in 3.5 us.  So h takes two hops.  The owner of a cell stores its new
// values at device scope into the group's ring, as in k_lstm2_regw.  The workgroups of an XCD share the work of bringing
// them over: each reads its part of the ring (4 KB), and stores it into a ring of its XCD with plain stores, which stay in
// that XCD's L2; from there all of them read everything, in chunks that the MFMAs of the chunk before hide.
// Both rings validate themselves (all-ones = not yet written) and have 4 slots:
//  * ring of the group: h_s (what step s reads) is in slot s % 4.  The owner stores h_{s+1} and re-arms h_{s-1}: it has seen
//    all of h_s, so every workgroup has finished step s-1, so every XCD had brought h_{s-1} over.
//  * ring of the XCD: a workgroup that brings its part of h_s over re-arms its part of h_{s-2}: it has seen all of h_{s-1}
//    there, of which every workgroup of the XCD brought its part when it had finished reading h_{s-2}.
// A re-arm is acknowledged (vmcnt(0) in front of the next publication) before anything that lets a reader ask for that slot.
// That the workgroups id % xcds share an XCD is checked at the start; if not, the copies are stored at device scope.
// Waits are bounded as everywhere.
// ---------------------------------------------------------------------------------------------
constexpr unsigned wide_lds_bytes(int MT, int NT, int LF) {
  return (unsigned)(kWaves * LF * kTileBytes + kWaves * MT * NT * kTileBytes);
}

// Fragments of h (16 bytes) that a workgroup brings over per thread at most: n / KE * 16 NT fragments over G / xcds workgroups.
constexpr int kWideForward = 2;

template <typename AT, int MT, int NT, int KS, int LF>
__global__ __launch_bounds__(kWgThreads) void k_lstm2_wide(const Lstm2Params p) {
  using E = Elem<AT>;
  using SN = Sentinel<AT>;
  using LM = LaneMax<AT>;
  constexpr int KE = E::KE, KM = E::KM, ES = (int)sizeof(AT);
  constexpr int TILES = MT * NT, EPT = (TILES + kWaves - 1) / kWaves, RF = MT * KS - LF;
  constexpr int CH = NT == 1 ? 4 : 2, NC = KS / CH;  // macro steps of h per chunk, chunks
  static_assert(KS % CH == 0 && LF >= 0 && RF > 0, "fragment counts");

  extern __shared__ __align__(16) unsigned char smem[];
  i32x4* Wl = (i32x4*)smem;                                            // [kWaves][LF][64]
  f32x4* red = (f32x4*)(smem + (size_t)kWaves * LF * kTileBytes);      // [kWaves][TILES][64]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = p.n, S = n / KM, nc = p.nc, G = p.wgs_per_group, X = p.xcds;
  // the workgroups of an XCD own neighbouring cells
  const int xcd = (int)blockIdx.x % X, member = (int)blockIdx.x / X;
  const int members = (G - xcd + X - 1) / X;
  const int r = xcd * (G / X) + min(xcd, G % X) + member;
  const int g = p.group_offset, b_base = g * p.Bg, rows = min(p.Bg, p.B - b_base);
  const int nsteps = p.nsteps;
  const long long bn = (long long)p.B * nc;
  const unsigned slot_bytes = (unsigned)((size_t)n * p.Bp * ES);
  unsigned char* hx_g = (unsigned char*)p.hx + (size_t)g * kHxRing * slot_bytes;
  unsigned char* hx_l = (unsigned char*)p.hxl + (size_t)xcd * kHxRing * slot_bytes;
  __amdgpu_buffer_rsrc_t ring = __builtin_amdgcn_make_buffer_rsrc((void*)hx_g, 0, kHxRing * slot_bytes, kBufFlags);
  __amdgpu_buffer_rsrc_t local = __builtin_amdgcn_make_buffer_rsrc((void*)hx_l, 0, kHxRing * slot_bytes, kBufFlags);
  const int kg = lane >> 4, jl = lane & 15;
  const int ks_count = S > wave ? (S - wave + kWaves - 1) / kWaves : 0;

  // W: fragments of this wavefront's share (zeros where there is none)
  i32x4 wreg[RF];
#pragma unroll
  for (int f = 0; f < MT * KS; ++f) {
    const int mt = f / KS, ks = f % KS, m = r * MT + mt;
    i32x4 v = i32x4{0, 0, 0, 0};
    if (ks < ks_count && m < n / 4) v = ((const i32x4*)p.Wp)[((size_t)m * S + wave + kWaves * ks) * 64 + lane];
    if (f < RF)
      wreg[f] = v;
    else
      Wl[(wave * LF + f - RF) * 64 + lane] = v;
  }

  // The (row, cell) pairs whose state this thread keeps.
  float c_state[EPT], h_prev[EPT];
  int e_cell[EPT], e_b[EPT];
  bool e_own[EPT], e_valid[EPT];  // the pair has a place in the ring; ... and exists for the caller
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = wave + kWaves * j;
    e_cell[j] = 4 * (r * MT + e / NT) + kg;
    e_b[j] = 16 * (e % NT) + jl;
    e_own[j] = e < TILES && e_cell[j] < n;
    e_valid[j] = e_own[j] && e_b[j] < rows && e_cell[j] < nc;
    c_state[j] = h_prev[j] = 0.f;
    if (e_valid[j]) {
      const long long bc = (long long)(b_base + e_b[j]) * nc + e_cell[j];
      c_state[j] = p.c0[bc];
      h_prev[j] = E::load(p.y0, bc);
    }
  }

  // This thread's fragments of the XCD's copy: offsets inside a slot (fragments of rows that do not exist are nobody's).
  const int frags = n / KE * p.Bp, part = (frags + members - 1) / members;
  unsigned f_off[kWideForward];
#pragma unroll
  for (int i = 0; i < kWideForward; ++i) {
    const int q = tid + kWgThreads * i, f = member * part + q;
    f_off[i] = q < part && f < frags && f % p.Bp < rows ? (unsigned)(f * kFragBytes) : kOobOffset;
  }
  unsigned b_off[NT];  // this lane's fragment of macro step `wave`
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) b_off[nt] = (unsigned)(((4 * wave + kg) * p.Bp + 16 * nt + jl) * kFragBytes);
  const unsigned ks_stride = (unsigned)(4 * kWaves * p.Bp * kFragBytes);  // from one macro step of the share to the next

  __shared__ int s_one_xcd;
  if (tid == 0) s_one_xcd = group_on_one_xcd(p.flags + (size_t)g * G + 2 * xcd, (unsigned)members, p.status, p.timeout_ticks) ? 1 : 0;
  __syncthreads();
  const bool one_xcd = s_one_xcd != 0;

  AT xin[EPT][4];
  float msk[EPT];
  auto fetch = [&](int s) {
    const size_t t = (size_t)frame_of(p, s);
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      msk[j] = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) xin[j][q] = (AT)0.f;
      if (e_valid[j]) {
        const AT* xp = (const AT*)p.X + (t * p.B + b_base + e_b[j]) * (size_t)p.ldX + e_cell[j];
#pragma unroll
        for (int q = 0; q < 4; ++q) xin[j][q] = xp[(size_t)q * nc];
        msk[j] = p.mask[t * p.B + b_base + e_b[j]];
      }
    }
  };
  // Bookkeeping of one repeated read: false when the wait is over for good.
  unsigned long long t0 = 0;
  auto keep_waiting = [&](unsigned& spins) {
    if ((spins++ & 15u) == 0) {
      if (__hip_atomic_load(p.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
      const unsigned long long now = wall_clock64();
      if (spins == 1) {
        t0 = now;
      } else if (now - t0 > p.timeout_ticks) {
        __hip_atomic_store(p.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
      }
    }
    return true;
  };
  auto incomplete = [&](const i32x4* v, int count) {
    unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < count; ++i)
#pragma unroll
      for (int w = 0; w < 4; ++w) m[w] = LM::fold(m[w], (unsigned)v[i][w]);
    return __any(LM::has_sentinel(LM::fold(LM::fold(m[0], m[1]), LM::fold(m[2], m[3])))) != 0;
  };

  i32x4 bf[2][CH * NT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int u = 0; u < CH * NT; ++u) bf[i][u] = i32x4{0, 0, 0, 0};
  fetch(0);
  int delay = p.poll_delay;
  for (int s = 0; s < nsteps; ++s) {
    const unsigned slot = (unsigned)(s & (kHxRing - 1)) * slot_bytes, old = (unsigned)((s + 2) & (kHxRing - 1)) * slot_bytes;
    // ---- bring this workgroup's part of h_s over
    {
      i32x4 fv[kWideForward];
      unsigned spins = 0;
      if (s > 0)
        for (int k = 0; k < delay; ++k) __builtin_amdgcn_s_sleep(1);
      do {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < kWideForward; ++i)
          fv[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ring, f_off[i], slot, kAuxDevice));
      } while (incomplete(fv, kWideForward) && keep_waiting(spins));
      // (a repeated read costs a trip to memory: the delay in front of the first adapts, as in k_lstm2_regw)
      if (spins)
        delay = min(delay + p.delay_inc, 64);
      else if (p.delay_inc && (s & p.delay_dec_mask) == p.delay_dec_mask && delay > 0)
        --delay;
      const u32x4 ones = u32x4{~0u, ~0u, ~0u, ~0u};
#pragma unroll
      for (int i = 0; i < kWideForward; ++i) {
        if (one_xcd) {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, fv[i]), local, f_off[i], slot, 0);
          __builtin_amdgcn_raw_buffer_store_b128(ones, local, f_off[i], old, 0);
        } else {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, fv[i]), local, f_off[i], slot, kAuxDevice);
          __builtin_amdgcn_raw_buffer_store_b128(ones, local, f_off[i], old, kAuxDevice);
        }
      }
    }
    // ---- the product, chunk by chunk
    auto load_chunk = [&](int c) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        if (16 * nt + jl < rows) {
#pragma unroll
          for (int u = 0; u < CH; ++u) {
            const int ks = c * CH + u;
            // (past the share: any complete fragment, against zeros of W)
            bf[c & 1][u * NT + nt] =
                __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(local, b_off[nt], slot + (ks < ks_count ? (unsigned)ks : 0u) * ks_stride, kAuxDevice));
          }
        }
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    load_chunk(0);
    unsigned spins = 0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (c + 1 < NC) load_chunk(c + 1);
      while (incomplete(bf[c & 1], CH * NT) && keep_waiting(spins)) load_chunk(c);
#pragma unroll
      for (int u = 0; u < CH; ++u)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const int f = mt * KS + c * CH + u;
          const i32x4 a = f < RF ? wreg[f < RF ? f : 0] : Wl[(wave * LF + f - RF) * 64 + lane];
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = E::mma(a, bf[c & 1][u * NT + nt], acc[mt][nt]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) red[(wave * TILES + mt * NT + nt) * 64 + lane] = acc[mt][nt];
    // everything this wavefront stored before (re-arms included) is acknowledged before its new values go out
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    asm volatile("" ::: "memory");
    __syncthreads();

    // ---- gates and cell update, new hidden values out
    float a_out[EPT][4], y_out[EPT];
    const unsigned nxt = (unsigned)((s + 1) & (kHxRing - 1)) * slot_bytes, arm = (unsigned)((s + 3) & (kHxRing - 1)) * slot_bytes;
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int e = wave + kWaves * j;
      y_out[j] = a_out[j][0] = a_out[j][1] = a_out[j][2] = a_out[j][3] = 0.f;
      if (e < TILES) {
        f32x4 gsum = red[e * 64 + lane];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) gsum += red[(w * TILES + e) * 64 + lane];
        const float m = msk[j];
        const float a0 = Act<AT>::tanh(gsum[0] + (float)xin[j][0]);
        const float a1 = Act<AT>::sigmoid(gsum[1] + (float)xin[j][1]);
        const float a2 = Act<AT>::sigmoid(gsum[2] + (float)xin[j][2]);
        const float a3 = Act<AT>::sigmoid(gsum[3] + (float)xin[j][3]);
        const float pc = c_state[j];
        const float c = (pc * a2 + a0 * a1) * m + pc * (1.f - m);
        const float y = E::round(Act<AT>::tanh(c) * a3 * m);
        const float hn = (p.op_flags & kOpNoCarry) ? y : E::round(y + h_prev[j] * (1.f - m));
        c_state[j] = c;
        h_prev[j] = hn;
        y_out[j] = y;
        a_out[j][0] = (p.op_flags & kOpH0IsCell) ? c : a0;
        a_out[j][1] = a1; a_out[j][2] = a2; a_out[j][3] = a3;
        if (e_own[j]) {
          const unsigned ho = (unsigned)((((e_cell[j] / KE) * p.Bp + e_b[j]) * KE + (e_cell[j] % KE)) * ES);
          SN::template store<kAuxDevice>(ring, ho + nxt, SN::bits(hn));
          SN::template store<kAuxDevice>(ring, ho + arm, SN::kSentinel);
        }
      }
    }
    // ---- while they travel: the op's outputs, and the next step's inputs
    const size_t t = (size_t)frame_of(p, s);
#pragma unroll
    for (int j = 0; j < EPT; ++j)
      if (e_valid[j]) {
        const size_t row = t * p.B + b_base + e_b[j];
#pragma unroll
        for (int q = 0; q < 4; ++q) E::store(p.H, row * 4 * nc + (size_t)q * nc + e_cell[j], a_out[j][q]);
        p.C[row * nc + e_cell[j]] = c_state[j];
        E::store(p.Y, row * (size_t)p.ldY + e_cell[j], y_out[j]);
      }
    if (s + 1 < nsteps) fetch(s + 1);
    __syncthreads();  // `red` may take the next step's partial tiles
  }

  // after a wait that ran into its bound: NaN as the final cell state and in the last visited frame of Y
  const bool expired = wait_expired(p.status);
  if (expired && tid == 0) report_expired(p.status);
  const size_t t_last = (size_t)frame_of(p, nsteps - 1);
#pragma unroll
  for (int j = 0; j < EPT; ++j)
    if (e_valid[j]) {
      const long long bc = (long long)(b_base + e_b[j]) * nc + e_cell[j];
      p.d[bc] = expired ? __builtin_nanf("") : c_state[j];
      if (p.hN) E::store(p.hN, bc, expired ? __builtin_nanf("") : h_prev[j]);
      if (expired) E::store(p.Y, (t_last * p.B + b_base + e_b[j]) * (size_t)p.ldY + e_cell[j], __builtin_nanf(""));
    }
}

}  // namespace rtn
