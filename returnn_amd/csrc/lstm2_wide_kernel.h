// gfx950 persistent kernel of the forward recurrence for layers so wide that the recurrent weights take the registers AND
// the LDS of the whole device.
#pragma once

#include <hip/hip_runtime.h>

#include "lstm2_kernels.h"

namespace rtn {

// ---------------------------------------------------------------------------------------------
// W of n = 4096 in bf16 is 128 MB: 512 KB for each of the 256 CUs, which have 512 KB of registers and 160 KB of LDS.
// Launches per step read W from memory every step (22.6 us at 6 TB/s); here a turn reads it once, and a step takes 4.1 us: T = 200,
// B = 16 4.58 ms as launches per step, 0.88 now, 0.05 of it for the packing.  What bounds a step: the matrix cores are busy for
// 2048 of its 9700 clocks, vector instructions issue in 1700, and half of the clocks a wavefront waits for memory -- the
// two hops of h.  (More of h in flight, 14 loads per wavefront instead of 8, in smaller chunks: 5 % slower.  What a chunk
// waits for is the last workgroup that brings its part over.)  (Fewer frames than pay for a turn's load of W run as launches per step: wide_turns_us in the host code.)
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
// A re-arm is acknowledged before anything that lets a reader ask for that slot: between it and the wavefront's next stores
// into the same ring lies the wait for the loads that bring the next h over, and a wavefront's memory operations are
// waited for in their order.
// That the workgroups id % xcds share an XCD is checked at the start; if not, the copies are stored at device scope.
// Waits are bounded as everywhere.
// ---------------------------------------------------------------------------------------------
// Fragments in LDS of a wavefront in the order the product takes them: how many come before tile mt of macro step ks.
constexpr int wide_lds_slot(int MT, int KS, int RF, int ks, int mt) {
  int count = 0;
  for (int k = 0; k <= ks; ++k)
    for (int m = 0; m < MT; ++m)
      if ((k < ks || m < mt) && m * KS + k >= RF) ++count;
  return count;
}

// What a staged step's streams take in LDS: X in, H out of the same places; Y; C.  (0: no such build, see WideStage.)
constexpr unsigned wide_stage_bytes(int MT, int NT, int LF, int ES) {
  return LF && ES == 4 ? 0u : (unsigned)(16 * NT * 4 * MT * (4 * ES + ES + 4));
}

constexpr unsigned wide_lds_bytes(int MT, int NT, int LF, int ES) {
  return (unsigned)(kWaves * LF * kTileBytes + kWaves * MT * NT * kTileBytes) + wide_stage_bytes(MT, NT, LF, ES);
}

// The op's streams of a workgroup in pieces of CB bytes of a row: PR pieces of each of X's and H's four blocks and of Y, PC of
// C.  64 pieces of one stream are a unit, a wavefront's access; the units are dealt to the wavefronts, SL to each at most.
template <typename AT, int MT, int NT>
struct WideStage {
  static constexpr int ES = (int)sizeof(AT), RC = 4 * MT, CB = (RC * ES) % 16 == 0 ? 16 : 8;
  static constexpr int PR = RC * ES / CB, PC = RC * 4 / CB;
  static constexpr int UH = NT * PR, UC = (16 * NT * PC + 63) / 64, UY = (16 * NT * PR + 63) / 64;
  static constexpr int SL = (UH + UC + UY + kWaves - 1) / kWaves;
  static constexpr int kC = 16 * NT * RC * 4 * ES, kY = kC + 16 * NT * RC * 4;  // where C and Y begin
};

// Fragments of h (16 bytes) that a workgroup brings over per thread at most: n / KE * 16 NT fragments over G / xcds workgroups.
constexpr int kWideForward = 2;

// STAGED: the op's streams go through LDS.  X comes in as up to 16 bytes of a row per thread, H, Y and C leave so; a thread by
// itself has 2 or 4 bytes of 4 cells next to each other, and every one of the 11 accesses per step touches 16 lines for a few bytes
// of each.  us per 200 steps without / with it: bf16 n = 4096 with 1, 4 and 16 rows 793 / 778, 805 / 785, 949 / 877, n = 2560 with 16 and 32
// rows 767 / 696, 1182 / 960; float32 n = 1280 with 16 rows 1356 / 1240, n = 2048 with 3 and 32 rows 1261 / 1258, 2231 / 2103.  (n = 4096, 16 rows
// without any streams: 823.)  h as one store of 8 or 16 bytes per row of a tile instead of one per cell, the lanes' values brought
// together first: 871, 697 and 971, 1262, 1282 and 2087; not kept.
// Where rows may begin anywhere (p.nc < p.n), and in float32 beyond n = 2048, where W leaves no room, pair by pair.
template <typename AT, int MT, int NT, int KS, int LF, bool STAGED>
__global__ __launch_bounds__(kWgThreads) void k_lstm2_wide(const Lstm2Params p) {
  using E = Elem<AT>;
  using SN = Sentinel<AT>;
  using LM = LaneMax<AT>;
  constexpr int KE = E::KE, KM = E::KM, ES = (int)sizeof(AT);
  constexpr int TILES = MT * NT, EPT = (TILES + kWaves - 1) / kWaves, RF = MT * KS - LF;
  constexpr int CH = NT == 1 ? 4 : 2, NB = 3, NC = KS / CH;  // macro steps of h per chunk, chunks in flight, chunks
  static_assert(KS % CH == 0 && LF >= 0 && RF > 0, "fragment counts");

  extern __shared__ __align__(16) unsigned char smem[];
  i32x4* Wl = (i32x4*)smem;                                            // [kWaves][LF][64]
  f32x4* red = (f32x4*)(smem + (size_t)kWaves * LF * kTileBytes);      // [kWaves][TILES][64]
  using Stage = WideStage<AT, MT, NT>;
  constexpr int RC = Stage::RC, CB = Stage::CB, SL = Stage::SL;
  unsigned char* stage = (unsigned char*)(red + kWaves * TILES * 64);  // X and H [4][16 NT][RC], C [16 NT][RC], Y [16 NT][RC]
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
      Wl[(wave * LF + wide_lds_slot(MT, KS, RF, ks, mt)) * 64 + lane] = v;
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
    start_state<AT>(p, e_valid[j], (b_base + e_b[j]) * nc + e_cell[j], &c_state[j], &h_prev[j]);
  }

  // This thread's fragments of the XCD's copy: offsets inside a slot (fragments of rows that do not exist are nobody's).
  const int frags = n / KE * p.Bp, part = (frags + members - 1) / members;
  unsigned f_off[kWideForward];
#pragma unroll
  for (int i = 0; i < kWideForward; ++i) {
    const int q = tid + kWgThreads * i, f = member * part + q;
    f_off[i] = q < part && f < frags && f % p.Bp < rows ? (unsigned)(f * kFragBytes) : kOobOffset;
  }
  // This lane's fragment of macro step `wave`.  Lanes of rows that do not exist load beyond the buffer (zeros): a branch around
  // the loads would have the compiler wait for all of them at every use, since any of them could be the last one issued.
  unsigned b_off[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) b_off[nt] = 16 * nt + jl < rows ? (unsigned)(((4 * wave + kg) * p.Bp + 16 * nt + jl) * kFragBytes) : kOobOffset;
  const unsigned ks_stride = (unsigned)(4 * kWaves * p.Bp * kFragBytes);  // from one macro step of the share to the next

  __shared__ int s_one_xcd;
  if (wave == 0) s_one_xcd = group_on_one_xcd(p.flags + (size_t)g * G + 2 * xcd, (unsigned)members, p.status, p.timeout_ticks) ? 1 : 0;
  __syncthreads();
  const bool one_xcd = s_one_xcd != 0;

  // The op's streams, a pair per thread or (STAGED) a piece of a row: gate inputs and mask come in one step ahead, behind the loads of the product; a step's
  // outputs leave behind the next step's.  Without a branch: pairs and frames that do not exist have offsets beyond any
  // frame.  (With branches the compiler has to wait for these loads and stores, and the
  // trip to memory they take, wherever it waits for a chunk of h.)
  unsigned x_at[EPT], h_at[EPT], y_at[EPT], c_at[EPT], m_at[EPT];  // byte offsets inside a frame
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const long long row = b_base + e_b[j];
    x_at[j] = e_valid[j] ? (unsigned)((row * p.ldX + e_cell[j]) * ES) : kOobOffset;
    h_at[j] = e_valid[j] ? (unsigned)((row * 4 * nc + e_cell[j]) * ES) : kOobOffset;
    y_at[j] = e_valid[j] ? (unsigned)((row * p.ldY + e_cell[j]) * ES) : kOobOffset;
    c_at[j] = e_valid[j] ? (unsigned)((row * nc + e_cell[j]) * 4) : kOobOffset;
    m_at[j] = e_valid[j] ? (unsigned)(row * 4) : kOobOffset;
  }
  const unsigned frame_x = (unsigned)((size_t)p.B * p.ldX * ES), frame_h = (unsigned)((size_t)p.B * 4 * nc * ES), frame_y = (unsigned)((size_t)p.B * p.ldY * ES),
                 frame_c = (unsigned)(bn * 4), frame_m = (unsigned)(p.B * 4), gate = (unsigned)(nc * ES);  // (gate: from one of a row's four blocks to the next)
  // A staged unit's stream, and this thread's piece of it: its offset in X's frame (H's units) and in the output's, and where it
  // is in LDS.
  using Piece = std::conditional_t<CB == 16, i32x4, i32x2>;
  unsigned xp_at[SL], op_at[SL], lp_at[SL];
  Piece xp[SL];
  if constexpr (STAGED) {
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      const int u = wave + kWaves * i;
      const bool is_h = u < Stage::UH, is_c = !is_h && u < Stage::UH + Stage::UC;
      const int k = 64 * (is_h ? u : is_c ? u - Stage::UH : u - Stage::UH - Stage::UC) + lane;  // the piece of the stream
      const int per_row = is_c ? Stage::PC : Stage::PR, block = k / (16 * NT * per_row), row = k / per_row % (16 * NT);
      const int in_block = block * nc, cell = 4 * r * MT + k % per_row * (CB / (is_c ? 4 : ES));
      const bool there = u < Stage::UH + Stage::UC + Stage::UY && block < (is_h ? 4 : 1) && row < rows && cell < nc;
      const long long at = b_base + row;
      xp_at[i] = is_h && there ? (unsigned)((at * p.ldX + in_block + cell) * ES) : kOobOffset;
      op_at[i] = !there ? kOobOffset : is_h ? (unsigned)((at * 4 * nc + in_block + cell) * ES) : is_c ? (unsigned)((at * nc + cell) * 4) : (unsigned)((at * p.ldY + cell) * ES);
      lp_at[i] = block < (is_h ? 4 : 1) ? (unsigned)((is_h ? 0 : is_c ? Stage::kC : Stage::kY) + k * CB) : 0u;
    }
  }
  AT xin[EPT][4], xnext[EPT][4];
  float msk[EPT], mnext[EPT];
  // (frames that do not exist: all offsets beyond; not a buffer of no bytes, whose range check a scalar offset would wrap)
  auto frame = [&](const void* base, int s, unsigned bytes, bool there) {
    return __builtin_amdgcn_make_buffer_rsrc((unsigned char*)base + (there ? frame_of(p, s) : 0) * (long long)bytes, 0, bytes, kBufFlags);
  };
  auto fetch = [&](int s) {
    const bool there = s < nsteps;
    __amdgpu_buffer_rsrc_t xr = frame(p.X, s, frame_x, there), mr = frame(p.mask, s, frame_m, there);
    if constexpr (STAGED) {
#pragma unroll
      for (int i = 0; i < SL; ++i) {
        if (kWaves * i >= Stage::UH) continue;
        const unsigned at = there ? xp_at[i] : kOobOffset;
        if constexpr (CB == 16)
          xp[i] = __builtin_bit_cast(Piece, __builtin_amdgcn_raw_buffer_load_b128(xr, at, 0, 0));
        else
          xp[i] = __builtin_bit_cast(Piece, __builtin_amdgcn_raw_buffer_load_b64(xr, at, 0, 0));
      }
    }
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const unsigned at = there ? x_at[j] : kOobOffset;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if constexpr (STAGED)
          continue;
        else if constexpr (ES == 2)
          xnext[j][q] = __builtin_bit_cast(AT, __builtin_amdgcn_raw_buffer_load_b16(xr, at, q * gate, 0));
        else
          xnext[j][q] = __builtin_bit_cast(AT, __builtin_amdgcn_raw_buffer_load_b32(xr, at, q * gate, 0));
      }
      mnext[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(mr, there ? m_at[j] : kOobOffset, 0, 0));
    }
  };
  auto take = [&]() {
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
#pragma unroll
      for (int q = 0; q < 4 && !STAGED; ++q) xin[j][q] = xnext[j][q];
      msk[j] = mnext[j];
    }
  };
  AT a_out[EPT][4], y_out[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) a_out[j][0] = a_out[j][1] = a_out[j][2] = a_out[j][3] = y_out[j] = (AT)0.f;
  auto put = [&](int s) {
    const bool there = s >= 0;
    __amdgpu_buffer_rsrc_t hr = frame(p.H, s, frame_h, there), yr = frame(p.Y, s, frame_y, there), cr = frame(p.C, s, frame_c, there);
    if constexpr (STAGED) {
#pragma unroll
      for (int i = 0; i < SL; ++i) {
        const int u = wave + kWaves * i;
        const Piece v = *(const Piece*)(stage + lp_at[i]);
        __amdgpu_buffer_rsrc_t rs = u < Stage::UH ? hr : u < Stage::UH + Stage::UC ? cr : yr;
        const unsigned at = there ? op_at[i] : kOobOffset;
        if constexpr (CB == 16)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rs, at, 0, 0);
        else
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rs, at, 0, 0);
      }
      return;
    }
    auto store = [&](AT v, __amdgpu_buffer_rsrc_t rs, unsigned off, unsigned block) {
      if constexpr (ES == 2)
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), rs, off, block, 0);
      else
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rs, off, block, 0);
    };
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) store(a_out[j][q], hr, there ? h_at[j] : kOobOffset, q * gate);
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, c_state[j]), cr, there ? c_at[j] : kOobOffset, 0, 0);
      store(y_out[j], yr, there ? y_at[j] : kOobOffset, 0);
    }
  };
  // X of the step, in the places that H of the step before has been read from.
  auto stage_x = [&]() {
    if constexpr (STAGED) {
#pragma unroll
      for (int i = 0; i < SL; ++i)
        if (wave + kWaves * i < Stage::UH) *(Piece*)(stage + lp_at[i]) = xp[i];
    }
  };
  auto staged_pair = [&](int j) { return (e_b[j] * RC + (e_cell[j] - 4 * r * MT)); };  // a pair's place in a staged block
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
  // Running maxima over the elements of fragments, and whether one of them was not written yet.
  auto fold = [&](unsigned (&m)[4], const i32x4& v) {
#pragma unroll
    for (int w = 0; w < 4; ++w) m[w] = LM::fold(m[w], (unsigned)v[w]);
  };
  auto seen_mark = [&](const unsigned (&m)[4]) { return __any(LM::has_sentinel(LM::fold(LM::fold(m[0], m[1]), LM::fold(m[2], m[3])))) != 0; };

  i32x4 bf[NB][CH * NT];
  fetch(0);
  take();
  RTN_TRACE_DECL
  // float32, two tiles of cells and one of rows (1024 < n <= 2048, up to 16 rows): a delay that adapts, from 4 units on.  us per step without / with
  // it: 1, 2, 4 and 8 rows of n = 1088, 1280, 1536, 1722 and 2048, 120 and 1200 steps, all 1.4 ... 2.9 % less with it (n = 1722, 2 rows 6.20 / 6.05; n = 2048,
  // 8 rows 6.61 / 6.51 in 120 steps); 16 rows 0 ... 2.9 % less (n = 1088 6.69 / 6.52), n = 1280 in 1200 steps 6.66 / 6.82.  (Fixed at 4 units 6.12 where it takes
  // 6.05; from 20 units on, 120 steps of n = 1722 take 6.67.)  The other float32 builds lose by it or are level: 32 rows of n = 1280, 1722, 2048 10.99 / 11.17,
  // 11.03 / 11.19, 11.03 / 11.19; n = 2304, 2 and 16 rows 10.14 / 10.11, 10.84 / 10.98; n = 2816 10.25 / 10.22, 11.04 / 11.18.
  constexpr bool kAdapts = sizeof(AT) == 4 && MT == 2 && NT == 1;
  int delay = 4;
  for (int s = 0; s < nsteps; ++s) {
    const unsigned slot = (unsigned)(s & (kHxRing - 1)) * slot_bytes, old = (unsigned)((s + 2) & (kHxRing - 1)) * slot_bytes;
    // ---- bring this workgroup's part of h_s over
    {
      // (No delay in front of the first read, as the kernels whose CUs read all of h across the XCDs have it: a repeat is 4 KB per CU and
      // costs the others nothing.  us per step of 600 without / with one that adapts: n = 4096, 16 rows 4.41 / 4.51, one row 3.71 / 3.78; n = 2560, 16 rows 3.73 / 3.83,
      // 32 rows 5.74 / 5.87.  In float32 one of the builds gains by one: see kAdapts.)
      if constexpr (kAdapts)
        if (s > 0)
          for (int k = 0; k < delay; ++k) __builtin_amdgcn_s_sleep(1);
      i32x4 fv[kWideForward];
      unsigned spins = 0;
      bool again;
      do {
        asm volatile("" ::: "memory");
        unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < kWideForward; ++i)
          fv[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ring, f_off[i], slot, kAuxDevice));
#pragma unroll
        for (int i = 0; i < kWideForward; ++i) fold(m, fv[i]);
        again = seen_mark(m) && keep_waiting(spins);
      } while (again);
      if constexpr (kAdapts) {
        if (spins)
          delay = min(delay + p.delay_inc, 64);
        else if (p.delay_inc && (s & p.delay_dec_mask) == p.delay_dec_mask && delay > 0)
          --delay;
      }
      RTN_TRACE_MARK(0)  // h_s arrives across the XCDs
      RTN_TRACE_ADD(6, spins)
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
    // ---- the product, chunk by chunk; a chunk is checked behind the MFMAs of the one before (checked in front of its own, with
    // the matrix core idle meanwhile, each of them cost 0.1 us)
    auto load_chunk = [&](int c) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int u = 0; u < CH; ++u) {
          const int ks = c * CH + u;
          // (past the share: any complete fragment, against zeros of W)
          bf[c % NB][u * NT + nt] =
              __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(local, b_off[nt], slot + (ks < ks_count ? (unsigned)ks : 0u) * ks_stride, kAuxDevice));
        }
    };
    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    unsigned spins = 0;
    auto complete = [&](int c, bool mark) {  // read chunk c again until it is complete
      while (mark && keep_waiting(spins)) {
        load_chunk(c);
        unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < CH * NT; ++u) fold(m, bf[c % NB][u]);
        mark = seen_mark(m);
      }
    };
    load_chunk(0);
    // the fragments in LDS are read WP ahead of their MFMA (read where they are needed, each of them cost 80 clocks)
    constexpr int WP = LF ? 2 : 1;
    i32x4 wl[WP];
    if constexpr (LF > 0) {
#pragma unroll
      for (int i = 0; i < WP; ++i) wl[i] = Wl[(wave * LF + i) * 64 + lane];
    }
    {
      unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < CH * NT; ++u) fold(m, bf[0][u]);
      complete(0, seen_mark(m));
    }
    // (the others behind it: asked for together with the first one, they are in the way of its repeats)
#pragma unroll
    for (int c = 1; c < NB - 1; ++c) load_chunk(c);
    RTN_TRACE_MARK(1)  // brought over, first chunk back
    RTN_TRACE_ADD(7, spins)
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (c + NB - 1 < NC) load_chunk(c + NB - 1);
      if (c + NB - 1 == NC - 1 || (NC < NB && c == 0)) {
        put(s - 1);
        stage_x();
        fetch(s + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < CH; ++u) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const int f = mt * KS + c * CH + u, q = wide_lds_slot(MT, KS, RF, c * CH + u, mt);
          const i32x4 a = f < RF ? wreg[f < RF ? f : 0] : wl[q % WP];
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = E::mma(a, bf[c % NB][u * NT + nt], acc[mt][nt]);
          if (f >= RF && q + WP < LF) wl[q % WP] = Wl[(wave * LF + q + WP) * 64 + lane];
        }
        if (c + 1 < NC)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) fold(m, bf[(c + 1) % NB][u * NT + nt]);
      }
      const bool mark = c + 1 < NC && seen_mark(m);
      __builtin_amdgcn_sched_barrier(0);
      if (c + 1 < NC) complete(c + 1, mark);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) red[(wave * TILES + mt * NT + nt) * 64 + lane] = acc[mt][nt];
    RTN_TRACE_MARK(2)  // product
    __syncthreads();
    RTN_TRACE_MARK(3)  // barrier

    // ---- gates and cell update, new hidden values out
    const unsigned nxt = (unsigned)((s + 1) & (kHxRing - 1)) * slot_bytes, arm = (unsigned)((s + 3) & (kHxRing - 1)) * slot_bytes;
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int e = wave + kWaves * j;
      if (e < TILES) {
        f32x4 part[kWaves];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) part[w] = red[(w * TILES + e) * 64 + lane];
        __builtin_amdgcn_sched_barrier(0);
        f32x4 gsum = part[0];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) gsum += part[w];
        const float m = msk[j];
        AT* const hs = (AT*)stage + staged_pair(j);  // X's and H's place in the first block
        constexpr int block = 16 * NT * RC;
        if constexpr (STAGED) {
#pragma unroll
          for (int q = 0; q < 4; ++q) xin[j][q] = hs[q * block];
        }
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
        y_out[j] = (AT)y;
        a_out[j][0] = (AT)((p.op_flags & kOpH0IsCell) ? c : a0);
        a_out[j][1] = (AT)a1; a_out[j][2] = (AT)a2; a_out[j][3] = (AT)a3;
        if constexpr (STAGED) {
#pragma unroll
          for (int q = 0; q < 4; ++q) hs[q * block] = a_out[j][q];
          ((float*)(stage + Stage::kC))[staged_pair(j)] = c;
          ((AT*)(stage + Stage::kY))[staged_pair(j)] = (AT)y;
        }
        if (e_own[j]) {
          const unsigned ho = (unsigned)((((e_cell[j] / KE) * p.Bp + e_b[j]) * KE + (e_cell[j] % KE)) * ES);
          SN::template store<kAuxDevice>(ring, ho + nxt, SN::bits(hn));
          SN::template store<kAuxDevice>(ring, ho + arm, SN::kSentinel);
        }
      }
    }
    RTN_TRACE_MARK(4)  // gates, new values out
    take();
    __syncthreads();  // `red` may take the next step's partial tiles
    RTN_TRACE_MARK(5)  // next inputs, barrier
  }
  RTN_TRACE_FLUSH(p, blockIdx.x)

  put(nsteps - 1);
  if constexpr (STAGED) __syncthreads();  // (the mark below goes over what another thread has stored)

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
