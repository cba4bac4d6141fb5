// gfx950 persistent kernel of the gradient recurrence for layers whose recurrent weights take the registers AND the LDS of the
// CUs of a batch group.
#pragma once

#include <hip/hip_runtime.h>

#include "lstm2_bwd_kernels.h"
#include "lstm2_wide_kernel.h"

namespace rtn {

// ---------------------------------------------------------------------------------------------
// W of n = 2048 in bf16 is 32 MB, and what bounds k_lstm2_bwd_regw there is not W but how many rows a launch takes: a workgroup
// with one tile of 16 values of k reads all of its group's derivatives every frame (16 rows x 4n values, 256 KB), 128 of them are a group of
// 16 rows, and the device holds two such groups.  Here a workgroup has MT = 2 tiles for the same 256 KB: four groups at once.
// What bounds a frame (6.3 us at n = 2048) is those 256 KB on their way from the XCD's L2, 40 KB per microsecond and CU of the 150 that its
// path takes: 12 loads per wavefront in flight are what the registers have room for.  Of a frame's 14 000 clocks the MFMAs are 2048, vector
// instructions 2800, and half of them a wavefront waits for memory.
// us per gradient call of 64 frames, k_lstm2_bwd_regw / here: n = 2048, 48, 64, 100 and 256 rows 737 / 588, 877 / 743, 1446 / 1149, 2939 / 2380, two
// problems of 32 rows 842 / 699; n = 1792, 100 rows 1479 / 1121; n = 1536, 48, 64 and 160 rows 685 / 455, 784 / 551, 1754 / 1326; n = 1280, 64 rows 700 / 437.
// (Chunks of 2 macro steps, six of them in flight: 783 at n = 2048 and 64 rows; the next frame's inputs behind the last chunk: 773.)
//
//  * W: 2 x KST fragments per wavefront, all but the last LF of them in registers, those in LDS, as in k_lstm2_wide.
//  * exchange: in two hops, as there.  The owner of a cell stores its derivatives at device scope into the group's ring; the workgroups
//    of a group on one XCD share the work of bringing a frame over into a ring of that XCD, from where all of them read
//    everything in chunks behind the MFMAs of the chunk before.  A group has X / slots XCDs to itself (slots: groups the
//    grid has room for).  Both rings have kExRing slots and validate themselves, and the order of their re-arms is that of k_lstm2_wide:
//    frame f's derivatives are stored when all of frame f - 1's have been seen, and with them what frame f - 2 left in a
//    slot is re-armed; a workgroup that brings its part of frame f over re-arms its part of frame f - 2, of which everybody on
//    the XCD has finished the product when frame f - 1 was complete there.
//  * frame: pointwise part, stores, next frame's inputs asked for, the other workgroups' derivatives brought over, product, sum
//    over the wavefronts.  The inputs' way from memory and the hand-over take as long as each other and go in parallel.
// ---------------------------------------------------------------------------------------------
// Fragments (16 bytes) that a thread brings over per frame at most.
constexpr int kBwdWideForward = 2;

template <typename AT, int MT, int KST, int LF>
__global__ __launch_bounds__(kWgThreads) void k_lstm2_bwd_wide(const Lstm2BwdMulti multi) {
  using E = Elem<AT>;
  using SN = Sentinel<AT>;
  using LM = LaneMax<AT>;
  constexpr int KE = E::KE, KM = E::KM, ES = (int)sizeof(AT);
  constexpr int RF = MT * KST - LF, CH = 4, NB = 3, NC = KST / CH, NACC = 2;
  constexpr int Bp = 16, kRedGroup = 20, KGW = 16 * MT / KE;
  static_assert(KST % CH == 0 && NC > NB && CH % NACC == 0 && LF > 2 && 4 * KGW * Bp == kWgThreads, "fragment counts; a piece of the derivatives per thread");

  // id -> group of the launch, all problems counted through (gg), and the workgroup's place in it
  const int X = multi.xcds, xpg = X / multi.slots;
  const int xcd = (int)blockIdx.x % X, member = (int)blockIdx.x / X, members = (int)gridDim.x / X;
  const int gg = xcd / xpg, which = gg / multi.q[0].groups;
  if (which >= multi.count) return;
  const Lstm2BwdPersistent q = multi.q[which];
  const Lstm2BwdParams& p = q.p;
  const int g = q.group_offset + gg - which * q.groups, rank = (xcd % xpg) * members + member;
  const int n = p.n, n4 = 4 * n, nc = p.nc, k0 = rank * 16 * MT;
  const int b_base = g * q.Bg, rows = min(q.Bg, p.B - b_base);
  const long long bn = (long long)p.B * nc;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  extern __shared__ __align__(16) unsigned char bwd_smem[];
  i32x4* Wl = (i32x4*)bwd_smem;  // [kWaves][LF][64]
  __shared__ f32x4 red[kWaves][MT][4 * kRedGroup];
  __shared__ i32x4 stage[4 * KGW * Bp];  // [gate][piece][row]: the workgroup's derivatives of a frame in ring order
  __shared__ int s_one_xcd;
  if (wave == 0) s_one_xcd = (int)group_on_one_xcd(q.sync + 2 * (size_t)(g * xpg + xcd % xpg), (unsigned)members, q.status, q.timeout_ticks);

  const unsigned frame_bytes = (unsigned)((size_t)p.B * 4 * nc * ES);
  const unsigned dx_frame_bytes = (unsigned)((size_t)p.B * p.ldDX * ES), dy_frame_bytes = (unsigned)((size_t)p.B * p.ldDY * ES);
  const unsigned ex_frame = (unsigned)((size_t)n4 * Bp * ES);  // one slot of a ring: [4n/KM][4][Bp][16 bytes]
  __amdgpu_buffer_rsrc_t ring = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)q.ex + (size_t)g * kExRing * ex_frame, 0, kExRing * ex_frame, kBufFlags);
  __amdgpu_buffer_rsrc_t local = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)q.exl + (size_t)xcd * kExRing * ex_frame, 0, kExRing * ex_frame, kBufFlags);

  // W: wavefront w has the macro steps [w * ksb, (w + 1) * ksb) of j, as far as they reach (zeros beyond)
  const int ksb = q.ksb, ks_here = max(0, min(ksb, n4 / KM - ksb * wave));
  i32x4 wreg[RF];
#pragma unroll
  for (int f = 0; f < MT * KST; ++f) {
    const int mt = f / KST, ks = f % KST;
    const AT* Wr = (const AT*)p.W + (size_t)(k0 + 16 * mt + (lane & 15)) * n4 + (size_t)KM * ksb * wave + KE * (lane >> 4);
    const i32x4 v = (ks < ks_here) ? *(const i32x4*)(Wr + (size_t)KM * ks) : i32x4{0, 0, 0, 0};
    if (f < RF)
      wreg[f] = v;
    else
      Wl[(wave * LF + wide_lds_slot(MT, KST, RF, ks, mt)) * 64 + lane] = v;
  }
  // this lane's first B fragment of the XCD's ring (rows that do not exist: beyond the buffer, zeros)
  const unsigned b_off = (lane & 15) < rows ? (unsigned)(((ks_here ? ksb * wave * 4 : 0) + (lane >> 4)) * Bp + (lane & 15)) * 16u : kOobOffset;
  constexpr unsigned ks_stride = 4 * Bp * 16;
  // the fragments this thread brings over
  const int frags = n4 / KE * Bp, part = (frags + members - 1) / members;
  unsigned f_off[kBwdWideForward];
#pragma unroll
  for (int i = 0; i < kBwdWideForward; ++i) {
    const int at = tid + kWgThreads * i, f = member * part + at;
    f_off[i] = at < part && f < frags && f % Bp < rows ? (unsigned)(f * 16) : kOobOffset;
  }
  // this thread's piece of the workgroup's derivatives: where it goes
  const int o_row = tid & (Bp - 1), o_gate = (tid / Bp) / KGW, o_piece = (tid / Bp) % KGW, o_cell = k0 + o_piece * KE;
  const unsigned o_ring = o_row < rows ? (unsigned)((((o_gate * n + k0) / KE + o_piece) * Bp + o_row) * 16) : kOobOffset;
  const unsigned o_dx = o_row < rows && o_cell < nc ? (unsigned)(((size_t)(b_base + o_row) * p.ldDX + (size_t)o_gate * nc + o_cell) * ES) : kOobOffset;

  // The (row, k) pairs of this thread: one in each tile.
  const int kl = tid & 15, bl = tid >> 4, b = b_base + ((bl < rows) ? bl : 0);
  const int red_at = (kl >> 2) * kRedGroup + bl, red_comp = kl & 3;
  bool act[MT];
  unsigned off_h[MT], off_dy[MT], off_c[MT];  // byte offsets inside a frame; out of range (0 comes back) for cells beyond nc
  float dyw[MT], dc[MT], dx0[MT][4];
  // (no branch around the load: behind one that some lanes skip, a full register file has cost those lanes values)
  __amdgpu_buffer_rsrc_t rs_dd = __builtin_amdgcn_make_buffer_rsrc((void*)q.Dd, 0, q.Dd ? (unsigned)(bn * 4) : 0u, kBufFlags);
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int k = k0 + 16 * j + kl;
    act[j] = bl < rows && k < nc;
    off_h[j] = k < nc ? (unsigned)(((long long)b * 4 * nc + k) * ES) : kOobOffset;
    off_dy[j] = k < nc ? (unsigned)(((long long)b * p.ldDY + k) * ES) : kOobOffset;
    off_c[j] = k < nc ? (unsigned)(((long long)b * nc + k) * 4) : kOobOffset;
    dyw[j] = 0.f;
    dc[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_dd, act[j] ? off_c[j] : kOobOffset, 0, 0));
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) dx0[j][gq] = 0.f;
  }
  // Inputs of a frame, as the loads bring them; without branches around them, as in k_lstm2_bwd_regw.
  unsigned in_gate[MT][4], in_dy[MT], in_pc[MT], in_ph[MT];
  float in_m;
  auto widen = [](unsigned raw) {
    if constexpr (ES == 2)
      return __builtin_bit_cast(float, raw << 16);
    else
      return __builtin_bit_cast(float, raw);
  };
  auto fetch = [&](long long t, long long prev_t) {
    const bool from_h = (p.op_flags & kOpH0IsCell) != 0 && prev_t >= 0;
    const float* csrc = prev_t < 0 ? p.c0 : p.C + prev_t * bn;
    __amdgpu_buffer_rsrc_t rs_c = __builtin_amdgcn_make_buffer_rsrc((void*)csrc, 0, from_h ? 0u : (unsigned)(bn * 4), kBufFlags);
    __amdgpu_buffer_rsrc_t rs_ph = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)p.H + (size_t)(prev_t < 0 ? 0 : prev_t) * frame_bytes, 0,
                                                                     from_h ? frame_bytes : 0u, kBufFlags);
    __amdgpu_buffer_rsrc_t rs_h = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)p.H + (size_t)t * frame_bytes, 0, frame_bytes, kBufFlags);
    __amdgpu_buffer_rsrc_t rs_dy = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)p.DY + (size_t)t * dy_frame_bytes, 0, dy_frame_bytes, kBufFlags);
    auto load = [](__amdgpu_buffer_rsrc_t rs, unsigned off, int soff) -> unsigned {
      if constexpr (ES == 2)
        return __builtin_amdgcn_raw_buffer_load_b16(rs, off, soff, 0);
      else
        return __builtin_amdgcn_raw_buffer_load_b32(rs, off, soff, 0);
    };
#pragma unroll
    for (int j = 0; j < MT; ++j) {
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) in_gate[j][gq] = load(rs_h, off_h[j], gq * nc * ES);
      in_dy[j] = load(rs_dy, off_dy[j], 0);
      in_pc[j] = __builtin_amdgcn_raw_buffer_load_b32(rs_c, off_c[j], 0, 0);
      in_ph[j] = load(rs_ph, off_h[j], 0);
    }
    in_m = p.mask[t * p.B + b];
  };
  const int F = q.nframes;
  auto frame = [&](int f) { return q.t_end - (long long)f * q.step; };

  unsigned long long t0 = 0;
  auto keep_waiting = [&](unsigned& spins) {  // bookkeeping of one repeated read: false when the wait is over for good
    if ((spins++ & 15u) == 0) {
      if (__hip_atomic_load(q.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
      const unsigned long long now = wall_clock64();
      if (spins == 1) {
        t0 = now;
      } else if (now - t0 > q.timeout_ticks) {
        __hip_atomic_store(q.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
      }
    }
    return true;
  };
  auto fold = [&](unsigned (&m)[4], const i32x4& v) {
#pragma unroll
    for (int w = 0; w < 4; ++w) m[w] = LM::fold(m[w], (unsigned)v[w]);
  };
  auto seen_mark = [&](const unsigned (&m)[4]) { return __any(LM::has_sentinel(LM::fold(LM::fold(m[0], m[1]), LM::fold(m[2], m[3])))) != 0; };

  __syncthreads();  // s_one_xcd, W in LDS
  const bool one_xcd = s_one_xcd != 0;

  i32x4 bf[NB][CH];
  // d_h of the thread's pairs from the derivatives of the f-th frame, added to dyw
  auto gemm = [&](int f) {
    const unsigned slot = (unsigned)(f & (kExRing - 1)) * ex_frame, old = (unsigned)((f + 2) & (kExRing - 1)) * ex_frame;
    {
      i32x4 fv[kBwdWideForward];
      unsigned spins = 0;
      bool again;
      do {
        asm volatile("" ::: "memory");  // other workgroups write this memory: really load again
        unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < kBwdWideForward; ++i) fv[i] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ring, f_off[i], slot, kAuxDevice));
#pragma unroll
        for (int i = 0; i < kBwdWideForward; ++i) fold(m, fv[i]);
        again = seen_mark(m) && keep_waiting(spins);
      } while (again);
      const u32x4 ones = u32x4{~0u, ~0u, ~0u, ~0u};
#pragma unroll
      for (int i = 0; i < kBwdWideForward; ++i) {
        if (one_xcd) {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, fv[i]), local, f_off[i], slot, 0);
          __builtin_amdgcn_raw_buffer_store_b128(ones, local, f_off[i], old, 0);
        } else {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, fv[i]), local, f_off[i], slot, kAuxDevice);
          __builtin_amdgcn_raw_buffer_store_b128(ones, local, f_off[i], old, kAuxDevice);
        }
      }
    }
    auto load_chunk = [&](int c) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int u = 0; u < CH; ++u) {
        const int ks = c * CH + u;  // (past the share: any complete fragment, against zeros of W)
        bf[c % NB][u] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(local, b_off, slot + (ks < ks_here ? (unsigned)ks : 0u) * ks_stride, kAuxDevice));
      }
    };
    f32x4 acc[MT][NACC];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int a = 0; a < NACC; ++a) acc[mt][a] = f32x4{0.f, 0.f, 0.f, 0.f};
    unsigned spins = 0;
    auto complete = [&](int c, bool mark) {  // read chunk c again until it is complete
      while (mark && keep_waiting(spins)) {
        load_chunk(c);
        unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < CH; ++u) fold(m, bf[c % NB][u]);
        mark = seen_mark(m);
      }
    };
    load_chunk(0);
    constexpr int WP = 2;  // the fragments in LDS are read WP ahead of their MFMA
    i32x4 wl[WP];
#pragma unroll
    for (int i = 0; i < WP; ++i) wl[i] = Wl[(wave * LF + i) * 64 + lane];
    {
      unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < CH; ++u) fold(m, bf[0][u]);
      complete(0, seen_mark(m));
    }
#pragma unroll
    for (int c = 1; c < NB - 1; ++c) load_chunk(c);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (c + NB - 1 < NC) load_chunk(c + NB - 1);
      __builtin_amdgcn_sched_barrier(0);
      unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < CH; ++u) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const int at = mt * KST + c * CH + u, l = wide_lds_slot(MT, KST, RF, c * CH + u, mt);
          const i32x4 a = at < RF ? wreg[at < RF ? at : 0] : wl[l % WP];
          acc[mt][u % NACC] = E::mma(a, bf[c % NB][u], acc[mt][u % NACC]);
          if (at >= RF && l + WP < LF) wl[l % WP] = Wl[(wave * LF + l + WP) * 64 + lane];
        }
        if (c + 1 < NC) fold(m, bf[(c + 1) % NB][u]);
      }
      const bool mark = c + 1 < NC && seen_mark(m);
      __builtin_amdgcn_sched_barrier(0);
      if (c + 1 < NC) complete(c + 1, mark);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[wave][mt][(lane >> 4) * kRedGroup + (lane & 15)] = acc[mt][0] + acc[mt][1];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) sum += ((const float*)&red[w][j][red_at])[red_comp];
      dyw[j] += sum;
    }
    // (`red` is written again behind the barrier of the next frame's staging, `stage` behind the one above)
  };

  const bool raw_dh = (p.op_flags & kOpRawDh) != 0;
  fetch(frame(0), F > 1 ? frame(1) : -1);
  for (int f = 0; f < F; ++f) {
    if (f > 0) gemm(f - 1);
    // pointwise part of the frame (returnn/native_op.py:1123-1180)
    const float m = in_m;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const float dy = widen(in_dy[j]), a_fg = widen(in_gate[j][2]);
      const float pc = __builtin_bit_cast(float, in_pc[j]) + widen(in_ph[j]);
      const float err_y = raw_dh ? dy * m + dyw[j] : (dy + dyw[j]) * m;
      const float err_c = dc[j] * m;
      float dx[4];
      const float err_cell = bwd_cell<AT>(p.op_flags, widen(in_gate[j][0]), widen(in_gate[j][1]), a_fg, widen(in_gate[j][3]), pc, err_y, err_c, dx);
      dc[j] = a_fg * err_cell + dc[j] * (1.f - m);
      const int col = 16 * j + kl;
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const int at = ((gq * KGW + col / KE) * Bp + bl) * KE + col % KE;  // element index inside `stage`
        if constexpr (ES == 2)
          ((unsigned short*)stage)[at] = (unsigned short)SN::bits(dx[gq]);
        else
          ((unsigned*)stage)[at] = SN::bits(dx[gq]);
        dx0[j][gq] = raw_dh ? dx[gq] : dx[gq] + dx0[j][gq] * (1.f - m);
      }
      dyw[j] = (p.op_flags & kOpNoCarry) ? 0.f : dyw[j] * (1.f - m);
    }
    __syncthreads();  // the frame's derivatives of this workgroup are staged
    {
      const u32x4 v = __builtin_bit_cast(u32x4, stage[tid]);
      __amdgpu_buffer_rsrc_t rs_dx = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)p.DX + (size_t)frame(f) * dx_frame_bytes, 0, dx_frame_bytes, kBufFlags);
      __builtin_amdgcn_raw_buffer_store_b128(v, ring, o_ring, (unsigned)(f & (kExRing - 1)) * ex_frame, kAuxDevice);
      __builtin_amdgcn_raw_buffer_store_b128(u32x4{~0u, ~0u, ~0u, ~0u}, ring, o_ring, (unsigned)((f + 2) & (kExRing - 1)) * ex_frame, kAuxDevice);
      __builtin_amdgcn_raw_buffer_store_b128(v, rs_dx, o_dx, 0, 0);  // the op's output: a plain stream
    }
    const int fn = min(f + 1, F - 1);  // (past the end: the last frame's again, unused)
    fetch(frame(fn), fn + 1 < F ? frame(fn + 1) : -1);
  }
  gemm(F - 1);

  // After a wait that ran into its bound: NaN, as in k_lstm2_bwd_regw.
  const bool expired = wait_expired(q.status);
  if (expired && tid == 0) report_expired(q.status);
  const float nan = __builtin_nanf("");
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    if (act[j]) {
      const long long k = k0 + 16 * j + kl, at = (long long)b * nc + k;
      E::store(q.Dy0, at, expired ? nan : dyw[j]);
      p.Dc0[at] = expired ? nan : dc[j];
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) E::store(p.dx0, (long long)b * 4 * nc + k + (long long)gq * nc, expired ? nan : dx0[j][gq]);
    }
  }
}

}  // namespace rtn
