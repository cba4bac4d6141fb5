// gfx950 kernel of the NativeLstm2 forward op for bfloat16 groups of up to 8 rows: the recurrent product in sparse matrix instructions.
#pragma once

#include "lstm2_kernels.h"

namespace rtn {

// Frames per turn of the streams, and LDS copies of every stream.
constexpr int kSparseBatch = 4;
constexpr int kSparseCopies = 2 * kSparseBatch;
// LDS (bytes): partial tiles (two steps), then kSparseCopies copies each of X, H, Y, C and the mask of 8 rows.
struct SparseLds {
  unsigned red, xl, hs, ys, cs, ml, total;
  unsigned x_copy, y_copy, c_copy;
};
__host__ __device__ constexpr SparseLds sparse_lds(int MT) {
  SparseLds l{};
  l.x_copy = 8u * 32u * MT;
  l.y_copy = 8u * 8u * MT;
  l.c_copy = 8u * 16u * MT;
  unsigned off = 0;
  l.red = off; off += 2u * kWaves * (MT / 2) * kTileBytes;
  l.xl = off; off += kSparseCopies * l.x_copy;
  l.hs = off; off += kSparseCopies * l.x_copy;
  l.ys = off; off += kSparseCopies * l.y_copy;
  l.cs = off; off += kSparseCopies * l.c_copy;
  l.ml = off; off += kSparseCopies * 32u;
  l.total = off;
  return l;
}

// idx: the places of the two values stored of every four, 2 bits each
__device__ __forceinline__ f32x4 smfmac(i32x4 h, i32x8 w, f32x4 c, int idx) {
  return __builtin_amdgcn_smfmac_f32_16x16x64_bf16(__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x16, w), c, idx, 0, 0);
}

// Decomposition, exchange and order of a step are k_lstm2_regw's; what differs:
//
// The product of a dense W and a dense h in v_smfmac_f32_16x16x64_bf16.  That instruction multiplies a 16 x 64 operand of which two in
// every four values along k are zero and not stored with a dense 64 x 16 one, in the 16 clocks of the dense 16x16x32: twice the k.
// Here h is the operand with the zeros and W the dense one.  A group of at most 8 rows would leave half of the 16 rows to padding, so
// every row of h takes two: one holds its values of macro step 2a at places 0 and 1 of every four, the other those of step 2a + 1
// at places 2 and 3, and W's two steps are interleaved to match (a lane's registers hold two k of step 2a and two of step 2a + 1 in turn).
// Nothing is left out and no product is rounded: the two rows of a result are the sums over the wavefront's even and its odd macro steps,
// added before the partial tile leaves for LDS -- the two chains of additions (two_chains) that every kernel of these widths makes, the
// same bits from all of them.  MT * KS / 2 matrix instructions per wavefront and step in place of MT * KS, no masking and shifting of h into
// operand forms, and h comes in as 1 KB of consecutive memory per load.  (In the instruction's result a lane has one gate column and two rows'
// sums; with 16 cells of one gate per tile a lane has all gates of a cell.)
//
// The streams X, mask, H, Y and C move in turns of four frames.  What a wavefront loads and stores ends in the order it was issued, and a
// CU's first-level cache answers its wavefronts in order as well, so a load of X holds up every load of h behind it for as long as
// memory takes (0.84 us under this load).  Moved frame by frame, as k_lstm2_regw does, a pair of 32 rows of n = 1024 took 1.31 us per step (1.13
// with no streams at all); in turns of four, X, H and the rest each in a step of their own, 1.25 (all in one step 1.34: loads and
// stores then meet in memory), and chunks of 16 bytes fill the wavefronts.  Chunks lie in LDS without padding, rotated by row so
// that 8 rows of 8 cells touch every bank once.
// What bounds it, n = 1024: of 1.25 us the MFMAs are 0.28, partial tiles through LDS, gates and stores 0.5, the hand-over 0.35.  us per step before
// (two tiles in one accumulator of the dense instruction) and now: pair of 32 rows 1.38 / 1.25, pair of 16 rows 1.38 / 1.19, one row 1.32 / 1.11,
// n = 768, 24 rows 1.35 / 1.16; n = 512, 32 rows 1.06 / 0.89; n = 256, 100 rows 1.03 / 0.89.
template <int MT, int KS, bool TAIL>
__global__ __launch_bounds__(kWgThreads) void k_lstm2_sparse(const Lstm2Multi multi) {
  static_assert((MT == 2 || MT == 4 || MT == 8) && KS % 2 == 0 && two_chains<__bf16>(KS), "no such build");
  using AT = __bf16;
  using E = Elem<AT>;
  using SN = Sentinel<AT>;
  using LM = LaneMax<AT>;
  // (workgroup ids as k_lstm2_regw deals them in XCD-local plans, the only ones with groups of so few rows)
  const int X = multi.xcds, G = multi.p[0].wgs_per_group, per = multi.p[0].groups;
  const int xcd = (int)blockIdx.x % X, slot = (int)blockIdx.x / X, gg = (slot / G) * X + xcd, which = gg / per;
  if (which >= multi.count) return;
  int g = gg - which * per;
  const int r = slot % G;
  const Lstm2Params p = multi.p[which];
  constexpr int ES = 2, KM = E::KM, NP = KS / 2;  // NP: pairs of macro steps per wavefront
  constexpr int CELLS = 4 * MT, UNITS = MT / 2;   // a unit: 8 cells of 8 rows, one per lane of a wavefront
  constexpr int FB = kSparseBatch;
  constexpr SparseLds L = sparse_lds(MT);

  extern __shared__ __align__(16) unsigned char smem[];
  typedef f32x4 RedBuf[kWaves][UNITS][64];
  RedBuf* red = (RedBuf*)(smem + L.red);  // [2]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = p.n, S = n / KM, nc = p.nc, nsteps = p.nsteps;
  g += p.group_offset;
  const int b_base = g * p.Bg;
  const int rows = min(p.Bg, p.B - b_base);
  const long long bn = (long long)p.B * nc;
  const int cell0 = CELLS * r;
  const int kg = lane >> 4, jl = lane & 15;

  // ---- streams: 16-byte chunks of a frame (8 rows); this wavefront's chunks of a turn of FB frames are XI chunks per lane of X and
  // of H (frames xf, xf + 2) and one of Y, C and the mask (frame `wave`).  Chunks that do not exist carry an out-of-range offset.
  constexpr int CPS = MT / 2, XROW = 4 * CPS;     // chunks of one (row, gate), and of a row of X or H
  constexpr int XI = MT == 8 ? 2 : 1;
  typedef Chunk<16> CK;
  auto sw_x = [](int row) { return (row ^ (row >> 2)) & (XROW - 1); };
  auto sw_y = [](int row) { return MT == 8 ? (row >> 2) & 1 : 0; };
  auto sw_c = [](int row) { return MT == 8 ? (row >> 1) & 3 : MT == 4 ? (row >> 2) & 1 : 0; };
  const int xf = MT == 8 ? wave >> 1 : wave;
  const int xc = MT == 8 ? 64 * (wave & 1) + lane : lane;  // chunk of the frame
  const bool xc_there = xc < 8 * XROW;
  unsigned xoff, hoff, yoff, coff;
  {
    const int row = xc / XROW, gp = (xc % XROW) ^ sw_x(row), gate = gp / CPS, part = gp % CPS;
    const bool there = xc_there && row < rows && cell0 + (part + 1) * 8 <= nc;
    xoff = there ? (unsigned)(((long long)(b_base + row) * p.ldX + gate * nc + cell0) * ES + part * 16) : kOobOffset;
    hoff = there ? (unsigned)(((long long)(b_base + row) * 4 * nc + gate * nc + cell0) * ES + part * 16) : kOobOffset;
  }
  {
    const int row = lane / CPS, part = (lane % CPS) ^ sw_y(row);
    yoff = lane < 8 * CPS && row < rows && cell0 + (part + 1) * 8 <= nc ? (unsigned)(((long long)(b_base + row) * p.ldY + cell0) * ES + part * 16) : kOobOffset;
  }
  {
    const int row = lane / MT, in = lane % MT, cl = 8 * ((in >> 1) ^ sw_c(row)) + 4 * (in & 1);
    coff = lane < 8 * MT && row < rows && cell0 + cl + 4 <= nc ? (unsigned)(((b_base + row) * nc + cell0 + cl) * 4) : kOobOffset;
  }
  const unsigned moff = lane < rows ? (unsigned)((b_base + lane) * 4) : kOobOffset;
  // where this lane's chunks lie inside a copy (lanes without one: the chunk of another lane, which they only read)
  const unsigned xlds = (unsigned)(xc_there ? xc : 0) * 16, ylds = (unsigned)(lane % (8 * CPS)) * 16, clds = (unsigned)(lane % (8 * MT)) * 16;
  const unsigned frame_x = (unsigned)((size_t)p.B * p.ldX * ES), frame_h = (unsigned)((size_t)p.B * 4 * nc * ES),
                 frame_y = (unsigned)((size_t)p.B * p.ldY * ES), frame_c = (unsigned)(bn * 4), frame_m = (unsigned)(p.B * 4);
  const long long step_x = (long long)p.step * frame_x, step_h = (long long)p.step * frame_h, step_y = (long long)p.step * frame_y,
                  step_c = (long long)p.step * frame_c, step_m = (long long)p.step * frame_m;
  // The frames of the next turn (X and mask in, outputs out); signed steps: the op may run backwards in time.
  const unsigned char* x_at = (const unsigned char*)p.X + (long long)p.first * frame_x + xf * step_x;
  const unsigned char* m_at = (const unsigned char*)p.mask + (long long)p.first * frame_m + wave * step_m;
  unsigned char* h_at = (unsigned char*)p.H + (long long)p.first * frame_h + xf * step_h;
  unsigned char* y_at = (unsigned char*)p.Y + (long long)p.first * frame_y + wave * step_y;
  unsigned char* c_at = (unsigned char*)p.C + (long long)p.first * frame_c + wave * step_c;
  CK::T xv[XI], fh[XI], fy, fc;
  float mv = 0.f;
  auto fetch = [&](int s0) {  // X and mask of frames s0 ... s0 + FB - 1 (s0: the next turn's) into registers
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)(x_at + 2 * i * step_x), 0, s0 + xf + 2 * i < nsteps ? frame_x : 0u, kBufFlags);
      xv[i] = CK::load(xr, xoff);
    }
    __amdgpu_buffer_rsrc_t mr = __builtin_amdgcn_make_buffer_rsrc((void*)m_at, 0, s0 + wave < nsteps ? frame_m : 0u, kBufFlags);
    mv = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(mr, moff, 0, 0));
    x_at += FB * step_x;
    m_at += FB * step_m;
  };
  auto put = [&](int s0) {  // registers -> the copies of those frames
    const unsigned c0 = (unsigned)s0 & (kSparseCopies - 1);
    if (xc_there) {
#pragma unroll
      for (int i = 0; i < XI; ++i) *(CK::T*)(smem + L.xl + (c0 + xf + 2 * i) * L.x_copy + xlds) = xv[i];
    }
    if (lane < 8) *(float*)(smem + L.ml + (c0 + wave) * 32 + lane * 4) = mv;
  };
  auto flush_read_h = [&](int s0) {  // staged outputs of frames s0 ... s0 + FB - 1 -> registers
    const unsigned c0 = (unsigned)s0 & (kSparseCopies - 1);
#pragma unroll
    for (int i = 0; i < XI; ++i) fh[i] = *(const CK::T*)(smem + L.hs + (c0 + xf + 2 * i) * L.x_copy + xlds);
  };
  auto flush_read_yc = [&](int s0) {
    const unsigned c0 = (unsigned)s0 & (kSparseCopies - 1);
    fy = *(const CK::T*)(smem + L.ys + (c0 + wave) * L.y_copy + ylds);
    fc = *(const CK::T*)(smem + L.cs + (c0 + wave) * L.c_copy + clds);
  };
  auto flush_h = [&](int s0) {  // ... -> H, Y, C (frames that do not exist: buffers of no bytes)
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int f = s0 + xf + 2 * i;
      __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc((void*)(h_at + 2 * i * step_h), 0, f >= 0 && f < nsteps ? frame_h : 0u, kBufFlags);
      CK::store(fh[i], hr, hoff);
    }
    h_at += s0 >= 0 ? FB * step_h : 0;
  };
  auto flush_yc = [&](int s0) {
    const int f = s0 + wave;
    const bool there = f >= 0 && f < nsteps;
    __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc((void*)y_at, 0, there ? frame_y : 0u, kBufFlags);
    __amdgpu_buffer_rsrc_t cr = __builtin_amdgcn_make_buffer_rsrc((void*)c_at, 0, there ? frame_c : 0u, kBufFlags);
    CK::store(fy, yr, yoff);
    CK::store(fc, cr, coff);
    y_at += s0 >= 0 ? FB * step_y : 0;
    c_at += s0 >= 0 ? FB * step_c : 0;
  };

  // ---- the recurrence
  const unsigned hx_buf_bytes = (unsigned)((size_t)n * p.Bp * ES);
  unsigned char* hx_g = (unsigned char*)p.hx + (size_t)g * kHxRing * hx_buf_bytes;
  __amdgpu_buffer_rsrc_t ring_rs = __builtin_amdgcn_make_buffer_rsrc((void*)hx_g, 0, kHxRing * hx_buf_bytes, kBufFlags);
  const int ks_count = (S > wave) ? (S - wave + kWaves - 1) / kWaves : 0;  // macro steps of this wave

  // W of this wavefront's share, for the whole sequence; pairs past the share hold zeros and meet zeros.
  i32x8 w[MT][NP];
  unsigned foff[NP];  // where this lane's fragments of h are inside a ring buffer
  {
    const int pairs = sparse_pairs(S);
#pragma unroll
    for (int a = 0; a < NP; ++a) {
      foff[a] = 2 * a + sparse_row_half(jl) < ks_count && sparse_row(jl) < rows ? (unsigned)((((kWaves * a + wave) * 4 + kg) * 16 + jl) * kFragBytes) : kOobOffset;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        i32x4 x = i32x4{0, 0, 0, 0}, y = x;
        if (2 * a < ks_count) {
          const i32x4* src = (const i32x4*)p.Wp + ((size_t)(r * MT + mt) * pairs + kWaves * a + wave) * 128 + lane;
          x = src[0];
          y = src[64];
        }
        w[mt][a] = i32x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
      }
    }
  }

  // The (sequence, cell) pair whose state this thread keeps: row lane / 8, cell lane % 8 of unit `wave`.
  const int unit = min(wave, UNITS - 1), row = lane >> 3, cl = 8 * unit + (lane & 7), cell = cell0 + cl;
  const bool active = UNITS >= kWaves || wave < UNITS;  // uniform over the wavefront
  const bool valid = active && row < rows && cell < nc;
  const unsigned e_hoff = sparse_hx(row, cell) * ES;
  unsigned goff[4];  // the pair's gates in a copy of X or H
#pragma unroll
  for (int q = 0; q < 4; ++q) goff[q] = (unsigned)(row * (16 * XROW) + ((q * CPS + unit) ^ sw_x(row)) * 16 + (lane & 7) * ES);
  const unsigned y_in = (unsigned)(row * 16 * CPS + (unit ^ sw_y(row)) * 16 + (lane & 7) * ES);
  const unsigned c_in = (unsigned)(row * 16 * MT + (unit ^ sw_c(row)) * 32 + (lane & 7) * 4);
  float c_state, h_prev;
  start_state<AT>(p, valid, (b_base + row) * nc + cell, &c_state, &h_prev);
  // The tail (see k_lstm2_regw): first cell of the chunk of X, H and Y, and of C, that the width cuts.
  const int tail_x = nc - nc % 8 - cell0, tail_c = nc - nc % 4 - cell0;
  const bool has_tail = TAIL && nc % 8 != 0 && tail_x >= 0 && tail_x < CELLS;  // uniform over the workgroup
  const bool in_tail = valid && cl >= tail_x;
  AT x_tail[4] = {(AT)0.f, (AT)0.f, (AT)0.f, (AT)0.f};
  auto fetch_tail = [&](int s) {  // the tail's gate inputs of step s, from memory
    if (in_tail) {
      const AT* xp = (const AT*)p.X + ((size_t)frame_of(p, s) * p.B + b_base + row) * (size_t)p.ldX + cell;
#pragma unroll
      for (int q = 0; q < 4; ++q) x_tail[q] = xp[(size_t)q * nc];
    }
  };

  __shared__ int s_local;  // (that all workgroups of a group share an XCD is checked, as in k_lstm2_regw)
  if (wave == 0)
    s_local = group_on_one_xcd(p.flags + (size_t)g * p.wgs_per_group, (unsigned)p.wgs_per_group, p.status, p.timeout_ticks) ? 1 : 0;

  auto run = [&](auto ex_tag) {
    constexpr int EX = decltype(ex_tag)::value;
    constexpr int AUXS = (EX == kExDevice) ? kAuxDevice : 0, AUXL = kAuxDevice;
    i32x4 bf[NP];
#pragma unroll
    for (int a = 0; a < NP; ++a) bf[a] = i32x4{0, 0, 0, 0};
    auto issue = [&](int s) {  // the loads of this wave's fragments of ring buffer s % 4
      const unsigned soff = (unsigned)(s & (kHxRing - 1)) * hx_buf_bytes;
      asm volatile("" ::: "memory");  // other workgroups write this memory: really load again
      if constexpr (EX == kExNoWait) return;
      if (sparse_row(jl) < rows) {
#pragma unroll
        for (int a = 0; a < NP; ++a) bf[a] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ring_rs, foff[a], soff, AUXL));
      }
    };
    AT x_in[2][4];
    float m_in[2];
    auto load_gate_inputs = [&](int s, auto par_tag) {  // of step s, from its copy
      constexpr int PAR = decltype(par_tag)::value;
      const unsigned copy = (unsigned)s & (kSparseCopies - 1);
      const unsigned char* xin = smem + L.xl + copy * L.x_copy;
#pragma unroll
      for (int q = 0; q < 4; ++q) x_in[PAR][q] = *(const AT*)(xin + goff[q]);
      m_in[PAR] = *(const float*)(smem + L.ml + copy * 32 + row * 4);
    };
    float x_f[4], m_f = 0.f, keep_c = 0.f, keep_h = 0.f;
    auto widen_gate_inputs = [&](auto par_tag) {
      constexpr int PAR = decltype(par_tag)::value;
#pragma unroll
      for (int q = 0; q < 4; ++q) x_f[q] = (float)x_in[PAR][q];
      m_f = m_in[PAR];
      const float om = 1.f - m_f;
      keep_c = c_state * om;
      keep_h = h_prev * om;
    };
    RTN_TRACE_DECL
    constexpr bool spread_after_all = EX == kExDevice;
    int delay = EX == kExNoWait ? 0 : spread_after_all ? 20 : p.poll_delay;
    const int delay_inc = spread_after_all ? 2 : p.delay_inc;
    const int idx = sparse_row_half(jl) ? (int)0xEEEEEEEE : 0x44444444;
    // One time step; PH = s % FB.  The streams' turn, behind the MFMAs, with PH == 1: X and mask of the four frames that start with
    // s + 3 are asked for; they go to LDS with PH == 2 and are read there from the step after that on.  The last four frames' outputs
    // (a barrier lies behind their staging) go out with PH == 2 (H) and PH == 3 (Y and C).
    auto step = [&](int s, auto ph_tag) {
      constexpr int PH = decltype(ph_tag)::value, PAR = PH & 1;
      unsigned stage = (unsigned)s & (kSparseCopies - 1);
      asm volatile("" : "+s"(stage));
      // (the accumulators have to be cleared by instructions of their own, which go here, where nothing else is to do)
      f32x4 acc[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+v"(acc[mt]));
      }
      unsigned long long t0 = 0;
      unsigned spins = 0;
      for (;;) {
        unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
        for (int a = 0; a < NP; ++a)
#pragma unroll
          for (int q = 0; q < 4; ++q) m[q] = LM::fold(m[q], (unsigned)bf[a][q]);
        const unsigned seen = LM::fold(LM::fold(m[0], m[1]), LM::fold(m[2], m[3]));
        if (EX == kExNoWait || !__any(LM::has_sentinel(seen))) break;
        if ((spins++ & 15u) == 0) {
          if (__hip_atomic_load(p.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
          const unsigned long long now = wall_clock64();
          if (spins == 1) {
            t0 = now;
          } else if (now - t0 > p.timeout_ticks) {
            __hip_atomic_store(p.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
          }
        }
        issue(s);
      }
      RTN_TRACE_MARK(0)
      // Everything this wave stored before (re-arm stores included) is acknowledged, and X that was asked for is there.
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
      asm volatile("" ::: "memory");
      if (spins)
        delay = min(delay + delay_inc, 64);
      else if (delay_inc && (s & p.delay_dec_mask) == p.delay_dec_mask && delay > 0)
        --delay;
      RTN_TRACE_MARK(7)

      // The MFMAs in chunks of one per accumulator or less, a full scheduling fence between chunks, the step's other work dealt to them.
      RedBuf& redbuf = red[PAR];
      constexpr int CHUNK = MT < 4 ? MT : 4, NCH = NP * MT / CHUNK;
#pragma unroll
      for (int c = 0; c < NCH; ++c) {
        auto at = [&](int want) { return c == (want < NCH ? want : NCH - 1); };
        if (PH == 2 && at(0)) flush_read_h(s - FB - 2);
        if (PH == 3 && at(0)) flush_read_yc(s - FB - 3);
        if (at(1)) load_gate_inputs(s + 1, IntTag<1 - PAR>{});
        if (PH == 2 && at(2)) put(s + 2);
        if (PH == 2 && at(3)) flush_h(s - FB - 2);
        if (PH == 3 && at(3)) flush_yc(s - FB - 3);
        if (PH == 1 && at(5)) fetch(s + FB - 1);
        if (at(5)) widen_gate_inputs(IntTag<PAR>{});
#pragma unroll
        for (int u = 0; u < CHUNK; ++u) {
          const int a = c * CHUNK / MT, mt = c * CHUNK % MT + u;
          acc[mt] = smfmac(bf[a], w[mt][a], acc[mt], idx);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x096, 3, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (MT >= 4) {
        // tile 4 v + gate: the lane's cell is number lane % 16 of the v-th sixteen, rows 2 (lane / 16) and 2 (lane / 16) + 1
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
          f32x4 v;
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = acc[4 * (u >> 1) + q][u & 1] + acc[4 * (u >> 1) + q][2 + (u & 1)];
          redbuf[wave][2 * (u >> 1) + (jl >> 3)][(2 * kg + (u & 1)) * 8 + (jl & 7)] = v;
        }
      } else {
        // 8 cells: lane % 16 is cell lane % 8, and its upper half the last two gates
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          float* dst = (float*)&redbuf[wave][0][(2 * kg + q) * 8 + (jl & 7)] + 2 * (jl >> 3);
          *(f32x2*)dst = f32x2{acc[0][q] + acc[0][2 + q], acc[1][q] + acc[1][2 + q]};
        }
      }
      if (has_tail && in_tail) {
#pragma unroll
        for (int q = 0; q < 4; ++q) x_f[q] = (float)x_tail[q];
      }
      RTN_TRACE_MARK(1)
      __syncthreads();  // the one barrier of a step
      RTN_TRACE_MARK(2)

      float g_act[4], y_out = 0.f;
      if (active) {
        f32x4 part[kWaves];
#pragma unroll
        for (int v = 0; v < kWaves; ++v) part[v] = redbuf[v][unit][lane];
        __builtin_amdgcn_sched_barrier(0);
        f32x4 gsum = part[0];
#pragma unroll
        for (int v = 1; v < kWaves; ++v) gsum += part[v];
        const float a0 = Act<AT>::tanh(gsum[0] + x_f[0]);
        const float a1 = Act<AT>::sigmoid(gsum[1] + x_f[1]);
        const float a2 = Act<AT>::sigmoid(gsum[2] + x_f[2]);
        const float a3 = Act<AT>::sigmoid(gsum[3] + x_f[3]);
        const float c = (c_state * a2 + a0 * a1) * m_f + keep_c;
        const float y = E::round(Act<AT>::tanh(c) * a3 * m_f);
        const float hn = (p.op_flags & kOpNoCarry) ? y : E::round(y + keep_h);
        c_state = c;
        h_prev = hn;
        g_act[0] = (p.op_flags & kOpH0IsCell) ? c : a0;
        g_act[1] = a1; g_act[2] = a2; g_act[3] = a3;
        y_out = y;
        // New hidden values out; re-arm the elements everybody read one step ago (rows the group does not have own slots too).
        const unsigned nxt = (unsigned)((s + 1) & (kHxRing - 1)) * hx_buf_bytes, arm = (unsigned)((s + 3) & (kHxRing - 1)) * hx_buf_bytes;
        SN::template store<AUXS>(ring_rs, e_hoff + nxt, SN::bits(hn));
        SN::template store<AUXS>(ring_rs, e_hoff + arm, SN::kSentinel);
        RTN_TRACE_MARK(3)
        unsigned char* hq = smem + L.hs + stage * L.x_copy;
#pragma unroll
        for (int q = 0; q < 4; ++q) *(AT*)(hq + goff[q]) = (AT)g_act[q];
        *(AT*)(smem + L.ys + stage * L.y_copy + y_in) = (AT)y_out;
        *(float*)(smem + L.cs + stage * L.c_copy + c_in) = c_state;
      }
      if (has_tail) {
        if (in_tail) {
          const size_t at = (size_t)frame_of(p, s) * p.B + b_base + row;
#pragma unroll
          for (int q = 0; q < 4; ++q) ((AT*)p.H)[at * 4 * nc + (size_t)q * nc + cell] = (AT)g_act[q];
          ((AT*)p.Y)[at * (size_t)p.ldY + cell] = (AT)y_out;
          if (cl >= tail_c) p.C[at * nc + cell] = c_state;
        }
        if (s + 1 < nsteps) fetch_tail(s + 1);
      }
      if (s + 1 < nsteps) {
        for (int k = 0; k < delay; ++k) __builtin_amdgcn_s_sleep(1);
        issue(s + 1);
      }
      RTN_TRACE_MARK(4)
    };
    fetch(0);
    put(0);
    __syncthreads();
    load_gate_inputs(0, IntTag<0>{});
    if (has_tail) fetch_tail(0);
    issue(0);
    for (int s = 0; s < nsteps; s += FB) {
      step(s, IntTag<0>{});
      if (s + 1 < nsteps) step(s + 1, IntTag<1>{});
      if (s + 2 < nsteps) step(s + 2, IntTag<2>{});
      if (s + 3 < nsteps) step(s + 3, IntTag<3>{});
    }
    RTN_TRACE_ADD(6, (unsigned long long)delay << 40)
    RTN_TRACE_FLUSH(p, which * p.groups * p.wgs_per_group + (g - p.group_offset) * p.wgs_per_group + r)
  };
  __syncthreads();  // s_local
  if (!TAIL && p.exchange == kExNoWait) {
    if (tid == 0) __hip_atomic_store(p.status, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if constexpr (!TAIL) run(IntTag<kExNoWait>{});
  } else if (s_local) {
    run(IntTag<kExLocal>{});
  } else {
    run(IntTag<kExDevice>{});
  }
  __syncthreads();  // the last step's outputs are staged
  // (As in k_lstm2_regw: an expired wait must show in what a consumer reads.)
  const bool expired = wait_expired(p.status);
  if (expired && tid == 0) report_expired(p.status);
  // the frames since the last turns of the loop
  for (int s0 = nsteps >= 3 ? (nsteps - 3) / FB * FB : 0; s0 < nsteps; s0 += FB) {
    flush_read_h(s0);
    flush_h(s0);
  }
  for (int s0 = nsteps >= 4 ? (nsteps - 4) / FB * FB : 0; s0 < nsteps; s0 += FB) {
    flush_read_yc(s0);
    if (expired && s0 + wave == nsteps - 1) fy = CK::fill(kNanWords<AT>);
    flush_yc(s0);
  }
  if (valid) {
    const long long bc = (long long)(b_base + row) * nc + cell;
    p.d[bc] = expired ? __builtin_nanf("") : c_state;
    if (p.hN) E::store(p.hN, bc, expired ? __builtin_nanf("") : h_prev);
  }
  if (expired && has_tail) {  // the tail's cells of the last frame, which went out by themselves (see k_lstm2_regw)
    const int l = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0)), bl = l >> 3, in = 8 * unit + (l & 7);
    if (active && bl < rows && in >= tail_x && cell0 + in < nc)
      E::store(p.Y, ((long long)frame_of(p, nsteps - 1) * p.B + b_base + bl) * p.ldY + cell0 + in, __builtin_nanf(""));
  }
}

}  // namespace rtn
