// gfx950 kernel of the NativeLstm2 forward op for batches that take the register kernel several launches: two launches' rows
// in one, taken in turn step by step.
#pragma once

#include "lstm2_kernels.h"

namespace rtn {

// LDS: the partial tiles of either set, then per set one copy of X and the mask and of the staged H, Y and C.
struct DualLds {
  unsigned red, xl, hs, ys, cs, ml, set, total;  // xl ... ml: inside a set's part, which starts at red + index * set behind the tiles
  unsigned x_row, y_row, c_row;
};
__host__ __device__ constexpr DualLds dual_lds(int es, int MT) {
  DualLds l{};
  const unsigned cells = 4u * MT;
  l.x_row = 4u * cells * es + kRowPad;
  l.y_row = cells * es + kRowPad;
  l.c_row = cells * 4u + kRowPad;
  l.red = 2u * kWaves * MT * kTileBytes;
  unsigned off = 0;
  l.xl = off; off += 16u * l.x_row + 16u;
  l.hs = off; off += 16u * l.x_row + 16u;
  l.ys = off; off += (16u * l.y_row + 15u) / 16u * 16u;
  l.cs = off; off += 16u * l.c_row;
  l.ml = off; off += 16u * 4u + 16u;
  l.set = off;
  l.total = l.red + 2u * l.set;
  return l;
}

// A workgroup holds its slice of W in registers as k_lstm2_regw does and works on TWO groups of up to 16 rows with it: group
// g of multi.p[0] and group g of multi.p[1] (the same problem at another group_offset).  A step of one group is a chain --
// hidden state in, MFMAs, partial tiles through LDS, gates, hidden state out and to every other CU of the XCD -- of which the
// matrix cores take a fifth and the hand-over about half; here the one group's hand-over runs while the other's products and
// gates are worked on.  Each half step asks for the other group's hidden state behind its MFMAs (it left its writers half a
// step ago), so that what remains exposed are the two groups' own MFMAs, barriers and gates.
// With two barriers per step one LDS copy of every stream is enough: X and the mask of one group move from registers to LDS
// in the other group's half, staged outputs leave in the own group's next half.
// What bounds it now is how fast one wavefront per SIMD issues: of 7500 clocks per wavefront and step of both groups (bf16
// n = 1024, B = 256: 3.3 us, 4.3 in turns) the matrix cores are busy for 2050, vector instructions issue in 2300, 2200 go by with an
// instruction waiting for its turn and 1600 with none to issue; 23 % of the clocks the LDS is busy are bank conflicts.  (The gates
// of one group woven into the other's MFMAs left the hand-over exposed: 842 us against 690.)
// SPREAD: groups over all XCDs, for layers of 1024 < n <= 2048, which no XCD holds.  There a step alone is mostly hand-over (of 7400 clocks
// of 32 rows of n = 2048 the matrix cores had 1400): n = 2048, B = 64, T = 64 4.3 us per step of both, 5.7 in turns; n = 1280, B = 90 3.8, 9.5 in the
// three turns that two tiles of rows per workgroup made.  What is left of it, 8800 clocks per step of both: MFMAs 2050, vector instructions 2100, 3200 with an
// instruction waiting for its turn, 2000 with none to issue (all 256 registers are taken, and 12 more in scratch).
// The order of additions is that of k_lstm2_regw: the same bits.
template <typename AT, int MT, int KS, bool SPREAD>
__global__ __launch_bounds__(kWgThreads) void k_lstm2_dual(const Lstm2Multi multi) {
  using E = Elem<AT>;
  using SN = Sentinel<AT>;
  using LM = LaneMax<AT>;
  constexpr int KE = E::KE, KM = E::KM, ES = (int)sizeof(AT);
  constexpr int EPT = MT / kWaves, CELLS = 4 * MT, ROWS = 16;
  static_assert(MT == kWaves || MT == 2 * kWaves, "one or two pairs per thread in the pointwise part");
  typedef AT Cells __attribute__((ext_vector_type(EPT)));  // the thread's cells of a row
  constexpr DualLds L = dual_lds(ES, MT);
  const Lstm2Params p = multi.p[0];
  const int X = multi.xcds, G = p.wgs_per_group;
  int g, r;
  if constexpr (SPREAD) {
    map_block(p, (int)blockIdx.x, g, r);
  } else {
    const int xcd = (int)blockIdx.x % X, slot = (int)blockIdx.x / X;
    g = (slot / G) * X + xcd;
    r = slot % G;
  }
  if (g >= p.groups) return;

  extern __shared__ __align__(16) unsigned char smem[];
  typedef f32x4 RedBuf[kWaves][MT][64];
  RedBuf* red = (RedBuf*)smem;  // [2]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = p.n, S = n / KM, nc = p.nc, nsteps = p.nsteps;
  const long long bn = (long long)p.B * nc;
  const int group[2] = {g + p.group_offset, g + multi.p[1].group_offset};
  const int kg = lane >> 4, jl = lane & 15;

  // Streams, as in k_lstm2_regw; offsets are relative to a group's first row, rows beyond the batch end lie behind the frame.
  constexpr int SEG = CELLS * ES, CPS = SEG / 16, XCH = (ROWS * 4 * CPS + kWgThreads - 1) / kWgThreads;
  constexpr int SEGC = CELLS * 4;
  static_assert(ROWS * CPS <= 64 && ROWS * (SEGC / 16) <= 128, "wavefront 0 moves Y, wavefronts 1 and 2 move C");
  typedef Chunk<16> CK;
  const int cell0 = CELLS * r;
  unsigned xoff[XCH], hoff[XCH], xlds[XCH];
  // (a chunk of Y or of C per thread, by wavefront: one load from LDS and one store where one of each left most lanes without any)
  const bool moves_y = wave == 0;
  unsigned ycoff = kOobOffset, yclds = 0;
#pragma unroll
  for (int i = 0; i < XCH; ++i) {
    const int c = tid + kWgThreads * i;
    const int row = c / (4 * CPS), gate = (c / CPS) % 4, part = c % CPS;
    const bool there = row < p.Bg && cell0 + (part + 1) * KE <= nc;
    xoff[i] = there ? (unsigned)(((long long)row * p.ldX + gate * nc + cell0) * ES + part * 16) : kOobOffset;
    hoff[i] = there ? (unsigned)(((long long)row * 4 * nc + gate * nc + cell0) * ES + part * 16) : kOobOffset;
    xlds[i] = row < ROWS ? (unsigned)(row * L.x_row + gate * SEG + part * 16) : (unsigned)(ROWS * L.x_row);
  }
  if (moves_y) {
    const int row = tid / CPS, part = tid % CPS;
    if (row < p.Bg && cell0 + (part + 1) * KE <= nc) ycoff = (unsigned)(((long long)row * p.ldY + cell0) * ES + part * 16);
    yclds = L.ys + (unsigned)(min(row, ROWS - 1) * L.y_row + part * 16);
  } else {
    const int c = tid - 64, row = c / (SEGC / 16), part = c % (SEGC / 16);
    if (row < p.Bg && cell0 + (part + 1) * 4 <= nc) ycoff = (unsigned)((row * nc + cell0) * 4 + part * 16);
    yclds = L.cs + (unsigned)(min(row, ROWS - 1) * L.c_row + part * 16);
  }
  const unsigned moff = tid < p.Bg ? (unsigned)(tid * 4) : kOobOffset;
  const long long frame_x = (long long)p.B * p.ldX * ES, frame_h = (long long)p.B * 4 * nc * ES, frame_y = (long long)p.B * p.ldY * ES,
                  frame_c = bn * 4, frame_m = (long long)p.B * 4;

  // ---- per group
  const unsigned hx_buf_bytes = (unsigned)((size_t)n * p.Bp * ES);
  __amdgpu_buffer_rsrc_t ring[2];
  const unsigned char *x_at[2], *m_at[2];  // the frame that is fetched next, at the group's first row
  unsigned char *h_at[2], *yc_at[2];  // the frame whose staged outputs leave next
  unsigned left_x[2], left_h[2], left_yc[2], left_m[2];  // bytes of a frame from the group's first row on (0: no such row)
  unsigned frag[2];  // this lane's fragment of macro step `wave` in a ring buffer; out of range: a row the group does not have
  int rows[2];
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const long long b0 = (long long)group[d] * p.Bg, t0 = frame_of(p, 0);
    rows[d] = (int)max(0LL, min((long long)p.Bg, p.B - b0));
    ring[d] = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)p.hx + (size_t)group[d] * kHxRing * hx_buf_bytes, 0, kHxRing * hx_buf_bytes, kBufFlags);
    const long long bs = min(b0, (long long)p.B);
    x_at[d] = (const unsigned char*)p.X + t0 * frame_x + bs * p.ldX * ES;
    m_at[d] = (const unsigned char*)p.mask + t0 * frame_m + bs * 4;
    h_at[d] = (unsigned char*)p.H + t0 * frame_h + bs * 4 * nc * ES;
    yc_at[d] = moves_y ? (unsigned char*)p.Y + t0 * frame_y + bs * p.ldY * ES : (unsigned char*)p.C + t0 * frame_c + bs * nc * 4;
    left_x[d] = (unsigned)(frame_x - bs * p.ldX * ES);
    left_h[d] = (unsigned)(frame_h - bs * 4 * nc * ES);
    left_yc[d] = moves_y ? (unsigned)(frame_y - bs * p.ldY * ES) : (unsigned)(frame_c - bs * nc * 4);
    left_m[d] = (unsigned)(frame_m - bs * 4);
    frag[d] = jl < rows[d] ? (unsigned)(((4 * wave + kg) * p.Bp + jl) * kFragBytes) : kOobOffset;
  }
  const long long step_x = (long long)p.step * frame_x, step_h = (long long)p.step * frame_h, step_yc = (long long)p.step * (moves_y ? frame_y : frame_c),
                  step_m = (long long)p.step * frame_m;
  CK::T xv[2][XCH];
  float mv[2] = {0.f, 0.f};
  auto fetch = [&](auto set_tag, bool enabled) {  // the next frame of X and the mask into registers
    constexpr int D = decltype(set_tag)::value;
    __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)x_at[D], 0, enabled ? left_x[D] : 0u, kBufFlags);
    __amdgpu_buffer_rsrc_t mr = __builtin_amdgcn_make_buffer_rsrc((void*)m_at[D], 0, enabled ? left_m[D] : 0u, kBufFlags);
#pragma unroll
    for (int i = 0; i < XCH; ++i) xv[D][i] = CK::load(xr, xoff[i]);
    mv[D] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(mr, moff, 0, 0));
    x_at[D] += step_x;
    m_at[D] += step_m;
  };
  auto put = [&](auto set_tag) {  // registers -> LDS
    constexpr int D = decltype(set_tag)::value;
    unsigned char* base = smem + L.red + D * L.set;
#pragma unroll
    for (int i = 0; i < XCH; ++i) *(CK::T*)(base + L.xl + xlds[i]) = xv[D][i];
    ((float*)(base + L.ml))[tid < ROWS ? tid : ROWS] = mv[D];
  };
  CK::T fh[XCH], fyc;
  auto flush_read = [&](auto set_tag) {  // staged outputs -> registers
    constexpr int D = decltype(set_tag)::value;
    const unsigned char* base = smem + L.red + D * L.set;
#pragma unroll
    for (int i = 0; i < XCH; ++i) fh[i] = *(const CK::T*)(base + L.hs + xlds[i]);
    fyc = *(const CK::T*)(base + yclds);
  };
  auto flush_write = [&](auto set_tag, bool enabled) {  // ... -> H, Y, C (a frame that does not exist: a buffer of no bytes)
    constexpr int D = decltype(set_tag)::value;
    __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc((void*)h_at[D], 0, enabled ? left_h[D] : 0u, kBufFlags);
    __amdgpu_buffer_rsrc_t ycr = __builtin_amdgcn_make_buffer_rsrc((void*)yc_at[D], 0, enabled ? left_yc[D] : 0u, kBufFlags);
#pragma unroll
    for (int i = 0; i < XCH; ++i) CK::store(fh[i], hr, hoff[i]);
    CK::store(fyc, ycr, ycoff);
    h_at[D] += enabled ? step_h : 0;
    yc_at[D] += enabled ? step_yc : 0;
  };

  // W: this wavefront's macro steps of the workgroup's tiles; slots past its share hold zeros and meet the fragment of slot 0.
  const int ks_count = S > wave ? (S - wave + kWaves - 1) / kWaves : 0;
  i32x4 wreg[MT][KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      wreg[mt][ks] = i32x4{0, 0, 0, 0};
      if (ks < ks_count) wreg[mt][ks] = ((const i32x4*)p.Wp)[((size_t)(r * MT + mt) * S + wave + kWaves * ks) * 64 + lane];
    }

  // The (sequence, cell) pairs of this thread, the same in both groups.
  // (Two pairs per thread are neighbouring cells: half the accesses to LDS and to the ring, two conversions in one.)
  float c_state[2][EPT], h_prev[2][EPT];
  unsigned e_hoff[EPT], e_cl[EPT];
  const unsigned e_row = (unsigned)jl;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int cl = EPT * (kWaves * wave + kg) + j, cell = cell0 + cl;
    e_cl[j] = (unsigned)cl;
    e_hoff[j] = (unsigned)((((cell / KE) * p.Bp + jl) * KE + (cell % KE)) * ES);
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      c_state[d][j] = h_prev[d][j] = 0.f;
      if (jl < rows[d] && cell < nc) {
        const long long bc = ((long long)group[d] * p.Bg + jl) * nc + cell;
        c_state[d][j] = p.c0[bc];
        h_prev[d][j] = E::load(p.y0, bc);
      }
    }
  }

  // That all workgroups of a group share an XCD is checked (both groups of a workgroup have the same workgroups).
  __shared__ int s_local;
  if (!SPREAD && wave == 0) s_local = group_on_one_xcd(p.flags + (size_t)group[0] * G, (unsigned)G, p.status, p.timeout_ticks) ? 1 : 0;

  auto run = [&](auto ex_tag) {
    constexpr int AUXS = decltype(ex_tag)::value == kExDevice ? kAuxDevice : 0, AUXL = kAuxDevice;
    RTN_TRACE_DECL
    constexpr int SETS = SPREAD ? 1 : 2;  // (SPREAD: a group's registers are free when the other group's are asked for)
    i32x4 bf[SETS][KS];
    auto load = [&](auto set_tag, int s, int ks) {
      constexpr int D = decltype(set_tag)::value;
      const unsigned soff = (unsigned)(s & (kHxRing - 1)) * hx_buf_bytes + (ks < ks_count ? ks : 0) * (unsigned)(4 * kWaves * kFragBytes) * p.Bp;
      bf[D % SETS][ks] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ring[D], frag[D], soff, AUXL));
    };
    auto issue = [&](auto set_tag, int s) {  // read the hidden state that enters step s
      asm volatile("" ::: "memory");
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) load(set_tag, s, ks);
      asm volatile("" ::: "memory");
    };
    auto half = [&](int s, auto set_tag) {
      constexpr int D = decltype(set_tag)::value, O = 1 - D;
      unsigned char* const base = smem + L.red + D * L.set;
      auto complete = [&]() {
        unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int w = 0; w < 4; ++w) m[w] = LM::fold(m[w], (unsigned)bf[D % SETS][ks][w]);
        return !__any(LM::has_sentinel(LM::fold(LM::fold(m[0], m[1]), LM::fold(m[2], m[3]))));
      };
      // (The first look stands outside the loop: behind these loads stand the other group's stores, for which a wait that
      // also has to serve the loop's own reads would wait too.)
      if (!complete()) {
        unsigned long long t0 = 0;
        unsigned spins = 0;
        do {
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
          issue(set_tag, s);
        } while (!complete());
      }
      RTN_TRACE_MARK(0)  // wait for h_{s-1}
      // (Vector memory operations of a wavefront end in the order they were issued: with h_{s-1}, asked for behind the stores
      // of this group's step s-1, the re-arming stores of that step have ended too, before anything of step s goes out.)
      Cells x_in[4];
      const unsigned char* xin = base + L.xl + e_row * L.x_row + e_cl[0] * ES;
#pragma unroll
      for (int q = 0; q < 4; ++q) x_in[q] = *(const Cells*)(xin + q * SEG);
      const float m = ((const float*)(base + L.ml))[e_row];
      flush_read(set_tag);
      put(IntTag<O>{});
      if (SPREAD) flush_write(set_tag, s > 0);
      // The other group's hidden state is asked for between the MFMAs of the second half, a load every MT / 2 of them (a CU
      // takes 16 clocks for each of the four wavefronts' loads): it was handed over a quarter of a step before, about the time
      // it takes to be visible on the other CUs.  (n = 1024, B = 256: 669 us for 200 steps; all loads behind the last MFMA 690,
      // behind the barrier 735, behind the gates 797, at the end 852; all in the middle 710, in front of the MFMAs 807.)
      asm volatile("" ::: "memory");
      // (Two chains of additions per wavefront: four tiles at a time, and a four's partial tiles are added and leave for LDS behind the
      // next one's MFMAs.)
      constexpr int CHAINS = two_chains<AT>(KS) ? 2 : 1, GRP = CHAINS == 2 ? 4 : MT;
      f32x4 acc[GRP][CHAINS];
#pragma unroll
      for (int i = 0; i < KS * MT; ++i) {
        const int ks = i / GRP % KS, mt = i / (GRP * KS) * GRP + i % GRP;
        if (!SPREAD && i >= KS * MT / 2 && i % (MT / 2) == 0) {
          __builtin_amdgcn_sched_barrier(0);
          load(IntTag<O>{}, D ? s + 1 : s, i / (MT / 2) - KS);
        }
        if (ks < CHAINS) acc[mt % GRP][ks] = f32x4{0.f, 0.f, 0.f, 0.f};
        acc[mt % GRP][ks % CHAINS] = E::mma(wreg[mt][ks], bf[D % SETS][ks], acc[mt % GRP][ks % CHAINS]);
        __builtin_amdgcn_sched_group_barrier(0x008, sizeof(AT) == 2 ? 1 : 4, 0);
        __builtin_amdgcn_sched_group_barrier(0x096, 3, 0);
        if (CHAINS == 2 && ks == KS - 1) {
          asm("" : "+v"(acc[mt % GRP][0]), "+v"(acc[mt % GRP][CHAINS - 1]));  // (accumulation registers would be copied for the additions)
          red[D][wave][mt][lane] = acc[mt % GRP][0] + acc[mt % GRP][CHAINS - 1];
        }
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      // SPREAD: the hand-over takes longer than the half step between, and a read that comes too early is made again, 64 KB per CU
      // through the memory fabric (n = 2048, B = 64, T = 64, us per step of both: in the second half of the MFMAs 5.4, here 4.3, behind the
      // barrier 4.3, behind the gates 5.0, at the end 5.1; here with a delay of 2 / 4 / 8 units of 64 clocks in front 4.5 / 4.7 / 4.8).
      if (SPREAD) issue(IntTag<O>{}, D ? s + 1 : s);
      // The other group's X for the half step after next: behind the loads of h, which would wait for it otherwise.
      fetch(IntTag<O>{}, D ? s + 2 < nsteps : s + 1 < nsteps);
      if constexpr (CHAINS == 1) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) red[D][wave][mt][lane] = acc[mt][0];
      }
      RTN_TRACE_MARK(1)  // MFMAs, streams, partial tiles to LDS
      __syncthreads();
      RTN_TRACE_MARK(2)  // barrier
      unsigned h_bits[EPT];
      float g_act[EPT][4], y_out[EPT];
#pragma unroll
      for (int j = 0; j < EPT; ++j) {
        f32x4 part[kWaves];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) part[w] = red[D][w][e_cl[j] >> 2][16 * (e_cl[j] & 3) + jl];
        __builtin_amdgcn_sched_barrier(0);
        f32x4 gsum = part[0];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) gsum += part[w];
        const float a0 = Act<AT>::tanh(gsum[0] + (float)x_in[0][j]);
        const float a1 = Act<AT>::sigmoid(gsum[1] + (float)x_in[1][j]);
        const float a2 = Act<AT>::sigmoid(gsum[2] + (float)x_in[2][j]);
        const float a3 = Act<AT>::sigmoid(gsum[3] + (float)x_in[3][j]);
        const float om = 1.f - m, pc = c_state[D][j];
        const float c = (pc * a2 + a0 * a1) * m + pc * om;
        const float y = E::round(Act<AT>::tanh(c) * a3 * m);
        const float hn = (p.op_flags & kOpNoCarry) ? y : E::round(y + h_prev[D][j] * om);
        c_state[D][j] = c;
        h_prev[D][j] = hn;
        h_bits[j] = SN::bits(hn);
        g_act[j][0] = (p.op_flags & kOpH0IsCell) ? c : a0;
        g_act[j][1] = a1; g_act[j][2] = a2; g_act[j][3] = a3;
        y_out[j] = y;
      }
      const unsigned nxt = (unsigned)((s + 1) & (kHxRing - 1)) * hx_buf_bytes, arm = (unsigned)((s + 3) & (kHxRing - 1)) * hx_buf_bytes;
      if constexpr (EPT == 2) {
        __builtin_amdgcn_raw_buffer_store_b32(h_bits[0] | h_bits[EPT - 1] << 16, ring[D], e_hoff[0] + nxt, 0, AUXS);
        __builtin_amdgcn_raw_buffer_store_b32(0xFFFFFFFFu, ring[D], e_hoff[0] + arm, 0, AUXS);
      } else {
        SN::template store<AUXS>(ring[D], e_hoff[0] + nxt, h_bits[0]);
        SN::template store<AUXS>(ring[D], e_hoff[0] + arm, SN::kSentinel);
      }
      RTN_TRACE_MARK(3)  // gates, exchange stores
      // (Staged outputs of the step before leave here, behind everything that the other group's hidden state could wait for.)
      if (!SPREAD) flush_write(set_tag, s > 0);
      unsigned char* hq = base + L.hs + e_row * L.x_row + e_cl[0] * ES;
      Cells v;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int j = 0; j < EPT; ++j) v[j] = (AT)g_act[j][q];
        *(Cells*)(hq + q * SEG) = v;
      }
      struct __attribute__((aligned(4 * EPT))) { float c[EPT]; } cs;
#pragma unroll
      for (int j = 0; j < EPT; ++j) {
        v[j] = (AT)y_out[j];
        cs.c[j] = c_state[D][j];
      }
      *(Cells*)(base + L.ys + e_row * L.y_row + e_cl[0] * ES) = v;
      *(decltype(cs)*)(base + L.cs + e_row * L.c_row + e_cl[0] * 4) = cs;
      RTN_TRACE_MARK(4)  // staging
    };
    fetch(IntTag<0>{}, true);
    fetch(IntTag<1>{}, true);
    put(IntTag<0>{});
    fetch(IntTag<0>{}, nsteps > 1);
    issue(IntTag<0>{}, 0);
    __syncthreads();
    for (int s = 0; s < nsteps; ++s) {
      half(s, IntTag<0>{});
      half(s, IntTag<1>{});
    }
    RTN_TRACE_FLUSH(p, g * G + r)
  };
  __syncthreads();  // s_local
  if constexpr (SPREAD) {
    run(IntTag<kExDevice>{});
  } else if (s_local) {
    run(IntTag<kExLocal>{});
  } else {
    run(IntTag<kExDevice>{});
  }
  __syncthreads();  // the last step's outputs are staged
  // (As in k_lstm2_regw: an expired wait must show in what a consumer reads.)
  const bool expired = wait_expired(p.status);
  if (expired && tid == 0) report_expired(p.status);
  auto finish = [&](auto set_tag) {
    constexpr int D = decltype(set_tag)::value;
    flush_read(set_tag);
    if (expired && moves_y) fyc = CK::fill(kNanWords<AT>);
    flush_write(set_tag, true);
#pragma unroll
    for (int j = 0; j < EPT; ++j)
      if (jl < rows[D] && cell0 + (int)e_cl[j] < nc) {
        const long long bc = ((long long)group[D] * p.Bg + jl) * nc + cell0 + e_cl[j];
        p.d[bc] = expired ? __builtin_nanf("") : c_state[D][j];
        if (p.hN) E::store(p.hN, bc, expired ? __builtin_nanf("") : h_prev[D][j]);
      }
  };
  finish(IntTag<0>{});
  finish(IntTag<1>{});
}

}  // namespace rtn
