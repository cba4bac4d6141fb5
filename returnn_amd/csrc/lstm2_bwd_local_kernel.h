// gfx950 persistent kernel of the NativeLstm2 gradient op for batch groups of up to 8 rows that sit on one XCD each.
#pragma once

#include "lstm2_bwd_kernels.h"
#include "lstm2_sparse_kernel.h"

namespace rtn {

// ---------------------------------------------------------------------------------------------------------------
// The frame of k_lstm2_bwd_regw (decomposition, exchange ring, bounded waits and who re-arms what are described there), for
// groups whose ring of 8 rows per frame stays in one XCD's L2.  A workgroup is 4 wavefronts with W in their registers; one
// load takes two macro steps of the contraction at once (lanes of rows 0-7 step 2a, lanes of rows 8-15 step 2a + 1, 1 KB of
// consecutive memory).  In bfloat16 that is the stored operand of a sparse matrix instruction as it is (see k_lstm2_sparse): rows 8-15 name
// the places of step 2a + 1 among W's interleaved words, and one instruction per tile takes both steps.  The two halves of a row's sum are added across the lanes.
//
// What bounds a frame is the ring: the stores are visible to the XCD after some 500 clocks, then every CU takes in all of the
// group's derivatives (64 KB at n = 1024: 550 clocks to issue the loads and 950 until the last is back, measured with nothing
// else on the way), then 512 clocks of MFMAs per wavefront, the sum over the wavefronts and the gates.  So
//  * the product begins on the first half of the registers and checks the second behind the first one's MFMAs;
//  * the MFMAs of a register go to accumulators of their own with a fence behind (left alone, the scheduler lines up those of
//    one accumulator, each waiting for the one before);
//  * nothing that does not need the errors is left to the time between the product and the stores: the gates' factors are
//    worked out while the stores travel;
//  * derivatives go from the lanes that have them to the ring, 8 or 16 bytes each (see Quad), without LDS and a barrier;
//  * inputs are asked for behind most of the MFMAs, when the other wavefronts' ring loads are through, and for four frames at once (kBwdBatch).
// Nothing in the loop may be reached with loads in flight that the frame's own path does not have there: the compiler then waits
// for all of them, and a fetch from memory that was just asked for stood between the sum and the stores (0.15 us of a frame).
//
// Measured (gradient op, us per frame with the weight gradient, k_lstm2_bwd_regw / this): bf16 n = 1024, both directions of 32 rows
// 2.74 / 2.50, one direction 2.60 / 2.31; n = 768 2.51 / 2.23; n = 512, 32 rows 1.90 / 1.64; n = 128, both of 8 rows 1.74 / 1.38; n = 64,
// 4 rows 1.42 / 1.03; float32 n = 500, both of 40 rows 5.26 / 4.89; n = 256, 100 rows 3.69 / 3.09; n = 64, both of 32 rows 1.56 / 1.25.
// With the sparse product and inputs in turns (whole backward pass of a layer over 500 frames, us before / now): bf16 n = 1024, both directions of 32 rows
// 1580 / 1525, n = 768, 32 rows 1272 / 1168, n = 512, both of 32 rows 1124 / 1025, n = 256, both of 16 rows 767 / 690, n = 128, 8 rows 608 / 554; float32
// n = 256, 30 rows 869 / 859, n = 64, 8 rows 546 / 525.
// ---------------------------------------------------------------------------------------------------------------

// Four elements (8 or 16 bytes) per lane, and the transposition of 4 x 4 of them over the lanes of a quad: with it lane i, which
// owns cell i of four, moves gate i of all four in one piece -- the derivatives on their way to the ring and to DX, the gates
// of a frame on their way in.  (The derivatives went through LDS, with a barrier, to the threads that stored 16-byte pieces: 400 of the
// 1200 clocks between the sum and the stores; the gates were a load each: 8 loads per frame and pair instead of 4 cost 0.3 of 2.5 us.)
template <typename AT>
struct Quad;
template <>
struct Quad<float> {
  typedef u32x4 T;
  static __device__ __forceinline__ unsigned selector(int) { return 0; }
  static __device__ __forceinline__ T transpose(T v, int lane, unsigned) { return __builtin_bit_cast(T, quad_transpose(__builtin_bit_cast(f32x4, v), lane)); }
  static __device__ __forceinline__ T pack(const unsigned (&g)[4]) { return T{g[0], g[1], g[2], g[3]}; }
  static __device__ __forceinline__ float get(T v, int k) { return __builtin_bit_cast(float, (unsigned)v[k]); }
  static __device__ __forceinline__ T load(__amdgpu_buffer_rsrc_t rs, unsigned off) { return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0)); }
  template <int AUX>
  static __device__ __forceinline__ void store(T v, __amdgpu_buffer_rsrc_t rs, unsigned off, unsigned soff = 0) { __builtin_amdgcn_raw_buffer_store_b128(v, rs, off, soff, AUX); }
  static __device__ __forceinline__ T ones() { return T{~0u, ~0u, ~0u, ~0u}; }
};
template <>
struct Quad<__bf16> {
  typedef u32x2 T;
  // (bytes of v_perm_b32) even lanes: the low halves, their own first; odd lanes: the high halves, their own second
  static __device__ __forceinline__ unsigned selector(int lane) { return lane & 1 ? 0x03020706u : 0x05040100u; }
  template <int PERM>
  static __device__ __forceinline__ unsigned from_lane(unsigned v) { return (unsigned)__builtin_amdgcn_mov_dpp((int)v, PERM, 0xF, 0xF, true); }
  static __device__ __forceinline__ T transpose(T v, int lane, unsigned sel) {
    const bool upper = (lane & 2) != 0;
    const unsigned keep = upper ? v[1] : v[0], got = from_lane<0x4E>(upper ? v[0] : v[1]);  // with the lane 2 away
    const unsigned lo = upper ? got : keep, hi = upper ? keep : got;                        // of lanes lane % 2 and lane % 2 + 2
    return T{__builtin_amdgcn_perm(from_lane<0xB1>(lo), lo, sel), __builtin_amdgcn_perm(from_lane<0xB1>(hi), hi, sel)};
  }
  static __device__ __forceinline__ T pack(const unsigned (&g)[4]) { return T{g[0] | (g[1] << 16), g[2] | (g[3] << 16)}; }
  static __device__ __forceinline__ float get(T v, int k) { return __builtin_bit_cast(float, k & 1 ? v[k >> 1] & 0xFFFF0000u : v[k >> 1] << 16); }
  static __device__ __forceinline__ T load(__amdgpu_buffer_rsrc_t rs, unsigned off) { return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0)); }
  template <int AUX>
  static __device__ __forceinline__ void store(T v, __amdgpu_buffer_rsrc_t rs, unsigned off, unsigned soff = 0) { __builtin_amdgcn_raw_buffer_store_b64(v, rs, off, soff, AUX); }
  static __device__ __forceinline__ T ones() { return T{~0u, ~0u}; }
};

// Frames whose inputs are asked for at once, but where a wavefront's share of W is 64 fragments (or 32 in float32), whose ring loads and products take
// so long that the burst is felt more than a frame's loads are: us per frame one at a time / four: bf16 n = 512, both directions of 32 rows 1.75 / 1.45,
// n = 1024 2.52 / 2.63, float32 n = 500, both of 40 rows 5.21 / 5.25, n = 256, 30 rows 1.36 / 1.33.  (A load from memory holds up the ring loads
// behind it in the CU's first-level cache: see k_lstm2_sparse.)
constexpr int kBwdBatch = 4;

// RQ > 0 (float32, groups of at most 4 RQ rows): the product in v_mfma_f32_4x4x1, whose 16 blocks of 4 rows x 4 values of k are
// 4 rows x 64 products in 8 clocks, the rate of the 16x16x4 without its padding of 8 rows to 16.  With MT tiles of 16 values
// of k, 4 MT blocks take one element of the contraction range and 4 / MT of them go at once: lane group kg of a fragment
// holds elements 4 kg ... 4 kg + 3, and of every 4 MT blocks the one that holds the wanted rows of register i's element is
// broadcast to the others.  The 4 / MT partial sums are added across the lanes before they go through LDS.
template <int MT, int ABID>
__device__ __forceinline__ f32x4 bwd_quad_mma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, MT == 4 ? 4 : MT == 2 ? 3 : 2, ABID, 0); }
// Two macro steps whose fragments share a register (rows 0-7 and 8-15 of every lane group); I counts (e, i, macro step, quad).
template <int MT, int RQ, int... I>
__device__ __forceinline__ void bwd_quad_steps(const i32x4 (&w0)[MT], const i32x4 (&w1)[MT], const i32x4& xbits, f32x4 (&acc)[RQ][2], std::integer_sequence<int, I...>) {
  const f32x4 x = __builtin_bit_cast(f32x4, xbits);
  f32x4 w[2][MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    w[0][i] = __builtin_bit_cast(f32x4, w0[i]);
    w[1][i] = __builtin_bit_cast(f32x4, w1[i]);
  }
  (([&] {
     constexpr int rq = I % RQ, up = I / RQ % 2, i = I / (2 * RQ) % MT, e = I / (2 * RQ * MT);
     acc[rq][up] = bwd_quad_mma<MT, 4 * i + rq + 2 * up>(x[e], w[up][i][e], acc[rq][up]);
   }()),
   ...);
}
// a + b of the lanes 32 (SHIFT = 32) or 16 apart: lanes without the bit get a's sum, lanes with it b's.
template <int SHIFT>
__device__ __forceinline__ f32x4 lane_pair_sum(f32x4 a, f32x4 b) {
  f32x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const unsigned x = __builtin_bit_cast(unsigned, (float)a[j]), y = __builtin_bit_cast(unsigned, (float)b[j]);
    const u32x2 t = SHIFT == 32 ? __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(x, y, false, false))
                                : __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(x, y, false, false));
    const unsigned lo = t[0], hi = t[1];
    r[j] = __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
  }
  return r;
}

template <typename AT, int KSB, int MT, int RQ = 0>
__global__ __launch_bounds__(kWgThreads) void k_lstm2_bwd_local(const Lstm2BwdMulti multi) {
  constexpr bool QUAD = RQ > 0;
  static_assert(KSB % 2 == 0 && QUAD == (sizeof(AT) == 4) && RQ <= 2, "paired loads; float32 in quads of rows, bfloat16 in sparse matrix instructions");
  // tiles whose pairs a thread keeps: with at most 8 rows the threads of the upper 8 row slots take every other tile (SPLIT)
  constexpr bool SPLIT = MT % 2 == 0;
  constexpr int PT = SPLIT ? MT / 2 : MT;
  const int kb = multi.q[0].p.n / (16 * MT), groups_now = multi.q[0].groups;
  const int xcd = (int)blockIdx.x % multi.xcds, slot = (int)blockIdx.x / multi.xcds;
  const int gg = (slot / kb) * multi.xcds + xcd;  // group of the launch, all problems counted through
  const int which = gg / groups_now;
  const int bid = (gg - which * groups_now) * kb + slot % kb;
  if (which >= multi.count) return;
  const Lstm2BwdPersistent q = multi.q[which];
  using E = Elem<AT>;
  using SN = Sentinel<AT>;
  using LM = LaneMax<AT>;
  constexpr int KE = E::KE, KM = E::KM, ES = (int)sizeof(AT);
  const Lstm2BwdParams& p = q.p;
  // partial tiles of the wavefronts, in two copies: no barrier between the sums of one frame and the partial tiles of the next
  // (QUAD: [quad][k] of 4 rows each, two quads of up to 32 values of k in one 64 lanes wide slot)
  // (else: [tile][quad of rows][k] of 4 rows each, two tiles in one slot, see gemm)
  constexpr int kRedSlots = QUAD ? (MT == 4 ? RQ : 1) : (MT + 1) / 2;
  __shared__ f32x4 red2[2][kWaves][kRedSlots][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = p.n, n4 = 4 * n;
  const int kblocks = n / (16 * MT);  // workgroups per group; each owns MT tiles of 16 values of k
  const int g = q.group_offset + bid / kblocks, k0 = (bid % kblocks) * 16 * MT;
  const int b_base = g * q.Bg;
  const int rows = min(q.Bg, p.B - b_base);
  const int nc = p.nc;
  const long long bn = (long long)p.B * nc;
  const unsigned frame_bytes = (unsigned)((size_t)p.B * 4 * nc * ES);
  const unsigned dx_frame_bytes = (unsigned)((size_t)p.B * p.ldDX * ES), dy_frame_bytes = (unsigned)((size_t)p.B * p.ldDY * ES);
  // the exchange ring of this group: kExRing frames of [4n/KM][4][8][16 bytes]
  const unsigned ex_frame = (unsigned)((size_t)n4 * 8 * ES);
  __amdgpu_buffer_rsrc_t ring = __builtin_amdgcn_make_buffer_rsrc((unsigned char*)q.ex + (size_t)g * kExRing * ex_frame, 0, kExRing * ex_frame, kBufFlags);

  // An XCD-local plan rests on all workgroups of a group being on one XCD: checked here.
  __shared__ int s_local;
  if (wave == 0) s_local = (int)group_on_one_xcd(q.sync + 2 * (size_t)g, (unsigned)kblocks, q.status, q.timeout_ticks);
  __syncthreads();
  const bool local = s_local != 0;

  // A fragments: this wavefront's macro steps [wave*ksb, (wave+1)*ksb) of the 16*MT rows of W, as far as the 4n/KM macro
  // steps reach.  Slots beyond them hold zeros in W and read nothing, so that any width whose share per wavefront is at most
  // KSB runs on this kernel.
  const int ksb = q.ksb;
  const int ks_here = max(0, min(ksb, n4 / KM - ksb * wave));  // uniform over the wavefront
  // (bfloat16: a register pair of macro steps 2a and 2a + 1 is interleaved word by word, see k_lstm2_sparse; lane group g holds elements
  // 8 (g / 2) + 4 (g % 2) ... + 3 and those 16 further of either.)
  i32x4 wreg[QUAD ? MT : 1][KSB];
  i32x8 wsp[QUAD ? 1 : MT][KSB / 2];
  if constexpr (!QUAD) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const AT* Wr = (const AT*)p.W + (size_t)(k0 + 16 * mt + (lane & 15)) * n4 + (size_t)KM * ksb * wave + 4 * (lane >> 4);
#pragma unroll
      for (int a = 0; a < KSB / 2; ++a) {
        i32x2 v[2][2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int h = 0; h < 2; ++h) v[u][h] = 2 * a + u < ks_here ? *(const i32x2*)(Wr + KM * (2 * a + u) + 16 * h) : i32x2{0, 0};
        wsp[mt][a] = i32x8{v[0][0][0], v[1][0][0], v[0][0][1], v[1][0][1], v[0][1][0], v[1][1][0], v[0][1][1], v[1][1][1]};
      }
    }
  } else {
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    // (QUAD: register i of a lane is k = lane % (16 MT), elements 4 (i + MT * (lane / (16 MT))) ... + 3 of the macro step)
    const AT* Wr = (const AT*)p.W + (size_t)(k0 + (QUAD ? lane & (16 * MT - 1) : 16 * mt + (lane & 15))) * n4 + (size_t)KM * ksb * wave +
                   KE * (QUAD ? mt + MT * (lane / (16 * MT)) : lane >> 4);
#pragma unroll
    for (int ks = 0; ks < KSB; ++ks) wreg[mt][ks] = (ks < ks_here) ? *(const i32x4*)(Wr + (size_t)KM * ks) : i32x4{0, 0, 0, 0};
  }
  }
  // Byte offsets of this lane's B fragments inside a ring frame.  The lanes of rows the group lacks and slots without a share
  // carry an out-of-range one: 0 comes back and no memory is touched.  (The offsets stay in registers over the frames, which measured faster than
  // instruction immediates.)
  const int places = (lane & 8) ? (int)0xEEEEEEEE : 0x44444444;  // rows 8-15 hold the odd macro step's values: places 2 and 3 of every four
  constexpr int NB = KSB / 2;                   // registers of B fragments
  constexpr int PARTS = NB >= 8 ? 2 : 1, N1 = NB / PARTS;  // ... checked and multiplied in parts (four of them: no faster)
  i32x4 bf[NB];
  unsigned foff[NB];
#pragma unroll
  for (int a = 0; a < NB; ++a)
    foff[a] = (lane & 7) < rows && 2 * a + ((lane >> 3) & 1) < ks_here ? (unsigned)((ksb * wave + 2 * a + ((lane >> 3) & 1)) * 512 + ((lane >> 4) * 8 + (lane & 7)) * 16) : 0x80000000u;

  // The (row, k) pairs of this thread: one in each of its tiles.
  const int kl = tid & 15;
  const int bl = SPLIT ? (tid & 127) >> 4 : tid >> 4;  // row slot
  const int upper = SPLIT ? tid >> 7 : 0;              // SPLIT: which of a pair of tiles
  auto tile_of = [&](int j) { return SPLIT ? 2 * j + upper : j; };
  const int b = b_base + ((bl < rows) ? bl : 0);
  bool act[PT];  // the pair exists: the group has the row and the caller the cell
  long long idx[PT], io[PT];
  unsigned off_gates[PT], off_h0[PT], off_dy[PT], off_c[PT];  // byte offsets inside a frame of H (gate lane % 4 of the quad's cells; the pair's own first block), DY and C; out of range (0 comes back) for cells beyond nc
  unsigned ring_at[PT], dx_at[PT];  // where the four cells of gate lane % 4 go, inside a frame of the ring and of DX (out of range: nowhere)
  float dyw[PT], dc[PT], dx0[PT][4];
  // (no branch around the load: behind one that some lanes skip, a full register file has cost those lanes values)
  __amdgpu_buffer_rsrc_t rs_dd = __builtin_amdgcn_make_buffer_rsrc((void*)q.Dd, 0, q.Dd ? (unsigned)(bn * 4) : 0u, kBufFlags);
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    const int mt = tile_of(j);
    const int k = k0 + 16 * mt + kl;
    act[j] = bl < rows && k < nc;
    idx[j] = (long long)b * nc + k;
    io[j] = (long long)b * 4 * nc + k;
    off_dy[j] = k < nc ? (unsigned)(((long long)b * p.ldDY + k) * ES) : kOobOffset;
    off_c[j] = k < nc ? (unsigned)(idx[j] * 4) : kOobOffset;
    const int gate = kl & 3, first = k & ~3;  // (nc is a multiple of 4)
    off_h0[j] = k < nc ? (unsigned)(io[j] * ES) : kOobOffset;
    off_gates[j] = first < nc ? (unsigned)(((long long)b * 4 * nc + (long long)gate * nc + first) * ES) : kOobOffset;
    ring_at[j] = bl < rows ? (unsigned)((((gate * n + first) / KE * 8 + bl) * KE + first % KE) * ES) : kOobOffset;
    dx_at[j] = bl < rows && first < nc ? (unsigned)(((long long)b * p.ldDX + (long long)gate * nc + first) * ES) : kOobOffset;
    dyw[j] = 0.f;
    dc[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_dd, act[j] ? off_c[j] : kOobOffset, 0, 0));
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) dx0[j][gq] = 0.f;
  }
  // where a pair's element of the summed tile is
  const int red_lane = QUAD ? (RQ == 2 ? (bl >> 2) & 1 : 0) * (MT == 4 ? 64 : 32) + kl : 16 * ((bl >> 2) & 1) + kl;  // (+ 32 for an odd tile)
  const int red_comp = bl & 3;

  // Inputs of a frame: asked for behind the MFMAs of the product two frames before it, turned into the factors of the pointwise
  // part a frame before it.  (A wavefront's loads count as returned in the order they were issued: asked for in front of the
  // ring's loads, they made the wait for the ring a wait for memory.)  No branches around the loads and no arithmetic on what
  // they bring until then: a register that gets its value on two paths, or feeds an instruction, makes the compiler wait for
  // every load in flight there.  Frames that do not exist are buffers of no bytes.
  // (as the loads bring them: an element widened any earlier would be waited for among the MFMAs)
  typedef Quad<AT> QD;
  const unsigned quad_sel = QD::selector(lane);
  typedef std::conditional_t<ES == 2, unsigned short, unsigned> Raw;
  constexpr int FB = MT * KSB >= 64 || (QUAD && KSB >= 32) ? 1 : kBwdBatch;
  typename QD::T nx_gates[FB][PT];
  Raw nx_dy[FB][PT];
  unsigned nx_pc[FB][PT], nx_m[FB];
  BwdCell<AT> cell[PT];
  float in_dy[PT], in_m;
  auto widen = [](Raw raw) {
    if constexpr (ES == 2)
      return __builtin_bit_cast(float, (unsigned)raw << 16);
    else
      return __builtin_bit_cast(float, raw);
  };
  auto load = [](__amdgpu_buffer_rsrc_t rs, unsigned off, int soff) -> Raw {
    if constexpr (ES == 2)
      return __builtin_amdgcn_raw_buffer_load_b16(rs, off, soff, 0);
    else
      return __builtin_amdgcn_raw_buffer_load_b32(rs, off, soff, 0);
  };
  const unsigned m_off = (unsigned)(b * 4);
  const bool h0_cell = (p.op_flags & kOpH0IsCell) != 0;
  // The frame that is fetched next: its ordinal, and where it lies in H, DY, C (the frame before it) and the mask.
  int nf = 0;
  bool cell_from_h[FB];  // what nx_pc holds
  const long long stride_h = -(long long)q.step * frame_bytes, stride_dy = -(long long)q.step * dy_frame_bytes, stride_c = -(long long)q.step * bn * 4,
                  stride_m = -(long long)q.step * p.B * 4;
  const unsigned char *at_h = (const unsigned char*)p.H + q.t_end * (long long)frame_bytes, *at_dy = (const unsigned char*)p.DY + q.t_end * (long long)dy_frame_bytes,
                      *at_c = (const unsigned char*)p.C + (q.t_end - q.step) * bn * 4, *at_m = (const unsigned char*)(p.mask + q.t_end * p.B);
  auto fetch_gates = [&](int slot) {
    __amdgpu_buffer_rsrc_t rs_h = __builtin_amdgcn_make_buffer_rsrc((void*)at_h, 0, nf < q.nframes ? frame_bytes : 0u, kBufFlags);
#pragma unroll
    for (int j = 0; j < PT; ++j) nx_gates[slot][j] = QD::load(rs_h, off_gates[j]);
    at_h += stride_h;
  };
  auto fetch_errors = [&](int slot) {
    const bool there = nf < q.nframes;
    __amdgpu_buffer_rsrc_t rs_dy = __builtin_amdgcn_make_buffer_rsrc((void*)at_dy, 0, there ? dy_frame_bytes : 0u, kBufFlags);
    __amdgpu_buffer_rsrc_t rs_m = __builtin_amdgcn_make_buffer_rsrc((void*)at_m, 0, there ? (unsigned)(p.B * 4) : 0u, kBufFlags);
#pragma unroll
    for (int j = 0; j < PT; ++j) nx_dy[slot][j] = load(rs_dy, off_dy[j], 0);
    nx_m[slot] = __builtin_amdgcn_raw_buffer_load_b32(rs_m, m_off, 0, 0);
    at_dy += stride_dy;
    at_m += stride_m;
  };
  // The cell state of the frame before: C, c0 in front of the first frame, or (kOpH0IsCell) the word of H that holds the pair's
  // element of its first block.  (Behind fetch_gates: at_h is the frame before the one fetched.)
  auto fetch_cell = [&](int slot) {
    const bool first = q.nframes - nf == 1;
    const bool from_h = cell_from_h[slot] = h0_cell && !first;
    const unsigned char* src = first ? (const unsigned char*)p.c0 : from_h ? at_h : at_c;
    __amdgpu_buffer_rsrc_t rs_c = __builtin_amdgcn_make_buffer_rsrc((void*)src, 0, nf >= q.nframes ? 0u : from_h ? frame_bytes : (unsigned)(bn * 4), kBufFlags);
#pragma unroll
    for (int j = 0; j < PT; ++j) nx_pc[slot][j] = __builtin_amdgcn_raw_buffer_load_b32(rs_c, from_h ? off_h0[j] & ~3u : off_c[j], 0, 0);
    at_c += stride_c;
    ++nf;
  };
  auto fetch = [&](int slot) {
    fetch_gates(slot);
    fetch_errors(slot);
    fetch_cell(slot);
  };
  auto take_next = [&](int slot) {  // what was asked for becomes the current frame's inputs
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const typename QD::T g = QD::transpose(nx_gates[slot][j], lane, quad_sel);
      float before = __builtin_bit_cast(float, nx_pc[slot][j]);
      if constexpr (ES == 2)
        if (cell_from_h[slot]) before = __builtin_bit_cast(float, off_h0[j] & 2 ? nx_pc[slot][j] & 0xFFFF0000u : nx_pc[slot][j] << 16);
      cell[j] = BwdCell<AT>::of(p.op_flags, QD::get(g, 0), QD::get(g, 1), QD::get(g, 2), QD::get(g, 3), before);
      in_dy[j] = widen(nx_dy[slot][j]);
      asm volatile("" : "+v"(in_dy[j]));
    }
    in_m = __builtin_bit_cast(float, nx_m[slot]);
    // (of registers of their own from here on: used as the loads left them, they would be waited for behind the next fetch)
    asm volatile("" : "+v"(in_m));
  };
  const int F = q.nframes;
  unsigned char* at_dx = (unsigned char*)p.DX + q.t_end * (long long)dx_frame_bytes;
  const long long stride_dx = -(long long)q.step * dx_frame_bytes;

  auto issue = [&](int f, int from = 0) {  // the loads of frame ordinal f's derivatives, register `from` and up
    const unsigned slot = (unsigned)(f & (kExRing - 1)) * ex_frame;
    asm volatile("" ::: "memory");  // other workgroups write this memory: really load again
#pragma unroll
    for (int a = 0; a < NB; ++a)
      if (a >= from) bf[a] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(ring, foff[a], slot, kAuxDevice));
  };
  // One fixed delay for all wavefronts in front of the first read.  (A group that was planned for one XCD and found itself on
  // several takes the adaptive delay of a spread plan.)
  int delay = local ? q.poll_delay : 20;
  const int delay_inc = local ? q.delay_inc : 2;
  bool aborted = false;
  // d_h of the thread's pairs from DX of frame t (whose first read has been issued): wait, MFMA, sum over the
  // wavefronts; added to dyw.
  RTN_BTRACE_DECL
  // (four independent running maxima: one chain of dependent packed operations needs a wait state after every one of them,
  // and there are up to 128 of them here)
  auto fold = [&](unsigned (&m)[4], const i32x4& v) {
#pragma unroll
    for (int w = 0; w < 4; ++w) m[w] = LM::fold(m[w], (unsigned)v[w]);
  };
  auto seen_mark = [&](const unsigned (&m)[4]) { return __any(LM::has_sentinel(LM::fold(LM::fold(m[0], m[1]), LM::fold(m[2], m[3])))) != 0; };
  auto marked = [&](int from) {  // among the registers of the part that begins at `from`
    unsigned m[4] = {0, 0, 0, 0};
#pragma unroll
    for (int a = 0; a < NB; ++a)
      if (a >= from && a < from + N1) fold(m, bf[a]);
    return seen_mark(m);
  };
  // Reads registers `from` and up again until the part that begins there is complete; returns the number of repeats.  (Behind a
  // first look outside: the loads of the other part may still be on their way there.)
  auto read_again = [&](int t, int from) {
    unsigned long long t0 = 0;
    unsigned spins = 0;
    do {
      if ((spins++ & 15u) == 0) {
        if (__hip_atomic_load(q.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) { aborted = true; break; }
        const unsigned long long now = wall_clock64();
        if (spins == 1) {
          t0 = now;
        } else if (now - t0 > q.timeout_ticks) {
          __hip_atomic_store(q.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          aborted = true;
          break;
        }
      }
      issue(t, from);
    } while (marked(from));
    return spins;
  };
  auto gemm = [&](int t, auto ph_tag) {  // t: ordinal of the frame whose derivatives go through the product
    constexpr int PH = decltype(ph_tag)::value;  // (t + 1) % FB
    RTN_BTRACE_MARK(4)  // pointwise tail, delay, first read, factors of the next frame
    auto& red = red2[t & 1];
    // (at least four accumulators keep the MFMA pipeline full)
    constexpr int NACC = MT >= 4 ? 1 : 4 / MT;
    f32x4 part[MT][NACC];
    if constexpr (!QUAD) {  // (cleared here, where nothing else is to do)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int a = 0; a < NACC; ++a) {
          part[mt][a] = f32x4{0.f, 0.f, 0.f, 0.f};
          asm volatile("" : "+v"(part[mt][a]));
        }
    }
    f32x4 quad[QUAD ? RQ : 1][2];
    unsigned spins = 0;
    if (marked(0)) spins = read_again(t, 0);
    RTN_BTRACE_MARK(0)  // wait for the frame's DX
    RTN_BTRACE_ADD(6, spins)
    if (spins)
      delay = min(delay + delay_inc, 64);
    else if (delay_inc && delay > 0)
      delay -= ((t & q.delay_dec_mask) == q.delay_dec_mask) ? 1 : 0;
    // W lives in accumulation registers where it is at most half of that file: the B fragments fill up to half of
    // the ordinary registers, and a matrix instruction reads an A operand from either file (without this the compiler
    // parks part of W there anyway and copies four registers back in front of every MFMA, which halves the MFMA rate).
    if constexpr (QUAD && MT * KSB <= 32) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int ks = 0; ks < KSB; ++ks) asm volatile("" : "+a"(wreg[mt][ks]));
    }
#pragma unroll
    for (int q = 0; q < (QUAD ? RQ : 1); ++q) quad[q][0] = quad[q][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Register by register, with a fence behind and a piece of the other work -- the check of the next part, the fetch of the
    // next inputs -- between its MFMAs.
    unsigned m2[4] = {0, 0, 0, 0};
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      if (a > 0 && a % N1 == 0) {
        if (seen_mark(m2)) (void)read_again(t, a);
#pragma unroll
        for (int w = 0; w < 4; ++w) m2[w] = 0;
      }
      if (PH == 1 % FB) {
        if (a == (NB >= 3 ? NB - 3 : 0)) {
#pragma unroll
          for (int i = 1; i <= FB / 2; ++i) fetch((PH + i) % FB);
        }
        if (FB > 1 && a == NB - 1) {
#pragma unroll
          for (int i = FB / 2 + 1; i <= FB; ++i) fetch((PH + i) % FB);
        }
        if (FB == 1) {
          if (a == (NB >= 3 ? NB - 3 : 0)) fetch_gates(0);
          if (a == (NB >= 3 ? NB - 2 : NB - 1)) fetch_errors(0);
          if (a == NB - 1) fetch_cell(0);
        }
      }
      if (a + N1 < NB) fold(m2, bf[a + N1]);
      if constexpr (QUAD) {
        i32x4 w0[MT], w1[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          w0[mt] = wreg[mt][2 * a];
          w1[mt] = wreg[mt][2 * a + 1];
        }
        bwd_quad_steps<MT, RQ>(w0, w1, bf[a], quad, std::make_integer_sequence<int, 8 * MT * RQ>());
#pragma unroll
        for (int i = 0; i < 8 * MT * RQ; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // an MFMA of 8 clocks takes two issue turns of 4 ...
          __builtin_amdgcn_sched_group_barrier(0x096, 1, 0);  // ... one of which anything else may have
        }
      } else {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          part[mt][a % NACC] = smfmac(bf[a], wsp[mt][a], part[mt][a % NACC], places);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x096, 3, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (QUAD) {
      f32x4 sum[RQ];
#pragma unroll
      for (int q = 0; q < RQ; ++q) sum[q] = quad[q][0] + quad[q][1];
      if constexpr (MT == 4) {
#pragma unroll
        for (int q = 0; q < RQ; ++q) red[wave][q][lane] = sum[q];
      } else {
        f32x4 acc = lane_pair_sum<32>(sum[0], sum[RQ - 1]);
        if constexpr (MT == 1) acc = lane_pair_sum<16>(acc, acc);
        red[wave][0][lane] = acc;
      }
    } else {
      // Rows 0-7 of a result are the sums over the even macro steps, 8-15 those over the odd ones, 32 lanes away: added, an even tile's sums
      // end up in the lower lanes and the odd tile's beside it in the upper ones, one slot for both.
#pragma unroll
      for (int slot = 0; slot < kRedSlots; ++slot) {
        f32x4 tile[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int mt = 2 * slot + k < MT ? 2 * slot + k : 2 * slot;
          tile[k] = part[mt][0];
#pragma unroll
          for (int a = 1; a < NACC; ++a) tile[k] += part[mt][a];
        }
        red[wave][slot][lane] = lane_pair_sum<32>(tile[0], tile[1]);
      }
    }
    RTN_BTRACE_MARK(1)  // MFMA, partial tiles to LDS
    __syncthreads();
    RTN_BTRACE_MARK(2)  // barrier
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const int mt = tile_of(j);
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        if constexpr (QUAD)
          sum += ((const float*)(&red[w][0][0] + red_lane + 16 * mt))[red_comp];
        else
          sum += ((const float*)&red[w][mt >> 1][red_lane + 32 * (mt & 1)])[red_comp];
      }
      dyw[j] += sum;
    }
    // (this copy of `red` is written again two frames from now, behind the next frame's barrier above)
    RTN_BTRACE_MARK(3)  // sum over the wavefronts
  };

  const bool raw_dh = (p.op_flags & kOpRawDh) != 0;
  // Where a frame's derivatives go.
  unsigned to = 0, arm = 0;
  unsigned char* dx_to = nullptr;
  auto aim = [&](int f) {
    to = (unsigned)(f & (kExRing - 1)) * ex_frame;
    arm = (unsigned)((f + 2) & (kExRing - 1)) * ex_frame;
    dx_to = at_dx;
    at_dx += stride_dx;
    asm volatile("" : "+s"(to), "+s"(arm), "+s"(dx_to));  // scalar arithmetic ahead of the wait, not behind it
  };
  auto pointwise = [&](int f, int next) {
    __amdgpu_buffer_rsrc_t rs_dx = __builtin_amdgcn_make_buffer_rsrc(dx_to, 0, dx_frame_bytes, kBufFlags);
    // pointwise part of frame t (returnn/native_op.py:1123-1180); the derivatives out as soon as they are there, then all-ones
    // into the slot that was read two frames ago, DX, and what the errors carry on
    const float m = in_m;
    float dx[PT][4], err_cell[PT];
    typename QD::T out[PT];
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const float err_y = raw_dh ? in_dy[j] * m + dyw[j] : (in_dy[j] + dyw[j]) * m;
      err_cell[j] = cell[j].apply(err_y, dc[j] * m, dx[j]);
      const unsigned bits[4] = {SN::bits(dx[j][0]), SN::bits(dx[j][1]), SN::bits(dx[j][2]), SN::bits(dx[j][3])};
      out[j] = QD::transpose(QD::pack(bits), lane, quad_sel);
    }
    if (local) {
#pragma unroll
      for (int j = 0; j < PT; ++j) QD::template store<0>(out[j], ring, ring_at[j], to);
#pragma unroll
      for (int j = 0; j < PT; ++j) QD::template store<0>(QD::ones(), ring, ring_at[j], arm);
    } else {
#pragma unroll
      for (int j = 0; j < PT; ++j) QD::template store<kAuxDevice>(out[j], ring, ring_at[j], to);
#pragma unroll
      for (int j = 0; j < PT; ++j) QD::template store<kAuxDevice>(QD::ones(), ring, ring_at[j], arm);
    }
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      QD::template store<0>(out[j], rs_dx, dx_at[j]);
      dc[j] = cell[j].a_fg * err_cell[j] + dc[j] * (1.f - m);
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) dx0[j][gq] = raw_dh ? dx[j][gq] : dx[j][gq] + dx0[j][gq] * (1.f - m);
      dyw[j] = (p.op_flags & kOpNoCarry) ? 0.f : dyw[j] * (1.f - m);
    }
    RTN_BTRACE_MARK(5)  // pointwise part, stores
    // while the derivatives travel: what the next frame's pointwise part can do without the errors, and after the delay the
    // first read of this frame's ring slot
    take_next(next);
    if (!aborted)
      for (int d = 0; d < delay; ++d) __builtin_amdgcn_s_sleep(1);
    issue(f);
  };
  fetch(0);
  take_next(0);
  fetch(1 % FB);
  aim(0);
  // (The first frame in front of the loop: a way into its pointwise part without a product in front, on which loads are still
  // in flight, made every frame wait for the inputs it had just asked for.)
  if (F > 0) pointwise(0, 1 % FB);
  for (int f = 1; f <= F; f += FB) {
    auto frame = [&](int f, auto ph_tag) {
      aim(f);
      gemm(f - 1, ph_tag);
      if (f < F) pointwise(f, (decltype(ph_tag)::value + 1) % FB);
    };
    frame(f, IntTag<1 % FB>{});
    if constexpr (FB > 1) {
      if (f + 1 > F) break;
      frame(f + 1, IntTag<2 % FB>{});
    }
    if constexpr (FB > 2) {
      if (f + 2 > F) break;
      frame(f + 2, IntTag<3>{});
      if (f + 3 > F) break;
      frame(f + 3, IntTag<0>{});
    }
  }
  RTN_BTRACE_ADD(7, (unsigned long long)delay)
  RTN_BTRACE_FLUSH()
  // After a wait that ran into its bound the gradients are wrong without looking it: the workgroups that see the mark
  // hand out NaN, so that a caller who never asks for the status still finds a non-finite gradient.
  const bool expired = wait_expired(q.status);
  if (expired && tid == 0) report_expired(q.status);
  const float nan = __builtin_nanf("");
#pragma unroll
  for (int j = 0; j < PT; ++j) {
    if (act[j]) {
      E::store(q.Dy0, idx[j], expired ? nan : dyw[j]);
      p.Dc0[idx[j]] = expired ? nan : dc[j];
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) E::store(p.dx0, io[j] + (long long)gq * nc, expired ? nan : dx0[j][gq]);
    }
  }
}

}  // namespace rtn
