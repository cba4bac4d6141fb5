// The instantiations of the persistent kernels, in parts: this file is compiled once per value of RTN_TABLE_PART
// (see build.py), each compilation defines the table functions of one part (lstm2_kernel_tables.h).
#include <hip/hip_runtime.h>

#include "lstm2_kernel_tables.h"

#ifndef RTN_TABLE_PART
#error "compile with -DRTN_TABLE_PART=<1..17>"
#endif

namespace rtn {
namespace {

// Forward.  HI: the builds with 8 or 16 macro steps of the contraction per wavefront, else those with 2 or 4.  (bfloat16 with 16: regw_table_16.)
template <typename AT, bool HI, bool TAIL>
RegwKernel regw_table(int MT, int NT, int KSMAX, bool half) {
  if (half) {
#define RTN_CASE(mt, ks) \
  if (MT == mt && NT == 1 && KSMAX == ks) return &k_lstm2_regw<AT, mt, 1, ks, true, TAIL>;
    if constexpr (sizeof(AT) == 4) {  // (bfloat16: k_lstm2_sparse)
      if constexpr (HI) {
        RTN_CASE(2, 8) RTN_CASE(4, 8) RTN_CASE(8, 8)
      } else {
        RTN_CASE(2, 2) RTN_CASE(2, 4)
        RTN_CASE(4, 2) RTN_CASE(4, 4)
      }
    }
#undef RTN_CASE
    return nullptr;
  }
#define RTN_CASE(mt, nt, ks) \
  if (MT == mt && NT == nt && KSMAX == ks) return &k_lstm2_regw<AT, mt, nt, ks, false, TAIL>;
  if constexpr (HI) {
    RTN_CASE(1, 1, 8) RTN_CASE(1, 2, 8) RTN_CASE(1, 4, 8)
    RTN_CASE(2, 1, 8) RTN_CASE(2, 2, 8) RTN_CASE(2, 4, 8)
    RTN_CASE(4, 1, 8) RTN_CASE(4, 2, 8)
    RTN_CASE(8, 1, 8)
    if constexpr (sizeof(AT) == 4) {
      RTN_CASE(1, 1, 16) RTN_CASE(1, 2, 16)
      RTN_CASE(2, 1, 16) RTN_CASE(2, 2, 16)
    }
  } else {
    RTN_CASE(1, 1, 2) RTN_CASE(1, 2, 2) RTN_CASE(1, 4, 2)
    RTN_CASE(2, 1, 2) RTN_CASE(2, 2, 2) RTN_CASE(2, 4, 2)
    RTN_CASE(4, 1, 2) RTN_CASE(4, 2, 2)
    RTN_CASE(1, 1, 4) RTN_CASE(1, 2, 4) RTN_CASE(1, 4, 4)
    RTN_CASE(2, 1, 4) RTN_CASE(2, 2, 4) RTN_CASE(2, 4, 4)
    RTN_CASE(4, 1, 4) RTN_CASE(4, 2, 4)
  }
#undef RTN_CASE
  return nullptr;
}

// Forward, bfloat16 with 16 macro steps per wavefront.
template <bool TAIL>
RegwKernel regw_table_16(int MT, int NT) {
#define RTN_CASE(mt, nt) \
  if (MT == mt && NT == nt) return &k_lstm2_regw<__bf16, mt, nt, 16, false, TAIL>;
  RTN_CASE(1, 1) RTN_CASE(1, 2)
  RTN_CASE(2, 1) RTN_CASE(2, 2)
  RTN_CASE(4, 1)
#undef RTN_CASE
  return nullptr;
}

// Forward, float32 in quads of rows.
template <bool TAIL>
RegwKernel regw_table_quad(int MT, int KSMAX, int RQ) {
#define RTN_CASE(mt, ks) \
  if (MT == mt && KSMAX == ks) \
    return RQ == 1 ? &k_lstm2_regw<float, mt, 1, ks, false, TAIL, 1> : RQ == 2 ? &k_lstm2_regw<float, mt, 1, ks, false, TAIL, 2> : RQ == 3 ? &k_lstm2_regw<float, mt, 1, ks, false, TAIL, 3> : nullptr;
  RTN_CASE(4, 4) RTN_CASE(4, 8)
  RTN_CASE(8, 8)
#undef RTN_CASE
  if (MT == 4 && KSMAX == 2 && RQ == 1) return &k_lstm2_regw<float, 4, 1, 2, false, TAIL, 1>;
  return nullptr;
}

// Gradient.
template <typename AT, bool HALF>
BwdRegwKernel bwd_regw_table(int KSB, int MT, int WV) {
#define RTN_CASE(ks, mt, wv) \
  if (KSB == ks && MT == mt && WV == wv) return &k_lstm2_bwd_regw<AT, ks, mt, wv, 0, HALF>;
  RTN_CASE(2, 1, 4) RTN_CASE(4, 1, 4) RTN_CASE(8, 1, 4) RTN_CASE(16, 1, 4) RTN_CASE(32, 1, 4)
  if constexpr (sizeof(AT) == 2) { RTN_CASE(64, 1, 4) }
  RTN_CASE(2, 2, 4) RTN_CASE(4, 2, 4) RTN_CASE(8, 2, 4) RTN_CASE(16, 2, 4) RTN_CASE(32, 2, 4)
  RTN_CASE(2, 4, 4) RTN_CASE(4, 4, 4) RTN_CASE(8, 4, 4) RTN_CASE(16, 4, 4)
  RTN_CASE(2, 1, 8) RTN_CASE(4, 1, 8) RTN_CASE(8, 1, 8) RTN_CASE(16, 1, 8)
  RTN_CASE(2, 2, 8) RTN_CASE(4, 2, 8) RTN_CASE(8, 2, 8) RTN_CASE(16, 2, 8)
  RTN_CASE(2, 4, 8) RTN_CASE(4, 4, 8) RTN_CASE(8, 4, 8) RTN_CASE(16, 4, 8)
  RTN_CASE(2, 1, 16) RTN_CASE(4, 1, 16) RTN_CASE(8, 1, 16)
  RTN_CASE(2, 2, 16) RTN_CASE(4, 2, 16) RTN_CASE(8, 2, 16)
  RTN_CASE(2, 4, 16) RTN_CASE(4, 4, 16) RTN_CASE(8, 4, 16)
#undef RTN_CASE
  return nullptr;
}

// (groups of up to 8 rows on one XCD each; RQ: float32 in quads of rows)
template <typename AT, int RQ>
BwdRegwKernel bwd_local_table(int KSB, int MT) {
#define RTN_CASE(ks, mt) \
  if (KSB == ks && MT == mt) return &k_lstm2_bwd_local<AT, ks, mt, RQ>;
  RTN_CASE(2, 1) RTN_CASE(4, 1) RTN_CASE(8, 1) RTN_CASE(16, 1) RTN_CASE(32, 1)
  RTN_CASE(2, 2) RTN_CASE(4, 2) RTN_CASE(8, 2) RTN_CASE(16, 2) RTN_CASE(32, 2)
  RTN_CASE(2, 4) RTN_CASE(4, 4) RTN_CASE(8, 4) RTN_CASE(16, 4)
#undef RTN_CASE
  return nullptr;
}

template <typename AT>
BwdRegwKernel bwd_regw_lds_table() { return &k_lstm2_bwd_regw<AT, 16, 1, 8, 16>; }

}  // namespace

#if RTN_TABLE_PART == 1
RegwKernel regw_table_bf16_lo(int MT, int NT, int KSMAX, bool half, bool tail) { return tail ? regw_table<__bf16, false, true>(MT, NT, KSMAX, half) : regw_table<__bf16, false, false>(MT, NT, KSMAX, half); }
#elif RTN_TABLE_PART == 2
RegwKernel regw_table_bf16_hi(int MT, int NT, int KSMAX, bool half, bool tail) { return tail ? regw_table<__bf16, true, true>(MT, NT, KSMAX, half) : regw_table<__bf16, true, false>(MT, NT, KSMAX, half); }
#elif RTN_TABLE_PART == 3
RegwKernel regw_table_f32_lo(int MT, int NT, int KSMAX, bool half, bool tail) { return tail ? regw_table<float, false, true>(MT, NT, KSMAX, half) : regw_table<float, false, false>(MT, NT, KSMAX, half); }
#elif RTN_TABLE_PART == 4
RegwKernel regw_table_f32_hi(int MT, int NT, int KSMAX, bool half, bool tail) { return tail ? regw_table<float, true, true>(MT, NT, KSMAX, half) : regw_table<float, true, false>(MT, NT, KSMAX, half); }
#elif RTN_TABLE_PART == 5
BwdRegwKernel bwd_regw_table_bf16_half(int KSB, int MT, int WV) { return bwd_regw_table<__bf16, true>(KSB, MT, WV); }
#elif RTN_TABLE_PART == 6
BwdRegwKernel bwd_regw_table_bf16_full(int KSB, int MT, int WV) { return bwd_regw_table<__bf16, false>(KSB, MT, WV); }
BwdRegwKernel bwd_regw_lds_table_bf16() { return bwd_regw_lds_table<__bf16>(); }
BwdWideBuild bwd_wide_build(int steps) {
  if (steps > 32 && steps <= 48) return {&k_lstm2_bwd_wide<__bf16, 2, 48, 4>, 2, 4};
  if (steps > 48 && steps <= 64) return {&k_lstm2_bwd_wide<__bf16, 2, 64, 36>, 2, 36};
  return {nullptr, 0, 0};
}
#elif RTN_TABLE_PART == 7
BwdRegwKernel bwd_regw_table_f32_half(int KSB, int MT, int WV) { return bwd_regw_table<float, true>(KSB, MT, WV); }
#elif RTN_TABLE_PART == 8
BwdRegwKernel bwd_regw_table_f32_full(int KSB, int MT, int WV) { return bwd_regw_table<float, false>(KSB, MT, WV); }
BwdRegwKernel bwd_regw_lds_table_f32() { return bwd_regw_lds_table<float>(); }
#elif RTN_TABLE_PART == 9
// Ascending by the width that MT tiles on 256 CUs and KS macro steps per wavefront take, then by rows.  What bounds NT: W,
// 4 MT NT accumulator registers and two chunks of h per wavefront in 512 registers.
WideBuild wide_kernel(int dtype, int n, int cus, int rows) {
#define RTN_WIDE(at, dt, mt, nt, ks, lf) {&k_lstm2_wide<at, mt, nt, ks, lf, false>, wide_stage_bytes(mt, nt, lf, (int)sizeof(at)) ? &k_lstm2_wide<at, mt, nt, ks, lf, !(lf && sizeof(at) == 4)> : nullptr, dt, mt, nt, ks, lf}
  static const WideBuild builds[] = {
      RTN_WIDE(float, 0, 2, 1, 32, 0), RTN_WIDE(float, 0, 2, 2, 32, 0), RTN_WIDE(float, 0, 3, 1, 44, 36),
      RTN_WIDE(__bf16, 1, 3, 1, 24, 0), RTN_WIDE(__bf16, 1, 3, 2, 24, 0), RTN_WIDE(__bf16, 1, 4, 1, 32, 35),
  };
#undef RTN_WIDE
  WideBuild best = {nullptr, nullptr, 0, 0, 0, 0, 0};
  for (const WideBuild& b : builds) {
    if (b.dtype != dtype) continue;
    const int KM = dtype == 1 ? 32 : 16;
    if ((n / 4 + b.MT - 1) / b.MT > cus || (n / KM + kWaves - 1) / kWaves > b.KS) continue;
    if (best.kernel && (b.MT != best.MT || b.KS != best.KS)) break;  // (the narrowest builds that take the width)
    best = b;
    if (rows <= 16 * b.NT) break;
  }
  return best;
}
// Four rows per workgroup: float32 up to n = 64, bf16 up to 128.  Measured at T = 4, 32 and 300 with B = 4 ... 1024, us per call, against k_lstm2_regw: T = 300, B = 4 /
// 1024: float32 n = 32 184 / 204 against 312 / 396, n = 64 211 / 250 against 310 / 473; bf16 n = 32 121 / 143 against 249 / 296, n = 64 186 / 209
// against 248 / 349, n = 96 213 / 281 against 253 / 505, n = 128 263 / 338 against 255 / 547.  Beyond, 8 wavefronts' MFMAs on one CU take longer than a
// hand-over: float32 n = 96 / 128 1.36 / 1.64 us per step against 1.03, bf16 n = 160 1.7 against 0.85.
// One row per workgroup: float32 up to n = 128 (there 1.01 us per step against 1.06 of k_lstm2_regw with few rows, 1.07 against 1.39 with 256), where W takes
// half of the CU's registers; bf16 up to 128 (12 wavefronts for n = 160 have too few registers each).
SoloBuild solo_kernel(int dtype, int n, bool one_row) {
#define RTN_SOLO(at, s) if (n <= s * Elem<at>::KM) return {&k_lstm2_solo<at, s>, 64 * solo_waves<at>(s), kSoloRows};
#define RTN_SOLO_ROW(at, s) if (n <= s * Elem<at>::KM) return {&k_lstm2_solo_row<at, s>, 64 * solo_waves<at>(s), 1};
  if (one_row && dtype == 1) {
    RTN_SOLO_ROW(__bf16, 1) RTN_SOLO_ROW(__bf16, 2) RTN_SOLO_ROW(__bf16, 3) RTN_SOLO_ROW(__bf16, 4)
  } else if (one_row) {
    RTN_SOLO_ROW(float, 2) RTN_SOLO_ROW(float, 4) RTN_SOLO_ROW(float, 6) RTN_SOLO_ROW(float, 8)
  } else if (dtype == 1) {
    RTN_SOLO(__bf16, 1) RTN_SOLO(__bf16, 2) RTN_SOLO(__bf16, 3) RTN_SOLO(__bf16, 4)
  } else {
    RTN_SOLO(float, 2) RTN_SOLO(float, 4)
  }
#undef RTN_SOLO
#undef RTN_SOLO_ROW
  return {nullptr, 0, 0};
}
#elif RTN_TABLE_PART == 10
RegwKernel regw_table_f32_quad_tail(int MT, int KSMAX, int RQ) { return regw_table_quad<true>(MT, KSMAX, RQ); }
#elif RTN_TABLE_PART == 11
RegwKernel regw_table_f32_quad_tail(int MT, int KSMAX, int RQ);
RegwKernel regw_table_f32_quad(int MT, int KSMAX, bool tail, int RQ) { return tail ? regw_table_f32_quad_tail(MT, KSMAX, RQ) : regw_table_quad<false>(MT, KSMAX, RQ); }
#elif RTN_TABLE_PART == 12
BwdRegwKernel bwd_local_table_f32_two(int KSB, int MT);
BwdRegwKernel bwd_local_table_f32(int KSB, int MT, int RQ) { return RQ == 1 ? bwd_local_table<float, 1>(KSB, MT) : RQ == 2 ? bwd_local_table_f32_two(KSB, MT) : nullptr; }
#elif RTN_TABLE_PART == 13
BwdRegwKernel bwd_local_table_f32_two(int KSB, int MT) { return bwd_local_table<float, 2>(KSB, MT); }
#elif RTN_TABLE_PART == 14
RegwKernel dual_kernel(int MT, int KSMAX, bool local) {
  if (local) return MT == 8 && KSMAX == 8 ? &k_lstm2_dual<__bf16, 8, 8, false> : nullptr;
  return MT == 4 && KSMAX == 16 ? &k_lstm2_dual<__bf16, 4, 16, true> : nullptr;
}
#elif RTN_TABLE_PART == 15
BwdRegwKernel bwd_local_table_bf16(int KSB, int MT) { return bwd_local_table<__bf16, 0>(KSB, MT); }
#elif RTN_TABLE_PART == 16
RegwKernel sparse_kernel(int MT, int KSMAX, bool tail) {
#define RTN_CASE(mt, ks) \
  if (MT == mt && KSMAX == ks) return tail ? &k_lstm2_sparse<mt, ks, true> : &k_lstm2_sparse<mt, ks, false>;
  RTN_CASE(2, 2) RTN_CASE(2, 4) RTN_CASE(2, 8)
  RTN_CASE(4, 2) RTN_CASE(4, 4) RTN_CASE(4, 8)
  RTN_CASE(8, 8)
#undef RTN_CASE
  return nullptr;
}
#elif RTN_TABLE_PART == 17
RegwKernel regw_table_bf16_16(int MT, int NT, bool tail) { return tail ? regw_table_16<true>(MT, NT) : regw_table_16<false>(MT, NT); }
#else
#error "RTN_TABLE_PART must be 1..17"
#endif

}  // namespace rtn
