// Which build of the persistent kernels serves which decomposition.  The kernels are templates with many
// instantiations; they are compiled in several parts, each a compilation of lstm2_kernel_tables.hip with another value
// of RTN_TABLE_PART, so that the parts build side by side.  The host code asks these functions for a kernel and launches
// it through the pointer.
#pragma once

#include "lstm2_bwd_kernels.h"
#include "lstm2_bwd_local_kernel.h"
#include "lstm2_bwd_wide_kernel.h"
#include "lstm2_kernels.h"
#include "lstm2_dual_kernel.h"
#include "lstm2_solo_kernel.h"
#include "lstm2_sparse_kernel.h"
#include "lstm2_wide_kernel.h"

namespace rtn {

typedef void (*RegwKernel)(const Lstm2Multi);
typedef void (*BwdRegwKernel)(const Lstm2BwdMulti);

// Forward register kernel k_lstm2_regw<AT, MT, NT, KSMAX, HALF, TAIL>; null if the decomposition has no build.
// "lo": KSMAX of 2 or 4 macro steps per wavefront, "hi": 8 or 16.
RegwKernel regw_table_bf16_lo(int MT, int NT, int KSMAX, bool half, bool tail);
RegwKernel regw_table_bf16_hi(int MT, int NT, int KSMAX, bool half, bool tail);
RegwKernel regw_table_bf16_16(int MT, int NT, bool tail);
RegwKernel regw_table_f32_lo(int MT, int NT, int KSMAX, bool half, bool tail);
RegwKernel regw_table_f32_hi(int MT, int NT, int KSMAX, bool half, bool tail);

// k_lstm2_sparse<MT, KSMAX, TAIL>: bfloat16 groups of up to 8 rows.
RegwKernel sparse_kernel(int MT, int KSMAX, bool tail);

// Forward kernel for small layers k_lstm2_solo<AT, S, R>: the build for width n (one_row: the one with a row per workgroup, if
// the width has it); kernel null: none.
struct SoloBuild {
  RegwKernel kernel;
  int threads, rows;
};
SoloBuild solo_kernel(int dtype, int n, bool one_row);

// k_lstm2_dual<__bf16, MT, KSMAX, !local>: two turns of a large batch in one launch; null if the decomposition has no build.
RegwKernel dual_kernel(int MT, int KSMAX, bool local);

// Forward kernel for wide layers k_lstm2_wide<AT, MT, NT, KS, LF, STAGED>.
typedef void (*WideKernel)(const Lstm2Params);
struct WideBuild {
  WideKernel kernel, staged;  // staged: for rows that begin on 16 bytes; null: none
  int dtype, MT, NT, KS, LF;
};
// The build for a layer of width n on `cus` CUs and `rows` rows per launch; the last one in the list if rows are more than
// any build for that width takes; kernel null: none.
WideBuild wide_kernel(int dtype, int n, int cus, int rows);

// Persistent gradient kernel k_lstm2_bwd_regw<AT, KSB, MT, WV, 0, HALF>; KSB: fragments of W per tile and wavefront,
// MT: tiles of 16 values of k per workgroup, WV: wavefronts per workgroup.  "half": groups of at most 8 rows.
BwdRegwKernel bwd_regw_table_bf16_half(int KSB, int MT, int WV);
BwdRegwKernel bwd_regw_table_bf16_full(int KSB, int MT, int WV);
BwdRegwKernel bwd_regw_table_f32_half(int KSB, int MT, int WV);
BwdRegwKernel bwd_regw_table_f32_full(int KSB, int MT, int WV);
// k_lstm2_bwd_local<AT, KSB, MT, RQ>: groups of at most 8 rows on one XCD each; float32: of at most 4 RQ rows, the product in quads.
BwdRegwKernel bwd_local_table_bf16(int KSB, int MT);
BwdRegwKernel bwd_local_table_f32(int KSB, int MT, int RQ);
// The variants with half of a wavefront's share of W in registers and half in LDS (one tile per workgroup).
BwdRegwKernel bwd_regw_lds_table_bf16();
BwdRegwKernel bwd_regw_lds_table_f32();
// k_lstm2_bwd_wide<__bf16, MT, KST, LF>: the build for `steps` macro steps per wavefront; kernel null: none.
struct BwdWideBuild {
  BwdRegwKernel kernel;
  int tiles, lds_fragments;
};
BwdWideBuild bwd_wide_build(int steps);

// k_lstm2_regw<float, MT, 1, KSMAX, false, TAIL, RQ>: the product in quads of rows.
RegwKernel regw_table_f32_quad(int MT, int KSMAX, bool tail, int RQ);

// rq > 0: the product in quads of rows (float32)
inline RegwKernel regw_kernel(int dtype, int MT, int NT, int KSMAX, bool half, bool tail, int rq) {
  if (rq > 0) return dtype == 0 && NT == 1 ? regw_table_f32_quad(MT, KSMAX, tail, rq) : nullptr;
  if (half && dtype == 1 && two_chains<__bf16>(KSMAX)) return sparse_kernel(MT, KSMAX, tail);
  if (dtype == 1 && KSMAX == 16) return half ? nullptr : regw_table_bf16_16(MT, NT, tail);
  const bool lo = KSMAX <= 4;
  if (dtype == 1 /* RTN_DTYPE_BF16 */) return lo ? regw_table_bf16_lo(MT, NT, KSMAX, half, tail) : regw_table_bf16_hi(MT, NT, KSMAX, half, tail);
  return lo ? regw_table_f32_lo(MT, NT, KSMAX, half, tail) : regw_table_f32_hi(MT, NT, KSMAX, half, tail);
}

}  // namespace rtn
