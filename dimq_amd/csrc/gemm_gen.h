// The general pre-laid path (gemm_gen.hip): any codebook Linear or Conv2d as
// one fp16 GEMM whose operands a first launch lays out.
#pragma once

#include "gemm_kernel.h"

namespace dimq {

// What a call's first launch writes where, and how the GEMM is cut.
struct GenPlan {
  bool ok = false;
  bool conv = false, a4 = false, hilo = false;
  bool direct_x = false;  // the activations are read in place
  int splits = 1;         // k ranges (> 1: fp32 partial outputs and a second pass)
  int64_t cg = 0;         // channels per group padded to 8 (Linear: K padded to a stage)
  int64_t kp = 0;         // k of one weight plane: taps * cg, padded to a stage
  int64_t step = 0;       // images (Linear: rows) laid out and multiplied at a time
  int64_t pixels = 0;     // rows of the laid-out activations: those of `step` images
  int64_t planes = 0;     // flag words per row (0: fp16 activations or codes, no range guard)
  int64_t off_rs = 0, off_x = 0, off_flags = 0, off_zero = 0, off_part = 0;
  int64_t bytes = 0;      // workspace
};

// p: the call's arguments (for a4 the activations themselves, with act_scale /
// act_zp).  Only sizes, layouts and dtypes are read; `in_place`: x may be read
// in place (16-byte aligned).
GenPlan gen_plan(const GemmArgs& p, int bits, int x_dtype, bool a4, bool in_place);

// Runs the plan's launches.  `ws` is 256-byte aligned and holds plan.bytes.
int launch_gen(const GemmArgs& p, const GenPlan& plan, int bits, int x_dtype, void* ws, hipStream_t s);

// k ranges (1: no split) of a GEMM with `tiles` tiles of `stages` k stages that
// take us_per_stage on a CU of their own.  Splitting fills a chip that has
// fewer tiles than CUs, for a second launch over the fp32 partial outputs: 5 us
// and their bytes at 4 TB/s.  A range more has to save a tenth.
int split_ranges(int64_t tiles, int64_t stages, double us_per_stage, int64_t outputs);

// y = epilogue(rs * sum over the splits of part + bias); part holds `splits`
// planes in y's element order.  guard: sums that are not finite are recomputed.
void launch_split_reduce(const GemmArgs& p, const float* part, int splits, const float* rs, int x_dtype, int bits,
                         bool guard, bool tapmajor, hipStream_t s);

// The two launches of a split codebook GEMM on gemm_big_kernel: the arguments
// of the first, and the workspace of its partial outputs.
inline int64_t split_bytes(int splits, int64_t M, int64_t ldy) {
  return (static_cast<int64_t>(splits) * M * ldy * 4 + 255) / 256 * 256;
}
inline GemmArgs split_args(const GemmArgs& p, int splits, void* ws) {
  GemmArgs q = p;
  q.splits = splits;
  q.y = ws;
  q.y_dt = DIMQ_F32;
  q.bias = nullptr;
  q.epi = Epi{};
  return q;
}

}  // namespace dimq
