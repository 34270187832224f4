// The small-launch GEMM (gemm_small.hip) as gemm.hip's dispatch sees it.
#pragma once

#include "common.hpp"

namespace dlt {

enum class SmallElem { BF16, FP8, MX, F32 };

// bm x bn tiles, K in `pieces` of piece_stages 128-byte stages; bm == 0: not worth it.
struct SmallPlan {
  int bm, bn, pieces, piece_stages;
};

// The fastest plan for one m x n x k problem on `cus` compute units with `scratch` bytes for the
// K pieces' sums (0: K stays whole), if it beats big_us, the 256 x 256 tiles' estimate.
SmallPlan small_plan(SmallElem e, int64_t m, int64_t n, int64_t k, int cus, int64_t scratch,
                     double big_us);

// Runs the plan: operands checked by the caller as for gemm.hip (F32: gemm_f32.hip, C, bias and
// residual fp32, residual + (acc + bias)). gate: EPI_GATE_RESIDUAL.
void gemm_small(SmallElem e, const SmallPlan& plan, const difflet_gemm_problem& q, int64_t n,
                int64_t k, bool gate, int64_t rows_per_batch, void* scratch, hipStream_t s);

// Compute units of the current device (gemm.hip).
int gemm_device_cus();

}  // namespace dlt
