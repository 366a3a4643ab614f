// Product of more than 16 tokens with a plain VQ weight whose codebook LDS holds (see table_gemm.hip).
#pragma once

#include "vq_call.hpp"

namespace npamd {

struct TablePlan {
  int tile;  // -1: the kernel does not take the call
  float us;
};
// The tile of least estimate for M tokens, and that estimate.
TablePlan plan_table_gemm(int M, int N, int K, int nc);
// Takes the call (c.k_in as in npamd_vq_gemv_blocks) if its estimate is below `other_us`; 1 when it does not.
int launch_table_gemm(const VqCall& c, float other_us);
// The GEMV with a workgroup per 32 tokens, us (dense_gemm.hip).  kind: 0 VQ, 1 residual VQ, 4 and 8 bits per weight.
float gemv_blocks_us(int kind, int table_rows, int M, int N, int K);

}  // namespace npamd
