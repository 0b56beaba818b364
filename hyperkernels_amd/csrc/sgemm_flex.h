// sgemm_flex.h - fp32 GEMM on the fp32 MFMA for small products and rows of any alignment
// (sgemm_flex.hip).
#pragma once

#include "hk_host.h"

namespace hk {

struct SgemmFlexCall {
  bool ta, tb;
  int M, N, K, batch;  // K > 0, leading dimensions in [4, 2^21)
  const float* A;
  int64_t lda, sA;
  const float* B;
  int64_t ldb, sB;
  F32Out out;
};
// Index of the tile shape for a product: the least modelled time among those that form an output's sum
// from min_chains serial ones at least, or from as many as any shape does.
int sgemm_flex_plan(int M, int N, int K, int batch, int min_chains);
hipError_t sgemm_flex_run(int shape, const SgemmFlexCall& call, hipStream_t stream);

}  // namespace hk
