// bgemm_flex.h - the BF16 GEMM on small tiles and on operands of any alignment (bgemm_flex.hip).
#pragma once

#include "hk_host.h"

namespace hk {

namespace gemm {
struct Epi;
}

// How such a product runs: tile shape `tile` (an id, 0: none), `used` k splits of kps k each, and
// the modelled time (us).
struct FlexPlan {
  int tile, used, kps;
  double cost;
};
// split_k == 0: the library's choice of splits. ragged: rows that are no whole 16-byte vectors.
FlexPlan bgemm_flex_plan(int M, int N, int K, int batch, int split_k, bool ragged);
// Rows of one output tile of a plan's tile shape (0 for none).
int bgemm_flex_tile_rows(int tile);

struct FlexCall {
  bool ta, tb;
  int M, N, K, batch;
  const hk_bf16* A;
  int64_t lda, sA;
  const hk_bf16* B;
  int64_t ldb, sB;
  hk_bf16* C;
  int64_t ldc, sC;
  const gemm::Epi* ep;  // NULL with part or out
  int used, kps;
  float* part;          // used > 1: the fp32 partials [split][batch][M][part_pitch(N)]
  const F32Out* out;    // not NULL: fp32 C instead (used == 1, N % 8 == 0)
};
hipError_t bgemm_flex_run(int tile, const FlexCall& call, hipStream_t stream);

}  // namespace hk
