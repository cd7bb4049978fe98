// Host side of the MX e4m3 GEMM on the tiles of gemm_mid.h (gemm_mid_fp8.hip).
#pragma once
#include "gemm_mid_api.h"

namespace dnn {

// A, W: e4m3 rows of Kb bytes; sx: e8m0 per row and 128 columns of A; sw: per column
// of the output.  qo: the output is quantised in the epilogue (GELU, e4m3 rows of
// ldq bytes with kpo columns, scales sxo) and C not written.
struct Mid8Args : MidRows {
  const uint8_t* A;
  const uint8_t* W;
  const uint32_t* sx;
  const float* sw;
  uint8_t* qo;
  uint8_t* sxo;
  int Kb, ldq, kpo;
};

int mid8_blocks(int tile);  // workgroups of a tile that share a CU
int mid8_launch(int tile, const Mid8Args& a, const QkvScatter* scat, hipStream_t st);

}  // namespace dnn
