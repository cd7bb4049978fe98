// Host side of the GEMM for 65 to a few thousand rows (gemm_mid.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "common.h"

namespace dnn {

struct MidArgs {
  const bf16_t* A;
  const bf16_t* W;
  void* C;
  const float* bias;
  const bf16_t* R;
  const float2* rowstat;
  const float* colsum;
  float* part;  // splits > 1: fp32 parts [splits][M][N]
  int lda, ldw, ldc, ldr, M, N, K, splits, act, f32;
};

struct QkvScatter;
struct MidPlan {
  int tile;    // index into the tile table, < 0: the 256 x 256 kernel is the faster one
  int splits;  // workgroups over K
  float us;    // estimated time
};

// `ws_bytes`: room for parts (0: no split).  `scatter`: head-major output, no split.
MidPlan mid_plan(int M, int N, int K, long long ws_bytes, bool scatter);
// Whether M rows still run faster on the decode kernels (`norm`: with a folded norm; `frag`: with the weight's fragment-order copy).
bool mid_skinny(int M, int N, int K, bool norm, bool frag, long long ws_bytes);
// Bytes of a decode workspace that parts may use: its last 4 KiB hold the decode stream kernel's tickets.
inline long long mid_ws(const void* ws, long long bytes) { return ws == nullptr ? 0 : bytes - 4096; }
int mid_launch(int tile, const MidArgs& a, const QkvScatter* scat, hipStream_t st);  // a.splits workgroups over K

}  // namespace dnn
