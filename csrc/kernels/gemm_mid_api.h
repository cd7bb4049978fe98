// Host side of the GEMM for 65 to a few thousand rows (gemm_mid.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "common.h"

namespace dnn {

// Output rows and their epilogue.
struct MidRows {
  void* C;
  const float* bias;
  const bf16_t* R;
  int ldc, ldr, M, N, act, f32;
};

struct MidArgs : MidRows {
  const bf16_t* A;
  const bf16_t* W;
  const float2* rowstat;
  const float* colsum;
  // Row statistics by way of partials {mean, sum of squared deviations} of 32 columns of a row: written with the
  // bf16 output [M][N / 32], or read for the folded norm instead of rowstat [M][K / 32]
  float2* parts_out;
  const float2* parts;
  float eps;
  int rms;
  float* part;  // splits > 1: fp32 parts [splits][M][N]
  int lda, ldw, K, splits;
};

struct QkvScatter;
struct MidPlan {
  int tile;    // index into the tile table, < 0: the 256 x 256 kernel is the faster one
  int splits;  // workgroups over K
  float us;    // estimated time
  int cols;    // leading columns as 256 x 256 tiles in a launch of their own, the rest as above (0: none)
};

// `ws_bytes`: room for parts (0: no split).  `kind`: bf16, with the columns in one launch
// or in two, or tiles that the MX e4m3 kernel has (K then in 128-byte K-tiles x 64),
// all or with whole 128 columns.
enum MidKind : unsigned { MID_BF16 = 0, MID_BF16_WHOLE = 1, MID_MX = 2, MID_MX_QUANT = 3 };
MidPlan mid_plan(int M, int N, int K, long long ws_bytes, unsigned kind);
// Whether M rows still run faster on the decode kernels (`norm`: with a folded norm; `frag`: with the weight's fragment-order copy).
bool mid_skinny(int M, int N, int K, bool norm, bool frag, long long ws_bytes);
// Bytes of a decode workspace that parts may use: its last 4 KiB hold the decode stream kernel's tickets.
inline long long mid_ws(const void* ws, long long bytes) { return ws == nullptr ? 0 : bytes - 4096; }
// Widest rows whose partials a workgroup merges, and what the columns of a product with partials divide by.
constexpr int MID_PARTS_K = 2048, MID_PARTS_N = 64;
int mid_blocks(int tile);  // workgroups of a tile (K whole) that share a CU
// The same on a kernel with that epilogue alone (gemm_mid_plain.hip); -3, nothing launched: there is none.
int mid_plain_launch(int tile, const MidArgs& a, hipStream_t st);
int mid_launch(int tile, const MidArgs& a, const QkvScatter* scat, hipStream_t st);  // a.splits workgroups over K

}  // namespace dnn
