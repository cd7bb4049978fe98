// Decode steps of a row or two by partial products (decode_row.hip).
#pragma once
#include <hip/hip_runtime.h>

constexpr int DECODE_ROWS = 2;  // rows that such a step may have

// A block's projections: fragment-order bf16 copies, fp32 vectors.
struct RowBlock {
  const void *w_qkv, *w_o, *w_up, *w_down;
  const float *cs_qkv, *b_qkv, *b_o, *cs_up, *b_up, *b_down;
};

extern "C" {
long long dnn_decode_row_parts(int M, int d, int H, int Hkv, int hd, int S);
int dnn_decode_row_blocks(const RowBlock* blocks, int n, const void* x, void* a, void* h, void* qkv, void* f, float* parts,
                          char* kc, char* vc, long long kv_block, int M, int d, int H, int Hkv, int hd, int S,
                          const int* pos, float scale, float eps, hipStream_t st);
// attn_decode_qkv of heads of 64 whose output goes on through W_o: part[h][b][:] = head h of row b times the
// columns of wo (fragment order, N = K = 64 H) that read it
int dnn_attn_decode_proj(const void* qkv, int ldq, void* kc, void* vc, const void* wo, float* part, int B, int H, int S,
                         const int* pos, float scale, hipStream_t st);
}
