#pragma once
// Decode projections laid out for one shape each (gemm_lean.hip).
#include "gemm_epilogue.h"

namespace dnn {

enum SkNorm { NORM_NONE = 0, NORM_RMS = 1, NORM_LN = 2 };

typedef float f32x2 __attribute__((ext_vector_type(2)));

// 16 OCP e4m3 weight bytes -> 16 bf16 (exact: every e4m3 value is a bf16
// value).  gfx950's v_cvt_scalef32_pk_bf16_fp8 (scale 1.0) turns two bytes into
// a packed bf16 pair in one op: 8 VALU per 16 B instead of 8 fp32 converts + 8
// repacks — the decode weight stream is VALU-paced at batch 1.
__device__ __forceinline__ void w8_to_bf16(const i32x4& w, bf16x8& lo, bf16x8& hi) {
  bf16x2v o[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    o[2 * i] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((uint32_t)w[i], 1.0f, false);
    o[2 * i + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((uint32_t)w[i], 1.0f, true);
  }
  __builtin_memcpy(&lo, &o[0], 16);
  __builtin_memcpy(&hi, &o[4], 16);
}

struct LeanArgs {
  const uint8_t* A;
  int lda_b;
  const uint8_t* W;
  const float* sw;
  bf16_t* C;
  int ldc;
  const float* bias;
  const bf16_t* R;
  int ldr, M, N;
  const float* colsum;
  float eps;
  const float2* rs_in;  // LayerNorm: partials of A's rows (epi_rowstat16)
  int rs_in_ld;
  float2* rs_out;
  int rs_out_ld;
};

// C[M,N] = act(norm(A) W^T * sw + bias) (+ R) where the shape is one of those laid out: false, nothing launched, elsewhere.
bool dnn_gemm_lean(const LeanArgs& p, int nch, int act, int norm, bool w8, hipStream_t st);

}  // namespace dnn
