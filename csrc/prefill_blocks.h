// The launches of one prefill pass through a stage's blocks, issued in one call.
//
// A pass of a few hundred tokens is a chain of 5 to 9 launches a block of 3 to 10 us
// each; issued one by one from Python (10 us a launch: argument checks, tensor views,
// the call) the device waits for the host: GPT-2, 66 to 256 tokens, 680 us for 63
// launches that run 300.  The sequence and what it computes are those of
// runtime/transformer.py TransformerStage.step with T > 1 and folded norms, and so are the
// kernels but for two that only this call launches: the q | k | v product that rotates
// (dnn_gemm_bf16_qkv_rope: the bits of product and pass) and the attention that quantises its
// rows (dnn_flash_attn_mx: the bytes of attention and quantiser).  Weights come as pointers of
// this call, read from the stage's layers.
#pragma once
#include <cstdint>
#include <vector>

#include "kernels/api.h"
#include "kernels/gemm_mid_api.h"

namespace dnn {

// A projection: row-major weight (bf16, or e4m3 rows of kp bytes with column scales),
// bias, row sums (folded LayerNorm), fragment-order copy; null where there is none.
struct PrefillProj {
  const void* w;
  const float *scale, *bias, *colsum;
  const void* frag;
};
struct PrefillBlock {
  PrefillProj qkv, o, up, down;
};

struct PrefillPass {
  int B, T, d, H, Hkv, hd, S, ffn, n_up, act, norm;
  float eps, scale;
  int skinny_rows, skinny_max;  // rows that always / may run on the decode kernels (ops/gemm.py skinny_rows)
  int fp8, scatter;
  const void* x;                // (B T, d) input rows; a block's residual stream is h
  void *h, *a, *qkv, *q, *att, *f;
  void *q8, *sx, *q8b, *sxb;    // fp8: MX activations and scales, those of the c_fc output
  float* s8;                    // fp8: row scales of activations that are not MX
  void* parts;                  // partials of the row statistics of h, [rows][d / 32], or null
  const float* ones;
  char *kc, *vc;                // this stage's caches at the first sequence, one block's bytes apart
  long long kv_block;
  const int* pos;
  const float *cosT, *sinT;
  void* ws;
  long long ws_bytes;
  hipStream_t st;
  int more;                     // another call runs the blocks behind these
  bool have;                    // `parts` holds the partials of x; after run(), of h
  const char* what = "";

  int rows() const { return B * T; }
  static int kpad(int k) { return (k + 127) / 128 * 128; }

  bool skinny(int N, int K, bool norm_in, bool frag, long long wsb) const {
    const int M = rows();
    if (fp8) return M <= 64 || (M <= skinny_max && ((M + 127) / 128) * ((N + 127) / 128) < 192);
    if (M <= skinny_rows || M > skinny_max) return M <= skinny_rows;
    return dnn_gemm_is_skinny(M, N, K, norm_in, frag, wsb) != 0;
  }
  bool mx(int N) const { return rows() >= 256 && N >= 256; }

  int quant_norm(const void* in) {
    what = "layernorm_q8_mx";
    return dnn_layernorm_q8_mx(in, d, nullptr, nullptr, q8, kpad(d), sx, rows(), d, kpad(d), eps, norm == 1, st);
  }

  // out = act(norm(in) W^T + bias), in (rows, d).  fp8: row_scale: one scale a row, else MX; quant: the
  // output leaves as MX e4m3 in q8b / sxb
  int norm_proj(const void* in, const PrefillProj& p, void* out, int ldo, int N, int act_, bool row_scale, bool quant) {
    const int M = rows();
    if (skinny(N, d, true, p.frag != nullptr, ws_bytes)) {
      what = fp8 ? "gemm_skinny_w8" : "gemm_skinny_norm";
      return fp8 ? dnn_gemm_skinny_w8(in, d, p.w, kpad(d), p.scale, out, ldo, p.bias, nullptr, 0, M, N, d, act_, norm,
                                      p.colsum, eps, st, p.frag, ws, ws_bytes)
                 : dnn_gemm_skinny_norm(in, d, p.w, d, out, ldo, p.bias, nullptr, 0, M, N, d, act_, norm, p.colsum,
                                        eps, st, p.frag, ws, ws_bytes);
    }
    if (fp8 && row_scale) {
      what = "layernorm_q8";
      if (const int rc = dnn_layernorm_q8(in, d, ones, nullptr, q8, kpad(d), s8, M, d, kpad(d), eps, norm == 1, st, 0))
        return rc;
      what = "gemm_fp8";
      return dnn_gemm_fp8(q8, s8, p.w, p.scale, out, ldo, p.bias, nullptr, 0, M, N, kpad(d), act_, st);
    }
    if (fp8) {
      if (const int rc = quant_norm(in)) return rc;
      what = "gemm_fp8_mx";
      return dnn_gemm_fp8_mx(q8, sx, p.w, p.scale, out, ldo, p.bias, nullptr, 0, M, N, kpad(d), act_,
                             quant ? q8b : nullptr, quant ? kpad(N) : 0, quant ? sxb : nullptr, quant ? kpad(N) : 0, st);
    }
    what = "gemm_bf16_parts";
    int wrote;
    return dnn_gemm_bf16_parts(in, d, p.w, d, out, ldo, p.bias, nullptr, 0, M, N, d, act_, st, nullptr, norm, eps,
                               (float*)a, have ? parts : nullptr, p.colsum, nullptr, &wrote, ws, ws_bytes);
  }

  // h = in W^T + bias + res, in (rows, K); qin, sin: in as MX e4m3, where its producer left it so; read: the
  // next projection takes h's partials (`have`: they were written)
  int res_proj(const void* in, const PrefillProj& p, const void* res, int K, const void* qin, const void* sin, bool read) {
    const int M = rows();
    have = false;
    if (!fp8) {
      what = "gemm_bf16_parts";
      int wrote = 0;
      const int rc = dnn_gemm_bf16_parts(in, K, p.w, K, h, d, p.bias, res, d, M, d, K, 0, st, p.frag, 0, 0.f, nullptr,
                                         nullptr, nullptr, read ? parts : nullptr, &wrote, ws, ws_bytes);
      have = wrote != 0;
      return rc;
    }
    if (skinny(d, K, false, true, ws_bytes)) {
      what = "gemm_skinny_w8";
      return dnn_gemm_skinny_w8(in, K, p.w, kpad(K), p.scale, h, d, p.bias, res, d, M, d, K, 0, 0, nullptr, 0.f, st,
                                p.frag, ws, ws_bytes);
    }
    if (qin == nullptr) {
      qin = q8, sin = sx;
      what = "quant_fp8_mx";
      if (const int rc = dnn_quant_fp8_mx(in, K, q8, kpad(K), sx, M, K, kpad(K), st)) return rc;
    }
    what = "gemm_fp8_mx";
    return dnn_gemm_fp8_mx(qin, sin, p.w, p.scale, h, d, p.bias, res, d, M, d,
                           kpad(K), 0, nullptr, 0, nullptr, 0, st);
  }

  // q, K and V of a block straight to q and the caches: 1 done, 0 not this shape, < 0 or > 1 failed
  int scattered(const void* in, const PrefillProj& p, void* k, void* v, int& rc) {
    const int N = (H + 2 * Hkv) * hd;
    rc = 0;
    if (!scatter || skinny(N, d, true, fp8 || p.frag != nullptr, 0)) return 0;
    if (cosT != nullptr) {
      if (fp8 || norm != 1 || p.bias != nullptr || p.colsum != nullptr) return 0;
      what = "gemm_bf16_qkv_rope";
      rc = dnn_gemm_bf16_qkv_rope(in, d, p.w, d, eps, (float*)a, q, k, v, pos, B, T, H, Hkv, hd, S, d, cosT, sinT,
                                  mid_ws(ws, ws_bytes), st);
      if (rc != -3) return 1;
      rc = 0;
      return 0;
    }
    if (fp8) {
      if (N % 32 != 0) return 0;
      if ((rc = quant_norm(in))) return 0;
      what = "gemm_fp8_qkv_scatter_mx";
      rc = dnn_gemm_fp8_qkv_scatter_mx(q8, sx, p.w, p.scale, p.bias, q, k, v, pos, B, T, H, Hkv, hd, S, kpad(d), st);
      return 1;
    }
    what = "gemm_bf16_qkv_scatter_parts";
    rc = dnn_gemm_bf16_qkv_scatter_parts(in, d, p.w, d, p.bias, norm, eps, (float*)a, have ? parts : nullptr, p.colsum, q, k,
                                         v, pos, B, T, H, Hkv, hd, S, d, st);
    if (rc == -3) {  // off the tiles with the scatter epilogue: projection rows instead
      rc = 0;
      return 0;
    }
    return 1;
  }

  // fp8: every projection runs on the decode kernels or on MX activations
  bool covered() const {
    if (!fp8) return true;
    const int N[3] = {(H + 2 * Hkv) * hd, d, n_up}, K[3] = {d, H * hd, d};
    for (int i = 0; i < 3; ++i)
      if (!skinny(N[i], K[i], true, true, 0) && !mx(N[i])) return false;
    // a quantised c_fc output needs a c_proj that reads it
    return act != 2 || skinny(n_up, d, true, true, 0) || !skinny(d, ffn, false, true, 0);
  }

  int run(const std::vector<PrefillBlock>& blocks) {
    const void* in = x;
    const int nq = (H + 2 * Hkv) * hd;
    const int one_group = fp8 && rows() > skinny_max;  // e4m3 activations follow (attention.hip flash_two_groups)
    // the attention quantises its rows itself where the projection behind it takes MX rows
    const bool att_quant = one_group && hd == 64 && !skinny(d, H * hd, false, true, ws_bytes);
    const bool up_quant = fp8 && act == 2 && !skinny(n_up, d, true, true, 0);
    const bool part = parts != nullptr && !fp8;
    for (size_t i = 0; i < blocks.size(); ++i) {
      const PrefillBlock& L = blocks[i];
      // who reads h's partials: not the decode kernels, and none is behind the last block
      const bool read_up = part && !skinny(n_up, d, true, L.up.frag != nullptr, ws_bytes) &&
                           dnn_gemm_takes_parts(rows(), n_up, d, d, d, act, 0, ws_bytes);
      const bool read_qkv = part && scatter && cosT == nullptr && (more || i + 1 < blocks.size()) &&
                            !skinny(nq, d, true, L.qkv.frag != nullptr, 0) && dnn_gemm_takes_parts(rows(), nq, d, d, d, 0, 1, 0);
      void *k = kc + i * kv_block, *v = vc + i * kv_block;
      int rc;
      bool mx_att = false;
      if (scattered(in, L.qkv, k, v, rc)) {
        if (rc) return rc;
        if (att_quant) {
          what = "flash_attn_mx";
          rc = dnn_flash_attn_mx(q, k, v, q8, kpad(H * hd), sx, B, T, H, Hkv, hd, S, pos, scale, st);
          mx_att = rc != -3;
        }
        if (!mx_att) {
          what = "flash_attn";
          rc = dnn_flash_attn(q, k, v, att, B, T, H, Hkv, hd, S, pos, scale, st, 0, one_group);
        }
      } else {
        if (rc) return rc;
        if ((rc = norm_proj(in, L.qkv, qkv, nq, nq, 0, true, false))) return rc;
        if (cosT == nullptr) {
          what = "flash_attn_qkv";
          rc = dnn_flash_attn_qkv(qkv, nq, k, v, att, B, T, H, Hkv, hd, S, pos, scale, st, 0, one_group);
        } else {
          what = "qkv_split";
          if ((rc = dnn_qkv_split(qkv, q, k, v, B, T, H, Hkv, hd, S, pos, cosT, sinT, 1, st))) return rc;
          what = "flash_attn";
          rc = dnn_flash_attn(q, k, v, att, B, T, H, Hkv, hd, S, pos, scale, st, 0, one_group);
        }
      }
      if (rc) return rc;
      if ((rc = res_proj(att, L.o, in, H * hd, mx_att ? q8 : nullptr, mx_att ? sx : nullptr, read_up))) return rc;
      if ((rc = norm_proj(h, L.up, f, ffn, n_up, act, false, up_quant))) return rc;
      if ((rc = res_proj(f, L.down, h, ffn, up_quant ? q8b : nullptr, up_quant ? sxb : nullptr, read_qkv))) return rc;
      in = h;
    }
    return 0;
  }
};

}  // namespace dnn
