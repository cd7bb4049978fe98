// C ABI of the decoder kernels with an fp32 residual and a paged KV cache
// (residual_rows.hip, token_gate.hip, gemm_f32.hip,
// paged_attention.hip, latent_attention.hip, poly_norm.hip).  As in api.h: every
// function enqueues on `st`; 0 = success, negative = rejected shape.
#pragma once
#include <hip/hip_runtime.h>
#include "glu_clamp.h"

struct RowsArgs {
  const float* x_in;   // residual rows (nullptr: 0)
  const int* xidx;     // optional gather of x rows (no x_out then), xrows entries exist
  const void* y;       // sublayer output rows (nullptr: none)
  const int* yidx;     // optional gather of y rows
  const float* y_w;    // RMS-norm weight of y (nullptr: y as it is)
  float* x_out;        // updated residual (may be x_in)
  void* copy;          // optional copy of x' as a GEMM operand
  const float* n_w;    // norm weight of h (nullptr: no h)
  void* h;
  int xrows, yrows, ldx, ldy, ldcopy, ldh, M, N, NP;
  float mult, eps;
  // optional parts (zero: absent)
  const float* x_add = nullptr;     // fp32 rows joined to x as they are (stride ldadd)
  const void* y2 = nullptr;         // second sublayer output, RMS-normed with y2_w, joined like y
  const float* y2_w = nullptr;
  const void* ys = nullptr;         // weighted rows joined to y: sum over t < top of ysw[m * top + t] * ys[ysi[m * top + t]]
  const int* ysi = nullptr;
  const float* ysw = nullptr;
  const float* n_b = nullptr;       // with it the norm is tanh(n_alpha x') * n_w + n_b (no mean, no variance)
  const int* pos = nullptr;         // with freq: a sinusoidal position vector joins x (columns < N), entry 2i
  const double* freq = nullptr;     //   sin, 2i + 1 cos of 2 pi * pos * freq[i] (freq in turns)
  int ldadd = 0, ldy2 = 0, ldys = 0, ysrows = 0, top = 0;
  float n_alpha = 0.f;
  int y_joined = 0;                 // with ys: y_w norms the joined row instead of y alone
  // token shift (with n_w): h <- h + (h of the sequence's token before - h) * sh_mu, zeros before the first
  const float* sh_mu = nullptr;
  float* sh_state = nullptr;        // [slot][NP]: h of every sequence's last token, before the shift
  const int* sh_start = nullptr;    // per row: first / last row of its sequence's portion, slot, position
  const int* sh_last = nullptr;
  const int* sh_slots = nullptr;
  const int* sh_pos = nullptr;
  int sh_nslots = 0, sh_rows = 1;   // sh_rows: neighbouring rows of one group of threads
};

// One sequence's key range, masks and scales of a paged attention launch.
struct PagedAttnArgs {
  const void* qkv;     // rows [q H*DK | k G*DK | v G*DV | gate H ...], row stride ldq
  void* kp;            // key pages   [page][G][64][DK]
  void* vp;            // value pages [page][G][64][DV]
  const int* table;    // block table: page of (slot, position / 64); < 0: none
  const int* slots;    // per row: block-table row
  const int* pos;      // per row: position of the token
  void* out;           // [row][H*DV], row stride ldo
  int ldq, ldo, ldt, npages, M;
  int H, G, DK, DV;
  int gate;            // first column of the output gate logits in qkv, -1: none
  int window, keep;    // key j seen by query i: j <= i and (i - j < window or j < keep)
  float scale;
  // optional parts (zero: absent)
  const float* kscale = nullptr;  // [page][64]: factor of every key's scores (fp32, all heads)
  const float* slopes = nullptr;  // [H]: slope_h * (i - j) is taken off the scaled score
  int gate_el = 0;                // the gate has a column per head and value (H*DV) instead of one per head
  int shared = 0;                 // values are the keys: vp == kp, rows [q H*DK | k G*DK | ...]
  int written = 0;                // the cache already holds the rows' keys and values (paged_decode does not store them)
  const float* sinks = nullptr;   // [H]: a score per head that joins the softmax and has no value
};

// Query / key norm over whole projections, and the cache write of shared
// keys = values:  q <- q * rsqrt(mean(q^2) + eps) * qw * temp(pos) in place,
// page keys <- k as projected, kscale <- rsqrt(mean(k^2) + eps); qw holds the
// product of both norm weights.  temp = 1 + t_coef * ln(floor((pos + 1) / t_every) + 1).
struct QkNormArgs {
  void* qkv;
  void* kp;
  float* kscale;
  const float* qw;  // [H*DK]
  const int* table;
  const int* slots;
  const int* pos;
  int ldq, ldt, npages, M, H, G, DK, nq, nk;  // nq, nk: true widths of the projections
  int t_every;                                 // 0: no temperature
  float t_coef, eps;
};

// out = a N(z) + b N(z^2) + c N(z^3) + e in place, N(y) = y / sqrt(mean(y^2) + eps);
// rows of n values, zero up to the next 16 bytes.
struct PolyNormArgs {
  void* z;
  const float* w;  // {a, b, c, e}
  int ld, M, n;
  float eps;
};

// Rotation of pairs of values (neighbours, or i and i + pairs: the kernel's
// choice): freq[i] turns per position, cos and sin times mag.
struct RopeTable {
  const double* freq = nullptr;
  int pairs = 0;
  float mag = 1.f;
};

// Rows [q H*DK | k G*DK | v G*DV | ...]: every head of q and k is rotated (value
// i of a head with value i + rope.pairs, the rest pass) and divided by its root
// mean square over `dim` values; q in place, k and v into the cache pages.
struct QkHeadsArgs {
  void* qkv;
  void* kp;            // [page][G][64][DK]
  void* vp;            // [page][G][64][DV]
  const int* table;
  const int* slots;
  const int* pos;
  RopeTable rope;
  int ldq, ldt, npages, M, H, G, DK, DV, dim;
  float eps;
};

// Rows [query latent QP | latent CP | shared key part RP]: RMS norms of the two
// latents (true widths QN, CN) with weights qw, cw and rotation of the key part,
// in place; [latent | key part] goes into the cache [page][64][CP + RP].
struct LatentPrepArgs {
  void* rows;
  void* kp;
  const float* qw;
  const float* cw;
  const int* table;
  const int* slots;
  const int* pos;
  RopeTable rope;
  int ld, ldt, npages, M, QN, QP, CN, CP, RP;
  float eps;
};

// Causal attention of every head over latent cache rows; out = sum of latents.
struct LatentAttnArgs {
  const void* qlat;    // rows [H][CP], stride ldql
  const void* qrot;    // rows: head h at h * hs, RP columns, stride ldqr
  const void* kp;      // [page][64][CP + RP]
  const int* table;
  const int* slots;
  const int* pos;
  void* out;           // rows [H][CP], stride ldo
  const void* gate;    // rows [H] of gate logits, stride ldg (nullptr: none)
  int ldql, ldqr, hs, ldo, ldg, ldt, npages, M, H, CP, RP;
  float scale;
};

// The same attention over keys and values of every head, for portions whose
// sequences' cache rows were gathered and projected.
struct LatentKeysArgs {
  const void* q;       // rows [H][DP + RP], stride ldq
  const void* kv;      // key rows [H][DP | VP], stride ldkv
  const void* krot;    // key rows [RP], stride ldr
  const int* pos;
  void* out;           // rows [H][VP], stride ldo
  const void* gate;    // rows [H] of gate logits, stride ldg (nullptr: none)
  int ldq, ldkv, ldr, ldo, ldg, M, H, DP, RP, VP, keys;
  float scale;
};

extern "C" {
int dnn_poly_norm(const PolyNormArgs* a, int f32, hipStream_t st);
int dnn_rope_rows(void* x, int ld, int hs, int M, int H, int RP, const int* pos, const RopeTable* r, int f32,
                  hipStream_t st);
int dnn_latent_prep(const LatentPrepArgs* a, int f32, hipStream_t st);
int dnn_latent_attn(const LatentAttnArgs* a, const int* tiles, int ntiles, int rows, int splits, int per_token, float* ws,
                    long long ws_elems, hipStream_t st);  // rows: packed rows of a tile, 32 or 64
int dnn_latent_gather(const void* kp, int cols, const int* table, int ldt, int npages, const int* ent, int nent, void* out,
                      int rows, hipStream_t st);
int dnn_latent_prefill(const LatentKeysArgs* a, const int* tiles, int ntiles, hipStream_t st);
int dnn_latent_attn_f32(const LatentAttnArgs* a, hipStream_t st);
int dnn_rows_update(const RowsArgs* a, int y_f32, int out_f32, hipStream_t st);
// g = gelu_tanh(x W^T) * table[tok]: bf16, wsh = W in fragment order; _f32: from z = x W^T
int dnn_token_gate(const void* x, int ldx, const void* w, int ldw, const void* wsh, int K, const void* table, int ldt,
                   int off, const int* tok, int V, void* g, int ldg, int M, int n, int np, hipStream_t st);
int dnn_token_gate_f32(const float* z, int ldz, const float* table, int ldt, int off, const int* tok, int V, float* g,
                       int ldg, int M, int n, int np, hipStream_t st);
int dnn_qk_norm(const QkNormArgs* a, int f32, hipStream_t st);
int dnn_qk_heads(const QkHeadsArgs* a, int f32, hipStream_t st);
int dnn_xielu_f32(float* z, int ld, int M, int n, const float* c, hipStream_t st);  // in place
int dnn_glu_f32(const float* gu, int ldi, float* out, int ldo, int M, int F, int act, const GluClamp* clamp,
                hipStream_t st);
int dnn_gemm_f32(const float* A, int lda, const float* W, int ldw, float* C, int ldc, const float* bias, int M, int N,
                 int K, hipStream_t st);
int dnn_paged_write(const PagedAttnArgs* a, int f32, hipStream_t st);
int dnn_paged_prefill(const PagedAttnArgs* a, const int* tiles, int ntiles, hipStream_t st);
int dnn_paged_mixed(const PagedAttnArgs* a, const int* tiles, int ntiles, const int* rows, int nrows, int splits, float* ws,
                    long long ws_elems, hipStream_t st);
int dnn_paged_decode(const PagedAttnArgs* a, const int* rows, int nrows, int splits, float* ws, long long ws_elems,
                     hipStream_t st);
int dnn_paged_attn_f32(const PagedAttnArgs* a, hipStream_t st);
}
