// A block of a decode step of one or two rows in four launches: partial products
// instead of finished ones between them (LayerNorm folded into the projections,
// heads of 64, bf16).
//
//   q | k | v   the rows (residual + bias + four partials of the block before),
//               their statistics, the product
//   attention   a head's output times the 64 columns of W_o that read it: one
//               partial a head (attention_stream.h, PROJ)
//   c_fc        residual + bias + a partial a head, statistics, product, GELU
//   c_proj      four slices of K, four partials
//
// Such a step is a chain of launches of 3 to 6 us whatever they read: what one of them
// costs is its start, a round trip for its rows, one for its weights and a short
// reduction.  So a launch less (the attention's projection: 3.2 us) and slices of K for
// the longest one (c_proj: 96 chunks on 48 workgroups, 5.7) pay for partials that
// every workgroup behind adds up once more (12 to 36 KB from the L2 a row).  And a launch
// begins with a cold instruction cache: these kernels are 0.8 to 2.5 KB straight through,
// with every size a template argument, where the general ones are 4 KB of it and 1.3 us
// slower in a step (not by themselves).
//
// GPT-2, 12 blocks and the head, graph, us of the separate launches : this: one row behind 100 tokens 268 :
// 186, behind 900 313 : 225; two rows 275 : 209, 318 : 242.  A row more is 20 us of partials: three
// would take 230 (separate 280), four 255.  us a block, one row behind 100 and 1000 tokens, two rows behind both:
// width 256 17.1 : 12.2, 20.6 : 15.0, 18.1 : 13.4, 20.8 : 16.0; 768 18.1 : 13.8, 20.7 : 17.4, 18.1 : 15.7, 20.8 : 18.8; 1024
// 22.4 : 16.1, 26.2 : 19.1, 22.5 : 17.5, 26.5 : 20.4.
//
// The rows are rounded to bf16 where the separate launches store them, sums are fp32.
#include "attention_row.h"
#include "common.h"
#include "gemm_epilogue.h"

namespace dnn {

constexpr int RP_SLICES = 4;  // partials of c_proj

struct RowProj {
  const bf16_t* x;      // (M, K) rows: the residual; without PRO the operand, its slices side by side
  const float* parts;   // PRO: [NP][M][K]
  const float* pbias;   // of the product that the partials are of
  bf16_t* h;            // PRO: the rows with their partials, one workgroup writes them
  const uint8_t* w;     // fragment order (ops/gemm.py shuffle_weight)
  const float *colsum, *bias;
  void* out;            // PRO: bf16 (M, N), else partials [slice][M][N]
  float eps;
  int M, N;
};

// mean and sum of squared deviations of two sets of n values each
__device__ __forceinline__ void rp_merge(float& mean, float& m2, float mo, float qo, float n) {
  const float d = mo - mean;
  mean = 0.5f * (mean + mo);
  m2 = m2 + qo + d * d * (0.5f * n);
}

// One workgroup per 16 columns (and slice): 4 waves of CH chunks of 32 k, the lower and the
// upper half of a wave's chunks in sums of their own.  MR rows.
template <int CH, int NP, int MR, bool PRO, int ACT>
__global__ __launch_bounds__(256) void row_proj_kernel(RowProj p) {
  constexpr int K = CH * 128;  // of this workgroup
  constexpr int XW = PRO ? K / 256 : 1;
  static_assert(!PRO || (K % 256 == 0 && K <= 1024), "whole waves, four values a thread");
  __shared__ __attribute__((aligned(16))) bf16_t xs[PRO ? MR : 1][PRO ? K : 8];
  __shared__ float2 st[MR][XW];
  __shared__ f32x4 red[8][4 * MR];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slice = blockIdx.y, c4 = lane >> 4, mrow = min(lane & 15, MR - 1);
  const i32x4* wp = reinterpret_cast<const i32x4*>(p.w) +
                    ((size_t)blockIdx.x * (CH * 4 * gridDim.y) + slice * CH * 4 + wave * CH) * 64 + lane;
  f32x4 part[PRO && NP ? NP : 1][MR], pb = {0.f, 0.f, 0.f, 0.f};
  bf16x4 xr[MR];
  i32x4 wv[CH], av[CH];
  const int k = min(tid * 4, K - 4);
  if constexpr (PRO) {  // the rows' operands are asked for first: they come from the L2, the weights from memory
#pragma unroll
    for (int m = 0; m < MR; ++m) {
#pragma unroll
      for (int i = 0; i < NP; ++i)
        part[i][m] = *reinterpret_cast<const f32x4*>(p.parts + ((size_t)i * p.M + min(m, p.M - 1)) * K + k);
      xr[m] = *reinterpret_cast<const bf16x4*>(p.x + (size_t)min(m, p.M - 1) * K + k);
    }
    if (NP) pb = *reinterpret_cast<const f32x4*>(p.pbias + k);
  } else {
    const bf16_t* xp = p.x + (size_t)min(mrow, p.M - 1) * K * gridDim.y + slice * K + wave * CH * 32 + c4 * 8;
#pragma unroll
    for (int u = 0; u < CH; ++u) av[u] = *reinterpret_cast<const i32x4*>(xp + u * 32);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < CH; ++u) wv[u] = __builtin_nontemporal_load(wp + u * 64);
  const int n = blockIdx.x * 16 + c4 * 4;
  f32x4 cs, bs;
  if constexpr (PRO) {
    cs = *reinterpret_cast<const f32x4*>(p.colsum + n);
    bs = *reinterpret_cast<const f32x4*>(p.bias + n);
  }
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (PRO) {
    if (wave < XW) {
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NP; ++i) v = i == 0 ? part[0][m] : v + part[i][m];
        bf16x4 o = xr[m];
        if constexpr (NP > 0) {
          v += pb;
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = (short)f2bf(v[j] + bf2f_s(xr[m][j]));
        }
        *reinterpret_cast<bf16x4*>(&xs[m][k]) = o;
        if (blockIdx.x == 0 && m < p.M) *reinterpret_cast<bf16x4*>(p.h + (size_t)m * K + k) = o;
        float e[4], s = 0.f, q = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) s += e[j] = bf2f_s(o[j]);
        float mean = 0.25f * s;
#pragma unroll
        for (int j = 0; j < 4; ++j) q = fmaf(e[j] - mean, e[j] - mean, q);
        rp_merge(mean, q, dpp_f<0xB1>(mean), dpp_f<0xB1>(q), 4.f);
        rp_merge(mean, q, dpp_f<0x4E>(mean), dpp_f<0x4E>(q), 8.f);
        rp_merge(mean, q, dpp_f<0x141>(mean), dpp_f<0x141>(q), 16.f);
        rp_merge(mean, q, dpp_f<0x140>(mean), dpp_f<0x140>(q), 32.f);
        f32x2 a = lanes16(mean), b = lanes16(q);
        mean = a[0], q = b[0];
        rp_merge(mean, q, a[1], b[1], 64.f);
        a = lanes32(mean), b = lanes32(q);
        mean = a[0], q = b[0];
        rp_merge(mean, q, a[1], b[1], 128.f);
        if (lane == 0) st[m][wave] = float2{mean, q};
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < CH; ++u) av[u] = *reinterpret_cast<const i32x4*>(&xs[mrow][(wave * CH + u) * 32 + c4 * 8]);
  }
  f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int u = 0; u < CH; ++u)
    acc[u / (CH / 2)] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[u]),
                                                                __builtin_bit_cast(bf16x8, av[u]), acc[u / (CH / 2)], 0, 0, 0);
  if ((lane & 15) < MR) {
    red[wave * 2][c4 * MR + mrow] = acc[0];
    red[wave * 2 + 1][c4 * MR + mrow] = acc[1];
  }
  __syncthreads();
  if (wave != 0 || (lane & 15) >= p.M) return;
  f32x4 r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = red[i][c4 * MR + mrow];
#pragma unroll
  for (int i = 1; i < 8; ++i) r[0] += r[i];
  if constexpr (!PRO) {
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.out) + ((size_t)slice * p.M + mrow) * p.N + n) = r[0];
  } else {
    float mean = 0.f, m2 = 0.f;
#pragma unroll
    for (int i = 0; i < XW; ++i) mean += st[mrow][i].x;
    mean *= 1.f / XW;
#pragma unroll
    for (int i = 0; i < XW; ++i) m2 += fmaf(256.f * (st[mrow][i].x - mean), st[mrow][i].x - mean, st[mrow][i].y);
    const float rstd = rsqrtf(m2 * (1.f / K) + p.eps);
    f32x4 y = rstd * (r[0] - mean * cs) + bs;
    if constexpr (ACT == ACT_GELU) {
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = gelu_erf(y[j]);
    }
    *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(p.out) + (size_t)mrow * p.N + n) =
        make_uint2(pack2bf(y[0], y[1]), pack2bf(y[2], y[3]));
  }
}

}  // namespace dnn

using namespace dnn;

// Widths whose heads and chunks the kernels are laid out for.
static int row_chunks(int d) { return d == 256 ? 2 : d == 768 ? 6 : d == 1024 ? 8 : 0; }

template <int CH, int MR>
static void row_launch(const RowProj& p, int np, bool gelu, hipStream_t st) {
  constexpr int H = CH * 2;  // heads of 64
  const dim3 grid(p.N / 16);
  if (gelu)
    hipLaunchKernelGGL((row_proj_kernel<CH, H, MR, true, ACT_GELU>), grid, dim3(256), 0, st, p);
  else if (np)
    hipLaunchKernelGGL((row_proj_kernel<CH, RP_SLICES, MR, true, ACT_NONE>), grid, dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((row_proj_kernel<CH, 0, MR, true, ACT_NONE>), grid, dim3(256), 0, st, p);
}
template <int MR>
static void row_launch_d(int ch, const RowProj& p, int np, bool gelu, hipStream_t st) {
  if (ch == 2) row_launch<2, MR>(p, np, gelu, st);
  else if (ch == 6) row_launch<6, MR>(p, np, gelu, st);
  else row_launch<8, MR>(p, np, gelu, st);
}
template <int MR>
static void row_slices_d(int ch, const RowProj& p, hipStream_t st) {
  const dim3 grid(p.N / 16, RP_SLICES);
  if (ch == 2) hipLaunchKernelGGL((row_proj_kernel<2, 0, MR, false, ACT_NONE>), grid, dim3(256), 0, st, p);
  else if (ch == 6) hipLaunchKernelGGL((row_proj_kernel<6, 0, MR, false, ACT_NONE>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((row_proj_kernel<8, 0, MR, false, ACT_NONE>), grid, dim3(256), 0, st, p);
}

// fp32 elements of `parts` that a step of M rows of width d uses, 0: not a step for these kernels.
// Caches below 2048 keys: from there on the separate attention splits a head's keys over workgroups, this one never, and
// each of a head's H / 2 groups of columns reads them again: 3.0 us more a block for 1000 keys more where the split one
// pays 0.7 (width 768, one row, a cache of 2047 keys behind 2000 tokens 20.5, the split one of 4096 21.4 there and 22.7
// behind 4000).  The cache's size is what the host knows.
extern "C" long long dnn_decode_row_parts(int M, int d, int H, int Hkv, int hd, int S) {
  if (M < 1 || M > DECODE_ROWS || row_chunks(d) == 0 || hd != 64 || H * hd != d || H != Hkv || S < 1 || S >= 2048) return 0;
  return (long long)M * d * (H + RP_SLICES);
}

// The blocks of a step of M rows (one token of each sequence) but for the last c_proj: x (M, d) in; f (M, 4 d) and the
// residual h of the last block out.  a: rows of scratch; parts: dnn_decode_row_parts.  K and V caches of the first block,
// kv_block bytes apart.  -3, nothing launched: not these sizes.
extern "C" int dnn_decode_row_blocks(const RowBlock* blocks, int n, const void* x, void* a, void* h, void* qkv, void* f,
                                     float* parts, char* kc, char* vc, long long kv_block, int M, int d, int H, int Hkv,
                                     int hd, int S, const int* pos, float scale, float eps, hipStream_t st) {
  const int ch = row_chunks(d);
  if (n < 1 || dnn_decode_row_parts(M, d, H, Hkv, hd, S) == 0) return -3;
  float* const p_att = parts;                          // [H][M][d]
  float* const p_out = parts + (size_t)M * d * H;      // [RP_SLICES][M][d]
  const bool one = M == 1;
  for (int i = 0; i < n; ++i) {
    const RowBlock& L = blocks[i];
    RowProj q = {(const bf16_t*)(i ? h : x), p_out, i ? blocks[i - 1].b_down : nullptr, (bf16_t*)a, (const uint8_t*)L.w_qkv,
                 L.cs_qkv, L.b_qkv, qkv, eps, M, 3 * d};
    one ? row_launch_d<1>(ch, q, i, false, st) : row_launch_d<2>(ch, q, i, false, st);
    const int rc = dnn_attn_decode_proj(qkv, 3 * d, kc + i * kv_block, vc + i * kv_block, L.w_o, p_att, M, H, S, pos, scale, st);
    if (rc) return rc;
    RowProj u = {(const bf16_t*)a, p_att, L.b_o, (bf16_t*)h, (const uint8_t*)L.w_up, L.cs_up, L.b_up, f, eps, M, 4 * d};
    one ? row_launch_d<1>(ch, u, H, true, st) : row_launch_d<2>(ch, u, H, true, st);
    if (i + 1 == n) break;
    RowProj o = {(const bf16_t*)f, nullptr, nullptr, nullptr, (const uint8_t*)L.w_down, nullptr, nullptr, p_out, 0.f, M, d};
    one ? row_slices_d<1>(ch, o, st) : row_slices_d<2>(ch, o, st);
  }
  return (int)hipGetLastError();
}
