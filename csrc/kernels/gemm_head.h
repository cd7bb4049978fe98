// Decode vocabulary head with the greedy argmax's first pass ("head" kernel,
// the tied 50304-wide head toward its byte floor).
//
//   logits[m, n] = bf16( rstd[m] (A[m,:] . W'[n,:] - mean[m] colsum[n]) + bias'[n] )
//   part[m, wg]  = argmax over this workgroup's columns of logits[m, :]
//
// (ln_f folded into W' on the host, ops/gemm.py fold_norm; bf16 or OCP e4m3
// W8A16 weights in fragment order, ops/gemm.py shuffle_weight.)  The argmax
// of every row is then one small merge over the workgroups' partials
// (sampler.hip argmax_final_kernel) instead of a second pass over the
// 64 x 50304 logits.
//
// Why a separate kernel.  At 64 rows and K = 768 a column tile's weights
// (24 KiB) are as many bytes as the activations it multiplies (96 KiB shared
// by every tile): gemm_skinny re-reads the activations from L2 once per
// workgroup of 4 column tiles and each wave waits a round trip per 2-chunk
// batch — 26 us for 77 MB (2.9 TB/s).  Here a persistent workgroup per CU
// keeps the activation rows in LDS for all of its column tiles:
//   * the activations (16 or 64 rows, padded by clamping) go to LDS once per K
//     pass by LDS-DMA, 16-B slot j of row r at j ^ (r & 15) inside each 256-B
//     group (conflict-free fragment reads; swizzle applied on the source);
//   * a wave for each 16-column tile of the workgroup's contiguous tile range
//     (equal bytes per CU, at most 16 tiles); a wave streams its tile's K range in groups of
//     GS chunks (1 KiB each) into two register buffers, the next group issued
//     before the current one is multiplied: up to 2 x GS KiB in flight per
//     wave, 100 to 200 KiB per CU.  With 8 waves and 12 or 13 tiles five waves had two
//     tiles and three had one, and the workgroup took as long as two;
//   * what the epilogue reads by column (scales, column sums, bias) is loaded first of all: behind
//     the products it was a trip to memory that nothing hid;
//   * up to 16 rows there is one row tile: a quarter of the image, of its reads and of the products;
//   * the LayerNorm / RMSNorm statistics of the rows come from the LDS
//     image (shifted by each row's first element, as gemm_skinny);
//   * epilogue per tile: channel scale (W8), folded norm, bias, bf16 round,
//     8-B stores, and the argmax of the rounded values per row;
//     the waves' winners meet in LDS and the workgroup writes one
//     {value bits, index} partial per row (ties -> smallest index).
// A longer K than the LDS image holds runs in passes (CPP chunks each): the
// image is restaged between passes and the accumulators stay in registers.
//
// us with the merge of the partials behind it, 8 waves of up to two tiles : this (the bytes at 4.77 TB/s: 16.2,
// 33.7, 16.9), 50257 columns, 1 and 64 rows: K = 768 24.1 : 19.5, 27.1 : 25.2; 1600 40.3 : 33.0, 44.2 : 40.1; 1600 in
// e4m3 33.0 : 20.4, 36.3 : 33.1.  Above 16 rows the image, statistics and epilogue of 64 rows (4 to 5 us) stay.
#pragma once
#include "gemm_stream.h"

namespace dnn {

constexpr int HEAD_WAVES = 16;  // at most, a wave a tile

template <bool W8, int MT, int NCH, int CPP, int GS>
struct HeadCfg {
  static constexpr int ACH = W8 ? 128 : 64;  // A bytes per row per 64-B weight chunk
  static constexpr int AU = W8 ? 2 : 1;      // A fragments (16 B) per chunk and m-tile
  static constexpr int NP = (NCH + CPP - 1) / CPP;
  static constexpr int KP = CPP * ACH;       // image row bytes (a multiple of 256)
  static constexpr int ROWS = MT * 16;
  static constexpr int LDS = ROWS * KP + (2 * ROWS + 2 * HEAD_WAVES * ROWS) * 4;
  static_assert(KP % 256 == 0, "image rows are whole 256-B swizzle groups");
  static_assert(ROWS * KP % 1024 == 0, "whole LDS-DMA instructions");
};

// one group of GS weight chunks [c0, c0 + GS) of column tile `tile` (chunks
// past c1 clamp to c1 - 1: loaded, never multiplied)
template <int NCH, int GS>
__device__ __forceinline__ void head_wload(i32x4 (&buf)[GS], const uint8_t* __restrict__ Wsh, int tile, int c0, int c1,
                                           int lane) {
  const uint8_t* wp = Wsh + (size_t)tile * NCH * 1024 + lane * 16;
#pragma unroll
  for (int j = 0; j < GS; ++j) {
    const int cc = min(c0 + j, c1 - 1);
    buf[j] = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(wp + (size_t)cc * 1024));
  }
}

// MFMAs of `n` chunks (local chunk index cl0..) of one group against the image
template <bool W8, int MT, int KP, int AU, int ACH, int GS>
__device__ __forceinline__ void head_mma(f32x4 (&acc)[MT], const i32x4 (&buf)[GS], int n, int cl0, const char* img,
                                         int fr, int fg) {
#pragma unroll
  for (int j = 0; j < GS; ++j) {
    if (j < n) {  // wave-uniform
      bf16x8 af[MT][AU];
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int h = 0; h < AU; ++h) {
          const int row = 16 * t + fr;
          const int slot = ((cl0 + j) * ACH + fg * (ACH / 4) + 16 * h) >> 4;
          af[t][h] = *reinterpret_cast<const bf16x8*>(img + row * KP + ((slot ^ (row & 15)) << 4));
        }
      if constexpr (W8) {
        bf16x8 wlo, whi;
        bf16x2v o[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          o[2 * i] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((uint32_t)buf[j][i], 1.0f, false);
          o[2 * i + 1] = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((uint32_t)buf[j][i], 1.0f, true);
        }
        __builtin_memcpy(&wlo, &o[0], 16);
        __builtin_memcpy(&whi, &o[4], 16);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wlo, af[t][0], acc[t], 0, 0, 0);
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(whi, af[t][AU - 1], acc[t], 0, 0, 0);
        }
      } else {
        bf16x8 wf;
        __builtin_memcpy(&wf, &buf[j], 16);
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, af[t][0], acc[t], 0, 0, 0);
      }
    }
    // one chunk's fragments at a time: hoisting every chunk's LDS reads of the
    // group ahead of its MFMAs would need 4 x AU x 4 VGPRs per chunk and spill
    __builtin_amdgcn_sched_barrier(0);
  }
}

__device__ __forceinline__ void head_amax(float& best, int& bi, float v, int i) {
  if (v > best || (v == best && i < bi)) {
    best = v;
    bi = i;
  }
}

// NORM: 0 none, 1 RMSNorm, 2 LayerNorm (folded; colsum for LN).  MT: row tiles of 16, 1 or 4.
template <bool W8, int NORM, int NCH, int CPP, int GS, int MT = 4>
__global__ __launch_bounds__(HEAD_WAVES * 64, 1) void gemm_head_kernel(const uint8_t* __restrict__ A, int lda_b,
                                                           const uint8_t* __restrict__ Wsh,
                                                           const float* __restrict__ sw,
                                                           const float* __restrict__ colsum,
                                                           const float* __restrict__ bias, float eps,
                                                           bf16_t* __restrict__ C, int ldc, int M, int N, int kelems,
                                                           int2* __restrict__ part) {
  using Cfg = HeadCfg<W8, MT, NCH, CPP, GS>;
  constexpr int ROWS = Cfg::ROWS;
  constexpr int ACH = Cfg::ACH, AU = Cfg::AU, NP = Cfg::NP, KP = Cfg::KP;
  constexpr int KPS = KP / 16;  // 16-B slots per image row
  extern __shared__ __attribute__((aligned(1024))) char hd_lds[];
  float* st_mean = reinterpret_cast<float*>(hd_lds + ROWS * KP);
  float* st_rstd = st_mean + ROWS;
  float* xbest = st_rstd + ROWS;                                  // [waves][rows]
  int* xidx = reinterpret_cast<int*>(xbest + HEAD_WAVES * ROWS);  // [waves][rows]

  const int tid = threadIdx.x, lane = tid & 63, nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fg = lane >> 4;
  const int ntile16 = (N + 15) >> 4;
  // the workgroup's contiguous tile range (12-13 of GPT-2's 3142 tiles on 256
  // CUs: every CU streams the same bytes), a wave each (host: nw >= wt1 - wt0)
  const int wt0 = (int)((long long)blockIdx.x * ntile16 / gridDim.x);
  const int wt1 = (int)((long long)(blockIdx.x + 1) * ntile16 / gridDim.x);
  const bool has = wt0 + wave < wt1;  // wave-uniform; a wave without a tile reads the first one's lines and drops them
  const int tile = has ? wt0 + wave : wt0;
  const int kbA = kelems * 2;

  // the epilogue's operands (absent ones read a valid address, ``pre`` decides their use)
  const int n0 = tile * 16 + fg * 4, nn = min(n0, (N - 4) & ~3);  // host: N >= 16
  const bool vec = ((reinterpret_cast<uintptr_t>(sw) | reinterpret_cast<uintptr_t>(colsum) |
                     reinterpret_cast<uintptr_t>(bias)) & 15) == 0;
  const bool pre = vec && n0 + 3 < N;
  const float* dummy = reinterpret_cast<const float*>(A);
  f32x4 cs = f32x4{0.f, 0.f, 0.f, 0.f}, bs = cs, sc = cs;
  if constexpr (NORM == 2) cs = *reinterpret_cast<const f32x4*>(vec ? colsum + nn : dummy);
  bs = *reinterpret_cast<const f32x4*>(vec && bias != nullptr ? bias + nn : dummy);
  if constexpr (W8) sc = *reinterpret_cast<const f32x4*>(vec ? sw + nn : dummy);
  __builtin_amdgcn_sched_barrier(0);

  // statistics: wave w < 2 MT owns rows 8w..8w+7, 8 lanes per row (host: nw >= 2 MT)
  const int srow = 8 * wave + (lane >> 3), ssub = lane & 7;
  const bool stats = NORM != 0 && wave < 2 * MT;
  float shift = 0.f, s1 = 0.f, s2 = 0.f;

  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int pc0 = p * CPP;
    const int pc1 = min(NCH, pc0 + CPP);
    const int npc = pc1 - pc0;
    const int ng = (npc + GS - 1) / GS;  // groups per tile in this pass (compile-time after unrolling)
    // the first group's weights, the activation image of this pass (ROWS x KP bytes) by LDS-DMA, the second
    // group: the weights' stream goes on while the waves meet and the image lands
    i32x4 wa[GS], wb[GS];
    head_wload<NCH, GS>(wa, Wsh, tile, pc0, pc1, lane);
    if (p > 0) __syncthreads();  // every wave is done reading the previous image
    for (int q = wave; q < ROWS * KP / 1024; q += nw) {
      const int o = q * 1024 + lane * 16;
      const int r = o / KP;
      const int sl = (o % KP) >> 4;
      const int s = sl ^ (r & 15);
      const int row = min(r, M - 1);
      const int kb = min(pc0 * ACH + s * 16, kbA - 16);
      glds16(A + (size_t)row * lda_b + kb, hd_lds + q * 1024);
    }
    if (ng > 1) head_wload<NCH, GS>(wb, Wsh, tile, pc0 + GS, pc1, lane);
    __syncthreads();  // waits for all of them: an LDS-DMA is not ordered with plain loads behind it

    // statistics of this pass's K range
    if (stats) {
      const char* rp = hd_lds + srow * KP;
      if constexpr (NORM == 2) {
        if (p == 0) shift = bf2f(*reinterpret_cast<const bf16_t*>(rp + ((0 ^ (srow & 15)) << 4)));
      }
#pragma unroll 4
      for (int i = 0; i < KPS / 8; ++i) {  // KPS / 8 is even; odd rows half a 256-B group on: no bank twice
        const int sl = (i ^ (srow & 1)) * 8 + ssub, s = sl ^ (srow & 15);
        if (pc0 * ACH + s * 16 < kbA) {
          const bf16x8 x8 = *reinterpret_cast<const bf16x8*>(rp + sl * 16);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float x = bf2f_s(x8[e]) - shift;
            if constexpr (NORM == 2) s1 += x;
            s2 = fmaf(x, x, s2);
          }
        }
      }
    }

    // two register buffers: a group computes while the next one lands
    for (int g = 0; g < ng; g += 2) {
      head_mma<W8, MT, KP, AU, ACH, GS>(acc, wa, min(GS, npc - g * GS), g * GS, hd_lds, fr, fg);
      if (g + 2 < ng) head_wload<NCH, GS>(wa, Wsh, tile, pc0 + (g + 2) * GS, pc1, lane);
      if (g + 1 < ng) {
        head_mma<W8, MT, KP, AU, ACH, GS>(acc, wb, min(GS, npc - (g + 1) * GS), (g + 1) * GS, hd_lds, fr, fg);
        if (g + 3 < ng) head_wload<NCH, GS>(wb, Wsh, tile, pc0 + (g + 3) * GS, pc1, lane);
      }
    }
  }

  // ---- row statistics -> LDS
  if constexpr (NORM != 0) {
    s1 = group_sum<8>(s1);
    s2 = group_sum<8>(s2);
    if (stats && ssub == 0) {
      const float invk = 1.f / (float)kelems, d = s1 * invk;
      const float var = NORM == 2 ? fmaxf(s2 * invk - d * d, 0.f) : s2 * invk;
      st_mean[srow] = NORM == 2 ? shift + d : 0.f;
      st_rstd[srow] = rsqrtf(var + eps);
    }
    __syncthreads();
  }

  // ---- epilogue + argmax (lane: row 16 t + fr, columns n0..n0+3)
  float best[MT];
  int bi[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    best[t] = -INFINITY;
    bi[t] = 0x7fffffff;
  }
  if (has) {
    if (!pre) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool ok = n0 + r < N;
        cs[r] = (NORM == 2 && ok) ? colsum[n0 + r] : 0.f;
        bs[r] = (bias != nullptr && ok) ? bias[n0 + r] : 0.f;
        sc[r] = (W8 && ok) ? sw[n0 + r] : 1.f;
      }
    } else if (bias == nullptr) {
      bs = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = 16 * t + fr;
      float mean = 0.f, rstd = 1.f;
      if constexpr (NORM != 0) {
        mean = st_mean[m];
        rstd = st_rstd[m];
      }
      uint32_t pk[2];
      float rv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[t][r];
        if constexpr (W8) v *= sc[r];
        if constexpr (NORM == 2) v = rstd * (v - mean * cs[r]);
        if constexpr (NORM == 1) v *= rstd;
        v += bs[r];
        const bf16_t b = f2bf(v);
        rv[r] = bf2f(b);
        if (r & 1)
          pk[r >> 1] |= (uint32_t)b << 16;
        else
          pk[r >> 1] = (uint32_t)b;
      }
      if (m < M) {
        bf16_t* cp = C + (size_t)m * ldc + n0;
        if (n0 + 3 < N) {
          *reinterpret_cast<uint2*>(cp) = make_uint2(pk[0], pk[1]);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n0 + r < N) cp[r] = (bf16_t)((pk[r >> 1] >> (16 * (r & 1))) & 0xffff);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n0 + r < N) head_amax(best[t], bi[t], rv[r], n0 + r);
      }
    }
  }
  // ---- winners: the 4 lane groups, then the waves, then one partial per row
#pragma unroll
  for (int t = 0; t < MT; ++t) {
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
      const float ov = __shfl_xor(best[t], o, 64);
      const int oi = __shfl_xor(bi[t], o, 64);
      head_amax(best[t], bi[t], ov, oi);
    }
    if (lane < 16) {
      xbest[wave * ROWS + 16 * t + lane] = best[t];
      xidx[wave * ROWS + 16 * t + lane] = bi[t];
    }
  }
  __syncthreads();
  if (tid < ROWS && tid < M) {
    float b = xbest[tid];
    int i = xidx[tid];
    for (int w = 1; w < nw; ++w) head_amax(b, i, xbest[w * ROWS + tid], xidx[w * ROWS + tid]);
    part[(size_t)tid * gridDim.x + blockIdx.x] = make_int2(__float_as_int(b), i);
  }
}

}  // namespace dnn
