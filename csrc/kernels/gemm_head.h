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
//   * the activations (all 64 rows, padded by clamping) go to LDS once per K
//     pass by LDS-DMA, 16-B slot j of row r at j ^ (r & 15) inside each 256-B
//     group (conflict-free fragment reads; swizzle applied on the source);
//   * 8 waves, each owning at most two 16-column tiles of the workgroup's
//     contiguous tile range (equal bytes per CU); a wave streams a tile's K range in groups of
//     GS chunks (1 KiB each) into two register buffers, the next group issued
//     before the current one is multiplied: up to 2 x GS KiB in flight per
//     wave, 8 x that per CU;
//   * the LayerNorm / RMSNorm statistics of the 64 rows come from the LDS
//     image (shifted by each row's first element, as gemm_skinny);
//   * epilogue per tile: channel scale (W8), folded norm, bias, bf16 round,
//     8-B stores, and the running argmax of the rounded values per row;
//     the 8 waves' winners meet in LDS and the workgroup writes one
//     {value bits, index} partial per row (ties -> smallest index).
// A longer K than the LDS image holds runs in passes (CPP chunks each): the
// image is restaged between passes and the accumulators stay in registers.
#pragma once
#include "gemm_stream.h"

namespace dnn {

template <bool W8, int NCH, int CPP, int GS>
struct HeadCfg {
  static constexpr int ACH = W8 ? 128 : 64;  // A bytes per row per 64-B weight chunk
  static constexpr int AU = W8 ? 2 : 1;      // A fragments (16 B) per chunk and m-tile
  static constexpr int NP = (NCH + CPP - 1) / CPP;
  static constexpr int KP = CPP * ACH;       // image row bytes (a multiple of 256)
  static constexpr int LDS = 64 * KP + (2 * 64 + 2 * 8 * 64) * 4;
  static_assert(KP % 256 == 0, "image rows are whole 256-B swizzle groups");
  static_assert(64 * KP % 1024 == 0, "whole LDS-DMA instructions");
};

template <bool W8, int NCH, int CPP, int GS>
constexpr int head_lds_bytes() {
  return HeadCfg<W8, NCH, CPP, GS>::LDS;
}

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
template <bool W8, int KP, int AU, int ACH, int GS>
__device__ __forceinline__ void head_mma(f32x4 (&acc)[4], const i32x4 (&buf)[GS], int n, int cl0, const char* img,
                                         int fr, int fg) {
#pragma unroll
  for (int j = 0; j < GS; ++j) {
    if (j < n) {  // wave-uniform
      bf16x8 af[4][AU];
#pragma unroll
      for (int t = 0; t < 4; ++t)
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
        for (int t = 0; t < 4; ++t) {
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wlo, af[t][0], acc[t], 0, 0, 0);
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(whi, af[t][AU - 1], acc[t], 0, 0, 0);
        }
      } else {
        bf16x8 wf;
        __builtin_memcpy(&wf, &buf[j], 16);
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, af[t][0], acc[t], 0, 0, 0);
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

// NORM: 0 none, 1 RMSNorm, 2 LayerNorm (folded; colsum for LN).
template <bool W8, int NORM, int NCH, int CPP, int GS>
__global__ __launch_bounds__(512, 1) void gemm_head_kernel(const uint8_t* __restrict__ A, int lda_b,
                                                           const uint8_t* __restrict__ Wsh,
                                                           const float* __restrict__ sw,
                                                           const float* __restrict__ colsum,
                                                           const float* __restrict__ bias, float eps,
                                                           bf16_t* __restrict__ C, int ldc, int M, int N, int kelems,
                                                           int2* __restrict__ part) {
  using Cfg = HeadCfg<W8, NCH, CPP, GS>;
  constexpr int ACH = Cfg::ACH, AU = Cfg::AU, NP = Cfg::NP, KP = Cfg::KP;
  constexpr int KPS = KP / 16;  // 16-B slots per image row
  extern __shared__ __attribute__((aligned(1024))) char hd_lds[];
  float* st_mean = reinterpret_cast<float*>(hd_lds + 64 * KP);
  float* st_rstd = st_mean + 64;
  float* xbest = st_rstd + 64;                          // [8 waves][64 rows]
  int* xidx = reinterpret_cast<int*>(xbest + 8 * 64);  // [8 waves][64 rows]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 15, fg = lane >> 4;
  const int ntile16 = (N + 15) >> 4;
  // the workgroup's contiguous tile range (12-13 of GPT-2's 3142 tiles on 256
  // CUs: every CU streams the same bytes), its waves round-robin inside it
  const int wt0 = (int)((long long)blockIdx.x * ntile16 / gridDim.x);
  const int wt1 = (int)((long long)(blockIdx.x + 1) * ntile16 / gridDim.x);
  const int tl[2] = {wt0 + wave, wt0 + wave + 8};
  const bool has0 = tl[0] < wt1;  // wave-uniform
  const bool has1 = tl[1] < wt1;
  const int kbA = kelems * 2;

  // statistics: wave w owns rows 8w..8w+7, 8 lanes per row
  const int srow = 8 * wave + (lane >> 3), ssub = lane & 7;
  float shift = 0.f, s1 = 0.f, s2 = 0.f;

  f32x4 acc[2][4];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[k][t] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int pc0 = p * CPP;
    const int pc1 = min(NCH, pc0 + CPP);
    const int npc = pc1 - pc0;
    const int ng = (npc + GS - 1) / GS;  // groups per tile in this pass (compile-time after unrolling)
    if (p > 0) __syncthreads();          // every wave is done reading the previous image
    // the activation image of this pass (64 rows x KP bytes) by LDS-DMA, then
    // the first two groups' weights; the barrier waits for the image only
    // (loads retire in issue order), the weights land under the statistics
#pragma unroll
    for (int q = wave; q < 64 * KP / 1024; q += 8) {
      const int o = q * 1024 + lane * 16;
      const int r = o / KP;
      const int sl = (o % KP) >> 4;
      const int s = sl ^ (r & 15);
      const int row = min(r, M - 1);
      const int kb = min(pc0 * ACH + s * 16, kbA - 16);
      glds16(A + (size_t)row * lda_b + kb, hd_lds + q * 1024);
    }
    i32x4 wa[GS], wb[GS];
    const int t0c = has0 ? tl[0] : ntile16 - 1;
    const int t1c = has1 ? tl[1] : t0c;
    // item i: tile i / ng, group i % ng
    const int nit = (has1 ? 2 : 1) * ng;
    head_wload<NCH, GS>(wa, Wsh, t0c, pc0, pc1, lane);
    if (nit > 1) {
      head_wload<NCH, GS>(wb, Wsh, ng > 1 ? t0c : t1c, pc0 + (ng > 1 ? GS : 0), pc1, lane);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * GS) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(GS) : "memory");
    }
    __syncthreads();

    // statistics of this pass's K range
    if constexpr (NORM != 0) {
      const char* rp = hd_lds + srow * KP;
      if constexpr (NORM == 2) {
        if (p == 0) shift = bf2f(*reinterpret_cast<const bf16_t*>(rp + ((0 ^ (srow & 15)) << 4)));
      }
#pragma unroll 4
      for (int sl = ssub; sl < KPS; sl += 8) {
        const int s = sl ^ (srow & 15);
        if (pc0 * ACH + s * 16 < kbA) {
          const bf16x8 x8 = *reinterpret_cast<const bf16x8*>(rp + sl * 16);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float x = bf2f_s(x8[i]) - shift;
            if constexpr (NORM == 2) s1 += x;
            s2 = fmaf(x, x, s2);
          }
        }
      }
    }

    // items, two register buffers: item i computes while item i + 1 lands
    for (int i = 0; i < nit; i += 2) {
      {
        const int k = i / ng, g = i % ng;
        const int c0 = g * GS, n = min(GS, npc - c0);
        if (k == 0)
          head_mma<W8, KP, AU, ACH, GS>(acc[0], wa, n, c0, hd_lds, fr, fg);
        else
          head_mma<W8, KP, AU, ACH, GS>(acc[1], wa, n, c0, hd_lds, fr, fg);
        if (i + 2 < nit) {
          const int k2 = (i + 2) / ng, g2 = (i + 2) % ng;
          head_wload<NCH, GS>(wa, Wsh, k2 ? t1c : t0c, pc0 + g2 * GS, pc1, lane);
        }
      }
      if (i + 1 < nit) {
        const int k = (i + 1) / ng, g = (i + 1) % ng;
        const int c0 = g * GS, n = min(GS, npc - c0);
        if (k == 0)
          head_mma<W8, KP, AU, ACH, GS>(acc[0], wb, n, c0, hd_lds, fr, fg);
        else
          head_mma<W8, KP, AU, ACH, GS>(acc[1], wb, n, c0, hd_lds, fr, fg);
        if (i + 3 < nit) {
          const int k3 = (i + 3) / ng, g3 = (i + 3) % ng;
          head_wload<NCH, GS>(wb, Wsh, k3 ? t1c : t0c, pc0 + g3 * GS, pc1, lane);
        }
      }
    }
  }

  // ---- row statistics -> LDS
  if constexpr (NORM != 0) {
    s1 = group_sum<8>(s1);
    s2 = group_sum<8>(s2);
    if (ssub == 0) {
      const float invk = 1.f / (float)kelems, d = s1 * invk;
      const float var = NORM == 2 ? fmaxf(s2 * invk - d * d, 0.f) : s2 * invk;
      st_mean[srow] = NORM == 2 ? shift + d : 0.f;
      st_rstd[srow] = rsqrtf(var + eps);
    }
    __syncthreads();
  }

  // ---- epilogue per tile + running argmax (lane: row 16 t + fr, columns n..n+3)
  float best[4];
  int bi[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    best[t] = -INFINITY;
    bi[t] = 0x7fffffff;
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (k == 0 ? !has0 : !has1) continue;  // wave-uniform
    const int n0 = tl[k] * 16 + fg * 4;
    float cs[4], bs[4], sc[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = n0 + r;
      const bool ok = n < N;
      cs[r] = (NORM == 2 && ok) ? colsum[n] : 0.f;
      bs[r] = (bias != nullptr && ok) ? bias[n] : 0.f;
      sc[r] = (W8 && ok) ? sw[n] : 1.f;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
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
        float v = acc[k][t][r];
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
  // ---- winners: the 4 lane groups, then the 8 waves, then one partial per row
#pragma unroll
  for (int t = 0; t < 4; ++t) {
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
      const float ov = __shfl_xor(best[t], o, 64);
      const int oi = __shfl_xor(bi[t], o, 64);
      head_amax(best[t], bi[t], ov, oi);
    }
    if (lane < 16) {
      xbest[wave * 64 + 16 * t + lane] = best[t];
      xidx[wave * 64 + 16 * t + lane] = bi[t];
    }
  }
  __syncthreads();
  if (tid < 64 && tid < M) {
    float b = xbest[tid];
    int i = xidx[tid];
#pragma unroll
    for (int w = 1; w < 8; ++w) head_amax(b, i, xbest[w * 64 + tid], xidx[w * 64 + tid]);
    part[(size_t)tid * gridDim.x + blockIdx.x] = make_int2(__float_as_int(b), i);
  }
}

}  // namespace dnn
