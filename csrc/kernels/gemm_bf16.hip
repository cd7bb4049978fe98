// bf16 GEMM on CDNA4 MFMA with fused epilogues.
//
//   C[M,N] = act(A[M,K] . W[N,K]^T + bias[N]) (+ residual[M,N])
//
// W is the nn.Linear layout [out, in], so both operands are K-contiguous and
// every MFMA fragment is one 16-byte LDS read. Replaces the implicit torch ops
// of the reference's stage forwards: CIFAR fc1 (cifar_model_parts.py:13,55),
// nanoGPT c_attn / c_proj / c_fc / lm_head (partitions/gpt_model_parts.py:20-21,
// 32-33,46-49) and the Llama projections.
//
// Decode-sized M (<= 64) goes to the weight-streaming kernels of gemm_skinny.hip,
// row counts between that and a full chip of 256 x 256 tiles (gemm_tile.h) to the
// smaller tiles of gemm_mid.h.  Operands are staged global->LDS with 16-byte
// global_load_lds into buffers whose 128-B rows are XOR-swizzled on the SOURCE
// address (chunk ^= (row>>1)&7), which makes the ds_read_b128 fragment reads
// conflict-free.  Block ids are remapped so tiles sharing A panels run on one XCD.
#include <type_traits>

#include "api.h"
#include "gemm_epilogue.h"
#include "gemm_mid_api.h"
#include "gemm_mid_fp8.h"
#include "gemm_tile.h"

namespace dnn {

// ---------------------------------------------------------------------------
// fp8 (OCP e4m3fn) on the same 256^2 4-phase schedule: a K-tile is 128 fp8 =
// 128 B per row, so every LDS half-tile, glds piece and swizzle is
// byte-identical to the bf16 kernel's BK = 64 and the staging code is shared.
// Per (i, j) and K-tile ONE v_mfma_scale_f32_16x16x128_f8f6f4 (unit E8M0 block
// scales, 2x the bf16 rate) replaces the two bf16 16x16x32: lane group g feeds
// chunks g and 4+g of its row as its 32 "k" bytes — the same permutation of k
// for both operands, so the dot product is unchanged and the fragment reads are
// exactly the bf16 kernel's (conflict-free) ones.  Epilogue: per-token scale
// sa[m] and per-channel scale sw[n] on the fp32 accumulators, then the shared
// bias / act / residual / SwiGLU epilogues (16-B paired stores).
// ---------------------------------------------------------------------------
typedef int i32x8_t __attribute__((ext_vector_type(8)));

__device__ __forceinline__ i32x8_t f8_cat(const bf16x8& lo, const bf16x8& hi) {
  i32x8_t r;
  const i32x4 a = __builtin_bit_cast(i32x4, lo), b = __builtin_bit_cast(i32x4, hi);
  r[0] = a[0]; r[1] = a[1]; r[2] = a[2]; r[3] = a[3];
  r[4] = b[0]; r[5] = b[1]; r[6] = b[2]; r[7] = b[3];
  return r;
}

template <int MI, int NJ, bool WAIT = true>
__device__ __forceinline__ void bg_mfma_f8(f32x4 (&acc)[MI][NJ], const bf16x8 (&a)[MI][2], const bf16x8 (&b)[NJ][2]) {
  if constexpr (WAIT) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_setprio(1);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(f8_cat(b[j][0], b[j][1]), f8_cat(a[i][0], a[i][1]),
                                                                   acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
  __builtin_amdgcn_s_setprio(0);
}

// MX e8m0 scales of the activations on the scaled MFMA (MXA, common.h
// mx_index: one dword per lane per 128-row half-tile and K-tile, byte i =
// fragment i): acc carries the activation scales, the epilogue only the
// weight channel scale.
template <int MI, int NJ, bool WAIT = true>
__device__ __forceinline__ void bg_mfma_f8x(f32x4 (&acc)[MI][NJ], const bf16x8 (&a)[MI][2], const bf16x8 (&b)[NJ][2],
                                            uint32_t s) {
  static_assert(MI == 4, "one op_sel byte per A fragment");
  if constexpr (WAIT) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_setprio(1);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const i32x8_t bj = f8_cat(b[j][0], b[j][1]);
    acc[0][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bj, f8_cat(a[0][0], a[0][1]), acc[0][j], 0, 0, 0,
                                                                 0x7f7f7f7f, 0, s);
    acc[1][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bj, f8_cat(a[1][0], a[1][1]), acc[1][j], 0, 0, 0,
                                                                 0x7f7f7f7f, 1, s);
    acc[2][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bj, f8_cat(a[2][0], a[2][1]), acc[2][j], 0, 0, 0,
                                                                 0x7f7f7f7f, 2, s);
    acc[3][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bj, f8_cat(a[3][0], a[3][1]), acc[3][j], 0, 0, 0,
                                                                 0x7f7f7f7f, 3, s);
  }
  __builtin_amdgcn_s_setprio(0);
}

// QOUT (GELU c_fc of the MX prefill): the epilogue quantises its own output
// tile for the next GEMM — e4m3 bytes q_out[M][ldq] with one e8m0 scale per
// (row, 128 columns) from the tile's columns alone (the 4 waves sharing a row
// agree through LDS), so the c_proj input never exists in bf16 and no
// quantise pass reads it back.  Columns >= N are written as zeros up to kpo.
template <int ACT, bool SCATTER = false, int NQ = 2, bool MXA = false, bool QOUT = false>
__global__ __launch_bounds__(512, 1) void gemm_fp8_256_kernel(
    const uint8_t* __restrict__ A8, const float* __restrict__ sa, const uint8_t* __restrict__ W8,
    const float* __restrict__ sw, bf16_t* __restrict__ C, int ldc, const float* __restrict__ bias,
    const bf16_t* __restrict__ R, int ldr, int M, int N, int Kb, QkvScatter scat = {},
    const uint32_t* __restrict__ sx = nullptr, uint8_t* __restrict__ qo = nullptr, int ldq = 0,
    uint8_t* __restrict__ sxo = nullptr, int kpo = 0) {
  // (QOUT reuses the operand LDS after the main loop: see the epilogue)
  static_assert(NQ == 1 || NQ == 2, "256x256 or 256x128 tiles");
  static_assert(!MXA || NQ == 2, "MX activations: 256^2 tiles");
  static_assert(!QOUT || (MXA && ACT == ACT_GELU && !SCATTER), "quantised output: the MX c_fc");
  constexpr int TN = 128 * NQ;  // NQ = 1: the 256x128 variant (tail-split launches), as the bf16 kernel's
  constexpr int SCL_LDS = MXA ? 2 * 2 * 8 * 256 : 0;  // activation scales: [K-tile & 1][half][wave]
  __shared__ __attribute__((aligned(1024))) char smem[8 * BG_HALF + EPI_LDS + SCL_LDS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntn = (N + TN - 1) / TN, ntm = (M + BG_M - 1) / BG_M;
  int tm, tn;
  tile_coords(xcd_remap(blockIdx.x, ntm * ntn), ntm, ntn, tm, tn);
  const int m0 = tm * BG_M, n0 = tn * TN;
  const int wr = wave >> 2, wc = wave & 3;
  const int nk = Kb / 128;
  const int gan = g_gemm_anatomy;
  // epilogue operands in LDS (epi_operands_dma): channel scales, bias (SCATTER:
  // by the global column), per-row activation scales (not MXA); uniform
  char* epi = smem + 8 * BG_HALF;
  const int boff = SCATTER ? scat.c_off : 0;
  const bool epv = (N & 3) == 0 && (MXA || (M & 3) == 0) && M >= 4 && N >= 4 &&
                   ((reinterpret_cast<uintptr_t>(sw) | reinterpret_cast<uintptr_t>(bias) |
                     reinterpret_cast<uintptr_t>(sa)) & 15) == 0;
  if (epv)
    epi_operands_dma(bias != nullptr ? bias + boff : nullptr, sw, nullptr, MXA ? nullptr : sa, n0, N, m0, M, epi,
                     wave, lane);
  // byte-identical staging: view the e4m3 rows as bf16 rows of half the length
  const bf16_t* A = reinterpret_cast<const bf16_t*>(A8);
  const bf16_t* W = reinterpret_cast<const bf16_t*>(W8);
  const int lda = Kb / 2, ldw = Kb / 2;

  f32x4 acc[2][NQ][4][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < NQ; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[a][b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto half = [&](int u, int h) { return smem + (u * 4 + h) * BG_HALF; };
  BgRows ra, rb;
  if constexpr (NQ == 2) {
    ra.init(A, lda, m0, M, wave, lane);
    rb.init(W, ldw, n0, N, wave, lane);
  }
  auto stA = [&](int u, int h, int t) {
    t = t < nk ? t : nk - 1;
    if constexpr (NQ == 2) ra.stage(h, t, half(u, h), wave);
    else stage_half(A, lda, m0 + h * 128, M, t * BG_K, half(u, h), wave, lane);
  };
  auto stB = [&](int u, int h, int t) {
    t = t < nk ? t : nk - 1;
    if constexpr (NQ == 2) rb.stage(h, t, half(u, 2 + h), wave);
    else stage_half(W, ldw, n0 + h * 128, N, t * BG_K, half(u, 2 + h), wave, lane);
  };

  bf16x8 af[4][2], b0[2][2], b1[2][2];
  const int arow = wr * 64, brow = wc * 32;
  if constexpr (NQ == 1) {
    // the bf16 kernel's 2-phase K-tile (256x128), one scaled MFMA per tile pair
    stA(0, 0, 0);
    stB(0, 0, 0);
    stA(0, 1, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    bg_barrier();
    if (wr == 1) bg_barrier();
    auto ktile1 = [&](const int t, auto ucst) {
      constexpr int u = decltype(ucst)::value;
      bg_read<2>(b0, half(u, 2), brow, lane);
      __builtin_amdgcn_sched_barrier(0);
      bg_read<4>(af, half(u, 0), arow, lane);
      stA(u ^ 1, 0, t + 1);
      stB(u ^ 1, 0, t + 1);
      asm volatile("s_waitcnt vmcnt(4)" ::: "memory");  // A1 of tile t landed
      bg_barrier();
      bg_mfma_f8<4, 2>(acc[0][0], af, b0);
      bg_barrier();
      bg_read<4>(af, half(u, 1), arow, lane);
      stA(u ^ 1, 1, t + 1);
      asm volatile("s_waitcnt vmcnt(2)" ::: "memory");  // A0 / B0 of tile t+1 landed
      bg_barrier();
      bg_mfma_f8<4, 2>(acc[1][0], af, b0);
      bg_barrier();
    };
    int t = 0;
    for (; t + 1 < nk; t += 2) {
      ktile1(t, std::integral_constant<int, 0>{});
      ktile1(t + 1, std::integral_constant<int, 1>{});
    }
    if (t < nk) ktile1(t, std::integral_constant<int, 0>{});
  } else {
  // MXA: the scale dwords of a K-tile (half-tiles 0 / 1 of A), a wave's own copy in LDS;
  // tile t + 1's are sent for in tile t's first phase, ahead of its half-tile, so the wait
  // there finds tile t's behind all that may be in flight.  (Loaded to registers they were
  // carried around the loop, and the compiler waited for everything in flight, vmcnt(0),
  // before every second tile's first product: 2048 x 6400 x 1600 with GELU 41.5 us, now 39.0.)
  uint32_t scl[2] = {0x7f7f7f7fu, 0x7f7f7f7fu};
  char* const scl_lds = smem + 8 * BG_HALF + EPI_LDS + wave * 256;
  const int nb64 = mx_mpad(M) >> 6;
  auto ldsx = [&](int t, int u) {
    t = t < nk ? t : nk - 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t* p = sx + ((size_t)t * nb64 + min((m0 >> 6) + 2 * h + wr, nb64 - 1)) * 16;
      asm("" : "+s"(p));  // scalar base (BgRows::stage)
      __builtin_amdgcn_global_load_lds((const GLB_AS void*)(p + (lane & 15)), (LDS_AS void*)(scl_lds + (u * 2 + h) * 2048), 4,
                                       0, 0);
    }
  };
  auto rdsx = [&](int u) {
#pragma unroll
    for (int h = 0; h < 2; ++h) scl[h] = *reinterpret_cast<const uint32_t*>(scl_lds + (u * 2 + h) * 2048 + lane * 4);
  };
  bf16x8 a1[4][2];
  constexpr int FLY = MXA ? 12 : 10;  // the schedule of gemm_tile.h
  if constexpr (MXA) ldsx(0, 0);
  stA(0, 0, 0);
  stB(0, 0, 0);
  stB(0, 1, 0);
  stA(0, 1, 0);
  stA(1, 0, 1);
  stB(1, 0, 1);
  stB(1, 1, 1);
  bg_landed<10>();
  bg_barrier();
  if (wr == 1) bg_barrier();
  bg_read<4>(af, half(0, 0), arow, lane);

  auto mm = [&](f32x4 (&c)[4][2], const bf16x8 (&aa)[4][2], const bf16x8 (&bb)[2][2], uint32_t s, auto wait) {
    constexpr bool W = decltype(wait)::value;
    if constexpr (MXA) bg_mfma_f8x<4, 2, W>(c, aa, bb, s);
    else bg_mfma_f8<4, 2, W>(c, aa, bb);
  };
  auto ktile = [&](const int t, auto ucst) {
    constexpr int u = decltype(ucst)::value;
    bg_read<2>(b0, half(u, 2), brow, lane);
    if constexpr (MXA) ldsx(t + 1, u ^ 1);
    stA(u ^ 1, 1, t + 1);
    bg_landed<FLY>();
    if constexpr (MXA) rdsx(u);
    bg_barrier();
    mm(acc[0][0], af, b0, scl[0], std::true_type{});
    bg_barrier();
    bg_read<2>(b1, half(u, 3), brow, lane);
    stA(u, 0, t + 2);
    bg_landed<FLY>();
    bg_barrier();
    mm(acc[0][1], af, b1, scl[0], std::true_type{});
    bg_barrier();
    bg_read<4>(a1, half(u, 1), arow, lane);
    stB(u, 0, t + 2);
    bg_landed<FLY>();
    bg_barrier();
    mm(acc[1][1], a1, b1, scl[1], std::true_type{});
    bg_barrier();
    bg_read<4>(af, half(u ^ 1, 0), arow, lane);
    stB(u, 1, t + 2);
    bg_landed<FLY>();
    bg_barrier();
    mm(acc[1][0], a1, b0, scl[1], std::false_type{});
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    bg_barrier();
  };
  int t = (gan & 2) ? nk : 0;
  for (; t + 1 < nk; t += 2) {
    ktile(t, std::integral_constant<int, 0>{});
    ktile(t + 1, std::integral_constant<int, 1>{});
  }
  if (t < nk) ktile(t, std::integral_constant<int, 0>{});
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (wr == 0) bg_barrier();
  if (gan & 1) {  // anatomy probe: no stores
    if (acc[0][0][0][0][0] == 1.2345e-30f) C[0] = 0;
    return;
  }

  // Channel scales and (QOUT, or where the LDS copy is whole) bias of the lane's columns, held
  // from here on: looked up at every product they put three paths and a wait around each, and
  // the epilogue of 2048 x 4800 x 1600 took as long as its 13 K-tiles (31.3 us; 26.5 with the
  // scatter's addresses formed once as well, 2048 x 6400 x 1600 with GELU 39.0 : 37.6; without
  // activation 31.4 : 28.5, 8192 rows 108.7 : 99.5).  MX with ReLU looks them up: where it holds
  // them, the compiler spills operands in every K-tile (2048 x 1600 x 6400 59 : 84).
  constexpr bool HELD = !(MXA && ACT == ACT_RELU);
  f32x4 cs[NQ][2], bs[NQ][2];
  if constexpr (HELD) {
#pragma unroll
    for (int nq = 0; nq < NQ; ++nq)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n0 + nq * 128 + wc * 32 + j * 16 + (lane >> 4) * 4;
        bs[nq][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (epv) {  // the LDS copy (columns past N are not stored)
          cs[nq][j] = *reinterpret_cast<const f32x4*>(epi + EPI_C + 4 * (n - n0));
          if (bias != nullptr) bs[nq][j] = *reinterpret_cast<const f32x4*>(epi + EPI_B + 4 * (n - n0));
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            cs[nq][j][r] = n + r < N ? sw[n + r] : 0.f;
            if (QOUT) bs[nq][j][r] = (bias != nullptr && n + r < N) ? bias[n + r] : 0.f;
          }
        }
        if constexpr (QOUT) {  // columns past N leave as zeros: here once, not at every value (with gelu_erf's form 2048 x 6400 x 1600 37.8 -> 35.5 us)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (n + r >= N) cs[nq][j][r] = bs[nq][j][r] = 0.f;
          }
        }
      }
  }
  if constexpr (QOUT) {
    // bias + GELU in place, then per (row, 128-column half nq) amax: the lane's
    // 8 columns, the 4 lane rows of the wave (xor 16 / 32), the 4 waves of the
    // wave row through LDS (the operand buffers are dead), one barrier
    float* red = reinterpret_cast<float*>(smem);  // [mq][nq][i][wr][16][wc]
    __syncthreads();  // every wave past its last operand read and DMA (vmcnt(0) above)
#pragma unroll
    for (int mq = 0; mq < 2; ++mq)
#pragma unroll
      for (int nq = 0; nq < NQ; ++nq)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float am = 0.f;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            f32x4 v = acc[mq][nq][i][j] * cs[nq][j] + bs[nq][j];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              v[r] = gelu_erf(v[r]);
              am = fmaxf(am, fabsf(v[r]));
            }
            acc[mq][nq][i][j] = v;
          }
          am = max16(am);
          am = max32(am);
          if (lane < 16) red[((((mq * 2 + nq) * 4 + i) * 2 + wr) * 16 + lane) * 4 + wc] = am;
        }
    __syncthreads();
    const int mpad = mx_mpad(M);
#pragma unroll
    for (int mq = 0; mq < 2; ++mq)
#pragma unroll
      for (int nq = 0; nq < NQ; ++nq)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 a4 =
              *reinterpret_cast<const f32x4*>(red + ((((mq * 2 + nq) * 4 + i) * 2 + wr) * 16 + (lane & 15)) * 4);
          float inv;
          const uint32_t e = e8m0_of(fmaxf(fmaxf(a4[0], a4[1]), fmaxf(a4[2], a4[3])), inv);
          const f32x4 v0 = acc[mq][nq][i][0] * inv, v1 = acc[mq][nq][i][1] * inv;
          int x = __builtin_amdgcn_cvt_pk_fp8_f32(v0[0], v0[1], 0, false);
          x = __builtin_amdgcn_cvt_pk_fp8_f32(v0[2], v0[3], x, true);
          int y = __builtin_amdgcn_cvt_pk_fp8_f32(v1[0], v1[1], 0, false);
          y = __builtin_amdgcn_cvt_pk_fp8_f32(v1[2], v1[3], y, true);
          // as epi_pair_bf16: one permlane16_swap hands every lane 8 contiguous columns
          const auto sw2 = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)y, false, false);
          const int m = m0 + mq * 128 + arow + i * 16 + (lane & 15);
          const int q = lane >> 4;
          const int cb = n0 + nq * 128 + wc * 32;
          const int c = cb + ((q & 1) << 4) + ((q >> 1) << 3);
          if (m < M && c < kpo) *reinterpret_cast<uint2*>(qo + (size_t)m * ldq + c) = make_uint2(sw2[0], sw2[1]);
          const int t = (n0 + nq * 128) >> 7;
          if (wc == 0 && q == 0 && m < M && t * 128 < kpo) sxo[mx_index(m, t, mpad)] = (uint8_t)e;
        }
    return;
  }
  const bool badd = epv && bias != nullptr && !is_glu(ACT);  // uniform: bias added from the LDS copy
  const float* bias_e = badd ? nullptr : bias;
  // SCATTER: the destinations' parts (qkv_row), before any store; bias that is not in LDS
  QkvRow srow[2][4];
  QkvCol scol[NQ];
  if constexpr (SCATTER) {
#pragma unroll
    for (int mq = 0; mq < 2; ++mq)
#pragma unroll
      for (int i = 0; i < 4; ++i) srow[mq][i] = qkv_row(scat, min(m0 + mq * 128 + arow + i * 16 + (lane & 15), M - 1));
#pragma unroll
    for (int nq = 0; nq < NQ; ++nq) {
      const int nb = n0 + nq * 128 + wc * 32 + scat.c_off;
      scol[nq] = qkv_col(scat, pair_col(nb, lane));
      if (bias_e != nullptr && nb - scat.c_off < N) {
#pragma unroll
        for (int j = 0; j < 2; ++j) bs[nq][j] = *reinterpret_cast<const f32x4*>(bias_e + nb + j * 16 + (lane >> 4) * 4);
      }
    }
  }
  const bool vec = epi_vec_ok(C, ldc, bias, R, ldr);
  const bool pair = vec && epi_pair_ok(C, ldc, bias, R, ldr);
  // residual rows of the whole tile in flight before the first output (as in the bf16 kernel)
  const bool rpre = !is_glu(ACT) && pair && R != nullptr && n0 + TN - 1 < N;
  // the residual tile by LDS-DMA into the dead operand buffers (res_tile_dma;
  // anatomy bit 4 = the per-lane gathers below)
  const bool rdma = rpre && (gan & 4) == 0 && (ldr & 7) == 0 && (reinterpret_cast<uintptr_t>(R) & 15) == 0;
  bf16x4 rr[2][NQ][4][2];
  if (rdma) {
    __syncthreads();  // every wave past its last operand read and DMA (vmcnt(0) above)
    res_tile_dma<TN>(R, ldr, m0, n0, M, smem, wave, lane);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  } else if (rpre) {
#pragma unroll
    for (int mq = 0; mq < 2; ++mq)
#pragma unroll
      for (int nq = 0; nq < NQ; ++nq)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          epi_pair_res_load(m0 + mq * 128 + arow + i * 16 + (lane & 15), n0 + nq * 128 + wc * 32, M, R, ldr, lane,
                            rr[mq][nq][i][0], rr[mq][nq][i][1]);
  }
#pragma unroll
  for (int mq = 0; mq < 2; ++mq)
#pragma unroll
    for (int nq = 0; nq < NQ; ++nq)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + mq * 128 + arow + i * 16 + (lane & 15);
        const int nb = n0 + nq * 128 + wc * 32;
        // MXA: the activation scales are in acc
        const float rs = MXA ? 1.f
                             : (epv ? reinterpret_cast<const float*>(epi + EPI_SA)[m - m0] : (m < M ? sa[m] : 0.f));
        f32x4 v[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma clang fp contract(off)  // the product is rounded before the bias, on every path
          const int n = nb + j * 16 + (lane >> 4) * 4;
          f32x4 c4;
          if constexpr (HELD) {
            c4 = cs[nq][j];
          } else if (epv) {
            c4 = *reinterpret_cast<const f32x4*>(epi + EPI_C + 4 * (n - n0));
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) c4[r] = n + r < N ? sw[n + r] : 0.f;
          }
          v[j] = acc[mq][nq][i][j] * (c4 * rs);
          if constexpr (HELD) {
            if (badd || (SCATTER && bias != nullptr)) v[j] += bs[nq][j];
          } else {
            if (badd) v[j] += *reinterpret_cast<const f32x4*>(epi + EPI_B + 4 * (n - n0));
          }
        }
        if (SCATTER) {
          if (nb < N) epi_pair_scatter(v[0], v[1], m, M, srow[mq][i], scol[nq]);
        } else if (is_glu(ACT)) {
          epi_glu_pair<ACT, false>(v[0], v[1], m, nb / 2, M, N / 2, C, ldc, vec, lane);
        } else if (rdma) {
          const int rl = m - m0, cl = nb - n0 + (lane >> 4) * 4;
          epi_pair_bf16<ACT, true>(v[0], v[1], m, nb, M, C, ldc, bias_e, R, ldr, lane, res_tile_read<TN>(smem, rl, cl),
                                   res_tile_read<TN>(smem, rl, cl + 16));
        } else if (rpre) {
          epi_pair_bf16<ACT, true>(v[0], v[1], m, nb, M, C, ldc, bias_e, R, ldr, lane, rr[mq][nq][i][0],
                                   rr[mq][nq][i][1]);
        } else if (pair && nb + 31 < N) {
          epi_pair_bf16<ACT>(v[0], v[1], m, nb, (gan & 8) ? 0 : M, C, ldc, bias_e, R, ldr, lane);
        } else {
#pragma unroll
          for (int j = 0; j < 2; ++j)
            epi_t4<ACT, false>(v[j], m, nb + j * 16 + (lane >> 4) * 4, M, N, C, ldc, bias_e, R, ldr, vec);
        }
      }
}

// SwiGLU for the skinny path: h[m, j] = silu(g[m, j]) * u[m, j] where the skinny
// GEMM produced the packed [M, 2F] fp32/bf16 output.
__global__ void silu_mul_packed_kernel(const bf16_t* __restrict__ gu, int ld_in, bf16_t* __restrict__ out,
                                       int ld_out, int M, int F) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= M * F) return;
  const int m = idx / F, j = idx % F;
  const int grp = j / 16, c = j % 16;
  const float g = bf2f(gu[(size_t)m * ld_in + grp * 32 + c]);
  const float u = bf2f(gu[(size_t)m * ld_in + grp * 32 + 16 + c]);
  out[(size_t)m * ld_out + j] = f2bf(silu(g) * u);
}

}  // namespace dnn

// ------------------------------- host API ----------------------------------
using namespace dnn;

// Large-GEMM tile selection: 0 = auto (gemm_mid.hip mid_plan), 128 / 255 / 256
// force a tile (A/B benchmarking, tests).
static int g_gemm_tile = 0;
// Forced tile of gemm_mid.h's table and K split (tests, A/B); -1: chosen
static int g_mid_tile = -1, g_mid_splits = 1;
extern "C" int dnn_gemm_set_mid(int tile, int splits) {
  if (tile < -1 || tile > 6 || splits < 1 || splits > 16) return -1;
  g_mid_tile = tile;
  g_mid_splits = splits;
  return 0;
}
// Workgroups of a tile of that table (mx: of the e4m3 kernel's) that share a CU
extern "C" int dnn_gemm_mid_blocks(int tile, int mx) {
#ifndef DNN_DECODER_ONLY
  if (mx) return mid8_blocks(tile);
#endif
  return mx ? -1 : mid_blocks(tile);
}
// Rows up to which every bf16 GEMM streams its weights on the skinny kernels
// (A/B switch).  At M = 64 a wide-N head with warm weights runs faster on the
// 128^2 MFMA tiles (GPT-2 50304 x 768: 28.3 -> 22.5 us, x 1600: 52.7 -> 33.6,
// profiles/archive/r2_head_probe.jsonl), but inside the decode step (weights cold behind
// 1.27 GB of K/V) GPT-2 B=64 ran 0.588 -> 0.603 ms/step that way and GPT-2 XL
// B=64 4.507 -> 4.493 (profiles/archive/r2_decode_ab_skinny_max_m.jsonl): 64 stays.
static int g_skinny_max_m = 64;

extern "C" int dnn_gemm_set_skinny_max_m(int m) {
  if (m < 0 || m > 64) return -1;
  g_skinny_max_m = m;
  return 0;
}

// The decode kernels' rows: all up to g_skinny_max_m, beyond by estimate unless a tile is pinned
static bool skinny(int M, int N, int K, bool norm, bool frag, long long part_bytes) {
  return M <= g_skinny_max_m || (g_gemm_tile == 0 && g_mid_tile < 0 && mid_skinny(M, N, K, norm, frag, part_bytes));
}
extern "C" int dnn_gemm_is_skinny(int M, int N, int K, int norm, int frag, long long ws_bytes) {
  return skinny(M, N, K, norm != 0, frag != 0, ws_bytes - 4096);
}

// 256^2 epilogue: residual rows loaded ahead of the outputs (1) or per output row group (0)
static int g_res_prefetch = 1;

extern "C" int dnn_gemm_set_res_prefetch(int on) {
  g_res_prefetch = on ? 1 : 0;
  return 0;
}

extern "C" int dnn_gemm_set_anatomy(int bits) {
  return (int)hipMemcpyToSymbol(HIP_SYMBOL(g_gemm_anatomy), &bits, sizeof(int));
}

extern "C" int dnn_gemm_set_tile(int tile) {
  if (tile != 0 && tile != 128 && tile != 256 && tile != 255) return -1;  // 255: force 256x128
  g_gemm_tile = tile;
  return 0;
}

// Relative time of one 256x128 tile against one 256x256 tile (the auto rule
// picks 256x128 when ceil(tiles/256) x this beats the 256^2 rounds).  Off by
// default (measured, profiles/r4_gemm_tiles*.jsonl): at M = 32768 the 256x128
// tiles ran N=768 K=768 752 -> 672 TF/s, K=3072 1052 -> 1070, N=2304 885 ->
// 768, and the GPT-2 4-stage prefill 3.85 -> 3.76 M tok/s — the 2-phase
// schedule, one K-tile ahead, loses more per tile than the full last round
// saves; tile 255 keeps it selectable.
// the 256^2 + 256x128 tail split (A/B switch, a bit mask: 1 the bf16 kernel, 2 the fp8 one; DNN_SPLIT_TAIL
// sets the start value).  fp8 is off by default: GPT-2 XL prefill 259.5 -> 257.4 k tok/s with it
// (profiles/r4_prefill_ab_tail_split_gpt2xl.jsonl), bf16 GPT-2 +1.6 %
static int g_split_tail = [] {
  const char* e = getenv("DNN_SPLIT_TAIL");
  return e != nullptr ? atoi(e) : 1;
}();
extern "C" int dnn_gemm_set_split_tail(int on) {
  g_split_tail = on;
  return 0;
}

// Tail split rule: the columns of the 256^2 part (a multiple of 256), or 0.
// Applies when the 256^2 grid is whole rounds of 256 tiles plus one last
// column of tiles (1..256 columns wide) that fits one more round as 256x128
// tiles: GPT-2 (N 768 / 2304) and GPT-2 XL (N 1600 / 4800 / 6400) at M = 32768.
static int tail_split_cols(int M, int N, bool fp8 = false) {
  // fp8: bit 2 every tail, bit 4 only tails of >= 128 columns (GPT-2 XL c_attn / c_fc, not the 64-column
  // tail of the 1600-wide O / c_proj)
  if (!(g_split_tail & (fp8 ? 6 : 1)) || g_gemm_tile != 0) return 0;
  const int ntm = (M + 255) / 256, ntn = (N + 255) / 256;
  if (ntn < 2 || (ntm * (ntn - 1)) % 256 != 0) return 0;
  const int Na = (ntn - 1) * 256;
  if (fp8 && !(g_split_tail & 2) && N - Na < 128) return 0;
  if (ntm * ((N - Na + 127) / 128) > 256) return 0;
  return Na;
}

static float g_half_cost = 1e9f;
extern "C" int dnn_gemm_set_half_cost(float c) {
  if (!(c > 0.f)) return -1;
  g_half_cost = c;
  return 0;
}

// Partials of the row statistics for one call (dnn_gemm_bf16_parts, its scatter): what launch_gemm shall read in
// place of rowstat and write beside C; `wrote`: it did.
struct PartsReq {
  const float2* in = nullptr;
  float2* out = nullptr;
  float eps = 0.f;
  int rms = 0, wrote = 0;
};
static thread_local PartsReq g_parts;
struct PartsScope {
  explicit PartsScope(const PartsReq& r) { g_parts = r; }
  ~PartsScope() { g_parts = PartsReq{}; }
};

// The small tiles address a tile's rows with 32 bits.
static bool mid_narrow(int lda, int ldw) { return lda < 1 << 23 && ldw < 1 << 23; }

// Rows that 16-byte LDS-DMA may fetch.
static bool dma_rows(const void* A, int lda, const void* W, int ldw) {
  return (((uintptr_t)A | (uintptr_t)W) & 15) == 0 && lda % 8 == 0 && ldw % 8 == 0;
}

template <int ACT, bool F32>
static int launch_gemm(const void* A, int lda, const void* W, int ldw, void* C, int ldc, const float* bias,
                        const void* R, int ldr, int M, int N, int K, hipStream_t st, const void* Wsh,
                        const float2* rowstat, const float* colsum, void* ws, long long ws_bytes) {
  // decode-sized: the weight-streaming kernels (gemm_skinny.hip); a folded-norm
  // GEMM (rowstat) always takes the tile kernels: the skinny path folds its norm
  // itself, dnn_gemm_skinny_norm
  const long long part_bytes = mid_ws(ws, ws_bytes);
  // up to 256 rows what the small tiles cannot stage (dma_rows) goes to the decode kernels, whose loads are plain
  const bool narrow = mid_narrow(lda, ldw);
  if (rowstat == nullptr && g_parts.in == nullptr && (skinny(M, N, K, false, Wsh != nullptr, part_bytes) ||
                             (M <= 256 && (!narrow || !dma_rows(A, lda, W, ldw))))) {
    return dnn_gemm_skinny(A, lda, nullptr, W, ldw, nullptr, C, ldc, bias, R, ldr, M, N, K, ACT, F32 ? 1 : 0, 0, st, Wsh,
                           ws, ws_bytes);
  }
  // Tiles of gemm_mid.h, or 256 x 256 (and its tail split below) by estimated time
  const int tiles256 = ((M + BG_M - 1) / BG_M) * ((N + BG_N - 1) / BG_N);
  MidPlan plan{-1, 1, 0.f, 0};
  if (!narrow) {
  } else if (g_mid_tile >= 0) plan = {g_mid_tile, (long long)g_mid_splits * M * N * 4 <= part_bytes ? g_mid_splits : 1, 0.f, 0};
  else if (g_gemm_tile == 128) plan.tile = 2;
  else if (g_gemm_tile == 0 && (is_glu(ACT) || has_consts(ACT) || tail_split_cols(M, N) == 0))
    plan = mid_plan(M, N, K, part_bytes, has_consts(ACT) ? MID_BF16_WHOLE : MID_BF16);  // constants lie behind all N
  // partials are merged by one launch of the small tiles over all columns and all of K, and by nothing else
  if (g_parts.in != nullptr && (plan.tile < 0 || plan.cols != 0 || plan.splits != 1)) return -4;
  if (plan.tile >= 0) {
    MidArgs a{{C, bias, (const bf16_t*)R, ldc, ldr, M, N, ACT, F32 ? 1 : 0}, (const bf16_t*)A, (const bf16_t*)W,
              rowstat, colsum, nullptr, g_parts.in, g_parts.eps, g_parts.rms, (float*)ws, lda, ldw, K, plan.splits};
    // partials beside rows that leave as pairs of 16-byte stores with a residual (mid_rows)
    if (g_parts.out != nullptr && !F32 && ACT == ACT_NONE && R != nullptr && plan.cols == 0 && N % MID_PARTS_N == 0 &&
        (((uintptr_t)C | (uintptr_t)R | (uintptr_t)bias) & 15) == 0 && ldc % 8 == 0 && ldr % 8 == 0) {
      a.parts_out = g_parts.out;
      g_parts.wrote = 1;
    }
    if (const int n = plan.cols) {  // disjoint columns
      hipLaunchKernelGGL((gemm_bf16_256_kernel<ACT, F32>), dim3(((M + BG_M - 1) / BG_M) * (n / BG_N)), dim3(512), 0, st,
                         a.A, lda, a.W, ldw, C, ldc, bias, a.R, ldr, M, n, K, g_res_prefetch, rowstat, colsum);
      if (const hipError_t e = hipGetLastError()) return (int)e;
      a.C = (char*)C + (size_t)(is_glu(ACT) ? n / 2 : n) * (F32 ? 4 : 2);
      a.W += (size_t)n * ldw;
      a.N -= n;
      if (bias != nullptr) a.bias += n;
      if (a.R != nullptr) a.R += n;
      if (colsum != nullptr) a.colsum += n;
    }
    return mid_launch(plan.tile, a, nullptr, st);
  }
  const int tilesH = ((M + BG_M - 1) / BG_M) * ((N + 127) / 128);
  const bool half = g_gemm_tile == 255 || !bg_narrow(lda) || !bg_narrow(ldw) ||
                    (g_gemm_tile == 0 && (float)((tilesH + 255) / 256) * g_half_cost < (float)((tiles256 + 255) / 256));
  if (half) {
    hipLaunchKernelGGL((gemm_bf16_256_kernel<ACT, F32, false, 1>), dim3(tilesH), dim3(512), 0, st, (const bf16_t*)A,
                       lda, (const bf16_t*)W, ldw, C, ldc, bias, (const bf16_t*)R, ldr, M, N, K, g_res_prefetch,
                       rowstat, colsum);
    return (int)hipGetLastError();
  }
  // Tail split: when the 256^2 grid is full rounds plus a last
  // column of tiles that fills at most one more round as 256x128 tiles (GPT-2's
  // 768-wide O / c_proj at M = 32768: 256 tiles + a 128-tile column), the
  // first N - 256 columns run as 256^2 tiles and the last 256 as 256x128 tiles
  // in a second launch — 1 + 1/2 rounds instead of 2 full ones, no workspace
  // and no reduction (the two launches write disjoint columns).
  const int ntm256 = (M + BG_M - 1) / BG_M;
  const int Na = (!is_glu(ACT) && !has_consts(ACT)) ? tail_split_cols(M, N) : 0;  // constants lie behind all N
  if (Na > 0) {
    const int Nt = N - Na;
    const size_t cb = F32 ? sizeof(float) : sizeof(bf16_t);
    hipLaunchKernelGGL((gemm_bf16_256_kernel<ACT, F32>), dim3(ntm256 * (Na / 256)), dim3(512), 0, st,
                       (const bf16_t*)A, lda, (const bf16_t*)W, ldw, C, ldc, bias, (const bf16_t*)R, ldr, M, Na, K,
                       g_res_prefetch, rowstat, colsum);
    hipLaunchKernelGGL((gemm_bf16_256_kernel<ACT, F32, false, 1>), dim3(ntm256 * ((Nt + 127) / 128)), dim3(512), 0,
                       st, (const bf16_t*)A, lda, (const bf16_t*)W + (size_t)Na * ldw, ldw,
                       (void*)((char*)C + (size_t)Na * cb), ldc, bias != nullptr ? bias + Na : nullptr,
                       R != nullptr ? (const bf16_t*)R + Na : nullptr, ldr, M, Nt, K, g_res_prefetch, rowstat,
                       colsum != nullptr ? colsum + Na : nullptr);
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL((gemm_bf16_256_kernel<ACT, F32>), dim3(tiles256), dim3(512), 0, st, (const bf16_t*)A, lda,
                     (const bf16_t*)W, ldw, C, ldc, bias, (const bf16_t*)R, ldr, M, N, K, g_res_prefetch, rowstat,
                     colsum);
  return (int)hipGetLastError();
}

// rowstat (M float2 {rstd, -mean rstd}) / colsum (N floats, LayerNorm only):
// folded pre-norm epilogue, v = rstd acc - mean rstd colsum, before bias / act /
// residual (ops/gemm.py linear_norm at prefill sizes); nullptr = plain GEMM.
extern "C" int dnn_gemm_bf16(const void* A, int lda, const void* W, int ldw, void* C, int ldc, const float* bias,
                             const void* R, int ldr, int M, int N, int K, int act, int out_f32, hipStream_t st,
                             const void* Wsh, const float* rowstat, const float* colsum, void* ws,
                             long long ws_bytes) {
  if (K % 64 != 0 || M <= 0 || N <= 0) return -1;
  if (colsum != nullptr && rowstat == nullptr && g_parts.in == nullptr) return -1;
  const float2* rs = reinterpret_cast<const float2*>(rowstat);
#define DISPATCH(a)                                                                                  \
  if (act == a) {                                                                                    \
    if (out_f32) return launch_gemm<a, true>(A, lda, W, ldw, C, ldc, bias, R, ldr, M, N, K, st, Wsh, rs, colsum, ws, ws_bytes); \
    return launch_gemm<a, false>(A, lda, W, ldw, C, ldc, bias, R, ldr, M, N, K, st, Wsh, rs, colsum, ws, ws_bytes); \
  }
  DISPATCH(ACT_NONE)
#ifndef DNN_DECODER_ONLY  // the other families' epilogues: not in the decoder subset (ops/build.py)
  DISPATCH(ACT_RELU)
  DISPATCH(ACT_GELU)
  DISPATCH(ACT_SILU_MUL)
#endif
#undef DISPATCH
#define DISPATCH_BF16(a)                                                                                             \
  if (act == a && !out_f32) {                                                                                        \
    return launch_gemm<a, false>(A, lda, W, ldw, C, ldc, bias, R, ldr, M, N, K, st, Wsh, rs, colsum, ws, ws_bytes); \
  }
  DISPATCH_BF16(ACT_GELU_TANH_MUL)
  if (act == ACT_XIELU && bias == nullptr) return -2;
  DISPATCH_BF16(ACT_XIELU)
#ifdef DNN_DECODER_ONLY
  DISPATCH_BF16(ACT_SILU_MUL)
#endif
#undef DISPATCH_BF16
  return -2;
}

#ifndef DNN_DECODER_ONLY
// Whether a folded norm of these sizes and distances of rows can take its statistics from partials: one launch of the
// small tiles, K whole.
static bool takes_parts(int M, int N, int K, int lda, int ldw, long long part_bytes, int act, bool scatter) {
  if (g_gemm_tile != 0 || K % 64 != 0 || K > MID_PARTS_K || !mid_narrow(lda, ldw)) return false;
  if (scatter && tail_split_cols(M, N) != 0) return false;
  if (g_mid_tile >= 0) return scatter || g_mid_splits == 1;
  if (!is_glu(act) && tail_split_cols(M, N) != 0) return false;
  const MidPlan p = mid_plan(M, N, K, scatter ? 0 : part_bytes, scatter || has_consts(act) ? MID_BF16_WHOLE : MID_BF16);
  return p.tile >= 0 && p.cols == 0 && p.splits == 1;
}

extern "C" int dnn_gemm_takes_parts(int M, int N, int K, int lda, int ldw, int act, int scatter, long long ws_bytes) {
  return takes_parts(M, N, K, lda, ldw, ws_bytes - 4096, act, scatter != 0);
}

// GPT-2, 3 x 357 tokens: a statistics launch of 3.4 us ahead of every c_attn and c_fc, 784 a pass; as partials, which
// cost their writers 0.2 and their readers 0.6 each, 749.  Rows wider than MID_PARTS_K keep the launch: the
// partials of 4096 columns are as many bytes a workgroup as two of its K-tiles, and 700 rows' launch is 5 of 340 a block.
// dnn_gemm_bf16 with a folded norm (norm 1 RMS, 2 LayerNorm, 0 none) whose statistics come from `parts` (partials of A's
// rows, [M][K / 32]) where these sizes take them, else from a pass over A into `stats`; the partials
// of C's rows go to `parts_out` (null: none) where they can, `wrote` says whether.
extern "C" int dnn_gemm_bf16_parts(const void* A, int lda, const void* W, int ldw, void* C, int ldc, const float* bias,
                                   const void* R, int ldr, int M, int N, int K, int act, hipStream_t st, const void* Wsh,
                                   int norm, float eps, float* stats, const void* parts, const float* colsum,
                                   void* parts_out, int* wrote, void* ws, long long ws_bytes) {
  const bool read = norm != 0 && parts != nullptr && takes_parts(M, N, K, lda, ldw, mid_ws(ws, ws_bytes), act, false);
  *wrote = 0;
  if (norm != 0 && !read) {
    if (stats == nullptr) return -1;
    if (const int rc = dnn_row_stats(A, lda, stats, M, K, eps, norm == 1, st)) return rc;
  }
  PartsScope scope({read ? (const float2*)parts : nullptr, (float2*)parts_out, eps, norm == 1, 0});
  const int rc = dnn_gemm_bf16(A, lda, W, ldw, C, ldc, bias, R, ldr, M, N, K, act, 0, st, Wsh,
                               norm != 0 && !read ? stats : nullptr, norm != 0 ? colsum : nullptr, ws, ws_bytes);
  *wrote = g_parts.wrote;
  return rc;
}

extern "C" int dnn_gemm_bf16_qkv_scatter_parts(const void* A, int lda, const void* W, int ldw, const float* bias, int norm,
                                               float eps, float* stats, const void* parts, const float* colsum, void* q,
                                               void* kc, void* vc, const int* pos, int B, int T, int H, int Hkv, int hd,
                                               int S, int K, hipStream_t st) {
  const int N = (H + 2 * Hkv) * hd;
  const bool read = parts != nullptr && N % 32 == 0 && takes_parts(B * T, N, K, lda, ldw, 0, ACT_NONE, true);
  if (!read) {
    if (const int rc = dnn_row_stats(A, lda, stats, B * T, K, eps, norm == 1, st)) return rc;
  }
  PartsScope scope({read ? (const float2*)parts : nullptr, nullptr, eps, norm == 1, 0});
  return dnn_gemm_bf16_qkv_scatter(A, lda, W, ldw, bias, read ? nullptr : stats, colsum, q, kc, vc, pos, B, T, H, Hkv, hd, S,
                                   K, st);
}

extern "C" int dnn_silu_mul_packed(const void* gu, int ld_in, void* out, int ld_out, int M, int F, hipStream_t st) {
  const int n = M * F;
  hipLaunchKernelGGL(silu_mul_packed_kernel, dim3((n + 255) / 256), dim3(256), 0, st, (const bf16_t*)gu, ld_in,
                     (bf16_t*)out, ld_out, M, F);
  return (int)hipGetLastError();
}

// Prefill c_attn with the QKV scatter epilogue (gemm_bf16_256_kernel SCATTER):
// y = x W^T + bias (folded pre-norm when rowstat) written head-major: q ->
// (B, H, T, hd), k / v -> the (B, Hkv, S, hd) caches at rows pos[b] + t.  M =
// B*T.  Returns -3 when the shape does not fit the 256^2 path (the caller then
// uses the qkv row output + qkv_split).
extern "C" int dnn_gemm_bf16_qkv_scatter(const void* A, int lda, const void* W, int ldw, const float* bias,
                                         const float* rowstat, const float* colsum, void* q, void* kc, void* vc,
                                         const int* pos, int B, int T, int H, int Hkv, int hd, int S, int K,
                                         hipStream_t st) {
  const int M = B * T, N = (H + 2 * Hkv) * hd;
  if (K % 64 != 0 || M <= 0 || hd % 8 != 0 || (colsum != nullptr && rowstat == nullptr && g_parts.in == nullptr)) return -1;
  if (N % 32 != 0 || ((uintptr_t)bias & 15) != 0 || (M < 256 && !dma_rows(A, lda, W, ldw))) return -3;
  const int tiles = ((M + BG_M - 1) / BG_M) * ((N + BG_N - 1) / BG_N);
  if ((hd & (hd - 1)) != 0 || M >= (1 << 24)) return -3;
  QkvScatter sc{(bf16_t*)q, (bf16_t*)kc, (bf16_t*)vc, pos, T, H, Hkv, __builtin_ctz(hd), S, 1.0f / (float)T};
  if (g_gemm_tile == 0 && tail_split_cols(M, N) == 0 && mid_narrow(lda, ldw)) {
    MidPlan plan = mid_plan(M, N, K, 0, MID_BF16_WHOLE);
    if (g_mid_tile >= 0) plan.tile = g_mid_tile;
    if (plan.tile >= 0) {
      const MidArgs a{{q, bias, nullptr, hd, 0, M, N, ACT_NONE, 0}, (const bf16_t*)A, (const bf16_t*)W,
                      reinterpret_cast<const float2*>(rowstat), colsum, nullptr, g_parts.in, g_parts.eps, g_parts.rms,
                      nullptr, lda, ldw, K, 1};
      return mid_launch(plan.tile, a, &sc, st);
    }
  }
  if (g_parts.in != nullptr) return -4;  // only the small tiles merge partials
  if (M < 256) return -3;
  if (!bg_narrow(lda) || !bg_narrow(ldw)) {  // the 256 x 128 tiles address rows with 64 bits
    hipLaunchKernelGGL((gemm_bf16_256_kernel<ACT_NONE, false, true, 1>), dim3((M + BG_M - 1) / BG_M * ((N + 127) / 128)),
                       dim3(512), 0, st, (const bf16_t*)A, lda, (const bf16_t*)W, ldw, q, hd, bias, (const bf16_t*)nullptr, 0,
                       M, N, K, 0, reinterpret_cast<const float2*>(rowstat), colsum, sc);
    return (int)hipGetLastError();
  }
  // tail split as launch_gemm's (GPT-2 c_attn at M = 32768: 1024 + 128 tiles
  // -> 4 rounds of 256^2 + 1 round of 256x128); the bias is indexed by the
  // global column (c_off), the folded norm's colsum by the launch's own
  const int ntm256 = (M + BG_M - 1) / BG_M;
  const int Na = tail_split_cols(M, N);
  if (Na > 0) {
    const int Nt = N - Na;
    hipLaunchKernelGGL((gemm_bf16_256_kernel<ACT_NONE, false, true>), dim3(ntm256 * (Na / 256)), dim3(512), 0, st,
                       (const bf16_t*)A, lda, (const bf16_t*)W, ldw, q, hd, bias, (const bf16_t*)nullptr, 0, M, Na, K,
                       0, reinterpret_cast<const float2*>(rowstat), colsum, sc);
    QkvScatter tail = sc;
    tail.c_off = Na;
    hipLaunchKernelGGL((gemm_bf16_256_kernel<ACT_NONE, false, true, 1>), dim3(ntm256 * ((Nt + 127) / 128)),
                       dim3(512), 0, st, (const bf16_t*)A, lda, (const bf16_t*)W + (size_t)Na * ldw, ldw, q, hd, bias,
                       (const bf16_t*)nullptr, 0, M, Nt, K, 0, reinterpret_cast<const float2*>(rowstat),
                       colsum != nullptr ? colsum + Na : nullptr, tail);
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL((gemm_bf16_256_kernel<ACT_NONE, false, true>), dim3(tiles), dim3(512), 0, st, (const bf16_t*)A,
                     lda, (const bf16_t*)W, ldw, q, hd, bias, (const bf16_t*)nullptr, 0, M, N, K, 0,
                     reinterpret_cast<const float2*>(rowstat), colsum, sc);
  return (int)hipGetLastError();
}

// The same with RoPE: x W^T under an RMS norm whose statistics this call takes (into `stats`), q and K rotated, heads of
// 128.  A wave's 32 columns are 16 of a head's lower half and the same 16 of its upper half (the weight's rows are
// staged in that order), so a rotation is within a lane, and the pass that split and rotated the stored rows goes (6.3 us for 700 rows of
// 6144 columns, 33 for 8192, which is all but the traffic).  Four Llama-3 layers, us without and with: 700 rows 1410 : 1391, 4 x
// 2048 11279 : 11199, 8 x 512 5280 : 5220, 1500 2500 : 2467; the same bits.
// It needs tiles of 128 columns and all of K; where a split of K is the faster product by more than that pass takes, and
// for all else: -3 with nothing launched.
extern "C" int dnn_gemm_bf16_qkv_rope(const void* A, int lda, const void* W, int ldw, float eps, float* stats, void* q, void* kc,
                                      void* vc, const int* pos, int B, int T, int H, int Hkv, int hd, int S, int K,
                                      const float* cosT, const float* sinT, long long ws_bytes, hipStream_t st) {
  const int M = B * T, N = (H + 2 * Hkv) * hd;
  if (M <= 0 || cosT == nullptr || sinT == nullptr) return -1;
  if (hd != 128 || K % 64 != 0 || M >= (1 << 24) || !dma_rows(A, lda, W, ldw) || !mid_narrow(lda, ldw) || tail_split_cols(M, N) != 0 ||
      (((uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc | (uintptr_t)cosT | (uintptr_t)sinT) & 15) != 0)
    return -3;
  MidPlan plan = mid_plan(M, N, K, 0, MID_BF16);
  if (g_mid_tile >= 0) plan = {g_mid_tile, 1, 0.f, 0};
  else if (g_gemm_tile == 256) plan = {-1, 1, 0.f, 0};
  else if (g_gemm_tile != 0 ||
           plan.us > mid_plan(M, N, K, ws_bytes, MID_BF16).us + 3.f + (float)M * N * 4.f / 5.5e6f) return -3;
  if (plan.tile == 0 || plan.tile == 1 || (plan.tile < 0 && M < 256)) return -3;
  QkvScatter sc{(bf16_t*)q, (bf16_t*)kc, (bf16_t*)vc, pos, T, H, Hkv, 7, S, 1.0f / (float)T, 0, cosT, sinT};
  if (const int rc = dnn_row_stats(A, lda, stats, M, K, eps, 1, st)) return rc;
  const float2* rs = reinterpret_cast<const float2*>(stats);
  const int n = plan.tile < 0 ? N : plan.cols;  // columns of the 256 x 256 kernel
  if (n > 0) {
    hipLaunchKernelGGL((gemm_bf16_256_kernel<ACT_NONE, false, true, 2, false, true>),
                       dim3((M + BG_M - 1) / BG_M * ((n + BG_N - 1) / BG_N)), dim3(512), 0, st, (const bf16_t*)A, lda,
                       (const bf16_t*)W, ldw, q, hd, (const float*)nullptr, (const bf16_t*)nullptr, 0, M, n, K, 0, rs,
                       (const float*)nullptr, sc);
    if (const hipError_t e = hipGetLastError()) return (int)e;
  }
  if (n == N) return 0;
  sc.c_off = n;
  const MidArgs a{{q, nullptr, nullptr, hd, 0, M, N - n, ACT_NONE, 0}, (const bf16_t*)A, (const bf16_t*)W + (size_t)n * ldw, rs,
                  nullptr, nullptr, nullptr, eps, 1, nullptr, lda, ldw, K, 1};
  return mid_launch(plan.tile, a, &sc, st);
}

// fp8 (W8A8) c_attn with the QKV scatter epilogue: A8 / sa the per-token
// e4m3 activations (layernorm_q8), W8 / sw the e4m3 weight, Kb its row bytes.
extern "C" int dnn_gemm_fp8_qkv_scatter(const void* A8, const float* sa, const void* W8, const float* sw,
                                        const float* bias, void* q, void* kc, void* vc, const int* pos, int B, int T,
                                        int H, int Hkv, int hd, int S, int Kb, hipStream_t st) {
  const int M = B * T, N = (H + 2 * Hkv) * hd;
  if (Kb % 128 != 0 || M <= 0 || hd % 8 != 0 || sa == nullptr || sw == nullptr) return -1;
  if (N % 32 != 0 || M < 256 || ((uintptr_t)bias & 15) != 0 || !bg_narrow(Kb / 2)) return -3;
  const int tiles = ((M + BG_M - 1) / BG_M) * ((N + BG_N - 1) / BG_N);
  if ((hd & (hd - 1)) != 0 || M >= (1 << 24)) return -3;
  QkvScatter sc{(bf16_t*)q, (bf16_t*)kc, (bf16_t*)vc, pos, T, H, Hkv, __builtin_ctz(hd), S, 1.0f / (float)T};
  const int Na = tail_split_cols(M, N, true);  // GPT-2 XL c_attn (N = 4800): 2304 + 256 half tiles
  if (Na > 0) {
    const int ntm256 = (M + BG_M - 1) / BG_M, Nt = N - Na;
    hipLaunchKernelGGL((gemm_fp8_256_kernel<ACT_NONE, true>), dim3(ntm256 * (Na / 256)), dim3(512), 0, st,
                       (const uint8_t*)A8, sa, (const uint8_t*)W8, sw, (bf16_t*)q, hd, bias, (const bf16_t*)nullptr, 0,
                       M, Na, Kb, sc);
    QkvScatter tail = sc;
    tail.c_off = Na;
    hipLaunchKernelGGL((gemm_fp8_256_kernel<ACT_NONE, true, 1>), dim3(ntm256 * ((Nt + 127) / 128)), dim3(512), 0,
                       st, (const uint8_t*)A8, sa, (const uint8_t*)W8 + (size_t)Na * Kb, sw + Na, (bf16_t*)q, hd, bias,
                       (const bf16_t*)nullptr, 0, M, Nt, Kb, tail);
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL((gemm_fp8_256_kernel<ACT_NONE, true>), dim3(tiles), dim3(512), 0, st, (const uint8_t*)A8, sa,
                     (const uint8_t*)W8, sw, (bf16_t*)q, hd, bias, (const bf16_t*)nullptr, 0, M, N, Kb, sc);
  return (int)hipGetLastError();
}

// fp8 256^2 GEMM (see gemm_fp8_256_kernel); Kb = row bytes of A and W (multiple
// of 128), sa per-row, sw per-column scales.  Called by dnn_gemm_fp8 when the
// 256^2 tiles fill the chip.  -3: rows too wide for the tiles' 32-bit row offsets.
extern "C" int dnn_gemm_fp8_256(const void* A, const float* sa, const void* W, const float* sw, void* C, int ldc,
                                const float* bias, const void* R, int ldr, int M, int N, int Kb, int act,
                                hipStream_t st) {
  if (Kb % 128 != 0 || M <= 0 || N <= 0 || sa == nullptr || sw == nullptr) return -1;
  if (is_glu(act) && N % 16 != 0) return -1;
  if (!bg_narrow(Kb / 2)) return -3;
  const int tiles = ((M + BG_M - 1) / BG_M) * ((N + BG_N - 1) / BG_N);
  // tail split (as launch_gemm's): GPT-2 XL O / c_proj (N = 1600) and c_fc (N = 6400) at M = 32768
  const int Na = !is_glu(act) ? tail_split_cols(M, N, true) : 0;
  const int ntm256 = (M + BG_M - 1) / BG_M, Nt = N - Na;
#define F8L(a)                                                                                                    \
  if (act == a) {                                                                                                 \
    if (Na > 0) {                                                                                                 \
      hipLaunchKernelGGL((gemm_fp8_256_kernel<a>), dim3(ntm256 * (Na / 256)), dim3(512), 0, st,                   \
                         (const uint8_t*)A, sa, (const uint8_t*)W, sw, (bf16_t*)C, ldc, bias, (const bf16_t*)R,    \
                         ldr, M, Na, Kb);                                                                         \
      hipLaunchKernelGGL((gemm_fp8_256_kernel<a, false, 1>), dim3(ntm256 * ((Nt + 127) / 128)), dim3(512), 0, st, \
                         (const uint8_t*)A, sa, (const uint8_t*)W + (size_t)Na * Kb, sw + Na, (bf16_t*)C + Na,    \
                         ldc, bias != nullptr ? bias + Na : nullptr,                                              \
                         R != nullptr ? (const bf16_t*)R + Na : nullptr, ldr, M, Nt, Kb);                         \
      return (int)hipGetLastError();                                                                              \
    }                                                                                                             \
    hipLaunchKernelGGL((gemm_fp8_256_kernel<a>), dim3(tiles), dim3(512), 0, st, (const uint8_t*)A, sa,            \
                       (const uint8_t*)W, sw, (bf16_t*)C, ldc, bias, (const bf16_t*)R, ldr, M, N, Kb);            \
    return (int)hipGetLastError();                                                                                \
  }
  F8L(ACT_NONE) F8L(ACT_RELU) F8L(ACT_GELU) F8L(ACT_SILU_MUL)
#undef F8L
  return -2;
}

// Tile of gemm_mid.h for an MX product, -1: the 256 x 256 kernel.  A K-tile of 128
// bytes takes a tile as long as the bf16 kernel's K-tile of 64: the same estimate.
static int mx_mid_tile(int M, int N, int Kb, bool quant) {
  if (g_gemm_tile != 0 || Kb >= 1 << 24) return -1;  // the small tiles address a tile's rows with 32 bits
  if (g_mid_tile >= 0 && g_mid_tile < 5) return quant && g_mid_tile < 2 ? 2 : g_mid_tile;
  return mid_plan(M, N, Kb / 2, 0, quant ? MID_MX_QUANT : MID_MX).tile;
}

// MX-scaled W8A8 GEMM: A8 [M][Kb]
// e4m3 with e8m0 scales sx per (row, 128-column K-tile) (common.h mx_index;
// dnn_quant_fp8_mx / dnn_layernorm_q8_mx / a QOUT epilogue write them), W8 /
// sw per-channel e4m3.  qo != nullptr (act GELU): the output is quantised in
// the epilogue instead (QOUT: qo [M][ldq] e4m3 with scales sxo, kpo columns,
// the next GEMM's MX input) and C is not written.  -3: not a 256^2 shape (the
// caller keeps the per-row path).
extern "C" int dnn_gemm_fp8_mx(const void* A8, const void* sx, const void* W8, const float* sw, void* C, int ldc,
                               const float* bias, const void* R, int ldr, int M, int N, int Kb, int act, void* qo,
                               int ldq, void* sxo, int kpo, hipStream_t st) {
  if (Kb % 128 != 0 || M <= 0 || N <= 0 || sx == nullptr || sw == nullptr) return -1;
  if (M < 256 || N < 256 || !bg_narrow(Kb / 2)) return -3;
  if (qo != nullptr && (act != ACT_GELU || sxo == nullptr || kpo % 128 != 0 || kpo < N || ldq < kpo ||
                        (ldq & 7) != 0 || ((uintptr_t)qo & 7) != 0))
    return -1;
  if (is_glu(act) && N % 16 != 0) return -1;
  const int tiles = ((M + BG_M - 1) / BG_M) * ((N + BG_N - 1) / BG_N);
  const uint32_t* sxw = reinterpret_cast<const uint32_t*>(sx);
  const int mid = mx_mid_tile(M, N, Kb, qo != nullptr);
  if (mid >= 0 && act <= ACT_SILU_MUL) {
    const Mid8Args a{{C, bias, (const bf16_t*)R, ldc, ldr, M, N, act, 0}, (const uint8_t*)A8, (const uint8_t*)W8, sxw, sw,
                     (uint8_t*)qo, (uint8_t*)sxo, Kb, ldq, kpo};
    return mid8_launch(mid, a, nullptr, st);
  }
  if (qo != nullptr) {
    hipLaunchKernelGGL((gemm_fp8_256_kernel<ACT_GELU, false, 2, true, true>), dim3(tiles), dim3(512), 0, st,
                       (const uint8_t*)A8, (const float*)nullptr, (const uint8_t*)W8, sw, (bf16_t*)nullptr, 0, bias,
                       (const bf16_t*)nullptr, 0, M, N, Kb, QkvScatter{}, sxw, (uint8_t*)qo, ldq, (uint8_t*)sxo, kpo);
    return (int)hipGetLastError();
  }
#define F8M(a)                                                                                                      \
  if (act == a) {                                                                                                   \
    hipLaunchKernelGGL((gemm_fp8_256_kernel<a, false, 2, true>), dim3(tiles), dim3(512), 0, st, (const uint8_t*)A8, \
                       (const float*)nullptr, (const uint8_t*)W8, sw, (bf16_t*)C, ldc, bias, (const bf16_t*)R, ldr, M, \
                       N, Kb, QkvScatter{}, sxw);                                                                   \
    return (int)hipGetLastError();                                                                                  \
  }
  F8M(ACT_NONE) F8M(ACT_RELU) F8M(ACT_GELU) F8M(ACT_SILU_MUL)
#undef F8M
  return -2;
}

// fp8 c_attn with the QKV scatter epilogue on MX-scaled activations
// (dnn_layernorm_q8_mx): as dnn_gemm_fp8_qkv_scatter, sx instead of sa.
extern "C" int dnn_gemm_fp8_qkv_scatter_mx(const void* A8, const void* sx, const void* W8, const float* sw,
                                           const float* bias, void* q, void* kc, void* vc, const int* pos, int B, int T,
                                           int H, int Hkv, int hd, int S, int Kb, hipStream_t st) {
  const int M = B * T, N = (H + 2 * Hkv) * hd;
  if (Kb % 128 != 0 || M <= 0 || hd % 8 != 0 || sx == nullptr || sw == nullptr) return -1;
  if (N % 32 != 0 || M < 256 || N < 256 || ((uintptr_t)bias & 15) != 0 || !bg_narrow(Kb / 2)) return -3;
  if ((hd & (hd - 1)) != 0 || M >= (1 << 24)) return -3;
  QkvScatter sc{(bf16_t*)q, (bf16_t*)kc, (bf16_t*)vc, pos, T, H, Hkv, __builtin_ctz(hd), S, 1.0f / (float)T};
  const int mid = mx_mid_tile(M, N, Kb, false);
  if (mid >= 0) {
    const Mid8Args a{{q, bias, nullptr, hd, 0, M, N, ACT_NONE, 0}, (const uint8_t*)A8, (const uint8_t*)W8,
                     reinterpret_cast<const uint32_t*>(sx), sw, nullptr, nullptr, Kb, 0, 0};
    return mid8_launch(mid, a, &sc, st);
  }
  const int tiles = ((M + BG_M - 1) / BG_M) * ((N + BG_N - 1) / BG_N);
  hipLaunchKernelGGL((gemm_fp8_256_kernel<ACT_NONE, true, 2, true>), dim3(tiles), dim3(512), 0, st, (const uint8_t*)A8,
                     (const float*)nullptr, (const uint8_t*)W8, sw, (bf16_t*)q, hd, bias, (const bf16_t*)nullptr, 0, M,
                     N, Kb, sc, reinterpret_cast<const uint32_t*>(sx));
  return (int)hipGetLastError();
}
#endif  // DNN_DECODER_ONLY
