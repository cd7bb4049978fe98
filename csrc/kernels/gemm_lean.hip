// Decode projections of up to 64 rows whose slices of K lie in registers ("lean"):
//   C[M,N] = epi(A[M,K] . W[N,K]^T), W in fragment order, bf16 or e4m3 (W8A16).
//
// At these sizes a launch in a decode step costs its start, one round trip for what it
// reads and the code itself: every launch begins with a cold instruction cache, and 4 to 5
// KB of a kernel that is laid out for every shape are 1 to 2 us of fetches (GPT-2's
// 2304 x 768 of 64 rows: 5.0 us launched over and over by itself, 7.4 in its step).  So
// the shape is compile-time down to the chunk: NW waves of NB batches of CB chunks are K, D
// batches of a wave in flight straight to registers (a wave's slices of A and W are its own,
// nothing is shared before the sums meet), one barrier, and the waves that finish a tile
// have its epilogue's operands by then: 1.2 to 5.8 KB, of which the e4m3 c_fc's was 28.
//
// A wave reads its slice of every row whole and turns it to fragments in LDS of its own.  Read as fragments, a load is 16
// pieces of 64 bytes of 16 rows, half a line each: GPT-2's step of 64 rows is 501 us so, 482 through LDS, XL's 326 and 310.
//
// us a launch in the step, GPT-2 (bf16) of 64 rows 2304 x 768 7.4 -> 4.6, 3072 x 768 7.0 -> 5.0, 768 x 768 5.4
// -> 4.8, 768 x 3072 7.1 -> 4.9; XL (e4m3) of 64 rows 4800 x 1600 10.7 -> 6.3, 6400 x 1600 11.2 -> 6.6,
// 1600 x 1600 5.8 -> 4.9, 1600 x 6400 11.6 -> 7.8.  Batches in flight, waves and their chunks matter
// little (within 1 % of the step from one batch to all of K, 4 to 8 waves); tiles do: lean_gemm.
#include <utility>

#include "gemm_lean.h"

namespace dnn {

template <int NW, int CB, int NB, int D, int MT, int NT, bool W8, int NORM, int ACT, bool RES>
struct Lean {
  static constexpr int K = NW * CB * NB * (W8 ? 64 : 32), ROWS = 16 * MT;
  static constexpr int LPR = NW * 64 / ROWS;  // threads a row for the merge of its statistics
  static constexpr int TPR = LPR >= 64 ? 64 : LPR >= 32 ? 32 : LPR >= 16 ? 16 : LPR >= 8 ? 8 : 4;
  static constexpr int SPT = (K / 16 + TPR - 1) / TPR;
  // a batch of a wave's rows on its way through LDS: pieces of 16 bytes a row, and an odd number of them between rows
  static constexpr int PB = CB * (W8 ? 8 : 4), STRIDE = (PB + 1) * 16, NX = MT * PB / 4, WAVE = ROWS * STRIDE, LDS = NW * WAVE;
};

// ST: W goes past the L2's order of use (bytes read once; us a step of Llama-3's 32 rows, QKV with and without 399 and 414).
template <int NW, int CB, int NB, int D, int MT, int NT, bool W8, int NORM, int ACT, bool RES, bool ST>
__global__ __launch_bounds__(NW * 64) void gemm_lean_kernel(LeanArgs p) {
  using L = Lean<NW, CB, NB, D, MT, NT, W8, NORM, ACT, RES>;
  constexpr int AU = W8 ? 2 : 1, ACH = 64 * AU, TS = MT * NT, CH = CB * NB, TW = (TS + NW - 1) / NW;
  static_assert(D <= NB, "batches in flight");
  extern __shared__ __attribute__((aligned(16))) char lean_rows[];
  __shared__ f32x4 red[NW][TS][64];
  __shared__ float2 st[NORM == NORM_LN ? L::ROWS : 1];
  __shared__ float ss[NORM == NORM_RMS ? NW : 1][NORM == NORM_RMS ? L::ROWS : 1];
  // the row tiles of a column tile follow each other on one XCD
  const int n0 = (blockIdx.z * 8 + blockIdx.x) * (16 * NT), m0 = blockIdx.y * (16 * MT);
  if (n0 >= p.N) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, c4 = lane >> 4;
  float2 rp[L::SPT], rp0;
  const int srow = tid / L::TPR, sub = tid % L::TPR;
  if constexpr (NORM == NORM_LN) {
    const float2* q = p.rs_in + (size_t)min(m0 + min(srow, L::ROWS - 1), p.M - 1) * p.rs_in_ld;
    rp0 = q[0];
#pragma unroll
    for (int i = 0; i < L::SPT; ++i) rp[i] = q[min(sub + i * L::TPR, L::K / 16 - 1)];
  }
  i32x4 xr[D][L::NX], wv[D][NT][CB];
  const uint8_t* xp[L::NX];
  const uint8_t* wp[NT];
#pragma unroll
  for (int i = 0; i < L::NX; ++i) {
    const int q = lane + i * 64;
    xp[i] = p.A + (size_t)min(m0 + q / L::PB, p.M - 1) * p.lda_b + wave * (CH * ACH) + q % L::PB * 16;
  }
#pragma unroll
  for (int j = 0; j < NT; ++j)
    wp[j] = p.W + ((size_t)min(n0 / 16 + j, p.N / 16 - 1) * (NW * CH) + wave * CH) * 1024 + lane * 16;
  auto load = [&](auto bc) __attribute__((always_inline)) {
    constexpr int b = decltype(bc)::value, d = b % D;
#pragma unroll
    for (int i = 0; i < L::NX; ++i) xr[d][i] = *reinterpret_cast<const i32x4*>(xp[i] + b * (CB * ACH));
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int u = 0; u < CB; ++u) {
        const i32x4* q = reinterpret_cast<const i32x4*>(wp[j] + (b * CB + u) * 1024);
        wv[d][j][u] = ST ? __builtin_nontemporal_load(q) : *q;
      }
  };
  [&]<int... B>(std::integer_sequence<int, B...>) __attribute__((always_inline)) {
    (load(std::integral_constant<int, B>{}), ...);
  }(std::make_integer_sequence<int, D>{});
  // the tiles that this wave finishes, and their operands (absent ones from a dummy address)
  f32x4 cs[TW], bs[TW], sc[TW];
  bf16x4 rr[TW];
  int n[TW], m[TW];
#pragma unroll
  for (int i = 0; i < TW; ++i) {
    const int tile = min(wave + i * NW, TS - 1);
    n[i] = min(n0 + tile / MT * 16, p.N - 16) + c4 * 4;
    m[i] = m0 + tile % MT * 16 + r16;
    bs[i] = *reinterpret_cast<const f32x4*>(p.bias != nullptr ? p.bias + n[i] : reinterpret_cast<const float*>(p.W));
    if constexpr (NORM == NORM_LN) cs[i] = *reinterpret_cast<const f32x4*>(p.colsum + n[i]);
    if constexpr (W8) sc[i] = *reinterpret_cast<const f32x4*>(p.sw + n[i]);
    if constexpr (RES) rr[i] = *reinterpret_cast<const bf16x4*>(p.R + (size_t)min(m[i], p.M - 1) * p.ldr + n[i]);
  }
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NORM == NORM_LN) {
    const float2 mr = rowstat_merge<NORM_LN, L::TPR, L::SPT>(rp, rp0, sub, L::K, p.eps);
    if (sub == 0 && srow < L::ROWS) st[srow] = mr;
  }
  f32x4 acc[NT][MT];
  float sq[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    sq[t] = 0.f;
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  char* mine = lean_rows + wave * L::WAVE;
  const char* from = mine + r16 * L::STRIDE + c4 * (16 * AU);
  auto comp = [&](auto bc) __attribute__((always_inline)) {
    constexpr int d = decltype(bc)::value % D;
#pragma unroll
    for (int i = 0; i < L::NX; ++i) {
      const int q = lane + i * 64;
      *reinterpret_cast<i32x4*>(mine + q / L::PB * L::STRIDE + q % L::PB * 16) = xr[d][i];
    }
    // other lanes read what this one stored, and the next batch lies where this one did: the fences keep both orders (a
    // wave's LDS operations run in them)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int u = 0; u < CB; ++u) {
      bf16x8 a[MT][AU];
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int h = 0; h < AU; ++h)
          a[t][h] = *reinterpret_cast<const bf16x8*>(from + t * (16 * L::STRIDE) + u * ACH + h * 16);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        bf16x8 w[AU];
        if constexpr (W8) w8_to_bf16(wv[d][j][u], w[0], w[AU - 1]);
        else w[0] = __builtin_bit_cast(bf16x8, wv[d][j][u]);
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int h = 0; h < AU; ++h)
            acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[h], a[t][h], acc[j][t], 0, 0, 0);
      }
      if constexpr (NORM == NORM_RMS) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
          for (int h = 0; h < AU; ++h) {
            const i32x4 v4 = __builtin_bit_cast(i32x4, a[t][h]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const bf16x2v v = __builtin_bit_cast(bf16x2v, (uint32_t)v4[i]);
              sq[t] = __builtin_amdgcn_fdot2_f32_bf16(v, v, sq[t], false);
            }
          }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  [&]<int... B>(std::integer_sequence<int, B...>) __attribute__((always_inline)) {
    (([&]() __attribute__((always_inline)) {
       comp(std::integral_constant<int, B>{});
       __builtin_amdgcn_sched_barrier(0);
       if constexpr (B + D < NB) {
         load(std::integral_constant<int, B + D>{});
         __builtin_amdgcn_sched_barrier(0);
       }
     }()),
     ...);
  }(std::make_integer_sequence<int, NB>{});
  if constexpr (NORM == NORM_RMS) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const float s = add32(add16(sq[t]));
      if (lane < 16) ss[wave][t * 16 + lane] = s;
    }
  }
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int t = 0; t < MT; ++t) red[wave][j * MT + t][lane] = acc[j][t];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TW; ++i) {
    const int tile = wave + i * NW, nt = n0 + tile / MT * 16;
    if (tile >= TS || nt >= p.N) return;
    f32x4 v[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) v[w] = red[w][tile][lane];
    f32x4 y = v[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) y += v[w];
    if constexpr (W8) y *= sc[i];
    if constexpr (NORM == NORM_LN) {
      const float2 mr = st[m[i] - m0];
      y = mr.y * (y - mr.x * cs[i]);
    }
    if constexpr (NORM == NORM_RMS) {
      float q = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) q += ss[w][m[i] - m0];
      y *= rsqrtf(q * (1.f / L::K) + p.eps);
    }
    if (p.bias != nullptr) y += bs[i];
    if constexpr (ACT == ACT_GELU) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = gelu_erf(y[e]);
    }
    if constexpr (RES) {
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] += bf2f_s(rr[i][e]);
    }
    if constexpr (is_glu(ACT)) {  // 8 gate columns, then their 8 up columns
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[e]), __float_as_uint(y[e]), false, false);
        v[e] = glu_gate<ACT>(__uint_as_float(h[0])) * __uint_as_float(h[1]);
      }
      if (lane < 32 && m[i] < p.M)
        *reinterpret_cast<uint2*>(p.C + (size_t)m[i] * p.ldc + nt / 2 + c4 * 4) = make_uint2(pack2bf(v[0], v[1]), pack2bf(v[2], v[3]));
      continue;
    }
    const uint2 o = make_uint2(pack2bf(y[0], y[1]), pack2bf(y[2], y[3]));
    if (m[i] < p.M) *reinterpret_cast<uint2*>(p.C + (size_t)m[i] * p.ldc + n[i]) = o;
    if (RES && p.rs_out != nullptr)
      epi_rowstat16(f32x4{__uint_as_float(o.x << 16), __uint_as_float(o.x & 0xffff0000u), __uint_as_float(o.y << 16),
                          __uint_as_float(o.y & 0xffff0000u)},
                    m[i], nt, p.M, p.N, p.rs_out, p.rs_out_ld, lane);
  }
}

template <int NW, int CB, int NB, int D, int MT, int NT, bool W8, int NORM, int ACT, bool RES, bool ST = false>
static void lean_launch(const LeanArgs& p, hipStream_t st) {
  const int cols = (p.N / 16 + NT - 1) / NT;
  hipLaunchKernelGGL((gemm_lean_kernel<NW, CB, NB, D, MT, NT, W8, NORM, ACT, RES, ST>),
                     dim3(8, (p.M + 16 * MT - 1) / (16 * MT), (cols + 7) / 8), dim3(NW * 64),
                     (Lean<NW, CB, NB, D, MT, NT, W8, NORM, ACT, RES>::LDS), st, p);
}

// False, nothing done, where the shape is not one of those laid out.
template <int ACT, int NORM, bool W8>
static bool lean_gemm(const LeanArgs& p, int nch, hipStream_t st) {
  constexpr bool RES = NORM == NORM_NONE;
  if constexpr (!(NORM == NORM_LN && (ACT == ACT_NONE || ACT == ACT_GELU)) && !(RES && ACT == ACT_NONE) &&
                !(NORM == NORM_RMS && (ACT == ACT_NONE || ACT == ACT_SILU_MUL) && !W8)) {
    return false;
  } else {
    // The tiles, from whole steps (us; GPT-2 behind 100 tokens, XL behind 64, Llama-3 of 4 layers behind 100):
    //   GPT-2 QKV, c_fc        16 rows 1 x 1 tiles 251, 1 x 2 259, 2 x 2 266; 32 rows 311, 307, 321; 64 rows 358, 352, 351
    //   its O, c_proj          1 x 1 at every number of rows (64 rows, 1 x 2 and 2 x 1: 354; c_proj 367)
    //   XL e4m3 QKV, c_fc      8 rows 1 x 2 tiles 138, 1 x 4 142; 24 rows 181, 159; 64 rows 266, 232, 2 x 4 230
    //   its O, c_proj          48 rows 1 x 1 213, 212, 1 x 2 211, 211; 8 rows 138, 138; 139, 146
    //   Llama-3 QKV            16 rows 1 x 2 tiles 375, 1 x 3 378, 2 x 3 388; 32 rows 416, 398, 407, 2 x 2 399; 64 rows 514,
    //                          502, 481, 504 (before: 383, 414, 541)
    //   its O                  32 rows 1 x 1 424, 2 x 1 406; 64 rows 550, on 8 waves 523, on 4 520
    //   its gate | up          8 rows 1 x 1 343 (before: 335), 16 rows 371 (383), 1 x 2 381; 32 rows 2 x 2 429 (gemm_stream 414)
    //   its down               2 x 1 32 rows 419, 64 rows 603, 4 x 1 583 (gemm_stream 414, 541)
    // Two rows or fewer of GPT-2's widths: decode_row.hip.  These are the widths of GPT-2, XL in e4m3 and Llama-3 8B; GPT-2 medium
    // and large, XL in bf16 and others in e4m3 have not been laid out or measured, and run on the general kernels.
    auto al = [](const void* x, int a) { return ((uintptr_t)x & (a - 1)) == 0; };
    if (p.W == nullptr || p.M < 1 || p.M > 64 || p.N % 16 != 0 || p.N > (RES ? 4096 : is_glu(ACT) ? 65536 : 8192) || (is_glu(ACT) && p.bias != nullptr) || (p.R != nullptr) != RES ||
        (!RES && p.rs_out != nullptr) || p.lda_b % 16 != 0 || p.ldc % 4 != 0 || !al(p.A, 16) || !al(p.C, 8) ||
        !al(p.bias, 16) || !al(p.colsum, 16) || !al(p.sw, 16) || (RES && (p.ldr % 4 != 0 || !al(p.R, 8))) ||
        (NORM == NORM_LN && (p.rs_in == nullptr || p.colsum == nullptr)))
      return false;
#define LEAN(NWV, CBV, NBV, DV, MTV, NTV) lean_launch<NWV, CBV, NBV, DV, MTV, NTV, W8, NORM, ACT, RES>(p, st)
#define LEAN_ONCE(NWV, CBV, NBV, DV, MTV, NTV) lean_launch<NWV, CBV, NBV, DV, MTV, NTV, W8, NORM, ACT, RES, true>(p, st)
    const int M = p.M;
    if constexpr (!W8 && NORM == NORM_LN) {
      if (nch != 24) return false;
      if (M <= 16) LEAN(4, 6, 1, 1, 1, 1);
      else if (M <= 48) LEAN(4, 6, 1, 1, 1, 2);
      else LEAN(4, 6, 1, 1, 2, 2);
    } else if constexpr (!W8 && NORM == NORM_RMS && is_glu(ACT)) {
      if (nch != 128 || M <= 8 || M > 16) return false;
      LEAN_ONCE(4, 8, 4, 2, 1, 1);
    } else if constexpr (!W8 && NORM == NORM_RMS) {
      // Fewer columns leave CUs idle, each wave with an eighth of K to itself; more of them are a second round.  us a launch, general :
      // this (two small launches of 8 with it), 16 rows N 4096 13.4 : 14.5, 4608 15.6 : 13.4, 8192 17.5 : 16.7; 1 row 4608
      // 15.1 : 14.3, 6144 15.8 : 16.2 (in a step of 4 layers 4 to 12 less), 8192 17.4 : 19.2; 32 rows 4096 14.9 : 15.9, 4608 19.9 : 16.4,
      // 6144 20 : 16.9, 6656 21 : 25; 48 rows 2560 14.5 : 17, 3072 20 : 17.7, 6144 25.6 : 19.3, 6656 26 : 28; 64 rows 2048 14.2 : 17.1,
      // 2560 20.3 : 17.3, 8192 31 : 29.5.
      if (nch != 128 || p.N <= (M <= 32 ? 4096 : M <= 48 ? 2560 : 2048) || (p.N > 6144 && (M <= 8 || (M > 16 && M <= 48))))
        return false;
      if (M <= 16) LEAN_ONCE(8, 4, 4, 2, 1, 2);
      else if (M <= 32) LEAN_ONCE(8, 4, 4, 2, 1, 3);
      else LEAN_ONCE(8, 4, 4, 2, 2, 3);
    } else if constexpr (!W8) {
      if (nch == 24) LEAN(4, 6, 1, 1, 1, 1);
      else if (nch == 96) LEAN(4, 6, 4, 2, 1, 1);
      else if (nch != 128 || (M > 32 && p.N <= 1024)) return false;  // 64 rows, 64 columns 11.1 : 12.0, 768 12.5 : 12.9, 1280 13.8 : 13.0
      else if (M <= 16) LEAN_ONCE(8, 4, 4, 4, 1, 1);
      else if (M <= 32) LEAN(8, 4, 4, 3, 2, 1);
      else LEAN_ONCE(4, 8, 4, 2, 2, 1);
    } else if constexpr (NORM == NORM_LN) {
      if (nch != 25) return false;
      if (M <= 16) LEAN(5, 5, 1, 1, 1, 2);
      else if (M <= 48) LEAN(5, 1, 5, 2, 1, 4);
      else LEAN(5, 1, 5, 2, 2, 4);
    } else {
      if (nch == 25) {
        if (M <= 32) LEAN(5, 5, 1, 1, 1, 1);
        else LEAN(5, 1, 5, 3, 1, 2);
      } else if (nch == 100) {
        if (M <= 32) LEAN(10, 1, 10, 4, 1, 1);
        else LEAN(10, 1, 10, 2, 1, 2);
      } else {
        return false;
      }
    }
#undef LEAN
#undef LEAN_ONCE
    return true;
  }
}

bool dnn_gemm_lean(const LeanArgs& p, int nch, int act, int norm, bool w8, hipStream_t st) {
#define LG(A, N)                                                                                  \
  if (act == A && norm == N) return w8 ? lean_gemm<A, N, true>(p, nch, st) : lean_gemm<A, N, false>(p, nch, st);
  LG(ACT_NONE, NORM_LN) LG(ACT_GELU, NORM_LN) LG(ACT_NONE, NORM_NONE) LG(ACT_NONE, NORM_RMS) LG(ACT_SILU_MUL, NORM_RMS)
#undef LG
  return false;
}

}  // namespace dnn
