// bf16 GEMM for row counts between decode and large prefill (65 to a few thousand
// rows, where 256 x 256 tiles leave most CUs idle): tiles of 64 to 256 rows with a
// deep LDS pipeline, and the K range over several workgroups where the tiles alone
// do not fill the chip (gemm_mid.hip mid_plan chooses).
#pragma once
#include "common.h"
#include "gemm_epilogue.h"
#include "gemm_mid_api.h"
#include "gemm_tile.h"

namespace dnn {

template <int BM_, int BN_, int WM_, int WN_, int S_, int PW_ = 0>
struct MidTile {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, S = S_, PW = PW_;
  static constexpr int CW = WM * WN;                           // waves that multiply
  static constexpr int NW = PW ? PW : CW;                      // waves that stage: PW > 0, others than those
  static constexpr int THREADS = (CW + PW) * 64;
  static constexpr int I = BM / WM / 16, J = BN / WN / 16;      // 16 x 16 tiles of a wave
  static constexpr int PA = BM / 8 / NW, PB = BN / 8 / NW;      // 1-KiB pieces a wave stages of either operand
  static constexpr int STAGE = (BM + BN) * 128;                 // bytes of one K-tile of both operands
  static_assert(J % 2 == 0 && PA >= 1 && PB >= 1 && S >= 2, "");
};

// The tile table (costs: gemm_mid.hip MID).  Heights of 192 and 96 rows: between the powers of two a
// row count leaves half a tile empty or a chip half full, and 192 x 128 has room for four K-tiles where 256 x 128
// has for three.  us, the best of the others : these: 700 x 6144 x 4096 51.8 : 43.4, 1500 x 4096 x 4096 57.0 : 49.9, 1400 x
// 3072 x 768 17.4 : 14.9, 700 x 4096 x 14336 in 2 95.2 : 86; 96 rows: 380 x 6144 x 4096 38.3 : 35.0, 700 x 4096 x 4096 34.3 : 33.0.
// (192 x 64, 128 x 192 and 192 x 192 are best nowhere by more than 2 %.)
// 64 x 64: five K-tiles are what two workgroups a CU have room for.  us with four : five: 64 x 64 x 3072 11.1 : 10.6, 1071 x
// 768 x 3072 13.5 : 12.8, 700 x 6144 x 4096 72.2 : 71.0; six and more (one workgroup a CU) gain nothing over five.  Exactly half
// a CU's LDS: a kernel that keeps more beside its K-tiles needs a tile of its own (gemm_mid_fp8.hip).
typedef MidTile<64, 64, 2, 2, 5> Mid0;
typedef MidTile<128, 64, 2, 2, 6> Mid1;
typedef MidTile<128, 128, 2, 4, 4> Mid2;
typedef MidTile<256, 128, 4, 2, 3> Mid3;
typedef MidTile<128, 256, 2, 4, 3> Mid4;
typedef MidTile<192, 128, 4, 2, 4> Mid5;
typedef MidTile<96, 128, 2, 2, 5> Mid6;
// The same where K is split: four waves that only stage (mid_stage), so that no product
// waits for a request to be taken.  us with and without, parts and their sum: 512 x 4096 x
// 18432 in 4 77.8 : 83.8, 500 x 4096 x 21504 in 4 89.4 : 94.0; split 192 x 128 tiles 3 to 5 %.  Smaller tiles gain nothing, and whole ones lack the registers for their epilogue.
template <class T>
struct MidSplit {
  typedef T type;
};
template <>
struct MidSplit<Mid3> {
  typedef MidTile<256, 128, 4, 2, 3, 4> type;
};
template <>
struct MidSplit<Mid4> {
  typedef MidTile<128, 256, 2, 4, 3, 4> type;
};
template <>
struct MidSplit<Mid5> {
  typedef MidTile<192, 128, 4, 2, 4, 4> type;
};

// s_waitcnt operand: at most `vm` vector-memory and `lgkm` LDS operations outstanding
constexpr int wait_imm(int vm, int lgkm) { return (vm & 15) | (vm >> 4) << 14 | 7 << 4 | lgkm << 8; }

// Columns n .. n + 3 of a vector of N.
__device__ __forceinline__ f32x4 mid_cols(const float* b, int n, int N) {
  if (n + 3 < N && (reinterpret_cast<uintptr_t>(b) & 15) == 0) return *reinterpret_cast<const f32x4*>(b + n);
  f32x4 v;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = n + r < N ? b[n + r] : 0.f;
  return v;
}

template <int ACT>
__device__ __forceinline__ f32x4 mid_act(f32x4 v, const f32x2& xc) {
  if constexpr (ACT == ACT_GELU) {
    const f32x2 g0 = gelu_erf2(f32x2{v[0], v[1]}), g1 = gelu_erf2(f32x2{v[2], v[3]});
    return f32x4{g0[0], g0[1], g1[0], g1[1]};
  }
  act_xielu<ACT>(v, xc);
  if constexpr (ACT == ACT_RELU) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r], 0.f);
  }
  return v;
}

// Whether a wave's whole columns leave as pairs of 16-byte stores (uniform).
__device__ __forceinline__ bool mid_pair(const MidRows& p, int nw, int J) {
  return !p.f32 && epi_vec_ok(p.C, p.ldc, p.bias, p.R, p.ldr) && epi_pair_ok(p.C, p.ldc, p.bias, p.R, p.ldr) &&
         nw + J * 16 <= p.N;
}

// 4 finished columns of a row: residual and store, bf16 or fp32.
__device__ __forceinline__ void epi_t4_any(const f32x4& v, int m, int n, int M, int N, const MidRows& p, const bf16_t* R,
                                           bool vec) {
  if (p.f32) epi_t4<ACT_NONE, true>(v, m, n, M, N, p.C, p.ldc, nullptr, R, p.ldr, vec);
  else epi_t4<ACT_NONE, false>(v, m, n, M, N, p.C, p.ldc, nullptr, R, p.ldr, vec);
}

// Epilogues of their own (gemm_mid_plain.hip), where the host knows that every wave's columns are whole and leave as
// pairs of 16-byte bf16 stores: an activation, and what else there is.  MID_ANY: whatever the arguments say.
enum MidEpi { MID_ANY = -1, MID_RES = 8, MID_STAT = 16, MID_COLS = 32, MID_BIAS = 64, MID_STATS_OUT = 128 };
constexpr int mid_epi_act(int epi) { return epi & 7; }

// Whether rows leave as those epilogues store them (epi_vec_ok, epi_pair_ok), from waves of `cols` columns; at: more
// vectors that are read 16 bytes at a time.
inline bool mid_plain_ok(const MidRows& a, int cols, const float* at) {
  const uintptr_t p = (uintptr_t)a.C | (uintptr_t)a.bias | (uintptr_t)a.R | (uintptr_t)at;
  return !a.f32 && a.act >= 0 && a.act <= 7 && a.N % cols == 0 && (p & 15) == 0 && a.ldc % 8 == 0 &&
         (a.R == nullptr || a.ldr % 4 == 0);
}

// What the epilogue of a wave reads, loaded ahead of the loop: behind it statistics and
// column sums, bias, then residual rows were up to three trips to memory, 0.5 us each, of
// kernels that take 6 to 40 (with residual, 1071 x 768 x 768 and x 3072: 11.8 us on average,
// now 10.8).  The residual only where there are registers for it.
template <int I, int J>
struct MidPre {
  static constexpr bool RES = I * J <= 8;
  float2 rs[I];
  f32x4 cs[J], bs[J];
  bf16x4 rr[RES ? I : 1][J / 2][2];
  bool res;  // rr is loaded
  template <int EPI>
  __device__ __forceinline__ void load_plain(const MidRows& p, const float2* rowstat, const float* scale, int mw, int nw, int lane) {
    const int n = min(nw, p.N - J * 16) + (lane >> 4) * 4;  // a wave past the columns reads the last ones
    if (rowstat != nullptr) {
#pragma unroll
      for (int i = 0; i < I; ++i) rs[i] = rowstat[min(mw + i * 16, p.M - 1)];
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
      if constexpr ((EPI & MID_COLS) != 0) cs[j] = *reinterpret_cast<const f32x4*>(scale + n + j * 16);
      if constexpr ((EPI & MID_BIAS) != 0) bs[j] = *reinterpret_cast<const f32x4*>(p.bias + n + j * 16);
    }
    if constexpr (RES && (EPI & MID_RES) != 0) res_load(p, mw, nw, lane, rr);
  }
  template <int R>
  static __device__ __forceinline__ void res_load(const MidRows& p, int mw, int nw, int lane, bf16x4 (&r)[R][J / 2][2]) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int jp = 0; jp < J / 2; ++jp)
        epi_pair_res_load(mw + i * 16, min(nw, p.N - J * 16) + jp * 32, p.M, p.R, p.ldr, lane, r[i % R][jp][0], r[i % R][jp][1]);
  }
  // rows m of this lane from mw on, the wave's columns from nw on; `scale`: per column (colsum, channel scale) or null
  __device__ __forceinline__ void load(const MidRows& p, const float2* rowstat, const float* scale, int mw, int nw, int lane,
                                       bool rows) {
    const int M = p.M, N = p.N, n = nw + (lane >> 4) * 4;
#pragma unroll
    for (int i = 0; i < I; ++i) rs[i] = rowstat != nullptr ? rowstat[min(mw + i * 16, M - 1)] : float2{1.f, 0.f};
#pragma unroll
    for (int j = 0; j < J; ++j) {
      cs[j] = scale != nullptr ? mid_cols(scale, n + j * 16, N) : f32x4{0.f, 0.f, 0.f, 0.f};
      bs[j] = p.bias != nullptr && !is_glu(p.act) ? mid_cols(p.bias, n + j * 16, N) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    res = false;
    if constexpr (RES) {
      if (rows && p.R != nullptr && !is_glu(p.act) && mid_pair(p, nw, J)) {
        res = true;
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
          for (int jp = 0; jp < J / 2; ++jp)
            epi_pair_res_load(mw + i * 16, nw + jp * 32, M, p.R, p.ldr, lane, rr[i][jp][0], rr[i][jp][1]);
      }
    }
  }
};

// Bias and an elementwise activation on a wave's accumulators.
template <int I, int J, bool ALL = true>
__device__ __forceinline__ void mid_bias_act(f32x4 (&acc)[I][J], const float* bias, const f32x4 (&bs)[J], int act, int N) {
#pragma clang fp contract(off)  // a product in front (norm, channel scale) is rounded before the bias
  if (bias != nullptr) {
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int i = 0; i < I; ++i) acc[i][j] += bs[j];
  }
  if (act == ACT_GELU) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j] = mid_act<ACT_GELU>(acc[i][j], f32x2{});
  } else if (act == ACT_RELU) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j] = mid_act<ACT_RELU>(acc[i][j], f32x2{});
  } else if (ALL && act == ACT_XIELU) {
    const f32x2 xc = act_consts<ACT_XIELU>(bias, N);
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j] = mid_act<ACT_XIELU>(acc[i][j], xc);
  }
}

// Staging of K-tiles (128 bytes of a row): uniform tile bases, per-lane offsets of
// the wave's 1-KiB pieces of 8 rows, 16-byte chunks swizzled by row.
template <class T>
struct MidSource {
  const char* a;
  const char* b;
  char* lds;
  int nk, wave;
  uint32_t oa[T::PA], ob[T::PB];
  template <bool ROPE = false>  // ROPE: rope_row (gemm_tile.h), of whole 128s
  __device__ __forceinline__ void init(const char* A, int lda, int m0, int M, const char* W, int ldw, int n0, int N, int k0,
                                       int nk_, char* smem, int wave_, int lane) {
    a = A + (size_t)m0 * lda + (size_t)k0 * 128;
    b = W + (size_t)n0 * ldw + (size_t)k0 * 128;
    lds = smem, nk = nk_, wave = wave_;
#pragma unroll
    for (int q = 0; q < T::PA; ++q) {
      const int rl = (q * T::NW + wave) * 8 + (lane >> 3);
      oa[q] = (uint32_t)min(rl, M - 1 - m0) * (uint32_t)lda + (uint32_t)((lane & 7) ^ swz_chunk(rl)) * 16u;
    }
#pragma unroll
    for (int q = 0; q < T::PB; ++q) {
      const int rl = (q * T::NW + wave) * 8 + (lane >> 3);
      ob[q] = (uint32_t)min(ROPE ? (rl & ~127) + rope_row(rl & 127) : rl, N - 1 - n0) * (uint32_t)ldw + (uint32_t)((lane & 7) ^ swz_chunk(rl)) * 16u;
    }
  }
  // Part i of n of K-tile t; past the end: a harmless refill, so that the waits count alike
  __device__ __forceinline__ void stage(int t, int buf, int i, int n) const {
    const size_t k = (size_t)min(t, nk - 1) * 128;
    char* d = lds + buf * T::STAGE + wave * 1024;
#pragma unroll
    for (int q = T::PA * i / n; q < T::PA * (i + 1) / n; ++q) glds16(a + k + oa[q], d + q * T::NW * 1024);
#pragma unroll
    for (int q = T::PB * i / n; q < T::PB * (i + 1) / n; ++q) glds16(b + k + ob[q], d + T::BM * 128 + q * T::NW * 1024);
  }
};

// {mean, sum of squared deviations} of 32 stored columns of a row, 8 of them in each of the lanes l, l ^ 16, l ^ 32, l ^ 48.
__device__ __forceinline__ void mid_part_out(const uint4& x, int m, int nb, const MidRows& p, float2* out, int lane) {
  const uint32_t w[4] = {x.x, x.y, x.z, x.w};
  float v[8], s = 0.f, q = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    v[i] = __uint_as_float(i & 1 ? w[i >> 1] & 0xffff0000u : w[i >> 1] << 16);
    s += v[i];
  }
  const float mean = add32(add16(s)) * (1.f / 32.f);
#pragma unroll
  for (int i = 0; i < 8; ++i) q = fmaf(v[i] - mean, v[i] - mean, q);
  q = add32(add16(q));
  if (lane < 16 && m < p.M) out[(size_t)m * (p.N >> 5) + (nb >> 5)] = make_float2(mean, q);
}

// The rows' {rstd, -mean rstd} from their partials, TPR lanes a row and two partials a load.  As rowstat_merge
// (gemm_epilogue.h): shifted by the first partial's mean, so that no |mean| / std cancels.  load() ahead of the first
// requests, merge() behind them; the rows go to their lanes by way of LDS: behind the K-tiles where there is room
// (written ahead of the loop's first barrier), else where they were, behind the loop.
template <class T>
struct MidParts {
  static constexpr int TPR = T::THREADS / T::BM >= 4 ? 4 : 2, B = 4;  // lanes a row, loads a lane and batch
  static constexpr int TILES = T::S * T::STAGE;
  static constexpr int CU = TILES > 80 * 1024 ? 160 * 1024 : 80 * 1024;  // as many workgroups a CU as without
  static constexpr bool ROOM = TILES + T::BM * 8 <= CU;
  static constexpr int LDS = TILES + (ROOM ? T::BM * 8 : 0);
  f32x4 p[B];
  float2 r;
  const f32x4* row;
  int n2, sub;
  __device__ __forceinline__ void batch(int b) {
#pragma unroll
    for (int i = 0; i < B; ++i) p[i] = row[min(sub + (b + i) * TPR, n2 - 1)];
  }
  __device__ __forceinline__ void load(const MidArgs& a, int m0, int tid) {
    n2 = a.K >> 6, sub = tid % TPR;
    row = reinterpret_cast<const f32x4*>(a.parts) + (size_t)min(m0 + min(tid / TPR, T::BM - 1), a.M - 1) * n2;
    batch(0);
  }
  __device__ __forceinline__ void put(char* lds, int tid) const {
    if (sub == 0 && tid / TPR < T::BM) reinterpret_cast<float2*>(lds)[tid / TPR] = r;
  }
  __device__ __forceinline__ void merge(const MidArgs& a, char* lds, int tid) {
    const float c = a.rms ? 0.f : dpp_f<TPR == 4 ? 0x00 : 0xA0>(p[0][0]);  // quad_perm: the row's first lane
    float s1 = 0.f, s2 = 0.f, sm = 0.f;
    for (int b = 0;; b += B) {
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const bool in = sub + (b + i) * TPR < n2;
        const float d = in ? p[i][0] - c : 0.f, e = in ? p[i][2] - c : 0.f;
        s1 += d + e;
        s2 = fmaf(d, d, fmaf(e, e, s2));
        sm += in ? p[i][1] + p[i][3] : 0.f;
      }
      if ((b + B) * TPR >= n2) break;  // uniform
      batch(b + B);
    }
    s1 = group_sum<TPR>(s1) * 32.f;
    s2 = group_sum<TPR>(s2) * 32.f;
    sm = group_sum<TPR>(sm);
    const float invk = 1.f / (float)a.K, d = a.rms ? 0.f : s1 * invk;
    const float rstd = rsqrtf(fmax_nan((sm + s2) * invk - d * d, 0.f) + a.eps);
    r = make_float2(rstd, a.rms ? 0.f : -(c + d) * rstd);
    if constexpr (ROOM) put(lds + TILES, tid);
  }
  template <int I>
  __device__ __forceinline__ void share(char* lds, int tid, int row0, float2 (&rs)[I]) const {
    if constexpr (!ROOM) {
      __syncthreads();
      put(lds, tid);
      __syncthreads();
    }
    const float2* st = reinterpret_cast<const float2*>(lds + (ROOM ? TILES : 0));
#pragma unroll
    for (int i = 0; i < I; ++i) rs[i] = st[row0 + i * 16];
  }
};

// A wave's accumulators to head-major q / K / V (host: N % 32 == 0).
template <int I, int J>
__device__ __forceinline__ void mid_scatter(f32x4 (&acc)[I][J], int mw, int nw, int M, int N, const float* bias,
                                            const f32x4 (&bs)[J], int lane, const QkvScatter& scat) {
  QkvRow row[I];
  QkvCol col[J / 2];
#pragma unroll
  for (int i = 0; i < I; ++i) row[i] = qkv_row(scat, min(mw + i * 16, M - 1));
#pragma unroll
  for (int jp = 0; jp < J / 2; ++jp) col[jp] = qkv_col(scat, pair_col(nw + jp * 32, lane));
  mid_bias_act<I, J, false>(acc, bias, bs, ACT_NONE, N);
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int jp = 0; jp < J / 2; ++jp)
      if (nw + jp * 32 < N) epi_pair_scatter(acc[i][2 * jp], acc[i][2 * jp + 1], mw + i * 16, M, row[i], col[jp]);
}

// The same with q and K rotated (host: heads of 128, no bias; rows staged by rope_row).
template <int I, int J>
__device__ __forceinline__ void mid_rope(f32x4 (&acc)[I][J], int mw, int nw, int M, int N, int lane, const QkvScatter& scat) {
  QkvRow row[I];
  QkvCol col[J / 2];
  f32x4 co[I][J / 2], si[I][J / 2];
#pragma unroll
  for (int i = 0; i < I; ++i) row[i] = qkv_row(scat, min(mw + i * 16, M - 1));
#pragma unroll
  for (int jp = 0; jp < J / 2; ++jp) {
    col[jp] = qkv_col(scat, rope_pair_col(nw + jp * 32 + scat.c_off, lane));
#pragma unroll
    for (int i = 0; i < I; ++i) {
      co[i][jp] = rope_load(scat.cosT, row[i].p, nw + jp * 32, lane);
      si[i][jp] = rope_load(scat.sinT, row[i].p, nw + jp * 32, lane);
    }
  }
  const int rotated = ((scat.H + scat.Hkv) << 7) - scat.c_off;
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int jp = 0; jp < J / 2; ++jp) {
      if (nw + jp * 32 < rotated) rope_pair(acc[i][2 * jp], acc[i][2 * jp + 1], co[i][jp], si[i][jp]);
      if (nw + jp * 32 < N) epi_pair_scatter(acc[i][2 * jp], acc[i][2 * jp + 1], mw + i * 16, M, row[i], col[jp]);
    }
}

// A wave's accumulators (rows mw + 16 i of this lane, columns from nw on) through the epilogue to C.
// ALL: with fp32 rows and the activations that only bf16 weights have.
template <int I, int J, bool ALL = true>
__device__ __forceinline__ void mid_rows(f32x4 (&acc)[I][J], int mw, int nw, int lane, const MidRows& p,
                                         const MidPre<I, J>& pre, float2* parts_out = nullptr) {
  const int M = p.M, N = p.N, fg = lane >> 4;
  const bool f32 = ALL && p.f32;
  const bool vec = epi_vec_ok(p.C, p.ldc, p.bias, p.R, p.ldr);
  if (is_glu(p.act)) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int jp = 0; jp < J / 2; ++jp) {
        const f32x4 &x0 = acc[i][2 * jp], &x1 = acc[i][2 * jp + 1];
        const int m = mw + i * 16, c = (nw + jp * 32) / 2;
        if (ALL && p.act == ACT_GELU_TANH_MUL) epi_glu_pair<ACT_GELU_TANH_MUL, false>(x0, x1, m, c, M, N / 2, p.C, p.ldc, vec, lane);
        else if (f32) epi_glu_pair<ACT_SILU_MUL, true>(x0, x1, m, c, M, N / 2, p.C, p.ldc, vec, lane);
        else epi_glu_pair<ACT_SILU_MUL, false>(x0, x1, m, c, M, N / 2, p.C, p.ldc, vec, lane);
      }
    return;
  }
  mid_bias_act<I, J, ALL>(acc, p.bias, pre.bs, p.act, N);
  bf16_t* C = reinterpret_cast<bf16_t*>(p.C);
  const bool pair = mid_pair(p, nw, J);
  if (MidPre<I, J>::RES && pre.res) {
#pragma unroll
    for (int i = 0; i < (MidPre<I, J>::RES ? I : 1); ++i)
#pragma unroll
      for (int jp = 0; jp < J / 2; ++jp) {
        uint4 x;
        epi_pair_bf16<ACT_NONE, true>(acc[i][2 * jp], acc[i][2 * jp + 1], mw + i * 16, nw + jp * 32, M, C, p.ldc, nullptr,
                                      p.R, p.ldr, lane, pre.rr[i][jp][0], pre.rr[i][jp][1], f32x2{}, &x);
        if (parts_out != nullptr) mid_part_out(x, mw + i * 16, nw + jp * 32, p, parts_out, lane);
      }
  } else if (!MidPre<I, J>::RES && pair && p.R != nullptr) {  // every residual load before the first output
    bf16x4 rr[I][J / 2][2];
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int jp = 0; jp < J / 2; ++jp)
        epi_pair_res_load(mw + i * 16, nw + jp * 32, M, p.R, p.ldr, lane, rr[i][jp][0], rr[i][jp][1]);
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int jp = 0; jp < J / 2; ++jp) {
        uint4 x;
        epi_pair_bf16<ACT_NONE, true>(acc[i][2 * jp], acc[i][2 * jp + 1], mw + i * 16, nw + jp * 32, M, C, p.ldc, nullptr,
                                      p.R, p.ldr, lane, rr[i][jp][0], rr[i][jp][1], f32x2{}, &x);
        if (parts_out != nullptr) mid_part_out(x, mw + i * 16, nw + jp * 32, p, parts_out, lane);
      }
  } else if (pair) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int jp = 0; jp < J / 2; ++jp)
        epi_pair_bf16<ACT_NONE>(acc[i][2 * jp], acc[i][2 * jp + 1], mw + i * 16, nw + jp * 32, M, C, p.ldc, nullptr, nullptr,
                                0, lane);
  } else if (f32) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j)
        epi_t4<ACT_NONE, true>(acc[i][j], mw + i * 16, nw + j * 16 + fg * 4, M, N, p.C, p.ldc, nullptr, p.R, p.ldr, vec);
  } else {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j)
        epi_t4<ACT_NONE, false>(acc[i][j], mw + i * 16, nw + j * 16 + fg * 4, M, N, p.C, p.ldc, nullptr, p.R, p.ldr, vec);
  }
}

// epi_glu_pair (gemm_epilogue.h) of whole columns in bf16.
template <int ACT>
__device__ __forceinline__ void mid_glu_plain(const f32x4& a0, const f32x4& a1, int m, int ncol0, const MidRows& p, int lane) {
  f32x4 v;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a0[r]), __float_as_uint(a1[r]), false, false);
    const float g = __uint_as_float(s[0]), u = __uint_as_float(s[1]);
    if constexpr (ACT == ACT_GELU_TANH_MUL) v[r] = gelu_tanh(g) * u;
    else v[r] = g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f)) * u;
  }
  if (m < p.M)
    *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(p.C) + (size_t)m * p.ldc + ncol0 + (lane >> 4) * 4) =
        make_uint2(pack2bf(v[0], v[1]), pack2bf(v[2], v[3]));
}

// The same where the epilogue is known (MidEpi).
template <int I, int J, int EPI>
__device__ __forceinline__ void mid_rows_plain(f32x4 (&acc)[I][J], int mw, int nw, int lane, const MidRows& p,
                                               const MidPre<I, J>& pre, float2* parts_out) {
  constexpr int ACT = mid_epi_act(EPI);
  constexpr bool PRE = MidPre<I, J>::RES;
  if (nw >= p.N) return;
  if constexpr (is_glu(ACT)) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int jp = 0; jp < J / 2; ++jp)
        mid_glu_plain<ACT>(acc[i][2 * jp], acc[i][2 * jp + 1], mw + i * 16, (nw + jp * 32) / 2, p, lane);
    return;
  }
  {
#pragma clang fp contract(off)  // as mid_bias_act
    if constexpr ((EPI & MID_BIAS) != 0) {
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int i = 0; i < I; ++i) acc[i][j] += pre.bs[j];
    }
  }
  if constexpr (ACT != ACT_NONE) {
    const f32x2 xc = act_consts<ACT>(p.bias, p.N);
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j] = mid_act<ACT>(acc[i][j], xc);
  }
  constexpr bool RES = (EPI & MID_RES) != 0;
  bf16x4 rl[RES && !PRE ? I : 1][J / 2][2];
  if constexpr (RES && !PRE) MidPre<I, J>::res_load(p, mw, nw, lane, rl);  // every residual load before the first output
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int jp = 0; jp < J / 2; ++jp) {
      const int m = mw + i * 16, nb = nw + jp * 32;
      bf16_t* C = reinterpret_cast<bf16_t*>(p.C);
      if constexpr (!RES) {
        epi_pair_bf16<ACT_NONE>(acc[i][2 * jp], acc[i][2 * jp + 1], m, nb, p.M, C, p.ldc, nullptr, nullptr, 0, lane);
      } else {
        uint4 x;
        const bf16x4 r0 = PRE ? pre.rr[PRE ? i : 0][jp][0] : rl[PRE ? 0 : i][jp][0], r1 = PRE ? pre.rr[PRE ? i : 0][jp][1] : rl[PRE ? 0 : i][jp][1];
        epi_pair_bf16<ACT_NONE, true>(acc[i][2 * jp], acc[i][2 * jp + 1], m, nb, p.M, C, p.ldc, nullptr, p.R, p.ldr, lane, r0, r1,
                                      f32x2{}, &x);
        if constexpr ((EPI & MID_STATS_OUT) != 0) mid_part_out(x, m, nb, p, parts_out, lane);
      }
    }
}

// Loop: a K-tile of 64 is multiplied in two halves of 32; the second half's
// fragments are read behind the first row of products of the first, the next
// tile's first half behind the first row of the second, one barrier a tile.  The
// requests for tile t + S - 1 go out between the rows of products.
//
// What bounds it: the operands' way from L2 to LDS.  With 128 x 128 tiles on 192
// CUs a K-tile takes 0.47 us (32 KB a CU: 13 TB/s over the chip) where its products
// take 0.22 and its LDS traffic 0.33; larger tiles need fewer bytes per product but
// more splits.  Touching later lines from a wave of its own, waves of 64 x 32 in
// place of 64 x 64, or padded rows did not change that.
//
// T::PW > 0: other waves stage, and `src` only says where (mid_stage keeps the same barriers).
// `behind`: run behind the first requests.
struct MidNone {
  __device__ __forceinline__ void operator()() const {}
};
template <class T, class F = MidNone>
__device__ __forceinline__ void mid_loop(const MidSource<T>& src, int wm, int wn, int lane, f32x4 (&acc)[T::I][T::J],
                                         F behind = F{}) {
  constexpr bool OWN = T::PW == 0;
  constexpr int I = T::I, J = T::J, S = T::S, L = T::PA + T::PB;
  // fragment reads: lane (r, g) reads 16 B of row r at chunks g and 4 + g
  const int fr = lane & 15, fg = lane >> 4;
  const int arow = wm * (I * 16) + fr, brow = wn * (J * 16) + fr;
  const int ao[2] = {arow * 128 + ((fg ^ swz_chunk(arow)) << 4), arow * 128 + (((4 + fg) ^ swz_chunk(arow)) << 4)};
  const int bo[2] = {T::BM * 128 + brow * 128 + ((fg ^ swz_chunk(brow)) << 4),
                     T::BM * 128 + brow * 128 + (((4 + fg) ^ swz_chunk(brow)) << 4)};
  // The operands of a K-tile in two halves of 32: F[x] = 16 x 32 fragments of A, then of B.
  bf16x8 f[2][I + J];
  auto read = [&](auto hc, int buf) {
    constexpr int h = decltype(hc)::value;
    const char* d = src.lds + buf * T::STAGE;
#pragma unroll
    for (int j = 0; j < J; ++j) f[h][I + j] = *reinterpret_cast<const bf16x8*>(d + bo[h] + j * 2048);
#pragma unroll
    for (int i = 0; i < I; ++i) f[h][i] = *reinterpret_cast<const bf16x8*>(d + ao[h] + i * 2048);
  };
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mma = [&](auto hc, int i) {
    constexpr int h = decltype(hc)::value;
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[h][I + j], f[h][i], acc[i][j], 0, 0, 0);
  };
  constexpr auto h0 = std::integral_constant<int, 0>{};
  constexpr auto h1 = std::integral_constant<int, 1>{};
  if constexpr (OWN) {
#pragma unroll
    for (int q = 0; q < S - 1; ++q) src.stage(q, q, 0, 1);
    behind();
    __builtin_amdgcn_s_waitcnt(wait_imm((S - 2) * L, 0));
  }
  bg_barrier();
  read(h0, 0);
  int cur = 0;
  for (int t = 0; t < src.nk; ++t) {
    const int prev = cur == 0 ? S - 1 : cur - 1, next = cur == S - 1 ? 0 : cur + 1;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < I; ++i) {
      mma(h0, i);
      __builtin_amdgcn_sched_barrier(0);
      if (i == 0) read(h1, cur);
      if constexpr (OWN) src.stage(t + S - 1, prev, i, I);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (OWN) __builtin_amdgcn_s_waitcnt(wait_imm((S - 2) * L, 0));  // tile t + 1 landed, tile t read
    else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                   // tile t read
    bg_barrier();
#pragma unroll
    for (int i = 0; i < I; ++i) {
      mma(h1, i);
      __builtin_amdgcn_sched_barrier(0);
      if (i == 0) read(h0, next);
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
    cur = next;
  }
  __builtin_amdgcn_s_waitcnt(wait_imm(0, 0));
}

// The waves that only stage: tile t + S - 1 goes to the buffer that tile t - 1 left at the
// barrier before, tile t + 1 has landed at the next one; as many barriers as mid_loop.
template <class T>
__device__ __forceinline__ void mid_stage(const MidSource<T>& src) {
  constexpr int S = T::S, L = T::PA + T::PB;
#pragma unroll
  for (int q = 0; q < S - 1; ++q) src.stage(q, q, 0, 1);
  __builtin_amdgcn_s_waitcnt(wait_imm((S - 2) * L, 0));
  bg_barrier();
  int prev = S - 1;
  for (int t = 0; t < src.nk; ++t) {
    src.stage(t + S - 1, prev, 0, 1);
    __builtin_amdgcn_s_waitcnt(wait_imm((S - 2) * L, 0));
    bg_barrier();
    prev = prev == S - 1 ? 0 : prev + 1;
  }
  __builtin_amdgcn_s_waitcnt(wait_imm(0, 0));
}

enum MidOut { MID_ROWS = 0, MID_SCATTER = 1, MID_PART = 2, MID_ROPE = 3 };

// MERGE: the folded norm's statistics from partials (a variant of its own: a load under a branch is waited for where
// the branch ends, ahead of the first request)
// EPI: MidEpi
template <class T, MidOut OUT, bool MERGE, int EPI = MID_ANY>
__global__ __launch_bounds__(T::THREADS, 2) void gemm_mid_kernel(MidArgs p, QkvScatter scat) {
  constexpr bool PART = OUT == MID_PART;
  static_assert(EPI == MID_ANY || (OUT == MID_ROWS && T::PW == 0 && (!MERGE || (EPI & MID_STAT) != 0)), "");
  static_assert(PART ? !MERGE : T::PW == 0, "");
  constexpr int I = T::I, J = T::J;
  // S * STAGE bytes (MERGE: MidParts::LDS), given at launch: with the size in the kernel the compiler sees one
  // wave per SIMD and moves accumulators of the four-wave tiles to AGPRs and back in
  // the loop (a tile of 192 x 128 rows at 700 x 6144 x 4096: 47 -> 78 us)
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = p.M, N = p.N;
  const int ntn = (N + T::BN - 1) / T::BN, ntm = (M + T::BM - 1) / T::BM, tiles = ntm * ntn;
  int id = xcd_remap(blockIdx.x, tiles * p.splits), sp = 0;
  if constexpr (PART) {
    sp = id / tiles;
    id -= sp * tiles;
  }
  int tm, tn;
  tile_coords(id, ntm, ntn, tm, tn);
  const int m0 = tm * T::BM, n0 = tn * T::BN;
  const int cw = wave - T::PW;  // < 0: stages
  const int wm = cw / T::WN, wn = cw % T::WN, fr = lane & 15, fg = lane >> 4;
  int nk = p.K >> 6, k0 = 0;
  if constexpr (PART) {
    k0 = (int)((long long)nk * sp / p.splits);
    nk = (int)((long long)nk * (sp + 1) / p.splits) - k0;
  }
  MidSource<T> src;
  src.template init<OUT == MID_ROPE>(reinterpret_cast<const char*>(p.A), p.lda * 2, m0, M, reinterpret_cast<const char*>(p.W),
                                     p.ldw * 2, n0, N, k0, nk, smem, wave, lane);
  if constexpr (T::PW > 0) {
    if (cw < 0) {
      mid_stage<T>(src);
      return;
    }
  }
  const int mw = m0 + wm * (I * 16) + fr, nw = n0 + wn * (J * 16);  // the lane's first row, the wave's first column
  MidPre<I, J> pre;
  if constexpr (EPI != MID_ANY) pre.template load_plain<EPI>(p, !MERGE && (EPI & MID_STAT) != 0 ? p.rowstat : nullptr, p.colsum, mw, nw, lane);
  else if constexpr (OUT == MID_ROPE) pre.template load_plain<MID_STAT>(p, p.rowstat, nullptr, mw, nw, lane);
  else if constexpr (!PART) pre.load(p, p.rowstat, p.colsum, mw, nw, lane, OUT == MID_ROWS);
  f32x4 acc[I][J];
  MidParts<T> parts;
  if constexpr (MERGE) {
    parts.load(p, m0, tid);
    mid_loop<T>(src, wm, wn, lane, acc, [&]() { parts.merge(p, smem, tid); });
    parts.share(smem, tid, wm * (I * 16) + fr, pre.rs);
  } else {
    mid_loop<T>(src, wm, wn, lane, acc);
  }

  if constexpr (PART) {
    float* d = p.part + (size_t)sp * M * N;
#pragma unroll
    for (int i = 0; i < I; ++i) {
      const int m = m0 + wm * (I * 16) + i * 16 + fr;
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int n = n0 + wn * (J * 16) + j * 16 + fg * 4;  // host: N % 4 == 0
        if (m < M && n < N) *reinterpret_cast<f32x4*>(d + (size_t)m * N + n) = acc[i][j];
      }
    }
    return;
  }
  if constexpr (EPI != MID_ANY) {
    if constexpr ((EPI & MID_STAT) != 0) {
#pragma unroll
      for (int i = 0; i < I; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j) {
          if constexpr ((EPI & MID_COLS) != 0) acc[i][j] = acc[i][j] * pre.rs[i].x + pre.rs[i].y * pre.cs[j];
          else acc[i][j] *= pre.rs[i].x;
        }
    }
    mid_rows_plain<I, J, EPI>(acc, mw, nw, lane, p, pre, p.parts_out);
    return;
  }
  if constexpr (OUT == MID_ROPE) {
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j] *= pre.rs[i].x;
    mid_rope<I, J>(acc, mw, nw, M, N, lane, scat);
    return;
  }
  if (MERGE || p.rowstat != nullptr) {  // the folded norm, in the 256 x 256 kernel's order of operations
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int j = 0; j < J; ++j) acc[i][j] = acc[i][j] * pre.rs[i].x + pre.rs[i].y * pre.cs[j];
  }
  if constexpr (OUT == MID_SCATTER) mid_scatter<I, J>(acc, mw, nw, M, N, p.bias, pre.bs, lane, scat);
  else mid_rows<I, J>(acc, mw, nw, lane, p, pre, p.parts_out);
}

// Sum of the parts and the epilogue.  A thread: 4 columns of one row (gated: 4
// gate columns and the 4 up columns that belong to them).  Bound by reading the
// parts (they were just written: mostly from the last-level cache).
template <int GLU>
__global__ __launch_bounds__(256) void gemm_mid_reduce(MidArgs p) {
  const int m = blockIdx.y, M = p.M, N = p.N;
  const int q = blockIdx.x * 256 + threadIdx.x;  // group of 4 output columns
  const int n = GLU ? (q >> 1) * 16 + (q & 1) * 4 : q * 4;
  if (n >= N) return;
  const size_t slab = (size_t)M * N;
  const float* d = p.part + (size_t)m * N + n;
  f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f}, u = v;
  for (int s = 0; s < p.splits; ++s) {
    v += *reinterpret_cast<const f32x4*>(d + s * slab);
    if (GLU) u += *reinterpret_cast<const f32x4*>(d + s * slab + 8);
  }
  if (p.rowstat != nullptr) {
    v = epi_norm4(v, m, n, M, N, p.rowstat, p.colsum);
    if (GLU) u = epi_norm4(u, m, n + 8, M, N, p.rowstat, p.colsum);
  }
  const bool vec = epi_vec_ok(p.C, p.ldc, p.bias, p.R, p.ldr);
  if (GLU) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = (p.act == ACT_GELU_TANH_MUL ? gelu_tanh(v[r]) : silu(v[r])) * u[r];
    epi_t4_any(v, m, q * 4, M, N / 2, p, nullptr, vec);
    return;
  }
  f32x4 a[1][1] = {{v}};
  const f32x4 b[1] = {p.bias != nullptr ? mid_cols(p.bias, n, N) : f32x4{0.f, 0.f, 0.f, 0.f}};
  mid_bias_act<1, 1>(a, p.bias, b, p.act, N);
  if (p.parts_out != nullptr) {  // host: bf16, whole groups of 8 threads
    f32x4 x;
    epi_t4<ACT_NONE, false>(a[0][0], m, n, M, N, p.C, p.ldc, nullptr, p.R, p.ldr, vec, nullptr, 1.f, &x);
    const float mean = group_sum<8>(x[0] + x[1] + (x[2] + x[3])) * (1.f / 32.f);
    x -= mean;
    const float s = group_sum<8>(x[0] * x[0] + x[1] * x[1] + (x[2] * x[2] + x[3] * x[3]));
    if ((threadIdx.x & 7) == 0) p.parts_out[(size_t)m * (N >> 5) + (n >> 5)] = make_float2(mean, s);
    return;
  }
  epi_t4_any(a[0][0], m, n, M, N, p, p.R, vec);
}

template <class T, MidOut OUT, bool MERGE = false, int EPI = MID_ANY>
static int mid_start(const MidArgs& a, const QkvScatter& scat, hipStream_t st) {
  constexpr int LDS = MERGE ? MidParts<T>::LDS : T::S * T::STAGE;
  static const hipError_t room =
      hipFuncSetAttribute((const void*)gemm_mid_kernel<T, OUT, MERGE, EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (room != hipSuccess) return (int)room;
  const int tiles = ((a.M + T::BM - 1) / T::BM) * ((a.N + T::BN - 1) / T::BN);
  hipLaunchKernelGGL((gemm_mid_kernel<T, OUT, MERGE, EPI>), dim3(tiles * a.splits), dim3(T::THREADS), LDS, st, a, scat);
  return (int)hipGetLastError();
}

}  // namespace dnn
