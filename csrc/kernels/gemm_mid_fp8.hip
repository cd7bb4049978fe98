// e4m3 GEMM with MX activations (common.h mx_index) on the tiles of gemm_mid.h: row
// counts where the 256 x 256 tiles (gemm_bf16.hip gemm_fp8_256_kernel) leave CUs
// idle.  A K-tile is 128 columns = 128 bytes of a row, so staging, LDS images and a
// tile's time are those of the bf16 kernel's K-tile of 64.
#include "gemm_mid.h"
#include "gemm_mid_fp8.h"

namespace dnn {

typedef int i32x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ i32x8 mid8_cat(const bf16x8& lo, const bf16x8& hi) {
  const i32x4 a = __builtin_bit_cast(i32x4, lo), b = __builtin_bit_cast(i32x4, hi);
  return i32x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

// One product of 16 x 16 x 128; byte B of s scales the row fragment.
template <int B>
__device__ __forceinline__ f32x4 mid8_mfma(const i32x8& b, const i32x8& a, const f32x4& c, uint32_t s) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b, a, c, 0, 0, 0, 0x7f7f7f7f, B, s);
}

// PLAIN: rows of a projection with bias and residual alone, whole columns (mid_plain_ok): 4 to 9 KB of code for 11 to 34
// (gemm_mid_plain.hip).  us a launch, 2048 x 1600 of K = 1600 and 6400 on 128 x 128: 24.4 -> 23.8 on average.
enum Mid8Out { MID8_ROWS = 0, MID8_SCATTER = 1, MID8_QUANT = 2, MID8_PLAIN = 3 };

// Loop: a product needs both halves of a K-tile, so a tile's fragments are double
// buffered in registers: behind the first row of products of tile t the requests for
// t + S - 1 go out (their buffer was read an iteration ago), then tile t + 1 is
// awaited and read while the other rows are multiplied; one barrier a tile.  A
// wave's row scales (a dword per 64 rows, gemm_fp8_256_kernel) are staged beside the
// operands.  256 x 128 on 2048 x 4800 x 1600: 33 us as 256 x 256, 23 now.
template <class T, Mid8Out OUT>
__global__ __launch_bounds__(T::NW * 64, 2) void gemm_mid_fp8_kernel(Mid8Args p, QkvScatter scat) {
  constexpr int I = T::I, J = T::J, S = T::S, L = T::PA + T::PB + 1;
  static_assert(I == 4 || I == 2, "a wave's rows lie in one block of 64");
  extern __shared__ __attribute__((aligned(1024))) char smem[];  // S * (STAGE + NW * 256) bytes
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = p.M, N = p.N;
  const int ntn = (N + T::BN - 1) / T::BN, ntm = (M + T::BM - 1) / T::BM;
  int tm, tn;
  tile_coords(xcd_remap(blockIdx.x, ntm * ntn), ntm, ntn, tm, tn);
  const int m0 = tm * T::BM, n0 = tn * T::BN;
  const int wm = wave / T::WN, wn = wave % T::WN;
  const int nk = p.Kb >> 7;
  MidSource<T> src;
  src.init(reinterpret_cast<const char*>(p.A), p.Kb, m0, M, reinterpret_cast<const char*>(p.W), p.Kb, n0, N, 0, nk, smem,
           wave, lane);
  const int nb64 = mx_mpad(M) >> 6;
  const uint32_t* sx = p.sx + (size_t)min((m0 + wm * (I * 16)) >> 6, nb64 - 1) * 16 + (lane & 15);
  char* const scl = smem + S * T::STAGE + wave * 256;
  const int sshift = I == 2 ? 16 * (wm & 1) : 0;  // 32 rows: the upper or lower two bytes
  auto stage_scale = [&](int t, int buf) {
    __builtin_amdgcn_global_load_lds((const GLB_AS void*)(sx + (size_t)min(t, nk - 1) * nb64 * 16),
                                     (LDS_AS void*)(scl + buf * T::NW * 256), 4, 0, 0);
  };
  const int fr = lane & 15, fg = lane >> 4;
  const int arow = wm * (I * 16) + fr, brow = wn * (J * 16) + fr;
  const int ao[2] = {arow * 128 + ((fg ^ swz_chunk(arow)) << 4), arow * 128 + (((4 + fg) ^ swz_chunk(arow)) << 4)};
  const int bo[2] = {T::BM * 128 + brow * 128 + ((fg ^ swz_chunk(brow)) << 4),
                     T::BM * 128 + brow * 128 + (((4 + fg) ^ swz_chunk(brow)) << 4)};
  const int mw = m0 + wm * (I * 16) + fr, nw = n0 + wn * (J * 16);
  MidPre<I, J> pre;  // cs: the channel scales
  constexpr int EPI = MID_RES | MID_BIAS;
  if constexpr (OUT == MID8_PLAIN) pre.template load_plain<EPI | MID_COLS>(p, nullptr, p.sw, mw, nw, lane);
  else pre.load(p, nullptr, p.sw, mw, nw, lane, OUT == MID8_ROWS);
  bf16x8 fa[2][I][2], fb[2][J][2];
  uint32_t fs[2];
  auto read = [&](auto uc, int buf) {
    constexpr int u = decltype(uc)::value;
    const char* d = smem + buf * T::STAGE;
    fs[u] = *reinterpret_cast<const uint32_t*>(scl + buf * T::NW * 256 + lane * 4) >> sshift;
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) fb[u][j][h] = *reinterpret_cast<const bf16x8*>(d + bo[h] + j * 2048);
#pragma unroll
    for (int i = 0; i < I; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) fa[u][i][h] = *reinterpret_cast<const bf16x8*>(d + ao[h] + i * 2048);
  };
  f32x4 acc[I][J];
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mma = [&](auto uc, auto ic) {
    constexpr int u = decltype(uc)::value, i = decltype(ic)::value;
    const i32x8 a = mid8_cat(fa[u][i][0], fa[u][i][1]);
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] = mid8_mfma<i>(mid8_cat(fb[u][j][0], fb[u][j][1]), a, acc[i][j], fs[u]);
  };
  constexpr auto c0 = std::integral_constant<int, 0>{};
  constexpr auto c1 = std::integral_constant<int, 1>{};
  constexpr auto c2 = std::integral_constant<int, (I > 2 ? 2 : 1)>{};
  constexpr auto c3 = std::integral_constant<int, (I > 2 ? 3 : 1)>{};
#pragma unroll
  for (int q = 0; q < S - 1; ++q) {
    src.stage(q, q, 0, 1);
    stage_scale(q, q);
  }
  __builtin_amdgcn_s_waitcnt(wait_imm((S - 2) * L, 0));
  bg_barrier();
  read(c0, 0);
  int cur = 0;
  auto ktile = [&](int t, auto uc) {
    constexpr auto un = std::integral_constant<int, decltype(uc)::value ^ 1>{};
    const int prev = cur == 0 ? S - 1 : cur - 1, next = cur == S - 1 ? 0 : cur + 1;
    __builtin_amdgcn_s_setprio(1);
    mma(uc, c0);
    __builtin_amdgcn_sched_barrier(0);
    src.stage(t + S - 1, prev, 0, 1);
    stage_scale(t + S - 1, prev);
    __builtin_amdgcn_s_waitcnt(wait_imm((S - 2) * L, 0));  // tile t + 1 landed; tile t was read
    bg_barrier();
    read(un, next);
    __builtin_amdgcn_sched_barrier(0);
    mma(uc, c1);
    if constexpr (I > 2) {
      mma(uc, c2);
      mma(uc, c3);
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    cur = next;
  };
  int t = 0;
  for (; t + 1 < nk; t += 2) {
    ktile(t, c0);
    ktile(t + 1, c1);
  }
  if (t < nk) ktile(t, c0);
  __builtin_amdgcn_s_waitcnt(wait_imm(0, 0));

  if constexpr (OUT == MID8_QUANT) {
    // bias + GELU, then e4m3 with a scale per row and 128 columns: the columns of the
    // lane, of its four lane rows, and of the waves beside it through LDS
    constexpr int G = 128 / (J * 16);  // waves of 128 columns
    static_assert(T::BN % 128 == 0 && T::WN % G == 0, "whole blocks of 128 columns");
    float* red = reinterpret_cast<float*>(smem);  // [row of the tile][wn]
    __syncthreads();                              // every wave past its last operand read and DMA
#pragma unroll
    for (int i = 0; i < I; ++i) {
      float am = 0.f;
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const f32x4 v = mid_act<ACT_GELU>(acc[i][j] * pre.cs[j] + pre.bs[j], f32x2{});  // zeros past N: mid_cols
#pragma unroll
        for (int r = 0; r < 4; ++r) am = fmaxf(am, fabsf(v[r]));
        acc[i][j] = v;
      }
      am = max16(am);
      am = max32(am);
      if (lane < 16) red[(wm * (I * 16) + i * 16 + lane) * T::WN + wn] = am;
    }
    __syncthreads();
    const int mpad = mx_mpad(M);
#pragma unroll
    for (int i = 0; i < I; ++i) {
      float am = 0.f;
#pragma unroll
      for (int g = 0; g < G; ++g) am = fmaxf(am, red[(wm * (I * 16) + i * 16 + fr) * T::WN + wn / G * G + g]);
      float inv;
      const uint32_t e = e8m0_of(am, inv);
      const int m = mw + i * 16;
#pragma unroll
      for (int jp = 0; jp < J / 2; ++jp) {
        const f32x4 v0 = acc[i][2 * jp] * inv, v1 = acc[i][2 * jp + 1] * inv;
        int x = __builtin_amdgcn_cvt_pk_fp8_f32(v0[0], v0[1], 0, false);
        x = __builtin_amdgcn_cvt_pk_fp8_f32(v0[2], v0[3], x, true);
        int y = __builtin_amdgcn_cvt_pk_fp8_f32(v1[0], v1[1], 0, false);
        y = __builtin_amdgcn_cvt_pk_fp8_f32(v1[2], v1[3], y, true);
        const auto sw2 = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)y, false, false);
        const int c = nw + jp * 32 + ((fg & 1) << 4) + ((fg >> 1) << 3);
        if (m < M && c < p.kpo) *reinterpret_cast<uint2*>(p.qo + (size_t)m * p.ldq + c) = make_uint2(sw2[0], sw2[1]);
      }
      const int t128 = nw >> 7;
      if (wn % G == 0 && fg == 0 && m < M && t128 * 128 < p.kpo) p.sxo[mx_index(m, t128, mpad)] = (uint8_t)e;
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) acc[i][j] *= pre.cs[j];
  if constexpr (OUT == MID8_PLAIN) mid_rows_plain<I, J, EPI>(acc, mw, nw, lane, p, pre, nullptr);
  else if constexpr (OUT == MID8_SCATTER) mid_scatter<I, J>(acc, mw, nw, M, N, p.bias, pre.bs, lane, scat);
  else mid_rows<I, J, false>(acc, mw, nw, lane, p, pre);
}

// 64 x 64: four K-tiles in flight.  With the scales' 1 KiB a K-tile five are 87,040 bytes, one workgroup a CU where the
// estimate counts on two (gemm_mid.hip MID8).  us with five : four: 500 x 2304 x 768 8.5 :
// 6.1, 1000 12.2 : 9.2, 1800 19.7 : 13.7, 1350 x 768 x 768 8.4 : 5.9, 820 x 4800 x 1600 22.6 : 15.6.
typedef MidTile<64, 64, 2, 2, 4> Mid0Mx;

template <class T>
constexpr int mid8_lds() { return T::S * (T::STAGE + T::NW * 256); }
static_assert(2 * mid8_lds<Mid0Mx>() <= 160 * 1024, "two workgroups a CU");

template <class T>
static int blocks() {
  int n = 0;
  const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void*)gemm_mid_fp8_kernel<T, MID8_ROWS>,
                                                                    T::NW * 64, mid8_lds<T>());
  return e == hipSuccess ? n : -1;
}

int mid8_blocks(int tile) {
  switch (tile) {
    case 0: return blocks<Mid0Mx>();
    case 1: return blocks<Mid1>();
    case 2: return blocks<Mid2>();
    case 3: return blocks<Mid3>();
    case 4: return blocks<Mid4>();
  }
  return -1;
}

template <class T, Mid8Out OUT>
static int start(const Mid8Args& a, const QkvScatter& scat, hipStream_t st) {
  constexpr int LDS = mid8_lds<T>();
  static const hipError_t room =
      hipFuncSetAttribute((const void*)gemm_mid_fp8_kernel<T, OUT>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  if (room != hipSuccess) return (int)room;
  const int tiles = ((a.M + T::BM - 1) / T::BM) * ((a.N + T::BN - 1) / T::BN);
  hipLaunchKernelGGL((gemm_mid_fp8_kernel<T, OUT>), dim3(tiles), dim3(T::NW * 64), LDS, st, a, scat);
  return (int)hipGetLastError();
}

template <class T>
static int launch(const Mid8Args& a, const QkvScatter* scat, hipStream_t st) {
  if (a.qo != nullptr) {
    if constexpr (T::BN % 128 == 0) return start<T, MID8_QUANT>(a, QkvScatter{}, st);
    return -1;
  }
  if (scat != nullptr) return start<T, MID8_SCATTER>(a, *scat, st);
  if (a.act == ACT_NONE && a.R != nullptr && a.bias != nullptr && mid_plain_ok(a, T::J * 16, a.sw))
    return start<T, MID8_PLAIN>(a, QkvScatter{}, st);
  return start<T, MID8_ROWS>(a, QkvScatter{}, st);
}

int mid8_launch(int tile, const Mid8Args& a, const QkvScatter* scat, hipStream_t st) {
  switch (tile) {
    case 0: return launch<Mid0Mx>(a, scat, st);
    case 1: return launch<Mid1>(a, scat, st);
    case 2: return launch<Mid2>(a, scat, st);
    case 3: return launch<Mid3>(a, scat, st);
    case 4: return launch<Mid4>(a, scat, st);
  }
  return -1;
}

}  // namespace dnn
