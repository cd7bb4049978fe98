// Gated token input of a decoder layer: g = gelu_tanh(x W^T) * e[token], the
// projection and the product with the token's table row in one launch (bf16
// operands, fp32 accumulation; fp32 variant: the product alone, after
// gemm_f32).  W has few rows (the side dimension, padded to 64), so a plain
// GEMM grid would leave most CUs idle:
//
//   few rows    a workgroup takes 16 columns of 16 or 32 rows; eight waves split
//               K (one round trip for K <= 4096) over W in fragment order
//               (ops/gemm.py shuffle_weight) and reduce through LDS; K of 1024, 2048
//               and 4096 has kernels of its own
//   more rows   64 x 64 tiles on the loop of gemm_mid.h
#include "common.h"
#include "gemm_mid.h"
#include "residual_api.h"

namespace dnn {

struct TokenGate {
  const bf16_t* table;  // token rows, stride ldt; this layer's part starts at off
  const int* tok;
  bf16_t* g;
  int ldt, off, V, ldg, M, n;
};

// Table values of a lane's 4 consecutive columns c..c+3 of row m (transposed
// accumulators), 0 past the part; and the store of their products.
__device__ __forceinline__ void token_gate_row(const TokenGate& t, int m, int c, float (&e)[4]) {
  const bf16_t* p = t.table + (size_t)min(max(t.tok[min(m, t.M - 1)], 0), t.V - 1) * t.ldt + t.off;
#pragma unroll
  for (int r = 0; r < 4; ++r) e[r] = c + r < t.n ? bf2f(p[c + r]) : 0.f;
}
__device__ __forceinline__ void token_gate_store(const TokenGate& t, const f32x4& z, int m, int c,
                                                 const float (&e)[4]) {
  if (m >= t.M) return;
  *reinterpret_cast<uint2*>(t.g + (size_t)m * t.ldg + c) =
      make_uint2(pack2bf(gelu_tanh(z[0]) * e[0], gelu_tanh(z[1]) * e[1]),
                 pack2bf(gelu_tanh(z[2]) * e[2], gelu_tanh(z[3]) * e[3]));
}

constexpr int TG_WAVES = 8, TG_U = 16;  // waves that split K, 32-wide chunks each has in flight

// grid (columns / 16, rows / 16)
__global__ __launch_bounds__(64 * (TG_WAVES + 1)) void token_gate_skinny_kernel(const bf16_t* __restrict__ x, int ldx,
                                                                          const uint8_t* __restrict__ ws, int K,
                                                                          TokenGate t) {
  __shared__ f32x4 red[TG_WAVES][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = blockIdx.y * 16, nch = K / 32;
  const int m = m0 + (lane & 15);
  if (wave == TG_WAVES) {  // the last wave fetches the token rows meanwhile, then reduces
    const int c4 = blockIdx.x * 16 + (lane >> 4) * 4;
    float e[4];
    token_gate_row(t, m, c4, e);
    __syncthreads();
    f32x4 z = red[0][lane];
#pragma unroll
    for (int w = 1; w < TG_WAVES; ++w) z += red[w][lane];
    token_gate_store(t, z, m, c4, e);
    return;
  }
  const uint8_t* wp = ws + (size_t)blockIdx.x * nch * 1024 + lane * 16;
  const bf16_t* xp = x + (size_t)min(m, t.M - 1) * ldx + (lane >> 4) * 8;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int c0 = wave; c0 < nch; c0 += TG_WAVES * TG_U) {
    bf16x8 w[TG_U], a[TG_U];
#pragma unroll
    for (int u = 0; u < TG_U; ++u) {
      const int c = min(c0 + u * TG_WAVES, nch - 1);
      w[u] = *reinterpret_cast<const bf16x8*>(wp + (size_t)c * 1024);
      a[u] = *reinterpret_cast<const bf16x8*>(xp + c * 32);
    }
#pragma unroll
    for (int u = 0; u < TG_U; ++u)
      if (c0 + u * TG_WAVES < nch) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u], a[u], acc, 0, 0, 0);
  }
  red[wave][lane] = acc;
  __syncthreads();
}

// grid (rows / 16 R, columns / 16): eight waves of CH chunks are K, in H parts, everything of a wave in flight at once;
// wave r finishes the 16 rows r.  A wave reads its slice of every row whole (1 KB of K = 4096) and turns it to fragments
// in LDS of its own: read as fragments, 16 pieces of 64 bytes of rows 8 KB apart, 16 rows took 6.3 us of it against 4.4
// (one row, all lanes at one line: 3.6).  In XCDs' turns of rows, so an L2 holds 64 of 512 rows and W.
template <int CH, int R, int H>
struct TgLean {
  static constexpr int CP = CH / H, STRIDE = CP * 64 + 16;  // chunks a part, bytes of a staged row: 16 rows meet all banks
  static constexpr int LPR = CP * 4, RPI = 64 / LPR, NX = R * CP;  // lanes a row, rows a load, loads a part
  static constexpr int WAVE = 16 * R * STRIDE, LDS = TG_WAVES * WAVE;
};

template <int CH, int R, int H>
__global__ __launch_bounds__(64 * TG_WAVES) void token_gate_lean_kernel(const bf16_t* __restrict__ x, int ldx,
                                                                        const uint8_t* __restrict__ ws, TokenGate t) {
  using L = TgLean<CH, R, H>;
  extern __shared__ __attribute__((aligned(16))) char tg_rows[];
  __shared__ f32x4 red[TG_WAVES][R][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int mg = blockIdx.x * (16 * R), m0 = mg + (lane & 15), c4 = blockIdx.y * 16 + (lane >> 4) * 4;
  float e[4];
  if (wave < R) token_gate_row(t, m0 + wave * 16, c4, e);
  const uint8_t* wp = ws + ((size_t)blockIdx.y * TG_WAVES + wave) * (CH * 1024) + lane * 16;
  bf16x8 w[CH], xr[H][L::NX];
  const int xl = wave * (CH * 32) + lane % L::LPR * 8, xrow = L::LPR == 64 ? 0 : lane / L::LPR;
#pragma unroll
  for (int h = 0; h < H; ++h) {
#pragma unroll
    for (int i = 0; i < L::NX; ++i)
      xr[h][i] = *reinterpret_cast<const bf16x8*>(x + (size_t)min(mg + i * L::RPI + xrow, t.M - 1) * ldx + xl + h * (L::CP * 32));
#pragma unroll
    for (int u = 0; u < L::CP; ++u) w[h * L::CP + u] = *reinterpret_cast<const bf16x8*>(wp + (h * L::CP + u) * 1024);
  }
  __builtin_amdgcn_sched_barrier(0);
  f32x4 acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
  char* mine = tg_rows + wave * L::WAVE;
  char* to = mine + xrow * L::STRIDE + lane % L::LPR * 16;
  const char* from = mine + (lane & 15) * L::STRIDE + (lane >> 4) * 16;
#pragma unroll
  for (int h = 0; h < H; ++h) {
#pragma unroll
    for (int i = 0; i < L::NX; ++i) *reinterpret_cast<bf16x8*>(to + i * (L::RPI * L::STRIDE)) = xr[h][i];
    // other lanes read what this one stored, and the next part lies where this one did: the fences keep both orders (a
    // wave's LDS operations run in them)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int u = 0; u < L::CP; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r)
        acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            w[h * L::CP + u], *reinterpret_cast<const bf16x8*>(from + r * (16 * L::STRIDE) + u * 64), acc[r], 0, 0, 0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
#pragma unroll
  for (int r = 0; r < R; ++r) red[wave][r][lane] = acc[r];
  __syncthreads();
  if (wave >= R) return;
  f32x4 z = red[0][wave][lane];
#pragma unroll
  for (int v = 1; v < TG_WAVES; ++v) z += red[v][wave][lane];
  token_gate_store(t, z, m0 + wave * 16, c4, e);
}

template <int CH, int R, int H>
static int token_gate_lean(const TokenGate& t, const void* x, int ldx, const void* ws, int np, hipStream_t st) {
  hipLaunchKernelGGL((token_gate_lean_kernel<CH, R, H>), dim3((t.M + 16 * R - 1) / (16 * R), np / 16), dim3(64 * TG_WAVES),
                     (TgLean<CH, R, H>::LDS), st, (const bf16_t*)x, ldx, (const uint8_t*)ws, t);
  return (int)hipGetLastError();
}

template <class T>
__global__ __launch_bounds__(T::NW * 64, 2) void token_gate_tile_kernel(const bf16_t* __restrict__ x, int ldx,
                                                                        const bf16_t* __restrict__ w, int ldw, int np, int K,
                                                                        TokenGate t) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int I = T::I, J = T::J;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ntn = np / T::BN, b = xcd_remap(blockIdx.x, gridDim.x);
  const int m0 = b / ntn * T::BM, n0 = b % ntn * T::BN, wm = wave / T::WN, wn = wave % T::WN;
  const int mw = m0 + wm * (I * 16) + (lane & 15), cw = n0 + wn * (J * 16) + (lane >> 4) * 4;
  float e[I][J][4];  // gathered ahead of the loop
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) token_gate_row(t, mw + i * 16, cw + j * 16, e[i][j]);
  MidSource<T> src;
  src.init(reinterpret_cast<const char*>(x), ldx * 2, m0, t.M, reinterpret_cast<const char*>(w), ldw * 2, n0, np, 0, K / 64,
           smem, wave, lane);
  f32x4 acc[I][J];
  mid_loop<T>(src, wm, wn, lane, acc);
#pragma unroll
  for (int i = 0; i < I; ++i)
#pragma unroll
    for (int j = 0; j < J; ++j) token_gate_store(t, acc[i][j], mw + i * 16, cw + j * 16, e[i][j]);
}

// g[m, c] = gelu_tanh(z[m, c]) * table[token[m], off + c] for c < n, 0 up to np.
__global__ __launch_bounds__(256) void token_gate_f32_kernel(const float* __restrict__ z, int ldz,
                                                             const float* __restrict__ table, int ldt, int off,
                                                             const int* __restrict__ tok, int V, float* __restrict__ g,
                                                             int ldg, int M, int n, int np) {
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i >= (long)M * np) return;
  const int m = (int)(i / np), c = (int)(i % np);
  float v = 0.f;
  if (c < n) {
    const float x = z[(size_t)m * ldz + c];
    v = 0.5f * x * (1.0f + tanhf(0.797884560802865f * (x + 0.044715f * x * x * x))) *
        table[(size_t)min(max(tok[m], 0), V - 1) * ldt + off + c];
  }
  g[(size_t)m * ldg + c] = v;
}

}  // namespace dnn

using namespace dnn;

extern "C" int dnn_token_gate(const void* x, int ldx, const void* w, int ldw, const void* wsh, int K, const void* table,
                              int ldt, int off, const int* tok, int V, void* g, int ldg, int M, int n, int np,
                              hipStream_t st) {
  if (M <= 0 || n <= 0 || n > np || np % 64 != 0 || K <= 0 || K % 64 != 0 || off < 0 || off + n > ldt || V < 1) return -1;
  if (ldx % 8 != 0 || ldw % 8 != 0 || ldx < K || ldw < K || ldg % 4 != 0 || ldg < np || wsh == nullptr) return -1;
  if ((((uintptr_t)x | (uintptr_t)w | (uintptr_t)wsh) & 15) != 0 || ((uintptr_t)g & 7) != 0) return -1;
  const TokenGate t{(const bf16_t*)table, tok, (bf16_t*)g, ldt, off, V, ldg, M, n};
  // A K that eight waves hold: up to one round of 16 x 16 outputs a workgroup, then up to two of 32 x 16 (a third is
  // behind the tiles).  us, 16 x 16 : 32 x 16 : tiles, 256 columns: K 4096, 256 rows 4.7 : 6.2 : 7.0, 512 rows 8.0 :
  // 7.1 : 13.3, 1024 rows 15 : 12.2 : 15; K 1024, 512 rows 3.7 : 3.4 : 7.3, 1024 rows 5.9 : 5.4 : 7.3; 512 columns, 768
  // rows: K 2048 11.2 : 10.6 : 9.8, K 4096 22 : 19 : 16.
  const int groups = (M + 15) / 16 * (np / 16), pairs = (M + 31) / 32 * (np / 16);
  if (pairs <= 512 && (K == 4096 || K == 2048 || K == 1024)) {
    const bool one = groups <= 256;
    if (K == 4096) return one ? token_gate_lean<16, 1, 1>(t, x, ldx, wsh, np, st) : token_gate_lean<16, 2, 2>(t, x, ldx, wsh, np, st);
    if (K == 2048) return one ? token_gate_lean<8, 1, 1>(t, x, ldx, wsh, np, st) : token_gate_lean<8, 2, 1>(t, x, ldx, wsh, np, st);
    return one ? token_gate_lean<4, 1, 1>(t, x, ldx, wsh, np, st) : token_gate_lean<4, 2, 1>(t, x, ldx, wsh, np, st);
  }
  // Any K, few rows: rounds of 256 workgroups of 16 x 16 outputs, 6.4 us each for K up to 4096;
  // tiles 0.166 us a K-tile of 64 beside 4.9.  us, rounds : tiles: 100 x 64 x 512 7.1 : 6.2, 100 x
  // 256 x 1024 7.1 : 7.5, 512 x 256 x 4096 13.6 : 15.4, 1024 x 256 x 4096 26.5 : 15.7 (30 with the
  // six-stage loop of its own that read a tile's fragments between two barriers)
  const float rounds = (float)(((M + 15) / 16 * (np / 16) + 255) / 256), passes = (float)((K + 4095) / 4096);
  const bool narrow = ldx < 1 << 23 && ldw < 1 << 23;  // the tiles address their 64 rows with 32 bits
  if (M <= 64 || !narrow || 0.7f + 6.4f * rounds * passes < 4.9f + 0.166f * K / 64) {
    hipLaunchKernelGGL(token_gate_skinny_kernel, dim3(np / 16, (M + 15) / 16), dim3(64 * (TG_WAVES + 1)), 0, st,
                       (const bf16_t*)x, ldx, (const uint8_t*)wsh, K, t);
  } else {
    typedef Mid0 T;
    hipLaunchKernelGGL((token_gate_tile_kernel<T>), dim3((unsigned)((M + T::BM - 1) / T::BM * (np / T::BN))), dim3(T::NW * 64),
                       T::S * T::STAGE, st, (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, np, K, t);
  }
  return (int)hipGetLastError();
}

extern "C" int dnn_token_gate_f32(const float* z, int ldz, const float* table, int ldt, int off, const int* tok, int V,
                                  float* g, int ldg, int M, int n, int np, hipStream_t st) {
  if (M <= 0 || n <= 0 || n > np || off < 0 || off + n > ldt || V < 1 || ldg < np || ldz < n) return -1;
  hipLaunchKernelGGL(token_gate_f32_kernel, dim3((unsigned)(((long)M * np + 255) / 256)), dim3(256), 0, st, z, ldz,
                     table, ldt, off, tok, V, g, ldg, M, n, np);
  return (int)hipGetLastError();
}
