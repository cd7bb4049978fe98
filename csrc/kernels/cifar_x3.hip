// CIFAR-10 ConvNet at the reference's fp32 precision on bf16 MFMA ("bf16x3").
//
// The reference computes and ships fp32 (cifar_model_parts.py:7-26,
// node.py:45-48).  gfx950 has f32-input MFMA, but at 1/16 of the bf16 rate
// (cdna_hip_programming.md §3 "FP32-input MFMA"), so every fp32 operand here
// is split into two bf16 terms, x = hi + lo with hi = bf16(x), lo = bf16(x - hi)
// (|x - hi - lo| <= 2^-17 |x|), and each product is accumulated in fp32 as
//     a*b ~= a_hi*b_hi + a_hi*b_lo + a_lo*b_hi        (a_lo*b_lo < 2^-16 |ab| dropped)
// = 3 bf16 MFMAs per fp32 product: 5.3x the f32-MFMA rate at ~2^-16 relative
// error per product before fp32 accumulation.
//
// Kernels:
//  * cifar_stage0_x3_kernel: conv1+bias+ReLU+pool -> conv2+bias+ReLU+pool ->
//    NCHW flatten, fp32 in, fp32 (B,4096) out (reference ModelPart0_2Node,
//    cifar_model_parts.py:37-42); up to two images a workgroup (more: cifar_wino.hip).  Persistent, 512 threads: waves 0-3
//    ("producers") stage input image it+1 and run conv1 of image it, waves 4-7
//    ("consumers") run conv2 of image it-1, one barrier per image, so each SIMD
//    pairs a VALU/LDS-heavy wave with an MFMA-heavy one.  Per image: 32 conv1
//    tiles x 3 k-steps x 3 terms + 16 conv2 tiles x 18 k-steps x 3 terms = 1152
//    v_mfma_f32_32x32x16_bf16.  LDS (126,464 B): input double-buffered as
//    hi/lo HWC4 planes [34][40][4] (pitch 40: conflict-free conv1 b64 reads),
//    pooled conv1 map double-buffered as hi/lo planes [18][18][32] with the
//    16-B chunk XORed by (Y & 3), which makes every conv2 ds_read_b128 fragment
//    (four 16-lane groups) conflict-free; conv2 results leave straight from
//    the accumulators as 8-B fp32 stores (no LDS staging).
//  * cifar_fc1_x3_kernel: fc1 + bias + ReLU on the fp32 boundary tensor, the
//    split done in registers between LDS and the MFMAs (no split copy in HBM):
//    256x256x32 tiles, 8 waves of 64x128, per k32 step 3 x 32
//    mfma_f32_16x16x32_bf16 per wave (A_hi W_hi + A_hi W_lo + A_lo W_hi); K in
//    ranges where the tiles do not fill the chip, summed by cifar_fc1_sum_kernel.
//  * cifar_split3_kernel: fp32 (B,K) -> bf16 (B,3K) = [hi | hi | lo], the A
//    operand of fc1 where the kernel above does not write the output or fetch the
//    rows (one bf16 GEMM over K' = 3K against W' = [W_hi | W_lo | W_hi]).
//  * cifar_stage0_x3_band_kernel, cifar_fc1_few_kernel, cifar_head_few_kernel: the
//    same stages where the batch is too small to fill the chip with whole images.
//  * cifar_head_tail_x3_kernel: fc2 (512->10) + bias + softmax + per-row argmax
//    on fp32 hidden rows, 3-term split on mfma_f32_16x16x32_bf16.
#include <climits>
#include <type_traits>

#include "cifar_conv.h"
#include "gemm_epilogue.h"
#include "gemm_tile.h"

namespace dnn {

using namespace x3;

// SPLIT_OUT: the boundary leaves in the blocked hi/lo encoding
// (cifar_split_blocked_kernel) that cifar_fc1_x3_kernel<true> stages by DMA.
// keep: where given, a copy of the images is left there, from the registers they are
// split in; the kernel is bound by its products and HBM has room.  A copy kernel of
// its own in front took 301 us of a pass of 65536 images.
template <bool WIDE, bool SPLIT_OUT>
__global__ __launch_bounds__(512, 1) void cifar_stage0_x3_kernel(
    const float* __restrict__ x, float* __restrict__ out, const bf16_t* __restrict__ w1h,
    const bf16_t* __restrict__ w1l, const float* __restrict__ b1, const bf16_t* __restrict__ w2h,
    const bf16_t* __restrict__ w2l, const float* __restrict__ b2, float* __restrict__ keep, int B) {
  __shared__ __attribute__((aligned(16))) char smem[LDS_BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool producer = wave < 4;
  const int rw = wave & 3;
  const int rt = tid & 255;
  const int h = lane >> 5, r32 = lane & 31;
  const int n = B > (int)blockIdx.x ? (B - 1 - (int)blockIdx.x) / (int)gridDim.x + 1 : 0;

  // every halo (input and pooled map) is zero for the whole launch; interiors are rewritten per image
  for (int i = tid; i < LDS_BYTES / 16; i += 512) reinterpret_cast<uint4*>(smem)[i] = make_uint4(0, 0, 0, 0);

  __syncthreads();  // halos zeroed before any image is staged

  // The two roles run disjoint loops (wave-uniform branch, the same number of
  // barriers on both sides) so their resident operands never share live ranges:
  // producers hold conv1's split weights + the input prefetch, consumers the
  // 144 VGPRs of conv2's split weights.
  if (producer) {
    bf16x8 w1hf[3], w1lf[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      w1hf[s] = *reinterpret_cast<const bf16x8*>(w1h + r32 * 48 + s * 16 + h * 8);
      w1lf[s] = *reinterpret_cast<const bf16x8*>(w1l + r32 * 48 + s * 16 + h * 8);
    }
    const float bias = b1[r32];
    resident_fence(w1hf);
    resident_fence(w1lf);
    asm volatile("" ::"v"(bias));

    float pf[4][3];
    auto load_img = [&](int k) {
      const float* xb = x + (size_t)(blockIdx.x + (size_t)k * gridDim.x) * 3072;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < 3; ++c) pf[i][c] = xb[c * 1024 + rt + 256 * i];
    };
    auto stage_img = [&](int k) {  // prefetch registers -> padded HWC4 hi / lo planes
      char* xh = smem + xin_off(k, 0);
      char* xl = smem + xin_off(k, 1);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = rt + 256 * i, yy = p >> 5, xx = p & 31;
        uint2 vh, vl;
        split2(pf[i][0], pf[i][1], vh.x, vl.x);
        split2(pf[i][2], 0.f, vh.y, vl.y);
        const int o = ((yy + 1) * XW + xx + 1) * 8;
        *reinterpret_cast<uint2*>(xh + o) = vh;
        *reinterpret_cast<uint2*>(xl + o) = vl;
      }
      if (keep != nullptr) {
        float* kb = keep + (size_t)(blockIdx.x + (size_t)k * gridDim.x) * 3072;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int c = 0; c < 3; ++c) kb[c * 1024 + rt + 256 * i] = pf[i][c];
      }
    };
    if (n > 0) {
      load_img(0);
      stage_img(0);
      if (n > 1) load_img(1);
    }
    __syncthreads();
    for (int it = 0; it <= n; ++it) {
      if (it < n) {
#pragma unroll 1
        for (int t = rw; t < 32; t += 8)
          conv1_pair(smem + xin_off(it, 0), smem + a1_off(it, 0), t, t + 4, w1hf, w1lf, bias, lane);
        if (it + 1 < n) {
          stage_img(it + 1);
          if (it + 2 < n) load_img(it + 2);
        }
      }
      __syncthreads();
    }
  } else {
    const int oc2 = (rw & 1) * 32 + r32;
    bf16x8 w2hf[18], w2lf[18];
#pragma unroll
    for (int s = 0; s < 18; ++s) {
      w2hf[s] = *reinterpret_cast<const bf16x8*>(w2h + oc2 * 288 + s * 16 + h * 8);
      w2lf[s] = *reinterpret_cast<const bf16x8*>(w2l + oc2 * 288 + s * 16 + h * 8);
    }
    const float bias = b2[oc2];
    resident_fence(w2hf);
    resident_fence(w2lf);
    asm volatile("" ::"v"(bias));
    // lane base for (ky, channel-chunk parity): pixel row Y = 4*ty2 + (r32>>3) + ky,
    // Y & 3 = ((r32>>3) + ky) & 3 (4*ty2 = 0 mod 4), chunk = 2*par + h
    uint32_t lb[3][2];
#pragma unroll
    for (int ky = 0; ky < 3; ++ky)
#pragma unroll
      for (int par = 0; par < 2; ++par) {
        const int yr = (r32 >> 3) + ky;
        lb[ky][par] = (uint32_t)((yr * 18 + (r32 & 7)) * 64 + (((2 * par + h) ^ (yr & 3)) << 4));
      }

    auto conv2_img = [&](int k) {  // conv2 + bias + ReLU + pool of image k -> out (fp32, NCHW flatten)
      float* ob = out + (size_t)(blockIdx.x + (size_t)k * gridDim.x) * 4096 + oc2 * 64;
      const uint32_t plane = (uint32_t)(uintptr_t)(smem + a1_off(k, 0));
#pragma unroll 1
      for (int p = 0; p < 2; ++p) {
        const int ty2 = (rw >> 1) * 2 + p;
        const uint32_t rb = plane + ty2 * 4 * 18 * 64;
        uint32_t b[3][2];
#pragma unroll
        for (int ky = 0; ky < 3; ++ky)
#pragma unroll
          for (int par = 0; par < 2; ++par) b[ky][par] = rb + lb[ky][par];
        f32x16 acc[2] = {f32x16{}, f32x16{}};
        bf16x8 a0[4], a1[4];
        c2_issue<0>(b, a0);
        c2_step<0>(b, w2hf, w2lf, acc, a0, a1);
        if constexpr (WIDE) {
          // 16-B stores: lane half h holds pooled columns 4i+2h..+1 of both
          // tiles; one v_permlane32_swap per dword gives half 0 columns 0-3
          // (its own tile-0 pair + the other half's) and half 1 columns 4-7,
          // so a row leaves as one dwordx4 per lane instead of two dwordx2
#pragma unroll
          for (int qy = 0; qy < 2; ++qy) {
            const int g0 = (2 * qy) * 4;
            float v[2][2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              v[i][0] = fmaxf(fmax_nan(fmax_nan(acc[i][g0], acc[i][g0 + 1]), fmax_nan(acc[i][g0 + 4], acc[i][g0 + 5])) + bias, 0.f);
              v[i][1] = fmaxf(fmax_nan(fmax_nan(acc[i][g0 + 2], acc[i][g0 + 3]), fmax_nan(acc[i][g0 + 6], acc[i][g0 + 7])) + bias,
                              0.f);
            }
            const auto sx = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0][0]), __float_as_uint(v[1][0]), false,
                                                             false);
            const auto sy = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0][1]), __float_as_uint(v[1][1]), false,
                                                             false);
            const int PY = 2 * ty2 + qy;
            if constexpr (SPLIT_OUT) {  // k = oc2*64 + PY*8 + 4h + 0..3: one 8-B hi and one 8-B lo store
              uint2 hi, lo;
              split2(__uint_as_float(sx[0]), __uint_as_float(sy[0]), hi.x, lo.x);
              split2(__uint_as_float(sx[1]), __uint_as_float(sy[1]), hi.y, lo.y);
              char* bp = reinterpret_cast<char*>(ob - oc2 * 64) + (oc2 * 2 + (PY >> 2)) * 128 + ((PY & 3) * 8 + 4 * h) * 2;
              *reinterpret_cast<uint2*>(bp) = hi;
              *reinterpret_cast<uint2*>(bp + 64) = lo;
            } else {
              *reinterpret_cast<uint4*>(ob + PY * 8 + 4 * h) = make_uint4(sx[0], sy[0], sx[1], sy[1]);
            }
          }
        } else {
#pragma unroll
          for (int i = 0; i < 2; ++i) conv2_store<SPLIT_OUT>(ob - oc2 * 64, oc2, ty2, i, acc[i], bias, h);
        }
      }
    };

    __syncthreads();
    for (int it = 0; it <= n; ++it) {
      if (it >= 1) conv2_img(it - 1);
      __syncthreads();
    }
  }
}

// Stage 0 of a few images: one workgroup per image and band of 4 conv2 rows
// (ty2), so that 4 B workgroups share what one of the persistent kernel does in a
// row: conv1 of the 3 or 4 tile rows that the band's pooled map touches (waves
// 0-3, two pairs of tiles each; 1.5x the work of one image over the 4 bands), then
// conv2 of the band, one 32x32 tile a wave (waves 4-7, their weights loaded while
// conv1 runs).  Tiles, products and their order are those of the persistent kernel:
// the results are the same bits.  Bound by its chain (load, stage, conv1, barrier,
// 54 dependent MFMAs, store): 7.3 us where the persistent kernel takes 11.0 for one
// image.  Taken while the bands of all images run at once (4 B <= grid): with 256
// VGPRs a CU holds one workgroup, so beyond that the bands would queue.
template <bool SPLIT_OUT>
__global__ __launch_bounds__(512, 1) void cifar_stage0_x3_band_kernel(
    const float* __restrict__ x, float* __restrict__ out, const bf16_t* __restrict__ w1h,
    const bf16_t* __restrict__ w1l, const float* __restrict__ b1, const bf16_t* __restrict__ w2h,
    const bf16_t* __restrict__ w2l, const float* __restrict__ b2, float* __restrict__ keep) {
  constexpr int A1 = 2 * XPL;  // xin hi | lo, pooled map hi | lo
  __shared__ __attribute__((aligned(16))) char smem[A1 + 2 * A1PL];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rw = wave & 3, h = lane >> 5, r32 = lane & 31;
  const int ty2 = blockIdx.x & 3;
  const size_t img = blockIdx.x >> 2;

  float px[2][3];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int c = 0; c < 3; ++c) px[i][c] = x[img * 3072 + c * 1024 + tid + 512 * i];
  for (int i = tid; i < (A1 + 2 * A1PL) / 16; i += 512) reinterpret_cast<uint4*>(smem)[i] = make_uint4(0, 0, 0, 0);
  __syncthreads();  // halos are zero before the interior is written
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = tid + 512 * i, o = (((p >> 5) + 1) * XW + (p & 31) + 1) * 8;
    uint2 vh, vl;
    split2(px[i][0], px[i][1], vh.x, vl.x);
    split2(px[i][2], 0.f, vh.y, vl.y);
    *reinterpret_cast<uint2*>(smem + o) = vh;
    *reinterpret_cast<uint2*>(smem + XPL + o) = vl;
    if (keep != nullptr && (p >> 8) == ty2) {  // every band a quarter of the pixels
#pragma unroll
      for (int c = 0; c < 3; ++c) keep[img * 3072 + c * 1024 + p] = px[i][c];
    }
  }
  if (wave < 4) {
    bf16x8 w1hf[3], w1lf[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      w1hf[s] = *reinterpret_cast<const bf16x8*>(w1h + r32 * 48 + s * 16 + h * 8);
      w1lf[s] = *reinterpret_cast<const bf16x8*>(w1l + r32 * 48 + s * 16 + h * 8);
    }
    const float bias = b1[r32];
    __syncthreads();
    const int ty = 2 * ty2 - 1 + rw;  // conv1 tile row: pooled rows 2 ty, 2 ty + 1
    if (ty >= 0 && ty < 8) {
      conv1_pair(smem, smem + A1, 4 * ty, 4 * ty + 1, w1hf, w1lf, bias, lane);
      conv1_pair(smem, smem + A1, 4 * ty + 2, 4 * ty + 3, w1hf, w1lf, bias, lane);
    }
    __syncthreads();
  } else {
    const int oc2 = (rw & 1) * 32 + r32, i = rw >> 1;
    bf16x8 w2hf[18], w2lf[18];
#pragma unroll
    for (int s = 0; s < 18; ++s) {
      w2hf[s] = *reinterpret_cast<const bf16x8*>(w2h + oc2 * 288 + s * 16 + h * 8);
      w2lf[s] = *reinterpret_cast<const bf16x8*>(w2l + oc2 * 288 + s * 16 + h * 8);
    }
    const float bias = b2[oc2];
    resident_fence(w2hf);
    resident_fence(w2lf);
    __syncthreads();
    __syncthreads();
    f32x16 acc = {};
#pragma unroll
    for (int s = 0; s < 18; ++s) {
      const int ky = (s >> 1) / 3, kx = (s >> 1) % 3, yr = (r32 >> 3) + ky;
      const char* p = smem + A1 + ((4 * ty2 + yr) * 18 + 8 * i + (r32 & 7) + kx) * 64 + (((2 * (s & 1) + h) ^ (yr & 3)) << 4);
      const bf16x8 hi = *reinterpret_cast<const bf16x8*>(p), lo = *reinterpret_cast<const bf16x8*>(p + A1PL);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, w2hf[s], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hi, w2lf[s], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(lo, w2hf[s], acc, 0, 0, 0);
    }
    conv2_store<SPLIT_OUT>(out + img * 4096, oc2, ty2, i, acc, bias, h);
  }
}

// ---------------------------------------------------------------------------
// fc1 at fp32 precision: C = relu(A . W^T + bias), A fp32 [M][K], W = W_hi + W_lo
// (bf16 [N][K] each), C fp32.  256 x 256 tiles, 8 waves (4 M x 2 N) of 2 x 2
// quadrants of 32 x 64, k-steps of 32.  Both operands come by LDS-DMA in half-tiles
// of 128 rows (16 KiB: A as the fp32 it is, W as a hi and a lo plane of 64-byte
// rows), and the waves of column 1 run one barrier behind those of column 0, so that
// on every SIMD one wave reads and splits while the other multiplies.  A phase is one
// quadrant, 24 MFMAs:
//
//   ph1: read B0, fetch A1       | split A0 | stage B1[t+1] | C00
//   ph2:                         | split A1 | stage A0[t+2] | C10
//   ph3: read B1                 |          | stage B0[t+2] | C11
//   ph4: fetch A0[t+1]           |          | stage A1[t+2] | C01
//
// A wave fetches its 32 rows of a half of A as fp32 and splits them in registers in the
// next phase; two waves split the same rows.  (With 2 M x 4 N waves four do: the kernel
// is at the card's power limit, and the fewer vector operations count: 657 us at 65536
// x 512 x 4096, here 624.  Splitting once in LDS, in place, costs as much in LDS traffic:
// 640.  With A loaded to registers, split and written to LDS between two barriers: 681.
// A that arrives split: 549.)  A half-tile is staged again at the earliest two phases
// behind its last read, and a DMA has four to five phases until it is waited for.
//
// A's 16-byte chunk c (4 floats) of a row lies in slot ((c >> 1 | (c & 1) << 2) ^
// swz_chunk(row)): a lane's 8 floats are then slots g and 4 + g, which are read without
// conflicts.  W's chunk c of a 64-byte row lies at c ^ ((r >> 2) & 2).
//
// SPLIT_IN: A arrives pre-split in the blocked boundary encoding (see
// cifar_split_blocked_kernel: per row and 32-k block, 32 bf16 hi then 32 bf16
// lo, the same 128 bytes), and nothing is split here.
//
// splits > 1: K in that many ranges over the workgroups, whose sums are left in `part` [splits][M][N].
// ---------------------------------------------------------------------------
constexpr int F1_T = 256, F1_K = 32;

__device__ __forceinline__ int f1_swz(int r) { return (r >> 2) & 2; }

// The 24 products of a phase, between barriers: hi.hi, then W_lo A_hi, then W_hi A_lo of
// every accumulator
__device__ __forceinline__ void f1_mfma(f32x4 (&acc)[2][4], const bf16x8 (&a)[2][2], const bf16x8 (&b)[4][2]) {
  bg_barrier();
  __builtin_amdgcn_s_setprio(1);
#pragma unroll
  for (int jp = 0; jp < 4; jp += 2)  // the first fragments of W to arrive first
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
      for (int j = jp; j < jp + 2; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j][s == 1], a[i][s == 2], acc[i][j], 0, 0, 0);
  __builtin_amdgcn_s_setprio(0);
  bg_barrier();
}

template <bool SPLIT_IN>
__global__ __launch_bounds__(512, 1) void cifar_fc1_x3_kernel(const float* __restrict__ A, int lda,
                                                              const bf16_t* __restrict__ Wh,
                                                              const bf16_t* __restrict__ Wl, int ldw,
                                                              const float* __restrict__ bias, float* __restrict__ C,
                                                              int ldc, int M, int N, int K, int splits,
                                                              float* __restrict__ part) {
  __shared__ __attribute__((aligned(1024))) char smem[8 * BG_HALF];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntn = N / F1_T, ntm = (M + F1_T - 1) / F1_T;
  // columns fastest: the tiles of one panel of A run close together on one XCD, and its second
  // read hits L2 or the last-level cache (panels in groups of 8, rows fastest: no difference)
  const int id = xcd_remap(blockIdx.x, ntm * ntn * splits), sp = id / (ntm * ntn), tile = id - sp * ntm * ntn;
  const int tm = tile / ntn, tn = tile - tm * ntn;
  const int m0 = tm * F1_T, n0 = tn * F1_T;
  const int wr = wave & 3, wc = wave >> 2, fr = lane & 15, fg = lane >> 4;
  const int nkall = K / F1_K, k0 = nkall * sp / splits, nk = nkall * (sp + 1) / splits - k0;  // host: splits <= nkall
  auto half = [&](int u, int h) { return smem + (u * 4 + h) * BG_HALF; };  // h: A0, A1, B0, B1

  // A: pieces of 8 rows of 128 bytes, 2 of either half a wave: uniform row bases, the
  // lane's row (clamped for rows past the matrix) and chunk as 32-bit offsets
  const uint32_t ldb = (uint32_t)lda * 4u;
  const char* abase[4];
  uint32_t alim[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int r = min(m0 + (x >> 1) * 128 + ((x & 1) * 8 + wave) * 8, M - 1);
    abase[x] = reinterpret_cast<const char*>(A) + (size_t)r * ldb + (size_t)k0 * 128;
    alim[x] = (uint32_t)min(7, M - 1 - r) * ldb;
  }
  const int slot = (lane & 7) ^ ((wave & 1) * 4 + (lane >> 4));  // swz_chunk of the lane's row in its piece
  const uint32_t arow_off = (uint32_t)(lane >> 3) * ldb, achunk = (SPLIT_IN ? slot : (slot & 3) << 1 | slot >> 2) * 16u;
  auto stA = [&](int u, int h, int t) {
    t = t < nk ? t : nk - 1;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const char* p = abase[2 * h + i] + (size_t)t * 128;
      asm("" : "+s"(p));  // scalar base, 32-bit lane offset: not folded into per-lane addresses ahead of the loop
      glds16(p + (min(arow_off, alim[2 * h + i]) + achunk), half(u, h) + (i * 8 + wave) * 1024);
    }
  };
  // W: a wave stages 16 rows of 64 bytes of a half's hi and of its lo plane
  const char* wbase[2];
#pragma unroll
  for (int p = 0; p < 2; ++p)
    wbase[p] = reinterpret_cast<const char*>(p ? Wl : Wh) + (size_t)(n0 + wave * 16) * ldw * 2 + (size_t)k0 * 64;
  const uint32_t woff = (uint32_t)(lane >> 2) * (uint32_t)ldw * 2u + (uint32_t)((lane & 3) ^ f1_swz(lane >> 2)) * 16u;
  auto stB = [&](int u, int h, int t) {
    t = t < nk ? t : nk - 1;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const char* s = wbase[p] + (size_t)h * 256 * ldw + (size_t)t * 64;
      asm("" : "+s"(s));
      glds16(s + woff, half(u, 2 + h) + p * (BG_HALF / 2) + wave * 1024);
    }
  };

  f32x4 acc[2][2][2][4];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[a][b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  bf16x8 a0[2][2], a1[2][2], bb[4][2];
  f32x4 raw[2][2];
  const int arow = wr * 32 + fr, brow = wc * 64 + fr;
  // LDS offsets of the lane's fragments, moved from buffer to buffer: 128 KiB are more
  // than a read's immediate offset reaches, and registers for both would spill
  uint32_t ao[2], bo = 2 * BG_HALF + brow * 64 + ((fg ^ f1_swz(brow)) << 4);
#pragma unroll
  for (int s = 0; s < 2; ++s) ao[s] = arow * 128 + (((s * 4 + fg) ^ swz_chunk(arow)) << 4);
  auto fetch = [&](int h) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) raw[i][s] = *reinterpret_cast<const f32x4*>(smem + ao[s] + (h * BG_HALF + i * 2048));
  };
  auto fetched = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  auto split = [&](bf16x8 (&a)[2][2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (SPLIT_IN) {
#pragma unroll
        for (int s = 0; s < 2; ++s) a[i][s] = __builtin_bit_cast(bf16x8, raw[i][s]);
      } else {
        uint4 hi, lo;
        split2(raw[i][0][0], raw[i][0][1], hi.x, lo.x);
        split2(raw[i][0][2], raw[i][0][3], hi.y, lo.y);
        split2(raw[i][1][0], raw[i][1][1], hi.z, lo.z);
        split2(raw[i][1][2], raw[i][1][3], hi.w, lo.w);
        a[i][0] = __builtin_bit_cast(bf16x8, hi);
        a[i][1] = __builtin_bit_cast(bf16x8, lo);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // the next fragments take raw's registers
  };
  auto readB = [&](int h) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int p = 0; p < 2; ++p)
        bb[j][p] = *reinterpret_cast<const bf16x8*>(smem + bo + (h * BG_HALF + p * (BG_HALF / 2) + j * 1024));
    __builtin_amdgcn_sched_barrier(0);
  };

  // prologue: A0, B0 and A1 of tile 0 landed, four half-tiles in flight
  stA(0, 0, 0);
  stB(0, 0, 0);
  stA(0, 1, 0);
  stB(0, 1, 0);
  stA(1, 0, 1);
  stB(1, 0, 1);
  stA(1, 1, 1);
  bg_landed<8>();
  bg_barrier();
  if (wc == 1) bg_barrier();
  fetch(0);

  for (int t = 0, u = 0; t < nk; ++t, u ^= 1) {
    // ph1
    fetched();
    readB(0);
    split(a0);
    fetch(1);
    stB(u ^ 1, 1, t + 1);
    f1_mfma(acc[0][0], a0, bb);
    // ph2
    fetched();
    split(a1);
    stA(u, 0, t + 2);
    bg_landed<10>();  // B1 of tile t
    f1_mfma(acc[1][0], a1, bb);
    // ph3
    readB(1);
    stB(u, 0, t + 2);
    bg_landed<10>();  // A0 of tile t + 1
    f1_mfma(acc[1][1], a1, bb);
    // ph4
    fetched();
    ao[0] ^= 4 * BG_HALF, ao[1] ^= 4 * BG_HALF, bo ^= 4 * BG_HALF;
    fetch(0);
    stA(u, 1, t + 2);
    bg_landed<8>();  // B0 and A1 of tile t + 1
    f1_mfma(acc[0][1], a0, bb);
  }
  fetched();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (wc == 0) bg_barrier();

  // epilogue (transposed accumulators): row m0 + mq 128 + wr 32 + i 16 + (lane & 15), cols n..n+3
  if (splits > 1) {  // this range's sums: cifar_fc1_sum_kernel finishes
    float* d = part + (size_t)sp * M * N;
#pragma unroll
    for (int mq = 0; mq < 2; ++mq)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int m = m0 + mq * 128 + arow + i * 16;
        if (m < M) {
#pragma unroll
          for (int nq = 0; nq < 2; ++nq)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              *reinterpret_cast<f32x4*>(d + (size_t)m * N + n0 + nq * 128 + wc * 64 + j * 16 + fg * 4) = acc[mq][nq][i][j];
        }
      }
    return;
  }
  const bool vec = epi_vec_ok(C, ldc, bias, nullptr, 0);
#pragma unroll
  for (int mq = 0; mq < 2; ++mq)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int m = m0 + mq * 128 + arow + i * 16;
#pragma unroll
      for (int nq = 0; nq < 2; ++nq)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          epi_t4<ACT_RELU, true>(acc[mq][nq][i][j], m, n0 + nq * 128 + wc * 64 + j * 16 + fg * 4, M, N, C, ldc, bias,
                                 nullptr, 0, vec);
    }
}

// relu(sum of the parts + bias), 4 columns a thread; bound by reading the parts.
__global__ __launch_bounds__(256) void cifar_fc1_sum_kernel(const float* __restrict__ part, const float* __restrict__ bias,
                                                            float* __restrict__ C, int ldc, int M, int N, int splits) {
  const int n4 = N / 4, e = blockIdx.x * 256 + threadIdx.x, m = e / n4, n = (e - m * n4) * 4;
  if (m >= M) return;
  const float* d = part + (size_t)m * N + n;
  f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < splits; ++s) v += *reinterpret_cast<const f32x4*>(d + (size_t)s * M * N);
  v += *reinterpret_cast<const f32x4*>(bias + n);
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = fmaxf(v[r], 0.f);
  *reinterpret_cast<f32x4*>(C + (size_t)m * ldc + n) = v;
}

// Blocked boundary encoding of an fp32 (M,K) tensor, in place of the same
// 4 bytes per element: row r, 32-k block b holds 32 bf16 hi then 32 bf16 lo
// (hi + lo == x to ~2^-17 relative, the exact operand split of the x3 MFMAs).
// dir 0: fp32 -> blocked, dir 1: blocked -> fp32 (hi + lo).  K % 32 == 0.
__global__ __launch_bounds__(256) void cifar_split_blocked_kernel(const float* __restrict__ a, float* __restrict__ o,
                                                                  int M, int K, int dir) {
  const int per_row = K / 8;  // 8-element pieces
  const long total = (long)M * per_row;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const int m = (int)(e / per_row), k = (int)(e % per_row) * 8;
    char* rowp = reinterpret_cast<char*>(o + (size_t)m * K);
    const char* rowa = reinterpret_cast<const char*>(a + (size_t)m * K);
    const int hoff = (k >> 5) * 128 + (k & 31) * 2;
    if (dir == 0) {
      const float4 u = *reinterpret_cast<const float4*>(rowa + k * 4);
      const float4 v = *reinterpret_cast<const float4*>(rowa + k * 4 + 16);
      uint4 hi, lo;
      split2(u.x, u.y, hi.x, lo.x);
      split2(u.z, u.w, hi.y, lo.y);
      split2(v.x, v.y, hi.z, lo.z);
      split2(v.z, v.w, hi.w, lo.w);
      *reinterpret_cast<uint4*>(rowp + hoff) = hi;
      *reinterpret_cast<uint4*>(rowp + hoff + 64) = lo;
    } else {
      const uint4 hi = *reinterpret_cast<const uint4*>(rowa + hoff);
      const uint4 lo = *reinterpret_cast<const uint4*>(rowa + hoff + 64);
      const uint32_t h[4] = {hi.x, hi.y, hi.z, hi.w}, l[4] = {lo.x, lo.y, lo.z, lo.w};
      float r[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r[2 * i] = __uint_as_float(h[i] << 16) + __uint_as_float(l[i] << 16);
        r[2 * i + 1] = __uint_as_float(h[i] & 0xffff0000u) + __uint_as_float(l[i] & 0xffff0000u);
      }
      *reinterpret_cast<float4*>(rowp + k * 4) = float4{r[0], r[1], r[2], r[3]};
      *reinterpret_cast<float4*>(rowp + k * 4 + 16) = float4{r[4], r[5], r[6], r[7]};
    }
  }
}

// fp32 (M,K) -> bf16 (M,3K) rows [hi | hi | lo]; K % 8 == 0, plain loads: rows of a may start
// at any float.
// blocked = 1: a is in the blocked hi/lo encoding (the split is already done).
__global__ __launch_bounds__(256) void cifar_split3_kernel(const float* __restrict__ a, int lda,
                                                           bf16_t* __restrict__ o, int ldo, int M, int K,
                                                           int blocked) {
  const int per_row = K / 8;
  const long total = (long)M * per_row;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const int m = (int)(e / per_row), c = (int)(e % per_row) * 8;
    uint4 hi, lo;
    if (blocked) {
      const char* rowa = reinterpret_cast<const char*>(a + (size_t)m * lda) + (c >> 5) * 128 + (c & 31) * 2;
      hi = *reinterpret_cast<const uint4*>(rowa);
      lo = *reinterpret_cast<const uint4*>(rowa + 64);
    } else {
      const float4 u = *reinterpret_cast<const float4*>(a + (size_t)m * lda + c);
      const float4 v = *reinterpret_cast<const float4*>(a + (size_t)m * lda + c + 4);
      split2(u.x, u.y, hi.x, lo.x);
      split2(u.z, u.w, hi.y, lo.y);
      split2(v.x, v.y, hi.z, lo.z);
      split2(v.z, v.w, hi.w, lo.w);
    }
    bf16_t* r = o + (size_t)m * ldo + c;
    *reinterpret_cast<uint4*>(r) = hi;
    *reinterpret_cast<uint4*>(r + K) = hi;
    *reinterpret_cast<uint4*>(r + 2 * K) = lo;
  }
}

// fc2 (512->10) + bias + softmax + argmax on fp32 hidden rows (fc1+ReLU output).
// One wave per 16 rows and iteration, mfma_f32_16x16x32_bf16 with the 3-term split:
// A = hid rows (lane: row l&15, k 8*(l>>4)+j), B = W2 hi/lo padded to 16 classes in VGPRs.
__global__ __launch_bounds__(256) void cifar_head_tail_x3_kernel(const float* __restrict__ hid,
                                                                 const bf16_t* __restrict__ w2h,
                                                                 const bf16_t* __restrict__ w2l,
                                                                 const float* __restrict__ b2,
                                                                 float* __restrict__ probs, int* __restrict__ pred,
                                                                 int B) {
  const int lane = threadIdx.x & 63;
  const int gw = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int nw = (gridDim.x * blockDim.x) >> 6;
  const int col = lane & 15, kq = (lane >> 4) * 8;
  bf16x8 wfh[16], wfl[16];
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    wfh[s] = *reinterpret_cast<const bf16x8*>(w2h + col * 512 + s * 32 + kq);
    wfl[s] = *reinterpret_cast<const bf16x8*>(w2l + col * 512 + s * 32 + kq);
  }
  const float bias = col < 10 ? b2[col] : 0.f;
  for (int r0 = gw * 16; r0 < B; r0 += nw * 16) {
    const int row = r0 + (lane & 15);
    const int rc = row < B ? row : B - 1;
    const float* ap = hid + (size_t)rc * 512 + kq;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 16; ++s) {
      const float4 u = *reinterpret_cast<const float4*>(ap + s * 32);
      const float4 v = *reinterpret_cast<const float4*>(ap + s * 32 + 4);
      uint4 hi, lo;
      split2(u.x, u.y, hi.x, lo.x);
      split2(u.z, u.w, hi.y, lo.y);
      split2(v.x, v.y, hi.z, lo.z);
      split2(v.z, v.w, hi.w, lo.w);
      const bf16x8 ah = __builtin_bit_cast(bf16x8, hi), al = __builtin_bit_cast(bf16x8, lo);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, wfh[s], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, wfl[s], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, wfh[s], acc, 0, 0, 0);
    }
    // acc[r] = logit(row = r0 + (lane>>4)*4 + r, class = col)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float z = col < 10 ? acc[r] + bias : -INFINITY;
      float mx = z;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
      const float e = col < 10 ? expf(z - mx) : 0.f;
      float sum = e;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) sum += __shfl_xor(sum, o, 64);
      int cand = (z == mx) ? col : 16;  // smallest class index attaining the max (numpy semantics)
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) cand = min(cand, __shfl_xor(cand, o, 64));
      const int m = r0 + (lane >> 4) * 4 + r;
      if (m < B) {
        if (col < 10) probs[(size_t)m * 10 + col] = e / sum;
        if (col == 0) pred[m] = cand;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The head of a few images: fc1 as HS_S slices of K over HS_S x 32 workgroups, each
// reading its 16 columns x 512 k of W_hi and W_lo once for all rows, and a finish
// that sums the slices in order and, one workgroup a row, goes on to fc2, softmax
// and argmax.
//
// One row costs 8 MB of weights and nothing else: the GEMM over K' = 3 K that larger
// batches take reads 12.6 MB on 32 workgroups.  A wave holds its 64 k of the weights
// in registers and takes the rows 16 at a time (products and split of the fp32 rows
// as in the other fc1 paths); the 8 waves meet in LDS and the slice's sums leave as
// part[slice][row][512].  Slice = block & 7: the workgroups of one XCD share one
// slice of the rows in its L2.  One row: 3.8 + 3.4 us for the two launches; split,
// GEMM and tail took 3.2 + 16.8 + 9.8 us.
constexpr int HS_S = 8, HS_N = 512, HS_K = 4096;

template <bool BLOCKED>
__global__ __launch_bounds__(512) void cifar_fc1_few_kernel(const float* __restrict__ A, const bf16_t* __restrict__ Wh,
                                                            const bf16_t* __restrict__ Wl, float* __restrict__ part,
                                                            int M) {
  __shared__ __attribute__((aligned(16))) float red[2][8][32 * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, kq = (lane >> 4) * 8;
  const int slice = blockIdx.x & (HS_S - 1), n0 = (blockIdx.x / HS_S) * 16;
  const int k0 = slice * (HS_K / HS_S) + wave * 64;
  const size_t wo = (size_t)(n0 + r16) * HS_K + k0 + kq;
  bf16x8 wh[2], wl[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    wh[s] = *reinterpret_cast<const bf16x8*>(Wh + wo + s * 32);
    wl[s] = *reinterpret_cast<const bf16x8*>(Wl + wo + s * 32);
  }
  uint4 a[2][2][2];  // 16-row tile, k32 step, 32 B of the lane's row (fp32 k 0-3, 4-7 or hi, lo)
  auto load = [&](int m0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int m = min(m0 + i * 16 + r16, M - 1);
      const char* p = reinterpret_cast<const char*>(A + (size_t)m * HS_K + k0);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        a[i][s][0] = *reinterpret_cast<const uint4*>(p + s * 128 + (BLOCKED ? kq * 2 : kq * 4));
        a[i][s][1] = *reinterpret_cast<const uint4*>(p + s * 128 + (BLOCKED ? kq * 2 + 64 : kq * 4 + 16));
      }
    }
  };
  load(0);
  int buf = 0;
  for (int m0 = 0; m0 < M; m0 += 32, buf ^= 1) {
    f32x4 acc[2] = {f32x4{}, f32x4{}};
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        uint4 hi = a[i][s][0], lo = a[i][s][1];
        if constexpr (!BLOCKED) {
          const float4 u = __builtin_bit_cast(float4, a[i][s][0]), v = __builtin_bit_cast(float4, a[i][s][1]);
          split2(u.x, u.y, hi.x, lo.x);
          split2(u.z, u.w, hi.y, lo.y);
          split2(v.x, v.y, hi.z, lo.z);
          split2(v.z, v.w, hi.w, lo.w);
        }
        const bf16x8 ah = __builtin_bit_cast(bf16x8, hi), al = __builtin_bit_cast(bf16x8, lo);
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wh[s], ah, acc[i], 0, 0, 0);
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wl[s], ah, acc[i], 0, 0, 0);
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wh[s], al, acc[i], 0, 0, 0);
      }
    if (m0 + 32 < M) load(m0 + 32);
    // acc[i][r] = (row i * 16 + (lane & 15), column n0 + (lane >> 4) * 4 + r)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      *reinterpret_cast<f32x4*>(&red[buf][wave][(i * 16 + r16) * 16 + (lane >> 4) * 4]) = acc[i];
    __syncthreads();
    float v = red[buf][0][tid];
#pragma unroll
    for (int w = 1; w < 8; ++w) v += red[buf][w][tid];
    const int m = m0 + (tid >> 4);
    if (m < M) part[((size_t)slice * M + m) * HS_N + n0 + (tid & 15)] = v;
  }
}

// Row blockIdx.x: hid = relu(sum of the slices + b1) (stored where hid is given),
// then, with TAIL, logits = hid . W2^T + b2 (fp32 products with W2 = hi + lo, exact in
// fp32), softmax and the smallest class that attains the maximum.
template <bool TAIL>
__global__ __launch_bounds__(256) void cifar_head_few_kernel(const float* __restrict__ part,
                                                             const float* __restrict__ b1, float* __restrict__ hid,
                                                             const bf16_t* __restrict__ w2h,
                                                             const bf16_t* __restrict__ w2l,
                                                             const float* __restrict__ b2, float* __restrict__ probs,
                                                             int* __restrict__ pred, int M) {
  __shared__ __attribute__((aligned(16))) float hs[16 * 36];  // 32 k per slice of 36: 16-B reads of 4 slices, 4 banks apart
  __shared__ float zs[4][16];
  const int tid = threadIdx.x, m = blockIdx.x;
  const int cls = tid & 15, ks = tid >> 4;
  uint4 wh[4], wl[4];
  if constexpr (TAIL) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      wh[j] = *reinterpret_cast<const uint4*>(w2h + cls * HS_N + ks * 32 + j * 8);
      wl[j] = *reinterpret_cast<const uint4*>(w2l + cls * HS_N + ks * 32 + j * 8);
    }
  }
  float2 p[HS_S];
#pragma unroll
  for (int s = 0; s < HS_S; ++s)
    p[s] = *reinterpret_cast<const float2*>(part + ((size_t)s * M + m) * HS_N + 2 * tid);
  const float2 bb = *reinterpret_cast<const float2*>(b1 + 2 * tid);
  float2 v = p[0];
#pragma unroll
  for (int s = 1; s < HS_S; ++s) {
    v.x += p[s].x;
    v.y += p[s].y;
  }
  v.x = fmaxf(v.x + bb.x, 0.f);
  v.y = fmaxf(v.y + bb.y, 0.f);
  if (hid != nullptr) *reinterpret_cast<float2*>(hid + (size_t)m * HS_N + 2 * tid) = v;
  if constexpr (TAIL) {
    *reinterpret_cast<float2*>(hs + (tid >> 4) * 36 + (2 * tid & 31)) = v;
    __syncthreads();
    float z = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 u = *reinterpret_cast<const float4*>(hs + ks * 36 + j * 8);
      const float4 t = *reinterpret_cast<const float4*>(hs + ks * 36 + j * 8 + 4);
      const float hv[8] = {u.x, u.y, u.z, u.w, t.x, t.y, t.z, t.w};
      const uint32_t ph[4] = {wh[j].x, wh[j].y, wh[j].z, wh[j].w}, pl[4] = {wl[j].x, wl[j].y, wl[j].z, wl[j].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        z = fmaf(hv[2 * e], __uint_as_float(ph[e] << 16) + __uint_as_float(pl[e] << 16), z);
        z = fmaf(hv[2 * e + 1], __uint_as_float(ph[e] & 0xffff0000u) + __uint_as_float(pl[e] & 0xffff0000u), z);
      }
    }
    z = add16(z);
    z = add32(z);
    if ((tid & 63) < 16) zs[tid >> 6][cls] = z;
    __syncthreads();
    if (tid < 16) {
      z = tid < 10 ? zs[0][tid] + zs[1][tid] + zs[2][tid] + zs[3][tid] + b2[tid] : -INFINITY;
      float mx = z;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
      const float e = tid < 10 ? expf(z - mx) : 0.f;
      float sum = e;
      int cand = (z == mx) ? tid : 16;
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        sum += __shfl_xor(sum, o, 64);
        cand = min(cand, __shfl_xor(cand, o, 64));
      }
      if (tid < 10) probs[(size_t)m * 10 + tid] = e / sum;
      if (tid == 0) pred[m] = cand;
    }
  }
}

}  // namespace dnn

using namespace dnn;

// stage-0 boundary stores: 16-B (permlane32-paired, 1) or 8-B (0); A/B switch
static int g_s0_wide_store = 1;

extern "C" int dnn_cifar_s0_set_wide_store(int on) {
  g_s0_wide_store = on ? 1 : 0;
  return 0;
}

template <bool SPLIT_OUT>
static int launch_stage0_x3(const float* x, float* out, const void* w1h, const void* w1l, const float* b1,
                            const void* w2h, const void* w2l, const float* b2, float* keep, int B, int grid,
                            hipStream_t st) {
  if (g_s0_wide_store)
    hipLaunchKernelGGL((cifar_stage0_x3_kernel<true, SPLIT_OUT>), dim3(grid), dim3(512), 0, st, x, out,
                       (const bf16_t*)w1h, (const bf16_t*)w1l, b1, (const bf16_t*)w2h, (const bf16_t*)w2l, b2, keep, B);
  else
    hipLaunchKernelGGL((cifar_stage0_x3_kernel<false, SPLIT_OUT>), dim3(grid), dim3(512), 0, st, x, out,
                       (const bf16_t*)w1h, (const bf16_t*)w1l, b1, (const bf16_t*)w2h, (const bf16_t*)w2l, b2, keep, B);
  return (int)hipGetLastError();
}

// split_out = 1: the (B,4096) boundary in the blocked hi/lo encoding, else fp32.
// keep (null: none): (B,3,32,32), receives a copy of x; must not overlap x.
extern "C" int dnn_cifar_stage0_x3(const float* x, float* out, const void* w1h, const void* w1l, const float* b1,
                                   const void* w2h, const void* w2l, const float* b2, int B, int grid,
                                   hipStream_t st, int split_out, float* keep) {
  if (B <= 0) return 0;
  if (keep == x) keep = nullptr;
  if (grid <= 0) grid = 256;
  if (4L * B <= grid) {
    if (split_out)
      hipLaunchKernelGGL(cifar_stage0_x3_band_kernel<true>, dim3(4 * B), dim3(512), 0, st, x, out, (const bf16_t*)w1h,
                         (const bf16_t*)w1l, b1, (const bf16_t*)w2h, (const bf16_t*)w2l, b2, keep);
    else
      hipLaunchKernelGGL(cifar_stage0_x3_band_kernel<false>, dim3(4 * B), dim3(512), 0, st, x, out, (const bf16_t*)w1h,
                         (const bf16_t*)w1l, b1, (const bf16_t*)w2h, (const bf16_t*)w2l, b2, keep);
    return (int)hipGetLastError();
  }
  if (grid > B) grid = B;
  return split_out ? launch_stage0_x3<true>(x, out, w1h, w1l, b1, w2h, w2l, b2, keep, B, grid, st)
                   : launch_stage0_x3<false>(x, out, w1h, w1l, b1, w2h, w2l, b2, keep, B, grid, st);
}

// The ranges of K that dnn_cifar_fc1_x3 takes of those asked for: cifar_fc1_sum_kernel reads 16
// bytes at a time and counts quads of columns, whole workgroups of them, with 32 bits.
extern "C" int dnn_cifar_fc1_ranges(int M, int N, int splits, const float* C, const float* bias, const float* part) {
  const bool sum = (((uintptr_t)C | (uintptr_t)bias | (uintptr_t)part) & 15) == 0 && (long)M * (N / 4) <= INT_MAX - 255;
  return sum ? splits : 1;
}

extern "C" int dnn_cifar_fc1_x3(const float* A, int lda, const void* Wh, const void* Wl, int ldw, const float* bias,
                                float* C, int ldc, int M, int N, int K, hipStream_t st, int a_split, int splits,
                                float* part) {
  if (M <= 0) return 0;
  if (splits < 1 || splits > K / F1_K || (splits > 1 && part == nullptr)) return -1;
  splits = dnn_cifar_fc1_ranges(M, N, splits, C, bias, part);
  if (N % F1_T != 0 || K % F1_K != 0 || lda % 4 != 0 || ldw % 8 != 0 || ldc % 4 != 0) return -1;
  if ((((uintptr_t)A | (uintptr_t)Wh | (uintptr_t)Wl) & 15) != 0) return -1;  // 16-byte LDS-DMA
  if (lda >= 1 << 27 || ldw >= 1 << 27) return -1;  // 8 rows of A and 16 of W are addressed with 32 bits
  const int blocks = ((M + F1_T - 1) / F1_T) * (N / F1_T) * splits;
  if (a_split)
    hipLaunchKernelGGL(cifar_fc1_x3_kernel<true>, dim3(blocks), dim3(512), 0, st, A, lda, (const bf16_t*)Wh,
                       (const bf16_t*)Wl, ldw, bias, C, ldc, M, N, K, splits, part);
  else
    hipLaunchKernelGGL(cifar_fc1_x3_kernel<false>, dim3(blocks), dim3(512), 0, st, A, lda, (const bf16_t*)Wh,
                       (const bf16_t*)Wl, ldw, bias, C, ldc, M, N, K, splits, part);
  if (const hipError_t e = hipGetLastError()) return (int)e;
  if (splits > 1)
    hipLaunchKernelGGL(cifar_fc1_sum_kernel, dim3(((long)M * (N / 4) + 255) / 256), dim3(256), 0, st, part, bias, C, ldc, M, N,
                       splits);
  return (int)hipGetLastError();
}

extern "C" int dnn_cifar_split_blocked(const float* a, float* o, int M, int K, int dir, hipStream_t st) {
  if (M <= 0) return 0;
  if (K % 32 != 0 || a == o) return -1;
  const long total = (long)M * (K / 8);
  long blocks = (total + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(cifar_split_blocked_kernel, dim3((int)blocks), dim3(256), 0, st, a, o, M, K, dir);
  return (int)hipGetLastError();
}

extern "C" int dnn_cifar_split3(const float* a, int lda, void* o, int ldo, int M, int K, hipStream_t st, int blocked) {
  if (M <= 0) return 0;
  if (K % 8 != 0 || lda % 4 != 0 || ldo % 8 != 0 || ldo < 3 * K || (blocked && K % 32 != 0)) return -1;
  const long total = (long)M * (K / 8);
  long blocks = (total + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(cifar_split3_kernel, dim3((int)blocks), dim3(256), 0, st, a, lda, (bf16_t*)o, ldo, M, K, blocked);
  return (int)hipGetLastError();
}

extern "C" int dnn_cifar_head_tail_x3(const float* hid, const void* w2h, const void* w2l, const float* b2,
                                      float* probs, int* pred, int B, hipStream_t st) {
  if (B <= 0) return 0;
  int waves = (B + 15) / 16;
  int blocks = (waves + 3) / 4;
  if (blocks > 1024) blocks = 1024;
  hipLaunchKernelGGL(cifar_head_tail_x3_kernel, dim3(blocks), dim3(256), 0, st, hid, (const bf16_t*)w2h,
                     (const bf16_t*)w2l, b2, probs, pred, B);
  return (int)hipGetLastError();
}

// fc1 of a few rows into hid (M,512) and, where probs is given, fc2 + softmax + argmax
// (hid may then be null).  part: HS_S x M x 512 floats of scratch.
extern "C" int dnn_cifar_head_few(const float* A, int blocked, const void* Wh, const void* Wl, const float* b1,
                                  float* part, float* hid, const void* w2h, const void* w2l, const float* b2,
                                  float* probs, int* pred, int M, hipStream_t st) {
  if (M <= 0) return 0;
  if (probs == nullptr && hid == nullptr) return -1;
  if (blocked)
    hipLaunchKernelGGL(cifar_fc1_few_kernel<true>, dim3(HS_S * HS_N / 16), dim3(512), 0, st, A, (const bf16_t*)Wh,
                       (const bf16_t*)Wl, part, M);
  else
    hipLaunchKernelGGL(cifar_fc1_few_kernel<false>, dim3(HS_S * HS_N / 16), dim3(512), 0, st, A, (const bf16_t*)Wh,
                       (const bf16_t*)Wl, part, M);
  if (probs != nullptr)
    hipLaunchKernelGGL(cifar_head_few_kernel<true>, dim3(M), dim3(256), 0, st, part, b1, hid, (const bf16_t*)w2h,
                       (const bf16_t*)w2l, b2, probs, pred, M);
  else
    hipLaunchKernelGGL(cifar_head_few_kernel<false>, dim3(M), dim3(256), 0, st, part, b1, hid, (const bf16_t*)w2h,
                       (const bf16_t*)w2l, b2, probs, pred, M);
  return (int)hipGetLastError();
}
