// CIFAR stage 0 of many images: conv1 + bias + ReLU + pool -> conv2 + bias + ReLU + pool
// in fp32 (reference ModelPart0_2Node, cifar_model_parts.py:37-42), conv2 by Winograd's
// F(2 x 2, 3 x 3) (S. Winograd, "Arithmetic Complexity of Computations", 1980; A. Lavin, S. Gray,
// "Fast Algorithms for Convolutional Neural Networks", 2015): a 4 x 4 patch d of a channel becomes
// V = B^T d B, a 3 x 3 filter U = G g G^T, and the 2 x 2 outputs are A^T (sum over channels of
// U . V) A, 16 products where the window needs 36:
//
//   B^T = 1  0 -1  0    G = 1    0   0    A^T = 1  1  1  0
//         0  1  1  0        1/2 1/2 1/2         0  1 -1 -1
//         0 -1  1  0        1/2 -1/2 1/2
//         0  1  0 -1        0    0   1
//
// The direct form (cifar_x3.hip) is at the card's power limit: 81 % of its cycles on the matrix
// cores, at 1.75 of 2.4 GHz.  Here an image takes 672 units of its 1152 (a unit is one 32 x 32 x 16
// product; conv1 288, conv2 384 for 864) and twice the vector instructions.  65536 images, with their copy: 1796 ->
// 1475 us (9840 cycles an image at 1.85 GHz for 11350 at 1.75); 1024: 32.5 -> 28.3.
//
// What bounds it: a SIMD issues one vector instruction in 4.4 to 4.9 clocks, whichever wave it is from, and a
// phase (a quarter of an image) has 270 of them beside 1344 clocks of products; two waves leave gaps.  A wave for both
// roles, with conv2's output channels halved (each V formed twice): 13600 cycles.  The consumers' sums
// finished by themselves: 12100.  v_fma_mixlo / mixhi, which write half a register, take 8.4 clocks.
//
// Precision.  V, U and the sums behind them make an error of a product up to 1.7 times as large as
// the window does, so conv2's operands are two fp16 terms each, x = hi + lo to 2^-21 (two bf16 terms:
// 2^-17), three products; from 64 bits a stage is off by 3.0e-6 (direct: 4.8e-6, conv1's split in both).
// fp16 has few exponents, so both sides are scaled by powers of two, which
// round nothing: U so that the largest number of an output channel lies in [2^9, 2^10), the pooled map
// of an image so that what conv1 can reach at most (its weights' sum of magnitudes times the image's
// largest finite magnitude, plus the bias) lies below 2^13; V then stays below 2^15.  The scale of the
// map rides in conv1's bias addition, both inverses in conv2's.  An image whose range is too wide for one
// scale goes the direct way at the end (wide_range, direct_images), weights of such a spread take the direct form
// at all times (ops/cifar.py _winograd_range).  As every form that sums a patch before it multiplies: an output
// beside a part of its 4 x 4 patch that its own window does not see is off by 2^-21 of that part, so small outputs along
// an edge to values over 2^4 times theirs are further off than by the window, all of an image nearer.
//
// Work.  One workgroup a CU walks over images, 4 phases an image with one barrier each.  Waves 0-3
// ("producers") run conv1 of image it, two of its tile rows a phase, stage the next image, a quarter a phase, and
// finish 16 tiles of conv2.  Waves 4-7 ("consumers") run conv2 of image it - 1, 16 tiles (two rows of 8) a phase:
// wave I forms row I of V for all channels from the two map rows it needs, in the registers of the A operand
// (its neighbours' columns by DPP; a row of 16 lanes holds tiles (tx, ty & 1) at 2 tx + (ty & 1), so that
// a shift by two lanes shifts in zeros where the map ends), multiplies by its 4 of the 16 matrices of
// U (128 registers for 64 channels), and forms the two column sums.  What is left, sums over the 4 waves, goes
// through LDS: producer o finishes output channels 16 o to 16 o + 15 in the next phase.
//
// LDS (158,800 B): the split input (planes [33][40][4] bf16; a quarter of the next image takes the place of the
// rows that all waves have fetched), the pooled map twice (fp32 [17][16][32], halo rows shared, no halo
// columns), the sums between the waves twice, scales.  A pixel's 16-byte chunks and its place in a pair of pixels
// are swizzled (map_off) so that the reads of a patch's row are free of conflicts.
#include "cifar_conv.h"

namespace dnn {
namespace wino {

using namespace x3;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int WPL = 33 * XW * 8;              // one input plane; its last halo row is the next one's first
constexpr int MAP_OFF = 84 * 256;             // 2 WPL + a row of 320 B, to 256 B
constexpr int MAP_ROW = 16 * 128;
constexpr int MAP = 17 * MAP_ROW;
constexpr int EX_OFF = MAP_OFF + 2 * MAP + MAP_ROW;
constexpr int EX = 4 * 4 * 2 * 1024;          // [output channel group][consumer][column sum][lane] of 16 B
constexpr int SC_OFF = EX_OFF + 2 * EX;
constexpr int WIDE_OFF = SC_OFF + 4 * 16;     // behind the largest magnitudes of 4 images, by producer wave
constexpr int LDS_BYTES = WIDE_OFF + 16;
static_assert(2 * WPL + XW * 8 <= MAP_OFF && LDS_BYTES <= 160 * 1024, "");

__device__ __forceinline__ int map_base(int k) { return MAP_OFF + (k & 1) * MAP; }

// 16-byte chunk c (4 channels) of padded row y and column pair tx (columns 2 tx + cc) of a map
__device__ __forceinline__ int map_off(int y, int tx, int cc, int c) {
  const int f = (tx & 1) | ((tx >> 1) & 1) * 6;
  return y * MAP_ROW + tx * 256 + ((cc ^ ((y >> 1) & 1)) << 7) + ((c ^ f ^ ((y & 1) << 2)) << 4);
}

// The power of two that brings all of an image's pooled map below 2^13, and its inverse: m is the
// image's largest finite magnitude, b >= l1 m + bmax bounds the map.
__device__ __forceinline__ void map_scale(float m, float l1, float bmax, float& s, float& inv) {
  const uint32_t e = __float_as_uint(fmaf(m, l1, bmax)) >> 23;  // of b < 2^(e - 126)
  const uint32_t f = e < 39u ? 227u : 266u - e;                 // 2^-116 (b overflowed) .. 2^100
  s = __uint_as_float(f << 23);
  inv = __uint_as_float((254u - f) << 23);
}

// Is the range of an image of largest magnitude m too wide for one scale?  Two fp16 terms are off by 2^-21 of a magnitude
// of the map from 2^-3 on, and by up to 2^-24 below: 2^-37 of the bound.  Up to `most` the bound is at most 2^16 times
// what the biases bring to every output channel (ops/cifar.py _winograd_range), and that is 2^-21 beside
// them, less than the split of conv1's operands loses.
__device__ __forceinline__ bool wide_range(float m, float most) { return m > most; }

__device__ __forceinline__ float slots_max(const char* smem, int k) {
  const float4 v = *reinterpret_cast<const float4*>(smem + SC_OFF + (k & 3) * 16);
  return fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w));
}

// bias + ReLU + 2x2 max-pool of conv1 tile t in registers (max(a) + b == max(a + b) exactly), times the
// image's scale; a lane writes its channel of 4 pooled pixels (with a transpose over quads of lanes and one
// 16-byte write a tile 20 vector instructions more).  at: the lane's place in an even and in an odd padded
// row, pair of columns h of tile column 0 or 1 (the swizzle has a period of 4 pairs).
__device__ __forceinline__ void map_store(char* map, int tyc, const uint32_t (&at)[2], const f32x16& acc, float s, float bs) {
#pragma unroll
  for (int qy = 0; qy < 2; ++qy) {
    const int y = 2 * tyc + qy + 1, swap = (y >> 1) & 1;
    float v[2];
#pragma unroll
    for (int qx = 0; qx < 2; ++qx) {
      const int g0 = (2 * qy) * 4 + 2 * qx;
      v[qx] = fmaxf(fmaf(fmax_nan(fmax_nan(acc[g0], acc[g0 + 1]), fmax_nan(acc[g0 + 4], acc[g0 + 5])), s, bs), 0.f);
    }
    float* p = reinterpret_cast<float*>(map + at[y & 1] + y * MAP_ROW);
    p[0] = v[swap];
    p[32] = v[1 - swap];
  }
}

template <int CTRL>
__device__ __forceinline__ float shifted(float v) {  // lanes the shift leaves empty: 0
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float left(float v) { return shifted<0x112>(v); }   // row_shr:2
__device__ __forceinline__ float right(float v) { return shifted<0x102>(v); }  // row_shl:2

// 8 floats -> fp16 hi and lo (the difference to hi is exact in fp32).  A pair takes 4 vector instructions of
// 4.85 clocks; with v_fma_mixlo / mixhi, which write half a register, 3 but 22 clocks; what the compiler makes, 6.
__device__ __forceinline__ void split_f16(const float (&v)[8], f16x8& hi, f16x8& lo) {
  uint32_t h[4], l[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float d0, d1;
    h[e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(v[2 * e], v[2 * e + 1]));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(d0) : "v"(h[e]), "v"(v[2 * e]));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d1) : "v"(h[e]), "v"(v[2 * e + 1]));
    l[e] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(d0, d1));
  }
  hi = __builtin_bit_cast(f16x8, make_uint4(h[0], h[1], h[2], h[3]));
  lo = __builtin_bit_cast(f16x8, make_uint4(l[0], l[1], l[2], l[3]));
}

// acc[oc group] (+)= V U, hi.hi, hi.lo, lo.hi, the groups' chains interleaved
__device__ __forceinline__ void products(const f16x8& vh, const f16x8& vl, const f16x8 (&uh)[4], const f16x8 (&ul)[4],
                                         const f32x4 (&c)[4], f32x4 (&d)[4]) {
#pragma unroll
  for (int o = 0; o < 4; ++o) d[o] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, uh[o], c[o], 0, 0, 0);
#pragma unroll
  for (int o = 0; o < 4; ++o) d[o] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, ul[o], d[o], 0, 0, 0);
#pragma unroll
  for (int o = 0; o < 4; ++o) d[o] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl, uh[o], d[o], 0, 0, 0);
}

// Consumer wave I
template <int I>
__device__ __forceinline__ void consume(char* smem, const _Float16* __restrict__ u2h, const _Float16* __restrict__ u2l, int n,
                                        int lane) {
  const int r16 = lane & 15, g = lane >> 4;
  f16x8 uh[4][4], ul[4][4];  // [column j of V][output channel group]
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      const int at = (((I * 4 + j) * 64) + o * 16 + r16) * 32 + g * 8;
      uh[j][o] = *reinterpret_cast<const f16x8*>(u2h + at);
      ul[j][o] = *reinterpret_cast<const f16x8*>(u2l + at);
    }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int o = 0; o < 4; ++o) asm volatile("" ::"v"(uh[j][o]), "v"(ul[j][o]));

  // rows of the patch: V's row I is row RA of d, plus or minus row RB
  constexpr int RA = I == 0 ? 0 : I == 2 ? 2 : 1, RB = I == 0 || I == 1 ? 2 : I == 2 ? 1 : 3;
  const int ty = r16 & 1, tx = r16 >> 1;
  const int fa = map_off(2 * ty + RA, tx, 0, 2 * g), fb = map_off(2 * ty + RB, tx, 0, 2 * g);

  f32x4 da[2][2], db[2][2];  // [column][4 channels]
  auto fetch = [&](int G) {
    const char* ma = smem + map_base(G >> 2) + (G & 3) * 4 * MAP_ROW;
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        da[cc][e] = *reinterpret_cast<const f32x4*>(ma + (fa ^ (cc << 7 | e << 4)));
        db[cc][e] = *reinterpret_cast<const f32x4*>(ma + (fb ^ (cc << 7 | e << 4)));
      }
  };
  __syncthreads();  // image 0 is staged
  for (int p = 0; p < 4; ++p) __syncthreads();  // conv1 of image 0
  fetch(0);
#pragma unroll 1
  for (int G = 0; G < 4 * n; ++G) {
    float t0[8], t1[8], v[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float a0 = da[0][c >> 2][c & 3], b0 = db[0][c >> 2][c & 3];
      const float a1 = da[1][c >> 2][c & 3], b1 = db[1][c >> 2][c & 3];
      t0[c] = I == 1 ? a0 + b0 : a0 - b0;
      t1[c] = I == 1 ? a1 + b1 : a1 - b1;
    }
    const f32x4 zero[4] = {f32x4{}, f32x4{}, f32x4{}, f32x4{}};
    f16x8 vh, vl;
    f32x4 m1[4], s0[4], m2[4];
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = t0[c] + t1[c];
    split_f16(v, vh, vl);
    products(vh, vl, uh[1], ul[1], zero, m1);
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = t1[c] - t0[c];
    split_f16(v, vh, vl);
    products(vh, vl, uh[2], ul[2], zero, m2);
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = left(t1[c]) - t1[c];
    split_f16(v, vh, vl);
    products(vh, vl, uh[0], ul[0], m1, s0);
#pragma unroll
    for (int o = 0; o < 4; ++o) s0[o] += m2[o];  // m0 + m1 + m2
    char* ex = smem + EX_OFF + (G & 1) * EX + I * 2048 + lane * 16;
#pragma unroll
    for (int o = 0; o < 4; ++o) *reinterpret_cast<f32x4*>(ex + o * 8192) = s0[o];
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = t0[c] - right(t0[c]);
    split_f16(v, vh, vl);
    products(vh, vl, uh[3], ul[3], m2, m2);
    fetch(G + 1);  // its rows are in the map since the phase before last; behind the last tiles: unused
#pragma unroll
    for (int o = 0; o < 4; ++o) m1[o] -= m2[o];  // m1 - (m2 + m3)
#pragma unroll
    for (int o = 0; o < 4; ++o) *reinterpret_cast<f32x4*>(ex + o * 8192 + 1024) = m1[o];
    __syncthreads();
  }
}

// The sums of group G over the consumers' rows, bias, ReLU and pool for output channel oc (of group
// o) -> row ob of the boundary, 8-B stores of two pooled columns
template <bool SPLIT_OUT>
__device__ __forceinline__ void finish(const char* smem, int G, int o, int oc, float by, float bias, float* ob, int lane) {
  const char* ex = smem + EX_OFF + (G & 1) * EX + o * 8192 + lane * 16;
  f32x4 w[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int s = 0; s < 2; ++s) w[i][s] = *reinterpret_cast<const f32x4*>(ex + i * 2048 + s * 1024);
  float y[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float v[2][2];  // [output row][column]
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      v[0][s] = w[0][s][r] + w[1][s][r] + w[2][s][r];
      v[1][s] = w[1][s][r] - w[2][s][r] - w[3][s][r];
    }
    y[r] = fmaxf(fmaf(fmax_nan(fmax_nan(v[0][0], v[0][1]), fmax_nan(v[1][0], v[1][1])), by, bias), 0.f);
  }
  // tile 4 g + r: pooled column 2 g + (r >> 1), row 2 (G & 3) + (r & 1)
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int PY = 2 * (G & 3) + q, PX = 2 * (lane >> 4);
    if constexpr (SPLIT_OUT) {
      uint32_t hi, lo;
      split2(y[q], y[q + 2], hi, lo);
      char* bp = reinterpret_cast<char*>(ob) + (oc * 2 + (PY >> 2)) * 128 + ((PY & 3) * 8 + PX) * 2;
      *reinterpret_cast<uint32_t*>(bp) = hi;
      *reinterpret_cast<uint32_t*>(bp + 64) = lo;
    } else {
      *reinterpret_cast<float2*>(ob + oc * 64 + PY * 8 + PX) = make_float2(y[q], y[q + 2]);
    }
  }
}

// What a launch gets.  sc: conv1's largest sum of magnitudes, its largest bias magnitude, the largest magnitude
// of an image in range, 64 inverse scales of U.  u2h, u2l: [16][64][32] fp16.  keep: as in cifar_stage0_x3_kernel.
struct Args {
  const float* x;
  float* out;
  const bf16_t *w1h, *w1l;
  const float* b1;
  const bf16_t *w2h, *w2l;
  const _Float16 *u2h, *u2l;
  const float *b2, *sc;
  float* keep;
  int B;
};

// The images of this workgroup whose range is too wide, once more, with the direct conv2 (tiles, products and
// order of cifar_stage0_x3_kernel, one image after the other).  us of a launch without such an image, with one, with
// all (the direct form takes them as any other): 1024 images 34.6, 52, 102 (37.6), 65536 1450, 1610, 5170 (1710).  Weights of
// the reference's own initialisation reach it beyond magnitudes of 1200 to 2700; no raw pixel does (WINO_IMAGES).
template <bool SPLIT_OUT>
__device__ __forceinline__ void direct_images(char* smem, const Args& a, int n) {
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, r32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), rw = wave & 3;
  constexpr int A1 = 2 * XPL;  // xin hi | lo, pooled map hi | lo
  for (int k = 0; k < n; ++k) {
    const size_t img = blockIdx.x + (size_t)k * gridDim.x;
    float px[2][3], m = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int c = 0; c < 3; ++c) px[i][c] = a.x[img * 3072 + c * 1024 + tid + 512 * i];
      const float t = fmaxf(fmaxf(fabsf(px[i][0]), fabsf(px[i][1])), fabsf(px[i][2]));
      m = fmaxf(m, __float_as_uint(t) < 0x7f800000u ? t : 0.f);
    }
    m = wave_max(m);
    __syncthreads();  // the image before is done
    if (lane == 0) reinterpret_cast<float*>(smem + SC_OFF)[wave] = m;
    for (int i = tid; i < (A1 + 2 * A1PL) / 16; i += 512) reinterpret_cast<uint4*>(smem)[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    m = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) m = fmaxf(m, reinterpret_cast<const float*>(smem + SC_OFF)[i]);
    if (!wide_range(m, a.sc[2])) continue;  // the same for all
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int p = tid + 512 * i, o = (((p >> 5) + 1) * XW + (p & 31) + 1) * 8;
      uint2 vh, vl;
      split2(px[i][0], px[i][1], vh.x, vl.x);
      split2(px[i][2], 0.f, vh.y, vl.y);
      *reinterpret_cast<uint2*>(smem + o) = vh;
      *reinterpret_cast<uint2*>(smem + XPL + o) = vl;
    }
    __syncthreads();
    if (wave < 4) {
      bf16x8 w1hf[3], w1lf[3];
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        w1hf[s] = *reinterpret_cast<const bf16x8*>(a.w1h + r32 * 48 + s * 16 + h * 8);
        w1lf[s] = *reinterpret_cast<const bf16x8*>(a.w1l + r32 * 48 + s * 16 + h * 8);
      }
#pragma unroll 1
      for (int t = rw; t < 32; t += 8) conv1_pair(smem, smem + A1, t, t + 4, w1hf, w1lf, a.b1[r32], lane);
    }
    __syncthreads();
    if (wave >= 4) {
      const int oc = (rw & 1) * 32 + r32;
#pragma unroll 1
      for (int ty = (rw >> 1) * 2; ty < (rw >> 1) * 2 + 2; ++ty) {
#pragma unroll 1
        for (int i = 0; i < 2; ++i) {
          f32x16 acc = {};
#pragma unroll 2
          for (int s = 0; s < 18; ++s) {
            const int ky = (s >> 1) / 3, kx = (s >> 1) % 3, yr = (r32 >> 3) + ky;
            const char* p = smem + A1 + ((4 * ty + yr) * 18 + 8 * i + (r32 & 7) + kx) * 64 + (((2 * (s & 1) + h) ^ (yr & 3)) << 4);
            const bf16x8 ah = *reinterpret_cast<const bf16x8*>(p), al = *reinterpret_cast<const bf16x8*>(p + A1PL);
            const bf16x8 wh = *reinterpret_cast<const bf16x8*>(a.w2h + oc * 288 + s * 16 + h * 8);
            const bf16x8 wl = *reinterpret_cast<const bf16x8*>(a.w2l + oc * 288 + s * 16 + h * 8);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, wh, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, wl, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, wh, acc, 0, 0, 0);
          }
          conv2_store<SPLIT_OUT>(a.out + img * 4096, oc, ty, i, acc, a.b2[oc], h);
        }
      }
    }
  }
}

}  // namespace wino

using namespace wino;

template <bool SPLIT_OUT>
__global__ __launch_bounds__(512, 1) void cifar_stage0_wino_kernel(const Args a) {
  const float* __restrict__ x = a.x;
  float *__restrict__ out = a.out, *__restrict__ keep = a.keep;
  const float* __restrict__ sc = a.sc;
  __shared__ __attribute__((aligned(256))) char smem[wino::LDS_BYTES];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rw = wave & 3, rt = tid & 255, r32 = lane & 31, h = lane >> 5;
  const int n = (a.B - 1 - (int)blockIdx.x) / (int)gridDim.x + 1;  // host: grid <= B

  for (int i = tid; i < wino::LDS_BYTES / 16; i += 512) reinterpret_cast<uint4*>(smem)[i] = make_uint4(0, 0, 0, 0);
  __syncthreads();  // halos are zero before the interiors are written

  if (wave < 4) {
    bf16x8 w1hf[3], w1lf[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      w1hf[s] = *reinterpret_cast<const bf16x8*>(a.w1h + r32 * 48 + s * 16 + h * 8);
      w1lf[s] = *reinterpret_cast<const bf16x8*>(a.w1l + r32 * 48 + s * 16 + h * 8);
    }
    const int oc = rw * 16 + (lane & 15);
    const float bias = a.b1[r32], l1 = sc[0], bmax = sc[1], most = sc[2], bias2 = a.b2[oc], inv_w = sc[3 + oc];
    resident_fence(w1hf);
    resident_fence(w1lf);
    // all of them arrived: a wait left in the loop would be for the stores of the phase before as well
    asm volatile("" ::"v"(bias), "v"(l1), "v"(bmax), "v"(most), "v"(bias2), "v"(inv_w));

    float pf[4][3], big = 0.f;
    auto image = [&](int k) { return blockIdx.x + (size_t)min(k, n - 1) * gridDim.x; };
    auto load = [&](int k, int i) {  // behind the last image: that one again, not used
      const float* xb = x + image(k) * 3072;
#pragma unroll
      for (int c = 0; c < 3; ++c) pf[i][c] = xb[c * 1024 + rt + 256 * i];
    };
    auto stage = [&](int k, int i) {  // 8 rows: prefetch registers -> padded HWC4 hi / lo planes
      const int p = rt + 256 * i, o = (((p >> 5) + 1) * XW + (p & 31) + 1) * 8;
      uint2 vh, vl;
      split2(pf[i][0], pf[i][1], vh.x, vl.x);
      split2(pf[i][2], 0.f, vh.y, vl.y);
      *reinterpret_cast<uint2*>(smem + o) = vh;
      *reinterpret_cast<uint2*>(smem + WPL + o) = vl;
      // a pixel with an infinity or a NaN reaches no number: it bounds nothing
      float m = fmaxf(fmaxf(fabsf(pf[i][0]), fabsf(pf[i][1])), fabsf(pf[i][2]));
      m = __float_as_uint(m) < 0x7f800000u ? m : 0.f;
      big = i == 0 ? m : fmaxf(big, m);
      if (i == 3) {
        const float m64 = wave_max(big);
        if (lane == 0) *reinterpret_cast<float*>(smem + SC_OFF + (k & 3) * 16 + rw * 4) = m64;
      }
    };
    auto keep_rows = [&](int k, int i) {
      float* kb = keep + image(k) * 3072;
#pragma unroll
      for (int c = 0; c < 3; ++c) kb[c * 1024 + rt + 256 * i] = pf[i][c];
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) load(0, i);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      stage(0, i);
      if (keep != nullptr) keep_rows(0, i);
      load(1, i);
    }
    __syncthreads();
    // Phase p of image it: products of a pair of tiles, whose operands the phase before fetched; beside
    // them the pair before goes to the map, a quarter of the next image takes the place of the rows that
    // are fetched for good, and 16 tiles are finished.  The phases before tile 0 finish nothing: what they
    // store is stored over by the same lanes.
    bf16x8 fah[3], fal[3], fbh[3], fbl[3];
    f32x16 acca = {}, accb = {};
    float s = 0.f, bs = 0.f, inv;
    size_t step = (size_t)gridDim.x * 4096;
    asm("" : "+s"(step));  // not loaded from the launch's arguments again every phase
    float* ob = out + (size_t)blockIdx.x * 4096;
    float by = 0.f;  // inverse scale of the image that is being finished
    auto finish_scale = [&](int k) {
      float t;
      map_scale(slots_max(smem, k), l1, bmax, t, by);
      by *= inv_w;
    };
    const int xp = 2 * rw + h;  // pair of columns; tile column rw
    uint32_t at[2];
#pragma unroll
    for (int y = 0; y < 2; ++y)  // padded rows 0 and 1 hold their column 0 in place: not swapped
      at[y] = (uint32_t)(map_off(y, xp, 0, r32 >> 2) - y * MAP_ROW) + (r32 & 3) * 4;
    auto pair = [&](char* map, int p) {
      map_store(map, 2 * p, at, acca, s, bs);
      map_store(map, 2 * p + 1, at, accb, s, bs);
    };
    conv1_fetch<WPL>(smem, rw, fah, fal, lane);
    conv1_fetch<WPL>(smem, rw + 4, fbh, fbl, lane);
#pragma unroll 1
    for (int it = 0; it < n; ++it) {
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        f32x16 na = {}, nb = {};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          na = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fah[k], w1hf[k], na, 0, 0, 0);
          nb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fbh[k], w1hf[k], nb, 0, 0, 0);
          na = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fah[k], w1lf[k], na, 0, 0, 0);
          nb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fbh[k], w1lf[k], nb, 0, 0, 0);
          na = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fal[k], w1hf[k], na, 0, 0, 0);
          nb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fbl[k], w1hf[k], nb, 0, 0, 0);
        }
        pair(smem + map_base(p == 0 ? it + 1 : it), (p + 3) & 3);  // it + 1 is as odd as it - 1
        if (p == 1) ob += it > 1 ? step : 0;
        if (p == 1) finish_scale(it - 1);
        finish<SPLIT_OUT>(smem, 4 * it + p - 5, rw, oc, by, bias2, ob, lane);
        // image it in phase 0, its last quarter; then image it + 1
        const int k = p == 0 ? it : it + 1, i = (p + 3) & 3;
        stage(k, i);
        if (keep != nullptr && k < n) keep_rows(k, i);
        load(k + 1, i);
        conv1_fetch<WPL>(smem, rw + 8 * ((p + 1) & 3), fah, fal, lane);
        conv1_fetch<WPL>(smem, rw + 8 * ((p + 1) & 3) + 4, fbh, fbl, lane);
        acca = na;
        accb = nb;
        __syncthreads();
        if (p == 0) {
          const float m = slots_max(smem, it);
          map_scale(m, l1, bmax, s, inv);
          bs = bias * s;
          if (wide_range(m, most)) *reinterpret_cast<int*>(smem + WIDE_OFF) = 1;
        }
      }
    }
    pair(smem + map_base(n - 1), 3);
#pragma unroll 1
    for (int G = 4 * n - 5; G < 4 * n; ++G) {
      finish_scale(G >> 2);
      finish<SPLIT_OUT>(smem, G, rw, oc, by, bias2, out + image(max(G, 0) >> 2) * 4096, lane);
      if (G < 4 * n - 1) __syncthreads();
    }
  } else {
    switch (rw) {
      case 0: consume<0>(smem, a.u2h, a.u2l, n, lane); break;
      case 1: consume<1>(smem, a.u2h, a.u2l, n, lane); break;
      case 2: consume<2>(smem, a.u2h, a.u2l, n, lane); break;
      default: consume<3>(smem, a.u2h, a.u2l, n, lane);
    }
  }
  __syncthreads();
  if (*reinterpret_cast<const int*>(smem + WIDE_OFF)) direct_images<SPLIT_OUT>(smem, a, n);
}

}  // namespace dnn

using namespace dnn;

extern "C" int dnn_cifar_stage0_wino(const float* x, float* out, const void* w1h, const void* w1l, const float* b1,
                                     const void* w2h, const void* w2l, const void* u2h, const void* u2l, const float* b2,
                                     const float* sc, int B, int grid, hipStream_t st, int split_out, float* keep) {
  if (B <= 0) return 0;
  if (keep == x) keep = nullptr;
  if (grid <= 0) grid = 256;
  if (grid > B) grid = B;
  const Args a{x, out, (const bf16_t*)w1h, (const bf16_t*)w1l, b1, (const bf16_t*)w2h, (const bf16_t*)w2l,
               (const _Float16*)u2h, (const _Float16*)u2l, b2, sc, keep, B};
  if (split_out)
    hipLaunchKernelGGL(cifar_stage0_wino_kernel<true>, dim3(grid), dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL(cifar_stage0_wino_kernel<false>, dim3(grid), dim3(512), 0, st, a);
  return (int)hipGetLastError();
}
