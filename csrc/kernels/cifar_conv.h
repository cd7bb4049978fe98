// What the two forms of CIFAR stage 0 share (cifar_x3.hip: direct convolutions,
// cifar_wino.hip: conv2 by Winograd's F(2 x 2, 3 x 3)): the split of fp32 into two bf16
// terms, conv1's products on the staged image, and the pieces of the direct conv2.
#pragma once
#include "common.h"

namespace dnn {
namespace x3 {

// 2 floats -> packed bf16 hi pair and lo pair (element a in the low half).  Converted as
// pairs: 6 vector instructions, 10 where the compiler converts them one by one.
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf2));
  const float ah = __uint_as_float(hi << 16), bh = __uint_as_float(hi & 0xffff0000u);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a - ah, b - bh}, bf2));
}

__device__ __forceinline__ int dpp_xor1(int v) { return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false); }
__device__ __forceinline__ int dpp_xor2(int v) { return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false); }

constexpr int XW = 40;                        // xin row pitch (pixels); HWC4 bf16 = 8 B/pixel

// Where a lane's operands of conv1 tile t (4 x 8 pixels) begin in a staged plane, and one of them
__device__ __forceinline__ int conv1_lane(int t, int lane) {
  const int h = lane >> 5, r32 = lane & 31;
  return ((r32 >> 3) * XW + (r32 & 7) + 2 * h) * 8 + ((4 * (t >> 2)) * XW + 8 * (t & 3)) * 8;
}
__device__ __forceinline__ bf16x8 conv1_frag(const char* p) {
  const uint2 a = *reinterpret_cast<const uint2*>(p);
  const uint2 b = *reinterpret_cast<const uint2*>(p + 8);
  return __builtin_bit_cast(bf16x8, make_uint4(a.x, a.y, b.x, b.y));
}

// Operands of conv1 tile t of the staged image xh, whose lo plane is LO bytes behind
template <int LO>
__device__ __forceinline__ void conv1_fetch(const char* xh, int t, bf16x8 (&hi)[3], bf16x8 (&lo)[3], int lane) {
  const int o = conv1_lane(t, lane);
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    hi[s] = conv1_frag(xh + o + s * XW * 8);
    lo[s] = conv1_frag(xh + LO + o + s * XW * 8);
  }
}

constexpr int XPL = 34 * XW * 8;              // 10880: one input plane
constexpr int A1PL = 18 * 18 * 64;            // 20736: one pooled-conv1 plane [18][18][32] bf16
constexpr int A1_OFF = 4 * XPL;               // 43520
constexpr int LDS_BYTES = A1_OFF + 4 * A1PL;  // 126464

__device__ __forceinline__ int xin_off(int k, int lo) { return ((k & 1) * 2 + lo) * XPL; }
__device__ __forceinline__ int a1_off(int k, int lo) { return A1_OFF + ((k & 1) * 2 + lo) * A1PL; }

// conv2 A-fragment immediate offset for k-step S (tap = S>>1, kx = tap % 3),
// tile column I (tx2) and plane (LO): the lane/ky/parity part lives in the base.
template <int S, int I, int LO>
__device__ __forceinline__ constexpr int c2_imm() {
  return (8 * I + (S >> 1) % 3) * 64 + LO * A1PL;
}

// 4 reads of k-step S: [hi t0, hi t1, lo t0, lo t1]
template <int S>
__device__ __forceinline__ void c2_issue(const uint32_t (&b)[3][2], bf16x8 (&a)[4]) {
  constexpr int ky = (S >> 1) / 3, par = S & 1;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(a[0]) : "v"(b[ky][par]), "i"(c2_imm<S, 0, 0>()));
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(a[1]) : "v"(b[ky][par]), "i"(c2_imm<S, 1, 0>()));
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(a[2]) : "v"(b[ky][par]), "i"(c2_imm<S, 0, 1>()));
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(a[3]) : "v"(b[ky][par]), "i"(c2_imm<S, 1, 1>()));
}

// k-step S: issue step S+1's reads, wait for step S's (counted lgkmcnt; the
// caller has no other LDS op in flight), then 6 MFMAs alternating the two
// tiles' accumulators.  sched_barriers keep hipcc from hoisting MFMAs above
// the wait (cdna_hip_programming.md §5.7).
template <int S>
__device__ __forceinline__ void c2_step(const uint32_t (&b)[3][2], const bf16x8 (&wh)[18], const bf16x8 (&wl)[18],
                                        f32x16 (&acc)[2], bf16x8 (&cur)[4], bf16x8 (&nxt)[4]) {
  if constexpr (S + 1 < 18) {
    c2_issue<S + 1>(b, nxt);
    asm volatile("s_waitcnt lgkmcnt(4)" ::: "memory");
  } else {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  __builtin_amdgcn_sched_barrier(0);
  acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[0], wh[S], acc[0], 0, 0, 0);
  acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[1], wh[S], acc[1], 0, 0, 0);
  acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[0], wl[S], acc[0], 0, 0, 0);
  acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[1], wl[S], acc[1], 0, 0, 0);
  acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[2], wh[S], acc[0], 0, 0, 0);
  acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(cur[3], wh[S], acc[1], 0, 0, 0);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (S + 1 < 18) c2_step<S + 1>(b, wh, wl, acc, nxt, cur);
}

// hi / lo planes of the pooled conv1 map: bias + ReLU + 2x2 max-pool of tile t in
// registers (max(a)+b == max(a+b) exactly), quad-DPP gather of 4 channels of one
// pooled pixel per lane, hi/lo split, one 8-B store per plane
__device__ __forceinline__ void conv1_store(char* a1, int t, const f32x16& acc, float bias, int lane) {
  const int h = lane >> 5, r32 = lane & 31;
  const int q = ((r32 & 1) ? 2 : 0) + ((r32 & 2) ? 1 : 0);
  const int cb = r32 & ~3;
  const int ty = t >> 2, tx = t & 3;
  float v[4];
#pragma unroll
  for (int qy = 0; qy < 2; ++qy)
#pragma unroll
    for (int qx = 0; qx < 2; ++qx) {
      const int g0 = (2 * qy) * 4 + 2 * qx;
      v[qy * 2 + qx] = fmaxf(fmax_nan(fmax_nan(acc[g0], acc[g0 + 1]), fmax_nan(acc[g0 + 4], acc[g0 + 5])) + bias, 0.f);
    }
  const bool odd = r32 & 1;
  const int s0 = __float_as_int(odd ? v[0] : v[2]), s1 = __float_as_int(odd ? v[1] : v[3]);
  const float r0 = __int_as_float(dpp_xor1(s0)), r1 = __int_as_float(dpp_xor1(s1));
  uint32_t u0h, u0l, u1h, u1l;
  if (!odd) {
    split2(v[0], r0, u0h, u0l);
    split2(v[1], r1, u1h, u1l);
  } else {
    split2(r0, v[2], u0h, u0l);
    split2(r1, v[3], u1h, u1l);
  }
  const bool hi2 = r32 & 2;
  const uint32_t rch = (uint32_t)dpp_xor2((int)(hi2 ? u0h : u1h));
  const uint32_t rcl = (uint32_t)dpp_xor2((int)(hi2 ? u0l : u1l));
  const uint32_t mh = hi2 ? u1h : u0h, ml = hi2 ? u1l : u0l;
  uint2 wh, wl;
  wh.x = hi2 ? rch : mh;
  wh.y = hi2 ? mh : rch;
  wl.x = hi2 ? rcl : ml;
  wl.y = hi2 ? ml : rcl;
  const int Y = 2 * ty + (q >> 1) + 1, X = 4 * tx + 2 * h + (q & 1) + 1;
  const int o = (Y * 18 + X) * 64 + ((((cb >> 3) ^ (Y & 3))) << 4) + (cb & 7) * 2;
  *reinterpret_cast<uint2*>(a1 + o) = wh;
  *reinterpret_cast<uint2*>(a1 + A1PL + o) = wl;
}

// two conv1 tiles of the staged image xh at once: all 24 A-fragment reads up front, those of the two tiles in
// turn (tile by tile 512 images took 20.9 us for 20.5), two accumulation chains interleaved
__device__ __forceinline__ void conv1_pair(const char* xh, char* a1, int ta, int tb, const bf16x8 (&w1hf)[3],
                                           const bf16x8 (&w1lf)[3], float bias, int lane) {
  const int oa = conv1_lane(ta, lane), ob = conv1_lane(tb, lane);
  bf16x8 fah[3], fal[3], fbh[3], fbl[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    fah[s] = conv1_frag(xh + oa + s * XW * 8);
    fbh[s] = conv1_frag(xh + ob + s * XW * 8);
    fal[s] = conv1_frag(xh + XPL + oa + s * XW * 8);
    fbl[s] = conv1_frag(xh + XPL + ob + s * XW * 8);
  }
  f32x16 acca = {}, accb = {};
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    acca = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fah[s], w1hf[s], acca, 0, 0, 0);
    accb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fbh[s], w1hf[s], accb, 0, 0, 0);
    acca = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fah[s], w1lf[s], acca, 0, 0, 0);
    accb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fbh[s], w1lf[s], accb, 0, 0, 0);
    acca = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fal[s], w1hf[s], acca, 0, 0, 0);
    accb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fbl[s], w1hf[s], accb, 0, 0, 0);
  }
  conv1_store(a1, ta, acca, bias, lane);
  conv1_store(a1, tb, accb, bias, lane);
}

// bias + ReLU + 2x2 max-pool of conv2 tile (ty2, i) and channel oc2 -> row `out` of
// the (B,4096) boundary: 8-B stores of two pooled columns
template <bool SPLIT_OUT>
__device__ __forceinline__ void conv2_store(float* out, int oc2, int ty2, int i, const f32x16& acc, float bias, int h) {
#pragma unroll
  for (int qy = 0; qy < 2; ++qy) {
    float2 pv;
    const int g0 = (2 * qy) * 4;
    pv.x = fmaxf(fmax_nan(fmax_nan(acc[g0], acc[g0 + 1]), fmax_nan(acc[g0 + 4], acc[g0 + 5])) + bias, 0.f);
    pv.y = fmaxf(fmax_nan(fmax_nan(acc[g0 + 2], acc[g0 + 3]), fmax_nan(acc[g0 + 6], acc[g0 + 7])) + bias, 0.f);
    const int PY = 2 * ty2 + qy, PX = 4 * i + 2 * h;
    if constexpr (SPLIT_OUT) {
      uint32_t hi, lo;
      split2(pv.x, pv.y, hi, lo);
      char* bp = reinterpret_cast<char*>(out) + (oc2 * 2 + (PY >> 2)) * 128 + ((PY & 3) * 8 + PX) * 2;
      *reinterpret_cast<uint32_t*>(bp) = hi;
      *reinterpret_cast<uint32_t*>(bp + 64) = lo;
    } else {
      *reinterpret_cast<float2*>(out + oc2 * 64 + PY * 8 + PX) = pv;
    }
  }
}

template <int N>
__device__ __forceinline__ void resident_fence(const bf16x8 (&w)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" ::"v"(w[i]));
}

}  // namespace x3
}  // namespace dnn
