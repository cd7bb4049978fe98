#pragma once
// Decode attention that keeps the K/V stream running: every wave walks its own
// blocks of rows with the next block's keys in flight while it folds the values of
// this one, and no wave waits for another before the end.  Bound by the bytes of the
// caches: Llama-3 8B B=32 of 820 to 1100 keys 39.0 -> 24.3 us (5.2 TB/s; batches of keys,
// softmax over the split, batches of values before), of 560 21.7 -> 15.5 (all of a
// split's rows in flight at once before), B=64 of 1000 55 -> 42, B=1 of 2048 18.7 -> 10.2;
// GPT-2 B=64 of 385 to 512 18.5 -> 18.0, XL B=64 of 217 to 288 25.0 -> 20.0, of 60 17.6 -> 8.8;
// caches that memory holds, not the last-level cache.  Slower than before: 16384 keys of 25
// ungrouped heads, B=4, 80 -> 83, 32 ungrouped heads of 128, B=16 of 1024, 42.3 -> 43.2 (no
// model here has either).  Blocks of twice the rows: 0.5 us either way.
//
// Included by attention.hip inside namespace dnn (load_head8, bf16x2v).
//
// Values: a lane holds 8 dims (16 B) of a row, LPK = HD / 8 lanes a row, RG = 64 /
// LPK rows a load (1 KB in a row), U loads a block of R = U RG rows.
//  * One head a row (G = 1): keys in the same layout, scores by v_dot2 and a DPP sum
//    over the row's lanes, which leaves the score in every lane of the row -- where
//    the value row's 8 dims are.  Each group of LPK lanes runs its own softmax
//    (running maximum, sum, sums of values); nothing passes through LDS before the
//    groups and waves meet at the end.
//  * Grouped heads: scores of 16 keys x 16 head columns on MFMA (a block costs G
//    times the dot2s and sums the other way: 690 vector operations for 32 keys of
//    128 dims and 4 heads against 250), one softmax a wave, and its probabilities
//    reach the row layout as bf16 pairs through 64 B of LDS a row group, private to
//    the wave.
typedef uint16_t u16x2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float max_over_quarters(float v) { return max32(max16(v)); }  // lanes l, l ^ 16, l ^ 32, l ^ 48

// Sums of v[0..N) over the wave's row groups (LPK lanes apart), spread: quarter rr = lane
// >> 4 ends with values at(rr) .. at(rr) + N / 4 in v[0..N / 4): a swap and an add halve
// the values where a shuffle each would pass 4 N of them through the LDS unit.
template <int N, int LPK>
__device__ __forceinline__ int sum_row_groups(float (&v)[N], int lane) {
  if constexpr (LPK == 8) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] += dpp_f<0x128>(v[i]);  // row_ror:8
  }
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[i + N / 2]), false, false);
    v[i] = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  }
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + N / 4]), false, false);
    v[i] = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  }
  return ((lane >> 4) & 1) * (N / 2) + (lane >> 5) * (N / 4);
}

// PROJ (heads of 64, one workgroup a head and NW column tiles, blockIdx.y): the head's output, rounded to bf16 as it
// would be stored, times its 64 columns of W_o (wo, fragment order): part[head][row][N], N = 64 H.  The weights are
// asked for with the first keys.  Every column group forms the head's output for itself.
template <int HD, int G, int FM, bool NT, int NW, int U, bool PROJ = false>
__global__ __launch_bounds__(NW * 64) void attn_decode_stream_kernel(
    const bf16_t* __restrict__ q, int ldq, bf16_t* __restrict__ kc, bf16_t* __restrict__ vc, float* __restrict__ ws,
    int H, int Hkv, int S, const int* __restrict__ lens, const float* __restrict__ cosT,
    const float* __restrict__ sinT, float scale_log2, bf16_t* __restrict__ o_direct,
    const uint8_t* __restrict__ wo = nullptr, float* __restrict__ part = nullptr) {
  static_assert(!PROJ || (HD == 64 && G == 1), "two chunks of W_o a head");
  constexpr bool FUSED = FM != 0, ROPE = FM == 2;
  constexpr int LPK = HD / 8, RG = 64 / LPK, R = U * RG;
  static_assert(LPK == 8 || LPK == 16, "sums over row groups");
  constexpr bool MF = G > 1;
  constexpr int NT16 = R / 16, NKC = HD / 32;  // MF: key tiles of a block, k-steps of a tile
  static_assert(U % 2 == 0, "P.V folds row pairs");
  static_assert(!MF || (R % 16 == 0 && G <= 16), "MF: blocks of whole tiles");
  // MF: probabilities of a wave [row group][row pair][head][2]; q, the new key, the new value
  __shared__ __attribute__((aligned(16))) uint16_t pl[MF ? NW : 1][MF ? RG * U * G : PROJ ? HD : 8];
  __shared__ __attribute__((aligned(16))) uint16_t qkv[MF ? G + 2 : 1][HD];
  __shared__ __attribute__((aligned(16))) float red[NW * G * HD];
  __shared__ float mred[NW * G], lred[NW * G];

  const int bk = blockIdx.x, split = PROJ ? 0 : blockIdx.y, NS = PROJ ? 1 : gridDim.y;
  const int b = bk / Hkv, kvh = bk % Hkv;
  const int p_new = FUSED ? lens[b] : 0;
  const int len = FUSED ? min(p_new + 1, S) : min(lens[b], S);
  const int chunk = (len + NS - 1) / NS;
  const int k0 = split * chunk, k1 = min(len, k0 + chunk);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sub = lane % LPK, grp = lane / LPK;
  float* wsp = ws + ((size_t)bk * NS + split) * G * (HD + 2);
  const int ct = blockIdx.y * NW + wave;  // PROJ: the wave's column tile, and where its 4 columns' sums go
  float* const pdst = part + ((size_t)kvh * (gridDim.x / Hkv) + b) * (Hkv * HD) + ct * 16 + (lane >> 4) * 4;
  if (k0 >= k1) {  // nothing in this split (short context), or no key at all
    if (PROJ) {
      if (ct < Hkv * HD / 16 && (lane & 15) == 0) *reinterpret_cast<f32x4*>(pdst) = f32x4{0.f, 0.f, 0.f, 0.f};
    } else if (NS == 1) {
      for (int i = tid; i < G * HD; i += NW * 64) o_direct[(size_t)b * H * HD + kvh * G * HD + i] = 0;
    } else {
      for (int i = tid; i < G * (HD + 2); i += NW * 64) wsp[i] = (i % (HD + 2)) == HD ? -INFINITY : 0.f;
    }
    return;
  }
  const int n = k1 - k0;
  const bf16_t* kb = kc + (((size_t)b * Hkv + kvh) * S + k0) * HD;
  const bf16_t* vb = vc + (((size_t)b * Hkv + kvh) * S + k0) * HD + sub * 8;
  const bool own_new = FUSED && p_new < S && p_new >= k0 && p_new < k1;
  const int knew = own_new ? p_new - k0 : -1;

  const int hj = lane & 15, c4 = lane >> 4;
  i32x4 kr[MF ? NT16 * NKC : U], vr[U];
  auto load_v = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const i32x4* p = reinterpret_cast<const i32x4*>(vb + (size_t)min(blk * R + u * RG + grp, n - 1) * HD);
      vr[u] = NT ? __builtin_nontemporal_load(p) : *p;
    }
  };
  auto load_k = [&](int blk) __attribute__((always_inline)) {
    if constexpr (MF) {  // tile t, step k: key row t * 16 + hj, dims (c4 + 4 k) * 8
#pragma unroll
      for (int t = 0; t < NT16; ++t)
#pragma unroll
        for (int k = 0; k < NKC; ++k) {
          const i32x4* p = reinterpret_cast<const i32x4*>(kb + (size_t)min(blk * R + t * 16 + hj, n - 1) * HD +
                                                          (c4 + 4 * k) * 8);
          kr[t * NKC + k] = *p;
        }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const i32x4* p = reinterpret_cast<const i32x4*>(kb + (size_t)min(blk * R + u * RG + grp, n - 1) * HD + sub * 8);
        kr[u] = NT ? __builtin_nontemporal_load(p) : *p;
      }
    }
  };
  int blk = wave;
  uint32_t qp[4], nkp[4], nvp[4];  // G = 1: this lane's dims of q and the new row, as bf16 pairs
  bf16x8 qB[MF ? NKC : 1];         // MF: q^T, columns from G on zero
  const int pr = min(p_new, S - 1);
  if constexpr (MF) {
    // each 16 B of q, the new key and the new value once a workgroup, ahead of the
    // stream: loaded by every wave they were a third of all loads of a short context
    static_assert((G + 2) * LPK <= NW * 64, "one chunk a thread");
    const int hh = tid / LPK, cs = tid % LPK;
    float t8[8];
    if (hh <= G && (FUSED || hh < G))
      load_head8<HD, ROPE>(q + (size_t)b * ldq + (hh < G ? kvh * G + hh : H + kvh) * HD, cs, cosT, sinT, pr, t8);
    else if (FUSED && hh == G + 1)
      load_head8<HD, false>(q + (size_t)b * ldq + (H + Hkv + kvh) * HD, cs, nullptr, nullptr, 0, t8);
    __builtin_amdgcn_sched_barrier(0);
    load_k(blk);
    load_v(blk);
    __builtin_amdgcn_sched_barrier(0);
    if (hh < (FUSED ? G + 2 : G)) {
      uint4 c;
      c.x = pack2bf(t8[0], t8[1]);
      c.y = pack2bf(t8[2], t8[3]);
      c.z = pack2bf(t8[4], t8[5]);
      c.w = pack2bf(t8[6], t8[7]);
      *reinterpret_cast<uint4*>(&qkv[hh][cs * 8]) = c;
    }
    // LDS only: the K/V loads stay in flight across the barrier
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < NKC; ++k) {
      qB[k] = *reinterpret_cast<const bf16x8*>(&qkv[min(hj, G - 1)][(c4 + 4 * k) * 8]);
      if (hj >= G) qB[k] = bf16x8{};
    }
  } else {
    load_k(blk);
    load_v(blk);
    __builtin_amdgcn_sched_barrier(0);
    float t8[8];
    auto pack = [&](uint32_t (&d)[4]) {
#pragma unroll
      for (int j = 0; j < 4; ++j) d[j] = pack2bf(t8[2 * j], t8[2 * j + 1]);
    };
    load_head8<HD, ROPE>(q + (size_t)b * ldq + kvh * HD, sub, cosT, sinT, pr, t8);
    pack(qp);
    if constexpr (FUSED) {
      load_head8<HD, ROPE>(q + (size_t)b * ldq + (H + kvh) * HD, sub, cosT, sinT, pr, t8);
      pack(nkp);
      load_head8<HD, false>(q + (size_t)b * ldq + (H + Hkv + kvh) * HD, sub, nullptr, nullptr, 0, t8);
      pack(nvp);
    }
  }
  i32x4 wo_r[2];
  if constexpr (PROJ) {
    const i32x4* wp = reinterpret_cast<const i32x4*>(wo) + ((size_t)min(ct, Hkv * HD / 16 - 1) * (Hkv * 2) + kvh * 2) * 64 + lane;
    wo_r[0] = wp[0];
    wo_r[1] = wp[64];
    __builtin_amdgcn_sched_barrier(0);
  }

  // softmax state: G = 1, of the lane's row group; MF, of head hj over the wave (l: over the lane's keys).
  // The maximum starts finite: against -inf, scores that are -inf would make exp2(-inf + inf)
  float m = -FLT_MAX, l = 0.f, acc[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[g][j] = 0.f;
  for (; blk * R < n; blk += NW) {
    const bool more = (blk + NW) * R < n;
    const bool has_new = FUSED && knew >= blk * R && knew < blk * R + R;  // wave-uniform
    uint32_t pp[U / 2][G];  // probabilities of the lane's rows u, u + 1 as a bf16 pair
    if constexpr (MF) {
      if (has_new) {
#pragma unroll
        for (int t = 0; t < NT16; ++t)
          if (blk * R + t * 16 + hj == knew) {
#pragma unroll
            for (int k = 0; k < NKC; ++k) kr[t * NKC + k] = *reinterpret_cast<const i32x4*>(&qkv[G][(c4 + 4 * k) * 8]);
          }
      }
      f32x4 s[NT16];
#pragma unroll
      for (int t = 0; t < NT16; ++t) {
        s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < NKC; ++k)
          s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kr[t * NKC + k]), qB[k], s[t], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (more) load_k(blk + NW);
      __builtin_amdgcn_sched_barrier(0);
      // s[t][r] = (key t * 16 + c4 * 4 + r, head hj): row u * RG + grp of the value layout
      const int last = n - blk * R - c4 * 4;  // keys t * 16 + r < last exist
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < NT16; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[t][r] = t * 16 + r < last ? s[t][r] * scale_log2 : -INFINITY;
          mx = fmaxf(mx, s[t][r]);
        }
      const float mn = fmaxf(m, max_over_quarters(mx));
      const float al = mn == m ? 1.f : __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < NT16; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = __builtin_amdgcn_exp2f(s[t][r] - mn);
          sum += p;
          const int row = t * 16 + c4 * 4 + r, u = row / RG;
          if (hj < G) pl[wave][((row % RG) * (U / 2) + (u >> 1)) * G * 2 + hj * 2 + (u & 1)] = f2bf(p);
        }
      l = l * al + sum;
      // other lanes read what this one stored: the fence keeps the order (a wave's LDS
      // operations run in it), the vector type lets 16-bit stores be read in pairs
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int w = 0; w < U / 2; ++w)
#pragma unroll
        for (int g = 0; g < G; ++g)
          pp[w][g] = __builtin_bit_cast(
              uint32_t, *reinterpret_cast<const u16x2v*>(&pl[wave][((grp * (U / 2) + w) * G + g) * 2]));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (!__all(al == 1.f)) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const float ag = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(al), g));
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[g][j] *= ag;
        }
      }
    } else {
      if (has_new) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (blk * R + u * RG + grp == knew) kr[u] = i32x4{(int)nkp[0], (int)nkp[1], (int)nkp[2], (int)nkp[3]};
      }
      float p[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float d = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          d = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2v, qp[j]),
                                              __builtin_bit_cast(bf16x2v, (uint32_t)kr[u][j]), d, false);
        p[u] = group_sum<LPK>(d) * scale_log2;
      }
      __builtin_amdgcn_sched_barrier(0);
      if (more) load_k(blk + NW);
      __builtin_amdgcn_sched_barrier(0);
      const int last = n - blk * R - grp;  // rows u * RG < last exist
      float mn = m;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (u * RG < last) mn = fmaxf(mn, p[u]);
      const float al = mn == m ? 1.f : __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      float sum = 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        p[u] = u * RG < last ? __builtin_amdgcn_exp2f(p[u] - mn) : 0.f;
        sum += p[u];
      }
      l = l * al + sum;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[0][j] *= al;
#pragma unroll
      for (int w = 0; w < U / 2; ++w) pp[w][0] = pack2bf(p[2 * w], p[2 * w + 1]);
    }
    if (has_new) {
      i32x4 nv;
      if constexpr (MF)
        nv = *reinterpret_cast<const i32x4*>(&qkv[G + 1][sub * 8]);
      else
        nv = i32x4{(int)nvp[0], (int)nvp[1], (int)nvp[2], (int)nvp[3]};
#pragma unroll
      for (int u = 0; u < U; ++u)  // and past it (knew = n - 1): copies of the row as a slot's last owner left it
        if (blk * R + u * RG + grp >= knew) vr[u] = nv;
    }
#pragma unroll
    for (int u = 0; u < U; u += 2) {
      uint32_t pr[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        pr[2 * j] = __builtin_amdgcn_perm((uint32_t)vr[u + 1][j], (uint32_t)vr[u][j], 0x05040100u);
        pr[2 * j + 1] = __builtin_amdgcn_perm((uint32_t)vr[u + 1][j], (uint32_t)vr[u][j], 0x07060302u);
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          acc[g][j] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2v, pp[u / 2][g]),
                                                      __builtin_bit_cast(bf16x2v, pr[j]), acc[g][j], false);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) load_v(blk + NW);
    __builtin_amdgcn_sched_barrier(0);
  }

  // the wave's row groups, then the waves: a group without rows carries the lowest m, l = 0
  float mw = m, f = 1.f;
  if constexpr (!MF) {
    if constexpr (LPK == 8) mw = fmaxf(mw, dpp_f<0x128>(mw));  // row_ror:8
    mw = max_over_quarters(mw);
    f = m == mw ? 1.f : __builtin_amdgcn_exp2f(m - mw);
  }
  float ls = l * f;
  if constexpr (!MF && LPK == 8) ls += dpp_f<0x128>(ls);
  ls = add32(add16(ls));
  if (lane < G) {
    mred[wave * G + lane] = mw;
    lred[wave * G + lane] = ls;
  }
  {
    float v[G * 8];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int j = 0; j < 8; ++j) v[g * 8 + j] = MF ? acc[g][j] : acc[g][j] * f;
    const int at = sum_row_groups<G * 8, LPK>(v, lane);
    constexpr int NQ = G * 2;  // values a lane ends with
    if (LPK == 16 || (lane & 8) == 0) {
#pragma unroll
      for (int i = 0; i < NQ; i += 2)
        *reinterpret_cast<float2*>(red + (wave * G + (at + i) / 8) * HD + sub * 8 + (at + i) % 8) = float2{v[i], v[i + 1]};
    }
  }
  __syncthreads();
  for (int i = tid; i < G * HD; i += NW * 64) {
    const int g = i / HD, d = i % HD;
    float mw = mred[g];
#pragma unroll
    for (int w = 1; w < NW; ++w) mw = fmaxf(mw, mred[w * G + g]);
    float s = 0.f, ls = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = mred[w * G + g] == mw ? 1.f : __builtin_amdgcn_exp2f(mred[w * G + g] - mw);
      s += red[(w * G + g) * HD + d] * f;
      ls += lred[w * G + g] * f;
    }
    if constexpr (PROJ) {
      pl[0][d] = f2bf(ls > 0.f ? s / ls : 0.f);
    } else if (NS == 1) {
      o_direct[(size_t)b * H * HD + (kvh * G + g) * HD + d] = f2bf(ls > 0.f ? s / ls : 0.f);
    } else {
      wsp[g * (HD + 2) + d] = s;
      if (d == 0) {
        wsp[g * (HD + 2) + HD] = mw;
        wsp[g * (HD + 2) + HD + 1] = ls;
      }
    }
  }
  if constexpr (PROJ) {
    __syncthreads();
    f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 2; ++c)
      y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wo_r[c]),
                                                  *reinterpret_cast<const bf16x8*>(&pl[0][c * 32 + (lane >> 4) * 8]), y, 0, 0, 0);
    if (ct < Hkv * HD / 16 && (lane & 15) == 0) *reinterpret_cast<f32x4*>(pdst) = y;
  }
  // the new row into the cache, behind every load of the workgroup
  if (own_new && tid < LPK && (!PROJ || blockIdx.y == 0)) {
    const size_t at = (((size_t)b * Hkv + kvh) * S + p_new) * HD + sub * 8;
    uint4 wk, wv;
    if constexpr (MF) {
      wk = *reinterpret_cast<const uint4*>(&qkv[G][sub * 8]);
      wv = *reinterpret_cast<const uint4*>(&qkv[G + 1][sub * 8]);
    } else {
      wk = make_uint4(nkp[0], nkp[1], nkp[2], nkp[3]);
      wv = make_uint4(nvp[0], nvp[1], nvp[2], nvp[3]);
    }
    *reinterpret_cast<uint4*>(kc + at) = wk;
    *reinterpret_cast<uint4*>(vc + at) = wv;
  }
}
