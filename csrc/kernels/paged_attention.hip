// Attention over a paged KV cache, for batches of unequal sequences (gfx950).
//
// Cache: 64-key pages, keys [page][G][64][DK], values [page][G][64][DV] (DK and
// DV independent), addressed by a block table (slot, position / 64) -> page, so
// a sequence's keys may lie anywhere in the pool.  A query at position i sees
// key j when j <= i and (i - j < window or j < keep): a sliding window whose
// first `keep` keys stay visible; window = INT_MAX is plain causal attention.
// Only pages that hold a visible key are read.  The query heads of a KV head
// (H / G, any number) are packed with the queries into the 32 columns of the
// MFMA: column r of a sequence's chunk is (token r / R, head r % R), R = H / G.
// An optional output gate, sigmoid of a column of the projection row (one per
// head, or one per head and value), multiplies the head's output.  Optional
// score terms: a factor per cached key (a key norm that the cache does not
// hold) and a per-head slope times the distance, taken off.  A sink per head: a
// score that joins the softmax and has no value.  Values may be the keys
// themselves (one pool; qk_norm.hip writes it).
//
//   paged_write    new k / v rows -> pages
//   paged_prefill  chunks of >= 2 tokens; a workgroup takes 128 packed rows
//                  (4 waves x 32), pages staged through LDS
//   paged_decode   one token per sequence: 32-key units dealt to the 4 waves of
//                  a workgroup (and over `splits` workgroups), merged in LDS;
//                  the token's own k / v are written to the cache on the way
//   paged_attn_f32 fp32, one wave per (row, head): the exact mode
//
// Scores, softmax and accumulation are fp32; S^T = K Q^T keeps a query on one
// lane pair, so row maxima and sums are in registers, and O^T += V^T P^T takes
// P from the score registers and V^T by transposing LDS reads.
#include <algorithm>
#include <climits>

#include "attention_tile.h"
#include "residual_api.h"

namespace dnn {

__device__ __forceinline__ bool pa_sees(int i, int j, int window, int keep) {
  return j <= i && (i - j < window || j < keep);
}
// page index of (slot, block), -1 outside the table or the pool
__device__ __forceinline__ int pa_page(const PagedAttnArgs& a, int slot, int blk) {
  if (blk < 0 || blk >= a.ldt) return -1;
  const int p = a.table[(size_t)slot * a.ldt + blk];
  return p < a.npages ? p : -1;
}
// Visible key units of `unit` keys for queries qlo..qhi: the first ke units
// hold kept keys, wb..we the window.
struct Units {
  int ke, wb, total;
  __device__ __forceinline__ int at(int i) const { return i < ke ? i : wb + i - ke; }
};
__device__ __forceinline__ Units pa_units(int qlo, int qhi, int window, int keep, int unit) {
  const int we = qhi / unit + 1;
  Units u;
  u.ke = min((keep + unit - 1) / unit, we);
  u.wb = max(qlo >= window ? (qlo - window + 1) / unit : 0, u.ke);
  u.total = u.ke + max(we - u.wb, 0);
  return u;
}

// ---------------------------------------------------------------- cache write
template <typename T>
__global__ __launch_bounds__(256) void paged_write_kernel(PagedAttnArgs a) {
  constexpr int E = 16 / sizeof(T);
  const int ck = a.G * a.DK / E, cv = a.shared ? 0 : a.G * a.DV / E;
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i >= (long)a.M * (ck + cv)) return;
  const int m = (int)(i / (ck + cv));
  int c = (int)(i % (ck + cv));
  const int p = a.pos[m], page = pa_page(a, a.slots[m], p / PG);
  if (page < 0) return;
  const T* src = reinterpret_cast<const T*>(a.qkv) + (size_t)m * a.ldq + a.H * a.DK;
  T* dst;
  int d, g;
  if (c < ck) {
    g = c * E / a.DK;
    d = c * E - g * a.DK;
    src += c * E;
    dst = reinterpret_cast<T*>(a.kp) + (((size_t)page * a.G + g) * PG + p % PG) * a.DK + d;
  } else {
    c -= ck;
    g = c * E / a.DV;
    d = c * E - g * a.DV;
    src += a.G * a.DK + c * E;
    dst = reinterpret_cast<T*>(a.vp) + (((size_t)page * a.G + g) * PG + p % PG) * a.DV + d;
  }
  *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(src);
}

// ---------------------------------------------------------------- score terms
// Terms of the score beyond the dot product, for 4 consecutive keys key0.. of
// a page: s <- log2(e) * (s * kscale * scale - slope * (i - j)).
__device__ __forceinline__ bool pa_has_terms(const PagedAttnArgs& a) { return a.kscale != nullptr || a.slopes != nullptr; }
__device__ __forceinline__ f32x4 pa_kscale4(const PagedAttnArgs& a, int page, int key0) {
  if (a.kscale == nullptr) return f32x4{1.f, 1.f, 1.f, 1.f};
  return *reinterpret_cast<const f32x4*>(a.kscale + (size_t)page * PG + key0);
}
__device__ __forceinline__ float pa_slope(const PagedAttnArgs& a, int head) {
  return a.slopes != nullptr ? a.slopes[head] * LOG2E : 0.f;
}

// The softmax before any key (log2 units): empty, or the head's sink.
__device__ __forceinline__ void pa_begin(const PagedAttnArgs& a, int head, bool has, float& m, float& l) {
  has = has && a.sinks != nullptr;
  m = has ? a.sinks[head] * LOG2E : -INFINITY;
  l = has ? 1.f : 0.f;
}

__device__ __forceinline__ float pa_sigmoid(const PagedAttnArgs& a, int row, int col) {
  const float z = bf2f(reinterpret_cast<const bf16_t*>(a.qkv)[(size_t)row * a.ldq + a.gate + col]);
  return 1.0f / (1.0f + __expf(-z));
}
__device__ __forceinline__ float pa_gate_el(const PagedAttnArgs& a, int row, int col) {
  return a.gate >= 0 && a.gate_el ? pa_sigmoid(a, row, col) : 1.f;
}
__device__ __forceinline__ float pa_gate(const PagedAttnArgs& a, int row, int head) {
  if (a.gate < 0 || a.gate_el) return 1.f;
  const float z = bf2f(reinterpret_cast<const bf16_t*>(a.qkv)[(size_t)row * a.ldq + a.gate + head]);
  return 1.0f / (1.0f + __expf(-z));
}

// ---------------------------------------------------------------- prefill
// tiles: {first batch row of the chunk, its tokens, slot, first packed row}
template <int DK, int DV>
__device__ __forceinline__ void paged_prefill_tile(const PagedAttnArgs& a, const int4 t, const int g, char* smem) {
  char* ks = smem;
  char* vs = smem + PG * DK * 2;
  constexpr int NKS = DK / 16, NDT = DV / 32, CK = DK / 8, CV = DV / 8;
  constexpr int NIK = PG * CK / 256, NIV = PG * CV / 256;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int h = lane >> 5, r32 = lane & 31;
  const int R = a.H / a.G;
  const int tok0 = t.x, n = t.y, slot = t.z, row0 = t.w;
  const int p0 = a.pos[tok0];
  const int last = n - 1;
  const int wrow = row0 + wave * 32, row = wrow + r32;
  const int tk = min(row / R, last), head = g * R + row % R;
  const int q_abs = p0 + tk;
  const int wq_min = p0 + min(wrow / R, last), wq_max = p0 + min((wrow + 31) / R, last);
  const Units u = pa_units(p0 + min(row0 / R, last), p0 + min((row0 + 127) / R, last), a.window, a.keep, PG);

  bf16x8 qf[NKS];
  {
    const bf16_t* qp = reinterpret_cast<const bf16_t*>(a.qkv) + (size_t)(tok0 + tk) * a.ldq + head * DK + 8 * h;
#pragma unroll
    for (int s = 0; s < NKS; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + s * 16);
  }
  f32x16 o[NDT];
#pragma unroll
  for (int i = 0; i < NDT; ++i) o[i] = f32x16{};
  float m_i, l_i;
  pa_begin(a, head, true, m_i, l_i);
  const bool terms = pa_has_terms(a);
  const float sc0 = a.scale * LOG2E, sc = terms ? 1.f : sc0;
  const float slope = pa_slope(a, head);

  i32x4 pk[NIK], pv[NIV];
  auto fetch = [&](int i) __attribute__((always_inline)) {
    const int page = max(pa_page(a, slot, u.at(i)), 0);  // a missing page is never visible; stay in the pool
    const bf16_t* kb = reinterpret_cast<const bf16_t*>(a.kp) + ((size_t)page * a.G + g) * PG * DK;
    const bf16_t* vb = reinterpret_cast<const bf16_t*>(a.vp) + ((size_t)page * a.G + g) * PG * DV;
#pragma unroll
    for (int it = 0; it < NIK; ++it) pk[it] = *reinterpret_cast<const i32x4*>(kb + (it * 256 + tid) * 8);
#pragma unroll
    for (int it = 0; it < NIV; ++it) pv[it] = *reinterpret_cast<const i32x4*>(vb + (it * 256 + tid) * 8);
  };
  if (u.total > 0) fetch(0);
  for (int i = 0; i < u.total; ++i) {
    const int kb0 = u.at(i) * PG;
    __syncthreads();
#pragma unroll
    for (int it = 0; it < NIK; ++it) {
      const int e = it * 256 + tid, key = e / CK, c = e % CK;
      *reinterpret_cast<i32x4*>(ks + key * DK * 2 + (pa_swz<DK>(key, c) << 4)) = pk[it];
    }
#pragma unroll
    for (int it = 0; it < NIV; ++it) {
      const int e = it * 256 + tid, key = e / CV, c = e % CV;
      *reinterpret_cast<i32x4*>(vs + key * PaV<DV>::STRIDE + c * 16) = pv[it];
    }
    __syncthreads();
    if (i + 1 < u.total) fetch(i + 1);
    // any key of the page visible to the wave's queries wq_min..wq_max?
    if (kb0 > wq_max || (wq_min - (kb0 + PG - 1) >= a.window && kb0 >= a.keep)) continue;
    f32x16 s[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      s[kt] = f32x16{};
      const int key = kt * 32 + r32;
#pragma unroll
      for (int k = 0; k < NKS; ++k) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(ks + key * DK * 2 + (pa_swz<DK>(key, 2 * k + h) << 4));
        s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[k], s[kt], 0, 0, 0);
      }
    }
    if (terms) {
      const int page = max(pa_page(a, slot, u.at(i)), 0);
      const float off = -slope * (float)(q_abs - kb0);
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int k4 = kt * 32 + 8 * q + 4 * h;
          const f32x4 f = pa_kscale4(a, page, k4) * sc0;
          const float c = fmaf(slope, (float)k4, off);
#pragma unroll
          for (int j = 0; j < 4; ++j) s[kt][4 * q + j] = fmaf(s[kt][4 * q + j], f[j], fmaf(slope, (float)j, c));
        }
    }
    // every key visible to every query of the wave: no mask
    if (kb0 + PG - 1 > wq_min || !(wq_max - kb0 < a.window || kb0 + PG <= a.keep)) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (!pa_sees(q_abs, kb0 + kt * 32 + (e & 3) + 8 * (e >> 2) + 4 * h, a.window, a.keep)) s[kt][e] = -INFINITY;
    }
    const float alpha = pa_softmax<2>(s, sc, m_i, l_i);
    if (!__all(alpha == 1.f)) {
#pragma unroll
      for (int d = 0; d < NDT; ++d) o[d] *= alpha;
    }
    pa_pv<DV>(vs, s[0], o, lane);
    pa_pv<DV>(vs + 32 * PaV<DV>::STRIDE, s[1], o, lane);
  }
  if (row >= n * R) return;
  const float f = (l_i > 0.f ? 1.f / l_i : 0.f) * pa_gate(a, tok0 + tk, head);
  bf16_t* op = reinterpret_cast<bf16_t*>(a.out) + (size_t)(tok0 + tk) * a.ldo + head * DV;
#pragma unroll
  for (int d = 0; d < NDT; ++d)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = o[d][4 * q + j] * f;
      if (a.gate >= 0 && a.gate_el) {
        const bf16x4 z = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16_t*>(a.qkv) +
                                                          (size_t)(tok0 + tk) * a.ldq + a.gate + head * DV + d * 32 + 8 * q + 4 * h);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] *= 1.0f / (1.0f + __expf(-bf2f_s(z[j])));
      }
      *reinterpret_cast<uint2*>(op + d * 32 + 8 * q + 4 * h) = make_uint2(pack2bf(v[0], v[1]), pack2bf(v[2], v[3]));
    }
}

template <int DK, int DV>
__global__ __launch_bounds__(256, (DK + DV <= 256) ? 2 : 1) void paged_prefill_kernel(PagedAttnArgs a,
                                                                                      const int4* __restrict__ tiles) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  paged_prefill_tile<DK, DV>(a, tiles[blockIdx.y], blockIdx.x, smem);
}

// ---------------------------------------------------------------- decode
// A workgroup of NW waves: 32 query heads (at most) of KV head g of sequence e, part z of ns of its keys; rows[e] = the
// batch row.  ws (ns > 1): [e][H][ns][DV + 2] = {max, sum, O} partials.
//
// The token's own key and value are taken from the projection row by the wave that has their unit (the last one), and
// stored behind everything else: a store that the wave then waits for and reads back is a round trip more, and
// the page numbers of a wave are one load.  Eight waves where the launch leaves CUs idle: 32 heads over 8, 2 to 6
// sequences of 150 to 400 keys, 11.4 to 13.3 us with four waves and the store, 8.7 to 11.4 so: four dependent reads
// (row, slot, page, keys), 10 KB of code and two units of keys in turn.
constexpr int DU = 32;  // keys per unit

template <int DV, int NW>
__host__ __device__ constexpr int pa_dec_lds(int rt_rows) {
  const int v = NW * DU * (DV * 2 + 64), m = NW * rt_rows * (DV + 2) * 4;
  return v > m ? v : m;
}

template <int DK, int DV, int NW>
__device__ __forceinline__ void paged_decode_part(const PagedAttnArgs& a, const int* __restrict__ rows,
                                                  float* __restrict__ ws, const int grt, const int e, const int z,
                                                  const int ns, const bool written, char* smem) {
  constexpr int NKS = DK / 16, NDT = DV / 32, CV = DV / 8;
  constexpr int NIV = DU * CV / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, r32 = lane & 31;
  const int R = a.H / a.G, nrt = (R + 31) / 32;
  const int g = grt / nrt, rt = grt % nrt;
  const int rr = min(R - rt * 32, 32);  // query heads of this workgroup
  const int row = rows[e];
  const int slot = a.slots[row], p = a.pos[row];
  char* vs = smem + wave * DU * PaV<DV>::STRIDE;

  const Units u = pa_units(p, p, a.window, a.keep, DU);
  const int ub = (int)((long)u.total * z / ns), ue = (int)((long)u.total * (z + 1) / ns);

  const bf16_t* rowp = reinterpret_cast<const bf16_t*>(a.qkv) + (size_t)row * a.ldq;
  const bool own = !written && ue == u.total && ue > ub && wave == (u.total - 1 - ub) % NW;  // this wave has the token's unit
  auto store_own = [&]() {
    const int page = pa_page(a, slot, p / PG);
    if (page < 0) return;
    bf16_t* kd = reinterpret_cast<bf16_t*>(a.kp) + (((size_t)page * a.G + g) * PG + p % PG) * DK;
    bf16_t* vd = reinterpret_cast<bf16_t*>(a.vp) + (((size_t)page * a.G + g) * PG + p % PG) * DV;
    if (lane < DK / 8)
      *reinterpret_cast<uint4*>(kd + lane * 8) = *reinterpret_cast<const uint4*>(rowp + a.H * DK + g * DK + lane * 8);
    if (lane < DV / 8)
      *reinterpret_cast<uint4*>(vd + lane * 8) = *reinterpret_cast<const uint4*>(rowp + (a.H + a.G) * DK + g * DV + lane * 8);
  };
  // Heads of 256 have no register left for the row's own addresses, the pages and the gate (31 spilled for 18; 4 heads over 2, us a
  // launch and two small ones, 1 to 64 sequences of 300 keys 23 to 27 for 21 to 25, 32 of 4000 76 for 68): their token is stored
  // first and read back.
  constexpr bool WIDE = DK + DV >= 512;
  if constexpr (WIDE) {
    if (own) store_own();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  // pages of the wave's first 64 units, a lane each
  int pages = 0;
  if constexpr (!WIDE) {
    const int i = ub + wave + lane * NW;
    if (i < ue) pages = pa_page(a, slot, u.at(i) / (PG / DU));
  }
  bf16x8 qf[NKS];
  {
    const bf16_t* qp = rowp + (g * R + rt * 32 + min(r32, rr - 1)) * DK + 8 * h;
#pragma unroll
    for (int s = 0; s < NKS; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + s * 16);
  }
  f32x16 o[NDT];
#pragma unroll
  for (int i = 0; i < NDT; ++i) o[i] = f32x16{};
  float m_i, l_i;  // one wave of a token's workgroups brings the sink
  pa_begin(a, g * R + rt * 32 + min(r32, rr - 1), wave == 0 && z == 0, m_i, l_i);
  const bool terms = pa_has_terms(a);
  const float sc0 = a.scale * LOG2E, sc = terms ? 1.f : sc0;
  const float slope = pa_slope(a, g * R + rt * 32 + min(r32, rr - 1));

  bf16x8 kf[NKS];
  i32x4 pv[NIV];
  f32x4 ksc[4];
  auto load = [&](int i) __attribute__((always_inline)) {
    const int unit = u.at(i), k = (i - ub) / NW;
    const int page = max(!WIDE && k < 64 ? __builtin_amdgcn_readlane(pages, k) : pa_page(a, slot, unit / (PG / DU)), 0);
    const size_t k0 = ((size_t)page * a.G + g) * PG + (unit % (PG / DU)) * DU;
    const bf16_t* kb = reinterpret_cast<const bf16_t*>(a.kp) + (k0 + r32) * DK + 8 * h;
    const bf16_t* vb = reinterpret_cast<const bf16_t*>(a.vp) + k0 * DV;
    const int at = !WIDE && own && i == ue - 1 ? p - unit * DU : -1;  // the token's own row of the tile
    if (r32 == at) kb = rowp + (a.H + g) * DK + 8 * h;
    if (!a.shared) {
#pragma unroll
      for (int s = 0; s < NKS; ++s) kf[s] = *reinterpret_cast<const bf16x8*>(kb + s * 16);
    }
#pragma unroll
    for (int it = 0; it < NIV; ++it) {
      const int c = it * 64 + lane;
      pv[it] = *reinterpret_cast<const i32x4*>(c / CV == at ? rowp + (a.H + a.G) * DK + g * DV + c % CV * 8 : vb + c * 8);
    }
    if (terms) {
#pragma unroll
      for (int q = 0; q < 4; ++q) ksc[q] = pa_kscale4(a, page, (unit % (PG / DU)) * DU + 8 * q + 4 * h) * sc0;
    }
  };
  int i = ub + wave;
  constexpr bool AHEAD = NW == 4;  // eight waves have a unit or two each: the next one's loads ahead are code more than time
  if (AHEAD && i < ue) load(i);
  // the gate of the first value that this thread will store, ahead of the keys' arrival
  const int h0 = min(g * R + rt * 32 + tid / DV, a.H - 1);
  const float gate0 = pa_gate(a, row, h0) * pa_gate_el(a, row, h0 * DV + tid % DV);
  for (; i < ue; i += NW) {
    if constexpr (!AHEAD) load(i);
    const int kb0 = u.at(i) * DU;
    f32x16 s[1];
    s[0] = f32x16{};
    auto stage_v = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int it = 0; it < NIV; ++it) {
        const int c = it * 64 + lane;
        *reinterpret_cast<i32x4*>(vs + (c / CV) * PaV<DV>::STRIDE + (c % CV) * 16) = pv[it];
      }
    };
    if (a.shared) {  // the tile was read once, as values: the keys come from LDS
      stage_v();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int k = 0; k < NKS; ++k)
        kf[k] = *reinterpret_cast<const bf16x8*>(vs + r32 * PaV<DV>::STRIDE + (DK == DV ? 2 * k + h : 0) * 16);
    }
#pragma unroll
    for (int k = 0; k < NKS; ++k) s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[k], qf[k], s[0], 0, 0, 0);
    if (!a.shared) stage_v();
    if (terms) {
      const float off = -slope * (float)(p - kb0 - 4 * h);
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          s[0][4 * q + j] = fmaf(s[0][4 * q + j], ksc[q][j], fmaf(slope, (float)(8 * q + j), off));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (AHEAD && i + NW < ue) load(i + NW);
    if (kb0 + DU - 1 > p || !(p - kb0 < a.window || kb0 + DU <= a.keep)) {
#pragma unroll
      for (int q = 0; q < 16; ++q)
        if (!pa_sees(p, kb0 + (q & 3) + 8 * (q >> 2) + 4 * h, a.window, a.keep)) s[0][q] = -INFINITY;
    }
    const float alpha = pa_softmax<1>(s, sc, m_i, l_i);
    if (!__all(alpha == 1.f)) {
#pragma unroll
      for (int d = 0; d < NDT; ++d) o[d] *= alpha;
    }
    pa_pv<DV>(vs, s[0], o, lane);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }

  // merge the waves: {m, l, O[DV]} of each query head
  __syncthreads();
  float* mg = reinterpret_cast<float*>(smem);
  if (r32 < rr) {
    float* d = mg + (wave * rr + r32) * (DV + 2);
    if (h == 0) {
      d[0] = m_i;
      d[1] = l_i;
    }
#pragma unroll
    for (int t = 0; t < NDT; ++t)
#pragma unroll
      for (int q = 0; q < 16; ++q) d[2 + t * 32 + (q & 3) + 8 * (q >> 2) + 4 * h] = o[t][q];
  }
  __syncthreads();
  for (int x = tid; x < rr * DV; x += NW * 64) {
    const int r = x / DV, c = x % DV, head = g * R + rt * 32 + r;
    float m = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) m = fmaxf(m, mg[(w * rr + r) * (DV + 2)]);
    float l = 0.f, v = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float* d = mg + (w * rr + r) * (DV + 2);
      const float f = d[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(d[0] - m);
      l = fmaf(d[1], f, l);
      v = fmaf(d[2 + c], f, v);
    }
    if (ns == 1) {
      reinterpret_cast<bf16_t*>(a.out)[(size_t)row * a.ldo + head * DV + c] =
          f2bf((l > 0.f ? v / l : 0.f) * (!WIDE && x == tid ? gate0 : pa_gate(a, row, head) * pa_gate_el(a, row, head * DV + c)));
    } else {
      float* d = ws + (((size_t)e * a.H + head) * ns + z) * (DV + 2);
      if (c == 0) {
        d[0] = m;
        d[1] = l;
      }
      d[2 + c] = v;
    }
  }
  if (!WIDE && own) store_own();  // behind every read of the page by this workgroup; another one of the same head takes the row's own as well
}

// grid (G * head tiles, sequences, splits)
template <int DK, int DV, int NW>
__global__ __launch_bounds__(NW * 64, (DK + DV <= 256) ? 2 : 1) void paged_decode_kernel(PagedAttnArgs a,
                                                                                         const int* __restrict__ rows,
                                                                                         float* __restrict__ ws) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  paged_decode_part<DK, DV, NW>(a, rows, ws, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.z, a.written != 0, smem);
}

// Portions and single tokens of one step (their keys and values are in the pages): the tiles, then the sequences' parts,
// four waves each.  The few workgroups of the single tokens run beside the tiles instead of behind them: 128 to
// 160 workgroups of both, 12 to 13 and 16.4 us one after the other, 17.4 together.  So at every size: 1 to 256 sequences of 300 and
// 2000 keys beside 64 to 1536 new tokens, heads of 64 to 256, 1 to 16 KV heads, windows (180 combinations) take 0.54 to 0.97 of
// the two launches, one 1.02 (16 heads of 64, 256 sequences of 2000 keys beside one tile 401 : 409).
template <int DK, int DV>
__global__ __launch_bounds__(256, (DK + DV <= 256) ? 2 : 1) void paged_mixed_kernel(PagedAttnArgs a, const int4* __restrict__ tiles,
                                                                                    int ntiles, const int* __restrict__ rows,
                                                                                    int ns, float* __restrict__ ws) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int b = blockIdx.x, np = ntiles * a.G;
  if (b < np) {
    paged_prefill_tile<DK, DV>(a, tiles[b / a.G], b % a.G, smem);
    return;
  }
  const int per = a.G * ((a.H / a.G + 31) / 32), x = b - np;
  paged_decode_part<DK, DV, 4>(a, rows, ws, x % per, x / per / ns, x / per % ns, ns, true, smem);
}

// One workgroup per (sequence, head): the four waves take every fourth split.
__global__ __launch_bounds__(256) void paged_combine_kernel(PagedAttnArgs a, const int* __restrict__ rows, int ns,
                                                            const float* __restrict__ ws) {
  __shared__ float acc[4][256 + 2];
  const int e = blockIdx.x / a.H, head = blockIdx.x % a.H, row = rows[e];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float* d = ws + ((size_t)e * a.H + head) * ns * (a.DV + 2);
  float m = -INFINITY;
  for (int s = lane; s < ns; s += 64) m = fmaxf(m, d[(size_t)s * (a.DV + 2)]);
  m = wave_max(m);
  float l = 0.f, v[4] = {0.f, 0.f, 0.f, 0.f};
  for (int s = wave; s < ns; s += 4) {
    const float* q = d + (size_t)s * (a.DV + 2);
    const float f = q[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(q[0] - m);
    l = fmaf(q[1], f, l);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (lane + 64 * i < a.DV) v[i] = fmaf(q[2 + lane + 64 * i], f, v[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (lane + 64 * i < a.DV) acc[wave][lane + 64 * i] = v[i];
  if (lane == 0) acc[wave][256] = l;
  __syncthreads();
  const int c = threadIdx.x;
  if (c >= a.DV) return;
  l = acc[0][256] + acc[1][256] + acc[2][256] + acc[3][256];
  const float o = acc[0][c] + acc[1][c] + acc[2][c] + acc[3][c];
  reinterpret_cast<bf16_t*>(a.out)[(size_t)row * a.ldo + head * a.DV + c] =
      f2bf((l > 0.f ? o / l : 0.f) * pa_gate(a, row, head) * pa_gate_el(a, row, head * a.DV + c));
}

// ---------------------------------------------------------------- fp32
__global__ __launch_bounds__(256) void paged_attn_f32_kernel(PagedAttnArgs a) {
  __shared__ float qs[4][256], ps[4][PG];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int x = min((int)(blockIdx.x * 4 + wave), a.M * a.H - 1);  // surplus waves repeat the last row
  const int row = x / a.H, head = x % a.H, g = head / (a.H / a.G);
  const int slot = a.slots[row], p = a.pos[row];
  const float* rowp = reinterpret_cast<const float*>(a.qkv) + (size_t)row * a.ldq;
  for (int d = lane; d < a.DK; d += 64) qs[wave][d] = rowp[head * a.DK + d];
  __syncthreads();
  const Units u = pa_units(p, p, a.window, a.keep, PG);
  float m = a.sinks != nullptr ? a.sinks[head] : -INFINITY, l = a.sinks != nullptr ? 1.f : 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < u.total; ++i) {
    const int blk = u.at(i), page = pa_page(a, slot, blk);
    if (page < 0) continue;
    const int key = blk * PG + lane;
    const float* kr = reinterpret_cast<const float*>(a.kp) + (((size_t)page * a.G + g) * PG + lane) * a.DK;
    float s = -INFINITY;
    if (pa_sees(p, key, a.window, a.keep)) {
      s = 0.f;
      for (int d = 0; d < a.DK; d += 4) {
        const f32x4 k4 = *reinterpret_cast<const f32x4*>(kr + d);
        s = fmaf(k4[0], qs[wave][d], s);
        s = fmaf(k4[1], qs[wave][d + 1], s);
        s = fmaf(k4[2], qs[wave][d + 2], s);
        s = fmaf(k4[3], qs[wave][d + 3], s);
      }
      s *= a.scale;
      if (a.kscale != nullptr) s *= a.kscale[(size_t)page * PG + lane];
      if (a.slopes != nullptr) s -= a.slopes[head] * (float)(p - key);
    }
    const float m_new = fmaxf(m, wave_max(s));
    if (m_new == -INFINITY) continue;
    const float alpha = expf(m - m_new), pr = expf(s - m_new);
    l = l * alpha + wave_sum(pr);
    m = m_new;
    ps[wave][lane] = pr;
    __builtin_amdgcn_wave_barrier();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const float* vb = reinterpret_cast<const float*>(a.vp) + ((size_t)page * a.G + g) * PG * a.DV;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int d = lane + 64 * c;
      if (d >= a.DV) break;
      float v = o[c] * alpha;
      for (int j = 0; j < PG; ++j) v = fmaf(ps[wave][j], vb[(size_t)j * a.DV + d], v);
      o[c] = v;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  }
  float f = l > 0.f ? 1.f / l : 0.f;
  if (a.gate >= 0 && !a.gate_el) f *= 1.0f / (1.0f + expf(-rowp[a.gate + head]));
  float* op = reinterpret_cast<float*>(a.out) + (size_t)row * a.ldo + head * a.DV;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int d = lane + 64 * c;
    if (d >= a.DV) break;
    op[d] = o[c] * f * (a.gate >= 0 && a.gate_el ? 1.0f / (1.0f + expf(-rowp[a.gate + head * a.DV + d])) : 1.f);
  }
}

}  // namespace dnn

using namespace dnn;

static bool pa_ok(const PagedAttnArgs& a, int elem) {
  auto dim = [](int d) { return d == 64 || d == 128 || d == 256; };
  const int vec = 16 / elem;
  return a.M > 0 && a.G > 0 && a.H > 0 && a.H % a.G == 0 && dim(a.DK) && dim(a.DV) && a.ldq % vec == 0 &&
         a.ldo % 4 == 0 && a.ldo >= a.H * a.DV && a.ldq >= (a.H + a.G) * a.DK + (a.shared ? 0 : a.G * a.DV) &&
         (a.gate < 0 || a.gate + a.H * (a.gate_el ? a.DV : 1) <= a.ldq) && (!a.gate_el || a.gate % 4 == 0) &&
         (!a.shared || (a.kp == a.vp && a.DK == a.DV && a.written)) && ((uintptr_t)a.kscale & 15) == 0 && a.window > 0 && a.keep >= 0 && a.ldt > 0 && a.npages > 0 &&
         a.table != nullptr && a.slots != nullptr && a.pos != nullptr;
}

extern "C" int dnn_paged_write(const PagedAttnArgs* a, int f32, hipStream_t st) {
  if (!pa_ok(*a, f32 ? 4 : 2)) return -1;
  const long n = (long)a->M * a->G * (a->DK + (a->shared ? 0 : a->DV)) / (f32 ? 4 : 8);
  const dim3 grid((unsigned)((n + 255) / 256));
  if (f32) hipLaunchKernelGGL(paged_write_kernel<float>, grid, dim3(256), 0, st, *a);
  else hipLaunchKernelGGL(paged_write_kernel<bf16_t>, grid, dim3(256), 0, st, *a);
  return (int)hipGetLastError();
}

#define PA_DISPATCH(F)                                                           \
  {                                                                              \
    if (a->DK == 64 && a->DV == 64) F(64, 64)                                    \
    else if (a->DK == 64 && a->DV == 128) F(64, 128)                             \
    else if (a->DK == 64 && a->DV == 256) F(64, 256)                             \
    else if (a->DK == 128 && a->DV == 64) F(128, 64)                             \
    else if (a->DK == 128 && a->DV == 128) F(128, 128)                           \
    else if (a->DK == 128 && a->DV == 256) F(128, 256)                           \
    else if (a->DK == 256 && a->DV == 64) F(256, 64)                             \
    else if (a->DK == 256 && a->DV == 128) F(256, 128)                           \
    else F(256, 256)                                                             \
  }

extern "C" int dnn_paged_prefill(const PagedAttnArgs* a, const int* tiles, int ntiles, hipStream_t st) {
  if (!pa_ok(*a, 2) || ntiles <= 0 || ntiles > 65535 || !(a->scale > 0.f) || ((uintptr_t)tiles & 15) != 0) return -1;
  const dim3 grid(a->G, ntiles);
#define PF(K, V)                                                                                                     \
  hipLaunchKernelGGL((paged_prefill_kernel<K, V>), grid, dim3(256), PG * (K * 2 + PaV<V>::STRIDE), st, *a, \
                     (const int4*)tiles);
  PA_DISPATCH(PF)
#undef PF
  return (int)hipGetLastError();
}

static void launch_combine(const PagedAttnArgs* a, const int* rows, int nrows, int splits, const float* ws, hipStream_t st) {
  if (splits > 1)
    hipLaunchKernelGGL(paged_combine_kernel, dim3((unsigned)(nrows * a->H)), dim3(256), 0, st, *a, rows, splits, ws);
}
static bool pa_dec_ok(const PagedAttnArgs& a, int nrows, int splits, const float* ws, long long ws_elems) {
  return pa_ok(a, 2) && nrows > 0 && nrows <= 65535 && splits >= 1 && splits <= 256 && a.scale > 0.f &&
         (splits == 1 || (ws != nullptr && ws_elems >= (long long)nrows * a.H * splits * (a.DV + 2)));
}

extern "C" int dnn_paged_decode(const PagedAttnArgs* a, const int* rows, int nrows, int splits, float* ws,
                                long long ws_elems, hipStream_t st) {
  if (!pa_dec_ok(*a, nrows, splits, ws, ws_elems)) return -1;
  const int R = a->H / a->G, rr = R < 32 ? R : 32;
  const dim3 grid(a->G * ((R + 31) / 32), nrows, splits);
  // eight waves a workgroup where there is a CU for each and their tiles fit half its LDS
  const bool w8 = (long)grid.x * nrows * splits <= 256;
#define PD(K, V)                                                                                                          \
  {                                                                                                                       \
    constexpr bool fit = K + V <= 256;                                                                                    \
    if (fit && w8 && pa_dec_lds<V, 8>(rr) <= 80 * 1024)                                                                   \
      hipLaunchKernelGGL((paged_decode_kernel<K, V, fit ? 8 : 4>), grid, dim3(512), (pa_dec_lds<V, 8>(rr)), st, *a, rows, ws); \
    else                                                                                                                  \
      hipLaunchKernelGGL((paged_decode_kernel<K, V, 4>), grid, dim3(256), (pa_dec_lds<V, 4>(rr)), st, *a, rows, ws);        \
  }
  PA_DISPATCH(PD)
#undef PD
  launch_combine(a, rows, nrows, splits, ws, st);
  return (int)hipGetLastError();
}

// dnn_paged_prefill and dnn_paged_decode of one step whose rows' keys and values are written already, in one launch.
extern "C" int dnn_paged_mixed(const PagedAttnArgs* a, const int* tiles, int ntiles, const int* rows, int nrows, int splits,
                               float* ws, long long ws_elems, hipStream_t st) {
  if (!pa_dec_ok(*a, nrows, splits, ws, ws_elems) || ntiles <= 0 || ((uintptr_t)tiles & 15) != 0) return -1;
  const int R = a->H / a->G, rr = R < 32 ? R : 32;
  const long long wgs = (long long)ntiles * a->G + (long long)a->G * ((R + 31) / 32) * nrows * splits;
  if (wgs > INT_MAX) return -1;
#define PM(K, V)                                                                                                          \
  hipLaunchKernelGGL((paged_mixed_kernel<K, V>), dim3((unsigned)wgs), dim3(256),                                          \
                     (std::max(PG * (K * 2 + PaV<V>::STRIDE), pa_dec_lds<V, 4>(rr))), st, *a, (const int4*)tiles, ntiles, rows, \
                     splits, ws);
  PA_DISPATCH(PM)
#undef PM
  launch_combine(a, rows, nrows, splits, ws, st);
  return (int)hipGetLastError();
}

extern "C" int dnn_paged_attn_f32(const PagedAttnArgs* a, hipStream_t st) {
  if (!pa_ok(*a, 4)) return -1;
  hipLaunchKernelGGL(paged_attn_f32_kernel, dim3((unsigned)(((long)a->M * a->H + 3) / 4)), dim3(256), 0, st, *a);
  return (int)hipGetLastError();
}
