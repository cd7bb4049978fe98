// Gated delta rule (gfx950), per head with a matrix state (fp32,
// [slot][H][value][key channel]):
//   S <- g_t S,   u_t = beta_t (v_t - S^T k_t),   S <- S + k_t u_t^T,   y_t = S^T q_t
// with k and q as unit vectors (q also scaled) and g = exp(la).
//
//   delta_chunks  bf16, sequences of 2 tokens or more, on the MFMA
//   delta_steps   token by token in fp32: single decoded tokens, and the exact mode
//
// States are fp32 in pools by slot; a portion that begins at position 0 starts
// from zero.
#include "common.h"
#include "mixer_api.h"
#include "vec16.h"

namespace dnn {

typedef short s16x4 __attribute__((ext_vector_type(4)));
constexpr float LOG2E = 1.4426950408889634f;

// ---------------------------------------------------------------- token by token
// grid (H, VP / 64, sequences); LPR lanes share a state row (one value column),
// each holding float4s of it.  Both products with the state are summed at once:
// y = g S^T q + (k . q) u.
template <typename T, int NP>
__global__ __launch_bounds__(256) void delta_steps_kernel(DeltaArgs a) {
  constexpr int LPR = NP >= 64 ? 16 : NP / 4;  // lanes of a row
  constexpr int NI = NP / (4 * LPR);           // float4s of a lane and row
  constexpr int RPP = 256 / LPR, NR = 64 / RPP;
  const int h = blockIdx.x, v0 = blockIdx.y * 64;
  const int4 e = a.ent[blockIdx.z];
  const int slot = min(max(e.z, 0), a.nslots - 1);
  const int l = threadIdx.x % LPR, r0 = threadIdx.x / LPR;
  float* st = a.state + (((size_t)slot * a.H + h) * a.VP + v0) * NP;
  f32x4 S[NR][NI];
  const bool fresh = a.pos[e.x] == 0;
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      S[r][i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (!fresh) S[r][i] = *reinterpret_cast<const f32x4*>(st + (size_t)(r0 + r * RPP) * NP + i * 4 * LPR + l * 4);
    }
  for (int t = 0; t < e.y; ++t) {
    const int m = e.x + t;
    const T* row = reinterpret_cast<const T*>(a.rows) + (size_t)m * a.ld;
    const float beta = a.beta[(size_t)m * a.H + h], dec = expf(a.la[(size_t)m * a.H + h]);
    const T* qp = row + a.qcol + (h / a.qdiv) * NP + l * 4;
    const T* kp = row + a.kcol + (h / a.qdiv) * NP + l * 4;
    f32x4 q[NI], k[NI];
    float x[NR], qq = 0.f, kk = 0.f, kq = 0.f;
#pragma unroll
    for (int r = 0; r < NR; ++r) x[r] = to_f32(row[a.vcol + h * a.VP + v0 + r0 + r * RPP]);
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        q[i][j] = to_f32(qp[i * 4 * LPR + j]);
        k[i][j] = to_f32(kp[i * 4 * LPR + j]);
        qq = fmaf(q[i][j], q[i][j], qq);
        kk = fmaf(k[i][j], k[i][j], kk);
        kq = fmaf(k[i][j], q[i][j], kq);
      }
    const float rq = a.q_scale / sqrtf(group_sum<LPR>(qq) + a.unit_eps);
    const float rk = 1.0f / sqrtf(group_sum<LPR>(kk) + a.unit_eps);
    kq = group_sum<LPR>(kq) * rk * rq;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      q[i] *= rq;
      k[i] *= rk;
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      float sk = 0.f, sq = 0.f;
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          S[r][i][j] *= dec;
          sk = fmaf(S[r][i][j], k[i][j], sk);
          sq = fmaf(S[r][i][j], q[i][j], sq);
        }
      sk = group_sum<LPR>(sk);
      sq = group_sum<LPR>(sq);
      const float u = beta * (x[r] - sk);
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) S[r][i][j] = fmaf(k[i][j], u, S[r][i][j]);
      const int v = v0 + r0 + r * RPP;
      if (l == 0 && v < a.vdim)
        reinterpret_cast<T*>(a.y)[(size_t)m * a.ldy + h * a.vdim + v] = from_f32<T>(fmaf(u, kq, sq));
    }
  }
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int i = 0; i < NI; ++i)
      *reinterpret_cast<f32x4*>(st + (size_t)(r0 + r * RPP) * NP + i * 4 * LPR + l * 4) = S[r][i];
}

// ---------------------------------------------------------------- chunks
// 64 tokens at a time as four blocks of 16.  With A_t the running sum of la in
// the chunk and S the state before it,
//   u_t = beta_t (v_t - exp(A_t) S^T k_t - sum_{s < t} exp(A_t - A_s) (k_t . k_s) u_s)
//   y_t = exp(A_t) S^T q_t + sum_{s <= t} exp(A_t - A_s) (q_t . k_s) u_s
//   S  <- exp(A_L) S + sum_s k_s (exp(A_L - A_s) u_s)^T
// The u of a block depend on each other through a triangular 16 x 16 matrix T,
// and on the blocks before by products:  u = (1 + T)^-1 (r - T' u').
//
// Rows of T, T' and of the scores, and the inverse, do not need the state: four
// waves form them for all blocks.  Then every wave walks the blocks with 16 value
// columns of the state in its accumulators, which are the next product's operand
// as they lie.  The lengths of k and q enter as factors of fp32 results, so the
// operands k and q are exact.  The state, the u and every matrix enter the MFMA
// as two bf16 terms; the inverse is formed on the fp32 MFMA, doubling its size
// three times (no power of T is formed: keys that point alike make those large).
//
// PIPE: 8 waves.  Between two barriers four of them stage the operands of one
// chunk in LDS and form the matrices of the chunk before it, while the other
// four walk the one before that.  Else 4 waves do these in turn.
//
// A fragment of 32 columns holds for lane (t16 = lane & 15, g = lane >> 4) the
// columns 4 g + {0..3} and 16 + 4 g + {0..3} of row t16: the order in which two
// accumulator tiles hold 32 rows.
__device__ __forceinline__ uint32_t dr_pack2(float a, float b) {
  typedef float f32x2v __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v{a, b}), bf16x2v));
}
// Four values as bf16 and their remainders as bf16: about 16 bits of mantissa.
__device__ __forceinline__ void dr_split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  hi = dr_pack2(a, b);
  lo = dr_pack2(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xffff0000u));
}
__device__ __forceinline__ void dr_split4(const f32x4& v, uint2& hi, uint2& lo) {
  dr_split2(v[0], v[1], hi.x, lo.x);
  dr_split2(v[2], v[3], hi.y, lo.y);
}
__device__ __forceinline__ bf16x8 dr_frag(const uint2& a, const uint2& b) {
  const i32x4 v = {(int)a.x, (int)a.y, (int)b.x, (int)b.y};
  return __builtin_bit_cast(bf16x8, v);
}
__device__ __forceinline__ f32x4 dr_mfma(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// c + M1 M2 in fp32: m1 holds M1[t16][4 g + i], m2 and the result M2[4 g + i][t16]
__device__ __forceinline__ f32x4 dr_mul(const f32x4& m1, const f32x4& m2, f32x4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(m1[i], m2[i], c, 0, 0, 0);
  return c;
}

template <int NP, bool PIPE>
struct DeltaLds {
  static constexpr int PAIRS = NP / 32, KB = PAIRS * 1024;  // bytes of a block's k or q fragments
  static constexpr int RING = 8 * KB, NR = PIPE ? 3 : 1;    // k and q of a chunk; chunks staged at a time
  // rows of a block against n blocks take n KB: pairs of blocks as one fragment
  // per term, a last single block as one fragment of both terms
  static constexpr int O_T = 0, O_P = 6 * 1024, O_D = O_P + 10 * 1024;
  static constexpr int VST = 160, O_V = O_D + 4 * 1024;     // rows of v
  // per token: factors of k against the state, of q, of k into the state, then
  // the chunk's decay; sums of la, beta, 1 / length of k, scale / length of q
  static constexpr int O_C = O_V + 64 * VST, O_S = O_C + 3 * 256 + 16;
  static constexpr int SET = O_S + 4 * 256, TOTAL = NR * RING + (PIPE ? 2 : 1) * SET;
};
// Bytes before the rows of a block against n blocks
__device__ __forceinline__ constexpr int dr_base(int n) { return n * (n - 1) / 2 * 1024; }
// Place of lane (t16, g) among a block's k fragments: transposing reads of four
// rows spread over the banks.
__device__ __forceinline__ int dr_slot(int t16, int g) { return g * 16 + (t16 ^ ((g & 1) << 3)); }

template <int NP, bool PIPE>
__global__ __launch_bounds__(PIPE ? 512 : 256, 1) void delta_chunks_kernel(DeltaArgs a) {
  using L = DeltaLds<NP, PIPE>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int PAIRS = L::PAIRS;
  const int tid = threadIdx.x, lane = tid & 63, t16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
  const bool prepares = !PIPE || tid >= 256, walks = !PIPE || tid < 256;
  const int h = blockIdx.x, v0 = blockIdx.y * 64;
  const int4 e = a.ent[blockIdx.z];
  const int n = e.y, slot = min(max(e.z, 0), a.nslots - 1);
  float* state = a.state + (((size_t)slot * a.H + h) * a.VP + v0 + wave * 16 + t16) * NP + 4 * g;
  const bool fresh = a.pos[e.x] == 0;
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 S[2 * PAIRS];
#pragma unroll
  for (int i = 0; i < 2 * PAIRS; ++i) {
    S[i] = zero;
    if (walks && !fresh) S[i] = *reinterpret_cast<const f32x4*>(state + 16 * i);
  }
  const bf16_t* rows = reinterpret_cast<const bf16_t*>(a.rows) + (size_t)e.x * a.ld;
  const bf16_t* qb = rows + a.qcol + (h / a.qdiv) * NP + 4 * g;
  const bf16_t* kb = rows + a.kcol + (h / a.qdiv) * NP + 4 * g;
  const bf16_t* vb = rows + a.vcol + h * a.VP + v0 + (lane & 3) * 16;
  auto ring = [&](int c) __attribute__((always_inline)) { return smem + (PIPE ? c % 3 : 0) * L::RING; };
  auto set = [&](int c) __attribute__((always_inline)) { return smem + L::NR * L::RING + (PIPE ? c & 1 : 0) * L::SET; };

  // rows past the end repeat the last one: their step sizes are zero
  s16x4 pk[PAIRS][2], pq[PAIRS][2];
  i32x4 pv[2], cv[2];
  float pla = 0.f, pb = 0.f;
  auto fetch = [&](int c) __attribute__((always_inline)) {
    const size_t r = (size_t)min(c * 64 + wave * 16 + t16, n - 1) * a.ld;
#pragma unroll
    for (int i = 0; i < PAIRS; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        pk[i][j] = *reinterpret_cast<const s16x4*>(kb + r + i * 32 + j * 16);
        pq[i][j] = *reinterpret_cast<const s16x4*>(qb + r + i * 32 + j * 16);
      }
    const bf16_t* v = vb + (size_t)min(c * 64 + wave * 16 + (lane >> 2), n - 1) * a.ld;
#pragma unroll
    for (int j = 0; j < 2; ++j) pv[j] = *reinterpret_cast<const i32x4*>(v + j * 8);
    const size_t o = (size_t)(e.x + min(c * 64 + lane, n - 1)) * a.H + h;
    pla = a.la[o];
    pb = a.beta[o];
  };
  auto frag = [&](const s16x4 (&f)[2]) __attribute__((always_inline)) {
    return bf16x8{f[0][0], f[0][1], f[0][2], f[0][3], f[1][0], f[1][1], f[1][2], f[1][3]};
  };
  // 1 / length of the row of a lane's t16
  auto inv_len = [&](const s16x4 (&f)[PAIRS][2]) __attribute__((always_inline)) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < PAIRS; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x = bf2f_s(f[i][j >> 2][j & 3]);
        s = fmaf(x, x, s);
      }
    s = add16(s);
    s = add32(s);
    return 1.0f / sqrtf(s + a.unit_eps);
  };
  // what was fetched, of this wave's block, to LDS; v waits for the set of its chunk
  auto stage = [&](int c) __attribute__((always_inline)) {
    char* kr = ring(c) + wave * L::KB;
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      *reinterpret_cast<bf16x8*>(kr + i * 1024 + dr_slot(t16, g) * 16) = frag(pk[i]);
      *reinterpret_cast<bf16x8*>(kr + 4 * L::KB + i * 1024 + lane * 16) = frag(pq[i]);
    }
    const float rk = inv_len(pk), rq = inv_len(pq) * a.q_scale;
    float* sc = reinterpret_cast<float*>(set(c) + L::O_S);
    if (g == 0) {
      sc[128 + wave * 16 + t16] = rk;
      sc[192 + wave * 16 + t16] = rq;
    }
    if (wave == 0) {
      const bool live = c * 64 + lane < n;
      float A = live ? pla * LOG2E : 0.f;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const float u = __shfl_up(A, o, 64);
        if (lane >= o) A += u;
      }
      sc[lane] = A;
      sc[64 + lane] = live ? pb : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) cv[j] = pv[j];
  };
  // rows of block i against block j as operands
  auto put = [&](char* base, int blocks, int j, const f32x4& v) __attribute__((always_inline)) {
    uint2 hi, lo;
    dr_split4(v, hi, lo);
    char* p = base + (j >> 1) * 2048 + lane * 16;
    if ((j | 1) < blocks) {
      *reinterpret_cast<uint2*>(p + (j & 1) * 8) = hi;
      *reinterpret_cast<uint2*>(p + 1024 + (j & 1) * 8) = lo;
    } else {
      *reinterpret_cast<bf16x8*>(p) = dr_frag(hi, lo);
    }
  };
  auto prepare = [&](int c) __attribute__((always_inline)) {
    char* x = set(c);
    const char* kr = ring(c);
    const float* sc = reinterpret_cast<const float*>(x + L::O_S);
    auto four = [&](int o) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(sc + o + 4 * g); };
    // k_j . k_i and k_j . q_i: rows 4 g.. of block j, column t16 of block i
    auto scores = [&](int i, int j, f32x4& G, f32x4& Q) __attribute__((always_inline)) {
      G = zero, Q = zero;
#pragma unroll
      for (int p = 0; p < PAIRS; ++p) {
        const bf16x8 kj = *reinterpret_cast<const bf16x8*>(kr + j * L::KB + p * 1024 + dr_slot(t16, g) * 16);
        const bf16x8 ki = *reinterpret_cast<const bf16x8*>(kr + i * L::KB + p * 1024 + dr_slot(t16, g) * 16);
        const bf16x8 qi = *reinterpret_cast<const bf16x8*>(kr + (4 + i) * L::KB + p * 1024 + lane * 16);
        G = dr_mfma(kj, ki, G);
        Q = dr_mfma(kj, qi, Q);
      }
    };
    f32x4 G, Q;
    {  // this wave's block: T in both layouts, ta[i] = T[t16][4 g + i], tb[i] = T[4 g + i][t16]
      const int w = wave * 16, t = w + t16;
      scores(wave, wave, G, Q);
      const float At = sc[t], bt = sc[64 + t], kt = sc[128 + t], qt = sc[192 + t], Ae = sc[63];
      const f32x4 As = four(w), bs = four(64 + w), ks = four(128 + w);
      if (g == 0) {
        float* f = reinterpret_cast<float*>(x + L::O_C) + t;
        const float at = __builtin_amdgcn_exp2f(At);
        f[0] = kt * at;
        f[64] = qt * at;
        f[128] = kt * __builtin_amdgcn_exp2f(Ae - At);
        if (t == 0) f[192] = __builtin_amdgcn_exp2f(Ae);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
        *reinterpret_cast<i32x4*>(x + L::O_V + (w + (lane >> 2)) * L::VST + (lane & 3) * 32 + j * 16) = cv[j];
      f32x4 ta, tb, p, ea, eb;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int s = 4 * g + i;
        const float d = __builtin_amdgcn_exp2f(-fabsf(At - As[i])) * ks[i], y = kt * d * G[i];
        ta[i] = s < t16 ? bt * y : 0.f;
        tb[i] = t16 < s ? bs[i] * y : 0.f;
        p[i] = s <= t16 ? qt * d * Q[i] : 0.f;
        ea[i] = s == t16 ? 1.f : (s ^ t16) == 1 ? -ta[i] : 0.f;
        eb[i] = s == t16 ? 1.f : (s ^ t16) == 1 ? -tb[i] : 0.f;
      }
      put(x + L::O_P + dr_base(wave + 1), wave + 1, wave, p);
      // inverse of 1 + T: of 2 x 2 blocks, then E - E C E with C the lower left
      // quarter of blocks of twice the size
#pragma unroll
      for (int z = 2; z < 16; z *= 2) {
        f32x4 ca;
#pragma unroll
        for (int i = 0; i < 4; ++i) ca[i] = ((4 * g + i) ^ t16) / z == 1 ? ta[i] : 0.f;
        const f32x4 f = dr_mul(ca, eb, zero);  // C E
        const f32x4 ab = dr_mul(f, ea, zero), bb = z < 8 ? dr_mul(ea, f, zero) : zero;
        ea -= ab;
        eb -= bb;
      }
      uint2 hi, lo;
      dr_split4(ea * bs, hi, lo);  // the step sizes ride in its columns
      *reinterpret_cast<bf16x8*>(x + L::O_D + wave * 1024 + lane * 16) = dr_frag(hi, lo);
    }
    auto pair = [&](int i, int j) __attribute__((always_inline)) {
      scores(i, j, G, Q);
      const int t = i * 16 + t16;
      const float At = sc[t], kt = sc[128 + t], qt = sc[192 + t];
      const f32x4 As = four(j * 16), ks = four(128 + j * 16);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float d = __builtin_amdgcn_exp2f(At - As[r]) * ks[r];
        G[r] *= kt * d;
        Q[r] *= qt * d;
      }
      put(x + L::O_T + dr_base(i), i, j, G);
      put(x + L::O_P + dr_base(i + 1), i + 1, j, Q);
    };
    // (1 0) (3 0) | (2 0) (3 1) | (2 1) | (3 2)
    pair(wave == 0 ? 1 : wave == 3 ? 3 : 2, wave < 2 ? 0 : wave - 1);
    if (wave < 2) pair(3, wave);
  };
  auto walk = [&](int c) __attribute__((always_inline)) {  // the blocks in order (past the end every u is zero)
    const char* kr = ring(c);
    const char* m = set(c);
    bf16x8 sh[PAIRS], sl[PAIRS];
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      uint2 h0, h1, l0, l1;
      dr_split4(S[2 * p], h0, l0);
      dr_split4(S[2 * p + 1], h1, l1);
      sh[p] = dr_frag(h0, h1), sl[p] = dr_frag(l0, l1);
    }
    const float* cf = reinterpret_cast<const float*>(m + L::O_C);
    f32x4 x[4], y[4], U[4];
    uint2 uh[4], ul[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      x[b] = zero, y[b] = zero;
#pragma unroll
      for (int p = 0; p < PAIRS; ++p) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(kr + b * L::KB + p * 1024 + dr_slot(t16, g) * 16);
        const bf16x8 qf = *reinterpret_cast<const bf16x8*>(kr + (4 + b) * L::KB + p * 1024 + lane * 16);
        x[b] = dr_mfma(kf, sh[p], x[b]);
        y[b] = dr_mfma(qf, sh[p], y[b]);
        x[b] = dr_mfma(kf, sl[p], x[b]);
        y[b] = dr_mfma(qf, sl[p], y[b]);
      }
    }
    // acc + the sum over the u of the first `k` blocks (rows of a block against them at `base`)
    auto over = [&](const char* base, int k, f32x4 acc) __attribute__((always_inline)) {
      f32x4 low = zero;
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        if (j >= k) break;
        const bf16x8 f = *reinterpret_cast<const bf16x8*>(base + j * 1024 + lane * 16);
        if (j + 1 < k) {
          const bf16x8 lo = *reinterpret_cast<const bf16x8*>(base + j * 1024 + 1024 + lane * 16), u = dr_frag(uh[j], uh[j + 1]);
          acc = dr_mfma(f, u, acc);
          low = dr_mfma(f, dr_frag(ul[j], ul[j + 1]), low);
          low = dr_mfma(lo, u, low);
        } else {
          acc = dr_mfma(f, dr_frag(uh[j], uh[j]), acc);
          low = dr_mfma(f, dr_frag(ul[j], ul[j]), low);
        }
      }
      return acc + low;
    };
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int row = b * 16 + 4 * g;
      const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (LDS_AS s16x4*)(m + L::O_V + (row + (t16 >> 2)) * L::VST + (wave * 16 + 4 * (lane & 3)) * 2));
      const f32x4 c0 = *reinterpret_cast<const f32x4*>(cf + row);
      f32x4 r;
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = fmaf(-c0[i], x[b][i], bf2f_s(v[i]));
      if (b > 0) r -= over(m + L::O_T + dr_base(b), b, zero);
      uint2 hi, lo;
      dr_split4(r, hi, lo);
      const bf16x8 d = *reinterpret_cast<const bf16x8*>(m + L::O_D + b * 1024 + lane * 16);
      U[b] = dr_mfma(d, dr_frag(hi, hi), zero) + dr_mfma(d, dr_frag(lo, lo), zero);
      dr_split4(U[b], uh[b], ul[b]);
    }
    const int col = v0 + wave * 16 + t16;
    bf16_t* yp = reinterpret_cast<bf16_t*>(a.y) + (size_t)e.x * a.ldy + h * a.vdim + col;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int row = b * 16 + 4 * g;
      y[b] *= *reinterpret_cast<const f32x4*>(cf + 64 + row);
      y[b] = over(m + L::O_P + dr_base(b + 1), b + 1, y[b]);
    }
    if (v0 + 64 <= a.vdim && c * 64 + 64 <= n) {
      bf16_t* p = yp + (size_t)(c * 64 + 4 * g) * a.ldy;
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) p[(b * 16 + i) * a.ldy] = f2bf(y[b][i]);
    } else {
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = c * 64 + b * 16 + 4 * g + i;
          if (t < n && col < a.vdim) yp[(size_t)t * a.ldy] = f2bf(y[b][i]);
        }
    }
    const float dec = cf[192];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      U[b] *= *reinterpret_cast<const f32x4*>(cf + 128 + b * 16 + 4 * g);
      dr_split4(U[b], uh[b], ul[b]);
    }
    // 4 rows (tokens 4 g..) of channel 16 q + t16 of block b's keys
    auto col4 = [&](int b, int q) __attribute__((always_inline)) {
      return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (LDS_AS s16x4*)(kr + b * L::KB + (q >> 1) * 1024 + dr_slot(4 * g + (t16 >> 2), lane & 3) * 16 + (q & 1) * 8));
    };
#pragma unroll
    for (int q = 0; q < 2 * PAIRS; ++q) {
      S[q] *= dec;
#pragma unroll
      for (int b = 0; b < 4; b += 2) {
        const s16x4 k0 = col4(b, q), k1 = col4(b + 1, q);
        const bf16x8 f = {k0[0], k0[1], k0[2], k0[3], k1[0], k1[1], k1[2], k1[3]};
        S[q] = dr_mfma(f, dr_frag(uh[b], uh[b + 1]), S[q]);
        S[q] = dr_mfma(f, dr_frag(ul[b], ul[b + 1]), S[q]);
      }
    }
  };
  const int chunks = (n + 63) / 64;
  if (prepares) fetch(0);
  if constexpr (PIPE) {
    for (int i = 0; i < chunks + 2; ++i) {
      if (prepares) {
        if (i > 0 && i <= chunks) prepare(i - 1);
        if (i < chunks) {
          stage(i);
          fetch(i + 1);
        }
      } else if (i > 1) {
        walk(i - 2);
      }
      __syncthreads();
    }
  } else {
    for (int c = 0; c < chunks; ++c) {
      __syncthreads();  // the last chunk is read
      stage(c);
      __syncthreads();
      prepare(c);
      __syncthreads();
      fetch(c + 1);
      walk(c);
    }
  }
  if (!walks) return;
#pragma unroll
  for (int i = 0; i < 2 * PAIRS; ++i) *reinterpret_cast<f32x4*>(state + 16 * i) = S[i];
}

}  // namespace dnn

using namespace dnn;

static bool delta_ok(const DeltaArgs& a) {
  const int heads = a.qdiv > 0 ? (a.H - 1) / a.qdiv + 1 : 0;
  return a.M > 0 && a.H > 0 && a.qdiv > 0 && a.VP > 0 && a.VP % 64 == 0 && a.vdim > 0 && a.vdim <= a.VP && a.nent > 0 &&
         a.nent <= 65535 && a.nslots > 0 && (a.NP == 32 || a.NP == 64 || a.NP == 128 || a.NP == 256) && a.qcol >= 0 &&
         a.kcol >= 0 && a.vcol >= 0 && a.vcol + a.H * a.VP <= a.ld && a.qcol + heads * a.NP <= a.ld &&
         a.kcol + heads * a.NP <= a.ld && a.ldy >= a.H * a.vdim && ((uintptr_t)a.ent & 15) == 0 &&
         ((uintptr_t)a.state & 15) == 0 && a.state != nullptr && a.beta != nullptr && a.la != nullptr && a.pos != nullptr;
}

#define DELTA_NP(F)                                \
  switch (a->NP) {                                 \
    case 32: F(32) break;                          \
    case 64: F(64) break;                          \
    case 128: F(128) break;                        \
    default: F(256) break;                         \
  }

extern "C" int dnn_delta_steps(const DeltaArgs* a, int f32, hipStream_t st) {
  if (!delta_ok(*a)) return -1;
  const dim3 grid(a->H, a->VP / 64, a->nent);
#define DS(N)                                                                                     \
  {                                                                                               \
    if (f32) hipLaunchKernelGGL((delta_steps_kernel<float, N>), grid, dim3(256), 0, st, *a);      \
    else hipLaunchKernelGGL((delta_steps_kernel<bf16_t, N>), grid, dim3(256), 0, st, *a);         \
  }
  DELTA_NP(DS)
#undef DS
  return (int)hipGetLastError();
}

extern "C" int dnn_delta_chunks(const DeltaArgs* a, hipStream_t st) {
  if (!delta_ok(*a) || (a->ld | a->qcol | a->kcol | a->vcol) % 8 != 0 || ((uintptr_t)a->rows & 15) != 0) return -1;
  const dim3 grid(a->H, a->VP / 64, a->nent);
#define DC(N)                                                                                                   \
  {                                                                                                             \
    constexpr bool pipe = DeltaLds<N, true>::TOTAL <= 160 * 1024;                                               \
    constexpr int lds = DeltaLds<N, pipe>::TOTAL;                                                               \
    hipLaunchKernelGGL((delta_chunks_kernel<N, pipe>), grid, dim3(pipe ? 512 : 256), lds, st, *a);              \
  }
  DELTA_NP(DC)
#undef DC
  return (int)hipGetLastError();
}
