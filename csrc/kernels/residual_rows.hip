// Row kernels of decoder layers with an fp32 residual stream.
//
// rows_update: one pass over a row that joins sublayer outputs into the
// residual and prepares the next projection's input,
//   z  = y * [rsqrt(mean(y^2) + eps) * yw] [+ the same of y2] [+ sum_t w_t ys_t],
//        or the norm of y + sum_t w_t ys_t
//   x' = [x] [+ x_add] [+ position vector] + mult * z        (fp32)
//   copy = T(x')              the residual as a GEMM operand
//   h    = T(x' * rsqrt(mean(x'^2) + eps) * nw)               RMS norm, or
//        = T(tanh(alpha x') * nw + nb)                        dynamic tanh
//   h    = T(h + (h of the token before - h) * mu)              token shift of an RMS norm
// each part optional.  y rows may be gathered (the embedding: y = table,
// yidx = tokens, mult = the embedding scale), x rows too (the head's rows);
// ys are the rows of a mixture of experts, w_t their router weights.
// Rows are NP wide (padded, zeros past N); means are over the true width N.
// bf16 y / T in serving, fp32 in the exact mode.
//
// Token shift: a group of threads takes sh_rows neighbouring rows and keeps the
// last one's normed values in registers.  Where its rows continue a sequence, it
// forms the row before them once more (so x_out is not x_in).  The group that
// holds a sequence's first row of the step reads the state by slot, and forms
// the sequence's last row as well to store it there: no other group touches that
// state.
#include <algorithm>
#include "common.h"
#include "gemm_epilogue.h"
#include "residual_api.h"

namespace dnn {

__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 ld4(const bf16_t* p) {
  const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
  return f32x4{bf2f_s(v[0]), bf2f_s(v[1]), bf2f_s(v[2]), bf2f_s(v[3])};
}
__device__ __forceinline__ void st4(float* p, const f32x4& v) { *reinterpret_cast<f32x4*>(p) = v; }
__device__ __forceinline__ void st4(bf16_t* p, const f32x4& v) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pack2bf(v[0], v[1]), pack2bf(v[2], v[3]));
}

// Sum over the TPR threads of a row (TPR = 64: the wave; 256: the workgroup).
template <int TPR>
__device__ __forceinline__ float row_sum(float v, float* red) {
  v = wave_sum(v);
  if constexpr (TPR == 64) return v;
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

// Two sums at once over the TPR threads of a row.
template <int TPR>
__device__ __forceinline__ void row_sum2(float& u, float& v, float* red) {
  u = wave_sum(u);
  v = wave_sum(v);
  if constexpr (TPR == 64) return;
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = u, red[4 + wave] = v;
  __syncthreads();
  u = red[0] + red[1] + red[2] + red[3];
  v = red[4] + red[5] + red[6] + red[7];
}

// Entry c of the sinusoidal position vector: the angle in turns, reduced in
// fp64 before it becomes fp32.
__device__ __forceinline__ float pos_entry(int p, const double* freq, int c) {
  double t = (double)p * freq[c >> 1];
  t -= floor(t);
  const float a = 6.283185307179586f * (float)t;
  return (c & 1) != 0 ? cosf(a) : sinf(a);
}

// tanh for a bf16 result (straight line: one exponential, one reciprocal)
__device__ __forceinline__ float tanh_fast(float x) {
  return 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * 2.8853900817779268f));
}

// PART: what the row needs beyond x, y and an RMS norm, so that plain rows do
// not carry the registers of the rest.
enum RowsPart { ROWS_PLAIN = 0, ROWS_MORE = 1, ROWS_TWO = 2, ROWS_EXPERTS = 3, ROWS_POSITIONS = 4, ROWS_SHIFT = 5 };
// every part but PLAIN and SHIFT also has x_add and the dynamic tanh; MORE has nothing else
constexpr bool rows_more(int part) { return part != ROWS_PLAIN && part != ROWS_SHIFT; }

template <typename YT, typename OT, int TPR, int NC, int PART>
__global__ __launch_bounds__(256) void rows_update_kernel(RowsArgs a) {
  __shared__ float red[8];
  const int t = threadIdx.x % TPR;
  // few values per thread: the norm weights stay in registers over a
  // workgroup's rows, and everything of a row is one memory round trip
  constexpr bool PF = NC <= 4, TWO = PART == ROWS_TWO, SHIFT = PART == ROWS_SHIFT;
  constexpr bool NB = PF && rows_more(PART);
  f32x4 yw[PF ? NC : 1], nw[PF ? NC : 1], y2w[PF && TWO ? NC : 1], nb[NB ? NC : 1];
  f32x4 mu[PF && SHIFT ? NC : 1], prev[SHIFT ? NC : 1];
  if constexpr (PF) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = (t + TPR * i) * 4;
      if (c >= a.NP) continue;
      if (a.y_w != nullptr) yw[i] = ld4(a.y_w + c);
      if (a.n_w != nullptr) nw[i] = ld4(a.n_w + c);
      if constexpr (TWO) y2w[i] = ld4(a.y2_w + c);
      if constexpr (NB)
        if (a.n_b != nullptr) nb[i] = ld4(a.n_b + c);
      if constexpr (SHIFT) mu[i] = ld4(a.sh_mu + c);
    }
  }
  // TPR 256: rows are uniform over the workgroup
  int it = (SHIFT ? xcd_remap(blockIdx.x, gridDim.x) : (int)blockIdx.x) * (256 / TPR) + threadIdx.x / TPR;
  int it_end = a.M, step = gridDim.x * (256 / TPR);
  int beg = 0, end = 0, tail = 0;  // SHIFT: this group's rows, and the last row it also forms
  if constexpr (SHIFT) {
    it = __builtin_amdgcn_readfirstlane(it);  // uniform over the wave: the rows' indices are scalar loads
    beg = it * a.sh_rows;
    if (beg >= a.M) return;
    end = min(beg + a.sh_rows, a.M);
    it = beg > 0 && a.sh_start[beg] != beg ? beg - 1 : beg;
    tail = min(a.sh_last[end - 1], a.M - 1);
    it_end = a.sh_start[end - 1] >= beg && tail >= end ? end + 1 : end;
    step = 1;
#pragma unroll
    for (int i = 0; i < NC; ++i) prev[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (; it < it_end; it += step) {
  const int m = SHIFT && it >= end ? tail : it;
  const bool ghost = SHIFT && (it < beg || it >= end);  // formed for its normed values only
  const int xr = a.xidx != nullptr ? min(max(a.xidx[m], 0), a.xrows - 1) : m;
  f32x4 x[NC], y[NC], y2[PF && TWO ? NC : 1];
  const float* xp = a.x_in != nullptr ? a.x_in + (size_t)xr * a.ldx : nullptr;
  const YT* yp = nullptr;
  if (a.y != nullptr) {
    const int yr = a.yidx != nullptr ? min(max(a.yidx[m], 0), a.yrows - 1) : m;
    yp = reinterpret_cast<const YT*>(a.y) + (size_t)yr * a.ldy;
  }
  bool first = false, keeps = false;
  float* state = nullptr;
  if constexpr (SHIFT) {
    const int start = a.sh_start[m];
    first = start == m, keeps = a.sh_last[m] == m && start >= beg;
    state = a.sh_state + (size_t)min(max(a.sh_slots[m], 0), a.sh_nslots - 1) * a.NP;
    if (first && !ghost) {
      const bool fresh = a.sh_pos[m] == 0;
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        const int c = (t + TPR * i) * 4;
        prev[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (c < a.NP && !fresh) prev[i] = ld4(state + c);
      }
    }
  }
  const YT* y2p = TWO ? reinterpret_cast<const YT*>(a.y2) + (size_t)m * a.ldy2 : nullptr;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = (t + TPR * i) * 4;
    x[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    y[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (PF && TWO) y2[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (c < a.NP) {
      if (xp != nullptr) x[i] = ld4(xp + c);
      if (yp != nullptr) y[i] = ld4(yp + c);
      if constexpr (PF && TWO) y2[i] = ld4(y2p + c);
    }
  }
  if constexpr (TWO) {  // both outputs normalised
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = (t + TPR * i) * 4;
      f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (PF) v = y2[i];
      else if (c < a.NP) v = ld4(y2p + c);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s1 = fmaf(y[i][j], y[i][j], s1);
        s2 = fmaf(v[j], v[j], s2);
      }
    }
    row_sum2<TPR>(s1, s2, red);
    const float r1 = 1.0f / sqrtf(s1 / (float)a.N + a.eps), r2 = 1.0f / sqrtf(s2 / (float)a.N + a.eps);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = (t + TPR * i) * 4;
      if (c < a.NP)
        y[i] = y[i] * r1 * (PF ? yw[PF ? i : 0] : ld4(a.y_w + c)) + (PF ? y2[PF ? i : 0] * y2w[PF ? i : 0] : ld4(y2p + c) * ld4(a.y2_w + c)) * r2;
    }
  } else if (a.y_w != nullptr && !(PART == ROWS_EXPERTS && a.y_joined)) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) s = fmaf(y[i][j], y[i][j], s);
    const float r = 1.0f / sqrtf(row_sum<TPR>(s, red) / (float)a.N + a.eps);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = (t + TPR * i) * 4;
      if (c < a.NP) y[i] = y[i] * r * (PF ? yw[PF ? i : 0] : ld4(a.y_w + c));
    }
  }
  if constexpr (PART == ROWS_EXPERTS) {
    const int* si = a.ysi + (size_t)m * a.top;
    const float* sw = a.ysw + (size_t)m * a.top;
    for (int k = 0; k < a.top; k += 4) {  // four rows in flight
      const YT* p[4];
      float w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = min(k + u, a.top - 1);
        p[u] = reinterpret_cast<const YT*>(a.ys) + (size_t)min(max(si[q], 0), a.ysrows - 1) * a.ldys;
        w[u] = k + u < a.top ? sw[q] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        const int c = (t + TPR * i) * 4;
        if (c >= a.NP) continue;
        f32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = ld4(p[u] + c);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int j = 0; j < 4; ++j) y[i][j] = fmaf(w[u], v[u][j], y[i][j]);
      }
    }
    if (a.y_joined) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) s = fmaf(y[i][j], y[i][j], s);
      const float r = 1.0f / sqrtf(row_sum<TPR>(s, red) / (float)a.N + a.eps);
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        const int c = (t + TPR * i) * 4;
        if (c < a.NP) y[i] = y[i] * r * (PF ? yw[PF ? i : 0] : ld4(a.y_w + c));
      }
    }
  }
  if (rows_more(PART) && a.x_add != nullptr) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = (t + TPR * i) * 4;
      if (c < a.NP) x[i] = x[i] + ld4(a.x_add + (size_t)m * a.ldadd + c);
    }
  }
  if constexpr (PART == ROWS_POSITIONS) {
    const int p = a.pos[m];
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = (t + TPR * i) * 4 + j;
        if (c < a.N) x[i][j] += pos_entry(p, a.freq, c);
      }
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = (t + TPR * i) * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[i][j] = fmaf(a.mult, y[i][j], x[i][j]);
      s = fmaf(x[i][j], x[i][j], s);
    }
    if (c < a.NP && !ghost) {
      if (a.x_out != nullptr) st4(a.x_out + (size_t)m * a.ldx + c, x[i]);
      if (a.copy != nullptr) st4(reinterpret_cast<OT*>(a.copy) + (size_t)m * a.ldcopy + c, x[i]);
    }
  }
  if (a.n_w == nullptr) continue;
  if (rows_more(PART) && a.n_b != nullptr) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = (t + TPR * i) * 4;
      if (c >= a.NP) continue;
      const f32x4 w = PF ? nw[PF ? i : 0] : ld4(a.n_w + c), b = NB ? nb[NB ? i : 0] : ld4(a.n_b + c);
      f32x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = fmaf(sizeof(OT) == 2 ? tanh_fast(a.n_alpha * x[i][j]) : tanhf(a.n_alpha * x[i][j]), w[j], b[j]);
      st4(reinterpret_cast<OT*>(a.h) + (size_t)m * a.ldh + c, v);
    }
    continue;
  }
  const float r = 1.0f / sqrtf(row_sum<TPR>(s, red) / (float)a.N + a.eps);
  if constexpr (SHIFT) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = (t + TPR * i) * 4;
      if (c >= a.NP) continue;
      const f32x4 h = x[i] * r * (PF ? nw[PF ? i : 0] : ld4(a.n_w + c));
      if (!ghost) {
        const f32x4 w = PF ? mu[PF ? i : 0] : ld4(a.sh_mu + c);
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = fmaf(prev[i][j] - h[j], w[j], h[j]);
        st4(reinterpret_cast<OT*>(a.h) + (size_t)m * a.ldh + c, v);
      }
      if (keeps) st4(state + c, h);
      prev[i] = h;
    }
    continue;
  }
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = (t + TPR * i) * 4;
    if (c < a.NP) st4(reinterpret_cast<OT*>(a.h) + (size_t)m * a.ldh + c, x[i] * r * (PF ? nw[PF ? i : 0] : ld4(a.n_w + c)));
  }
  }
}

// rows_update in bf16 of rows 1024 NC wide with nothing extra: one row a workgroup, no bounds, everything loaded ahead
// of the first sum, one barrier a sum.  IN: the row comes from a table, is a residual and an output, or is the residual
// alone (by index).  YN: y is normed.  OUT: what is made of x' beside itself.
// A row is a trip to memory and two sums, and the launch of a step begins with no instructions in the cache, so the
// 0.5 to 2.3 KB of a form 4096 wide count against the general kernel's 4.1.  Within a step: 1 to 6 rows 4.2 to 4.8
// us -> 2.3 to 4, 512 rows 7 -> 5.4 to 6.1; a step's rows of 512 move 14 MB to 20 MB (2 to 3 us).
enum LeanIn { LEAN_TABLE = 0, LEAN_JOIN = 1, LEAN_ROWS = 2 };
enum LeanOut { LEAN_X = 0, LEAN_NORM = 1, LEAN_COPY = 2 };

template <int NC, int IN, bool YN, int OUT>
__global__ __launch_bounds__(256) void rows_lean_kernel(const float* x_in, const bf16_t* y, const int* idx, int rows,
                                                        const float* y_w, float* x_out, const float* n_w, bf16_t* out,
                                                        int ldx, int ldy, int ldo, int N, float mult, float eps) {
  __shared__ float red[8];
  const int wave = threadIdx.x >> 6, c = threadIdx.x * 4;
  const size_t m = blockIdx.x;
  size_t in = m;
  if constexpr (IN != LEAN_JOIN)
    if (idx != nullptr) in = (size_t)min(max(idx[m], 0), rows - 1);
  f32x4 xv[NC], yv[NC], yw[NC], nw[NC];
  bf16x4 yb[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    if constexpr (IN != LEAN_ROWS) yb[i] = *reinterpret_cast<const bf16x4*>(y + in * ldy + c + 1024 * i);
    if constexpr (IN != LEAN_TABLE) xv[i] = ld4(x_in + in * ldx + c + 1024 * i);
    if constexpr (YN) yw[i] = ld4(y_w + c + 1024 * i);
    if constexpr (OUT == LEAN_NORM) nw[i] = ld4(n_w + c + 1024 * i);
  }
#pragma unroll
  for (int i = 0; i < NC; ++i)
    if constexpr (IN != LEAN_ROWS) yv[i] = f32x4{bf2f_s(yb[i][0]), bf2f_s(yb[i][1]), bf2f_s(yb[i][2]), bf2f_s(yb[i][3])};
  if constexpr (YN) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) s = fmaf(yv[i][j], yv[i][j], s);
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[wave] = s;
    __syncthreads();
    const float r = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)N + eps);
#pragma unroll
    for (int i = 0; i < NC; ++i) yv[i] = yv[i] * r * yw[i];
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (IN != LEAN_ROWS) xv[i][j] = fmaf(mult, yv[i][j], IN == LEAN_JOIN ? xv[i][j] : 0.f);
      if constexpr (OUT == LEAN_NORM) s = fmaf(xv[i][j], xv[i][j], s);
    }
    if constexpr (IN != LEAN_ROWS) st4(x_out + m * ldx + c + 1024 * i, xv[i]);
    if constexpr (OUT == LEAN_COPY) st4(out + m * ldo + c + 1024 * i, xv[i]);
  }
  if constexpr (OUT == LEAN_NORM) {
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[4 + wave] = s;
    __syncthreads();
    const float r = 1.0f / sqrtf((red[4] + red[5] + red[6] + red[7]) / (float)N + eps);
#pragma unroll
    for (int i = 0; i < NC; ++i) st4(out + m * ldo + c + 1024 * i, xv[i] * r * nw[i]);
  }
}

// 1: not one of these forms.
template <int NC>
static int lean_launch(const RowsArgs& a, hipStream_t st) {
#define LEAN(IN, YN, OUT)                                                                                               \
  {                                                                                                                     \
    hipLaunchKernelGGL((rows_lean_kernel<NC, IN, YN, OUT>), dim3(a.M), dim3(256), 0, st, a.x_in, (const bf16_t*)a.y,    \
                       IN == LEAN_ROWS ? a.xidx : a.yidx, IN == LEAN_ROWS ? a.xrows : a.yrows, a.y_w, a.x_out, a.n_w,   \
                       (bf16_t*)(OUT == LEAN_COPY ? a.copy : a.h), a.ldx, a.ldy, OUT == LEAN_COPY ? a.ldcopy : a.ldh,   \
                       a.N, a.mult, a.eps);                                                                             \
    return (int)hipGetLastError();                                                                                      \
  }
  const bool norm = a.n_w != nullptr, copy = a.copy != nullptr;
  if (norm && copy) return 1;
  if (a.y == nullptr) {
    if (a.x_in == nullptr || a.x_out != nullptr || !norm) return 1;
    LEAN(LEAN_ROWS, false, LEAN_NORM)
  }
  if (a.x_out == nullptr) return 1;
  if (a.x_in == nullptr) {
    if (a.y_w != nullptr || !norm) return 1;
    LEAN(LEAN_TABLE, false, LEAN_NORM)
  }
  if (a.yidx != nullptr || a.xidx != nullptr) return 1;
  if (a.y_w == nullptr) {
    if (norm) LEAN(LEAN_JOIN, false, LEAN_NORM)
    if (copy) LEAN(LEAN_JOIN, false, LEAN_COPY)
    LEAN(LEAN_JOIN, false, LEAN_X)
  }
  if (norm) LEAN(LEAN_JOIN, true, LEAN_NORM)
  if (copy) LEAN(LEAN_JOIN, true, LEAN_COPY)
  LEAN(LEAN_JOIN, true, LEAN_X)
#undef LEAN
}

// The token shift of such rows (ROWS_SHIFT), a workgroup a row: it forms its own row and the one whose normed values it
// needs beside it -- the row before, or the sequence's last one, for the state, where its own is the first -- and both
// rows' loads are in flight and both rows' sums add up at once.  The general kernel's groups form theirs one after the other.  Bound as rows_lean_kernel is;
// us of 4096 columns, general : this: 1 row 4.9 : 4.0, 506 rows 9.3 : 7.3, 640 11.0 : 8.5, 1300 17.4 : 14.5, 2048 23.1 : 19.4 (a
// launch over and over; in a step 5 rows 7.3, 640 13.5 before).
template <int NC, int IN, bool YN>
__global__ __launch_bounds__(256) void rows_shift_kernel(RowsArgs a) {
  __shared__ float red[16];
  const int wave = threadIdx.x >> 6, c = threadIdx.x * 4, m = xcd_remap(blockIdx.x, gridDim.x);
  f32x4 x[2][NC], yw[NC], nw[NC], mu[NC], prev[NC];
  bf16x4 yb[2][NC];
  auto load = [&](int k, int row) __attribute__((always_inline)) {
    size_t yr = row;
    if constexpr (IN == LEAN_TABLE)
      if (a.yidx != nullptr) yr = (size_t)min(max(a.yidx[row], 0), a.yrows - 1);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      yb[k][i] = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16_t*>(a.y) + yr * a.ldy + c + 1024 * i);
      if constexpr (IN == LEAN_JOIN) x[k][i] = ld4(a.x_in + (size_t)row * a.ldx + c + 1024 * i);
    }
  };
  load(0, m);
  load(1, max(m - 1, 0));
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    if constexpr (YN) yw[i] = ld4(a.y_w + c + 1024 * i);
    nw[i] = ld4(a.n_w + c + 1024 * i);
    mu[i] = ld4(a.sh_mu + c + 1024 * i);
    prev[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const bool first = a.sh_start[m] == m;
  const int last = min(max(a.sh_last[m], m), a.M - 1);
  float* state = a.sh_state + (size_t)min(max(a.sh_slots[m], 0), a.sh_nslots - 1) * a.NP + c;
  if (first) {
    if (a.sh_pos[m] != 0) {
#pragma unroll
      for (int i = 0; i < NC; ++i) prev[i] = ld4(state + 1024 * i);
    }
    if (last != m) load(1, last);
  }
  f32x4 y[2][NC];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int i = 0; i < NC; ++i) y[k][i] = f32x4{bf2f_s(yb[k][i][0]), bf2f_s(yb[k][i][1]), bf2f_s(yb[k][i][2]), bf2f_s(yb[k][i][3])};
  // 1 / the root of the mean square of both rows
  auto norms = [&](const f32x4 (&v)[2][NC], float* sums, float (&r)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) s = fmaf(v[k][i][j], v[k][i][j], s);
      s = wave_sum(s);
      if ((threadIdx.x & 63) == 0) sums[4 * k + wave] = s;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k)
      r[k] = 1.0f / sqrtf((sums[4 * k] + sums[4 * k + 1] + sums[4 * k + 2] + sums[4 * k + 3]) / (float)a.N + a.eps);
  };
  float r[2];
  if constexpr (YN) {
    norms(y, red, r);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < NC; ++i) y[k][i] = y[k][i] * r[k] * yw[i];
  }
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int i = 0; i < NC; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j) x[k][i][j] = fmaf(a.mult, y[k][i][j], IN == LEAN_JOIN ? x[k][i][j] : 0.f);
      if (k == 0) st4(a.x_out + (size_t)m * a.ldx + c + 1024 * i, x[k][i]);
    }
  norms(x, red + 8, r);
  const bool keeps = first && a.sh_last[last] == last;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
#pragma clang fp contract(off)  // h is rounded before it is taken from the row before, as there
    const f32x4 h = x[0][i] * r[0] * nw[i], o = x[1][i] * r[1] * nw[i], p = first || m == 0 ? prev[i] : o;
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = fmaf(p[j] - h[j], mu[i][j], h[j]);
    st4((bf16_t*)a.h + (size_t)m * a.ldh + c + 1024 * i, v);
    if (keeps) st4(state + 1024 * i, last == m ? h : o);
  }
}

// 1: not one of these forms.
template <int NC>
static int shift_launch(const RowsArgs& a, hipStream_t st) {
  if (a.y == nullptr || a.x_out == nullptr || a.copy != nullptr || a.xidx != nullptr) return 1;
#define SHIFT(IN, YN)                                                                       \
  {                                                                                         \
    hipLaunchKernelGGL((rows_shift_kernel<NC, IN, YN>), dim3(a.M), dim3(256), 0, st, a);     \
    return (int)hipGetLastError();                                                          \
  }
  if (a.x_in == nullptr) {
    if (a.y_w != nullptr) return 1;
    SHIFT(LEAN_TABLE, false)
  }
  if (a.yidx != nullptr) return 1;
  if (a.y_w != nullptr) SHIFT(LEAN_JOIN, true)
  SHIFT(LEAN_JOIN, false)
#undef SHIFT
}

constexpr int ROWS_GRID = 2048;  // workgroups of a launch of many rows: they loop, eight to a CU

template <typename YT, typename OT, int PART>
static int rows_launch(const RowsArgs& a, hipStream_t st) {
  const int groups = PART == ROWS_SHIFT ? (a.M + a.sh_rows - 1) / a.sh_rows : a.M, cap = PART == ROWS_SHIFT ? groups : ROWS_GRID;
#define ROWS(TPR, NC)                                                                                             \
  {                                                                                                               \
    hipLaunchKernelGGL((rows_update_kernel<YT, OT, TPR, NC, PART>),                                               \
                       dim3(std::min((groups + 256 / TPR - 1) / (256 / TPR), cap)), dim3(256), 0, st, a);         \
    return (int)hipGetLastError();                                                                                \
  }
  // few rows (decode): a workgroup per row, so a row is one round trip deep
  if (a.M > 256) {
    if (a.NP <= 512) ROWS(64, 2)
    if (a.NP <= 1024) ROWS(64, 4)
  }
  if (a.NP <= 1024) ROWS(256, 1)
  if (a.NP <= 2048) ROWS(256, 2)
  if (a.NP <= 4096) ROWS(256, 4)
  if (a.NP <= 8192) ROWS(256, 8)
  if (a.NP <= 16384) ROWS(256, 16)
#undef ROWS
  return -1;
}

// fp32 gated activation of packed gate|up columns (8 gate, 8 up, ...): out = act(gate) * up.
__global__ __launch_bounds__(256) void glu_f32_kernel(const float* __restrict__ gu, int ldi, float* __restrict__ out,
                                                      int ldo, int M, int F, int act, GluClamp clamp) {
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i >= (long)M * F) return;
  const int m = (int)(i / F), c = (int)(i % F);
  const float* p = gu + (size_t)m * ldi + (c >> 3) * 16 + (c & 7);
  const float x = p[0];
  if (act == ACT_CLAMP_MUL) {
    const float g = fminf(x, clamp.limit), u = fminf(fmaxf(p[8], -clamp.limit), clamp.limit);
    out[(size_t)m * ldo + c] = g / (1.0f + expf(-clamp.alpha * g)) * (u + clamp.shift);
    return;
  }
  const float g = act == ACT_SILU_MUL ? x / (1.0f + expf(-x))
                                      : 0.5f * x * (1.0f + tanhf(0.797884560802865f * (x + 0.044715f * x * x * x)));
  out[(size_t)m * ldo + c] = g * p[8];
}

// Rows of z as the activation leaves them (gemm_epilogue.h), in fp32; c: its two constants.
__global__ __launch_bounds__(256) void xielu_f32_kernel(float* __restrict__ z, int ld, int M, int n,
                                                        const float* __restrict__ c) {
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i >= (long)M * n) return;
  float* p = z + (size_t)(i / n) * ld + i % n;
  const float v = *p;
  *p = fmaf(0.5f, v, v > 0.f ? c[0] * v * v : c[1] * (expm1f(v) - v));
}

}  // namespace dnn

using namespace dnn;

extern "C" int dnn_rows_update(const RowsArgs* a, int y_f32, int out_f32, hipStream_t st) {
  if (a->M <= 0 || a->N <= 0 || a->N > a->NP || a->NP % 4 != 0 || (a->ldx | a->ldy | a->ldcopy | a->ldh) % 4 != 0)
    return -1;
  if ((a->ldadd | a->ldy2 | a->ldys) % 4 != 0 || (a->y2 != nullptr && (a->y2_w == nullptr || a->y_w == nullptr)) ||
      (a->ys != nullptr && (a->ysi == nullptr || a->ysw == nullptr || a->top < 1 || a->ysrows < 1)) ||
      (a->y_joined && (a->ys == nullptr || a->y_w == nullptr)) ||
      (a->freq != nullptr && a->pos == nullptr))
    return -1;
  if ((a->xidx != nullptr && (a->xrows < 1 || a->x_out != nullptr)) || (a->yidx != nullptr && a->yrows < 1)) return -1;
  if (a->y2 != nullptr && (a->ys != nullptr || a->freq != nullptr)) return -1;
  if (a->ys != nullptr && a->freq != nullptr) return -1;
  if (a->sh_mu != nullptr &&
      (a->n_w == nullptr || a->n_b != nullptr || a->y2 != nullptr || a->ys != nullptr || a->freq != nullptr || a->x_add != nullptr ||
       a->sh_state == nullptr || a->sh_start == nullptr || a->sh_last == nullptr || a->sh_slots == nullptr || a->sh_pos == nullptr ||
       a->sh_nslots < 1 || a->sh_rows < 1 || (a->x_out != nullptr && a->x_out == a->x_in)))
    return -1;
  const bool more = a->x_add != nullptr || a->n_b != nullptr;
#define ROWS_PART(YT, OT)                                                                        \
  {                                                                                              \
    if (a->y2 != nullptr) return rows_launch<YT, OT, ROWS_TWO>(*a, st);                          \
    if (a->ys != nullptr) return rows_launch<YT, OT, ROWS_EXPERTS>(*a, st);                      \
    if (a->freq != nullptr) return rows_launch<YT, OT, ROWS_POSITIONS>(*a, st);                  \
    if (a->sh_mu != nullptr) return rows_launch<YT, OT, ROWS_SHIFT>(*a, st);                     \
    return more ? rows_launch<YT, OT, ROWS_MORE>(*a, st) : rows_launch<YT, OT, ROWS_PLAIN>(*a, st); \
  }
  if (y_f32 && out_f32) ROWS_PART(float, float)
  // Up to as many rows as workgroups are in flight at once: past that the general kernel keeps the norms' weights
  // over a workgroup's rows.
  if (!y_f32 && !out_f32 && !more && a->y2 == nullptr && a->ys == nullptr && a->freq == nullptr && a->M <= ROWS_GRID) {
    const bool shift = a->sh_mu != nullptr;
    const int rc = a->NP == 1024   ? shift ? shift_launch<1>(*a, st) : lean_launch<1>(*a, st)
                   : a->NP == 2048 ? shift ? shift_launch<2>(*a, st) : lean_launch<2>(*a, st)
                   : a->NP == 4096 ? shift ? shift_launch<4>(*a, st) : lean_launch<4>(*a, st)
                                   : 1;
    if (rc <= 0) return rc;
  }
  if (!y_f32 && !out_f32) ROWS_PART(bf16_t, bf16_t)
#undef ROWS_PART
  if (!y_f32 || a->y2 != nullptr || a->ys != nullptr || a->freq != nullptr || a->sh_mu != nullptr || more) return -1;
  return rows_launch<float, bf16_t, ROWS_PLAIN>(*a, st);
}

extern "C" int dnn_glu_f32(const float* gu, int ldi, float* out, int ldo, int M, int F, int act,
                           const GluClamp* clamp, hipStream_t st) {
  if (M <= 0 || F <= 0 || F % 8 != 0 || ldi < 2 * F || ldo < F || !is_glu(act) || (act == ACT_CLAMP_MUL && clamp == nullptr)) return -1;
  hipLaunchKernelGGL(glu_f32_kernel, dim3((unsigned)(((long)M * F + 255) / 256)), dim3(256), 0, st, gu, ldi, out, ldo,
                     M, F, act, clamp != nullptr ? *clamp : GluClamp{});
  return (int)hipGetLastError();
}

extern "C" int dnn_xielu_f32(float* z, int ld, int M, int n, const float* c, hipStream_t st) {
  if (M <= 0 || n <= 0 || ld < n || c == nullptr) return -1;
  hipLaunchKernelGGL(xielu_f32_kernel, dim3((unsigned)(((long)M * n + 255) / 256)), dim3(256), 0, st, z, ld, M, n, c);
  return (int)hipGetLastError();
}
