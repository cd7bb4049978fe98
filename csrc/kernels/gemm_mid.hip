// bf16 GEMM for 65 to a few thousand rows: the choice of tile and K split, and
// the launches (kernels: gemm_mid.h).
#include "gemm_mid.h"

namespace dnn {

// Tile table: rows, columns, whether two workgroups share a CU, and the constants of a
// tile's time in us: a (launch, first loads, epilogue), s (a K-tile of 64) and p (of s, where K is
// split: no epilogue, and waves that only stage), fitted to 1174 shapes (64 x 64
// with four K-tiles in flight).  As the kernels run now, over 589 other shapes (66 to 9400 rows, 768 to
// 28672 columns, K of 768 to 21504, weights cold), every tile with 1 to 8 splits, the estimate is off by 10 % (rms);
// what it picks takes 1.1 % longer than the best measured on average, 0.2 % in the median, 14 % at worst (67 x 6144 x
// 4096 20.5, 18.0 as 96 x 128 in 4; profiles/gemm_mid_estimate.md).
struct MidCost {
  int bm, bn, pairs;
  float a, s, p;
};
static constexpr MidCost MID[] = {{64, 64, 1, 2.97f, 0.220f, 0.83f},    {128, 64, 0, 3.04f, 0.332f, 0.94f},
                                  {128, 128, 0, 3.18f, 0.454f, 1.03f},  {256, 128, 0, 4.14f, 0.747f, 0.88f},
                                  {128, 256, 0, 3.88f, 0.752f, 0.92f},  {192, 128, 0, 3.67f, 0.602f, 0.92f},
                                  {96, 128, 0, 3.67f, 0.446f, 0.89f}};
static constexpr MidCost MID_256 = {256, 256, 0, 6.33f, 1.172f, 1.f};
// The e4m3 kernels on the first five and as 256 x 256, whole
static constexpr MidCost MID8[] = {{64, 64, 1, 1.89f, 0.252f, 1.f},   {128, 64, 0, 2.78f, 0.332f, 1.f},
                                   {128, 128, 0, 2.99f, 0.472f, 1.f}, {256, 128, 0, 4.14f, 0.707f, 1.f},
                                   {128, 256, 0, 4.07f, 0.754f, 1.f}};
static constexpr MidCost MID8_256 = {256, 256, 0, 4.93f, 1.198f, 1.f};
static constexpr int CUS = 256;

// Bytes a microsecond: weights, activations in and out, parts of a split
struct MidRates {
  float w, x, part;
};
static constexpr MidRates RATES = {7.3e6f, 1.9e6f, 3.2e6f}, RATES8 = {4.27e6f, 2.0e6f, 3.16e6f};

// Time of one tile size and split: K-tiles of the fullest CU, beside the time that reading the
// weights and moving the activations takes; a split adds its sum (one more launch, and the
// parts written and read).
static float mid_time(const MidCost& c, const MidRates& r, int M, int N, int K, int splits) {
  const long long wgs = (long long)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * splits;
  const int kt = (K / 64 + splits - 1) / splits, n = (int)((wgs + CUS - 1) / CUS);
  const float rounds = c.pairs ? (n / 2) * 1.73f + (n & 1) : (float)n;
  const float a = c.pairs ? c.a : c.a * (1.f + 0.5f * (n - 1));
  const float t = rounds * kt * (splits > 1 ? c.s * c.p : c.s), w = (float)N * K * 2.f / r.w + (float)M * (K + N) * 2.f / r.x;
  const float us = a + cbrtf(t * t * t + w * w * w);
  return splits == 1 ? us : us + 4.12f + (splits + 0.5f) * M * N * 4.f / r.part;
}

// The best tile and split of M x N, at most `best`.
static MidPlan best_tile(int M, int N, int K, long long ws_bytes, unsigned kind, MidPlan best) {
  const bool mx = kind >= MID_MX;
  for (int i = 0; i < (mx ? 5 : 7); ++i) {
    if (kind == MID_MX_QUANT && MID8[i].bn < 128) continue;
    for (int s = 1; s <= 8; ++s) {
      if (s > 1 && (N % 4 != 0 || M > 65535 || K / 64 / s < 3 || (long long)s * M * N * 4 > ws_bytes)) break;
      const float t = mx ? mid_time(MID8[i], RATES8, M, N, K, s) : mid_time(MID[i], RATES, M, N, K, s);
      if (t < best.us) best = {i, s, t, 0};
    }
  }
  return best;
}

static MidPlan best_plan(int M, int N, int K, long long ws_bytes, unsigned kind) {
  // the 256 x 256 kernel needs to be 5 % slower to lose: the estimate's error at
  // its sizes (12352 columns of 3000 rows: 257 us, 267 as 256 x 128)
  const bool mx = kind >= MID_MX;
  const float whole = mx ? mid_time(MID8_256, RATES8, M, N, K, 1) : mid_time(MID_256, RATES, M, N, K, 1);
  MidPlan best = best_tile(M, N, K, ws_bytes, kind, {-1, 1, M < 256 || N < 256 ? 1e30f : 0.95f * whole, 0});
  // Full rounds of 256 x 256 tiles and the columns that are left on the tile that
  // suits them: a last round that fills a third of the chip costs a whole one.  us as
  // the best single tile and in two: 700 x 28672 x 4096 168 : 155, 1700 rows 356 : 320,
  // 2600 x 12352 x 4096 256 : 222, 2600 x 6400 x 1600 80 : 65.
  const long long ntm = (M + 255) / 256, tiles = ntm * ((N + 255) / 256);
  if (kind == MID_BF16 && M >= 256 && tiles > CUS && tiles % CUS != 0) {
    const int cols = (int)(tiles / CUS * CUS / ntm) * 256;
    if (cols > 0 && cols < N) {
      MidPlan two = best_tile(M, N - cols, K, ws_bytes, kind, {-1, 1, 1e30f, 0});
      two.us += mid_time(MID_256, RATES, M, cols, K, 1);
      two.cols = cols;
      if (two.us < 0.95f * best.us) best = two;
    }
  }
  return best;
}

// The same by sizes: some 50 estimates take 3 us of host time, a table entry (per thread)
// nothing beside a launch.
MidPlan mid_plan(int M, int N, int K, long long ws_bytes, unsigned kind) {
  struct Entry {
    int M = 0, N = 0, K = 0;
    unsigned kind = 0;
    long long ws = 0;
    MidPlan plan{};
  };
  static thread_local Entry table[256];
  Entry& e = table[((unsigned)M * 2654435761u ^ (unsigned)N * 40503u ^ (unsigned)K * 97u ^ kind * 77u) >> 7 & 255];
  if (e.M != M || e.N != N || e.K != K || e.kind != kind || e.ws != ws_bytes)
    e = {M, N, K, kind, ws_bytes, best_plan(M, N, K, ws_bytes, kind)};
  return e.plan;
}

// Decode kernels (gemm_skinny.hip) on more than 64 rows against the tiles.  They take 16 rows
// and 32 columns a workgroup (16 up to 1024 columns), which share a CU and add up: the
// time is that of the fullest CU, in steps.  `frag`: the weight has its fragment-order
// copy; without it a step costs 1.6 times as much.  A folded norm rides along for 1 us; the
// tiles need a launch that adds 3.3 (also counted where partials of the row statistics spare it).  us, decode kernels : tiles: 132 rows x 768 x 768 5.3 : 5.8, 192 6.6 : 5.9; row-
// major 70 4.8 : 5.3; 192 x 768 x 3072 row-major 19.4 : 12.1; 70 x 1600 x 1600 7.1 : 7.1, 85
// 9.0 : 8.5; 256 x 4096 x 4096 88 : 18; with a norm 128 x 3072 x 768 9.0 : 9.7, 146 10.4 : 9.8,
// 135 x 2304 x 768 8.6 : 9.2, 167 9.6 : 9.1, 128 x 2816 x 512 6.4 : 7.4, 189 8.1 : 7.6, 256 x 1536 x
// 512 6.4 : 7.1, 65 x 4800 x 1600 12.8 : 11.7.
bool mid_skinny(int M, int N, int K, bool norm, bool frag, long long ws_bytes) {
  if (M > 256) return false;
  const bool one = N <= 1024;
  const int n = ((M + 15) / 16 * ((N + (one ? 15 : 31)) / (one ? 16 : 32)) + 255) / 256;
  const float base = one ? 2.9f + 0.0002f * K : 3.6f + 0.0006f * K;
  const float step = frag ? (one ? 0.45f + 0.0009f * K : 0.15f + 0.00152f * K)
                          : (one ? 0.4f + 0.0016f * K : 0.2f + 0.0025f * K);
  return base + n * step + (norm ? 1.f : 0.f) <
         mid_plan(M, N, K, ws_bytes, MID_BF16).us + (norm ? 3.3f : 0.f);
}

template <class T>
static int launch(const MidArgs& a, const QkvScatter* scat, hipStream_t st) {
#ifndef DNN_DECODER_ONLY
  if (a.parts != nullptr) {
    if (a.splits != 1) return -1;
    return scat != nullptr ? mid_start<T, MID_SCATTER, true>(a, *scat, st) : mid_start<T, MID_ROWS, true>(a, QkvScatter{}, st);
  }
#endif
#ifndef DNN_DECODER_ONLY
  if (scat != nullptr && scat->cosT != nullptr) {
    if constexpr (T::BN % 128 == 0) return mid_start<T, MID_ROPE>(a, *scat, st);
    return -1;
  }
#endif
  if (scat != nullptr) return mid_start<T, MID_SCATTER>(a, *scat, st);
  if (a.splits == 1) return mid_start<T, MID_ROWS>(a, QkvScatter{}, st);
  if (const int rc = mid_start<typename MidSplit<T>::type, MID_PART>(a, QkvScatter{}, st)) return rc;
  const bool glu = is_glu(a.act);
  const dim3 grid(((glu ? a.N / 2 : a.N) / 4 + 255) / 256, a.M);
  if (glu) hipLaunchKernelGGL((gemm_mid_reduce<1>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((gemm_mid_reduce<0>), grid, dim3(256), 0, st, a);
  return (int)hipGetLastError();
}

template <class T>
static int blocks() {
  int n = 0;
  const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void*)gemm_mid_kernel<T, MID_ROWS, false>,
                                                                    T::THREADS, T::S * T::STAGE);
  return e == hipSuccess ? n : -1;
}

int mid_blocks(int tile) {
  switch (tile) {
    case 0: return blocks<Mid0>();
    case 1: return blocks<Mid1>();
    case 2: return blocks<Mid2>();
    case 3: return blocks<Mid3>();
    case 4: return blocks<Mid4>();
    case 5: return blocks<Mid5>();
    case 6: return blocks<Mid6>();
  }
  return -1;
}

int mid_launch(int tile, const MidArgs& a, const QkvScatter* scat, hipStream_t st) {
  if (a.splits < 1 || (a.splits > 1 && (scat != nullptr || a.part == nullptr || a.N % 4 != 0 || a.K / 64 < a.splits ||
                                        a.M > 65535)))
    return -1;
  if (scat == nullptr && a.splits == 1) {
    if (const int rc = mid_plain_launch(tile, a, st); rc != -3) return rc;
  }
  switch (tile) {
    case 0: return launch<Mid0>(a, scat, st);
    case 1: return launch<Mid1>(a, scat, st);
    case 2: return launch<Mid2>(a, scat, st);
    case 3: return launch<Mid3>(a, scat, st);
    case 4: return launch<Mid4>(a, scat, st);
    case 5: return launch<Mid5>(a, scat, st);
    case 6: return launch<Mid6>(a, scat, st);
  }
  return -1;
}

}  // namespace dnn
