// The tiles of gemm_mid.h with one epilogue each: what a transformer block's projections need.
//
// The kernel for every epilogue is 17 to 60 KB; a launch begins with a cold instruction cache, and the way through
// branches that were not taken is fetched with the one that is.  One epilogue is 2 to 12.  us a launch in a pass: 1071 x
// 768 of K = 768 and 3072 with residual and statistics (64 x 64, 17 -> 3.2 KB) 11.0 -> 10.2 on average, 1071 x 3072 x 768
// with norm and GELU (128 x 128, 30 -> 7.4 KB) 14.1 -> 13.6, 700 x 4096 x 4096 with residual (96 x 128, 47 -> 4.4 KB) 34.4 ->
// 32.7, 700 x 6144 x 4096 with norm (192 x 128, 46 -> 3.6 KB) 46.4 -> 44.7.
#include "gemm_mid.h"

namespace dnn {

// The epilogue of `a` for waves of `cols` columns, MID_ANY where it is not one of the plain ones.
static int mid_epi(const MidArgs& a, int cols) {
  const bool stat = a.rowstat != nullptr || a.parts != nullptr, glu = is_glu(a.act);
  if (!mid_plain_ok(a, cols, a.colsum) || (a.colsum != nullptr && !stat) || (a.parts_out != nullptr && a.R == nullptr) ||
      (glu && (a.bias != nullptr || a.R != nullptr)))
    return MID_ANY;
  return a.act | (a.R != nullptr ? MID_RES : 0) | (stat ? MID_STAT : 0) | (a.colsum != nullptr ? MID_COLS : 0) |
         (a.bias != nullptr ? MID_BIAS : 0) | (a.parts_out != nullptr ? MID_STATS_OUT : 0);
}

template <class T>
static int plain(const MidArgs& a, hipStream_t st) {
  const int epi = mid_epi(a, T::J * 16);
#define EPI(E)                                                                           \
  if (epi == (E) && a.parts == nullptr) return mid_start<T, MID_ROWS, false, (E)>(a, QkvScatter{}, st);
  EPI(ACT_NONE)
  EPI(ACT_NONE | MID_BIAS)
  EPI(ACT_XIELU | MID_BIAS)
  EPI(ACT_GELU_TANH_MUL)
#ifndef DNN_DECODER_ONLY
  EPI(ACT_NONE | MID_RES)
  EPI(ACT_NONE | MID_RES | MID_BIAS)
  EPI(ACT_NONE | MID_RES | MID_BIAS | MID_STATS_OUT)
  EPI(ACT_NONE | MID_STAT)
  EPI(ACT_SILU_MUL | MID_STAT)
  constexpr int FC = ACT_GELU | MID_STAT | MID_COLS | MID_BIAS;
  EPI(FC)
  if (epi == FC) return mid_start<T, MID_ROWS, true, FC>(a, QkvScatter{}, st);
#endif
#undef EPI
  return -3;
}

int mid_plain_launch(int tile, const MidArgs& a, hipStream_t st) {
  switch (tile) {
    case 0: return plain<Mid0>(a, st);
    case 1: return plain<Mid1>(a, st);
    case 2: return plain<Mid2>(a, st);
    case 3: return plain<Mid3>(a, st);
    case 4: return plain<Mid4>(a, st);
    case 5: return plain<Mid5>(a, st);
    case 6: return plain<Mid6>(a, st);
  }
  return -3;
}

}  // namespace dnn
