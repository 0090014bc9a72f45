// Tile kernels of the TN product (weight gradient: A contiguous along M, B along N).
#include "gemm_tile.h"

namespace {
using namespace gemm_tile;

template <int BM, int BN>
int with_tile(int splits, const Args& a, hipStream_t st) {
  if (splits > 1) return launch<false, false, BM, BN, true, EPI_NONE>("gemm_bf16_tn", a, splits, st);
  return launch<false, false, BM, BN, false, EPI_NONE>("gemm_bf16_tn", a, 1, st);
}
}  // namespace

int ody_launch_gemm_tn(int BM, int BN, int splits, const gemm_tile::Args& a, hipStream_t st) {
  if (BM == 256 && BN == 256) return with_tile<256, 256>(splits, a, st);
  if (BM == 128 && BN == 256) return with_tile<128, 256>(splits, a, st);
  return with_tile<128, 128>(splits, a, st);
}
