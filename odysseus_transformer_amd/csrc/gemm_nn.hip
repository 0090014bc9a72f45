// Tile kernels of the NN product (input gradient: A contiguous along K, B along N).
#include "gemm_tile.h"

namespace {
using namespace gemm_tile;

template <int BM, int BN>
int with_tile(int epi, int splits, const Args& a, hipStream_t st) {
  if (epi == EPI_SWIGLU_BWD) return launch<true, false, BM, BN, false, EPI_SWIGLU_BWD>("gemm_bf16_nn_swiglu_bwd", a, 1, st);
  if (splits > 1) return launch<true, false, BM, BN, true, EPI_NONE>("gemm_bf16_nn", a, splits, st);
  return launch<true, false, BM, BN, false, EPI_NONE>("gemm_bf16_nn", a, 1, st);
}
}  // namespace

int ody_launch_gemm_nn(int epi, int BM, int BN, int splits, const gemm_tile::Args& a, hipStream_t st) {
  if (BM == 256 && BN == 256) return with_tile<256, 256>(epi, splits, a, st);
  if (BM == 128 && BN == 256) return with_tile<128, 256>(epi, splits, a, st);
  return with_tile<128, 128>(epi, splits, a, st);
}
