// Tile kernels of the NT product (forward: both operands contiguous along K).
#include "gemm_tile.h"

namespace {
using namespace gemm_tile;

template <int BM, int BN>
int with_tile(int epi, int splits, const Args& a, hipStream_t st) {
  if (epi == EPI_SWIGLU_FWD) return launch<true, true, BM, BN, false, EPI_SWIGLU_FWD>("gemm_bf16_nt_swiglu", a, 1, st);
  if (epi == EPI_ROPE) return launch<true, true, BM, BN, false, EPI_ROPE>("gemm_bf16_nt_rope", a, 1, st);
  if (splits > 1) return launch<true, true, BM, BN, true, EPI_NONE>("gemm_bf16_nt", a, splits, st);
  return launch<true, true, BM, BN, false, EPI_NONE>(a.add && a.add != a.C && a.K % BK == 0 ? "gemm_bf16_nt_residual" : "gemm_bf16_nt", a, 1, st);
}
}  // namespace

int ody_launch_gemm_nt(int epi, int BM, int BN, int splits, const gemm_tile::Args& a, hipStream_t st) {
  if (BM == 256 && BN == 256) return with_tile<256, 256>(epi, splits, a, st);
  if (BM == 128 && BN == 256) return with_tile<128, 256>(epi, splits, a, st);
  return with_tile<128, 128>(epi, splits, a, st);
}
