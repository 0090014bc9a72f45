// Products of the fp32 attention kernels on v_mfma_f32_32x32x2_f32 (described in attn_f32.hip).
#pragma once
#include "attn_params.h"
#include "attn_tile.h"

namespace f32tile {

constexpr int F_TILE = 32;            // rows of the streamed side per LDS tile
constexpr float LN2 = 0.6931471805599453f;

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// row of a 32-row tile that result register r of a lane in half g holds
__device__ __forceinline__ int acc_row(int r, int g) { return 8 * (r >> 2) + 4 * g + (r & 3); }

// One 32-row tile of a (rows, D) fp32 matrix on its way from global memory to LDS, brought by NT threads: 8 D / NT
// 16-byte pieces per thread, rows past `nvalid` read as zero.
template <int D, int NT>
struct TileRegs {
  static constexpr int N = 8 * D / NT, LD = D + 4;
  f32x4 v[N];
  __device__ __forceinline__ void fetch(const float* src, int64_t stride, int row0, int nvalid, int tid) {
#pragma unroll
    for (int c = 0; c < N; c++) {
      const int e = tid + c * NT, r = e / (D / 4), x = e % (D / 4);
      v[c] = (r < nvalid) ? *reinterpret_cast<const f32x4*>(src + (int64_t)(row0 + r) * stride + 4 * x)
                          : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  __device__ __forceinline__ void put(float* dst, int tid) const {
#pragma unroll
    for (int c = 0; c < N; c++) {
      const int e = tid + c * NT, r = e / (D / 4), x = e % (D / 4);
      *reinterpret_cast<f32x4*>(dst + r * LD + 4 * x) = v[c];
    }
  }
};

// The resident operand of a head_dim contraction: row `row` of a (rows, D) matrix in
// k-step order (element 4 j + t = column 8 j + 4 g + t), times `mul`.
template <int D>
__device__ __forceinline__ void load_row_frag(float (&f)[D / 2], const float* base, int64_t stride, int row, bool ok,
                                              int g, float mul) {
#pragma unroll
  for (int j = 0; j < D / 8; j++) {
    const f32x4 v = ok ? *reinterpret_cast<const f32x4*>(base + (int64_t)row * stride + 8 * j + 4 * g)
                       : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; t++) f[4 * j + t] = v[t] * mul;
  }
}

// acc (+)= T F^T for a 32-row LDS tile T (rows = MFMA rows) and a resident fragment F;
// two accumulation chains, summed by the caller.
template <int D>
__device__ __forceinline__ void tile_times_frag(const float* tile, int i, int g, const float (&f)[D / 2], f32x16& c0,
                                                f32x16& c1) {
  constexpr int LD = D + 4;
#pragma unroll
  for (int j = 0; j < D / 8; j++) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(tile + i * LD + 8 * j + 4 * g);
#pragma unroll
    for (int t = 0; t < 4; t++) {
      if (j & 1) c1 = mfma_f32(a[t], f[4 * j + t], c1);
      else c0 = mfma_f32(a[t], f[4 * j + t], c0);
    }
  }
}

// Two products of that kind at once, interleaved: each is the other's independent chain.
template <int D>
__device__ __forceinline__ void tiles_times_frags(const float* ta, const float (&fa)[D / 2], f32x16& ca, const float* tb,
                                                  const float (&fb)[D / 2], f32x16& cb, int i, int g) {
  constexpr int LD = D + 4;
#pragma unroll
  for (int j = 0; j < D / 8; j++) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(ta + i * LD + 8 * j + 4 * g);
    const f32x4 b = *reinterpret_cast<const f32x4*>(tb + i * LD + 8 * j + 4 * g);
#pragma unroll
    for (int t = 0; t < 4; t++) {
      ca = mfma_f32(a[t], fa[4 * j + t], ca);
      cb = mfma_f32(b[t], fb[4 * j + t], cb);
    }
  }
}

// acc[db] += T^T W for a 32-row LDS tile T (its 32 rows are contracted) and the weights
// W held in result-register order; D / 32 independent chains.
template <int D>
__device__ __forceinline__ void tile_t_times_regs(const float* tile, int i, int g, const f32x16& w,
                                                  f32x16 (&acc)[D / 32]) {
  constexpr int LD = D + 4;
#pragma unroll
  for (int ks = 0; ks < 16; ks++) {
    const float* row = tile + acc_row(ks, g) * LD + i;
#pragma unroll
    for (int db = 0; db < D / 32; db++) acc[db] = mfma_f32(row[32 * db], w[ks], acc[db]);
  }
}

// acc[db][r] is element (row i of the owner, column 32 db + 8 (r / 4) + 4 g + r % 4):
// four consecutive columns per register quad -> one 16-byte store each.
template <int D>
__device__ __forceinline__ void store_rows(float* dst, const f32x16 (&acc)[D / 32], int g, float mul, bool add) {
#pragma unroll
  for (int db = 0; db < D / 32; db++)
#pragma unroll
    for (int a = 0; a < 4; a++) {
      f32x4* out = reinterpret_cast<f32x4*>(dst + 32 * db + 8 * a + 4 * g);
      f32x4 v{acc[db][4 * a] * mul, acc[db][4 * a + 1] * mul, acc[db][4 * a + 2] * mul, acc[db][4 * a + 3] * mul};
      if (add) v += *out;
      *out = v;
    }
}

}  // namespace f32tile
