// Dense linears: C (M, N) = op(A) . op(B) for the three products of a linear
// layer (forward NT, dgrad NN, wgrad TN): the choice of a kernel and a plan, and the entry points.
//
// bf16 products run on gemm_tile.h (LDS tiles) or gemm_skinny.hip (few rows); the small kernel below only takes matrices whose
// row pitch does not fit those kernels' 32-bit tile offsets.  fp32 products: gemm_f32.hip.
#include <algorithm>
#include "gemm_tile.h"

namespace {

// ------------------------------------------------------------------ bf16, any pitch
constexpr int BK = 64;

// Operand tile in LDS.  KC = true: memory is (rows, K) row-major -> [ROWS][BK+8].
//                       KC = false: memory is (K, rows) row-major -> [BK][ROWS+32].
template <int ROWS, bool KC>
struct OperandTile {
  static constexpr int PITCH = KC ? (BK + 8) : (ROWS + 32);
  static constexpr int ELEMS = KC ? ROWS * PITCH : BK * PITCH;
  static constexpr int CHUNKS = ROWS * BK / 8 / 256;  // 16-byte chunks per thread
  bf16x8 r[CHUNKS];

  // row0: first row (M or N index) of the tile; k0: first K index
  __device__ __forceinline__ void gload(const bf16* base, int64_t ld, int row0, int k0, int nrows, int K, int tid) {
#pragma unroll
    for (int j = 0; j < CHUNKS; j++) {
      const int c = tid + 256 * j;
      int rr, kk;
      if (KC) { rr = c / (BK / 8); kk = (c % (BK / 8)) * 8; }
      else { kk = c / (ROWS / 8); rr = (c % (ROWS / 8)) * 8; }
      const int gr = row0 + rr, gk = k0 + kk;
      bool ok;
      const bf16* src;
      if (KC) { ok = gr < nrows && gk < K; src = base + (int64_t)gr * ld + gk; }   // K % 8 == 0: chunk all in or out
      else { ok = gk < K && gr < nrows; src = base + (int64_t)gk * ld + gr; }      // rows % 8 == 0 likewise
      r[j] = ok ? *reinterpret_cast<const bf16x8*>(src) : bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  __device__ __forceinline__ void sstore(bf16* lds, int tid) const {
#pragma unroll
    for (int j = 0; j < CHUNKS; j++) {
      const int c = tid + 256 * j;
      int rr, kk;
      if (KC) { rr = c / (BK / 8); kk = (c % (BK / 8)) * 8; *reinterpret_cast<bf16x8*>(lds + rr * PITCH + kk) = r[j]; }
      else { kk = c / (ROWS / 8); rr = (c % (ROWS / 8)) * 8; *reinterpret_cast<bf16x8*>(lds + kk * PITCH + rr) = r[j]; }
    }
  }
  // MFMA operand for tile rows [r32, r32+32), k-step ks (16 K values): lane (g, i) gets row r32+i, k = 16ks+8g..+7
  __device__ static __forceinline__ bf16x8 frag(const bf16* lds, int r32, int ks, int g, int i) {
    if (KC) {
      return *reinterpret_cast<const bf16x8*>(lds + (r32 + i) * PITCH + 16 * ks + 8 * g);
    } else {
      const bf16* p = lds + (16 * ks + 8 * g + ((i & 15) >> 2)) * PITCH + r32 + 16 * (i >> 4) + 4 * (i & 3);
      return concat4(lds_read_tr16(p), lds_read_tr16(p + 4 * PITCH));
    }
  }
};

// 64 WM x 64 WN tiles, 4 wavefronts in a 2 x 2 arrangement; operands are staged through registers and LDS in K-slabs of 64.
template <int WM, int WN, bool A_KC, bool B_KC>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(const bf16* __restrict__ A, const bf16* __restrict__ B,
                                                        bf16* __restrict__ C, const bf16* __restrict__ bias, int M,
                                                        int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
                                                        int accumulate, int tiles_m, int tiles_n) {
  constexpr int TM = 64 * WM, TN = 64 * WN;  // block tile
  typedef OperandTile<TM, A_KC> TA;
  typedef OperandTile<TN, B_KC> TB;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  bf16* As = reinterpret_cast<bf16*>(smem_raw);  // [2][TA::ELEMS]
  bf16* Bs = As + 2 * TA::ELEMS;                 // [2][TB::ELEMS]

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int wm = wave >> 1, wn = wave & 1;

  // Block -> tile.  Consecutive workgroup ids go round-robin over the 8 XCDs, each
  // with its own L2: give every XCD a contiguous range of tiles, and inside the
  // range walk down M in groups so that neighbours share the B panel.
  int pid = blockIdx.x;
  const int nblk = tiles_m * tiles_n;
  if (nblk % 8 == 0) pid = (pid % 8) * (nblk / 8) + pid / 8;
  constexpr int GROUP = 8;
  const int per_group = GROUP * tiles_n;
  const int gid = pid / per_group, first_m = gid * GROUP;
  const int gsz = min(tiles_m - first_m, GROUP);
  const int tm = first_m + (pid % per_group) % gsz, tn = (pid % per_group) / gsz;
  const int m0 = tm * TM, n0 = tn * TN;

  f32x16 acc[WM][WN];
#pragma unroll
  for (int a = 0; a < WM; a++)
#pragma unroll
    for (int b = 0; b < WN; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[a][b][r] = 0.f;

  TA ta;
  TB tb;
  const int nk = (K + BK - 1) / BK;
  ta.gload(A, lda, m0, 0, M, K, tid);
  tb.gload(B, ldb, n0, 0, N, K, tid);
  ta.sstore(As, tid);
  tb.sstore(Bs, tid);
  __syncthreads();

  for (int kt = 0; kt < nk; kt++) {
    const int buf = kt & 1;
    if (kt + 1 < nk) {
      ta.gload(A, lda, m0, (kt + 1) * BK, M, K, tid);
      tb.gload(B, ldb, n0, (kt + 1) * BK, N, K, tid);
    }
    const bf16* Ab = As + buf * TA::ELEMS;
    const bf16* Bb = Bs + buf * TB::ELEMS;
#pragma unroll
    for (int ks = 0; ks < BK / 16; ks++) {
      bf16x8 af[WM], bfr[WN];
#pragma unroll
      for (int a = 0; a < WM; a++) af[a] = TA::frag(Ab, 32 * (wm * WM + a), ks, g, i);
#pragma unroll
      for (int b = 0; b < WN; b++) bfr[b] = TB::frag(Bb, 32 * (wn * WN + b), ks, g, i);
#pragma unroll
      for (int a = 0; a < WM; a++)
#pragma unroll
        for (int b = 0; b < WN; b++) acc[a][b] = mfma32(bfr[b], af[a], acc[a][b]);  // rows = n, cols = m
    }
    if (kt + 1 < nk) {
      ta.sstore(As + (buf ^ 1) * TA::ELEMS, tid);
      tb.sstore(Bs + (buf ^ 1) * TB::ELEMS, tid);
    }
    __syncthreads();
  }

  // epilogue: lane (g, i) holds column m = i, rows n = 8*(r/4) + 4g + r%4
#pragma unroll
  for (int a = 0; a < WM; a++) {
    const int m = m0 + 32 * (wm * WM + a) + i;
    if (m >= M) continue;
#pragma unroll
    for (int b = 0; b < WN; b++) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int n = n0 + 32 * (wn * WN + b) + 8 * q + 4 * g;
        if (n >= N) continue;  // N % 8 == 0: a quad is all in or all out
        bf16* dst = C + (int64_t)m * ldc + n;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = acc[a][b][4 * q + e];
        if (bias) {
          const bf16x4 bv = *reinterpret_cast<const bf16x4*>(bias + n);
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] += (float)bv[e];
        }
        if (accumulate) {
          const bf16x4 old = *reinterpret_cast<const bf16x4*>(dst);
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] += (float)old[e];
        }
        bf16x4 w;
#pragma unroll
        for (int e = 0; e < 4; e++) w[e] = (bf16)v[e];
        *reinterpret_cast<bf16x4*>(dst) = w;
      }
    }
  }
}

__device__ __forceinline__ f32x4 sum_parts(const float* part, int splits, int64_t plane, int64_t at) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < splits; s++) v += *reinterpret_cast<const f32x4*>(part + s * plane + at);
  return v;
}
__device__ __forceinline__ void store_rounded(bf16* dst, f32x4 v) {
  bf16x4 w;
#pragma unroll
  for (int e = 0; e < 4; e++) w[e] = (bf16)v[e];
  *reinterpret_cast<bf16x4*>(dst) = w;
}

// C = sum over the K ranges of the fp32 partial tiles (+ bias, + add), rounded once; 4 elements per thread
__global__ __launch_bounds__(256) void gemm_splitk_sum_kernel(const float* __restrict__ part, int splits, bf16* C,
                                                              const bf16* __restrict__ bias, const bf16* add, int M, int N,
                                                              int64_t ldc, int64_t ld_add) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x, total = (int64_t)M * (N / 4);
  if (idx >= total) return;
  const int m = idx / (N / 4), n = (idx % (N / 4)) * 4;
  f32x4 v = sum_parts(part, splits, (int64_t)M * N, (int64_t)m * N + n);
  if (bias) {
    const bf16x4 bv = *reinterpret_cast<const bf16x4*>(bias + n);
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] += (float)bv[e];
  }
  if (add) {
    const bf16x4 old = *reinterpret_cast<const bf16x4*>(add + (int64_t)m * ld_add + n);
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] += (float)old[e];
  }
  store_rounded(C + (int64_t)m * ldc + n, v);
}

// The same for the rotary epilogue: a thread owns columns j .. j + 3 and j + 64 .. j + 67 of a head
__global__ __launch_bounds__(256) void gemm_splitk_rope_kernel(const float* __restrict__ part, int splits, bf16* __restrict__ C,
                                                               GemmEpi ep, int M, int N, int64_t ldc) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int per_row = N / 8;
  if (idx >= (int64_t)M * per_row) return;
  const int m = idx / per_row, k = idx % per_row, j = 4 * (k & 15), n = 128 * (k >> 4) + j;
  const f32x4 x1 = sum_parts(part, splits, (int64_t)M * N, (int64_t)m * N + n), x2 = sum_parts(part, splits, (int64_t)M * N, (int64_t)m * N + n + 64);
  f32x4 o1 = x1, o2 = x2;
  if (n < ep.I) {
    const bf16x8 cs = *reinterpret_cast<const bf16x8*>(ep.aux + (int64_t)m * ep.ld_aux + 2 * j);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float co = (float)cs[2 * e], sn = (float)cs[2 * e + 1];
      o1[e] = x1[e] * co - x2[e] * sn;
      o2[e] = x2[e] * co + x1[e] * sn;
    }
  }
  store_rounded(C + (int64_t)m * ldc + n, o1);
  store_rounded(C + (int64_t)m * ldc + n + 64, o2);
}

// Tile and number of K ranges of a product, by the time that the candidates were measured to take: us per slab of 64 k and round
// of blocks, for a round that fills the 256 compute units and (linearly down to) one that leaves most of them idle, when the
// clock is higher and memory less busy; two blocks of 128 x 128 share a compute unit.  Cutting K costs the fp32 partial tiles a
// trip through memory.  The larger tile wins wherever it fills its rounds (8192^3, NT: 1450 TFLOP/s with 256 x 256, 1295 with
// 128 x 256, 1200 with 128 x 128); with 1000 rows, for instance, 4096 x 11008 takes 156 us on its 64 tiles of 256 x 256, 99 us
// on 256 tiles of 128 x 128 and 84 us on 128 tiles of 128 x 256 with K in two ranges.
//
// Where a last round of 256 x 256 tiles would leave more than half of the units idle, its tiles are worked on as two half or four
// quarter tiles each, by other blocks of the same launch: a round of halves takes 0.58 of a whole one, of quarters 0.44 (0.27 where
// they are few).  (Same sums in the same order: the result does not depend on it.)  Same box, us whole / halves: QKV of 3001 tokens (288
// tiles) 183 / 150, gate_up of 1000 tokens (344) 183 / 161, of 3001 (1032) 484 / 453, four weight gradients over 1000 tokens 394 / 371.
// Halves / quarters: QKV of 3001 tokens 141 / 136, gate_up of 2100 (774) 333 / 325, of 3001 428 / 421, its input gradient of 5000 (320)
// 778 / 745.
//
// Twelve or sixteen ranges of K, of 40 slabs each or more, where every block then has a unit of its own (the model above knows no memory, which is
// what such products wait for) and eight ranges leave a third of the units idle (fewer than 24 quarter tiles) or read a matrix of few rows or columns
// twice over (more than 32).  us, eight / up to sixteen ranges, NN: 130 x 1024 x 50264 85 / 54, 48 x 2048 x 50264 78 / 49, 172 x 4096 x 50264, just
// written by another product, 140 / 102; what the lines keep out: 200 x 1536 x 33000 46 / 61, 128 x 4096 x 36864 67 / 72, 136 x 2048 x 45056 57 / 64,
// 1024 x 1024 x 57344 118 / 119, and, with shorter ranges, 80 x 4096 x 11008 25 / 27, 128 x 4096 x 28672 57 / 73.
struct Plan { int bm, bn, splits, cut, cut_parts; };

enum { ONE_RANGE = 1, FEW_RANGES = 8, MOST_RANGES = 16 };

Plan plan_bf16(int M, int N, int K, int most_ranges) {
  struct Tile { int bm, bn, per_cu; double idle_us, full_us; };
  static const Tile tiles[] = {{256, 256, 1, 0.80, 1.42}, {128, 256, 1, 0.55, 0.83}, {128, 128, 2, 0.35, 0.90}};
  const int slabs = (K + BK - 1) / BK, quarters = ((M + 127) / 128) * ((N + 127) / 128);
  const bool long_k = quarters < 24 || (quarters > 32 && (M < N ? M : N) <= 256);
  Plan best{256, 256, 1, 0, 1};
  double best_us = 1e30;
  for (const Tile& t : tiles) {
    const int64_t tiles_mn = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    for (int s = 1; s <= most_ranges; s += s < 8 ? 1 : 4) {
      if (s > 1 && slabs < (s > 8 ? 40 : 4) * s) break;
      if (s > 8 && !(long_k && tiles_mn * s <= 256)) break;
      const int64_t slots = 256 * t.per_cu, full = tiles_mn * s / slots, rest = tiles_mn * s % slots;
      double per_slab = full * t.full_us;
      if (rest) per_slab += t.idle_us + (t.full_us - t.idle_us) * rest / slots;
      double us = per_slab * ((slabs + s - 1) / s) + 4.0 * (full + (rest > 0));
      if (s > 1) us += 2.0 + (double)s * M * N * 8.0 / 6.0e6;
      if (us < best_us) best_us = us, best = Plan{t.bm, t.bn, s, 0, 1};
      if (t.bm != 256 || s != 1 || full == 0 || rest == 0) continue;
      for (int parts = 2; parts <= 4 && parts * rest <= 256; parts *= 2) {
        const Tile& h = tiles[parts / 2];
        const double last = h.idle_us + (h.full_us - h.idle_us) * parts * rest / (256 * h.per_cu);
        const double cut_us = (full * t.full_us + last) * slabs + 4.0 * (full + 1);
        if (cut_us < best_us) best_us = cut_us, best = Plan{t.bm, t.bn, 1, (int)rest, parts};
      }
    }
  }
  return best;
}

// a caller with less room for the partial tiles gets the best plan of those with at most eight ranges, or of those with one
Plan plan_with_workspace(int M, int N, int K, const void* workspace, size_t workspace_bytes) {
  if (workspace != nullptr && ody_aligned16(workspace))
    for (int most : {MOST_RANGES, FEW_RANGES}) {
      const Plan pl = plan_bf16(M, N, K, most);
      if ((size_t)pl.splits * M * N * sizeof(float) <= workspace_bytes) return pl;
    }
  return plan_bf16(M, N, K, ONE_RANGE);
}

bool vec16(const void* p, int64_t ld) { return ody_aligned16(p) && ld % 8 == 0; }
bool vec8(const void* p, int64_t ld) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0 && ld % 4 == 0; }

// whether the byte offsets inside a tile fit the tile kernel's 32 bits
bool tile_pitch_ok(int op, int64_t lda, int64_t ldb) {
  const int64_t kc = (int64_t)1 << 22, strided = (int64_t)1 << 24;
  return lda < (op == ODY_GEMM_TN ? strided : kc) && ldb < (op == ODY_GEMM_NT ? kc : strided);
}

template <bool A_KC, bool B_KC>
int launch_any_pitch(const gemm_tile::Args& a, int accumulate, hipStream_t st) {
  constexpr size_t smem = 2 * sizeof(bf16) * (OperandTile<128, A_KC>::ELEMS + OperandTile<128, B_KC>::ELEMS);
  auto kern = &gemm_bf16_kernel<2, 2, A_KC, B_KC>;
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, "ody_gemm")) return rc;
  const int tiles_m = (a.M + 127) / 128, tiles_n = (a.N + 127) / 128;
  ODY_LAUNCH("gemm_bf16_any_pitch", st, kern, dim3(tiles_m * tiles_n), dim3(256), smem, a.A, a.B, a.C, a.bias, a.M, a.N, a.K, a.lda, a.ldb,
             a.ldc, accumulate, tiles_m, tiles_n);
  return ody_check_launch("gemm_bf16");
}

int launch_tiles(int op, int epi, const Plan& pl, gemm_tile::Args a, hipStream_t st) {
  a.cut = pl.cut, a.cut_parts = pl.cut_parts;
  if (op == ODY_GEMM_NT) return ody_launch_gemm_nt(epi, pl.bm, pl.bn, pl.splits, a, st);
  if (op == ODY_GEMM_NN) return ody_launch_gemm_nn(epi, pl.bm, pl.bn, pl.splits, a, st);
  return ody_launch_gemm_tn(pl.bm, pl.bn, pl.splits, a, st);
}

// One bf16 product, C = A B (+ bias) (+ add); `add` may be C itself.
int gemm_bf16(int op, const bf16* A, const bf16* B, bf16* C, const bf16* bias, const bf16* add, int M, int N, int K, int64_t lda,
              int64_t ldb, int64_t ldc, int64_t ld_add, void* workspace, size_t workspace_bytes, hipStream_t st) {
  if (op == ODY_GEMM_NT && (add == nullptr || add == C) && ody_gemm_skinny_ok(EPI_NONE, M, N))
    return ody_launch_gemm_skinny(EPI_NONE, A, B, C, bias, M, N, K, lda, ldb, ldc, add != nullptr, GemmEpi{}, st);
  gemm_tile::Args a{};
  a.A = A, a.B = B, a.C = C, a.bias = bias, a.add = add;
  a.M = M, a.N = N, a.K = K, a.lda = lda, a.ldb = ldb, a.ldc = ldc, a.ld_add = ld_add;
  a.vec16 = vec16(C, ldc) && (!add || vec16(add, ld_add));
  if (!tile_pitch_ok(op, lda, ldb)) {
    ODY_REQUIRE(add == nullptr || add == C, ODY_ERR_UNSUPPORTED, "ody_gemm: row pitch too large for a separate addend");
    if (op == ODY_GEMM_NT) return launch_any_pitch<true, true>(a, add != nullptr, st);
    if (op == ODY_GEMM_NN) return launch_any_pitch<true, false>(a, add != nullptr, st);
    return launch_any_pitch<false, false>(a, add != nullptr, st);
  }
  const Plan pl = plan_with_workspace(M, N, K, workspace, workspace_bytes);
  if (pl.splits == 1) return launch_tiles(op, EPI_NONE, pl, a, st);
  a.part = static_cast<float*>(workspace);
  if (int rc = launch_tiles(op, EPI_NONE, pl, a, st)) return rc;
  const int64_t n4 = (int64_t)M * (N / 4);
  ODY_LAUNCH("gemm_splitk_sum", st, gemm_splitk_sum_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, a.part, pl.splits, C, bias,
             add, M, N, ldc, ld_add);
  return ody_check_launch("gemm_splitk_sum");
}

}  // namespace

extern "C" size_t ody_gemm_workspace_bytes(int op, int M, int N, int K, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  if (dtype == ODY_F32) return ody_gemm_f32_workspace(M, N, K);
  if (dtype != ODY_BF16) return 0;
  if (op == ODY_GEMM_NT && ody_gemm_skinny_ok(EPI_NONE, M, N)) return 0;
  const int splits = plan_bf16(M, N, K, MOST_RANGES).splits;
  return splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
}

extern "C" int ody_gemm(int op, const void* A, const void* B, void* C, const void* bias, int M, int N, int K,
                        int64_t lda, int64_t ldb, int64_t ldc, int accumulate, int dtype, void* workspace,
                        size_t workspace_bytes, void* stream) {
  ODY_REQUIRE(A && B && C, ODY_ERR_NULL, "ody_gemm: NULL pointer");
  ODY_REQUIRE(M > 0 && N > 0 && K > 0, ODY_ERR_BAD_SHAPE, "ody_gemm: M=%d N=%d K=%d", M, N, K);
  ODY_REQUIRE(op == ODY_GEMM_NT || op == ODY_GEMM_NN || op == ODY_GEMM_TN, ODY_ERR_UNSUPPORTED, "ody_gemm: op %d", op);
  const int a_cols = (op == ODY_GEMM_TN) ? M : K, b_cols = (op == ODY_GEMM_NT) ? K : N;
  ODY_REQUIRE(lda >= a_cols && ldb >= b_cols && ldc >= N, ODY_ERR_BAD_SHAPE,
              "ody_gemm: leading dimension smaller than the row length (lda=%lld ldb=%lld ldc=%lld)", (long long)lda,
              (long long)ldb, (long long)ldc);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == ODY_F32)
    return ody_launch_gemm_f32(op, (const float*)A, (const float*)B, (float*)C, (const float*)bias, M, N, K, lda, ldb, ldc,
                    accumulate ? (const float*)C : nullptr, ldc, workspace, workspace_bytes, st);
  ODY_REQUIRE(dtype == ODY_BF16, ODY_ERR_UNSUPPORTED, "ody_gemm: dtype %d unknown", dtype);
  // 16-byte vectors along the contiguous direction of every matrix
  ODY_REQUIRE(ody_aligned16(A) && ody_aligned16(B) && ((reinterpret_cast<uintptr_t>(C) & 7u) == 0) &&
                  (!bias || (reinterpret_cast<uintptr_t>(bias) & 7u) == 0),
              ODY_ERR_MISALIGNED, "ody_gemm: A and B must be 16-byte aligned, C and bias 8-byte aligned");
  ODY_REQUIRE(lda % 8 == 0 && ldb % 8 == 0 && ldc % 4 == 0, ODY_ERR_MISALIGNED,
              "ody_gemm: lda and ldb must be multiples of 8, ldc of 4");
  ODY_REQUIRE(N % 8 == 0 && a_cols % 8 == 0 && b_cols % 8 == 0, ODY_ERR_UNSUPPORTED,
              "ody_gemm: bf16 path needs N and the contiguous extents of A and B to be multiples of 8 "
              "(M=%d N=%d K=%d op=%d)", M, N, K, op);
  return gemm_bf16(op, (const bf16*)A, (const bf16*)B, (bf16*)C, (const bf16*)bias, accumulate ? (const bf16*)C : nullptr, M, N, K, lda,
                   ldb, ldc, ldc, workspace, workspace_bytes, st);
}

// ---------------------------------------------------------------------------
// Linears with the neighbouring elementwise operation in their epilogue
// ---------------------------------------------------------------------------
namespace {
int check_lin(const char* who, const void* a, const void* b, const void* c, int M, int N, int K, int dtype) {
  ODY_REQUIRE(a && b && c, ODY_ERR_NULL, "%s: NULL pointer", who);
  ODY_REQUIRE(M > 0 && N > 0 && K > 0, ODY_ERR_BAD_SHAPE, "%s: M=%d N=%d K=%d", who, M, N, K);
  ODY_REQUIRE(dtype == ODY_BF16 || dtype == ODY_F32, ODY_ERR_UNSUPPORTED, "%s: dtype %d unknown", who, dtype);
  return ODY_OK;
}

gemm_tile::Args fused_args(const void* a, const void* b, void* c, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
                           const GemmEpi& ep) {
  gemm_tile::Args r{};
  r.A = static_cast<const bf16*>(a), r.B = static_cast<const bf16*>(b), r.C = static_cast<bf16*>(c);
  r.M = M, r.N = N, r.K = K, r.lda = lda, r.ldb = ldb, r.ldc = ldc, r.vec16 = 1, r.ep = ep;
  return r;
}
}  // namespace

extern "C" int ody_linear_rope_ws(const void* x, const void* w, const void* table, void* y, int M, int N, int K, int n_rot, int D,
                                  int64_t ldx, int64_t ldw, int64_t ld_table, int64_t ldy, int dtype, void* workspace,
                                  size_t workspace_bytes, void* stream) {
  int rc = check_lin("ody_linear_rope", x, w, y, M, N, K, dtype);
  if (rc) return rc;
  ODY_REQUIRE(table != nullptr, ODY_ERR_NULL, "ody_linear_rope: table is NULL");
  ODY_REQUIRE(dtype == ODY_BF16 && D == 128, ODY_ERR_UNSUPPORTED, "ody_linear_rope: bf16 and head_dim 128 only");
  ODY_REQUIRE(n_rot >= 0 && N % D == 0 && n_rot <= N / D, ODY_ERR_BAD_SHAPE, "ody_linear_rope: N=%d n_rot=%d D=%d", N, n_rot, D);
  ODY_REQUIRE(ldx >= K && ldw >= K && ldy >= N, ODY_ERR_BAD_SHAPE, "ody_linear_rope: leading dimension smaller than the row length");
  ODY_REQUIRE(ld_table == D, ODY_ERR_BAD_SHAPE, "ody_linear_rope: the table's rows are D = %d elements apart, got %lld", D,
              (long long)ld_table);
  ODY_REQUIRE(vec16(table, ld_table) && vec16(y, ldy), ODY_ERR_MISALIGNED,
              "ody_linear_rope: table and y need 16-byte aligned rows");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const GemmEpi ep{static_cast<const bf16*>(table), nullptr, ld_table, 0, n_rot * D};
  if (ody_gemm_skinny_ok(EPI_ROPE, M, N) && vec16(x, ldx) && vec16(w, ldw) && K % 8 == 0)
    return ody_launch_gemm_skinny(EPI_ROPE, static_cast<const bf16*>(x), static_cast<const bf16*>(w), static_cast<bf16*>(y), nullptr,
                                  M, N, K, ldx, ldw, ldy, 0, ep, st);
  if (K % 8 == 0 && tile_pitch_ok(ODY_GEMM_NT, ldx, ldw) && vec16(x, ldx) && vec16(w, ldw)) {
    const Plan pl = plan_with_workspace(M, N, K, workspace, workspace_bytes);
    gemm_tile::Args a = fused_args(x, w, y, M, N, K, ldx, ldw, ldy, ep);
    if (pl.splits == 1) return launch_tiles(ODY_GEMM_NT, EPI_ROPE, pl, a, st);
    a.part = static_cast<float*>(workspace);
    if ((rc = launch_tiles(ODY_GEMM_NT, EPI_NONE, pl, a, st))) return rc;
    const int64_t n8 = (int64_t)M * (N / 8);
    ODY_LAUNCH("gemm_splitk_rope", st, gemm_splitk_rope_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, a.part, pl.splits, a.C, ep,
               M, N, ldy);
    return ody_check_launch("gemm_splitk_rope");
  }
  // rows that 16-byte pieces cannot address: the plain product, then the rotation in place (one more rounding of the rotated columns)
  rc = ody_gemm(ODY_GEMM_NT, x, w, y, nullptr, M, N, K, ldx, ldw, ldy, 0, dtype, nullptr, 0, stream);
  if (rc) return rc;
  return ody_launch_rope_from_table(y, table, M, n_rot, D, ldy, D, 0, st);
}

extern "C" int ody_linear_rope(const void* x, const void* w, const void* table, void* y, int M, int N, int K, int n_rot, int D,
                               int64_t ldx, int64_t ldw, int64_t ld_table, int64_t ldy, int dtype, void* stream) {
  return ody_linear_rope_ws(x, w, table, y, M, N, K, n_rot, D, ldx, ldw, ld_table, ldy, dtype, nullptr, 0, stream);
}

extern "C" int ody_linear_residual_ws(const void* x, const void* w, const void* residual, void* y, int M, int N, int K,
                                      int64_t ldx, int64_t ldw, int64_t ld_res, int64_t ldy, int dtype, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  int rc = check_lin("ody_linear_residual", x, w, y, M, N, K, dtype);
  if (rc) return rc;
  ODY_REQUIRE(residual != nullptr, ODY_ERR_NULL, "ody_linear_residual: residual is NULL");
  ODY_REQUIRE(ldx >= K && ldw >= K && ld_res >= N && ldy >= N, ODY_ERR_BAD_SHAPE,
              "ody_linear_residual: leading dimension smaller than the row length");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == ODY_BF16 && ody_gemm_skinny_ok(EPI_RESIDUAL, M, N) && vec16(x, ldx) && vec16(w, ldw) &&
      vec16(residual, ld_res) && vec16(y, ldy) && K % 8 == 0 && N % 8 == 0) {
    const GemmEpi ep{static_cast<const bf16*>(residual), nullptr, ld_res, 0, 0};
    return ody_launch_gemm_skinny(EPI_RESIDUAL, static_cast<const bf16*>(x), static_cast<const bf16*>(w), static_cast<bf16*>(y),
                                  nullptr, M, N, K, ldx, ldw, ldy, 0, ep, st);
  }
  if (dtype == ODY_BF16 && K % 8 == 0 && N % 8 == 0 && tile_pitch_ok(ODY_GEMM_NT, ldx, ldw) && vec16(x, ldx) && vec16(w, ldw) &&
      vec8(residual, ld_res) && vec8(y, ldy))   // the epilogues move at least four elements at a time
    return gemm_bf16(ODY_GEMM_NT, static_cast<const bf16*>(x), static_cast<const bf16*>(w), static_cast<bf16*>(y), nullptr,
                     static_cast<const bf16*>(residual), M, N, K, ldx, ldw, ldy, ld_res, workspace, workspace_bytes, st);
  if (dtype == ODY_F32)
    return ody_launch_gemm_f32(ODY_GEMM_NT, static_cast<const float*>(x), static_cast<const float*>(w), static_cast<float*>(y), nullptr, M, N, K, ldx,
                    ldw, ldy, static_cast<const float*>(residual), y == residual ? ldy : ld_res, workspace, workspace_bytes, st);
  // any other shape or alignment: y = residual, then y += x W^T (added in fp32 before the one rounding, as above)
  if (y != residual) {
    hipError_t e = hipMemcpy2DAsync(y, (size_t)ldy * sizeof(bf16), residual, (size_t)ld_res * sizeof(bf16), (size_t)N * sizeof(bf16), (size_t)M,
                                    hipMemcpyDeviceToDevice, st);
    ODY_REQUIRE(e == hipSuccess, ODY_ERR_LAUNCH, "ody_linear_residual: copy of the residual failed: %s", hipGetErrorString(e));
  }
  return ody_gemm(ODY_GEMM_NT, x, w, y, nullptr, M, N, K, ldx, ldw, ldy, 1, dtype, workspace, workspace_bytes, stream);
}

extern "C" int ody_linear_residual(const void* x, const void* w, const void* residual, void* y, int M, int N, int K,
                                   int64_t ldx, int64_t ldw, int64_t ld_res, int64_t ldy, int dtype, void* stream) {
  return ody_linear_residual_ws(x, w, residual, y, M, N, K, ldx, ldw, ld_res, ldy, dtype, nullptr, 0, stream);
}

extern "C" int ody_swiglu_fwd(const void* gate_up, void* h, int T, int I, int64_t ld_gu, int64_t ld_h, int dtype,
                              void* stream);
extern "C" int ody_swiglu_bwd(const void* gate_up, const void* dh, void* d_gate_up, int T, int I, int64_t ld_gu,
                              int64_t ld_dh, int64_t ld_dgu, int dtype, void* stream);

namespace {
// The kernel that writes h (and gate_up, unless it is NULL) in one launch.  Two thirds of what its epilogue stores is gate_up, behind
// the last slab where nothing hides it: without, 4096 x 22016 x 4096 takes 518 us instead of 537, 16384 rows 2053 instead of 2157.
// ODY_ERR_UNSUPPORTED, with nothing launched, for sizes
// and alignments that no kernel with that epilogue takes.
int linear_swiglu_fused(const void* x, const void* w_gate_up, void* gate_up, void* h, int T, int I, int K, int64_t ldx, int64_t ldw,
                        int64_t ld_gu, int64_t ld_h, hipStream_t st, bool launch) {
  if (K % 8 != 0 || !vec16(x, ldx) || !vec16(w_gate_up, ldw) || !vec16(h, ld_h) || (gate_up && !vec16(gate_up, ld_gu)))
    return ODY_ERR_UNSUPPORTED;
  const GemmEpi ep{nullptr, static_cast<bf16*>(h), 0, ld_h, I};
  if (ody_gemm_skinny_ok(EPI_SWIGLU_FWD, T, 2 * I))
    return !launch ? ODY_OK : ody_launch_gemm_skinny(EPI_SWIGLU_FWD, static_cast<const bf16*>(x), static_cast<const bf16*>(w_gate_up),
                                                     static_cast<bf16*>(gate_up), nullptr, T, 2 * I, K, ldx, ldw, ld_gu, 0, ep, st);
  if (I % 128 == 0 && tile_pitch_ok(ODY_GEMM_NT, ldx, ldw) && (int64_t)I * ldw < (1ll << 29))
    return !launch ? ODY_OK : launch_tiles(ODY_GEMM_NT, EPI_SWIGLU_FWD, plan_bf16(T, 2 * I, K, ONE_RANGE),
                                           fused_args(x, w_gate_up, gate_up, T, 2 * I, K, ldx, ldw, ld_gu, ep), st);
  return ODY_ERR_UNSUPPORTED;
}
}  // namespace

extern "C" int ody_linear_swiglu_h_fused(const void* x, const void* w_gate_up, int T, int I, int K, int64_t ldx, int64_t ldw, int dtype) {
  return T > 0 && I > 0 && K > 0 && dtype == ODY_BF16 &&
         linear_swiglu_fused(x, w_gate_up, nullptr, nullptr, T, I, K, ldx, ldw, 0, (int64_t)I % 8, nullptr, false) == ODY_OK;
}

extern "C" int ody_linear_swiglu_h(const void* x, const void* w_gate_up, void* h, int T, int I, int K, int64_t ldx, int64_t ldw,
                                   int64_t ld_h, int dtype, void* stream) {
  int rc = check_lin("ody_linear_swiglu_h", x, w_gate_up, h, T, I, K, dtype);
  if (rc) return rc;
  ODY_REQUIRE(ldx >= K && ldw >= K && ld_h >= I, ODY_ERR_BAD_SHAPE, "ody_linear_swiglu_h: leading dimension smaller than the row length");
  rc = dtype == ODY_BF16 ? linear_swiglu_fused(x, w_gate_up, nullptr, h, T, I, K, ldx, ldw, 0, ld_h, static_cast<hipStream_t>(stream), true)
                         : (int)ODY_ERR_UNSUPPORTED;
  ODY_REQUIRE(rc != ODY_ERR_UNSUPPORTED, ODY_ERR_UNSUPPORTED, "ody_linear_swiglu_h: T=%d I=%d K=%d needs a gate_up buffer", T, I, K);
  return rc;
}

extern "C" int ody_linear_swiglu(const void* x, const void* w_gate_up, void* gate_up, void* h, int T, int I, int K,
                                 int64_t ldx, int64_t ldw, int64_t ld_gu, int64_t ld_h, int dtype, void* stream) {
  int rc = check_lin("ody_linear_swiglu", x, w_gate_up, gate_up, T, I, K, dtype);
  if (rc) return rc;
  ODY_REQUIRE(h != nullptr, ODY_ERR_NULL, "ody_linear_swiglu: h is NULL");
  ODY_REQUIRE(ldx >= K && ldw >= K && ld_gu >= 2 * (int64_t)I && ld_h >= I, ODY_ERR_BAD_SHAPE,
              "ody_linear_swiglu: leading dimension smaller than the row length");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == ODY_BF16) {
    rc = linear_swiglu_fused(x, w_gate_up, gate_up, h, T, I, K, ldx, ldw, ld_gu, ld_h, st, true);
    if (rc != ODY_ERR_UNSUPPORTED) return rc;
  }
  rc = ody_gemm(ODY_GEMM_NT, x, w_gate_up, gate_up, nullptr, T, 2 * I, K, ldx, ldw, ld_gu, 0, dtype, nullptr, 0, stream);
  if (rc) return rc;
  return ody_swiglu_fwd(gate_up, h, T, I, ld_gu, ld_h, dtype, stream);
}

// The RMSNorm in front of a product of few rows, inside it: 16-byte rows, K % 8 == 0, rows that fit a block's LDS.
namespace {
bool norm_fits(const void* x, const void* norm_w, const void* w, const void* y, int M, int K, int64_t ldx, int64_t ldw, int64_t ldy) {
  return M <= ODY_SKINNY_NORM_MAX_M && (size_t)M * (K + 8) * sizeof(bf16) <= ODY_SKINNY_NORM_BYTES && K % 8 == 0 && vec16(x, ldx) && vec16(w, ldw) && vec16(y, ldy) && ody_aligned16(norm_w);
}
}  // namespace

extern "C" int ody_norm_linear_rope(const void* x, const void* norm_w, float eps, const void* w, const int64_t* position_ids,
                                    const float* inv_freq, void* y, int M, int N, int K, int n_rot, int D, int64_t ldx, int64_t ldw,
                                    int64_t ldy, int dtype, void* stream) {
  int rc = check_lin("ody_norm_linear_rope", x, w, y, M, N, K, dtype);
  if (rc) return rc;
  ODY_REQUIRE(norm_w && position_ids && inv_freq, ODY_ERR_NULL, "ody_norm_linear_rope: NULL pointer");
  ODY_REQUIRE(ldx >= K && ldw >= K && ldy >= N, ODY_ERR_BAD_SHAPE, "ody_norm_linear_rope: leading dimension smaller than the row length");
  ODY_REQUIRE(n_rot >= 0 && D > 0 && N % D == 0 && n_rot <= N / D, ODY_ERR_BAD_SHAPE, "ody_norm_linear_rope: N=%d n_rot=%d D=%d", N, n_rot, D);
  ODY_REQUIRE(dtype == ODY_BF16 && D == 128 && ody_gemm_skinny_ok(EPI_ROPE, M, N) && norm_fits(x, norm_w, w, y, M, K, ldx, ldw, ldy),
              ODY_ERR_UNSUPPORTED, "ody_norm_linear_rope: bf16, head_dim 128, few rows on 16-byte boundaries");
  GemmEpi ep{nullptr, nullptr, 0, 0, n_rot * D};
  ep.norm = static_cast<const bf16*>(norm_w), ep.eps = eps, ep.positions = position_ids, ep.inv_freq = inv_freq;
  return ody_launch_gemm_skinny(EPI_ROPE, static_cast<const bf16*>(x), static_cast<const bf16*>(w), static_cast<bf16*>(y), nullptr, M, N, K, ldx,
                                ldw, ldy, 0, ep, static_cast<hipStream_t>(stream));
}

extern "C" int ody_norm_linear_swiglu_h(const void* x, const void* norm_w, float eps, const void* w_gate_up, void* h, int T, int I, int K,
                                        int64_t ldx, int64_t ldw, int64_t ld_h, int dtype, void* stream) {
  int rc = check_lin("ody_norm_linear_swiglu_h", x, w_gate_up, h, T, I, K, dtype);
  if (rc) return rc;
  ODY_REQUIRE(norm_w != nullptr, ODY_ERR_NULL, "ody_norm_linear_swiglu_h: NULL pointer");
  ODY_REQUIRE(ldx >= K && ldw >= K && ld_h >= I, ODY_ERR_BAD_SHAPE, "ody_norm_linear_swiglu_h: leading dimension smaller than the row length");
  ODY_REQUIRE(dtype == ODY_BF16 && I < (1 << 30) && ody_gemm_skinny_ok(EPI_SWIGLU_FWD, T, 2 * I) &&
                  norm_fits(x, norm_w, w_gate_up, h, T, K, ldx, ldw, ld_h),
              ODY_ERR_UNSUPPORTED, "ody_norm_linear_swiglu_h: bf16, few rows on 16-byte boundaries, I a multiple of 16");
  GemmEpi ep{nullptr, static_cast<bf16*>(h), 0, ld_h, I};
  ep.norm = static_cast<const bf16*>(norm_w), ep.eps = eps;
  return ody_launch_gemm_skinny(EPI_SWIGLU_FWD, static_cast<const bf16*>(x), static_cast<const bf16*>(w_gate_up), nullptr, nullptr, T, 2 * I, K,
                                ldx, ldw, 0, 0, ep, static_cast<hipStream_t>(stream));
}

extern "C" size_t ody_linear_dgrad_swiglu_workspace_bytes(int T, int I, int K, int dtype) {
  if (T <= 0 || I <= 0 || K <= 0) return 0;
  if (dtype == ODY_BF16 && I % 128 == 0 && K % 8 == 0) return 0;
  return (((size_t)T * I * (dtype == ODY_BF16 ? 2 : 4)) + 255) & ~(size_t)255;
}

extern "C" int ody_linear_dgrad_swiglu(const void* dy, const void* w_down, const void* gate_up, void* d_gate_up, int T,
                                       int I, int K, int64_t ld_dy, int64_t ldw, int64_t ld_gu, int64_t ld_dgu, int dtype,
                                       void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_lin("ody_linear_dgrad_swiglu", dy, w_down, d_gate_up, T, I, K, dtype);
  if (rc) return rc;
  ODY_REQUIRE(gate_up != nullptr, ODY_ERR_NULL, "ody_linear_dgrad_swiglu: gate_up is NULL");
  ODY_REQUIRE(ld_dy >= K && ldw >= I && ld_gu >= 2 * (int64_t)I && ld_dgu >= 2 * (int64_t)I, ODY_ERR_BAD_SHAPE,
              "ody_linear_dgrad_swiglu: leading dimension smaller than the row length");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == ODY_BF16 && I % 128 == 0 && K % 8 == 0 && tile_pitch_ok(ODY_GEMM_NN, ld_dy, ldw) && vec16(dy, ld_dy) &&
      vec16(w_down, ldw) && vec16(gate_up, ld_gu) && vec16(d_gate_up, ld_dgu)) {
    const GemmEpi ep{static_cast<const bf16*>(gate_up), nullptr, ld_gu, 0, I};
    return launch_tiles(ODY_GEMM_NN, EPI_SWIGLU_BWD, plan_bf16(T, I, K, ONE_RANGE),
                        fused_args(dy, w_down, d_gate_up, T, I, K, ld_dy, ldw, ld_dgu, ep), st);
  }
  const size_t need = (size_t)T * I * (dtype == ODY_BF16 ? 2 : 4);
  ODY_REQUIRE(workspace != nullptr && workspace_bytes >= need && ody_aligned16(workspace), ODY_ERR_WORKSPACE,
              "ody_linear_dgrad_swiglu: this shape runs as two kernels and needs a 16-byte aligned workspace of %zu bytes "
              "for dh (got %zu)", need, workspace ? workspace_bytes : (size_t)0);
  rc = ody_gemm(ODY_GEMM_NN, dy, w_down, workspace, nullptr, T, I, K, ld_dy, ldw, I, 0, dtype, nullptr, 0, stream);
  if (rc) return rc;
  return ody_swiglu_bwd(gate_up, workspace, d_gate_up, T, I, ld_gu, I, ld_dgu, dtype, stream);
}
