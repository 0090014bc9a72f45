// fp32 products, C (M, N) = op(A) . op(B) (+ bias) (+ addend), any shape and alignment, on the bf16 matrix cores.
//
// An fp32 value is the sum of three bf16 values (split3.h); of the nine products of two such sums the six largest are formed, which
// leaves out at most a unit roundoff of fp32, 2^-24 of a product, and 2^-27.5 in the root mean square.  The largest one and the five others accumulate apart, so that
// the sum of the large terms is rounded once per 16 of K (the fp32 matrix instruction: every 2).  2-norm error against 64 bits, this
// / v_mfma_f32_32x32x2_f32 before it, N(0, 1) operands: K = 512 0.8e-7 to 1.3e-7 / 2.9e-7, 2048 1.3e-7 / 2.9e-7, 4096 4.0e-7 / 11.5e-7.  Operands on [1, 2), K = 4 to 4096:
// 2.8e-8 to 6.4e-8 / 3.8e-8 to 12.7e-8; all of them 0x1.00ff8p+0, where what is left out is largest and always of one sign: 5.9e-8 both.
//
// Six bf16 instructions take 192 matrix cycles where the fp32 one takes 512.  Bound by the rate of the matrix cores at the power limit
// where the product is large (4096^3: 70 % busy at 1.7 GHz), by the loads where it is small: a 64 x 64 tile moves 16 KB per 32 of K and
// its share of the splitting takes as many vector cycles as its products take matrix cycles.
//
// 4096^3, NT / TN: 1016 / 1023 -> 690 / 720 us (199 / 191 TFLOP/s).  The products of a layer of hidden 512 over 2048 tokens, us before /
// now: 2048 x 1536 x 512 37 / 29, x 2752 60 / 43, x 512 14.8 / 12, 2048 x 512 x 1376 34 / 26, 2048 x 512 x 2752 NN 61 / 46, 2752 x 512 x 2048
// TN 66 / 54, 512 x 512 x 2048 TN 17.6 / 16.7 (sum over all twelve 454 / 361).  Without SPLIT_UP, which is one more instruction an element
// and keeps the bits of operands below 2^-110, and with it, both on another box: 4096^3 NT / NN / TN 783 / 774 / 807 and 786 / 778 / 814;
// 2048 x 1536 x 512 29.9 and 30.5, 2048 x 2752 x 512 44.6 and 45.6, 512 x 1376 x 2048 TN 32.4 and 33.6 (the most).
//
// An input that is not finite, or from 2^111.99 on, makes 0 x infinity in a product that is none, and a result from 2^96 on is infinite before
// SPLIT_DOWN; a wavefront that finds a result that is not finite forms its tiles again on the fp32 instruction, straight from memory.
#include <algorithm>
#include <type_traits>
#include "gemm_tile.h"
#include "split3.h"

namespace {

constexpr int SK = 32;         // K slab
constexpr int PITCH = SK + 8;  // elements between the rows of a plane
// largest row pitch (exclusive) whose byte offsets inside a slab, 128 rows or 32 rows of K, stay below 2^31
constexpr int64_t max_pitch(bool kc) { return (int64_t)1 << (kc ? 22 : 24); }

// The share of one of TH threads in bringing ROWS rows x SK of K of an operand from global memory to its three planes [ROWS][PITCH]
// in LDS, as N loads of 4 floats.
//   KC (memory is (rows, K) row-major): a load is 4 k of a row, written as 8 bytes per plane.
//   else (memory is (K, rows)): the loads are 4 rows of N consecutive k, turned over in registers and written like the others.
// Either way the lanes of a row write its 64 bytes side by side, and 32 lanes rows 4 apart, whose 320 bytes put them on all the
// banks once.
template <int ROWS, bool KC, int TH>
struct Mover {
  static constexpr int N = ROWS * SK / 4 / TH, KL = KC ? 8 : SK / N;   // loads, lanes along K

  static __device__ __forceinline__ int k_of(int j, int t) { return KC ? 4 * (t & 7) : N * (t & (KL - 1)) + j; }
  static __device__ __forceinline__ int row_of(int j, int t) {   // of load j (KC), first one of all loads (else)
    const int q = t / KL;
    return KC ? TH / 8 * j + 4 * (q & 3) + ((q >> 2) & 3) + 16 * (q >> 4) : 4 * q;
  }
  // byte offset of a load in the slab, beyond the buffer's range for a row past the end; pitches below max_pitch
  static __device__ __forceinline__ unsigned offset(int j, int64_t ld, int row0, int nrows, int t) {
    const int rr = row_of(j, t), kk = k_of(j, t);
    return row0 + rr < nrows ? 4u * (unsigned)(KC ? rr * (int)ld + kk : kk * (int)ld + rr) : gemm_tile::PAST_END;
  }
  // base: first row of the tile, k = 0.  Without a branch: behind one the compiler loses count of the loads in flight and waits for
  // all of them.
  static __device__ __forceinline__ void fetch_vec(f32x4 (&r)[N], const float* base, int64_t ld, const unsigned (&off)[N], int k0, int k_end, int t) {
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base + (KC ? k0 : k0 * ld)), 0, 0x7fffffff, 0x00020000);
#pragma unroll
    for (int j = 0; j < N; j++)
      r[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, k0 + k_of(j, t) < k_end ? off[j] : gemm_tile::PAST_END, 0, 0));
  }
  // single floats; what lies outside reads as zero
  static __device__ __forceinline__ void fetch_any(f32x4 (&r)[N], const float* base, int64_t ld, int row0, int k0, int nrows, int k_end, int t) {
#pragma unroll
    for (int j = 0; j < N; j++) {
      const int row = row_of(j, t), k = k0 + k_of(j, t);
      const float* src = KC ? base + (int64_t)row * ld + k : base + (int64_t)k * ld + row;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const bool ok = KC ? (row0 + row < nrows && k + e < k_end) : (row0 + row + e < nrows && k < k_end);
        r[j][e] = ok ? src[e] : 0.f;
      }
    }
  }
  static __device__ __forceinline__ void put(const f32x4 (&r)[N], bf16* planes, int t) {
    constexpr int W = KC ? 4 : N;   // k of one write
#pragma unroll
    for (int e = 0; e < (KC ? N : 4); e++) {
      typename FloatVec<W>::type x;
#pragma unroll
      for (int j = 0; j < W; j++) x[j] = (KC ? r[e][j] : r[j][e]) * SPLIT_UP;
      const Split3<W> s(x);
      bf16* dst = planes + (KC ? row_of(e, t) : row_of(0, t) + e) * PITCH + k_of(0, t);
#pragma unroll
      for (int p = 0; p < 3; p++) *reinterpret_cast<typename Split3<W>::part*>(dst + p * ROWS * PITCH) = s.p[p];
    }
  }
};

// Both operands of a slab, brought by 256 threads.  64 + 64 rows: half of the threads bring one operand each, in pieces of 4 x 4 (pieces
// of 4 x 2, all threads both, took the weight gradients of 64 x 64 tiles from 34 to 53 us); more rows: all threads both.
template <int BM, int BN, bool A_KC, bool B_KC>
struct Slab {
  using MA = Mover<BM, A_KC, 256>;
  using MB = Mover<BN, B_KC, 256>;
  f32x4 ra[MA::N], rb[MB::N];
  unsigned oa[MA::N], ob[MB::N];
  const float *a, *b;
  int64_t lda, ldb;
  int m0, n0, M, N, t;
  __device__ __forceinline__ Slab(const float* A, const float* B, int64_t lda, int64_t ldb, int m0, int n0, int M, int N, int t)
      : a(A + (A_KC ? m0 * lda : m0)), b(B + (B_KC ? n0 * ldb : n0)), lda(lda), ldb(ldb), m0(m0), n0(n0), M(M), N(N), t(t) {
#pragma unroll
    for (int j = 0; j < MA::N; j++) oa[j] = MA::offset(j, lda, m0, M, t);
#pragma unroll
    for (int j = 0; j < MB::N; j++) ob[j] = MB::offset(j, ldb, n0, N, t);
  }
  template <bool VEC>
  __device__ __forceinline__ void fetch(int k0, int k_end) {   // past the range: zeros, nothing is read
    if (VEC) {
      MA::fetch_vec(ra, a, lda, oa, k0, k_end, t);
      MB::fetch_vec(rb, b, ldb, ob, k0, k_end, t);
    } else {
      MA::fetch_any(ra, a, lda, m0, k0, M, k_end, t);
      MB::fetch_any(rb, b, ldb, n0, k0, N, k_end, t);
    }
  }
  __device__ __forceinline__ void put(bf16* As, bf16* Bs) const {
    MA::put(ra, As, t);
    MB::put(rb, Bs, t);
  }
};
template <bool A_KC, bool B_KC>
struct Slab<64, 64, A_KC, B_KC> {
  using MA = Mover<64, A_KC, 128>;
  using MB = Mover<64, B_KC, 128>;
  f32x4 r[4];
  unsigned off[4];
  const float* base;
  int64_t ld;
  int row0, nrows, t;
  bool second;
  __device__ __forceinline__ Slab(const float* A, const float* B, int64_t lda, int64_t ldb, int m0, int n0, int M, int N, int tid)
      : t(tid & 127), second(__builtin_amdgcn_readfirstlane(tid >> 7)) {
    ld = second ? ldb : lda, row0 = second ? n0 : m0, nrows = second ? N : M;
    base = second ? B + (B_KC ? n0 * ldb : n0) : A + (A_KC ? m0 * lda : m0);
#pragma unroll
    for (int j = 0; j < 4; j++) off[j] = second ? MB::offset(j, ld, row0, nrows, t) : MA::offset(j, ld, row0, nrows, t);
  }
  template <bool VEC>
  __device__ __forceinline__ void fetch(int k0, int k_end) {
    if (A_KC == B_KC || !second) {
      if (VEC) MA::fetch_vec(r, base, ld, off, k0, k_end, t);
      else MA::fetch_any(r, base, ld, row0, k0, nrows, k_end, t);
    } else {
      if (VEC) MB::fetch_vec(r, base, ld, off, k0, k_end, t);
      else MB::fetch_any(r, base, ld, row0, k0, nrows, k_end, t);
    }
  }
  __device__ __forceinline__ void put(bf16* As, bf16* Bs) const {
    if (A_KC == B_KC || !second) MA::put(r, second ? Bs : As, t);
    else MB::put(r, Bs, t);
  }
};

// What each SIMD has room for: blocks per compute unit times G.
constexpr int waves_per_simd(int wm, int wn) { return wm + wn == 2 ? 4 : (wm + wn == 3 ? 3 : 2); }

// G groups of 4 wavefronts in a 2 x 2 arrangement, each wavefront owning WM x WN result tiles of 32 x 32.  A group takes every G-th
// slab of K through LDS of its own: split and written, then multiplied.  Odd groups do the one while even groups do the other, as
// different blocks of a compute unit do by chance; the groups' sums meet in LDS.  The product is computed as C^T = op(B)^T op(A)^T, so
// a lane holds 4 consecutive N per register quad and writes 16-byte pieces of C rows.
// splits > 1: a block takes one of so many ranges of slabs and writes fp32 partial results to part[split][M][N] (VEC only).
// VEC = false (unaligned pointers, or a contiguous extent that is no multiple of 4) moves single floats.
template <int WM, int WN, int G, bool A_KC, bool B_KC, bool VEC>
__global__ __launch_bounds__(256 * G, waves_per_simd(WM, WN)) void gemm_f32_kernel(
    const float* __restrict__ A, const float* __restrict__ B, float* C, const float* __restrict__ bias, int M, int N, int K, int64_t lda,
    int64_t ldb, int64_t ldc, const float* add, int64_t ld_add, int ntn, int splits, float* part) {
  constexpr int BM = 64 * WM, BN = 64 * WN;
  extern __shared__ __attribute__((aligned(16))) bf16 smem[];   // [G][A planes, B planes]
  const int tid = threadIdx.x, lane = tid & 63, wave = (tid >> 6) & 3, i = lane & 31, g = lane >> 5;
  const int group = __builtin_amdgcn_readfirstlane(tid >> 8), t = tid & 255;
  const int wm = wave >> 1, wn = wave & 1;
  // every XCD works on neighbouring tiles
  const int at = gemm_tile::xcd_position(blockIdx.x, gridDim.x), tiles = gridDim.x / splits, tile = at % tiles, split = at / tiles;
  const int m0 = (tile / ntn) * BM, n0 = (tile % ntn) * BN;
  bf16 *As = smem + group * 3 * (BM + BN) * PITCH, *Bs = As + 3 * BM * PITCH;

  f32x16 hi[WM][WN], lo[WM][WN];
#pragma unroll
  for (int a = 0; a < WM; a++)
#pragma unroll
    for (int b = 0; b < WN; b++)
#pragma unroll
      for (int r = 0; r < 16; r++) hi[a][b][r] = lo[a][b][r] = 0.f;

  int k_first = 0, k_last = K;
  if (VEC && part) {
    const int per = ((K + SK - 1) / SK + splits - 1) / splits * SK;
    k_first = min(split * per, K), k_last = min(k_first + per, K);
  }
  Slab<BM, BN, A_KC, B_KC> slab(A, B, lda, ldb, m0, n0, M, N, t);
  auto multiply = [&]() {
#pragma unroll
    for (int ks = 0; ks < SK / 16; ks++) {
      bf16x8 af[WM][3], bfr[WN][3];
#pragma unroll
      for (int p = 0; p < 3; p++) {
#pragma unroll
        for (int a = 0; a < WM; a++)
          af[a][p] = *reinterpret_cast<const bf16x8*>(As + (p * BM + 32 * (wm * WM + a) + i) * PITCH + 16 * ks + 8 * g);
#pragma unroll
        for (int b = 0; b < WN; b++)
          bfr[b][p] = *reinterpret_cast<const bf16x8*>(Bs + (p * BN + 32 * (wn * WN + b) + i) * PITCH + 16 * ks + 8 * g);
      }
#pragma unroll
      for (int a = 0; a < WM; a++)
#pragma unroll
        for (int b = 0; b < WN; b++) mfma_split3(bfr[b], af[a], hi[a][b], lo[a][b]);
    }
  };
  const int turns = (k_last - k_first + G * SK - 1) / (G * SK);
  int k0 = k_first + group * SK;
  slab.template fetch<VEC>(k0, k_last);
  if (G > 1 && (group & 1)) __syncthreads();
  for (int it = 0; it < turns; it++) {
    slab.put(As, Bs);
    k0 += G * SK;
    slab.template fetch<VEC>(k0, k_last);
    __syncthreads();
    multiply();
    __syncthreads();
  }
  if (G > 1 && !(group & 1)) __syncthreads();

#pragma unroll
  for (int a = 0; a < WM; a++)
#pragma unroll
    for (int b = 0; b < WN; b++) hi[a][b] += lo[a][b];
  if constexpr (G > 1) {
    static_assert(WM == 1 && WN == 1, "the groups' sums have to fit the planes' room");
    // the groups' sums through LDS, [group][wave][register quad][lane]; a group ends up with every G-th quad
    f32x4* sums = reinterpret_cast<f32x4*>(smem) + wave * 256 + lane;
#pragma unroll
    for (int q = 0; q < 4; q++) sums[group * 1024 + q * 64] = f32x4{hi[0][0][4 * q], hi[0][0][4 * q + 1], hi[0][0][4 * q + 2], hi[0][0][4 * q + 3]};
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (q % G != group) continue;
      f32x4 v = sums[q * 64];
#pragma unroll
      for (int s = 1; s < G; s++) v += sums[s * 1024 + q * 64];
#pragma unroll
      for (int e = 0; e < 4; e++) hi[0][0][4 * q + e] = v[e];
    }
  }
  bool finite = true;
#pragma unroll
  for (int a = 0; a < WM; a++)
#pragma unroll
    for (int b = 0; b < WN; b++)
#pragma unroll
      for (int r = 0; r < 16; r++)
        if ((r >> 2) % G == group) finite &= __builtin_fabsf(hi[a][b][r]) < INFINITY;
  if (__any(!finite)) {   // see above; rare
#pragma unroll
    for (int a = 0; a < WM; a++)
#pragma unroll
      for (int b = 0; b < WN; b++) {
        const int m = m0 + 32 * (wm * WM + a) + i, n = n0 + 32 * (wn * WN + b) + i;
        f32x16 c;
#pragma unroll
        for (int r = 0; r < 16; r++) c[r] = 0.f;
        for (int k1 = k_first; k1 < k_last; k1 += 2) {
          const int k = k1 + g;
          const float av = m < M && k < k_last ? A[A_KC ? (int64_t)m * lda + k : (int64_t)k * lda + m] : 0.f;
          const float bv = n < N && k < k_last ? B[B_KC ? (int64_t)n * ldb + k : (int64_t)k * ldb + n] : 0.f;
          c = __builtin_amdgcn_mfma_f32_32x32x2f32(bv, av, c, 0, 0, 0);
        }
        hi[a][b] = c;
      }
  } else {
#pragma unroll
    for (int a = 0; a < WM; a++)
#pragma unroll
      for (int b = 0; b < WN; b++) hi[a][b] *= SPLIT_DOWN;
  }
  // register r of lane (i, g) of tile (a, b): row m = 32 (wm WM + a) + i, column n = 32 (wn WN + b) + 8 (r / 4) + 4 g + r % 4
#pragma unroll
  for (int a = 0; a < WM; a++) {
    const int m = m0 + 32 * (wm * WM + a) + i;
    if (m >= M) continue;
#pragma unroll
    for (int b = 0; b < WN; b++) {
      const f32x16 v = hi[a][b];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        if (q % G != group) continue;
        const int n = n0 + 32 * (wn * WN + b) + 8 * q + 4 * g;
        if (VEC && part) {
          if (n < N)
            *reinterpret_cast<f32x4*>(part + ((int64_t)split * M + m) * N + n) = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
          continue;
        }
        float* dst = C + (int64_t)m * ldc + n;
        if (VEC && n + 3 < N) {
          f32x4 o{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
          if (bias) o += *reinterpret_cast<const f32x4*>(bias + n);
          if (add) o += *reinterpret_cast<const f32x4*>(add + (int64_t)m * ld_add + n);
          *reinterpret_cast<f32x4*>(dst) = o;
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++) {
            if (n + e >= N) continue;
            float o = v[4 * q + e];
            if (bias) o += bias[n + e];
            if (add) o += add[(int64_t)m * ld_add + n + e];
            dst[e] = o;
          }
        }
      }
    }
  }
}

// C (+)= sum of the fp32 partial results (+ bias); 4 elements per thread
__global__ __launch_bounds__(256) void gemm_f32_sum_kernel(const float* __restrict__ part, int splits, float* C,
                                                           const float* __restrict__ bias, int M, int N, int64_t ldc, const float* add,
                                                           int64_t ld_add) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)M * (N / 4)) return;
  const int m = idx / (N / 4), n = (idx % (N / 4)) * 4;
  const float* src = part + (int64_t)m * N + n;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < splits; s++) v += *reinterpret_cast<const f32x4*>(src + (int64_t)s * M * N);
  if (bias) v += *reinterpret_cast<const f32x4*>(bias + n);
  f32x4* dst = reinterpret_cast<f32x4*>(C + (int64_t)m * ldc + n);
  if (add) v += *reinterpret_cast<const f32x4*>(add + (int64_t)m * ld_add + n);
  *dst = v;
}

// Tile and ranges of K of an fp32 product, by the time that the candidates were measured to take (fitted to 800 products of 64 to 4096
// rows with 1 to 12 ranges; the pick is 1 % off the best of them in the mean, 9 % at most): us per slab of a compute unit
// with one, two or three blocks on it -- per four slabs for the 64 x 64 tile, whose one block has four groups --, a start per round of
// blocks, and the trip of the partial results.  Few tiles: 64 x 64 in groups, whose sums need no trip (2048 x 512 x 1376: 26.5 us, 128 x 64
// tiles in 4 ranges 31.8); more: 128 x 64 (2048 x 1536 x 512: 29.1, 64 x 64 in groups 38.7, 128 x 128 34.1); many: 128 x 128 (4096^3: 696,
// 128 x 64 759).
struct PlanF32 { int bm, bn, splits; };
PlanF32 plan_f32(int M, int N, int K, bool may_split) {
  struct Tile { int bm, bn, per_cu, groups; double slab_us[3]; };
  static const Tile tiles[] = {{64, 64, 1, 4, {1.87, 0, 0}}, {128, 64, 3, 1, {0.99, 1.43, 2.03}}, {128, 128, 2, 1, {1.63, 2.33, 0}}};
  const int slabs = (K + SK - 1) / SK;
  PlanF32 best{64, 64, 1};
  double best_us = 1e30;
  for (const Tile& t : tiles) {
    const int64_t tiles_mn = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    for (int s = 1; s <= (may_split ? 16 : 1) && (s == 1 || slabs >= 4 * s); s++) {
      const int64_t full = tiles_mn * s / (256 * t.per_cu), rest = tiles_mn * s % (256 * t.per_cu);
      const int turns = ((slabs + s - 1) / s + t.groups - 1) / t.groups;
      double us = 2.6 + full * (turns * t.slab_us[t.per_cu - 1] + 2.7);
      if (rest) us += turns * t.slab_us[(rest + 255) / 256 - 1] + 2.7;
      if (s > 1) us += 2.2 + (double)s * M * N * 8.0 / 5.5e6;
      if (us < best_us) best_us = us, best = PlanF32{t.bm, t.bn, s};
    }
  }
  return best;
}

template <int WM, int WN, int G, bool A_KC, bool B_KC, bool VEC>
int launch_kernel(const float* a, const float* b, float* c, const float* bias, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc,
                  const float* add, int64_t ld_add, int splits, float* part, hipStream_t st) {
  constexpr int BM = 64 * WM, BN = 64 * WN;
  constexpr size_t smem = sizeof(bf16) * G * 3 * (BM + BN) * PITCH;
  const int64_t ntm = (M + BM - 1) / BM, ntn = (N + BN - 1) / BN;
  ODY_REQUIRE(ntm * ntn * splits < ((int64_t)1 << 31), ODY_ERR_BAD_SHAPE, "ody_gemm: M=%d N=%d too large for one launch", M, N);
  auto kern = &gemm_f32_kernel<WM, WN, G, A_KC, B_KC, VEC>;
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, "ody_gemm")) return rc;
  ODY_LAUNCH("gemm_f32", st, kern, dim3((unsigned)(ntm * ntn * splits)), dim3(256 * G), smem, a, b, c, bias, M, N, K, lda, ldb, ldc, add, ld_add,
             (int)ntn, splits, part);
  return ody_check_launch("gemm_f32");
}

template <int WM, int WN, int G, bool A_KC, bool B_KC>
int launch_f32(const float* a, const float* b, float* c, const float* bias, int M, int N, int K, int64_t lda,
               int64_t ldb, int64_t ldc, const float* add, int64_t ld_add, bool vec, int splits, float* part, hipStream_t st) {
  const int rc = vec ? launch_kernel<WM, WN, G, A_KC, B_KC, true>(a, b, c, bias, M, N, K, lda, ldb, ldc, add, ld_add, splits, part, st)
                     : launch_kernel<WM, WN, G, A_KC, B_KC, false>(a, b, c, bias, M, N, K, lda, ldb, ldc, add, ld_add, 1, nullptr, st);
  if (rc || splits == 1) return rc;
  const int64_t n4 = (int64_t)M * (N / 4);
  ODY_LAUNCH("gemm_f32_sum", st, gemm_f32_sum_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, part, splits, c, bias, M, N, ldc,
             add, ld_add);
  return ody_check_launch("gemm_f32_sum");
}

template <bool A_KC, bool B_KC>
int dispatch_f32(const float* a, const float* b, float* c, const float* bias, int M, int N, int K, int64_t lda,
                 int64_t ldb, int64_t ldc, const float* add, int64_t ld_add, void* workspace, size_t workspace_bytes, hipStream_t st) {
  const bool vec = ody_aligned16(a) && ody_aligned16(b) && ody_aligned16(c) && (!bias || ody_aligned16(bias)) && lda < max_pitch(A_KC) &&
                   ldb < max_pitch(B_KC) && lda % 4 == 0 && ldb % 4 == 0 && ldc % 4 == 0 &&
                   (!add || (ody_aligned16(add) && ld_add % 4 == 0)) && N % 4 == 0 && (A_KC ? K : M) % 4 == 0 && (!B_KC || K % 4 == 0);
  PlanF32 pl = plan_f32(M, N, K, vec && workspace && ody_aligned16(workspace));
  if (pl.splits > 1 && workspace_bytes < (size_t)pl.splits * M * N * sizeof(float)) pl = plan_f32(M, N, K, false);
  float* part = pl.splits > 1 ? static_cast<float*>(workspace) : nullptr;
  if (pl.bm == 64) return launch_f32<1, 1, 4, A_KC, B_KC>(a, b, c, bias, M, N, K, lda, ldb, ldc, add, ld_add, vec, pl.splits, part, st);
  if (pl.bn == 64) return launch_f32<2, 1, 1, A_KC, B_KC>(a, b, c, bias, M, N, K, lda, ldb, ldc, add, ld_add, vec, pl.splits, part, st);
  return launch_f32<2, 2, 1, A_KC, B_KC>(a, b, c, bias, M, N, K, lda, ldb, ldc, add, ld_add, vec, pl.splits, part, st);
}

}  // namespace

size_t ody_gemm_f32_workspace(int M, int N, int K) {
  const int splits = plan_f32(M, N, K, true).splits;
  return splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
}

int ody_launch_gemm_f32(int op, const float* a, const float* b, float* c, const float* bias, int M, int N, int K, int64_t lda, int64_t ldb,
                        int64_t ldc, const float* add, int64_t ld_add, void* workspace, size_t workspace_bytes, hipStream_t st) {
  if (op == ODY_GEMM_NT) return dispatch_f32<true, true>(a, b, c, bias, M, N, K, lda, ldb, ldc, add, ld_add, workspace, workspace_bytes, st);
  if (op == ODY_GEMM_NN) return dispatch_f32<true, false>(a, b, c, bias, M, N, K, lda, ldb, ldc, add, ld_add, workspace, workspace_bytes, st);
  return dispatch_f32<false, false>(a, b, c, bias, M, N, K, lda, ldb, ldc, add, ld_add, workspace, workspace_bytes, st);
}
