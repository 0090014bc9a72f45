// Products with few rows, C (M, N) = A (M, K) . W (N, K)^T with M <= 16: a decoding step, or a handful of tokens.
//
// Bound by reading W once (an element of it serves M <= 16 multiply-adds), so the work is split for bytes in flight and
// not for operand reuse: a block owns NT groups of 16 rows of W, its wavefronts each take a share of K, and every wavefront
// loads its W fragments straight from global memory in the operand order of v_mfma_f32_16x16x32_bf16 -- no LDS, no barrier
// until the wavefronts' partial results are summed through LDS at the end.  The rows of A (all blocks read the same ones)
// come from cache; rows beyond M repeat row M - 1 and fall away with their unused result columns.
//
// Measured, weights cold, M = 1, us (TB/s): 4096 x 4096 8.0 (4.2), 4096 x 11008 19.3 (4.7), 32000 x 4096 45.3 (5.8), with the norm in front 22016 x 4096 33.0 (5.5),
// 6144 x 4096 13.0 (3.9), 5632 x 1024 5.2; of each about 1.7 between two launches and 1.2 until the first bytes arrive.  A unit takes some 64 KB of loads at a
// time and no more (deeper rings of loads to LDS, 96 KB a unit, changed nothing but the time at which what is behind them is issued), so what counts is
// that blocks are many and even: with two groups of 16 rows and 8 wavefronts a block everywhere, 22016 x 4096 ran 512 blocks in 20 us and the
// remaining 176 in 18, together 39.0 with the norm; the others 9.0, 20.5, 50.5, 16.0 and 6.4.
#include <type_traits>
#include "gemm_epi.h"

namespace {

#define FENCE() __builtin_amdgcn_sched_barrier(0)

// Sum over the lanes of a wavefront, by the tree of xor 1, 2, 4 .. 32 (within groups of equal values a mirrored lane is as good as an exchanged one)
__device__ __forceinline__ float wave_sum(float x) {
  auto dpp = [](float v, auto ctrl) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf, true)); };
  x += dpp(x, std::integral_constant<int, 0xb1>{});    // quad_perm [1, 0, 3, 2]
  x += dpp(x, std::integral_constant<int, 0x4e>{});    // quad_perm [2, 3, 0, 1]
  x += dpp(x, std::integral_constant<int, 0x141>{});   // row_half_mirror
  x += dpp(x, std::integral_constant<int, 0x140>{});   // row_mirror
  x += __shfl_xor(x, 16, 64);
  x += __shfl_xor(x, 32, 64);
  return x;
}

// NT groups a block, U steps of 32 k in flight per wavefront and group, and SK_WAVES wavefronts (ody_launch_gemm_skinny).
// NORM: A is x, and the product that of its RMS-normalised rows.  Every block normalises them for itself, into LDS, with the arithmetic of
// the RMSNorm kernel (another order of the sum), while its first fragments of W are on their way; EPI_ROPE then takes its angles from the positions too.  Weights
// cold, us without the norm / with it, one row: 6144 x 4096 with rotation 12.6 / 13.0, 22016 x 4096 SwiGLU 34.6 / 33.0 (the rows are read from LDS there), 5632 x 1024 5.6 / 5.2.  The norm's own launch takes 2.6, the
// table's 2.0, and each its gap and 5 of host work.  (The norm inside the K loop, on every fragment, took 0.3 and 3.4 us longer.)
// BATCH: all loads of a batch in front of its first product.  Left to the compiler, most of a later batch went out one or two loads at a time (NORM: 39 us for 33);
// where A's rows are many and blocks too, its order is the better one (22016 x 4096, M = 8: 41.4 / 38.4, but 6144 x 4096 13.8 / 17.4).
template <int NT, int U, int SK_WAVES, int EPI, bool NORM, bool BATCH>
__global__ __launch_bounds__(64 * SK_WAVES) void gemm_skinny_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                                    bf16* __restrict__ C, const bf16* __restrict__ bias, int M,
                                                                    int N, int K, int64_t lda, int64_t ldw, int64_t ldc,
                                                                    int accumulate, GemmEpi ep) {
  __shared__ f32x4 red[SK_WAVES][NT][64];
  __shared__ __attribute__((aligned(16))) bf16 angles[NORM && EPI == EPI_ROPE ? ODY_SKINNY_NORM_MAX_M : 1][16][2];
  extern __shared__ __attribute__((aligned(16))) bf16 rows[];   // NORM: [M][K + 8]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, q = lane >> 4;
  // a group of 16 rows of W: sixteen in a row, or, PAIRED, eight and their eight partners
  constexpr bool TWO = EPI == EPI_SWIGLU_FWD || EPI == EPI_ROPE, PAIRED = TWO && NT == 1;
  // first W row of group t of this block
  int row0[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    if (PAIRED) row0[t] = EPI == EPI_SWIGLU_FWD ? 8 * blockIdx.x : 128 * (blockIdx.x >> 3) + 8 * (blockIdx.x & 7);
    else if (EPI == EPI_SWIGLU_FWD) row0[t] = 16 * blockIdx.x + t * ep.I;                              // gate, up
    else if (EPI == EPI_ROPE) row0[t] = 128 * (blockIdx.x >> 2) + 16 * (blockIdx.x & 3) + 64 * t;      // j, j + 64 of a head
    else row0[t] = 16 * (NT * blockIdx.x + t);
  }
  const bf16* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) wp[t] = W + (int64_t)(PAIRED ? row0[t] + (c & 7) + (c >> 3) * (EPI == EPI_ROPE ? 64 : ep.I) : min(row0[t] + c, N - 1)) * ldw + 8 * q;
  const bf16* ap = (NORM ? rows + min(c, M - 1) * (K + 8) : A + (int64_t)min(c, M - 1) * lda) + 8 * q;

  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int steps = (K + 31) / 32, per = (steps + SK_WAVES - 1) / SK_WAVES;
  const int s0 = wave * per, s1 = min(s0 + per, steps);
  bf16x8 wf[U][NT], af[U];
  auto multiply = [&]() {
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int t = 0; t < NT; t++)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][t], af[u], acc[t], 0, 0, 0);   // rows = n, columns = m
  };
  int s = s0;
  const int whole = K / 32;   // steps that lie inside K for every lane
  const int s_whole = min(s1, whole);
  bool fetched = false;       // NORM: the first W fragments
  if constexpr (NORM) {
    fetched = s + U <= s_whole;
    float* sums = reinterpret_cast<float*>(red);   // [M][SK_WAVES]
    const int nvec = K / 8;
    bf16x8 first = bf16x8{0, 0, 0, 0, 0, 0, 0, 0}, scale = first;
    if (tid < nvec) first = *reinterpret_cast<const bf16x8*>(A + 8 * tid), scale = *reinterpret_cast<const bf16x8*>(ep.norm + 8 * tid);
    if (fetched) {
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int t = 0; t < NT; t++) wf[u][t] = *reinterpret_cast<const bf16x8*>(wp[t] + (int64_t)(s + u) * 32);
    }
    auto vector_of = [&](int r, int v) { return r == 0 && v == tid ? first : *reinterpret_cast<const bf16x8*>(A + (int64_t)r * lda + 8 * v); };
    for (int r = 0; r < M; r++) {
      float ss = 0.f;
      for (int v = tid; v < nvec; v += 64 * SK_WAVES) {
        const bf16x8 x = vector_of(r, v);
#pragma unroll
        for (int e = 0; e < 8; e++) ss = fmaf((float)x[e], (float)x[e], ss);
      }
      ss = wave_sum(ss);
      if (lane == 0) sums[r * SK_WAVES + wave] = ss;
    }
    if (EPI == EPI_ROPE && tid < 16 * M && (tid & 15) < (PAIRED ? 8 : 16)) {   // the angles of this block's columns, one per thread, rounded as the table's
      const float th = (float)ep.positions[tid >> 4] * ep.inv_freq[(row0[0] & 127) + (tid & 15)];
      angles[tid >> 4][tid & 15][0] = (bf16)cosf(th), angles[tid >> 4][tid & 15][1] = (bf16)sinf(th);
    }
    __syncthreads();
    for (int r = 0; r < M; r++) {
      float ss = 0.f;
#pragma unroll
      for (int w = 0; w < SK_WAVES; w++) ss += sums[r * SK_WAVES + w];
      const float rstd = rsqrtf(ss / (float)K + ep.eps);
      for (int v = tid; v < nvec; v += 64 * SK_WAVES) {
        const bf16x8 x = vector_of(r, v), n = v == tid ? scale : *reinterpret_cast<const bf16x8*>(ep.norm + 8 * v);
        bf16x8 y;
#pragma unroll
        for (int e = 0; e < 8; e++) y[e] = (bf16)((float)n[e] * (float)(bf16)((float)x[e] * rstd));
        *reinterpret_cast<bf16x8*>(rows + r * (K + 8) + 8 * v) = y;
      }
    }
    __syncthreads();
  }
  for (; s + U <= s_whole; s += U) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (!NORM || !fetched) {
#pragma unroll
        for (int t = 0; t < NT; t++) wf[u][t] = *reinterpret_cast<const bf16x8*>(wp[t] + (int64_t)(s + u) * 32);
      }
      af[u] = *reinterpret_cast<const bf16x8*>(ap + (int64_t)(s + u) * 32);
    }
    fetched = false;
    if (BATCH) FENCE();
    multiply();
  }
  if (s < s1) {   // the remainder, all of it in flight at once
    const bf16x8 zero = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < U; u++) {
      const bool in = s + u < s1 && (s + u) * 32 + 8 * q < K;   // K is a multiple of 8: a chunk is all in or out
#pragma unroll
      for (int t = 0; t < NT; t++) wf[u][t] = in ? *reinterpret_cast<const bf16x8*>(wp[t] + (int64_t)(s + u) * 32) : zero;
      af[u] = in ? *reinterpret_cast<const bf16x8*>(ap + (int64_t)(s + u) * 32) : zero;
    }
    multiply();
  }

#pragma unroll
  for (int t = 0; t < NT; t++) red[wave][t][lane] = acc[t];
  __syncthreads();
  // lane 16 q + c of the first wavefront owns row c of A and columns 4 q .. 4 q + 3 of every group of W rows
  const int row = c;
  if (tid >= 64 || row >= M || (PAIRED && q >= 2)) return;
  constexpr int NV = PAIRED ? 2 : NT;   // PAIRED: the partners' columns lie 32 lanes on
  f32x4 v[NV];
#pragma unroll
  for (int t = 0; t < NV; t++) {
    auto part = [&](int w) { return PAIRED ? red[w][0][lane + 32 * t] : red[w][t][lane]; };
    v[t] = part(0);
#pragma unroll
    for (int w = 1; w < SK_WAVES; w++) v[t] += part(w);
  }
  auto rounded = [](f32x4 x) {
    bf16x4 w;
#pragma unroll
    for (int e = 0; e < 4; e++) w[e] = (bf16)x[e];
    return w;
  };
  bf16* cp = C + (int64_t)row * ldc;
  if constexpr (EPI == EPI_SWIGLU_FWD) {
    const int n = row0[0] + 4 * q;
    if (n >= ep.I) return;
    const bf16x4 g4 = rounded(v[0]), u4 = rounded(v[1]);
    bf16x4 h4;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float a1 = (float)g4[e], a3 = (float)u4[e];
      h4[e] = (bf16)(a1 / (1.f + __expf(-a1)) * a3);
    }
    if (C) {   // NULL: only h is wanted
      *reinterpret_cast<bf16x4*>(cp + n) = g4;
      *reinterpret_cast<bf16x4*>(cp + ep.I + n) = u4;
    }
    *reinterpret_cast<bf16x4*>(ep.out2 + (int64_t)row * ep.ld_out2 + n) = h4;
  } else if constexpr (EPI == EPI_ROPE) {
    const int n = row0[0] + 4 * q, j = n & 127;
    f32x4 o1 = v[0], o2 = v[1];
    if (n < ep.I) {
      const bf16x8 cs = *reinterpret_cast<const bf16x8*>(NORM ? angles[row][4 * q] : ep.aux + (int64_t)row * ep.ld_aux + 2 * j);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float co = (float)cs[2 * e], sn = (float)cs[2 * e + 1];
        o1[e] = v[0][e] * co - v[1][e] * sn;
        o2[e] = v[1][e] * co + v[0][e] * sn;
      }
    }
    *reinterpret_cast<bf16x4*>(cp + n) = rounded(o1);
    *reinterpret_cast<bf16x4*>(cp + n + 64) = rounded(o2);
  } else {
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const int n = row0[t] + 4 * q;
      if (n >= N) continue;   // N % 8 == 0: four columns are all in or out
      if constexpr (EPI == EPI_RESIDUAL) {
        const bf16x4 r = *reinterpret_cast<const bf16x4*>(ep.aux + (int64_t)row * ep.ld_aux + n);
#pragma unroll
        for (int e = 0; e < 4; e++) v[t][e] += (float)r[e];
      } else {
        if (bias) {
          const bf16x4 b = *reinterpret_cast<const bf16x4*>(bias + n);
#pragma unroll
          for (int e = 0; e < 4; e++) v[t][e] += (float)b[e];
        }
        if (accumulate) {
          const bf16x4 o = *reinterpret_cast<const bf16x4*>(cp + n);
#pragma unroll
          for (int e = 0; e < 4; e++) v[t][e] += (float)o[e];
        }
      }
      *reinterpret_cast<bf16x4*>(cp + n) = rounded(v[t]);
    }
  }
}

template <int NT, int U, int SK_WAVES, int EPI, bool NORM = false, bool BATCH = true>
int launch(const char* name, const bf16* A, const bf16* W, bf16* C, const bf16* bias, int M, int N, int K, int64_t lda,
           int64_t ldw, int64_t ldc, int accumulate, const GemmEpi& ep, hipStream_t st) {
  const size_t smem = NORM ? sizeof(bf16) * M * (K + 8) : 0;
  auto kern = &gemm_skinny_kernel<NT, U, SK_WAVES, EPI, NORM, BATCH>;
  if (NORM)
    if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), ODY_SKINNY_NORM_BYTES, name)) return rc;
  ODY_LAUNCH(name, st, kern, dim3(((N + 15) / 16 + NT - 1) / NT), dim3(64 * SK_WAVES), smem, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep);
  return ody_check_launch(name);
}

// What a block takes.  us; weights cold unless "warm" (a matrix that the last-level cache holds, again and again).
//   M <= 4: one group of 16 rows, 8 wavefronts: 4096 x 4096 8.0 (8.9 otherwise), 2048 x 5632 9.0 / 9.7, with the norm 22016 x 4096 33.0 / 33.1.  Beyond 512 groups 4
//   wavefronts with twice the loads: 13312 x 2816, M = 4, 18.6 / 21.0, 32000 x 4096 45.3 / 44.8 and 46.8; where rows are long, too, but not with one row of A:
//   4096 x 11008, M = 4, 19.9 / 20.9 and 21.3, M = 1 19.3 / 19.3, 4096 x 14336, M = 1, 22.1 / 22.8.  (Warm, two
//   groups on 8 wavefronts would be ahead from three rows on: 32000 x 2048, M = 4, 22.9 / 21.7, 65536 x 1536 32.9 / 30.1, cold 27.3 / 28.0 and 39.7 / 42.3.)
//   M > 4: a group's fragments of A weigh as much as those of W.  Two groups share them where such blocks fill their last round of units, to 512 groups and from 800 on:
//   22016 x 4096, M = 8, 38.4 / 40.6, 6144 x 4096, M = 16, 15.2 / 15.9, 4608 x 3072, rotated, M = 16, 12.3 / 15.2 (one group); between the two, 1.1 to 1.5 rounds, they do not:
//   9216 x 2816, M = 5, 18.5, one group 14.5, 12288 x 4096, M = 5, 24.6 / 20.6.  Rows of 1792 to 2048 are two batches for each of 8 wavefronts, four for 4;
//   with 5 to 12 rows of A, 8 / 4 wavefronts: 50264 x 2048, M = 5, 43.1 / 45.2, M = 12 48.2 / 49.6, 32000 x 2048, M = 5, 27.1 / 29.2, M = 12 30.3 / 29.9, 32000 x 1920, M = 5, 25.2 / 29.8,
//   warm 16384 x 2048, M = 9, 12.6 / 13.7; beyond, 32000 x 1792, M = 5, 26.0 / 24.5, warm 32000 x 2176 24.0 / 23.0, 40960 x 2048, M = 16, 40.5 / 39.1.  Otherwise one group: 4096 x 11008, M = 8, 21.0 / 22.5, 3072 x 2048 6.0 / 7.7; 8 wavefronts
//   where groups are no more than units and K is short: 4096 x 4096, M = 5, 8.6 / 9.1, warm 7.2 / 7.5, or two batches for either, 2048 x 2048, M = 12, 6.1 / 6.3.
//   Pairs of rows (rotation, SwiGLU) with 257 to 512 groups: blocks of two whole groups are one for a unit, those of half and half up to two, and the second one's start shows.
//   Two / half and half: rotated, 6144 x 2048, M = 1, 7.3 / 8.2, M = 8 8.0 / 9.6, M = 12 8.4 / 9.2, 5120 x 4096, M = 1, 12.1 / 13.3; SwiGLU, 5632 x 1024, M = 6, warm, 4.6 / 4.9
//   (cold, M = 5, 5.8 / 5.6).  Beyond 448 groups of long rows they do not show it, 8192 x 4096, M = 1, 15.1 / 14.3, nor where more rows of A have 4 wavefronts, 6144 x 4096, M = 8,
//   13.6 / 13.6, SwiGLU, M = 16, 16.0 / 15.0.
template <int EPI>
int launch_for(const char* name, const bf16* A, const bf16* W, bf16* C, const bf16* bias, int M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc,
               int accumulate, const GemmEpi& ep, hipStream_t st) {
  const int groups = (N + 15) / 16;
  const bool one_each = groups > 256 && groups <= 512;   // of blocks of two groups, for a unit
  if constexpr (EPI == EPI_SWIGLU_FWD || EPI == EPI_ROPE)
    if (one_each && (K > 2048 ? M <= 4 && groups <= 448 : M <= 8 || EPI == EPI_ROPE))
      return launch<2, 8, 8, EPI, false, false>(name, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  if (M > 4 && M <= 12 && groups >= 1024 && K > 1792 && K <= 2048)
    return launch<2, 4, 8, EPI, false, false>(name, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  if (M > 4 && groups >= 1024) return launch<2, 4, 4, EPI, false, false>(name, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  if (M > 4 && (one_each || groups >= 800) && (K > 2048 || M > 8)) return launch<2, 4, 4, EPI>(name, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  const bool long_rows = M > 8 ? K > 2048 || K <= 1024 : K > 4096 && M > 4;
  if (M > 4 ? groups > 256 || long_rows : groups > 512 || (groups >= 256 && K > 4096 && M > 1))
    return launch<1, 8, 4, EPI>(name, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  return launch<1, 4, 8, EPI>(name, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
}

}  // namespace

bool ody_gemm_skinny_ok(int epi, int M, int N) {
  // One 16-row operand, up to which this is the faster one but for the longest rows (weights cold, us, M = 8 and 16 here / M = 17 in the tile kernel, which shares
  // both operands through LDS and cuts K over blocks: 6144 x 4096 13.7, 15.1 / 16.6; 4096 x 4096 9.4, 10.5 / 12.8; 2048 x 2048 5.6, 6.6 / 9.3; 22016 x 4096 37.9, 43.4 /
  // 48.6; 32000 x 4096 52.3, 59.4 / 64.7; 4096 x 11008 20.8, 24.4 / 24.1).  A second operand was tried with instances slower than these, 6144 x 4096, M = 32, 27.5 / 18.7; with
  // one the time of M = 8 grows by 8 to 18 % to M = 16, and by more for the loads of a second set of rows.
  if (M > ODY_SKINNY_MAX_M) return false;
  if (epi == EPI_SWIGLU_FWD) return N % 32 == 0;   // whole groups of 16 gate rows and of 16 up rows
  if (epi == EPI_ROPE) return N % 128 == 0;
  return epi == EPI_NONE || epi == EPI_RESIDUAL;
}

int ody_launch_gemm_skinny(int epi, const bf16* A, const bf16* W, bf16* C, const bf16* bias, int M, int N, int K, int64_t lda,
                           int64_t ldw, int64_t ldc, int accumulate, const GemmEpi& ep, hipStream_t st) {
  if (ep.norm) {
    if (epi == EPI_SWIGLU_FWD)
      return launch<1, 4, 8, EPI_SWIGLU_FWD, true>("gemm_skinny_norm_swiglu", A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
    return launch<1, 4, 8, EPI_ROPE, true>("gemm_skinny_norm_rope", A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  }
  if (epi == EPI_SWIGLU_FWD) return launch_for<EPI_SWIGLU_FWD>("gemm_skinny_swiglu", A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  if (epi == EPI_ROPE) return launch_for<EPI_ROPE>("gemm_skinny_rope", A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  if (epi == EPI_RESIDUAL) return launch_for<EPI_RESIDUAL>("gemm_skinny_residual", A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  return launch_for<EPI_NONE>("gemm_skinny", A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
}
