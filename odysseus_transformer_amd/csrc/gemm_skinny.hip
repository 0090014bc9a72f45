// Products with few rows, C (M, N) = A (M, K) . W (N, K)^T with M <= 16: a decoding step, or a handful of tokens.
//
// Bound by reading W once (an element of it serves M <= 16 multiply-adds), so the work is split for bytes in flight and
// not for operand reuse: a block owns NT groups of 16 rows of W, its wavefronts each take a share of K, and every wavefront
// loads its W fragments straight from global memory in the operand order of v_mfma_f32_16x16x32_bf16 -- no LDS, no barrier
// until the wavefronts' partial results are summed through LDS at the end.  The rows of A (all blocks read the same ones)
// come from cache; rows beyond M repeat row M - 1 and fall away with their unused result columns.
//
// Measured, weights cold, M = 1 (before: 128 x 128 tiles, one block per 128 columns): 4096 x 4096 68 -> 9.4 us (3.6 TB/s),
// 4096 x 11008 176 -> 22 us (4.1 TB/s), 22016 x 4096 76 -> 40 us (4.5 TB/s), 32000 x 4096 82 -> 54 us (4.9 TB/s; a copy of
// 1 GiB reaches 5.2).
#include "gemm_epi.h"

namespace {

constexpr int SK_WAVES = 8;

// NORM: A is x, and the product that of its RMS-normalised rows.  Every block normalises them for itself, into LDS, with the arithmetic of
// the RMSNorm kernel (another order of the sum), while its first fragments of W are on their way; EPI_ROPE then takes its angles from the positions too.  Weights
// cold, us without the norm / with it, one row: 6144 x 4096 with rotation 13.3 / 15.9, 22016 x 4096 SwiGLU 41.1 / 43.2, 5632 x 1024
// 5.9 / 6.8; four rows 13.6 / 18.1, 43.4 / 47.1, 6.1 / 8.6.  The norm's own launch takes 2.6, the table's 2.0, and each its gap and 5 of host
// work.  (The norm inside the K loop, on every fragment, took 16.2 and 46.6; a ring of fragments refilled one by one instead of a batch
// at a time, without the norm, 14.9 and 41.6.)
template <int NT, int U, int EPI, bool NORM>
__global__ __launch_bounds__(64 * SK_WAVES) void gemm_skinny_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                                    bf16* __restrict__ C, const bf16* __restrict__ bias, int M,
                                                                    int N, int K, int64_t lda, int64_t ldw, int64_t ldc,
                                                                    int accumulate, GemmEpi ep) {
  __shared__ f32x4 red[SK_WAVES][NT][64];
  __shared__ __attribute__((aligned(16))) bf16 angles[NORM && EPI == EPI_ROPE ? ODY_SKINNY_NORM_MAX_M : 1][16][2];
  extern __shared__ __attribute__((aligned(16))) bf16 rows[];   // NORM: [M][K + 8]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, q = lane >> 4;
  // first W row of group t of this block
  int row0[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    if (EPI == EPI_SWIGLU_FWD) row0[t] = 16 * blockIdx.x + t * ep.I;                                   // gate, up
    else if (EPI == EPI_ROPE) row0[t] = 128 * (blockIdx.x >> 2) + 16 * (blockIdx.x & 3) + 64 * t;      // j, j + 64 of a head
    else row0[t] = 16 * (NT * blockIdx.x + t);
  }
  const bf16* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) wp[t] = W + (int64_t)min(row0[t] + c, N - 1) * ldw + 8 * q;
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
#pragma unroll
      for (int d = 32; d > 0; d >>= 1) ss += __shfl_xor(ss, d, 64);
      if (lane == 0) sums[r * SK_WAVES + wave] = ss;
    }
    if (EPI == EPI_ROPE && tid < 16 * M) {   // the angles of this block's columns, one per thread, rounded as the table's
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
  if (tid >= 64 || row >= M) return;
  f32x4 v[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    v[t] = red[0][t][lane];
#pragma unroll
    for (int w = 1; w < SK_WAVES; w++) v[t] += red[w][t][lane];
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

template <int NT, int U, int EPI, bool NORM = false>
int launch(const char* name, int blocks, const bf16* A, const bf16* W, bf16* C, const bf16* bias, int M, int N, int K, int64_t lda,
           int64_t ldw, int64_t ldc, int accumulate, const GemmEpi& ep, hipStream_t st) {
  const size_t smem = NORM ? sizeof(bf16) * M * (K + 8) : 0;
  auto kern = &gemm_skinny_kernel<NT, U, EPI, NORM>;
  if (NORM)
    if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), ODY_SKINNY_NORM_BYTES, name)) return rc;
  ODY_LAUNCH(name, st, kern, dim3(blocks), dim3(64 * SK_WAVES), smem, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep);
  return ody_check_launch(name);
}

}  // namespace

bool ody_gemm_skinny_ok(int epi, int M, int N) {
  // one 16-row operand: with a second one the loads of A weigh as much as those of W, and the tile kernel, which shares both
  // through LDS and cuts K over blocks, is ahead (weights cold, us here / there: 6144 x 4096, M = 8: 17.8 / 17.6, 16: 20.8 / 17.8,
  // 32: 27.5 / 18.7; 4096 x 4096, M = 8: 10.7 / 14.0, 16: 12.2 / 13.9, 32: 15.5 / 14.2; 2048 x 2048, M = 16: 6.7 / 9.3)
  if (M > ODY_SKINNY_MAX_M) return false;
  if (epi == EPI_SWIGLU_FWD) return N % 32 == 0;   // whole groups of 16 gate rows and of 16 up rows
  if (epi == EPI_ROPE) return N % 128 == 0;
  return epi == EPI_NONE || epi == EPI_RESIDUAL;
}

int ody_launch_gemm_skinny(int epi, const bf16* A, const bf16* W, bf16* C, const bf16* bias, int M, int N, int K, int64_t lda,
                           int64_t ldw, int64_t ldc, int accumulate, const GemmEpi& ep, hipStream_t st) {
  const int groups = (N + 15) / 16;
  if (ep.norm) {
    if (epi == EPI_SWIGLU_FWD)
      return launch<2, 8, EPI_SWIGLU_FWD, true>("gemm_skinny_norm_swiglu", groups / 2, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
    return launch<2, 8, EPI_ROPE, true>("gemm_skinny_norm_rope", groups / 2, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  }
  if (epi == EPI_SWIGLU_FWD)
    return launch<2, 8, EPI_SWIGLU_FWD>("gemm_skinny_swiglu", groups / 2, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  if (epi == EPI_ROPE)
    return launch<2, 8, EPI_ROPE>("gemm_skinny_rope", groups / 2, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  const bool wide = groups >= 1024;
  if (epi == EPI_RESIDUAL) {
    if (wide) return launch<2, 8, EPI_RESIDUAL>("gemm_skinny_residual", (groups + 1) / 2, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
    return launch<1, 8, EPI_RESIDUAL>("gemm_skinny_residual", groups, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  }
  if (wide) return launch<2, 8, EPI_NONE>("gemm_skinny", (groups + 1) / 2, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
  return launch<1, 8, EPI_NONE>("gemm_skinny", groups, A, W, C, bias, M, N, K, lda, ldw, ldc, accumulate, ep, st);
}
