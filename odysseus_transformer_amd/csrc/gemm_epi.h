// What the epilogue of a bf16 product does besides rounding and storing.
//   EPI_RESIDUAL    C = A B + R                      (R = aux, row pitch ld_aux; one rounding, after the add)
//   EPI_SWIGLU_FWD  NT only.  B is the packed (2 I, K) gate_up weight.  Writes gate_up to C in its usual [gate | up] layout (C NULL:
//                   not at all) and h = silu(gate) * up to out2, computed from the rounded gate / up values exactly as the stand-alone SwiGLU
//                   kernel would.
//   EPI_ROPE        NT only, head_dim 128.  Columns below I (a multiple of 128) are rotated before the one rounding: with the
//                   cos / sin table of ody_rope_table in aux (row pitch ld_aux), column j < 64 of a head pairs with column j + 64
//   EPI_SWIGLU_BWD  the result is dh = dy Wd (N = I); with gate_up = aux the epilogue writes d_gate_up to C (pitch ldc, 2 I
//                   columns) as the stand-alone SwiGLU backward would from the rounded dh.
#pragma once
#include "ody_common.h"

enum { EPI_NONE = 0, EPI_RESIDUAL = 1, EPI_SWIGLU_FWD = 2, EPI_SWIGLU_BWD = 3, EPI_ROPE = 4 };
struct GemmEpi {
  const bf16* aux;
  bf16* out2;
  int64_t ld_aux, ld_out2;
  int I;
  // few rows only (gemm_skinny.hip): A is x, and the product that of its RMS-normalised rows (weight `norm` of K elements, or NULL);
  // EPI_ROPE takes its angles from positions[row] * inv_freq[j], rounded as ody_rope_table rounds them, where there is no table
  const bf16* norm;
  float eps;
  const int64_t* positions;
  const float* inv_freq;
};

// C (M, N) = A (M, K) . W (N, K)^T for few rows of A (gemm_skinny.hip); EPI_NONE also takes a bias and accumulation into C.
constexpr int ODY_SKINNY_MAX_M = 16;
// The norm in front of a product of few rows (GemmEpi::norm): every block normalises them for itself, so only where that is quicker than
// a launch of its own, and where the rows, 2 M (K + 8) bytes, fit the LDS.
constexpr int ODY_SKINNY_NORM_MAX_M = 4;
constexpr size_t ODY_SKINNY_NORM_BYTES = 64 << 10;
bool ody_gemm_skinny_ok(int epi, int M, int N);
int ody_launch_gemm_skinny(int epi, const bf16* A, const bf16* W, bf16* C, const bf16* bias, int M, int N, int K, int64_t lda,
                           int64_t ldw, int64_t ldc, int accumulate, const GemmEpi& ep, hipStream_t st);

// fp32 products (gemm_f32.hip), any shape and alignment; `add` may be C itself
size_t ody_gemm_f32_workspace(int M, int N, int K);
int ody_launch_gemm_f32(int op, const float* A, const float* B, float* C, const float* bias, int M, int N, int K, int64_t lda, int64_t ldb,
                        int64_t ldc, const float* add, int64_t ld_add, void* workspace, size_t workspace_bytes, hipStream_t st);
