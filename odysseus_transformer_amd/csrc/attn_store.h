// How the head_dim-128 backward kernels finish a row of dQ or dK.
#pragma once
#include "attn_params.h"

// dQ^T of one query held by lane group g (accumulator rows 8 (r >> 2) + 4 g + (r & 3) of each 32-wide slice of the
// head dimension) -> row qi of dq: scaled, then added to an fp32 or bf16 destination, rotated back by the rotary
// table, or rounded and stored.
__device__ __forceinline__ void store_dq_row(const AttnParams& p, const f32x16 (&dq)[4], int b, int h, int qi, int g) {
  if (qi >= p.Lq) return;
  if (p.dq_f32) {
    // fp32 destination (the ring step's running dq): exact accumulation over the key blocks, no rounding here
    float* dqp = static_cast<float*>(p.dq) + b * p.sdq.b + h * p.sdq.h + (int64_t)qi * p.sdq.l;
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        f32x4* dst = reinterpret_cast<f32x4*>(dqp + 32 * dt + 8 * a + 4 * g);
        f32x4 w = {0.f, 0.f, 0.f, 0.f};
        if (p.accumulate_dq) w = *dst;
#pragma unroll
        for (int e = 0; e < 4; e++) w[e] += dq[dt][4 * a + e] * p.scale;
        *dst = w;
      }
  } else if (p.rope_q) {
    // the gradient of the un-rotated projection: element d < 64 pairs with d + 64, both in this lane
    bf16* dqp = static_cast<bf16*>(p.dq) + b * p.sdq.b + h * p.sdq.h + (int64_t)qi * p.sdq.l;
    const bf16* trow = p.rope_q + ((int64_t)b * p.Lq + qi) * 128;
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        const bf16x8 cs = *reinterpret_cast<const bf16x8*>(trow + 2 * (32 * dt + 8 * a + 4 * g));
        bf16x4 w1, w2;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float c = (float)cs[2 * e], sn = (float)cs[2 * e + 1];
          const float g1 = dq[dt][4 * a + e] * p.scale, g2 = dq[dt + 2][4 * a + e] * p.scale;
          w1[e] = (bf16)(g1 * c + g2 * sn);
          w2[e] = (bf16)(g2 * c - g1 * sn);
        }
        *reinterpret_cast<bf16x4*>(dqp + 32 * dt + 8 * a + 4 * g) = w1;
        *reinterpret_cast<bf16x4*>(dqp + 32 * (dt + 2) + 8 * a + 4 * g) = w2;
      }
  } else {
    bf16* dqp = static_cast<bf16*>(p.dq) + b * p.sdq.b + h * p.sdq.h + (int64_t)qi * p.sdq.l;
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        bf16x4* dst = reinterpret_cast<bf16x4*>(dqp + 32 * dt + 8 * a + 4 * g);
        bf16x4 w, old = {0, 0, 0, 0};
        if (p.accumulate_dq) old = *dst;
#pragma unroll
        for (int e = 0; e < 4; e++) w[e] = (bf16)(dq[dt][4 * a + e] * p.scale + (float)old[e]);
        *dst = w;
      }
  }
}

// dK^T of one key, held alike -> row `key` of dk: scaled, rotated back by the rotary table, rounded and stored.
__device__ __forceinline__ void store_dk_row(const AttnParams& p, const f32x16 (&dk)[4], int b, int hk, int key, int g) {
  bf16* dkp = static_cast<bf16*>(p.dk) + b * p.sdk.b + hk * p.sdk.h + (int64_t)key * p.sdk.l;
  if (p.rope_k) {   // dK of the un-rotated projection: element d < 64 pairs with d + 64, both in this lane
    const bf16* trow = p.rope_k + ((int64_t)b * p.Lk + key) * 128;
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        const bf16x8 cs = *reinterpret_cast<const bf16x8*>(trow + 2 * (32 * dt + 8 * a + 4 * g));
        bf16x4 w1, w2;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float c = (float)cs[2 * e], sn = (float)cs[2 * e + 1];
          const float g1 = dk[dt][4 * a + e] * p.scale, g2 = dk[dt + 2][4 * a + e] * p.scale;
          w1[e] = (bf16)(g1 * c + g2 * sn);
          w2[e] = (bf16)(g2 * c - g1 * sn);
        }
        *reinterpret_cast<bf16x4*>(dkp + 32 * dt + 8 * a + 4 * g) = w1;
        *reinterpret_cast<bf16x4*>(dkp + 32 * (dt + 2) + 8 * a + 4 * g) = w2;
      }
  } else {
#pragma unroll
    for (int dt = 0; dt < 4; dt++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        bf16x4 wk;
#pragma unroll
        for (int e = 0; e < 4; e++) wk[e] = (bf16)(dk[dt][4 * a + e] * p.scale);
        *reinterpret_cast<bf16x4*>(dkp + 32 * dt + 8 * a + 4 * g) = wk;
      }
  }
}
