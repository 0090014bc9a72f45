// Flash-attention forward for few queries against many keys, bf16: a decoding step or a short chunk behind a cache.
//
// Bound by reading K and V once.  The rows of a block are ALL queries of ONE kv head -- the `group` query heads that share it
// times the Lq tokens, at most 64 -- so that no key is read twice, and the keys are cut into ranges (flash decoding): one
// 256-thread block per (batch, kv head, range), enough of them for two per compute unit.  Inside a block the four wavefronts
// take 32-key tiles in turn and keep their own running softmax; nothing is shared, so the loop has no barrier:
//
//      S^T = K Q^T          A: K rows, straight from global memory in operand order   B: Q^T (registers)
//      O^T += V^T P^T       A: V^T by transposing LDS reads of the wavefront's own tile   B: P^T = accumulator layout of S^T
//
// on v_mfma_f32_16x16x32_bf16 (lane = 16 q + c: A row c / B column c, k = 8 q .. 8 q + 7; accumulator column c, rows
// 4 q .. 4 q + 3).  The wavefronts' results are combined through LDS, the ranges by a second, small kernel with the
// arithmetic of the ring's block merge.
#include "attn_params.h"

namespace {

constexpr int DC_WAVES = 4, DC_TILE = 32, DC_BLOCK_KEYS = DC_WAVES * DC_TILE;
constexpr int DC_MAX_TOKENS = 32, DC_MAX_ROWS = 64, DC_MAX_SPLITS = 64;

// part_out [split][B][Lq][Hq][D], part_lse [split][B][Hq][Lq] (nsplit > 1)
template <int D, int MT>
__global__ __launch_bounds__(64 * DC_WAVES) void attn_decode_kernel(const AttnParams p, int nsplit, int keys_per_split,
                                                                    float* __restrict__ part_out, float* __restrict__ part_lse) {
  constexpr int KS = D / 32, DT = D / 16, VP = D + 16;   // V pitch: 16 rows of a transposing read hit every bank twice, the least possible
  constexpr int CPR = D / 8, RPL = 64 / CPR, VL = DC_TILE / RPL;   // 16-byte chunks per row, rows per load instruction, loads per tile
  constexpr int OP = D + 4;
  constexpr int VBYTES = DC_WAVES * DC_TILE * VP * 2, OBYTES = DC_WAVES * 16 * OP * 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[VBYTES > OBYTES ? VBYTES : OBYTES];
  __shared__ float sm[DC_WAVES][16 * MT], sl[DC_WAVES][16 * MT];

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int split = blockIdx.x % nsplit, bh = blockIdx.x / nsplit, hk = bh % p.Hkv, b = bh / p.Hkv;
  const int rows = p.group * p.Lq;
  const bf16* kp = static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const bf16* vp = static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h;
  bf16* Vs = reinterpret_cast<bf16*>(smem) + wave * DC_TILE * VP;

  // row r of the block: token r / group, query head hk * group + r % group
  bf16x8 qf[MT][KS];
  int lim[MT];      // last key the row sees
#pragma unroll
  for (int m = 0; m < MT; m++) {
    const int r = min(16 * m + c, rows - 1), qi = r / p.group, h = hk * p.group + r % p.group;
    const bf16* qp = static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h + (int64_t)qi * p.sq.l;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qf[m][ks] = *reinterpret_cast<const bf16x8*>(qp + 32 * ks + 8 * q);
    lim[m] = p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1;
  }
  f32x4 o[MT][DT];
  float mx[MT], l[MT];
#pragma unroll
  for (int m = 0; m < MT; m++) {
    mx[m] = -INFINITY, l[m] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[m][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float c2 = p.scale_log2e;
  const int k_first = split * keys_per_split, k_end = min(p.Lk, k_first + keys_per_split);
  const int safe = p.causal ? min(p.Lk - 1, p.off) : p.Lk - 1;   // keys up to here are seen by every row

  for (int k0 = k_first + wave * DC_TILE; k0 < k_end; k0 += DC_BLOCK_KEYS) {
    bf16x8 kf[2][KS], vr[VL];
#pragma unroll
    for (int st = 0; st < 2; st++) {
      const bf16* src = kp + (int64_t)min(k0 + 16 * st + c, p.Lk - 1) * p.sk.l + 8 * q;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) kf[st][ks] = *reinterpret_cast<const bf16x8*>(src + 32 * ks);
    }
#pragma unroll
    for (int j = 0; j < VL; j++)
      vr[j] = *reinterpret_cast<const bf16x8*>(vp + (int64_t)min(k0 + RPL * j + lane / CPR, p.Lk - 1) * p.sv.l + 8 * (lane % CPR));
    f32x4 s[MT][2];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
      for (int st = 0; st < 2; st++) {
        s[m][st] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ks++) s[m][st] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[st][ks], qf[m][ks], s[m][st], 0, 0, 0);
      }
    wavefront_sync();   // the tile before has been read
#pragma unroll
    for (int j = 0; j < VL; j++) *reinterpret_cast<bf16x8*>(Vs + (RPL * j + lane / CPR) * VP + 8 * (lane % CPR)) = vr[j];
    // keys of a lane: k0 + 16 st + 4 q + r
    const int last = min(k0 + DC_TILE, k_end) - 1;
    const bool mask = last > safe || last < k0 + DC_TILE - 1;
    bf16x8 pb[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
      if (mask) {
#pragma unroll
        for (int st = 0; st < 2; st++)
#pragma unroll
          for (int r = 0; r < 4; r++)
            if (k0 + 16 * st + 4 * q + r > min(lim[m], last)) s[m][st][r] = -INFINITY;
      }
      float t = fmaxf(fmaxf(fmaxf(s[m][0][0], s[m][0][1]), fmaxf(s[m][0][2], s[m][0][3])),
                      fmaxf(fmaxf(s[m][1][0], s[m][1][1]), fmaxf(s[m][1][2], s[m][1][3])));
      t = fmaxf(t, __shfl_xor(t, 16, 64));
      t = fmaxf(t, __shfl_xor(t, 32, 64));
      const float mn = fmaxf(mx[m], t), mu = mn == -INFINITY ? 0.f : mn;
      const float alpha = ody_exp2((mx[m] - mu) * c2);
      mx[m] = mn;
      float sum = 0.f;
#pragma unroll
      for (int st = 0; st < 2; st++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float e = ody_exp2(fmaf(s[m][st][r], c2, -mu * c2));
          sum += e;
          pb[m][4 * st + r] = (bf16)e;
        }
      l[m] = l[m] * alpha + sum;     // this lane's share of the row sum
#pragma unroll
      for (int dt = 0; dt < DT; dt++) o[m][dt] *= alpha;
    }
    // contraction index 8 q + j <-> key 16 (j >> 2) + 4 q + (j & 3)
    wavefront_sync();
    const bf16* vt = Vs + (4 * q + (c >> 2)) * VP + 4 * (c & 3);
#pragma unroll
    for (int dt = 0; dt < DT; dt++) {
      const bf16x8 a = concat4(lds_read_tr16(vt + 16 * dt), lds_read_tr16(vt + 16 * VP + 16 * dt));
#pragma unroll
      for (int m = 0; m < MT; m++) o[m][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[m], o[m][dt], 0, 0, 0);
    }
  }

  // ---- the four wavefronts' results of a row: common reference, weighted sum
#pragma unroll
  for (int m = 0; m < MT; m++) {
    l[m] += __shfl_xor(l[m], 16, 64);
    l[m] += __shfl_xor(l[m], 32, 64);
    if (q == 0) sm[wave][16 * m + c] = mx[m], sl[wave][16 * m + c] = l[m];
  }
  __syncthreads();
  float* Os = reinterpret_cast<float*>(smem);   // [wave][16][OP]
#pragma unroll
  for (int m = 0; m < MT; m++) {
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < DC_WAVES; w++) top = fmaxf(top, sm[w][16 * m + c]);
    const float ref = top == -INFINITY ? 0.f : top, mine = ody_exp2((mx[m] - ref) * c2);
#pragma unroll
    for (int dt = 0; dt < DT; dt++) *reinterpret_cast<f32x4*>(Os + (wave * 16 + c) * OP + 16 * dt + 4 * q) = o[m][dt] * mine;
    __syncthreads();
    // 16 rows x D / 4 vectors over the threads
#pragma unroll
    for (int e = 0; e < 16 * D / 4 / (64 * DC_WAVES); e++) {
      const int idx = tid + 64 * DC_WAVES * e, row = idx / (D / 4), d4 = idx % (D / 4), r = 16 * m + row;
      if (r < rows) {
        float t = -INFINITY, sum = 0.f;
#pragma unroll
        for (int w = 0; w < DC_WAVES; w++) t = fmaxf(t, sm[w][r]);
        const float tu = t == -INFINITY ? 0.f : t;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < DC_WAVES; w++) {
          sum += sl[w][r] * ody_exp2((sm[w][r] - tu) * c2);
          acc += *reinterpret_cast<const f32x4*>(Os + (w * 16 + row) * OP + 4 * d4);
        }
        acc *= sum > 0.f ? 1.f / sum : 0.f;
        const float lse = sum > 0.f ? (tu * c2 + __log2f(sum)) * ODY_LN2 : -INFINITY;
        const int qi = r / p.group, h = hk * p.group + r % p.group;
        if (nsplit > 1) {
          *reinterpret_cast<f32x4*>(part_out + ((((int64_t)split * p.B + b) * p.Lq + qi) * p.Hq + h) * D + 4 * d4) = acc;
          if (d4 == 0) part_lse[(((int64_t)split * p.B + b) * p.Hq + h) * p.Lq + qi] = lse;
        } else {
          bf16x4 w4;
#pragma unroll
          for (int k = 0; k < 4; k++) w4[k] = (bf16)acc[k];
          *reinterpret_cast<bf16x4*>(static_cast<bf16*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)qi * p.so.l + 4 * d4) = w4;
          if (d4 == 0) p.lse[((int64_t)b * p.Hq + h) * p.Lq + qi] = lse;
        }
      }
    }
    __syncthreads();
  }
}

// One block per (batch, query, head): the weights of its parts by one wavefront, then 256 / (D / 4) threads per column
// vector share the parts.
template <int D>
__global__ __launch_bounds__(256) void attn_decode_merge_kernel(const AttnParams p, int nsplit, const float* __restrict__ part_out,
                                                                const float* __restrict__ part_lse) {
  constexpr int C4 = D / 4, G = 256 / C4;
  __shared__ float w[DC_MAX_SPLITS];
  __shared__ f32x4 red[G][C4];
  const int tid = threadIdx.x, h = blockIdx.x % p.Hq, qi = (blockIdx.x / p.Hq) % p.Lq, b = blockIdx.x / (p.Hq * p.Lq);
  const int64_t plane_o = (int64_t)p.B * p.Lq * p.Hq * D, plane_l = (int64_t)p.B * p.Hq * p.Lq;
  const int64_t li = ((int64_t)b * p.Hq + h) * p.Lq + qi;
  if (tid < 64) {
    const float x = tid < nsplit ? part_lse[tid * plane_l + li] : -INFINITY;
    float m = x;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) m = fmaxf(m, __shfl_xor(m, s, 64));
    const float e = m == -INFINITY ? 0.f : __expf(x - m);
    float sum = e;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) sum += __shfl_xor(sum, s, 64);
    w[tid] = sum > 0.f ? e / sum : 0.f;
    if (tid == 0) p.lse[li] = sum > 0.f ? m + __logf(sum) : -INFINITY;
  }
  __syncthreads();
  const int d4 = tid % C4, g = tid / C4;
  const float* src = part_out + (((int64_t)b * p.Lq + qi) * p.Hq + h) * D + 4 * d4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = g; s < nsplit; s += G) acc += w[s] * *reinterpret_cast<const f32x4*>(src + s * plane_o);
  red[g][d4] = acc;
  __syncthreads();
  if (g == 0) {
#pragma unroll
    for (int k = 1; k < G; k++) acc += red[k][d4];
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = (bf16)acc[e];
    *reinterpret_cast<bf16x4*>(static_cast<bf16*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)qi * p.so.l + 4 * d4) = o;
  }
}

// Ranges of the keys: two blocks per compute unit, whole turns of the four wavefronts each, at most 64.
struct Ranges { int n, keys; };
Ranges ranges(int B, int Lk, int Hkv) {
  const int turns = (Lk + DC_BLOCK_KEYS - 1) / DC_BLOCK_KEYS;
  int n = (int)max((int64_t)1, min((int64_t)DC_MAX_SPLITS, (int64_t)512 / max((int64_t)1, (int64_t)B * Hkv)));
  const int per = (turns + min(n, turns) - 1) / min(n, turns);
  return Ranges{(turns + per - 1) / per, per * DC_BLOCK_KEYS};
}

size_t part_bytes(int n, int B, int Lq, int Hq, int D) { return (size_t)n * B * Lq * Hq * D * sizeof(float); }

template <int D, int MT>
int launch(const AttnParams& p, Ranges r, float* part_out, float* part_lse, hipStream_t st) {
  ODY_LAUNCH("attn_decode", st, (attn_decode_kernel<D, MT>), dim3(p.B * p.Hkv * r.n), dim3(64 * DC_WAVES), 0, p, r.n, r.keys, part_out,
             part_lse);
  int rc = ody_check_launch("attn_decode");
  if (rc || r.n == 1) return rc;
  ODY_LAUNCH("attn_decode_merge", st, (attn_decode_merge_kernel<D>), dim3(p.B * p.Lq * p.Hq), dim3(256), 0, p, r.n, part_out, part_lse);
  return ody_check_launch("attn_decode_merge");
}

template <int D>
int by_rows(const AttnParams& p, Ranges r, float* part_out, float* part_lse, hipStream_t st) {
  const int rows = p.group * p.Lq;
  if (rows <= 16) return launch<D, 1>(p, r, part_out, part_lse, st);
  if (rows <= 32) return launch<D, 2>(p, r, part_out, part_lse, st);
  return launch<D, 4>(p, r, part_out, part_lse, st);
}

}  // namespace

bool ody_attn_decode_ok(int Lq, int Hq, int Hkv, int D) {
  return (D == 64 || D == 128) && Lq <= DC_MAX_TOKENS && (int64_t)(Hq / Hkv) * Lq <= DC_MAX_ROWS;
}

size_t ody_attn_decode_workspace(int B, int Lq, int Lk, int Hq, int Hkv, int D) {
  const Ranges r = ranges(B, Lk, Hkv);
  return r.n == 1 ? 0 : part_bytes(r.n, B, Lq, Hq, D) + part_bytes(r.n, B, Lq, Hq, 1);
}

int ody_launch_attn_decode(const AttnParams& p, int D, void* workspace, size_t workspace_bytes, hipStream_t st) {
  Ranges r = ranges(p.B, p.Lk, p.Hkv);
  if (workspace == nullptr || workspace_bytes < ody_attn_decode_workspace(p.B, p.Lq, p.Lk, p.Hq, p.Hkv, D))
    r = Ranges{1, p.Lk};   // no room for the parts: one block per kv head walks all keys
  float* part_out = static_cast<float*>(workspace);
  float* part_lse = r.n == 1 ? nullptr : part_out + (size_t)r.n * p.B * p.Lq * p.Hq * D;
  return D == 64 ? by_rows<64>(p, r, part_out, part_lse, st) : by_rows<128>(p, r, part_out, part_lse, st);
}
