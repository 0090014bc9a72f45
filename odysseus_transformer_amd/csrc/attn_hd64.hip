// Flash attention for bf16 and head_dim 64, forward and backward, deterministic, without images or atomics.
//
// At head_dim 64 a (query, key) pair costs half the MFMA work of head_dim 128 and the same exp, conversions and sums: the
// vector pipe is the bound (forward: about 900 vector cycles per 512 matrix cycles of a 32 x 64 score tile), not LDS.  So, unlike
// the head_dim-128 kernels, operands that a product contracts over their row index are read with the transposing LDS read from
// the same tile as the row operands -- no transposed images, hence no pre-pass over V and K and half the tile bytes --, three
// or four wavefronts share a SIMD to keep the vector pipe fed, and the softmax of the forward does no work that the result does
// not need: a row's reference is the maximum of its first tile, nothing is compared or rescaled after it, and a block where a
// later score outgrew that by more than fp32 holds, in a row sum or in a sum of P V, walks its keys once more with a reference
// that follows.
//
// A block is 4 wavefronts of 32 rows each (queries; keys in the dK/dV kernel) against 64-row tiles of the other side, which go
// straight to LDS (direct loads, two stages).  GROUPS = 2 gives a block a second set of 4 wavefronts over the same rows, which
// takes every other tile; the sets add up through LDS at the end.  It is for calls with too few blocks to give every SIMD three
// wavefronts.
//
// The forward and dK/dV where there are blocks enough, and most calls' dQ, take the kernels of attn_hd64_pipe.hip (dispatch: end of this file).
//
// Tiles and fragments: attn_rowtile.h.
//
// Measured against the kernels these replace (register-staged tiles through padded LDS rows, rescaling on every tile, one block per
// kv head), us: 16 heads, L = 8192, causal: forward 207 -> 158 (870 TFLOP/s), dK/dV 415 -> 285, dQ 323 -> 213; 2 x 8 heads, L = 500,
// causal: 14 -> 10.7, 22.6 -> 16, 19.3 -> 11; 8 heads on 2 kv heads, L = 2000, full: 42 -> 26, 279 -> 45, 65 -> 30.  At the long
// shape the vector pipe is 70 % and the matrix pipe 46 % busy in the forward (16 % of the units' time is the causal tail), matrix 52 %
// and vector 45 % in dK/dV and dQ at 2.0 GHz.  Without effect: raised priority around the matrix steps, two wavefronts a SIMD
// instead of three in the backward.
//
// Error of the forward against 64 bits, standard normal inputs (running maximum / first tile's): 16 heads, L = 4096, causal 2.05e-3 /
// 2.11e-3; L = 700, full 2.21e-3 / 2.31e-3.  The roundings are the same ones; bf16 is finest just below a power of two, and that is
// where the largest P of a row lie if the reference is its maximum (an emulation in 64 bits that rounds P and out gives these figures).
#include <cfloat>
#include <type_traits>
#include <utility>
#include "attn_rowtile.h"

namespace {

using namespace rowtile;

constexpr int D = 64, KS = D / 16, DT = D / 32, TILE = ROWS * D;   // elements of a tile: 8 KB
constexpr int BLOCK_ROWS = 128;
typedef TileLoader<D, 4> Loader;

constexpr size_t KV_STAGE = 2 * TILE;                    // elements: two tiles
constexpr size_t QS_STAGE = 2 * TILE + 2 * 2 * ROWS;     // Q and dO tiles, -lse / scale and -delta of their rows in fp32
static_assert(2 * 2 * KV_STAGE * sizeof(bf16) >= 4 * 34 * 64 * sizeof(float) && 2 * 2 * QS_STAGE * sizeof(bf16) >= 4 * 64 * 64 * sizeof(float),
              "what a group hands over fits in the stages of two");

// ---------------------------------------------------------------------------------------------------------- forward
//   S^T = K Q^T      O^T += V^T P^T       lane = query column
template <int GROUPS>
__global__ __launch_bounds__(256 * GROUPS, 4) void attn_fwd_hd64_kernel(const AttnParams p) {
  constexpr size_t STAGE_BYTES = KV_STAGE * sizeof(bf16);
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int grp = wave >> 2, w4 = wave & 3;
  bf16* ring = reinterpret_cast<bf16*>(smem) + grp * 2 * KV_STAGE;   // [2][K tile | V tile]
  const BlockCoord bc = block_coord(p.Hq, p.B, p.causal);
  const int nqb = gridDim.x / (p.Hq * p.B);
  const int qblk = p.causal ? nqb - 1 - bc.rank : bc.rank;   // heaviest blocks first
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * BLOCK_ROWS, wq0 = q0 + w4 * 32, qi = wq0 + i;

  int n_end = p.causal ? min(p.Lk, min(q0 + BLOCK_ROWS, p.Lq) + p.off) : p.Lk;
  const int ntiles = n_end > 0 ? (n_end + ROWS - 1) / ROWS : 0;
  Loader lk, lv;
  lk.init(p.sk.l, w4, lane);
  lv.init(p.sv.l, w4, lane);
  const bf16* kp = static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const bf16* vp = static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h;
  auto load = [&](int t, int buf) {
    lk.load(ring + buf * KV_STAGE, kp, t * ROWS, p.Lk, w4);
    lv.load(ring + buf * KV_STAGE + TILE, vp, t * ROWS, p.Lk, w4);
  };

  bf16x8 qf[KS];
  load_rows(qf, static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h, p.sq.l, qi, p.Lq, g);
  const int lim = p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1;   // last key this lane's query sees
  const float c2 = p.scale_log2e;
  f32x16 o[DT];
  float ref;     // the row's reference in log2 units
  float l4[4];   // this lane's partial row sums

  // ONLINE = false: the reference of a row is the largest score of its first tile (a row that sees any key sees key 0) and stays.
  // ONLINE = true: it is the maximum so far, so that P <= 1 and P V overflows for no values that P = 1 would hold.
  const int iters = (ntiles + GROUPS - 1) / GROUPS;
  auto walk = [&](auto online) {
    constexpr bool ONLINE = decltype(online)::value;
    clear(o);
    ref = -FLT_MAX;   // no score is below it; not minus infinity, from which a masked score would be NaN
#pragma unroll
    for (int e = 0; e < 4; e++) l4[e] = 0.f;
    Readers<D> rd;
    rd.init(ring, g, i);
    auto tile = [&](int t, bool first) {
      const int n0 = t * ROWS;
      if (t >= ntiles || (p.causal && n0 > wq0 + 31 + p.off)) return;
      f32x16 s[2];
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int kt = 0; kt < 2; kt++) s[kt] = mfma32(row_frag(rd, 32 * kt, ks), qf[ks], ks == 0 ? f32x16{0} : s[kt]);
      if (n0 + ROWS > p.Lk || (p.causal && n0 + ROWS - 1 > wq0 + p.off)) {
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
          for (int r = 0; r < 16; r++)
            if (n0 + 32 * kt + acc_row(r, g) > lim) s[kt][r] = -INFINITY;
      }
      if (ONLINE || first) {
        float mx = fmaxf(s[0][0], s[1][0]);
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(mx, fmaxf(s[0][r], s[1][r]));
        mx = half_swap_max(mx) * c2;
        if (__builtin_amdgcn_ballot_w64(mx > ref) != 0) {
          const float next = fmaxf(ref, mx), alpha = ody_exp2(ref - next);
          ref = next;
#pragma unroll
          for (int e = 0; e < 4; e++) l4[e] *= alpha;
#pragma unroll
          for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
        }
      }
      auto half = [&](auto which) {
        constexpr int kt = decltype(which)::value;
        bf16x8 pb[2], vf[DT];
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const float x = ody_exp2(fmaf(s[kt][r], c2, -ref));
          l4[r & 3] += x;
          pb[r >> 3][r & 7] = (bf16)x;
        }
        tr_frags<ROWS + 32 * kt, 0>(vf, rd);
#pragma unroll
        for (int dt = 0; dt < DT; dt++) o[dt] = mfma32(vf[dt], pb[0], o[dt]);
        tr_frags<ROWS + 32 * kt + 16, 0>(vf, rd);
#pragma unroll
        for (int dt = 0; dt < DT; dt++) o[dt] = mfma32(vf[dt], pb[1], o[dt]);
      };
      half(std::integral_constant<int, 0>{});
      half(std::integral_constant<int, 1>{});
    };
    if (grp < ntiles) load(grp, 0);
    for (int it = 0; it < iters; it++) {
      const int t = grp + GROUPS * it;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();   // the tile has landed, and everyone is done with the one before
      if (t + GROUPS < ntiles) load(t + GROUPS, (it + 1) & 1);
      tile(t, it == 0);
      rd.move((it & 1) ? -(int)STAGE_BYTES : (int)STAGE_BYTES);
    }
    __syncthreads();   // everyone is done with the stages
  };
  walk(std::false_type{});
  {
    // a later score that outgrew its row's reference by more than fp32 holds left a row sum beyond any real one (or a NaN), or,
    // times large values, an infinity in O: 0 times the accumulators is 0 unless one of them is not finite
    int* flags = reinterpret_cast<int*>(smem);
    float zero[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int r = 0; r < 16; r++) zero[r & 3] = fmaf(o[dt][r], 0.f, zero[r & 3]);
    const bool finite = (zero[0] + zero[1]) + (zero[2] + zero[3]) == 0.f;
    const bool beyond = __builtin_amdgcn_ballot_w64(!finite || !(half_swap_sum((l4[0] + l4[1]) + (l4[2] + l4[3])) < 0x1p100f)) != 0;
    if (lane == 0) flags[wave] = beyond;
    __syncthreads();
    int any = 0;
#pragma unroll
    for (int w = 0; w < 4 * GROUPS; w++) any |= flags[w];
    __syncthreads();
    if (any) walk(std::true_type{});
  }

  float l = (l4[0] + l4[1]) + (l4[2] + l4[3]);
#pragma unroll 1
  for (int from = 1; from < GROUPS; from++) {
    float* patch = reinterpret_cast<float*>(smem) + w4 * 34 * 64;
    if (grp == from) {
      give(patch, o, lane);
      patch[32 * 64 + lane] = ref;
      patch[33 * 64 + lane] = l;
    }
    __syncthreads();
    if (grp == 0) {
      const float ref1 = patch[32 * 64 + lane], next = fmaxf(ref, ref1), a0 = ody_exp2(ref - next), a1 = ody_exp2(ref1 - next);
      take(patch, o, lane, a0, a1);
      l = l * a0 + patch[33 * 64 + lane] * a1;
      ref = next;
    }
    __syncthreads();
  }
  if (grp != 0) return;
  l = half_swap_sum(l);
  if (qi < p.Lq) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    store_row(static_cast<bf16*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)qi * p.so.l, o, inv, g);
    if (g == 0) p.lse[((int64_t)b * p.Hq + h) * p.Lq + qi] = l > 0.f ? (ref + __log2f(l)) * ODY_LN2 : -INFINITY;
  }
}

// ---------------------------------------------------------------------------------------------------------- backward
// Start values in fp32, either of them null where the call does not need it: -delta of every query row, (B, Hq, Lq), and -lse / scale,
// (B, Hq, Lq rounded up to whole tiles), minus infinity where P must be 0: past the end, or a query that saw no key.  8 lanes per row.
__global__ __launch_bounds__(256) void attn_bwd_hd64_rows_kernel(const AttnParams p, float* __restrict__ neg_delta,
                                                                 float* __restrict__ neg_lse) {
  const int lane8 = threadIdx.x & 7, qi = blockIdx.x * 32 + (threadIdx.x >> 3), h = blockIdx.y, b = blockIdx.z;
  float acc = 0.f;
  if (neg_delta && qi < p.Lq) {
    const bf16x8 ov = *reinterpret_cast<const bf16x8*>(static_cast<const bf16*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)qi * p.so.l + 8 * lane8);
    const bf16x8 dv = *reinterpret_cast<const bf16x8*>(static_cast<const bf16*>(p.dout) + b * p.sdo.b + h * p.sdo.h + (int64_t)qi * p.sdo.l + 8 * lane8);
#pragma unroll
    for (int e = 0; e < 8; e++) acc = fmaf((float)ov[e], (float)dv[e], acc);
  }
#pragma unroll
  for (int sft = 4; sft > 0; sft >>= 1) acc += __shfl_xor(acc, sft, 64);
  if (lane8 != 0) return;
  const int64_t head = (int64_t)b * p.Hq + h;
  const int rows = (p.Lq + ROWS - 1) / ROWS * ROWS;
  if (neg_delta && qi < p.Lq) neg_delta[head * p.Lq + qi] = -acc;
  if (neg_lse && qi < rows) {
    const float l = qi < p.Lq ? p.lse[head * p.Lq + qi] : INFINITY;
    neg_lse[head * rows + qi] = l == INFINITY || l == -INFINITY ? -INFINITY : -l / p.scale;
  }
}

//   S = Q K^T - lse / scale     dP = dO V^T - delta     dV^T += dO^T P     dK^T += Q^T (P o dP)      lane = key column
//
// S starts from -lse / scale of its rows, which the first wavefront of a group forms from lse once per tile: a register load beside
// the tile's direct loads, written to the tile's stage after the products of the tile before it.
//
// PART: the block takes ONE query head and leaves fp32 sums in part [dK | dV][B][Hq][Lk][D], which the kernel below adds over the
// heads of a group; otherwise it walks all query heads of its kv head.
template <int GROUPS, bool PART>
__global__ __launch_bounds__(256 * GROUPS, GROUPS == 1 ? 3 : 2) void attn_bwd_hd64_dkdv_kernel(const AttnParams p, const float* __restrict__ neg_delta,
                                                                            float* __restrict__ part) {
  constexpr size_t STAGE_BYTES = QS_STAGE * sizeof(bf16);
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int grp = wave >> 2, w4 = wave & 3;
  bf16* ring = reinterpret_cast<bf16*>(smem) + grp * 2 * QS_STAGE;   // [2][Q tile | dO tile | row values]
  const BlockCoord bc = block_coord(PART ? p.Hq : p.Hkv, p.B, p.causal);   // rank 0 = first key block = most query tiles
  const int b = bc.b, hk = PART ? bc.h / p.group : bc.h, h_first = PART ? bc.h : hk * p.group, heads = PART ? 1 : p.group;
  const int n0 = bc.rank * BLOCK_ROWS, wn0 = n0 + w4 * 32, key = wn0 + i;

  const int t_begin = p.causal ? max(0, n0 - p.off) / ROWS : 0, t_end = (p.Lq + ROWS - 1) / ROWS;
  const int ntq = max(0, t_end - t_begin), total = ntq * heads;
  // Tile `it` of the flattened (query head, query tile) range, last query tile first: the key blocks that run at one time on an
  // XCD then read the same Q and dO tiles.
  Loader lq, lo;
  lq.init(p.sq.l, w4, lane);
  lo.init(p.sdo.l, w4, lane);
  float l_next = INFINITY;   // first wavefront of a group: lse of row `lane` of the tile on its way
  auto load = [&](int it, int buf) {
    const int h = h_first + it / ntq, t = t_end - 1 - it % ntq;
    const int64_t head = ((int64_t)b * p.Hq + h) * p.Lq;
    if (w4 == 0) {
      l_next = INFINITY;
      if (t * ROWS + lane < p.Lq) l_next = p.lse[head + t * ROWS + lane];
    }
    bf16* st = ring + buf * QS_STAGE;
    lq.load(st, static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h, t * ROWS, p.Lq, w4);
    lo.load(st + TILE, static_cast<const bf16*>(p.dout) + b * p.sdo.b + h * p.sdo.h, t * ROWS, p.Lq, w4);
    if (w4 == 1) {   // rows past the end repeat the last one: their P is 0
      const float* src = neg_delta + head + min(t * ROWS + lane, p.Lq - 1);
      __builtin_amdgcn_global_load_lds((global_ptr)src, (lds_ptr)(st + 2 * TILE + 2 * ROWS), 4, 0, 0);
    }
  };
  // minus infinity for rows that must give P = 0: past the end, or a query that saw no key
  auto put_lse = [&](int buf) {
    if (w4 != 0) return;
    const bool none = l_next == INFINITY || l_next == -INFINITY;
    reinterpret_cast<float*>(ring + buf * QS_STAGE + 2 * TILE)[lane] = none ? -INFINITY : -l_next / p.scale;
  };
  if (grp < total) load(grp, 0);
  put_lse(0);

  bf16x8 kf[KS], vf[KS];
  load_rows(kf, static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h, p.sk.l, key, p.Lk, g);
  load_rows(vf, static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h, p.sv.l, key, p.Lk, g);
  const float c2 = p.scale_log2e;
  Readers<D> rd;
  rd.init(ring, g, i);
  f32x16 dk[DT], dv[DT];
  clear(dk);
  clear(dv);

  const int iters = (total + GROUPS - 1) / GROUPS;
  for (int n = 0; n < iters; n++) {
    const int it = grp + GROUPS * n, i0 = (t_end - 1 - it % max(ntq, 1)) * ROWS;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (it + GROUPS < total) load(it + GROUPS, (n + 1) & 1);
    const bf16* stage = ring + (n & 1) * QS_STAGE;
    const float* rv = reinterpret_cast<const float*>(stage + 2 * TILE) + 4 * g;
    auto sub_tile = [&](auto which) {
      __builtin_amdgcn_sched_barrier(0);   // one sub-tile's fragments at a time
      constexpr int mt = decltype(which)::value;
      const int m0 = i0 + 32 * mt;
      // every query of the sub-tile comes before every key of this wavefront: nothing to do
      if (it >= total || m0 >= p.Lq || (p.causal && m0 + 31 + p.off < wn0)) return;
      f32x16 s, dp;
#pragma unroll
      for (int a = 0; a < 4; a++) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(rv + 32 * mt + 8 * a);
        const f32x4 y = *reinterpret_cast<const f32x4*>(rv + ROWS + 32 * mt + 8 * a);
#pragma unroll
        for (int e = 0; e < 4; e++) s[4 * a + e] = x[e], dp[4 * a + e] = y[e];
      }
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        s = mfma32(row_frag(rd, 32 * mt, ks), kf[ks], s);
        dp = mfma32(row_frag(rd, ROWS + 32 * mt, ks), vf[ks], dp);
      }
      if (p.causal && m0 + p.off < wn0 + 31) {
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (m0 + acc_row(r, g) + p.off < key) s[r] = -INFINITY;
      }
      bf16x8 pf[2], dsf[2];
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const float pr = ody_exp2(s[r] * c2);
        pf[r >> 3][r & 7] = (bf16)pr;
        dsf[r >> 3][r & 7] = (bf16)(pr * dp[r]);
      }
      auto products = [&](auto half) {
        constexpr int ss = decltype(half)::value;
        bf16x8 of[DT], qf[DT];
        tr_frags<ROWS + 32 * mt + 16 * ss, 0>(of, rd);
        tr_frags<32 * mt + 16 * ss, 0>(qf, rd);
#pragma unroll
        for (int dt = 0; dt < DT; dt++) {
          dv[dt] = mfma32(of[dt], pf[ss], dv[dt]);
          dk[dt] = mfma32(qf[dt], dsf[ss], dk[dt]);
        }
      };
      products(std::integral_constant<int, 0>{});
      products(std::integral_constant<int, 1>{});
    };
    sub_tile(std::integral_constant<int, 0>{});
    sub_tile(std::integral_constant<int, 1>{});
    put_lse((n + 1) & 1);
    rd.move((n & 1) ? -(int)STAGE_BYTES : (int)STAGE_BYTES);
  }

#pragma unroll 1
  for (int from = 1; from < GROUPS; from++) {
    float* patch = reinterpret_cast<float*>(smem) + w4 * 64 * 64;
    __syncthreads();
    if (grp == from) {
      give(patch, dk, lane);
      give(patch + 32 * 64, dv, lane);
    }
    __syncthreads();
    if (grp == 0) {
      take(patch, dk, lane, 1.f, 1.f);
      take(patch + 32 * 64, dv, lane, 1.f, 1.f);
    }
  }
  if (grp != 0) return;
  if (key >= p.Lk) return;
  if (PART) {
    float* pk = part + (((int64_t)b * p.Hq + bc.h) * p.Lk + key) * D;
    float* pv = pk + (int64_t)p.B * p.Hq * p.Lk * D;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        f32x4 wk, wv;
#pragma unroll
        for (int e = 0; e < 4; e++) wk[e] = dk[dt][4 * a + e], wv[e] = dv[dt][4 * a + e];
        *reinterpret_cast<f32x4*>(pk + 32 * dt + 8 * a + 4 * g) = wk;
        *reinterpret_cast<f32x4*>(pv + 32 * dt + 8 * a + 4 * g) = wv;
      }
  } else {
    store_row(static_cast<bf16*>(p.dk) + b * p.sdk.b + hk * p.sdk.h + (int64_t)key * p.sdk.l, dk, p.scale, g);
    store_row(static_cast<bf16*>(p.dv) + b * p.sdv.b + hk * p.sdv.h + (int64_t)key * p.sdv.l, dv, 1.f, g);
  }
}

// dK, dV of a kv head = the sums of its query heads in their order; one thread per 4 elements
__global__ __launch_bounds__(256) void attn_bwd_hd64_sum_kernel(const AttnParams p, const float* __restrict__ part) {
  constexpr int Q = D / 4;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;   // over B * Hkv * Lk * D / 4
  if (idx >= (int64_t)p.B * p.Hkv * p.Lk * Q) return;
  const int d = 4 * (int)(idx % Q), key = (idx / Q) % p.Lk, hk = (idx / ((int64_t)Q * p.Lk)) % p.Hkv, b = idx / ((int64_t)Q * p.Lk * p.Hkv);
  const int64_t plane = (int64_t)p.B * p.Hq * p.Lk * D;
  const float* src = part + (((int64_t)b * p.Hq + hk * p.group) * p.Lk + key) * D + d;
  f32x4 sk = {0.f, 0.f, 0.f, 0.f}, sv = sk;
  for (int n = 0; n < p.group; n++, src += (int64_t)p.Lk * D) {
    sk += *reinterpret_cast<const f32x4*>(src);
    sv += *reinterpret_cast<const f32x4*>(src + plane);
  }
  bf16x4 wk, wv;
#pragma unroll
  for (int e = 0; e < 4; e++) wk[e] = (bf16)(sk[e] * p.scale), wv[e] = (bf16)sv[e];
  *reinterpret_cast<bf16x4*>(static_cast<bf16*>(p.dk) + b * p.sdk.b + hk * p.sdk.h + (int64_t)key * p.sdk.l + d) = wk;
  *reinterpret_cast<bf16x4*>(static_cast<bf16*>(p.dv) + b * p.sdv.b + hk * p.sdv.h + (int64_t)key * p.sdv.l + d) = wv;
}

//   S^T = K Q^T     dP^T = V dO^T - delta     dQ^T += K^T dS^T       lane = query column
template <int GROUPS>
__global__ __launch_bounds__(256 * GROUPS, GROUPS == 1 ? 3 : 2) void attn_bwd_hd64_dq_kernel(const AttnParams p,
                                                                                           const float* __restrict__ neg_delta) {
  constexpr size_t STAGE_BYTES = KV_STAGE * sizeof(bf16);
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int grp = wave >> 2, w4 = wave & 3;
  bf16* ring = reinterpret_cast<bf16*>(smem) + grp * 2 * KV_STAGE;
  const BlockCoord bc = block_coord(p.Hq, p.B, p.causal);
  const int nqb = gridDim.x / (p.Hq * p.B);
  const int qblk = p.causal ? nqb - 1 - bc.rank : bc.rank;
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * BLOCK_ROWS, wq0 = q0 + w4 * 32, qi = wq0 + i;

  int n_end = p.causal ? min(p.Lk, min(q0 + BLOCK_ROWS, p.Lq) + p.off) : p.Lk;
  const int ntiles = n_end > 0 ? (n_end + ROWS - 1) / ROWS : 0;
  Loader lk, lv;
  lk.init(p.sk.l, w4, lane);
  lv.init(p.sv.l, w4, lane);
  const bf16* kp = static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const bf16* vp = static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h;
  auto load = [&](int t, int buf) {
    lk.load(ring + buf * KV_STAGE, kp, t * ROWS, p.Lk, w4);
    lv.load(ring + buf * KV_STAGE + TILE, vp, t * ROWS, p.Lk, w4);
  };
  if (grp < ntiles) load(grp, 0);

  bf16x8 qf[KS], dof[KS];
  load_rows(qf, static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h, p.sq.l, qi, p.Lq, g);
  load_rows(dof, static_cast<const bf16*>(p.dout) + b * p.sdo.b + h * p.sdo.h, p.sdo.l, qi, p.Lq, g);
  const int64_t head = (int64_t)b * p.Hq + h;
  float lse2 = qi < p.Lq ? p.lse[head * p.Lq + qi] : INFINITY;
  if (lse2 == -INFINITY) lse2 = INFINITY;   // a query that saw no key: P = 0
  lse2 *= ODY_LOG2E;
  const float nd = qi < p.Lq ? neg_delta[head * p.Lq + qi] : 0.f;
  f32x16 start;   // dP starts from -delta: one add less per element
#pragma unroll
  for (int r = 0; r < 16; r++) start[r] = nd;
  const int lim = p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1;
  const float c2 = p.scale_log2e;
  Readers<D> rd;
  rd.init(ring, g, i);
  f32x16 dq[DT];
  clear(dq);

  const int iters = (ntiles + GROUPS - 1) / GROUPS;
  for (int it = 0; it < iters; it++) {
    const int t = grp + GROUPS * it;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + GROUPS < ntiles) load(t + GROUPS, (it + 1) & 1);
    auto sub_tile = [&](auto which) {
      __builtin_amdgcn_sched_barrier(0);   // one sub-tile's fragments at a time
      constexpr int kt = decltype(which)::value;
      const int k0 = t * ROWS + 32 * kt;
      if (t >= ntiles || k0 >= p.Lk || (p.causal && k0 > wq0 + 31 + p.off)) return;
      f32x16 s, dp;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        s = mfma32(row_frag(rd, 32 * kt, ks), qf[ks], ks == 0 ? f32x16{0} : s);
        dp = mfma32(row_frag(rd, ROWS + 32 * kt, ks), dof[ks], ks == 0 ? start : dp);
      }
      if (k0 + 32 > p.Lk || (p.causal && k0 + 31 > wq0 + p.off)) {
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (k0 + acc_row(r, g) > lim) s[r] = -INFINITY;
      }
      bf16x8 dsf[2];
#pragma unroll
      for (int r = 0; r < 16; r++) dsf[r >> 3][r & 7] = (bf16)(ody_exp2(fmaf(s[r], c2, -lse2)) * dp[r]);
      bf16x8 kf[DT];
      tr_frags<32 * kt, 0>(kf, rd);
#pragma unroll
      for (int dt = 0; dt < DT; dt++) dq[dt] = mfma32(kf[dt], dsf[0], dq[dt]);
      tr_frags<32 * kt + 16, 0>(kf, rd);
#pragma unroll
      for (int dt = 0; dt < DT; dt++) dq[dt] = mfma32(kf[dt], dsf[1], dq[dt]);
    };
    sub_tile(std::integral_constant<int, 0>{});
    sub_tile(std::integral_constant<int, 1>{});
    rd.move((it & 1) ? -(int)STAGE_BYTES : (int)STAGE_BYTES);
  }

#pragma unroll 1
  for (int from = 1; from < GROUPS; from++) {
    float* patch = reinterpret_cast<float*>(smem) + w4 * 32 * 64;
    __syncthreads();
    if (grp == from) give(patch, dq, lane);
    __syncthreads();
    if (grp == 0) take(patch, dq, lane, 1.f, 1.f);
  }
  if (grp != 0) return;
  if (qi >= p.Lq) return;
  store_dq(p, dq, b, h, qi, g);
}

inline size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
inline size_t delta_bytes(int B, int Lq, int Hq) { return align256((size_t)B * Hq * Lq * sizeof(float)); }
inline size_t lse_bytes(int B, int Lq, int Hq) { return align256((size_t)B * Hq * ((Lq + ROWS - 1) / ROWS * ROWS) * sizeof(float)); }
inline int64_t row_blocks(int B, int L, int H) { return (int64_t)B * H * ((L + BLOCK_ROWS - 1) / BLOCK_ROWS); }

// Fewer blocks than this leave SIMDs with one wavefront: two groups per block.  (More groups per block for all calls, which evens
// out a causal mask by itself, loses more to the wider barrier: dK/dV of 16 heads, L = 8192, with three groups 342 us against 311.)
constexpr int FEW_BLOCKS = 512;
// one block per query head instead of one per kv head where the latter leave compute units idle
inline bool split_heads(int B, int Lk, int Hq, int Hkv) { return Hq != Hkv && row_blocks(B, Lk, Hkv) < 1024; }

template <typename K, typename... A>
int launch(const char* name, K kern, int64_t blocks, int groups, size_t stage_elems, hipStream_t st, const A&... args) {
  const size_t smem = (size_t)groups * 2 * stage_elems * sizeof(bf16);
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, name)) return rc;
  ODY_LAUNCH(name, st, kern, dim3((unsigned)blocks), dim3(256 * groups), smem, args...);
  return ody_check_launch(name);
}

// The kernels of attn_hd64_pipe.hip address a tile with 32-bit byte offsets.
inline bool near(const AttnStrides& a, const AttnStrides& b) { return a.l < tile128::TILE_MAX_STRIDE && b.l < tile128::TILE_MAX_STRIDE; }

// The forward with 256-row blocks.  Before / with it, us:
//   Full.  A compute unit takes these blocks by whole rounds of 256, the former kernel's by half rounds, so that a last round at most half full goes to
//   the former one, unless there are rounds enough, the fewer the longer the rows, for the 5 to 17 % per round to make up for it.  512 keys: 16 heads,
//   L = 8192, 512 blocks, 26.5 / 25.3, 9 heads, 288 blocks, 19.4 / 23.4, 18 heads 32.9 / 34.5; 1000 keys, 4 x 64 heads, L = 1000, 91 / 79, 75 heads, 300 blocks,
//   34.9 / 37.5; 4096 keys, 57 heads, L = 2100, of whose last blocks half is empty, 155 / 177.  16 heads, L = 8192, 308 / 265.  None of 605 shapes from 192
//   blocks and 512 keys on is behind by more than 1 % this way.
//   Causal, where one block is many times as long as another, with three blocks for every unit or more, and work enough in all of them:
//   64 x 48 heads, L = 256, 768 blocks, 30.1 / 31.5, 128 x 64 heads of it 333 / 285; 8 x 48 heads, L = 512, 33.9 / 35.3, 32 x 64 heads 207 / 174;
//   1 x 24 heads, L = 8192, 235 / 213, 16 heads, 512 blocks, 179 / 173 by itself and 5 us behind before a backward; 48 heads, L = 4096, 128 / 117,
//   24 heads, 384 blocks, 76 / 79.
// A last block that is half empty costs its share of the rows.
//
// And with eight wavefronts a block, where that is one block for a unit, or causal, where two blocks to a unit from the start would leave the longer one
// alone on it, and blocks that take a unit each, longest first, do not.  Best of the other two / this one, us:
//   Full, more than one round of the former kernel's blocks and at most one of these: 4096 keys, 144 blocks, 70 / 60, 256 blocks 85 / 73, 1000 keys,
//   144 blocks, 26.9 / 24.0, 768 keys, 255 blocks, 27.4 / 25.4; not with 128 blocks, for which the former one has a unit each, 84 / 108 (8192 keys), and with
//   256 blocks not below 1024 keys: 700 22.3 / 23.1, 1000 27.4 / 27.6.
//   Causal, from 512 blocks of the former kernel to 512 of these: L = 8192, 8 heads, 126 / 112, 16 heads, 160 / 145; L = 4096, 16 heads, 68 / 62, 32 heads, 87 / 82,
//   L = 3000, 32 heads, 58 / 53; beyond, L = 8192, 18 heads, 176 / 179, L = 3000, 40 heads, 65.9 / 66.1, L = 2048, 48 heads, 43 / 45, or with a rectangle in front of the triangle, 3000
//   queries on 4096 keys, 27 heads, 79 / 81.
inline int fwd_pipe_groups(const AttnParams& p) {   // 0: not with 256-row blocks
  const int64_t halves = (p.Lq + BLOCK_ROWS - 1) / BLOCK_ROWS, blocks = (int64_t)p.B * p.Hq * ((halves + 1) / 2), former = (int64_t)p.B * p.Hq * halves;
  if (!near(p.sk, p.sv)) return 0;
  if (p.causal ? former >= FEW_BLOCKS && blocks <= 512 && 8 * (int64_t)p.off <= p.Lk && p.Lk >= (blocks <= 384 ? 3000 : 4096)
               : former > 256 && blocks <= 256 && p.Lk >= (former < FEW_BLOCKS ? 768 : 1024)) return 2;
  if ((halves & 1) && halves < 16) return 0;
  if (p.causal) return blocks >= 768 && blocks * p.Lk >= (1 << 21);
  const int64_t rounds = (blocks + 255) / 256, lost = 2 * rounds - (former + 255) / 256;   // half rounds
  if (former < FEW_BLOCKS || p.Lk < (rounds == 1 ? 640 : 512)) return 0;
  return lost == 0 || (lost == 1 && rounds > (p.Lk >= 2048 ? 2 : p.Lk >= 1024 ? 4 : 7));
}

// dQ in the order of attn_hd64_pipe.hip.  A unit holds two of its blocks and three of the former kernel's (one of eight wavefronts with fewer than 512).
// Before / with it, us: 384 blocks: L = 128 15.9 / 12.4, L = 512 24.2 / 19.1, L = 4096 106 / 85; 64 to 256 blocks 1.00 to 1.09; causal, 510 blocks, L = 700
// 26.5 / 20.6.  From 512 blocks on it wants rows long enough for a round of two blocks instead of three: L = 256, 768 blocks, 21.9 / 23.0; L = 384 24.1 / 25.2;
// L = 512 29.3 / 29.0; L = 1000 46.3 / 44.4; causal, where a block sees half of them, L = 384, 640 blocks, 19.4 / 21.9; L = 700 25.3 / 26.5; L = 1000 30.4 / 29.3;
// L = 2048 50.4 / 42.2.
inline bool dq_pipe_ok(const AttnParams& p, int64_t blocks) {
  return near(p.sk, p.sv) && (blocks < FEW_BLOCKS || p.Lk >= (p.causal ? 1000 : 512));
}

}  // namespace

int ody_launch_attn_fwd_hd64(const AttnParams& p, hipStream_t st) {
  if (const int groups = fwd_pipe_groups(p)) return ody_launch_attn_fwd_hd64_pipe(p, groups, st);
  const int64_t blocks = row_blocks(p.B, p.Lq, p.Hq);
  return blocks < FEW_BLOCKS ? launch("attn_fwd_hd64", &attn_fwd_hd64_kernel<2>, blocks, 2, KV_STAGE, st, p)
                             : launch("attn_fwd_hd64", &attn_fwd_hd64_kernel<1>, blocks, 1, KV_STAGE, st, p);
}

// [-delta | -lse / scale | fp32 dK / dV of every query head]; with less room -delta alone.  Without query heads to split, room for the second is
// asked where the dK / dV kernel of attn_hd64_pipe.hip reads it and has a quarter of the chip's units to run on: below, callers keep the
// workspace that they had, and the former kernel (whole backward, us, former / that one: 4 heads, L = 1000, 32 blocks, 42.7 / 40.1; 4 heads,
// L = 500 29.0 / 27.7; above the line 8 heads, L = 1000, 64 blocks, 42.9 / 40.1, 4 heads, L = 4000 125 / 114).
size_t ody_attn_bwd_hd64_workspace(int B, int Lq, int Lk, int Hq, int Hkv) {
  if (split_heads(B, Lk, Hq, Hkv))
    return delta_bytes(B, Lq, Hq) + lse_bytes(B, Lq, Hq) + align256((size_t)2 * B * Hq * Lk * D * sizeof(float));
  const bool pipe = Hq == Hkv && Lq > 5 * ROWS && row_blocks(B, Lk, Hq) >= 64;
  return delta_bytes(B, Lq, Hq) + (pipe ? lse_bytes(B, Lq, Hq) : 0);
}

int ody_launch_attn_bwd_hd64(const AttnParams& p, void* workspace, size_t workspace_bytes, hipStream_t st) {
  float* neg_delta = static_cast<float*>(workspace);
  float* neg_lse = reinterpret_cast<float*>(static_cast<char*>(workspace) + delta_bytes(p.B, p.Lq, p.Hq));
  float* part = reinterpret_cast<float*>(reinterpret_cast<char*>(neg_lse) + lse_bytes(p.B, p.Lq, p.Hq));
  const bool heads = split_heads(p.B, p.Lk, p.Hq, p.Hkv) && workspace_bytes >= ody_attn_bwd_hd64_workspace(p.B, p.Lq, p.Lk, p.Hq, p.Hkv);
  // dK / dV with one query head per block, in the order of attn_hd64_pipe.hip.  Whole backward before / with it, us: 16 heads, L = 8192, causal
  // 520 / 472, full 992 / 890; 8 heads of it 386 / 308; 16 heads, L = 4096, causal 206 / 164; 4 x 32 heads, L = 500, 57.1 / 52.3.  With fewer than 6
  // tiles of queries its prologue shows: 32 x 16 heads, L = 300, 96.2 / 97.5; 64 x 16 heads, L = 256, causal 113.7 / 116.  A unit holds two of its
  // blocks and three of the former kernel's, so that beyond 512 of them it wants rows long enough for the tail not to count: full, 8 x 32 heads,
  // L = 384, 0.98, L = 512 1.02; causal, 4 x 32 heads, L = 708, 59.0 / 63.0, 8 x 32 heads, L = 321, 0.88, 4 x 32 heads, L = 1000, 1.03.
  const int64_t blocks = row_blocks(p.B, p.Lk, p.Hq);
  const bool pipe = workspace_bytes >= delta_bytes(p.B, p.Lq, p.Hq) + lse_bytes(p.B, p.Lq, p.Hq) && (heads || p.group == 1) &&
                    p.Lq > ROWS * (blocks <= 512 ? 5 : p.causal ? 15 : 7) && near(p.sq, p.sdo);
  int rc;
  // Of a reused query side -delta alone is taken as it is: whether the call before wrote -lse / scale, and with this scale, depends on the keys
  // and the workspace that it had.
  if (!p.reuse_query_side || pipe) {
    const dim3 grid((p.Lq + ROWS - 1) / ROWS * (ROWS / 32), p.Hq, p.B);
    if (p.reuse_query_side)
      ODY_LAUNCH("attn_bwd_hd64_lse", st, attn_bwd_hd64_rows_kernel, grid, dim3(256), 0, p, nullptr, neg_lse);
    else
      ODY_LAUNCH("attn_bwd_hd64_rows", st, attn_bwd_hd64_rows_kernel, grid, dim3(256), 0, p, neg_delta, pipe ? neg_lse : nullptr);
    if ((rc = ody_check_launch("attn_bwd_hd64_rows"))) return rc;
  }
  const int64_t nkv = row_blocks(p.B, p.Lk, heads ? p.Hq : p.Hkv), nq = row_blocks(p.B, p.Lq, p.Hq);
  auto dkdv = [&](auto kern, int groups) { return launch("attn_bwd_hd64_dkdv", kern, nkv, groups, QS_STAGE, st, p, neg_delta, part); };
  if (pipe) rc = ody_launch_attn_bwd_hd64_dkdv_pipe(p, neg_delta, neg_lse, heads ? part : nullptr, st);
  else if (nkv < FEW_BLOCKS) rc = heads ? dkdv(&attn_bwd_hd64_dkdv_kernel<2, true>, 2) : dkdv(&attn_bwd_hd64_dkdv_kernel<2, false>, 2);
  else rc = heads ? dkdv(&attn_bwd_hd64_dkdv_kernel<1, true>, 1) : dkdv(&attn_bwd_hd64_dkdv_kernel<1, false>, 1);
  if (rc) return rc;
  if (heads) {
    const int64_t n = (int64_t)p.B * p.Hkv * p.Lk * (D / 4);
    ODY_LAUNCH("attn_bwd_hd64_sum", st, attn_bwd_hd64_sum_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, p, part);
    if ((rc = ody_check_launch("attn_bwd_hd64_sum"))) return rc;
  }
  if (dq_pipe_ok(p, nq)) return ody_launch_attn_bwd_hd64_dq_pipe(p, neg_delta, st);
  return nq < FEW_BLOCKS ? launch("attn_bwd_hd64_dq", &attn_bwd_hd64_dq_kernel<2>, nq, 2, KV_STAGE, st, p, neg_delta)
                         : launch("attn_bwd_hd64_dq", &attn_bwd_hd64_dq_kernel<1>, nq, 1, KV_STAGE, st, p, neg_delta);
}
