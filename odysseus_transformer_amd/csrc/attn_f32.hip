// fp32 attention (forward and backward) on the fp32 matrix cores, plus the delta
// pre-pass shared with the bf16 backward.
//
// These kernels serve the fp32 configuration, whose 1e-4 tolerance rules out bf16
// operands: head_dim 128, dropout, and the shortest forwards of head_dim 64, whose other calls are in attn_f32_parts.hip.  All products run on v_mfma_f32_32x32x2_f32 (lane = 32 g + i holds
// A[row i][k = g] and B[k = g][col i]; the 32 x 32 result sits in 16 registers,
// register r of lane (i, g) = row 8 (r / 4) + 4 g + r % 4, column i).
//
// A workgroup is 4 wavefronts of 32 rows each (queries in the forward and dQ kernels,
// keys in the dK / dV kernel); the other side is streamed in tiles of 32 rows through
// LDS, the next tile being fetched into registers while the current one is multiplied.
// As in the bf16 kernels the score tile is computed transposed where the wavefront owns
// queries (S^T = K Q^T), so one lane = one query and softmax statistics need no
// cross-lane traffic beyond one swap of the wavefront halves, and the result registers
// are directly the B operand of the next product.
//
// SPLIT instances serve calls with few rows, whose 128-row workgroups would leave compute units idle (and, under a causal
// mask, wait for the longest): the wavefronts (eight at head_dim 64) own the SAME 32 rows and take the streamed tiles in turn, each through
// LDS of its own (no barrier in the loop), and add their results up through LDS at the end.  8 heads x 64, L = 2048,
// causal: forward 160 -> 56 us, dQ 237 -> 73, dK / dV 298 -> 97; 8 x 64, L = 8192: 842 -> 689, 1262 -> 913, 1600 -> 1287.
// Where they do not serve, few_rows() below: 16 heads x 64, 4096 rows against 4096 full: 572 us whole, 691 split, against 32: 15
// and 57; 16 x 128, L = 4096, causal: 658 and 829.
//
// Two index permutations keep every LDS read conflict-free and 16 bytes wide where it
// can be:
//  * contraction over head_dim: k-step 4 j + t multiplies element 8 j + 4 g + t, so the
//    streamed operand is one 16-byte read per four MFMAs and the resident operand is
//    loaded once in the same order;
//  * contraction over the 32 streamed rows: k-step ks multiplies row 8 (ks / 4) + 4 g +
//    ks % 4, which is the row that result register ks of this lane already holds.
// Everything is deterministic: no atomics, fixed summation order.
#include <algorithm>
#include <cmath>
#include "attn_f32.h"

namespace {

using namespace f32tile;

constexpr int F_WAVES = 4;
constexpr int F_THREADS = 64 * F_WAVES;
constexpr int F_ROWS = 32 * F_WAVES;  // rows owned by a workgroup

// Geometry of an instance: who owns which rows, who streams which tiles, through which LDS.
template <int D, bool SPLIT>
struct Shape {
  static constexpr int LD = D + 4;
  // as many as the tiles in LDS allow: two per SIMD at head_dim 64, one at 128
  static constexpr int WAVES = SPLIT && D == 64 ? 8 : F_WAVES, THREADS = 64 * WAVES;
  static constexpr int ROWS = SPLIT ? 32 : F_ROWS;                 // rows owned by a workgroup
  static constexpr int LOADERS = SPLIT ? 64 : F_THREADS;           // threads that bring one tile
  static constexpr int STEP = SPLIT ? WAVES * F_TILE : F_TILE;   // streamed rows between two turns of a wavefront
  static constexpr int TILES = SPLIT ? WAVES : 1;                // tiles of each kind in LDS
  __device__ static __forceinline__ void sync() {
    if (SPLIT) wavefront_sync();   // its tiles are its own
    else __syncthreads();
  }
};

// SPLIT: the wavefronts' 32 x D results (result-register order, already on a common scale) through `lds` ([WAVES][32][LD],
// the streamed tiles' room), summed, times mul(row), to dst(row); `add`: onto what is there.
template <int D, int WAVES, typename Dst, typename Mul>
__device__ __forceinline__ void sum_wavefronts(float* lds, const f32x16 (&acc)[D / 32], int wave, int i, int g, int tid, int nrows, bool add,
                                               Dst dst, Mul mul) {
  constexpr int LD = D + 4;
  __syncthreads();
#pragma unroll
  for (int db = 0; db < D / 32; db++)
#pragma unroll
    for (int a = 0; a < 4; a++)
      *reinterpret_cast<f32x4*>(lds + (wave * 32 + i) * LD + 32 * db + 8 * a + 4 * g) =
          f32x4{acc[db][4 * a], acc[db][4 * a + 1], acc[db][4 * a + 2], acc[db][4 * a + 3]};
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 8 * D / (64 * WAVES); c++) {
    const int e = tid + c * 64 * WAVES, r = e / (D / 4), x = e % (D / 4);
    if (r >= nrows) continue;
    f32x4 v = *reinterpret_cast<const f32x4*>(lds + r * LD + 4 * x);
#pragma unroll
    for (int w = 1; w < WAVES; w++) v += *reinterpret_cast<const f32x4*>(lds + (w * 32 + r) * LD + 4 * x);
    v *= mul(r);
    f32x4* out = reinterpret_cast<f32x4*>(dst(r) + 4 * x);
    if (add) v += *out;
    *out = v;
  }
}

// ---------------------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------------------
// DROP (all three kernels): attention dropout (AttnParams::drop_*, ody_dropout_hash): row sums and lse are those of the
// full P; the entries that enter P V are the kept ones scaled by 1 / (1 - p), and dP counts only where an entry was kept.
template <int D, bool DROP, bool SPLIT>
__global__ __launch_bounds__((Shape<D, SPLIT>::THREADS), D == 64 ? (SPLIT ? 2 : 3) : 1) void attn_fwd_f32_kernel(const AttnParams p) {
  using S = Shape<D, SPLIT>;
  constexpr int LD = S::LD, NDB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float smem[];   // [TILES][K tile, V tile]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, g = lane >> 5;
  const BlockCoord bc = ody_block_coord(p.Hq, p.B);
  const int nqb = gridDim.x / (p.Hq * p.B);
  const int qblk = p.causal ? (nqb - 1 - bc.rank) : bc.rank;  // heaviest blocks first
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * S::ROWS, wq0 = SPLIT ? q0 : q0 + wave * 32, qi = wq0 + i;
  const int ltid = SPLIT ? lane : tid;
  float* Ks = smem + (SPLIT ? wave : 0) * 2 * F_TILE * LD;
  float* Vs = Ks + F_TILE * LD;
  const float* qp = static_cast<const float*>(p.q) + b * p.sq.b + h * p.sq.h;
  const float* kp = static_cast<const float*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const float* vp = static_cast<const float*>(p.v) + b * p.sv.b + hk * p.sv.h;

  float qf[D / 2];  // scores come out in the log2 domain
  load_row_frag<D>(qf, qp, p.sq.l, qi, qi < p.Lq, g, p.scale_log2e);
  f32x16 o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; db++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[db][r] = 0.f;
  float m = -INFINITY, l = 0.f;
  const unsigned drow = DROP ? ody_dropout_row(ody_dropout_head(p.drop_seed, b * p.Hq + h), qi) : 0u;

  // last key this lane's query sees, the first query of the wavefront sees, and the
  // key ranges the workgroup and the wavefront have to walk
  const int lim = p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1;
  const int lim_first = p.causal ? min(p.Lk - 1, wq0 + p.off) : p.Lk - 1;
  const int blk_hi = min(q0 + S::ROWS, p.Lq) - 1, wav_hi = min(wq0 + 32, p.Lq) - 1;
  const int n_end = max(0, p.causal ? min(p.Lk, blk_hi + p.off + 1) : p.Lk);
  const int w_end = (wq0 < p.Lq) ? max(0, p.causal ? min(p.Lk, wav_hi + p.off + 1) : p.Lk) : 0;

  TileRegs<D, S::LOADERS> kr, vr;
  const int n_first = SPLIT ? wave * F_TILE : 0;
  if (n_first < n_end) {
    kr.fetch(kp, p.sk.l, n_first, min(F_TILE, p.Lk - n_first), ltid);
    vr.fetch(vp, p.sv.l, n_first, min(F_TILE, p.Lk - n_first), ltid);
  }
  for (int n0 = n_first; n0 < n_end; n0 += S::STEP) {
    S::sync();
    kr.put(Ks, ltid);
    vr.put(Vs, ltid);
    S::sync();
    if (n0 + S::STEP < n_end) {
      kr.fetch(kp, p.sk.l, n0 + S::STEP, min(F_TILE, p.Lk - n0 - S::STEP), ltid);
      vr.fetch(vp, p.sv.l, n0 + S::STEP, min(F_TILE, p.Lk - n0 - S::STEP), ltid);
    }
    if (n0 >= w_end) continue;  // wavefront-uniform: nothing visible to this wavefront here

    f32x16 s, s1;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = s1[r] = 0.f;
    tile_times_frag<D>(Ks, i, g, qf, s, s1);
    s += s1;
    if (n0 + F_TILE - 1 > lim_first) {
#pragma unroll
      for (int r = 0; r < 16; r++)
        if (n0 + acc_row(r, g) > lim) s[r] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
    mx = half_swap_max(mx);
    const float m_new = fmaxf(m, mx);
    const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
    const float alpha = ody_exp2(m - m_use);
    m = m_new;
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      s[r] = ody_exp2(s[r] - m_use);
      sum += s[r];
      if (DROP && ody_dropout_hash(drow, n0 + acc_row(r, g)) < p.drop_thresh) s[r] = 0.f;
    }
    l = l * alpha + sum;
#pragma unroll
    for (int db = 0; db < NDB; db++) o[db] *= alpha;
    tile_t_times_regs<D>(Vs, i, g, s, o);
  }

  l = half_swap_sum(l);
  if constexpr (SPLIT) {
    __shared__ float sm[S::WAVES][32], sl[S::WAVES][32];
    if (g == 0) sm[wave][i] = m, sl[wave][i] = l;
    __syncthreads();
    float top = sm[0][i];
#pragma unroll
    for (int w = 1; w < S::WAVES; w++) top = fmaxf(top, sm[w][i]);
    const float mine = ody_exp2(m - (top == -INFINITY ? 0.f : top));
#pragma unroll
    for (int db = 0; db < NDB; db++) o[db] *= mine;
    auto total = [&](int r, float& ref) {
      float t = sm[0][r], sum = 0.f;
#pragma unroll
      for (int w = 1; w < S::WAVES; w++) t = fmaxf(t, sm[w][r]);
      ref = t == -INFINITY ? 0.f : t;
#pragma unroll
      for (int w = 0; w < S::WAVES; w++) sum += sl[w][r] * ody_exp2(sm[w][r] - ref);
      return sum;
    };
    float* ob = static_cast<float*>(p.out) + b * p.so.b + h * p.so.h;
    sum_wavefronts<D, S::WAVES>(smem, o, wave, i, g, tid, min(32, p.Lq - q0), false, [&](int r) { return ob + (int64_t)(q0 + r) * p.so.l; },
                      [&](int r) {
                        float ref;
                        const float sum = total(r, ref);
                        return sum > 0.f ? (DROP ? p.drop_scale : 1.f) / sum : 0.f;
                      });
    if (wave == 0 && g == 0 && qi < p.Lq) {
      float ref;
      const float sum = total(i, ref);
      p.lse[((int64_t)b * p.Hq + h) * p.Lq + qi] = sum > 0.f ? (ref + __log2f(sum)) * LN2 : -INFINITY;
    }
    return;
  }
  if (qi < p.Lq) {
    float* op = static_cast<float*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)qi * p.so.l;
    store_rows<D>(op, o, g, l > 0.f ? (DROP ? p.drop_scale : 1.f) / l : 0.f, false);
    if (g == 0) p.lse[((int64_t)b * p.Hq + h) * p.Lq + qi] = l > 0.f ? (m + __log2f(l)) * LN2 : -INFINITY;
  }
}

// ---------------------------------------------------------------------------------------
// dQ: the wavefront owns 32 queries, keys are streamed
// ---------------------------------------------------------------------------------------
template <int D, bool DROP, bool SPLIT>
__global__ __launch_bounds__((Shape<D, SPLIT>::THREADS), D == 64 && SPLIT ? 2 : 1) void attn_bwd_dq_f32_kernel(const AttnParams p) {
  using S = Shape<D, SPLIT>;
  constexpr int LD = S::LD, NDB = D / 32;
  extern __shared__ __attribute__((aligned(16))) float smem[];   // [TILES][K tile, V tile]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, g = lane >> 5;
  const BlockCoord bc = ody_block_coord(p.Hq, p.B);
  const int nqb = gridDim.x / (p.Hq * p.B);
  const int qblk = p.causal ? (nqb - 1 - bc.rank) : bc.rank;
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * S::ROWS, wq0 = SPLIT ? q0 : q0 + wave * 32, qi = wq0 + i;
  const int ltid = SPLIT ? lane : tid;
  float* Ks = smem + (SPLIT ? wave : 0) * 2 * F_TILE * LD;
  float* Vs = Ks + F_TILE * LD;
  const float* qp = static_cast<const float*>(p.q) + b * p.sq.b + h * p.sq.h;
  const float* dop = static_cast<const float*>(p.dout) + b * p.sdo.b + h * p.sdo.h;
  const float* kp = static_cast<const float*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const float* vp = static_cast<const float*>(p.v) + b * p.sv.b + hk * p.sv.h;

  float qf[D / 2], dof[D / 2];
  load_row_frag<D>(qf, qp, p.sq.l, qi, qi < p.Lq, g, p.scale_log2e);
  load_row_frag<D>(dof, dop, p.sdo.l, qi, qi < p.Lq, g, 1.f);
  const int64_t ri = ((int64_t)b * p.Hq + h) * p.Lq + qi;
  const float lse = (qi < p.Lq) ? p.lse[ri] : -INFINITY;
  const float lse2 = lse * ODY_LOG2E;
  const float delta = (qi < p.Lq) ? p.delta[ri] : 0.f;
  const unsigned drow = DROP ? ody_dropout_row(ody_dropout_head(p.drop_seed, b * p.Hq + h), qi) : 0u;
  // a query with no visible key (lse = -inf) contributes nothing
  const int lim = (lse == -INFINITY) ? -1 : (p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1);
  f32x16 dq[NDB];
#pragma unroll
  for (int db = 0; db < NDB; db++)
#pragma unroll
    for (int r = 0; r < 16; r++) dq[db][r] = 0.f;

  const int blk_hi = min(q0 + S::ROWS, p.Lq) - 1, wav_hi = min(wq0 + 32, p.Lq) - 1;
  const int n_end = max(0, p.causal ? min(p.Lk, blk_hi + p.off + 1) : p.Lk);
  const int w_end = (wq0 < p.Lq) ? max(0, p.causal ? min(p.Lk, wav_hi + p.off + 1) : p.Lk) : 0;

  TileRegs<D, S::LOADERS> kr, vr;
  const int n_first = SPLIT ? wave * F_TILE : 0;
  if (n_first < n_end) {
    kr.fetch(kp, p.sk.l, n_first, min(F_TILE, p.Lk - n_first), ltid);
    vr.fetch(vp, p.sv.l, n_first, min(F_TILE, p.Lk - n_first), ltid);
  }
  for (int n0 = n_first; n0 < n_end; n0 += S::STEP) {
    S::sync();
    kr.put(Ks, ltid);
    vr.put(Vs, ltid);
    S::sync();
    if (n0 + S::STEP < n_end) {
      kr.fetch(kp, p.sk.l, n0 + S::STEP, min(F_TILE, p.Lk - n0 - S::STEP), ltid);
      vr.fetch(vp, p.sv.l, n0 + S::STEP, min(F_TILE, p.Lk - n0 - S::STEP), ltid);
    }
    if (n0 >= w_end) continue;

    f32x16 s, dp;
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = dp[r] = 0.f;
    tiles_times_frags<D>(Ks, qf, s, Vs, dof, dp, i, g);  // S^T = K Q^T (log2 domain), dP^T = V dO^T
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const float pr = (n0 + acc_row(r, g) > lim) ? 0.f : ody_exp2(s[r] - lse2);
      float dpv = dp[r];
      if (DROP) dpv = ody_dropout_hash(drow, n0 + acc_row(r, g)) >= p.drop_thresh ? dpv * p.drop_scale : 0.f;
      s[r] = pr * (dpv - delta) * p.scale;  // dS^T
    }
    tile_t_times_regs<D>(Ks, i, g, s, dq);  // dQ^T += K^T dS^T
  }
  if constexpr (SPLIT) {
    float* qb = static_cast<float*>(p.dq) + b * p.sdq.b + h * p.sdq.h;
    sum_wavefronts<D, S::WAVES>(smem, dq, wave, i, g, tid, min(32, p.Lq - q0), p.accumulate_dq != 0,
                      [&](int r) { return qb + (int64_t)(q0 + r) * p.sdq.l; }, [](int) { return 1.f; });
    return;
  }
  if (qi < p.Lq) {
    float* dqp = static_cast<float*>(p.dq) + b * p.sdq.b + h * p.sdq.h + (int64_t)qi * p.sdq.l;
    store_rows<D>(dqp, dq, g, 1.f, p.accumulate_dq != 0);
  }
}

// ---------------------------------------------------------------------------------------
// dK / dV: the wavefront owns 32 keys, the queries of every head of the group are streamed.
// WHICH: 0 = dV only, 1 = dK only, 2 = both.  (At head_dim 128 the K and V fragments and both
// accumulators do not fit the register file together, so dV and dK take a pass each.)
// ---------------------------------------------------------------------------------------
template <int D, int WHICH, bool DROP, bool SPLIT>
__global__ __launch_bounds__((Shape<D, SPLIT>::THREADS), (D == 64 || (WHICH == 0 && !SPLIT)) ? 2 : 1) void attn_bwd_dkdv_f32_kernel(const AttnParams p) {
  using S = Shape<D, SPLIT>;
  constexpr int LD = S::LD, NDB = D / 32;
  constexpr bool DO_DV = (WHICH != 1), DO_DK = (WHICH != 0);
  extern __shared__ __attribute__((aligned(16))) float smem[];   // [TILES][Q tile, dO tile]
  __shared__ __attribute__((aligned(16))) float stats[S::TILES][2][F_TILE];  // lse in the log2 domain (+inf = row contributes nothing), delta
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 31, g = lane >> 5;
  const BlockCoord bc = ody_block_coord(p.Hkv, p.B);
  const int kblk = bc.rank;  // with causal masking the first key block is the heaviest
  const int hk = bc.h, b = bc.b;
  const int n0 = kblk * S::ROWS, wn0 = SPLIT ? n0 : n0 + wave * 32, ki = wn0 + i;
  const int ltid = SPLIT ? lane : tid;
  float* Qs = smem + (SPLIT ? wave : 0) * 2 * F_TILE * LD;
  float* Os = Qs + F_TILE * LD;
  float* Ls = stats[SPLIT ? wave : 0][0];
  float* Ds = stats[SPLIT ? wave : 0][1];
  const float* kp = static_cast<const float*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const float* vp = static_cast<const float*>(p.v) + b * p.sv.b + hk * p.sv.h;

  float kf[D / 2];
  float vf[DO_DK ? D / 2 : 1];
  load_row_frag<D>(kf, kp, p.sk.l, ki, ki < p.Lk, g, p.scale_log2e);
  if constexpr (DO_DK) load_row_frag<D>(vf, vp, p.sv.l, ki, ki < p.Lk, g, 1.f);
  f32x16 dk[DO_DK ? NDB : 1], dv[DO_DV ? NDB : 1];
#pragma unroll
  for (int db = 0; db < NDB; db++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      if constexpr (DO_DK) dk[db][r] = 0.f;
      if constexpr (DO_DV) dv[db][r] = 0.f;
    }

  // first query tile that sees the first key of the workgroup / of the wavefront
  const int i_begin = p.causal ? (max(0, n0 - p.off) / F_TILE) * F_TILE : 0;
  const int w_begin = p.causal ? max(0, wn0 - p.off) : 0;

  // turns over the query tiles of every head of the group
  const int ntq = p.Lq > i_begin ? (p.Lq - i_begin + F_TILE - 1) / F_TILE : 0, turns = ntq * p.group;
  TileRegs<D, S::LOADERS> qr, dor;
  float lr = 0.f, dr = 0.f;  // the first 32 loaders carry lse and delta of the next tile
  auto fetch = [&](int it) {
    const int h = hk * p.group + it / ntq, i0 = i_begin + (it % ntq) * F_TILE, valid = min(F_TILE, p.Lq - i0);
    qr.fetch(static_cast<const float*>(p.q) + b * p.sq.b + h * p.sq.h, p.sq.l, i0, valid, ltid);
    dor.fetch(static_cast<const float*>(p.dout) + b * p.sdo.b + h * p.sdo.h, p.sdo.l, i0, valid, ltid);
    if (ltid < F_TILE) {
      const int64_t rbase = ((int64_t)b * p.Hq + h) * p.Lq;
      const float x = (ltid < valid) ? p.lse[rbase + i0 + ltid] : -INFINITY;
      lr = (x == -INFINITY) ? INFINITY : x * ODY_LOG2E;
      dr = (ltid < valid) ? p.delta[rbase + i0 + ltid] : 0.f;
    }
  };
  const int it_first = SPLIT ? wave : 0, it_step = S::STEP / F_TILE;
  if (it_first < turns) fetch(it_first);
  {
    for (int it = it_first; it < turns; it += it_step) {
      const int h = hk * p.group + it / ntq, i0 = i_begin + (it % ntq) * F_TILE;
      const unsigned dh = DROP ? ody_dropout_head(p.drop_seed, b * p.Hq + h) : 0u;
      S::sync();
      qr.put(Qs, ltid);
      dor.put(Os, ltid);
      if (ltid < F_TILE) {
        Ls[ltid] = lr;
        Ds[ltid] = dr;
      }
      S::sync();
      if (it + it_step < turns) fetch(it + it_step);
      if (i0 + F_TILE <= w_begin || wn0 >= p.Lk) continue;  // wavefront-uniform

      // S = Q K^T (log2 domain): rows = queries, column = this lane's key; dP = dO V^T
      f32x16 s, dp;
#pragma unroll
      for (int r = 0; r < 16; r++) s[r] = dp[r] = 0.f;
      if constexpr (DO_DK) {
        tiles_times_frags<D>(Qs, kf, s, Os, vf, dp, i, g);
      } else {
        tile_times_frag<D>(Qs, i, g, kf, s, dp);
        s += dp;
      }
      f32x4 lv[4], dl[4];
#pragma unroll
      for (int a = 0; a < 4; a++) {
        lv[a] = *reinterpret_cast<const f32x4*>(Ls + 8 * a + 4 * g);
        dl[a] = *reinterpret_cast<const f32x4*>(Ds + 8 * a + 4 * g);
      }
      const int vis = p.causal ? ki - p.off - i0 : -1;  // tile row r is masked iff r < vis
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const float pr = (acc_row(r, g) < vis) ? 0.f : ody_exp2(s[r] - lv[r >> 2][r & 3]);
        bool keep = true;
        if (DROP) keep = ody_dropout_hash(ody_dropout_row(dh, i0 + acc_row(r, g)), ki) >= p.drop_thresh;
        s[r] = DROP ? (keep ? pr * p.drop_scale : 0.f) : pr;
        if constexpr (DO_DK) {
          const float dpv = DROP ? (keep ? dp[r] * p.drop_scale : 0.f) : dp[r];
          dp[r] = pr * (dpv - dl[r >> 2][r & 3]) * p.scale;  // dS
        }
      }
      if constexpr (DO_DV) tile_t_times_regs<D>(Os, i, g, s, dv);   // dV^T += dO^T P
      if constexpr (DO_DK) tile_t_times_regs<D>(Qs, i, g, dp, dk);  // dK^T += Q^T dS
    }
  }
  if constexpr (SPLIT) {
    if constexpr (DO_DK) {
      float* base = static_cast<float*>(p.dk) + b * p.sdk.b + hk * p.sdk.h;
      sum_wavefronts<D, S::WAVES>(smem, dk, wave, i, g, tid, min(32, p.Lk - n0), false, [&](int r) { return base + (int64_t)(n0 + r) * p.sdk.l; },
                        [](int) { return 1.f; });
    }
    if constexpr (DO_DV) {
      float* base = static_cast<float*>(p.dv) + b * p.sdv.b + hk * p.sdv.h;
      sum_wavefronts<D, S::WAVES>(smem, dv, wave, i, g, tid, min(32, p.Lk - n0), false, [&](int r) { return base + (int64_t)(n0 + r) * p.sdv.l; },
                        [](int) { return 1.f; });
    }
    return;
  }
  if (ki < p.Lk) {
    if constexpr (DO_DK) {
      float* dst = static_cast<float*>(p.dk) + b * p.sdk.b + hk * p.sdk.h + (int64_t)ki * p.sdk.l;
      store_rows<D>(dst, dk, g, 1.f, false);
    }
    if constexpr (DO_DV) {
      float* dst = static_cast<float*>(p.dv) + b * p.sdv.b + hk * p.sdv.h + (int64_t)ki * p.sdv.l;
      store_rows<D>(dst, dv, g, 1.f, false);
    }
  }
}

// delta[b, h, i] = sum_d dO[b, i, h, d] * O[b, i, h, d]; LPR lanes per row,
// 16-byte loads.
template <typename T, int D>
__global__ __launch_bounds__(256) void attn_delta_kernel(const AttnParams p) {
  constexpr int VEC = Vec16B<T>::N, LPR = D / VEC, RPB = 256 / LPR;
  typedef typename Vec16B<T>::type vec_t;
  const int tid = threadIdx.x, sub = tid % LPR;
  const int64_t row = (int64_t)blockIdx.x * RPB + tid / LPR;  // over B * Hq * Lq in (b, h, i) order
  const int64_t total = (int64_t)p.B * p.Hq * p.Lq;
  float acc = 0.f;
  if (row < total) {
    const int i = row % p.Lq;
    const int h = (row / p.Lq) % p.Hq;
    const int b = row / ((int64_t)p.Lq * p.Hq);
    const T* op = static_cast<const T*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)i * p.so.l + sub * VEC;
    const T* dp = static_cast<const T*>(p.dout) + b * p.sdo.b + h * p.sdo.h + (int64_t)i * p.sdo.l + sub * VEC;
    const vec_t ov = *reinterpret_cast<const vec_t*>(op);
    const vec_t dv = *reinterpret_cast<const vec_t*>(dp);
#pragma unroll
    for (int e = 0; e < VEC; e++) acc = fmaf((float)ov[e], (float)dv[e], acc);
  }
#pragma unroll
  for (int s = LPR / 2; s > 0; s >>= 1) acc += __shfl_xor(acc, s, 64);
  if (row < total && sub == 0) p.delta[row] = acc;
}

// Tiles of the streamed side that a row block walks: the longest walk and the mean.
struct Walk { double longest, mean; };
Walk walk(const AttnParams& p, bool own_keys) {
  double pairs = (double)p.Lq * p.Lk, longest = own_keys ? p.Lq : p.Lk;
  if (p.causal) {   // a query sees keys up to its own position + off; before that, none
    pairs = p.off >= 0 ? (double)p.Lq * (p.off + 0.5 * p.Lq) : 0.5 * p.Lk * p.Lk;
    if (own_keys) longest = std::min(p.Lq, p.Lk);
  }
  const double share = own_keys ? (double)p.group / p.Lk : 1.0 / p.Lq;
  if (own_keys) longest *= p.group;
  return Walk{std::ceil(longest / F_TILE), std::min(pairs * share, longest) / F_TILE};
}

// Whether the SPLIT instance is the faster one, in units of the time that a lone 128-row workgroup takes per tile (2.4 us in the
// forward of head_dim 64, 4.7 at 128).  That workgroup's walk is as long as its tiles; where several share a unit, the unit is
// at 0.9 per tile, and behind a causal mask's longest walk most of the unit idles at head_dim 64 (three workgroups share one) and
// little at 128 (one each).  A round of 256 split workgroups costs its start and end and 0.32 (head_dim 128: 0.34) per tile, and
// no less than one tile for each wavefront.  Fitted to 1100 shapes of 32 to 16384 rows and tokens, 1 to 256 heads, both masks:
// never slower than the whole instance by more than 2 us, and 0.2 % off the better one in the mean.  From 1024 whole workgroups on these
// are ahead, whole / split in us: 8 x 64, L = 16384, causal 2443 / 2629 forward, 4731 / 4955 dK / dV (dQ 3684 / 3522, the one exception
// of 42 timed); 2 x 16 x 64, L = 4096, causal 612 / 735, 1192 / 1351, dQ 928 / 975; 8 x 32 x 64, L = 512, causal 96 / 195, 194 / 323,
// 155 / 249; 32 x 128, L = 4096, causal 1277 / 1641 forward, dQ 1813 / 2116.
template <int D>
bool few_rows(int rows, int heads, Walk w) {
  constexpr double start = D == 64 ? 1.0 : 1.6, tile = D == 64 ? 0.32 : 0.34, idle = D == 64 ? 0.9 : 0.2;
  const int64_t whole = (int64_t)((rows + F_ROWS - 1) / F_ROWS) * heads, split = (int64_t)((rows + 31) / 32) * heads;
  if (whole >= 1024 || w.longest < 2) return false;
  const double rounds = (double)((split + 255) / 256), per_unit = 0.9 * whole / 256.0;
  return rounds * (start + tile * std::max(w.mean, (double)Shape<D, true>::WAVES)) <
         1.75 + std::max(w.longest, per_unit * w.mean + idle * (w.longest - w.mean));
}

template <int D, bool SPLIT, typename K>
int launch_one(const char* name, K kern, int rows, int heads, const AttnParams& p, hipStream_t st) {
  using S = Shape<D, SPLIT>;
  constexpr size_t smem = sizeof(float) * S::TILES * 2 * F_TILE * S::LD;
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, name)) return rc;
  ODY_LAUNCH(name, st, kern, dim3((unsigned)(((int64_t)rows + S::ROWS - 1) / S::ROWS * heads)), dim3(S::THREADS), smem, p);
  return ody_check_launch(name);
}

template <int D, bool DROP>
int launch_fwd(const AttnParams& p, hipStream_t st) {
  const int heads = p.Hq * p.B;
  const bool few = few_rows<D>(p.Lq, heads, walk(p, false));
  if constexpr (D == 64 && !DROP) {
    // a tile for each wavefront and no more: the products are over before splitting the operands pays (8 heads, 71 tokens: 9.8 us here,
    // 10.9 there; 300 tokens 15.6 and 14.0)
    if (few && p.Lk <= Shape<D, true>::STEP) return launch_one<D, true>("attn_fwd_f32_split", &attn_fwd_f32_kernel<D, DROP, true>, p.Lq, heads, p, st);
    return ody_launch_attn_fwd_f32_parts(p, st);
  } else {
    if (few) return launch_one<D, true>("attn_fwd_f32_split", &attn_fwd_f32_kernel<D, DROP, true>, p.Lq, heads, p, st);
    return launch_one<D, false>("attn_fwd_f32", &attn_fwd_f32_kernel<D, DROP, false>, p.Lq, heads, p, st);
  }
}

template <int D, bool DROP, bool SPLIT>
int launch_dkdv(const AttnParams& p, hipStream_t st) {
  const int heads = p.Hkv * p.B;
  if constexpr (D == 64) {
    return launch_one<D, SPLIT>(SPLIT ? "attn_bwd_dkdv_f32_split" : "attn_bwd_dkdv_f32", &attn_bwd_dkdv_f32_kernel<D, 2, DROP, SPLIT>, p.Lk, heads, p, st);
  } else {
    if (int rc = launch_one<D, SPLIT>(SPLIT ? "attn_bwd_dv_f32_split" : "attn_bwd_dv_f32", &attn_bwd_dkdv_f32_kernel<D, 0, DROP, SPLIT>, p.Lk, heads, p, st)) return rc;
    return launch_one<D, SPLIT>(SPLIT ? "attn_bwd_dk_f32_split" : "attn_bwd_dk_f32", &attn_bwd_dkdv_f32_kernel<D, 1, DROP, SPLIT>, p.Lk, heads, p, st);
  }
}

template <int D, bool DROP>
int launch_bwd(const AttnParams& p, hipStream_t st) {
  if constexpr (D == 64 && !DROP) {
    if (int rc = ody_launch_attn_bwd_dkdv_f32_parts(p, st)) return rc;
    return ody_launch_attn_bwd_dq_f32_parts(p, st);
  } else {
    const int rc = few_rows<D>(p.Lk, p.Hkv * p.B, walk(p, true)) ? launch_dkdv<D, DROP, true>(p, st) : launch_dkdv<D, DROP, false>(p, st);
    if (rc) return rc;
    const int heads = p.Hq * p.B;
    if (few_rows<D>(p.Lq, heads, walk(p, false))) return launch_one<D, true>("attn_bwd_dq_f32_split", &attn_bwd_dq_f32_kernel<D, DROP, true>, p.Lq, heads, p, st);
    return launch_one<D, false>("attn_bwd_dq_f32", &attn_bwd_dq_f32_kernel<D, DROP, false>, p.Lq, heads, p, st);
  }
}

template <typename T, int D>
int launch_delta(const AttnParams& p, hipStream_t st) {
  constexpr int RPB = 256 / (D / Vec16B<T>::N);
  const int64_t total = (int64_t)p.B * p.Hq * p.Lq;
  ODY_LAUNCH("attn_delta", st, (attn_delta_kernel<T, D>), dim3((unsigned)((total + RPB - 1) / RPB)), dim3(256), 0, p);
  return ody_check_launch("attn_delta");
}

}  // namespace

int ody_launch_attn_fwd_f32(const AttnParams& p, int D, hipStream_t st) {
  const bool drop = p.drop_thresh != 0;
  if (D == 64) return drop ? launch_fwd<64, true>(p, st) : launch_fwd<64, false>(p, st);
  if (D == 128) return drop ? launch_fwd<128, true>(p, st) : launch_fwd<128, false>(p, st);
  ody_set_error("fp32 attention: head_dim %d not built", D);
  return ODY_ERR_UNSUPPORTED;
}

int ody_launch_attn_bwd_f32(const AttnParams& p, int D, hipStream_t st) {
  const bool drop = p.drop_thresh != 0;
  if (D == 64) return drop ? launch_bwd<64, true>(p, st) : launch_bwd<64, false>(p, st);
  if (D == 128) return drop ? launch_bwd<128, true>(p, st) : launch_bwd<128, false>(p, st);
  ody_set_error("fp32 attention: head_dim %d not built", D);
  return ODY_ERR_UNSUPPORTED;
}

int ody_launch_attn_delta(const AttnParams& p, int D, int dtype, hipStream_t st) {
  if (dtype == ODY_F32 && D == 64) return launch_delta<float, 64>(p, st);
  if (dtype == ODY_F32 && D == 128) return launch_delta<float, 128>(p, st);
  if (dtype == ODY_BF16 && D == 64) return launch_delta<bf16, 64>(p, st);
  if (dtype == ODY_BF16 && D == 128) return launch_delta<bf16, 128>(p, st);
  ody_set_error("attention: head_dim %d / dtype %d not built", D, dtype);
  return ODY_ERR_UNSUPPORTED;
}
