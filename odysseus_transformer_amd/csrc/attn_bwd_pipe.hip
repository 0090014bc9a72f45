// Flash-attention backward, head_dim 128, bf16, on the tile machinery of attn_tile.h: direct
// global->LDS loads into rings (buffer loads: behind those of the flat kind the compiler waits for all LDS reads in flight in front of each use
// of one), 16-byte LDS reads only (an operand that a product
// contracts over its row index comes from the transposed images a pre-pass writes), fenced slots
// that fix the order of MFMAs, LDS reads and vector work.  Two kernels, no atomics: both recompute S
// from the saved log-sum-exp, and each owns its outputs.
//
// dQ kernel -- query-stationary, 4 wavefronts x 64 queries, one per SIMD, lane = query column, so lse and delta
// are per-lane scalars; two-deep rings of {K tile, V tile} and {K^T image}:
//
//      S^T = K Q^T            A: K rows (LDS)        B: Q^T (registers)
//      dP^T = V dO^T          A: V rows (LDS)        B: dO^T (registers)
//      dS^T = exp2(S^T c - lse) * (dP^T - delta)      dP^T starts at -delta
//      dQ^T += K^T dS^T       A: K^T image (LDS)     B: dS^T = accumulator layout
//
// A step forms S^T and dP^T of one 32-key sub-tile and then dQ^T of the one before, 16 products each; the vector work of the former runs under
// the last 32 of them, and every fragment read from LDS serves both halves of the queries.  Bound: power.  Against the kernel before (8 wavefronts of 32 queries,
// two per SIMD, a tile's parts one after the other), us, one box: 4 heads, L = 32768, causal 1420 / 1227 (constant operands 1076 / 879: the matrix
// pipe 61 / 75 % busy), 32 heads on 8, L = 16384 2910 / 2512, 4 heads, 8192 queries on 16384 keys 348 / 308.
//
// dK/dV kernel -- key-stationary (described where it is defined).
#include <algorithm>
#include <type_traits>
#include <utility>
#include "attn_store.h"
#include "attn_tile.h"

namespace {

using namespace tile128;

constexpr int D = 128, KS = D / 16, DT = D / 32;
#define FENCE() __builtin_amdgcn_sched_barrier(0)
#define INLINE __attribute__((always_inline))

// The same accumulators as one part's unscaled fp32 sum (a dQ kernel whose key range is cut into parts):
// dq_part [part][B][Lq][Hq][D]; attn_bwd_dq_sum_kernel adds the parts and finishes dq as store_dq_row would.
__device__ __forceinline__ void store_dq_part(float* __restrict__ dq_part, int part, const AttnParams& p,
                                              const f32x16 (&dq)[DT], int b, int h, int qi, int g) {
  if (qi >= p.Lq) return;
  float* dst = dq_part + ((((int64_t)part * p.B + b) * p.Lq + qi) * p.Hq + h) * D;
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int a = 0; a < 4; a++) {
      f32x4 w;
#pragma unroll
      for (int e = 0; e < 4; e++) w[e] = dq[dt][4 * a + e];
      *reinterpret_cast<f32x4*>(dst + 32 * dt + 8 * a + 4 * g) = w;
    }
}

// ---------------------------------------------------------------------------------
// dQ
// ---------------------------------------------------------------------------------
constexpr int DQ_WAVES = 8, DQ_BM = 32 * DQ_WAVES, DQ_THREADS = 64 * DQ_WAVES;   // of the kernel over kept dS

constexpr int DP_WAVES = 4, DP_QT = 2, DP_THREADS = 64 * DP_WAVES, DP_BN = 64;
constexpr int DP_ROWS = 2 * TILE_ELEMS;                         // a K tile and a V tile
static_assert(32 * DP_QT * DP_WAVES == DQ_BM, "the same blocks as the kernel over kept dS");
static_assert(DP_WAVES == 4, "the load split and the vmcnt waits assume 4 wavefronts");

// A product whose second operand lies in accumulation registers, with results in ordinary ones (see mfma32_onto)
__device__ __forceinline__ void mfma32_from_acc(f32x16& d, bf16x8 a, bf16x8 b, const f32x16& c) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %3" : "=&v"(d) : "v"(a), "a"(b), "v"(c));
}
__device__ __forceinline__ void mfma32_onto_acc(f32x16& d, bf16x8 a, bf16x8 b) {
  asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "a"(b));
}

// kparts > 1 (too few query blocks for the chip): block id = part + kparts * (the usual id), the block takes part
// `part` of its key tiles and leaves its unscaled fp32 sum in dq_part.
__global__ __launch_bounds__(DP_THREADS, 1) void attn_bwd_dq_pipe_kernel(const AttnParams p,
                                                                          const bf16* __restrict__ kimg, int kparts,
                                                                          float* __restrict__ dq_part) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  bf16* rring = reinterpret_cast<bf16*>(smem_raw);   // [2][DP_ROWS]
  bf16* iring = rring + 2 * DP_ROWS;                 // [2][IMG_ELEMS]

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5,
            i = lane & 31;
  const int kpart = blockIdx.x % kparts;
  const BlockCoord bc = ody_block_coord_of(blockIdx.x / kparts, p.Hq, p.B);
  const int nqb = gridDim.x / (p.Hq * p.B * kparts);
  const int qblk = p.causal ? (nqb - 1 - bc.rank) : bc.rank;   // heaviest blocks first
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * DQ_BM, wq0 = q0 + wave * 32 * DP_QT;

  const int q_hi = min(q0 + DQ_BM, p.Lq) - 1;
  int n_end = p.causal ? min(p.Lk, q_hi + p.off + 1) : p.Lk;
  if (n_end < 0) n_end = 0;
  int ntiles = (n_end + DP_BN - 1) / DP_BN;
  int t_first = 0;   // this block's part of the tiles: [t_first, ntiles)
  if (kparts > 1) {
    const int per = (ntiles + kparts - 1) / kparts;
    t_first = min(kpart * per, ntiles);
    ntiles = min(t_first + per, ntiles);
  }
  // end of those that this wavefront's queries see a key of, and of those that they see whole
  int w_end = ntiles, w_full = p.Lk / DP_BN;
  if (p.causal) {
    w_end = min(ntiles, max(t_first, (wq0 + 32 * DP_QT - 1 + p.off + DP_BN) / DP_BN));
    w_full = min(w_full, max(0, wq0 + p.off + 1) / DP_BN);
  }

  const float c2 = p.scale_log2e;

  // Direct loads: of the rows of tile `lr` and of the image of tile `li`, the last one again where there are no more.  Rows past the end read
  // zeros: they lie beyond the descriptor.
  const int last_tile = max(ntiles - 1, 0);   // (a block without tiles brings tile 0 and leaves it)
  int lr = min(t_first, last_tile), li = lr;
  const int krow = 2 * (int)p.sk.l, vrow = 2 * (int)p.sv.l;   // bytes
  const int klane = (4 * wave + (lane >> 4)) * krow + 16 * (lane & 15), vlane = (4 * wave + (lane >> 4)) * vrow + 16 * (lane & 15);
  const int ilane = 1024 * wave + 16 * lane;
  const bf16* ktp = static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h + (int64_t)lr * DP_BN * p.sk.l;
  const bf16* vtp = static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h + (int64_t)lr * DP_BN * p.sv.l;
  const bf16* kip = kimg + (((int64_t)b * p.Hkv + hk) * ((p.Lk + DP_BN - 1) / DP_BN) + lr) * IMG_ELEMS;
  int room = p.Lk - lr * DP_BN;   // rows from the tile's first one on
  auto bring = [&](const bf16* src, int bytes, bf16* dst, int off, int soff) INLINE {
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(src), (short)0, bytes, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_ptr)dst, 16, off, soff, 0, 0);
  };
  auto load_rows = [&](int j, int which) INLINE {   // a quarter j of the K tile, of the V tile
    bf16* dst = rring + (lr & 1) * DP_ROWS + (4 * j + wave) * GROUP_ELEMS;
    const int last = min(room, DP_BN) - 1;
    if (which == 0) bring(ktp, last * krow + 256, dst, klane + 16 * j * krow, 0);
    else bring(vtp, last * vrow + 256, dst + TILE_ELEMS, vlane + 16 * j * vrow, 0);
  };
  auto load_image = [&](int j) INLINE { bring(kip, IMG_BYTES, iring + (li & 1) * IMG_ELEMS + (4 * j + wave) * 512, ilane, 4096 * j); };
  auto next_rows = [&]() INLINE {
    const int to = min(lr + 1, last_tile), step = to - lr;
    lr = to;
    ktp += (int64_t)step * (DP_BN / 2 * krow);
    vtp += (int64_t)step * (DP_BN / 2 * vrow);
    room -= step * DP_BN;
  };
  auto next_image = [&]() INLINE {
    const int to = min(li + 1, last_tile), step = to - li;
    li = to;
    kip += step * IMG_ELEMS;
  };

  auto all_rows = [&]() INLINE {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      load_rows(j, 0);
      load_rows(j, 1);
    }
  };
  auto all_image = [&]() INLINE {
#pragma unroll
    for (int j = 0; j < 4; j++) load_image(j);
  };

  // The first tiles, and the queries' side behind the first rows: one wait for memory in front of the first products (attn_fwd_pipe.hip)
  all_rows();
  FENCE();
  bf16x8 qf[DP_QT][KS], dof[DP_QT][KS];
  f32x16 minus_delta[DP_QT];   // what dP starts from
  float lse2[DP_QT], delta[DP_QT];
  int lim[DP_QT];
  {
    const bf16* qp = static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h;
    const bf16* dop = static_cast<const bf16*>(p.dout) + b * p.sdo.b + h * p.sdo.h;
#pragma unroll
    for (int qt = 0; qt < DP_QT; qt++) {
      const int qi = wq0 + 32 * qt + i, row = min(qi, p.Lq - 1);   // rows past the end: the last one, whose results are not stored
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        qf[qt][ks] = *reinterpret_cast<const bf16x8*>(qp + (int64_t)row * p.sq.l + 16 * ks + 8 * g);
        dof[qt][ks] = *reinterpret_cast<const bf16x8*>(dop + (int64_t)row * p.sdo.l + 16 * ks + 8 * g);
      }
      const int64_t ri = ((int64_t)b * p.Hq + h) * p.Lq + row;
      lse2[qt] = p.lse[ri];
      delta[qt] = p.delta[ri];
      lim[qt] = p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1;
    }
  }
  FENCE();
  all_image();
  next_rows();
  all_rows();
  FENCE();
#pragma unroll
  for (int qt = 0; qt < DP_QT; qt++) {
#pragma unroll
    for (int ks = 0; ks < KS; ks++) asm volatile("" : "+v"(qf[qt][ks]), "+a"(dof[qt][ks]));
    if (lse2[qt] == -INFINITY || wq0 + 32 * qt + i >= p.Lq) lse2[qt] = INFINITY;   // a query that saw no key: P = 0
    lse2[qt] *= ODY_LOG2E;
#pragma unroll
    for (int r = 0; r < 16; r++) minus_delta[qt][r] = -delta[qt];
    asm volatile("" : "+v"(minus_delta[qt]), "+v"(lse2[qt]));
  }

  const int rbase = row_frag_base(g, i), ibase = image_frag_base(g, i);
  f32x16 dq[DP_QT][DT];
#pragma unroll
  for (int qt = 0; qt < DP_QT; qt++)
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int r = 0; r < 16; r++) dq[qt][dt][r] = 0.f;
  f32x16 s[DP_QT], dp[DP_QT];            // S, then P; dP, then dS
  bf16x8 dsf[DP_QT][2], dsf_next[DP_QT][2];
  // the steps of element e (query half e >> 4, register e & 15) of a sub-tile
  auto exponent = [&](int e, int t, int kt, auto masked) INLINE {
    const int qt = e >> 4, r = e & 15;
    float x = s[qt][r];
    if (decltype(masked)::value) x = t * DP_BN + acc_tile_row(r, g, kt) > lim[qt] ? -INFINITY : x;
    s[qt][r] = fmaf(x, c2, -lse2[qt]);
  };
  auto weight = [&](int e) INLINE { s[e >> 4][e & 15] = ody_exp2(s[e >> 4][e & 15]); };
  auto ds = [&](int e) INLINE { dp[e >> 4][e & 15] *= s[e >> 4][e & 15]; };
  auto pack = [&](int q) INLINE {   // elements 2 q and 2 q + 1
    const int qt = q >> 3, r = 2 * (q & 7);
    dsf_next[qt][r >> 3][r & 7] = (bf16)dp[qt][r], dsf_next[qt][r >> 3][(r & 7) + 1] = (bf16)dp[qt][r + 1];
  };
  constexpr int LGKM_4 = 0xc47f;   // s_waitcnt lgkmcnt(4): with the reads behind them in the order below, half of `fr` is there
  bf16x8 fr[8];
  auto kfrag = [&](const bf16* rows, int kt, int n) INLINE { return row_frag(rows, rbase, n, kt); };                 // k-step n
  auto vfrag = [&](const bf16* rows, int kt, int n) INLINE { return row_frag(rows + TILE_ELEMS, rbase, n, kt); };
  auto ifrag = [&](const bf16* im, int kt, int n) INLINE { return image_frag(im, ibase, n & 3, n >> 2, kt); };      // k-step n >> 2, columns 32 (n & 3)
  auto rslot = [&](int t) INLINE { return rring + (t & 1) * DP_ROWS; };
  auto islot = [&](int t) INLINE { return iring + (t & 1) * IMG_ELEMS; };
  auto barrier_rows = [&]() INLINE {     // the rows of the next tile have landed (behind them 4 loads of an image); everyone is done with those before
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    next_rows();
  };
  auto barrier_image = [&]() INLINE {    // likewise the image (behind it 8 loads of rows)
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    next_image();
  };

  // One step: S and dP of the sub-tile after (tile t, sub-tile KT), then dQ of this one: three parts of 16 products, with the vector work of the
  // sub-tile after under the last two.  A fragment serves both halves of the queries; `fr` holds those of a part when it begins and is left
  // with those of the next.
  auto step = [&](int t, auto kt_, auto masked) INLINE {
    constexpr int KT = decltype(kt_)::value, NKT = KT ^ 1;
    const int nt = KT ? t + 1 : t;
    const bf16 *rows = rslot(nt), *after = rslot(t + 1), *image = islot(t);   // after: of the sub-tile behind the next one
#pragma unroll
    for (int m = 0; m < 16; m++) {
      const int n = m >> 1, qt = m & 1;
      if ((m & 7) == 0) __builtin_amdgcn_s_waitcnt(LGKM_4);
      if (n == 0) mfma32_new(s[qt], fr[n], qf[qt][n]);
      else mfma32_onto(s[qt], fr[n], qf[qt][n]);
      FENCE();
      if (qt == 1) fr[n] = vfrag(rows, NKT, n);
      if (KT == 1 && (m & 7) == 4) load_rows(1, m >> 3);
      FENCE();
    }
    if (KT == 0) barrier_image();
#pragma unroll
    for (int m = 0; m < 16; m++) {
      const int n = m >> 1, qt = m & 1;
      if ((m & 7) == 0) __builtin_amdgcn_s_waitcnt(LGKM_4);
      if (n == 0) mfma32_from_acc(dp[qt], fr[n], dof[qt][n], minus_delta[qt]);
      else mfma32_onto_acc(dp[qt], fr[n], dof[qt][n]);
      FENCE();
      if (qt == 1) fr[n] = ifrag(image, KT, n);
      if (m >= 3) weight(2 * m - 6), weight(2 * m - 5);
      if (m >= 2) exponent(2 * m - 4, nt, NKT, masked), exponent(2 * m - 3, nt, NKT, masked);   // (S is 3 products old)
      if (KT == 0 && (m & 3) == 1) load_image(m >> 2);
      if (KT == 1 && (m & 7) == 4) load_rows(2, m >> 3);
      FENCE();
    }
    if (KT == 0) barrier_rows();
#pragma unroll
    for (int m = 0; m < 16; m++) {
      const int n = m >> 1, qt = m & 1;
      if ((m & 7) == 0) __builtin_amdgcn_s_waitcnt(LGKM_4);
      dq[qt][n & 3] = mfma32(fr[n], dsf[qt][n >> 2], dq[qt][n & 3]);
      FENCE();
      if (qt == 1) fr[n] = kfrag(after, KT, n);
      if (m <= 2) weight(2 * m + 26), weight(2 * m + 27);
      if (m <= 1) exponent(2 * m + 28, nt, NKT, masked), exponent(2 * m + 29, nt, NKT, masked);
      if (m >= 2) {   // all of dS and its operands before the next part takes the registers of S
#pragma unroll
        for (int e = 0; e < 3; e++)
          if (3 * (m - 2) + e < 32) ds(3 * (m - 2) + e);
      }
      if (m >= 4) {
        if (m < 12) pack(m - 4);
        else pack(2 * m - 16), pack(2 * m - 15);
      }
      if (KT == 0 && (m & 7) == 4) load_rows(0, m >> 3);
      if (KT == 1 && (m & 7) == 4) load_rows(3, m >> 3);
      FENCE();
    }
#pragma unroll
    for (int qt = 0; qt < DP_QT; qt++)
#pragma unroll
      for (int ss = 0; ss < 2; ss++) dsf[qt][ss] = dsf_next[qt][ss];
  };
  std::integral_constant<int, 0> c0;
  std::integral_constant<int, 1> c1;

  if (t_first < ntiles) {
    asm volatile("s_waitcnt vmcnt(12)" ::: "memory");   // the first tile's rows
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int t = t_first;
    if (t < w_end) {
      // S, P, dP and dS of the first sub-tile
      const bf16* rows = rslot(t);
#pragma unroll
      for (int n = 0; n < 8; n++) {
        const bf16x8 fk = kfrag(rows, 0, n), fv = vfrag(rows, 0, n);
#pragma unroll
        for (int qt = 0; qt < DP_QT; qt++) {
          if (n == 0) {
            mfma32_new(s[qt], fk, qf[qt][n]);
            mfma32_from_acc(dp[qt], fv, dof[qt][n], minus_delta[qt]);
          } else {
            mfma32_onto(s[qt], fk, qf[qt][n]);
            mfma32_onto_acc(dp[qt], fv, dof[qt][n]);
          }
        }
      }
      asm volatile("s_nop 15\n\ts_nop 7" : "+v"(s[0]), "+v"(s[1]), "+v"(dp[0]), "+v"(dp[1]));
#pragma unroll
      for (int e = 0; e < 32; e++) {
        exponent(e, t, 0, std::true_type{});
        weight(e);
        ds(e);
      }
#pragma unroll
      for (int q = 0; q < 16; q++) pack(q);
#pragma unroll
      for (int qt = 0; qt < DP_QT; qt++)
#pragma unroll
        for (int ss = 0; ss < 2; ss++) dsf[qt][ss] = dsf_next[qt][ss];
#pragma unroll
      for (int n = 0; n < 8; n++) fr[n] = kfrag(rows, 1, n);
      FENCE();
      for (; t + 1 < min(w_end, w_full); t++) {
        step(t, c0, std::false_type{});
        step(t, c1, std::false_type{});
      }
      for (; t < w_end; t++) {   // (behind the last tile a sub-tile is formed that nobody uses)
        step(t, c0, std::true_type{});
        step(t, c1, std::true_type{});
      }
    }
    // the other wavefronts' tiles: keep bringing this one's share of them
    for (; t < ntiles; t++) {
      barrier_image();
      all_image();
      barrier_rows();
      all_rows();
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

#pragma unroll
  for (int qt = 0; qt < DP_QT; qt++) {
    const int qi = wq0 + 32 * qt + i;
    if (kparts > 1) store_dq_part(dq_part, kpart, p, dq[qt], b, h, qi, g);
    else store_dq_row(p, dq[qt], b, h, qi, g);
  }
}

// ---------------------------------------------------------------------------------
// dK / dV
// ---------------------------------------------------------------------------------
// Key-stationary, 4 wavefronts x 64 keys, one per SIMD with its whole register file, lane = key column.  K and V
// rows stay in registers as B operands (128), dK^T and dV^T fill the accumulation registers (256); 64-query tiles of Q and dO stream
// through two-deep rings as row tiles (A operands of S and dP) and as transposed images (A operands of dV^T and
// dK^T); P and dS are accumulator tiles, which is the B-operand layout of the next product.
//
//      S  = Q K^T - lse/scale     the accumulators start at -lse/scale, so P = exp2(S c)
//      dP = dO V^T - delta        likewise -delta
//      dV^T += dO^T P             dK^T += Q^T (P o dP)
//
// The work goes by units of 32 queries x 32 keys.  While the 16 products of dV and dK of one unit and the 16 of S and dP of the next go through
// the matrix pipe, the exponentials, dS and the packing of that next unit are formed, two or three instructions under each product, so
// that both pipes are busy by the order of the instructions.  (Both halves of the keys in one go would read every fragment once instead of twice,
// but needs 70 registers more than there are.)  The order of the sums, and with it every bit of dK and dV, is that of the
// kernel before, which had 8 wavefronts of 32 keys, two per SIMD, each forming a unit's parts one after the other.  Bound: power.
// us before / here, two boxes: 4 heads, L = 32768, causal 1886 / 1640 (constant operands, where power is no bound, 1511 / 1160: the matrix pipe 58 / 75 %
// busy), 32 heads on 8, L = 16384 3861 / 3390, 4 heads, 8192 queries on 16384 keys 471 / 410.  Of the gain 2 % is one wait for four
// fragments in the place of four.
constexpr int KV_WAVES = 4, KV_KT = 2, KV_BN = 32 * KV_KT * KV_WAVES, KV_BQ = 64, KV_THREADS = 64 * KV_WAVES;
constexpr int KV_STAT_ELEMS = 64 * 8;                                    // start-value record of one tile: 1 KB, one direct load
constexpr int KV_ROWS = 2 * TILE_ELEMS + KV_STAT_ELEMS, KV_IMAGES = 2 * IMG_ELEMS;   // Q, dO tiles and start values; Q^T, dO^T images
static_assert(KV_WAVES == 4, "the load split and the vmcnt waits assume 4 wavefronts");

// dS kept for the dQ kernel (Lq and Lk multiples of 256; causal: Lq == Lk): one 128 KB block per (256-key block kb,
// 256-query block qb; causal: qb >= kb), laid out for the reader, which takes 64 keys x 256 queries at a time:
//   [64-key tile y = 0..3][64-query tile x = 0..3][chunk c = 0..7][key 0..63][8 bf16]
// Element j of chunk c is the query of tile row 32 (j >> 2) + 16 (c & 1) + 4 (j & 3) + ((c >> 1) & 1) + 2 (c >> 2) -- the
// order in which an accumulator holds the rows, i.e. image_pos(row) = 8 c + j.  Blocks of one (batch, head) are
// contiguous, key block after key block, and inside a key block by qb.  Entries of masked pairs are 0; the parts
// (y, x) of a diagonal block with y > x, whose keys all come after their queries, are never written (and never used).
constexpr int DS_PIECE = 64 * 8;                 // one (y, x, c): 1 KB
constexpr int DS_PART = 4 * 8 * DS_PIECE;        // one y: 32 KB
constexpr int DS_BLOCK_ELEMS = 4 * DS_PART;
// nbq, nbk: 256-row blocks of queries and of keys.  Causal (nbq == nbk): the blocks at or below the diagonal.
__host__ __device__ inline int64_t ds_blocks_per_head(int nbq, int nbk, bool causal) {
  return causal ? (int64_t)nbq * (nbq + 1) / 2 : (int64_t)nbq * nbk;
}
__host__ __device__ inline int64_t ds_block_index(int nbq, int kb, int qb, bool causal) {
  return causal ? (int64_t)kb * nbq - (int64_t)kb * (kb - 1) / 2 + (qb - kb) : (int64_t)kb * nbq + qb;
}

// S and dP do not start from zero: the accumulators of a sub-tile are loaded with -lse/scale and -delta of their
// rows, so that S comes out of the MFMAs as q.k - lse/scale and P = exp2(S c) costs one multiply and one exp per
// element.  A lane's 16 accumulator rows depend on its lane group only, so the 32 lanes of a group read the same 16
// floats (4 broadcast reads of 16 bytes per product).  The query-side pre-pass (attn_bwd_prepass_kernel) writes them:
// per (batch, head, tile) a table [sub-tile mt][0: -lse/scale, 1: -delta][lane group g][register r] of fp32 at the
// start of a 1 KB record, register r of group g being query acc_tile_row(r, g, mt).  Rows that must give P = 0
// (beyond Lq, or a query that saw no key) hold minus infinity.
//
// SPLIT = false: a block owns 256 keys of a kv head with one query head.
// SPLIT = true (grouped-query attention, or too few key blocks for the chip): a block owns 256 keys for ONE query
// head and part `bc.h % qparts` of that head's query tiles, and writes fp32 partial dK / dV to `part`, which
// attn_bwd_group_sum_kernel adds up over the group and the parts.  With few kv heads, or few keys against many
// queries (a ring step over a short key block), this is what gives the chip enough, and evenly sized, blocks.
//
// KEEP_DS = true (whole 256-row blocks on both sides; causal: self-attention): every dS tile also goes to p.ds, in the
// layout described at ds_block_index, and the dQ kernel below (attn_bwd_dq_kept_kernel) reads it back
// instead of computing S, dP and dS a second time.
template <bool SPLIT, bool KEEP_DS>
__global__ __launch_bounds__(KV_THREADS, 1) void attn_bwd_dkdv_pipe_kernel(const AttnParams p,
                                                                            const bf16* __restrict__ qimg,
                                                                            const bf16* __restrict__ doimg,
                                                                            const bf16* __restrict__ stats,
                                                                            float* __restrict__ part, int qparts) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  bf16* rring = reinterpret_cast<bf16*>(smem_raw);   // [2][KV_ROWS]
  bf16* iring = rring + 2 * KV_ROWS;                 // [2][KV_IMAGES]

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5,
            i = lane & 31;
  const BlockCoord bc = ody_block_coord(SPLIT ? p.Hq * qparts : p.Hkv, p.B);   // rank 0 = first key block = most query tiles
  const int h = SPLIT ? bc.h / qparts : bc.h, qpart = SPLIT ? bc.h % qparts : 0;   // (unless SPLIT, every head has keys of its own)
  const int hk = SPLIT ? h / p.group : h, b = bc.b;
  const int n0 = bc.rank * KV_BN, wn0 = n0 + wave * 32 * KV_KT;
  const int q_tiles = (p.Lq + KV_BQ - 1) / KV_BQ;

  const int t_begin = p.causal ? max(0, n0 - p.off) / KV_BQ : 0;   // first query tile that sees a key of this block
  int total = max(0, q_tiles - t_begin), t_top = q_tiles - 1;   // this block's tiles: t_top, t_top - 1, ... (total of them)
  if (SPLIT && qparts > 1) {
    const int per = (total + qparts - 1) / qparts;
    t_top -= qpart * per;
    total = max(0, min(per, total - qpart * per));
  }
  // (last query tile first: the key blocks of an XCD then read the same Q / dO tiles at the same time and share them through L2)
  // of them, those that see a key of this wavefront, and before them those that see all of its keys
  int w_total = total, w_full = total;
  if (p.causal) {
    w_total = min(total, max(0, t_top + 1 - max(0, wn0 - p.off) / KV_BQ));
    w_full = min(total, max(0, t_top + 1 - (max(0, wn0 + 32 * KV_KT - 1 - p.off) + KV_BQ - 1) / KV_BQ));
  }

  f32x16 dk[KV_KT][DT], dv[KV_KT][DT];
#pragma unroll
  for (int kh = 0; kh < KV_KT; kh++)
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int r = 0; r < 16; r++) dk[kh][dt][r] = dv[kh][dt][r] = 0.f;
  const float c2 = p.scale_log2e;

  // Direct loads: of the rows of tile `lr` (from the top) and of the images of tile `li`, the last one again where there are no more.
  // Rows past the end read zeros: they lie beyond the descriptor.
  const int last_tile = max(total - 1, 0), t_start = max(t_top, 0);   // (a block without tiles brings one and leaves it)
  int lr = 0, li = 0;
  const int qrow = 2 * (int)p.sq.l, orow = 2 * (int)p.sdo.l;   // bytes
  const int qlane = (4 * wave + (lane >> 4)) * qrow + 16 * (lane & 15), olane = (4 * wave + (lane >> 4)) * orow + 16 * (lane & 15);
  const int ilane = 1024 * wave + 16 * lane;
  const int64_t tile_id = ((int64_t)b * p.Hq + h) * q_tiles + t_start;
  const bf16* qtp = static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h + (int64_t)t_start * KV_BQ * p.sq.l;
  const bf16* otp = static_cast<const bf16*>(p.dout) + b * p.sdo.b + h * p.sdo.h + (int64_t)t_start * KV_BQ * p.sdo.l;
  const bf16* stp = stats + tile_id * KV_STAT_ELEMS;
  const bf16* qip = qimg + tile_id * IMG_ELEMS;
  const bf16* oip = doimg + tile_id * IMG_ELEMS;
  const int top_rows = min(KV_BQ, p.Lq - t_start * KV_BQ) - 1;
  int q_bytes = top_rows * qrow + 256, o_bytes = top_rows * orow + 256;
  auto bring = [&](const bf16* src, int bytes, bf16* dst, int off, int soff) INLINE {
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(src), (short)0, bytes, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_ptr)dst, 16, off, soff, 0, 0);
  };
  // a quarter j of the rows (two instructions per wavefront), of the images; every wavefront brings the whole record of start values
  auto load_rows = [&](int j, int which) INLINE {
    bf16* dst = rring + (lr & 1) * KV_ROWS + (4 * j + wave) * GROUP_ELEMS;
    if (which == 0) bring(qtp, q_bytes, dst, qlane + 16 * j * qrow, 0);
    else bring(otp, o_bytes, dst + TILE_ELEMS, olane + 16 * j * orow, 0);
  };
  auto load_stats = [&]() INLINE { bring(stp, 2 * KV_STAT_ELEMS, rring + (lr & 1) * KV_ROWS + 2 * TILE_ELEMS, ilane - 1024 * wave, 0); };
  auto load_images = [&](int j, int which) INLINE {
    bring(which ? oip : qip, IMG_BYTES, iring + (li & 1) * KV_IMAGES + which * IMG_ELEMS + (4 * j + wave) * 512, ilane, 4096 * j);
  };
  auto next_rows = [&]() INLINE {
    const int to = min(lr + 1, last_tile), step = to - lr;
    lr = to;
    qtp -= (int64_t)step * (KV_BQ / 2 * qrow);
    otp -= (int64_t)step * (KV_BQ / 2 * orow);
    stp -= step * KV_STAT_ELEMS;
    if (step) q_bytes = (KV_BQ - 1) * qrow + 256, o_bytes = (KV_BQ - 1) * orow + 256;
  };
  auto next_images = [&]() INLINE {
    const int to = min(li + 1, last_tile), step = to - li;
    li = to;
    qip -= step * IMG_ELEMS;
    oip -= step * IMG_ELEMS;
  };

  auto all_rows = [&]() INLINE {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      load_rows(j, 0);
      load_rows(j, 1);
    }
  };
  auto all_images = [&]() INLINE {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      load_images(j, 0);
      load_images(j, 1);
    }
  };

  // The first tiles, and this block's keys behind the first rows: one wait for memory in front of the first products (attn_fwd_pipe.hip).  Of the
  // second tile not the start values: those the first unit brings, like those of any tile.
  load_stats();
  all_rows();
  FENCE();
  bf16x8 kf[KV_KT][KS], vf[KV_KT][KS];
  {
    const bf16* kp = static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h;
    const bf16* vp = static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h;
#pragma unroll
    for (int kh = 0; kh < KV_KT; kh++) {
      const int key = min(wn0 + 32 * kh + i, p.Lk - 1);   // keys past the end: the last one, whose results are not stored
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        kf[kh][ks] = *reinterpret_cast<const bf16x8*>(kp + (int64_t)key * p.sk.l + 16 * ks + 8 * g);
        vf[kh][ks] = *reinterpret_cast<const bf16x8*>(vp + (int64_t)key * p.sv.l + 16 * ks + 8 * g);
      }
    }
  }
  FENCE();
  all_images();
  next_rows();
  all_rows();
  FENCE();
#pragma unroll
  for (int kh = 0; kh < KV_KT; kh++)
#pragma unroll
    for (int ks = 0; ks < KS; ks++) asm volatile("" : "+v"(kf[kh][ks]), "+v"(vf[kh][ks]));

  const int rbase = row_frag_base(g, i), ibase = image_frag_base(g, i);
  // + 32 kh: the first query that sees this lane's keys; less what of an accumulator's row goes by the lane (acc_tile_row), so that the mask compares
  // this one register with scalars: with a register per row the loops went to scratch memory
  const int key_off = p.causal ? wn0 + i - p.off - 16 * g : -(1 << 30);
  f32x16 s, dp;                          // S, then P; dP, then dS
  bf16x8 pf[2], dsf[2], pf_next[2], dsf_next[2];
  // a lane's 16 start values: quarter a of those of S (which = 0) or dP (1) of sub-tile mt
  auto start_values = [&](const bf16* rows, int mt, int which, int a, f32x16& x) INLINE {
    const f32x4 v = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(rows + 2 * TILE_ELEMS) + mt * 64 + which * 32 + g * 16 + 4 * a);
#pragma unroll
    for (int e = 0; e < 4; e++) x[4 * a + e] = v[e];
  };
  // the steps of element r of a unit: exponent, P, dS, and two elements together into the operands
  auto exponent = [&](int r, int t, int mt, int kh, auto masked) INLINE {
    float x = s[r] * c2;
    if (decltype(masked)::value) x = key_off > t * KV_BQ + acc_tile_row(r, 0, mt) - 32 * kh ? -INFINITY : x;   // queries before the key
    s[r] = x;
  };
  auto weight = [&](int r) INLINE { s[r] = ody_exp2(s[r]); };
  auto ds = [&](int r) INLINE { dp[r] *= s[r]; };
  auto pack = [&](bf16x8 (&dst)[2], const f32x16& src, int q) INLINE {
    dst[q >> 2][2 * q & 7] = (bf16)src[2 * q], dst[q >> 2][(2 * q & 7) + 1] = (bf16)src[2 * q + 1];
  };
  // s_waitcnt lgkmcnt(4), lgkmcnt(8): with the reads that are issued behind them in the order below, half of `fr` is there (one wait for four
  // fragments: the compiler's own would be one for each)
  constexpr int LGKM_4 = 0xc47f, LGKM_8 = 0xc87f;
  bf16x8 fr[8];
  auto qfrag = [&](const bf16* rows, int mt, int n) INLINE { return row_frag(rows, rbase, n, mt); };                   // k-step n
  auto ofrag = [&](const bf16* rows, int mt, int n) INLINE { return row_frag(rows + TILE_ELEMS, rbase, n, mt); };
  auto ifrag = [&](const bf16* im, int mt, int m) INLINE {   // m = 2 n + which: dO^T (0) or Q^T (1) image, k-step n >> 2, columns of 32 n & 3
    return image_frag(im + ((m & 1) ? 0 : IMG_ELEMS), ibase, (m >> 1) & 3, m >> 3, mt);
  };
  auto rslot = [&](int it) INLINE { return rring + (it & 1) * KV_ROWS; };
  auto islot = [&](int it) INLINE { return iring + (it & 1) * KV_IMAGES; };
  // (Where dS is kept its stores count as well, so that these waits are for a few more loads than they name.)
  auto barrier_rows = [&]() INLINE {     // the rows of the next tile have landed (behind them 8 loads of images); everyone is done with those before
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    next_rows();
  };
  auto barrier_images = [&]() INLINE {   // likewise the images (behind them 9 loads of rows and start values)
    asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    next_images();
  };
  auto keep = [&](bf16* ds_tile, int mt, int kh, int ss) INLINE {
    // Kept dS: dsf[ss] is chunk 4 mt + 2 ss + g of this lane's key, 512 contiguous bytes per half wavefront.  Streaming stores: the tiles are
    // read once, by another kernel.
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    __builtin_nontemporal_store(__builtin_bit_cast(u32x4, dsf[ss]),
                                reinterpret_cast<u32x4*>(ds_tile + (unsigned)((4 * mt + 2 * ss + g) * DS_PIECE + (32 * kh + i) * 8)));
  };

  // The work goes by units of 32 queries (sub-tile mt of tile it) x 32 keys (half kh).  One call: S and dP of the unit after (it, MT, KH), then dV
  // and dK of this one, 16 products each; the vector work of the unit after runs under these 32.  `fr` holds the first 8 fragments of either
  // part and is left with those of the next.
  auto unit = [&](int it, auto mt_, auto kh_, auto masked, bf16* ds_tile) INLINE {
    constexpr int MT = decltype(mt_)::value, KH = decltype(kh_)::value;
    constexpr int NKH = KH ^ 1, NMT = KH ? MT ^ 1 : MT;                  // the unit after
    constexpr int AMT = MT ^ 1;                                          // sub-tile of the unit behind that
    const int nt = KH && MT ? it + 1 : it, t = t_top - nt;
    const bf16 *rows = rslot(nt), *after = MT ? rslot(it + 1) : rslot(it), *images = islot(it);
#pragma unroll
    for (int m = 0; m < 16; m++) {
      if (m == 4) __builtin_amdgcn_s_waitcnt(LGKM_8);
      else if ((m & 3) == 0) __builtin_amdgcn_s_waitcnt(LGKM_4);
      if (m < 8) mfma32_onto(s, fr[m], kf[NKH][m]);
      else mfma32_onto(dp, fr[m - 8], vf[NKH][m - 8]);
      FENCE();
      if (m < 4) start_values(rows, NMT, 1, m, dp);
      fr[m & 7] = m < 8 ? ofrag(rows, NMT, m) : ifrag(images, MT, m - 8);
      if (m >= 11) weight(2 * m - 22), weight(2 * m - 21);
      if (m >= 10) exponent(2 * m - 20, t, NMT, NKH, masked), exponent(2 * m - 19, t, NMT, NKH, masked);   // (S is 3 products old)
      if (KEEP_DS && (m == 2 || m == 5)) keep(ds_tile, MT, KH, m == 5);
      // the rows of the tile after the next one: from the barrier in the third unit to the one in the first
      if (MT == 1 && KH == 1 && (m & 3) == 1) load_rows(m >> 2, 0);
      if (MT == 0 && KH == 0 && m == 3) load_stats();
      if (MT == 0 && KH == 0 && m == 7) barrier_images();
      // the images of the next one: from there on to the barrier in the third unit
      if (MT == 0 && KH == 1 && (m & 3) == 1) load_images(m >> 2, 1);
      FENCE();
    }
#pragma unroll
    for (int m = 0; m < 16; m++) {
      if (m == 12) __builtin_amdgcn_s_waitcnt(LGKM_8);
      else if ((m & 3) == 0) __builtin_amdgcn_s_waitcnt(LGKM_4);
      if (m & 1) dk[KH][(m >> 1) & 3] = mfma32(fr[m & 7], dsf[m >> 3], dk[KH][(m >> 1) & 3]);
      else dv[KH][(m >> 1) & 3] = mfma32(fr[m & 7], pf[m >> 3], dv[KH][(m >> 1) & 3]);
      FENCE();
      fr[m & 7] = m < 8 ? ifrag(images, MT, m + 8) : qfrag(after, AMT, m - 8);
      if (m <= 2) weight(2 * m + 10), weight(2 * m + 11);
      if (m <= 1) exponent(2 * m + 12, t, NMT, NKH, masked), exponent(2 * m + 13, t, NMT, NKH, masked);
      if (m >= 2 && m < 8) {   // S is done with by product 7: its start values must be there when the next part begins
#pragma unroll
        for (int r = 0; r < 3; r++)
          if (3 * (m - 2) + r < 16) ds(3 * (m - 2) + r);
      }
      if (m >= 3 && m < 7) pack(pf_next, s, 2 * m - 6), pack(pf_next, s, 2 * m - 5);
      if (m >= 8) pack(dsf_next, dp, m - 8);
      if (m == 8 || m == 9) start_values(after, AMT, 0, 2 * m - 16, s), start_values(after, AMT, 0, 2 * m - 15, s);
      if (MT == 1 && KH == 1 && (m & 3) == 1) load_rows(m >> 2, 1);
      if (MT == 1 && KH == 0 && m == 7) barrier_rows();
      if (MT == 0 && KH == 0 && (m & 3) == 1) load_images(m >> 2, 0);
      FENCE();
    }
#pragma unroll
    for (int ss = 0; ss < 2; ss++) pf[ss] = pf_next[ss], dsf[ss] = dsf_next[ss];
  };
  std::integral_constant<int, 0> c0;
  std::integral_constant<int, 1> c1;
  auto kept = [&](int it) INLINE -> bf16* {   // this wavefront's 64 keys of tile `it` among the kept dS
    if (!KEEP_DS) return nullptr;
    const int t = t_top - it, nbq = q_tiles / 4, nbk = p.Lk / KV_BN;
    return p.ds + (((int64_t)b * p.Hq + h) * ds_blocks_per_head(nbq, nbk, p.causal) + ds_block_index(nbq, bc.rank, t >> 2, p.causal)) * DS_BLOCK_ELEMS +
           ((wave * 4 + (t & 3)) * 8) * DS_PIECE;
  };

  if (total > 0) {
    asm volatile("s_waitcnt vmcnt(16)" ::: "memory");   // the first tile's rows
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int it = 0;
    if (w_total > 0) {
      // S, P, dP and dS of the first unit
      const bf16* rows = rslot(0);
#pragma unroll
      for (int a = 0; a < 4; a++) {
        start_values(rows, 0, 0, a, s);
        start_values(rows, 0, 1, a, dp);
      }
#pragma unroll
      for (int n = 0; n < 8; n++) {
        mfma32_onto(s, qfrag(rows, 0, n), kf[0][n]);
        mfma32_onto(dp, ofrag(rows, 0, n), vf[0][n]);
      }
      asm volatile("s_nop 15\n\ts_nop 7" : "+v"(s), "+v"(dp));
#pragma unroll
      for (int r = 0; r < 16; r++) {
        exponent(r, t_top, 0, 0, std::true_type{});
        weight(r);
        ds(r);
      }
#pragma unroll
      for (int q = 0; q < 8; q++) {
        pack(pf, s, q);
        pack(dsf, dp, q);
      }
#pragma unroll
      for (int a = 0; a < 4; a++) start_values(rows, 0, 0, a, s);
#pragma unroll
      for (int n = 0; n < 8; n++) fr[n] = qfrag(rows, 0, n);
      FENCE();
      for (; it + 1 < min(w_total, w_full); it++) {
        bf16* d = kept(it);
        unit(it, c0, c0, std::false_type{}, d);
        unit(it, c0, c1, std::false_type{}, d);
        unit(it, c1, c0, std::false_type{}, d);
        unit(it, c1, c1, std::false_type{}, d);
      }
      for (; it < w_total; it++) {   // (behind the last tile a unit is formed that nobody uses)
        bf16* d = kept(it);
        unit(it, c0, c0, std::true_type{}, d);
        unit(it, c0, c1, std::true_type{}, d);
        unit(it, c1, c0, std::true_type{}, d);
        unit(it, c1, c1, std::true_type{}, d);
      }
    }
    // the other wavefronts' tiles: keep bringing this one's share of them
    for (; it < total; it++) {
      load_stats();
      barrier_images();
      all_images();
      barrier_rows();
      all_rows();
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

#pragma unroll
  for (int kh = 0; kh < KV_KT; kh++) {
    const int key = wn0 + 32 * kh + i;
    if (key >= p.Lk) continue;
    if (SPLIT) {
      // part: [dK | dV][batch][query head][part of the queries][key][D] fp32, unscaled
      float* pk = part + (((int64_t)b * p.Hq * qparts + bc.h) * p.Lk + key) * D;
      float* pv = pk + (int64_t)p.B * p.Hq * qparts * p.Lk * D;
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int a = 0; a < 4; a++) {
          f32x4 wk, wv;
#pragma unroll
          for (int e = 0; e < 4; e++) wk[e] = dk[kh][dt][4 * a + e], wv[e] = dv[kh][dt][4 * a + e];
          *reinterpret_cast<f32x4*>(pk + 32 * dt + 8 * a + 4 * g) = wk;
          *reinterpret_cast<f32x4*>(pv + 32 * dt + 8 * a + 4 * g) = wv;
        }
    } else {
      bf16* dvp = static_cast<bf16*>(p.dv) + b * p.sdv.b + hk * p.sdv.h + (int64_t)key * p.sdv.l;
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int a = 0; a < 4; a++) {
          bf16x4 wv;
#pragma unroll
          for (int e = 0; e < 4; e++) wv[e] = (bf16)dv[kh][dt][4 * a + e];
          *reinterpret_cast<bf16x4*>(dvp + 32 * dt + 8 * a + 4 * g) = wv;
        }
      store_dk_row(p, dk[kh], b, hk, key, g);
    }
  }
}

// ---------------------------------------------------------------------------------
// dQ from the kept dS
// ---------------------------------------------------------------------------------
// One product, dQ^T += K^T dS^T, over the tiles that the dK/dV kernel (KEEP_DS) left in p.ds.  256 queries per block,
// 8 wavefronts x 32 queries: wavefront w owns chunks 4 (w & 1) ... + 3 of 64-query tile (w >> 1) of the block, lane i
// the query at position 32 (w & 1) + i of that tile's kept order.
//
//      A: K^T image (LDS, 16-byte reads), as in the dQ kernel at the top of this file
//      B: dS^T.  The tiles hold 8 queries of one key side by side, the product contracts over keys: the transposing
//         LDS read turns 4 keys x 16 queries into 4-key pieces per query, two of them make a fragment.
//
// 2 bytes per visible (query, key) pair for 256 flops: the kernel is bound by HBM, and what it needs is bytes in
// flight -- more than the LDS could take as landing room.  So the dS of a 64-key tile (32 one-KB pieces, 4 per
// wavefront) and its K^T image (2 KB per wavefront) travel through registers: four sets, loaded four tiles ahead,
// written to one of two LDS buffers the iteration before their tile is due.  (Direct loads to LDS for the images
// would put two kinds of loads on the one counter, and the compiler then waits for all of them every time.)
// The compiler places the waits for the register loads by counting the loads issued since, so these must leave in
// program order: no pass may move a load across this point, neither the optimizer nor the instruction scheduler.
#define ISSUE_ORDER()                    \
  do {                                   \
    asm volatile("" ::: "memory");       \
    __builtin_amdgcn_sched_barrier(0);   \
  } while (0)
constexpr int DS_PIECE_ELEMS = GROUP_ELEMS;   // 1 KB + 16 bytes: consecutive pieces start 4 banks apart
constexpr int DQK_DS_BUF = 32 * DS_PIECE_ELEMS, DQK_SETS = 4;
constexpr int DQK_LDS_ELEMS = 2 * DQK_DS_BUF + 2 * IMG_ELEMS;

//
// kparts > 1 (too few query blocks for the chip: a ring step of few queries against a long key block): block id =
// part + kparts * (the usual id), the block takes part `part` of its 256-key blocks and leaves its unscaled fp32 sum in
// dq_part [part][B][Lq][Hq][D]; attn_bwd_dq_sum_kernel adds the parts and finishes dq.
__global__ __launch_bounds__(DQ_THREADS) void attn_bwd_dq_kept_kernel(const AttnParams p, const bf16* __restrict__ kimg,
                                                                       int kparts, float* __restrict__ dq_part) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  bf16* dsbuf = reinterpret_cast<bf16*>(smem_raw);   // [2][DQK_DS_BUF]
  bf16* imgs = dsbuf + 2 * DQK_DS_BUF;               // [2][IMG_ELEMS]

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5,
            i = lane & 31;
  const int kpart = blockIdx.x % kparts;
  const BlockCoord bc = ody_block_coord_of(blockIdx.x / kparts, p.Hq, p.B);
  const int nqb = gridDim.x / (p.Hq * p.B * kparts);
  const int qblk = p.causal ? nqb - 1 - bc.rank : bc.rank;   // causal: heaviest blocks first
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int x = wave >> 1, mt = wave & 1, nbq = p.Lq / KV_BN, nbk = p.Lk / KV_BN;
  const bf16* kip = kimg + ((int64_t)b * p.Hkv + hk) * (p.Lk / 64) * IMG_ELEMS;
  const bf16* dsh = p.ds + ((int64_t)b * p.Hq + h) * ds_blocks_per_head(nbq, nbk, p.causal) * DS_BLOCK_ELEMS;
  // 64-key tiles: all of them, or (causal) those up to the block's last query; a multiple of DQK_SETS
  int ntiles = p.causal ? 4 * (qblk + 1) : 4 * nbk;
  const int last_tile = p.causal ? 4 * qblk + x : ntiles;   // of this wavefront's queries
  int t_first = 0;   // this block's part of the tiles: [t_first, ntiles), whole 256-key blocks
  if (kparts > 1) {
    const int per = 4 * ((ntiles / 4 + kparts - 1) / kparts);
    t_first = min(kpart * per, ntiles);
    ntiles = min(t_first + per, ntiles);
  }
  // position 32 mt + i of the tile's kept order = chunk 4 mt + (i >> 3), element i & 7
  const int qrow = qblk * DQ_BM + KV_BQ * x + 32 * ((i >> 2) & 1) + 16 * ((i >> 3) & 1) + 4 * (i & 3) + (i >> 4) + 2 * mt;
  auto store_part = [&](const f32x16 (&acc)[DT]) { store_dq_part(dq_part, kpart, p, acc, b, h, qrow, g); };

  u32x4 regs[DQK_SETS][6];
  // tile t: this wavefront's 4 of the 32 pieces (x, c) of key tile t & 3 of block (t >> 2, qblk) -- 32 KB in a row --
  // and its 2 of the 16 KB of the K^T image, into register set `set`
  auto issue = [&](int set, int t) {
    const bf16* src = dsh + ds_block_index(nbq, t >> 2, qblk, p.causal) * DS_BLOCK_ELEMS + (t & 3) * DS_PART;
#pragma unroll
    for (int n = 0; n < 4; n++) {   // piece 8 n + wave: query tile n of the block, chunk `wave`
      regs[set][n] = *reinterpret_cast<const u32x4*>(src + (unsigned)((8 * n + wave) * DS_PIECE + lane * 8));
      ISSUE_ORDER();
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
      regs[set][4 + j] = *reinterpret_cast<const u32x4*>(kip + (int64_t)t * IMG_ELEMS + (unsigned)(((DQ_WAVES * j + wave) * 64 + lane) * 8));
      ISSUE_ORDER();
    }
  };
  auto drain = [&](int set, int t) {
    bf16* buf = dsbuf + (t & 1) * DQK_DS_BUF;
#pragma unroll
    for (int n = 0; n < 4; n++)
      *reinterpret_cast<u32x4*>(buf + (8 * n + wave) * DS_PIECE_ELEMS + lane * 8) = regs[set][n];
    bf16* slot = imgs + (t & 1) * IMG_ELEMS;
#pragma unroll
    for (int j = 0; j < 2; j++)
      *reinterpret_cast<u32x4*>(slot + ((DQ_WAVES * j + wave) * 64 + lane) * 8) = regs[set][4 + j];
  };
  f32x16 dq[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) dq[dt][r] = 0.f;
  if (t_first >= ntiles) {   // a part without keys (causal: an early query block has fewer key blocks than parts)
    store_part(dq);
    return;
  }
#pragma unroll
  for (int u = 0; u < DQK_SETS; u++) issue(u, t_first + u);   // ntiles - t_first >= DQK_SETS

  const int ibase = image_frag_base(g, i);
  // the transposing read: inside 16 lanes, lane 4 k + m supplies key 4 k (+ the fragment's row offset) and queries
  // 4 m ... 4 m + 3 of the 16; queries 0-7 of the 16 are one chunk, 8-15 the next
  const int sbase = (8 * x + 4 * mt + 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1)) * DS_PIECE_ELEMS +
                    (16 * g + 4 * ((lane >> 2) & 3)) * 8 + 4 * (lane & 1);

  auto tile = [&](int t) {
    const bf16* Sp = dsbuf + (t & 1) * DQK_DS_BUF + sbase;
    const bf16* Ki = imgs + (t & 1) * IMG_ELEMS;
    constexpr int IPF = 4;
    bf16x8 ifr[IPF], dsf[2][2];
#pragma unroll
    for (int n = 0; n < IPF; n++) ifr[n] = image_frag(Ki, ibase, n & 3, 0, 0);
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
      for (int ss = 0; ss < 2; ss++)   // keys 32 (j >> 2) + 16 g + 4 (j & 3) + ss + 2 kt, j = 0..7
        dsf[kt][ss] = concat4(lds_read_tr16(Sp + (ss + 2 * kt) * 8), lds_read_tr16(Sp + (ss + 2 * kt) * 8 + 32 * 8));
    FENCE();
#pragma unroll
    for (int n = 0; n < 16; n++) {
      const int dt = n & 3, ss = (n >> 2) & 1, kt = n >> 3;
      dq[dt] = mfma32(ifr[n % IPF], dsf[kt][ss], dq[dt]);
      if (n + IPF < 16) {
        const int m = n + IPF;
        ifr[n % IPF] = image_frag(Ki, ibase, m & 3, (m >> 2) & 1, m >> 3);
      }
      FENCE();
    }
  };

  drain(0, t_first);
  ISSUE_ORDER();
  int t0 = t_first;
  do {   // not a `for`: its entry test would give the compiler a block to sink the loads above into, out of order
#pragma unroll
    for (int u = 0; u < DQK_SETS; u++) {
      const int t = t0 + u;
      // everyone is done with tile t - 1, and sees what the wavefronts wrote of tile t to LDS an iteration ago
      __syncthreads();
      // tile t + 1 has arrived (the compiler places the wait: all loads are of one kind, so it can count them);
      // tiles t + 2 and t + 3 may still be on their way, and tile t + 4 sets out
      // No branches around these (past the end: a write that nobody reads, and one more load of the last tile):
      // with branches the compiler loses count of the loads in flight and waits for all of them.
      ISSUE_ORDER();
      drain((u + 1) % DQK_SETS, t + 1);
      ISSUE_ORDER();
      issue(u, min(t + DQK_SETS, ntiles - 1));
      // (causal) tiles whose keys all come after this wavefront's queries were never written
      if (t <= last_tile) tile(t);
    }
  } while ((t0 += DQK_SETS) < ntiles);

  if (kparts > 1) store_part(dq);
  else store_dq_row(p, dq, b, h, qrow, g);
}

// dq = the sum of the fp32 parts of a key-split dQ kernel, finished like store_dq_row does; one thread per
// 4 elements d..d+3 of the first half of a (query, head) row and their partners d + 64 (the pairs of the rotary
// embedding)
__global__ __launch_bounds__(256) void attn_bwd_dq_sum_kernel(const AttnParams p, const float* __restrict__ dq_part, int kparts) {
  constexpr int Q = D / 8;
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;   // over B * Lq * Hq * D / 8
  const int64_t total = (int64_t)p.B * p.Lq * p.Hq * Q;
  if (idx >= total) return;
  const int d4 = idx % Q;
  const int h = (idx / Q) % p.Hq;
  const int qi = (idx / ((int64_t)Q * p.Hq)) % p.Lq;
  const int b = idx / ((int64_t)Q * p.Hq * p.Lq);
  const int64_t plane = (int64_t)p.B * p.Lq * p.Hq * D;
  const float* src = dq_part + (((int64_t)b * p.Lq + qi) * p.Hq + h) * D + 4 * d4;
  f32x4 s1 = {0.f, 0.f, 0.f, 0.f}, s2 = s1;
  for (int s = 0; s < kparts; s++) {
    s1 += *reinterpret_cast<const f32x4*>(src + s * plane);
    s2 += *reinterpret_cast<const f32x4*>(src + s * plane + D / 2);
  }
  s1 *= p.scale;
  s2 *= p.scale;
  if (p.dq_f32) {
    float* dqp = static_cast<float*>(p.dq) + b * p.sdq.b + h * p.sdq.h + (int64_t)qi * p.sdq.l + 4 * d4;
    if (p.accumulate_dq) {
      s1 += *reinterpret_cast<const f32x4*>(dqp);
      s2 += *reinterpret_cast<const f32x4*>(dqp + D / 2);
    }
    *reinterpret_cast<f32x4*>(dqp) = s1;
    *reinterpret_cast<f32x4*>(dqp + D / 2) = s2;
    return;
  }
  bf16* dqp = static_cast<bf16*>(p.dq) + b * p.sdq.b + h * p.sdq.h + (int64_t)qi * p.sdq.l + 4 * d4;
  bf16x4 w1, w2;
  if (p.rope_q) {
    const bf16x8 cs = *reinterpret_cast<const bf16x8*>(p.rope_q + ((int64_t)b * p.Lq + qi) * D + 8 * d4);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float c = (float)cs[2 * e], sn = (float)cs[2 * e + 1];
      w1[e] = (bf16)(s1[e] * c + s2[e] * sn);
      w2[e] = (bf16)(s2[e] * c - s1[e] * sn);
    }
  } else {
    if (p.accumulate_dq) {
      const bf16x4 o1 = *reinterpret_cast<const bf16x4*>(dqp), o2 = *reinterpret_cast<const bf16x4*>(dqp + D / 2);
#pragma unroll
      for (int e = 0; e < 4; e++) s1[e] += (float)o1[e], s2[e] += (float)o2[e];
    }
#pragma unroll
    for (int e = 0; e < 4; e++) w1[e] = (bf16)s1[e], w2[e] = (bf16)s2[e];
  }
  *reinterpret_cast<bf16x4*>(dqp) = w1;
  *reinterpret_cast<bf16x4*>(dqp + D / 2) = w2;
}

// dK, dV of a kv head = sum of the fp32 partials of its query heads and their `qparts` parts; one thread per 4 elements
// d..d+3 of the first half of a key row and their partners d + 64 (the pairs of the rotary embedding)
__global__ __launch_bounds__(256) void attn_bwd_group_sum_kernel(const AttnParams p, const float* __restrict__ part,
                                                                 int qparts) {
  constexpr int Q = D / 8;                                                // threads per key row
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;           // over B * Hkv * Lk * D / 8
  const int64_t total = (int64_t)p.B * p.Hkv * p.Lk * Q;
  if (idx >= total) return;
  const int d4 = idx % Q;
  const int key = (idx / Q) % p.Lk;
  const int hk = (idx / ((int64_t)Q * p.Lk)) % p.Hkv;
  const int b = idx / ((int64_t)Q * p.Lk * p.Hkv);
  const int64_t plane = (int64_t)p.B * p.Hq * qparts * p.Lk * D;
  f32x4 sk1 = {0.f, 0.f, 0.f, 0.f}, sk2 = sk1, sv1 = sk1, sv2 = sk1;
  for (int hg = 0; hg < p.group * qparts; hg++) {   // (query head of the group, part), in this fixed order
    const float* src = part + ((((int64_t)b * p.Hkv + hk) * p.group * qparts + hg) * p.Lk + key) * D + 4 * d4;
    sk1 += *reinterpret_cast<const f32x4*>(src);
    sk2 += *reinterpret_cast<const f32x4*>(src + D / 2);
    sv1 += *reinterpret_cast<const f32x4*>(src + plane);
    sv2 += *reinterpret_cast<const f32x4*>(src + plane + D / 2);
  }
  bf16x4 wk1, wk2, wv1, wv2;
  if (p.rope_k) {
    const bf16x8 cs = *reinterpret_cast<const bf16x8*>(p.rope_k + ((int64_t)b * p.Lk + key) * D + 8 * d4);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float c = (float)cs[2 * e], sn = (float)cs[2 * e + 1];
      const float g1 = sk1[e] * p.scale, g2 = sk2[e] * p.scale;
      wk1[e] = (bf16)(g1 * c + g2 * sn);
      wk2[e] = (bf16)(g2 * c - g1 * sn);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++) wk1[e] = (bf16)(sk1[e] * p.scale), wk2[e] = (bf16)(sk2[e] * p.scale);
  }
#pragma unroll
  for (int e = 0; e < 4; e++) wv1[e] = (bf16)sv1[e], wv2[e] = (bf16)sv2[e];
  bf16* dkp = static_cast<bf16*>(p.dk) + b * p.sdk.b + hk * p.sdk.h + (int64_t)key * p.sdk.l + 4 * d4;
  bf16* dvp = static_cast<bf16*>(p.dv) + b * p.sdv.b + hk * p.sdv.h + (int64_t)key * p.sdv.l + 4 * d4;
  *reinterpret_cast<bf16x4*>(dkp) = wk1;
  *reinterpret_cast<bf16x4*>(dkp + D / 2) = wk2;
  *reinterpret_cast<bf16x4*>(dvp) = wv1;
  *reinterpret_cast<bf16x4*>(dvp + D / 2) = wv2;
}

inline size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// Parts of the other side's range, for a kernel with `blocks` blocks that each walk `tiles` 64-row tiles.  As for the
// forward's key split: with fewer blocks than it takes to keep the chip's 256 compute units busy and balanced -- one
// block each when all are equally long, two each under a causal mask, where they are not and only a second, lighter
// block per unit lets the heaviest-first order even that out -- the range is cut into 2 or 4 parts of at least 16
// tiles (on average, when causal).
inline int range_parts(int64_t blocks, int tiles, bool causal) {
  const int64_t want = causal ? 512 : 256;
  int s = 1;
  while (s < 4 && blocks * s * 2 <= want && tiles >= 32 * s) s *= 2;
  return s;
}
// dK/dV: parts of the query range of a (256-key block, query head)
inline int query_parts(int B, int Lq, int Lk, int Hq, int Hkv, bool causal) {
  const int64_t blocks = (int64_t)B * Hq * ((Lk + KV_BN - 1) / KV_BN);   // already one per QUERY head when they are split
  return range_parts(blocks, (Lq + KV_BQ - 1) / KV_BQ, causal);
}
// dQ (either kernel): parts of the key range of a (256-query block, head)
inline int key_parts(int B, int Lq, int Lk, int Hq, bool causal) {
  return range_parts((int64_t)B * Hq * ((Lq + DQ_BM - 1) / DQ_BM), (Lk + 63) / 64, causal);
}
// fp32 partial dK / dV (grouped-query attention, or a split query range) and partial dQ (a split key range) share one
// region: the first is summed up before the second is written.  Sized for the larger of the causal and the unmasked
// policy, since the size query does not know the mask.
inline size_t partials_bytes(int B, int Lq, int Lk, int Hq, int Hkv) {
  const int qp = std::max(query_parts(B, Lq, Lk, Hq, Hkv, false), query_parts(B, Lq, Lk, Hq, Hkv, true));
  const int kp = std::max(key_parts(B, Lq, Lk, Hq, false), key_parts(B, Lq, Lk, Hq, true));
  const size_t kv = (Hq == Hkv && qp == 1) ? 0 : (size_t)2 * B * Hq * qp * Lk * D * sizeof(float);
  const size_t dq = kp == 1 ? 0 : (size_t)kp * B * Lq * Hq * D * sizeof(float);
  return align256(std::max(kv, dq));
}

}  // namespace

// workspace after delta: the transposed images of K, Q and dO, the per-tile start values and, for
// grouped-query attention, the fp32 partial dK / dV of every query head
size_t ody_attn_bwd_pipe_workspace(int B, int Lq, int Lk, int Hq, int Hkv) {
  return align256(ody_attn_images_bytes(B, Lk, Hkv)) + 2 * align256(ody_attn_images_bytes(B, Lq, Hq)) +
         align256((size_t)B * Hq * ((Lq + KV_BQ - 1) / KV_BQ) * KV_STAT_ELEMS * sizeof(bf16)) +
         partials_bytes(B, Lq, Lk, Hq, Hkv);
}

size_t ody_attn_bwd_pipe_ds_bytes(int B, int Lq, int Lk, int Hq, int causal) {
  if (Lq % KV_BN != 0 || Lk % KV_BN != 0 || (causal && Lq != Lk) || B <= 0 || Hq <= 0) return 0;
  return (size_t)B * Hq * ds_blocks_per_head(Lq / KV_BN, Lk / KV_BN, causal != 0) * DS_BLOCK_ELEMS * sizeof(bf16);
}

int ody_launch_attn_bwd_pipe(const AttnParams& p, void* workspace, hipStream_t st) {
  constexpr size_t smem_q = (size_t)2 * (DP_ROWS + IMG_ELEMS) * sizeof(bf16);
  constexpr size_t smem_kv = (size_t)2 * (KV_ROWS + KV_IMAGES) * sizeof(bf16);
  constexpr size_t smem_qs = (size_t)DQK_LDS_ELEMS * sizeof(bf16);
  static_assert(smem_qs <= 160 * 1024, "LDS of one CU");
  for (const auto& ks : {std::pair<const void*, size_t>{reinterpret_cast<const void*>(&attn_bwd_dq_pipe_kernel), smem_q},
                         {reinterpret_cast<const void*>(&attn_bwd_dq_kept_kernel), smem_qs},
                         {reinterpret_cast<const void*>(&attn_bwd_dkdv_pipe_kernel<false, false>), smem_kv},
                         {reinterpret_cast<const void*>(&attn_bwd_dkdv_pipe_kernel<true, false>), smem_kv},
                         {reinterpret_cast<const void*>(&attn_bwd_dkdv_pipe_kernel<false, true>), smem_kv},
                         {reinterpret_cast<const void*>(&attn_bwd_dkdv_pipe_kernel<true, true>), smem_kv}})
    if (int rc = ody_allow_dynamic_lds(ks.first, ks.second, "attn_bwd")) return rc;
  unsigned char* w = static_cast<unsigned char*>(workspace);
  bf16* kimg = reinterpret_cast<bf16*>(w);
  bf16* qimg = reinterpret_cast<bf16*>(w + align256(ody_attn_images_bytes(p.B, p.Lk, p.Hkv)));
  bf16* doimg = reinterpret_cast<bf16*>(w + align256(ody_attn_images_bytes(p.B, p.Lk, p.Hkv)) +
                                        align256(ody_attn_images_bytes(p.B, p.Lq, p.Hq)));
  bf16* stats = reinterpret_cast<bf16*>(reinterpret_cast<unsigned char*>(doimg) +
                                        align256(ody_attn_images_bytes(p.B, p.Lq, p.Hq)));
  int rc;
  // everything that depends on q, dout, out and lse only: delta, Q / dO images, start values
  if (!p.reuse_query_side && (rc = ody_launch_attn_bwd_prepass(p, qimg, doimg, stats, st))) return rc;
  float* part = reinterpret_cast<float*>(
      reinterpret_cast<unsigned char*>(stats) +
      align256((size_t)p.B * p.Hq * ((p.Lq + KV_BQ - 1) / KV_BQ) * KV_STAT_ELEMS * sizeof(bf16)));
  auto group_sum = [&](int qparts) {
    const int64_t n8 = (int64_t)p.B * p.Hkv * p.Lk * (D / 8);
    ODY_LAUNCH("attn_bwd_group_sum", st, attn_bwd_group_sum_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, p,
               part, qparts);
    return ody_check_launch("attn_bwd_group_sum");
  };
  const int qparts = query_parts(p.B, p.Lq, p.Lk, p.Hq, p.Hkv, p.causal != 0);
  // dK and dV are the same bits whether dS is kept or not; where that is a choice (rows in multiples of 256), a cut query range keeps a call on
  // the kernels below.  It costs what the others gain: causal, 4 heads, L = 2048 109 us here, 65 there, 8 heads, L = 3584 178 and 124
  const bool same_sums = qparts == 1 || ody_attn_bwd_pipe_ds_bytes(p.B, p.Lq, p.Lk, p.Hq, p.causal) == 0;
  // rows too far apart for the 32-bit offsets of a tile below: that kernel's are 64 bits wide
  const bool far = std::max(std::max(p.sq.l, p.sdo.l), std::max(p.sk.l, p.sv.l)) >= TILE_MAX_STRIDE;
  if (far || (!p.ds && same_sums && ody_attn_bwd_short_ok(p.B, p.Lq, p.Lk, p.Hq, p.causal))) {
    // the pre-pass wrote the query side whole: a later call that reuses it may run on the kernels below
    if ((rc = ody_launch_attn_bwd_short(p, stats, part, st)) || p.group == 1) return rc;
    return group_sum(1);
  }
  if ((rc = ody_launch_attn_images(p.k, p.sk, p.B, p.Lk, p.Hkv, kimg, nullptr, 0, st))) return rc;
  const int key_blocks = (p.Lk + KV_BN - 1) / KV_BN;
  if (p.group == 1 && qparts == 1) {
    if (p.ds)
      ODY_LAUNCH("attn_bwd_dkdv_pipe", st, (attn_bwd_dkdv_pipe_kernel<false, true>), dim3(key_blocks * p.Hkv * p.B),
                 dim3(KV_THREADS), smem_kv, p, qimg, doimg, stats, nullptr, 1);
    else
      ODY_LAUNCH("attn_bwd_dkdv_pipe", st, (attn_bwd_dkdv_pipe_kernel<false, false>), dim3(key_blocks * p.Hkv * p.B),
                 dim3(KV_THREADS), smem_kv, p, qimg, doimg, stats, nullptr, 1);
    if ((rc = ody_check_launch("attn_bwd_dkdv_pipe"))) return rc;
  } else {
    if (p.ds)
      ODY_LAUNCH("attn_bwd_dkdv_pipe", st, (attn_bwd_dkdv_pipe_kernel<true, true>), dim3(key_blocks * p.Hq * qparts * p.B),
                 dim3(KV_THREADS), smem_kv, p, qimg, doimg, stats, part, qparts);
    else
      ODY_LAUNCH("attn_bwd_dkdv_pipe", st, (attn_bwd_dkdv_pipe_kernel<true, false>), dim3(key_blocks * p.Hq * qparts * p.B),
                 dim3(KV_THREADS), smem_kv, p, qimg, doimg, stats, part, qparts);
    if ((rc = ody_check_launch("attn_bwd_dkdv_pipe"))) return rc;
    if ((rc = group_sum(qparts))) return rc;
  }
  dim3 gq(((p.Lq + DQ_BM - 1) / DQ_BM) * p.Hq * p.B);
  if (p.ds) {
    // what ody_attn_bwd_pipe_ds_bytes promised: whole 256-row blocks on both sides, queries and keys aligned
    ODY_REQUIRE(p.Lq % KV_BN == 0 && p.Lk % KV_BN == 0 && (!p.causal || p.off == 0) && KV_BN == DQ_BM, ODY_ERR_UNSUPPORTED,
                "attn_bwd: kept dS needs multiples of %d rows on both sides and, if causal, as many keys as queries", KV_BN);
    const int kparts = key_parts(p.B, p.Lq, p.Lk, p.Hq, p.causal != 0);
    ODY_LAUNCH("attn_bwd_dq_kept", st, attn_bwd_dq_kept_kernel, dim3(gq.x * kparts), dim3(DQ_THREADS), smem_qs, p, kimg, kparts,
               part);
    if ((rc = ody_check_launch("attn_bwd_dq_kept")) || kparts == 1) return rc;
    const int64_t n8 = (int64_t)p.B * p.Lq * p.Hq * (D / 8);
    ODY_LAUNCH("attn_bwd_dq_sum", st, attn_bwd_dq_sum_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, p, part, kparts);
    return ody_check_launch("attn_bwd_dq_sum");
  }
  const int kparts = key_parts(p.B, p.Lq, p.Lk, p.Hq, p.causal != 0);
  ODY_LAUNCH("attn_bwd_dq_pipe", st, attn_bwd_dq_pipe_kernel, dim3(gq.x * kparts), dim3(DP_THREADS), smem_q, p, kimg, kparts,
             part);
  if ((rc = ody_check_launch("attn_bwd_dq_pipe")) || kparts == 1) return rc;
  const int64_t n8 = (int64_t)p.B * p.Lq * p.Hq * (D / 8);
  ODY_LAUNCH("attn_bwd_dq_sum", st, attn_bwd_dq_sum_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, p, part, kparts);
  return ody_check_launch("attn_bwd_dq_sum");
}
