// Flash attention for bf16 and head_dim 128 where the kernels for long sequences (attn_fwd_pipe.hip, attn_bwd_pipe.hip) leave compute units
// idle or wait for latency: few blocks of 256 rows, each a few tiles long, behind passes that write transposed images.
//
// A block is 128 rows: 4 wavefronts of 32 rows, twice.  In the forward and for dQ the second four take every other key tile, so that the
// serial chain of tiles is half as long; the halves add up through LDS at the end.  For dK and dV the two sets share the tiles and the
// work: one holds dV, the other dK (S is formed twice, which costs less than the registers of both: a chain of three products instead of
// four).  Tiles come straight to LDS, two stages, and serve as row operands and, through the transposing read, as transposed ones
// (attn_rowtile.h), at half the LDS rate but without images: no pass that writes those of K and V (those of Q and dO come with the pre-pass, for later
// calls that reuse the query side).  All of the backward behind the pre-pass is one launch.
//
// The forward on more than a few tiles (the ring) takes a sub-tile of 32 keys of every tile per group instead, in the order of attn_fwd_pipe.hip: products,
// LDS reads and vector work of neighbouring sub-tiles under one another, loads four tiles ahead.
//
// What bounds it: latency of a chain of tiles in a block (2.2 us for 128 rows against 128 keys in the forward, 1.5 in the ring) on 1 block a unit.
// On the kernels for long sequences / here, us, launches included: forward of 4 x 8 heads, L = 331, causal 19.5 / 12.2 (three launches / one), backward on 2 kv
// heads 66 / 33.5 (five / three); 32 heads on 8, L = 1000, causal 38.3 / 20.4 and 110 / 69; 8 heads, L = 1500, full 40 / 23.8 and 129 / 58.
// Error against 64 bits, standard normal inputs, before / here: out 2.07e-3 / 1.96e-3 (4 x 8 heads, L = 331), 2.34e-3 / 2.31e-3 (640 rows,
// full); dQ, dK, dV the same within the spread of one input to the next (2.5e-3, 2.5e-3, 2.3e-3).
#include <algorithm>
#include <cfloat>
#include <type_traits>
#include <utility>
#include "attn_rowtile.h"
#include "attn_store.h"

namespace {

using namespace rowtile;

constexpr int D = 128, KS = D / 16, DT = D / 32, TILE = ROWS * D;   // elements of a tile: 16 KB
constexpr int BLOCK_ROWS = 128, WAVES = 8, GROUPS = 2;
constexpr size_t KV_STAGE = 2 * TILE;                    // elements: two tiles
constexpr size_t QS_STAGE = 2 * TILE + 512;              // Q and dO tiles, start values of S and dP (1 KB, written by the pre-pass)
constexpr size_t SMEM = GROUPS * 2 * KV_STAGE * sizeof(bf16);
static_assert(SMEM >= 4 * (16 * DT + 2) * 64 * sizeof(float) && SMEM >= 2 * QS_STAGE * sizeof(bf16) && SMEM <= 160 * 1024, "one block per unit");
typedef TileLoader<D, 4> GroupLoader;
constexpr int FW_STAGE = 2 * TILE;   // elements: K and V of a tile of the forward's ring of 4
static_assert(4 * FW_STAGE * sizeof(bf16) <= SMEM && 4 * QS_STAGE * sizeof(bf16) >= SMEM && 4 * QS_STAGE * sizeof(bf16) <= 160 * 1024, "the rings");
#define FENCE() __builtin_amdgcn_sched_barrier(0)
#define INLINE __attribute__((always_inline))
#define WAIT_LDS(n) asm volatile("s_waitcnt lgkmcnt(" #n ")" ::: "memory")

// A transposed fragment (tr_frags) whose reads are still under way: 16 rows from FIRST and FIRST + STEP on, 32 columns by the address pair
struct TrFrag {
  s16x4 lo, hi;
};
template <int FIRST, int STEP = 8>
__device__ __forceinline__ void read_tr(TrFrag& f, unsigned a0, unsigned a1) {
  asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%4\n\tds_read_b64_tr_b16 %1, %3 offset:%5"
               : "=&v"(f.lo), "=&v"(f.hi)
               : "v"(a0), "v"(a1), "n"(2 * FIRST * D), "n"(2 * (FIRST + STEP) * D));
}
// behind the wait for them
__device__ __forceinline__ void tie(TrFrag& f) { asm volatile("" : "+v"(f.lo), "+v"(f.hi)); }
__device__ __forceinline__ bf16x8 value(const TrFrag& f) {
  return concat4(__builtin_bit_cast(bf16x4, f.lo), __builtin_bit_cast(bf16x4, f.hi));
}
template <typename F, int... N>
__device__ __forceinline__ void each_of(const F& f, std::integer_sequence<int, N...>) {
  (f(std::integral_constant<int, N>{}), ...);
}
template <int COUNT, typename F>
__device__ __forceinline__ void each(const F& f) {
  each_of(f, std::make_integer_sequence<int, COUNT>{});
}

// ---------------------------------------------------------------------------------------------------------- forward
//   S^T = K Q^T      O^T += V^T P^T       lane = query column
__global__ __launch_bounds__(64 * WAVES, 2) void attn_fwd_short_kernel(const AttnParams p) {
  constexpr size_t STAGE_BYTES = KV_STAGE * sizeof(bf16);
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int grp = wave >> 2, w4 = wave & 3;
  bf16* ring = reinterpret_cast<bf16*>(smem) + grp * 2 * KV_STAGE;   // [2][K tile | V tile]
  const BlockCoord bc = ody_block_coord(p.Hq, p.B);
  const int nqb = gridDim.x / (p.Hq * p.B);
  const int qblk = p.causal ? nqb - 1 - bc.rank : bc.rank;   // heaviest blocks first
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * BLOCK_ROWS, wq0 = q0 + w4 * 32, qi = wq0 + i;

  int n_end = p.causal ? min(p.Lk, min(q0 + BLOCK_ROWS, p.Lq) + p.off) : p.Lk;
  const int ntiles = n_end > 0 ? (n_end + ROWS - 1) / ROWS : 0;
  GroupLoader lk, lv;
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
        bf16x8 pb[2], vf[2];
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const float x = ody_exp2(fmaf(s[kt][r], c2, -ref));
          l4[r & 3] += x;
          pb[r >> 3][r & 7] = (bf16)x;
        }
        auto product = [&](auto slice) {   // 16 keys, 64 columns of the head
          constexpr int ss = decltype(slice)::value & 1, hf = decltype(slice)::value >> 1;
          tr_frags<ROWS + 32 * kt + 16 * ss, hf>(vf, rd);
#pragma unroll
          for (int dt = 0; dt < 2; dt++) o[2 * hf + dt] = mfma32(vf[dt], pb[ss], o[2 * hf + dt]);
        };
        product(std::integral_constant<int, 0>{});
        product(std::integral_constant<int, 2>{});
        product(std::integral_constant<int, 1>{});
        product(std::integral_constant<int, 3>{});
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
    float* patch = reinterpret_cast<float*>(smem) + w4 * (16 * DT + 2) * 64;
    if (grp == from) {
      give(patch, o, lane);
      patch[16 * DT * 64 + lane] = ref;
      patch[(16 * DT + 1) * 64 + lane] = l;
    }
    __syncthreads();
    if (grp == 0) {
      const float ref1 = patch[16 * DT * 64 + lane], next = fmaxf(ref, ref1), a0 = ody_exp2(ref - next), a1 = ody_exp2(ref1 - next);
      take(patch, o, lane, a0, a1);
      l = l * a0 + patch[(16 * DT + 1) * 64 + lane] * a1;
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

// The same on more than a few tiles: a wavefront has one sub-tile of every tile of a ring of four, and forms S of the tile after (8 products) and P V of
// the present one (8), each product with one element of P and one or two LDS reads behind it; K rows are read half a turn ahead, V columns a quarter.
// Bound: the vector pipe and the reads from LDS beside the products, 1600 cycles a tile of 1024 of products, and the clock.  Before (products, vector
// work and the waits of the transposing reads one after the other, as above) / now, us, launch included: L = 1000, causal, 32 heads, 22.7 / 20.4,
// 16 heads 22.1 / 18.8; L = 2048, 8 heads, 36.8 / 28.4; L = 4096, 8 heads, against attn_fwd_pipe.hip's, 66 / 50.  Its fixed cost is 0.5 us more (a first
// pass through more code, two latencies in front of the loop): short rows are left to the loop above.
__global__ __launch_bounds__(64 * WAVES, 2) void attn_fwd_short_ring_kernel(const AttnParams p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int grp = wave >> 2, w4 = wave & 3;
  const BlockCoord bc = ody_block_coord(p.Hq, p.B);
  const int nqb = gridDim.x / (p.Hq * p.B);
  const int qblk = p.causal ? nqb - 1 - bc.rank : bc.rank;   // heaviest blocks first
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * BLOCK_ROWS, wq0 = q0 + w4 * 32, qi = wq0 + i;

  int n_end = p.causal ? min(p.Lk, min(q0 + BLOCK_ROWS, p.Lq) + p.off) : p.Lk;
  const int ntiles = n_end > 0 ? (n_end + ROWS - 1) / ROWS : 0;
  const bf16* kp = static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const bf16* vp = static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h;
  const int lim = p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1;   // last key this lane's query sees
  const float c2 = p.scale_log2e;
  bf16x8 qf[KS];
  f32x16 o[DT];
  float ref;     // the row's reference in log2 units
  float l4[4];   // this lane's partial row sums

  // The direct loads of a tile: halves of K (0, 1) and of V (2, 3), one instruction per wavefront each.  Rows past the end read zeros, and a tile past
  // the end nothing else: its loads are there to be counted.
  bf16* fring = reinterpret_cast<bf16*>(smem);   // [4][K tile | V tile]
  const int brow = 4 * wave + (lane >> 4), bcol = 16 * ((lane & 15) ^ swz<D>(brow)), krow = 2 * (int)p.sk.l, vrow = 2 * (int)p.sv.l;
  const int koff = brow * krow + bcol, voff = brow * vrow + bcol;
  auto load = [&](int t, int part) INLINE {
    const int rows = min(p.Lk - t * ROWS, ROWS), row = part < 2 ? krow : vrow;
    const bf16* src = (part < 2 ? kp : vp) + (int64_t)(t * ROWS) * (row / 2);
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(src), (short)0, t < ntiles ? (rows - 1) * row + 2 * D : 0, 0x00020000);
    bf16* dst = fring + (t & 3) * FW_STAGE + (part < 2 ? 0 : TILE) + (8 * (part & 1) + wave) * 512;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)dst, 16, (part < 2 ? koff : voff) + 32 * (part & 1) * row, 0, 0, 0);
  };
  // K of tile 0 and the queries first: what the first products wait for is not behind four tiles
  load(0, 0), load(0, 1);
  FENCE();
  fetch_rows(qf, static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h, p.sq.l, qi, p.Lq, g);
  FENCE();
#pragma unroll
  for (int t = 0; t < 4; t++) {
    if (t < 3) load(t + 1, 0), load(t + 1, 1);
    load(t, 2), load(t, 3);
  }
  settle_rows(qf, qi, p.Lq);
  // The reference of a row and a group is the largest score of its first two sub-tiles (a row that sees any key of the group's sees their first one) and
  // stays.  Of the first one alone it would do, but the further below a row's maximum it is, the coarser bf16 is where the large P lie (out of 32 heads,
  // L = 1000, 2.053e-3 from 64 bits, 2.033e-3 as in the loop above).  Sub-tile `grp` of every tile is this group's.
  const int sub_end = min(n_end, p.causal ? wq0 + 32 + p.off : n_end) - 32 * grp, sub_full = min(p.Lk, p.causal ? wq0 + 1 + p.off : p.Lk) - 32 * grp - 32;
  const int w_live = sub_end > 0 ? (sub_end + ROWS - 1) / ROWS : 0;   // sub-tiles with a key that this wavefront sees
  const int w_full = sub_full >= 0 ? sub_full / ROWS + 1 : 0;         // those of which all of its queries see all keys
  const int seen = lim - 32 * grp - 4 * g;   // last key this lane's query sees, from this lane's first one in tile 0 on
  f32x16 s[2];                       // of even and odd tiles
  bf16x8 pb[2][2], kfr[KS];          // P, alike; K rows: k-step n
  TrFrag vfr[2 * DT];                // V^T: 16 keys n / DT, columns 32 (n % DT)
  Readers<D> rd;
  rd.init(fring, g, i);
#pragma unroll
  for (int n = 0; n < KS; n++) rd.row[n] += 2 * 32 * D * grp, rd.tr[n] += 2 * 32 * D * grp;
  typedef const bf16x8 __attribute__((address_space(3))) * frag_ptr;
  // ODD: of the two tiles that the readers' place in the ring has
  auto read_k = [&](int n, int odd) INLINE { kfr[n] = *(frag_ptr)(uintptr_t)(rd.row[n] + odd * FW_STAGE * 2); };
  auto read_v = [&](auto n_, auto odd_) INLINE {
    constexpr int n = decltype(n_)::value, FIRST = decltype(odd_)::value * 2 * ROWS + ROWS + 16 * (n / DT);
    read_tr<FIRST>(vfr[n], rd.tr[2 * (n % DT)], rd.tr[2 * (n % DT) + 1]);
  };
  auto score = [&](int t, int par, int e, auto masked) INLINE {
    return decltype(masked)::value && acc_row(e, 0) > seen - t * ROWS ? -INFINITY : s[par][e];
  };
  // The vector work of a sub-tile in steps of a product's length from the first product of its S on: element e in step 10 + e; the products with
  // its first 8 elements begin in step 24.
  auto vector = [&](int step, int t, auto par_, auto masked) INLINE {
    constexpr int P = decltype(par_)::value;
    const int e = step - 10;
    if (e < 0 || e >= 16) return;
    const float x = ody_exp2(fmaf(score(t, P, e, masked), c2, -ref));
    l4[e & 3] += x;
    pb[P][e >> 3][e & 7] = (bf16)x;
  };
  std::integral_constant<int, 0> c0;
  std::integral_constant<int, 1> c1;
  // One call: S of the tile after t, then P V of tile t (P: t & 1), 8 products each; under them the vector work of both.
  auto unit = [&](int t, auto par_, auto masked) INLINE {
    constexpr int P = decltype(par_)::value;
    std::integral_constant<int, P ^ 1> other;
    auto slot = [&](auto m_) INLINE {
      constexpr int m = decltype(m_)::value;
      if (m == 8) {
        WAIT_LDS(0);
#pragma unroll
        for (int n = 0; n < 2 * DT; n++) tie(vfr[n]);
        // K of tile t + 2 and V of tile t + 1 have landed (behind them 6 loads); everyone is done with tile t
        asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      if (m < 8) s[P ^ 1] = mfma32(kfr[m & 7], qf[m & 7], m == 0 ? f32x16{0} : s[P ^ 1]);
      else o[m & 3] = mfma32(value(vfr[m & 7]), pb[P][(m & 7) >> 2], o[m & 3]);
      FENCE();
      if constexpr (m < 4) read_v(std::integral_constant<int, 4 + (m & 3)>{}, par_);
      if constexpr (m >= 8 && m < 12) read_k(2 * (m & 3), P), read_k(2 * (m & 3) + 1, P);
      if constexpr (m >= 12) read_v(std::integral_constant<int, m & 3>{}, other);
      if (m > 8 && (m & 1)) load(t + 4, (m - 9) >> 1);
      if (P == 1 && m == 4)
#pragma unroll
        for (int n = 0; n < KS; n++) rd.tr[n] += t & 2 ? -4 * FW_STAGE : 4 * FW_STAGE;
      if (P == 1 && m == 15)
#pragma unroll
        for (int n = 0; n < KS; n++) rd.row[n] += t & 2 ? 4 * FW_STAGE : -4 * FW_STAGE;
      vector(16 + m, t, par_, masked);
      vector(m, t + 1, other, masked);
      FENCE();
    };
    each<16>(slot);
  };
  auto clear_rows = [&]() INLINE {
    clear(o);
    ref = -FLT_MAX;   // no score is below it; not minus infinity, from which a masked score would be NaN
#pragma unroll
    for (int e = 0; e < 4; e++) l4[e] = 0.f;
  };
  clear_rows();
  if (ntiles > 0) {
    asm volatile("s_waitcnt vmcnt(14)" ::: "memory");   // K of tile 0
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int t = 0;
    if (w_live > 0) {
#pragma unroll
      for (int n = 0; n < KS; n++) read_k(n, 0);
#pragma unroll
      for (int n = 0; n < KS; n++) s[0] = mfma32(kfr[n], qf[n], n == 0 ? f32x16{0} : s[0]);
    }
    asm volatile("s_waitcnt vmcnt(10)" ::: "memory");   // K of tile 1, V of tile 0
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (w_live > 0) {
#pragma unroll
      for (int n = 0; n < KS; n++) read_k(n, 1);
      each<DT>([&](auto n) INLINE { read_v(n, c0); });
      // (S of the second one is formed again by the loop)
      float mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 16; e++) mx = fmaxf(mx, score(0, 0, e, std::true_type{}));
      if (w_live > 1) {
#pragma unroll
        for (int n = 0; n < KS; n++) s[1] = mfma32(kfr[n], qf[n], n == 0 ? f32x16{0} : s[1]);
#pragma unroll
        for (int e = 0; e < 16; e++) mx = fmaxf(mx, score(1, 1, e, std::true_type{}));
      }
      ref = fmaxf(ref, half_swap_max(mx) * c2);
#pragma unroll
      for (int m = 0; m < 16; m++) vector(m, 0, c0, std::true_type{});
#pragma unroll
      for (int n = 0; n < KS; n++) rd.row[n] += 4 * FW_STAGE;   // the loop reads rows two tiles ahead of columns
      FENCE();
      for (; t + 1 < w_live && t + 2 < w_full; t += 2) {
        unit(t, c0, std::false_type{});
        unit(t + 1, c1, std::false_type{});
      }
      for (; t + 1 < w_live; t += 2) {   // (behind the last tile one is formed that nobody uses)
        unit(t, c0, std::true_type{});
        unit(t + 1, c1, std::true_type{});
      }
      if (t < w_live) {   // an even tile is left
        each<DT>([&](auto n) INLINE { read_v(std::integral_constant<int, DT + decltype(n)::value>{}, c0); });
#pragma unroll
        for (int m = 0; m < 16; m++) vector(16 + m, t, c0, std::true_type{});
        WAIT_LDS(0);
#pragma unroll
        for (int n = 0; n < 2 * DT; n++) {
          tie(vfr[n]);
          o[n & 3] = mfma32(value(vfr[n]), pb[0][n >> 2], o[n & 3]);
        }
      } else {
        WAIT_LDS(0);   // the reads of the tile behind
#pragma unroll
        for (int n = 0; n < DT; n++) tie(vfr[n]);
      }
    }
    // the other wavefronts' tiles: keep bringing this one's share of them
    for (; t < ntiles; t++) {
      asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int j = 0; j < 4; j++) load(t + 4, j);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();   // everyone is done with the ring
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
    if (any) {   // once more, with the maximum so far as a row's reference, so that P <= 1 and P V overflows for no values that P = 1 would hold
      clear_rows();
      for (int t = 0; t < ntiles; t++) {
#pragma unroll
        for (int j = 0; j < 4; j++) load(t, j);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (t < w_live) {
          int own = lane;
          asm volatile("" : "+v"(own));   // so that no address of this is kept in a register meanwhile
          Readers<D> again;
          again.init(fring + (t & 3) * FW_STAGE + 32 * D * grp, own >> 5, own & 31);
#pragma unroll
          for (int n = 0; n < KS; n++) s[0] = mfma32(row_frag(again, 0, n), qf[n], n == 0 ? f32x16{0} : s[0]);
          float mx = -INFINITY;
#pragma unroll
          for (int e = 0; e < 16; e++) mx = fmaxf(mx, score(t, 0, e, std::true_type{}));
          const float next = fmaxf(ref, half_swap_max(mx) * c2), alpha = ody_exp2(ref - next);
          ref = next;
#pragma unroll
          for (int e = 0; e < 4; e++) l4[e] *= alpha;
#pragma unroll
          for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
#pragma unroll
          for (int m = 10; m < 26; m++) vector(m, t, c0, std::true_type{});
          auto product = [&](auto slice) INLINE {   // 16 keys, 64 columns of the head
            constexpr int ss = decltype(slice)::value >> 1, hf = decltype(slice)::value & 1;
            bf16x8 vf[2];
            tr_frags<ROWS + 16 * ss, hf>(vf, again);
#pragma unroll
            for (int dt = 0; dt < 2; dt++) o[2 * hf + dt] = mfma32(vf[dt], pb[0][ss], o[2 * hf + dt]);
          };
          each<4>(product);
        }
        __syncthreads();
      }
    }
  }

  float l = (l4[0] + l4[1]) + (l4[2] + l4[3]);
#pragma unroll 1
  for (int from = 1; from < GROUPS; from++) {
    float* patch = reinterpret_cast<float*>(smem) + w4 * (16 * DT + 2) * 64;
    if (grp == from) {
      give(patch, o, lane);
      patch[16 * DT * 64 + lane] = ref;
      patch[(16 * DT + 1) * 64 + lane] = l;
    }
    __syncthreads();
    if (grp == 0) {
      const float ref1 = patch[16 * DT * 64 + lane], next = fmaxf(ref, ref1), a0 = ody_exp2(ref - next), a1 = ody_exp2(ref1 - next);
      take(patch, o, lane, a0, a1);
      l = l * a0 + patch[(16 * DT + 1) * 64 + lane] * a1;
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
// dQ of 128 queries of a head: 4 wavefronts of 32 queries, two groups that take every other key tile.
//   S^T = K Q^T     dP^T = V dO^T - delta     dQ^T += K^T dS^T       lane = query column
__device__ __forceinline__ void dq_block(const AttnParams& p, unsigned char* smem, int q0, int h, int b) {
  constexpr size_t STAGE_BYTES = KV_STAGE * sizeof(bf16);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int grp = wave >> 2, w4 = wave & 3, hk = h / p.group, wq0 = q0 + w4 * 32, qi = wq0 + i;
  bf16* ring = reinterpret_cast<bf16*>(smem) + grp * 2 * KV_STAGE;   // [2][K tile | V tile]

  int n_end = p.causal ? min(p.Lk, min(q0 + BLOCK_ROWS, p.Lq) + p.off) : p.Lk;
  const int ntiles = n_end > 0 ? (n_end + ROWS - 1) / ROWS : 0;
  GroupLoader lk, lv;
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
  const float nd = qi < p.Lq ? -p.delta[head * p.Lq + qi] : 0.f;
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
      bf16x8 kf[2];
      auto product = [&](auto slice) {
        constexpr int ss = decltype(slice)::value & 1, hf = decltype(slice)::value >> 1;
        tr_frags<32 * kt + 16 * ss, hf>(kf, rd);
#pragma unroll
        for (int dt = 0; dt < 2; dt++) dq[2 * hf + dt] = mfma32(kf[dt], dsf[ss], dq[2 * hf + dt]);
      };
      product(std::integral_constant<int, 0>{});
      product(std::integral_constant<int, 2>{});
      product(std::integral_constant<int, 1>{});
      product(std::integral_constant<int, 3>{});
    };
    sub_tile(std::integral_constant<int, 0>{});
    sub_tile(std::integral_constant<int, 1>{});
    rd.move((it & 1) ? -(int)STAGE_BYTES : (int)STAGE_BYTES);
  }

  float* patch = reinterpret_cast<float*>(smem) + w4 * 16 * DT * 64;
  __syncthreads();
  if (grp == 1) give(patch, dq, lane);
  __syncthreads();
  if (grp == 1) return;
  take(patch, dq, lane, 1.f, 1.f);
  store_dq_row(p, dq, b, h, qi, g);
}

// The same in the order of attn_fwd_short_ring_kernel: a wavefront has one sub-tile of every tile, and forms S and dP of the tile after (16 products)
// and dQ of the present one (8) with the vector work of the former under them.
__device__ __forceinline__ void dq_ring_block(const AttnParams& p, unsigned char* smem, int q0, int h, int b) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int grp = wave >> 2, w4 = wave & 3, hk = h / p.group, wq0 = q0 + w4 * 32, qi = wq0 + i;
  const int n_end = p.causal ? min(p.Lk, min(q0 + BLOCK_ROWS, p.Lq) + p.off) : p.Lk;
  const int ntiles = n_end > 0 ? (n_end + ROWS - 1) / ROWS : 0;
  const bf16* kp = static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const bf16* vp = static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h;
  const float c2 = p.scale_log2e;
  bf16* ring = reinterpret_cast<bf16*>(smem);   // [4][K tile | V tile]
  const int brow = 4 * wave + (lane >> 4), bcol = 16 * ((lane & 15) ^ swz<D>(brow)), krow = 2 * (int)p.sk.l, vrow = 2 * (int)p.sv.l;
  const int koff = brow * krow + bcol, voff = brow * vrow + bcol;
  auto load = [&](int t, int part) INLINE {   // as in attn_fwd_short_ring_kernel
    const int rows = min(p.Lk - t * ROWS, ROWS), row = part < 2 ? krow : vrow;
    const bf16* src = (part < 2 ? kp : vp) + (int64_t)(t * ROWS) * (row / 2);
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(src), (short)0, t < ntiles ? (rows - 1) * row + 2 * D : 0, 0x00020000);
    bf16* dst = ring + (t & 3) * FW_STAGE + (part < 2 ? 0 : TILE) + (8 * (part & 1) + wave) * 512;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)dst, 16, (part < 2 ? koff : voff) + 32 * (part & 1) * row, 0, 0, 0);
  };
  // tile 0 and the queries first: what the first products wait for is not behind four tiles
#pragma unroll
  for (int j = 0; j < 4; j++) load(0, j);
  FENCE();
  bf16x8 qf[KS], dof[KS];
  fetch_rows(qf, static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h, p.sq.l, qi, p.Lq, g);
  fetch_rows(dof, static_cast<const bf16*>(p.dout) + b * p.sdo.b + h * p.sdo.h, p.sdo.l, qi, p.Lq, g);
  const int64_t head = (int64_t)b * p.Hq + h;
  float lse2 = p.lse[head * p.Lq + min(qi, p.Lq - 1)], delta = p.delta[head * p.Lq + min(qi, p.Lq - 1)];
  FENCE();
#pragma unroll
  for (int t = 1; t < 4; t++)
#pragma unroll
    for (int j = 0; j < 4; j++) load(t, j);
  settle_rows(qf, qi, p.Lq);
  settle_rows(dof, qi, p.Lq);
  asm volatile("" : "+v"(lse2), "+v"(delta));
  lse2 = qi >= p.Lq || lse2 == -INFINITY ? INFINITY : lse2 * ODY_LOG2E;   // past the end, or a query that saw no key: P = 0
  if (qi >= p.Lq) delta = 0.f;

  const int lim = p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1;   // last key this lane's query sees
  const int sub_end = min(n_end, p.causal ? wq0 + 32 + p.off : n_end) - 32 * grp, sub_full = min(p.Lk, p.causal ? wq0 + 1 + p.off : p.Lk) - 32 * grp - 32;
  const int w_live = sub_end > 0 ? (sub_end + ROWS - 1) / ROWS : 0;   // sub-tiles with a key that this wavefront sees
  const int w_full = sub_full >= 0 ? sub_full / ROWS + 1 : 0;         // those of which all of its queries see all keys
  const int seen = lim - 32 * grp - 4 * g;   // last key this lane's query sees, from this lane's first one in tile 0 on
  f32x16 s, dp, dq[DT];
  clear(dq);
  bf16x8 ds[2][2], fr[KS];   // dS of even and odd tiles; rows of K, then of V, k-step n
  TrFrag tf[DT];             // K^T: columns 32 n
  Readers<D> rd;
  rd.init(ring, g, i);
#pragma unroll
  for (int n = 0; n < KS; n++) rd.row[n] += 2 * 32 * D * grp, rd.tr[n] += 2 * 32 * D * grp;
  typedef const bf16x8 __attribute__((address_space(3))) * frag_ptr;
  auto read_row = [&](int n, int which, int odd) INLINE { fr[n] = *(frag_ptr)(uintptr_t)(rd.row[n] + odd * FW_STAGE * 2 + which * TILE * 2); };
  auto read_col = [&](auto n_, auto odd_) INLINE {   // 16 keys n / DT, columns 32 (n % DT)
    constexpr int n = decltype(n_)::value, FIRST = decltype(odd_)::value * 2 * ROWS + 16 * (n / DT);
    read_tr<FIRST>(tf[n % DT], rd.tr[2 * (n % DT)], rd.tr[2 * (n % DT) + 1]);
  };
  // The vector work of a sub-tile in steps of a product's length from the first product of its S on: element e becomes P in step 9 + 11 e / 16 and
  // dS in step 18 + 6 e / 16.
  auto vector = [&](int step, int t, auto par_, auto masked) INLINE {
    constexpr int P = decltype(par_)::value;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      if (18 + 6 * e / 16 == step) {
        dp[e] = (dp[e] - delta) * s[e];
        if (e & 1) ds[P][e >> 3][(e & 7) - 1] = (bf16)dp[e - 1], ds[P][e >> 3][e & 7] = (bf16)dp[e];
      }
      if (9 + 11 * e / 16 == step) {
        const float x = decltype(masked)::value && acc_row(e, 0) > seen - t * ROWS ? -INFINITY : s[e];
        s[e] = ody_exp2(fmaf(x, c2, -lse2));
      }
    }
  };
  std::integral_constant<int, 0> c0;
  std::integral_constant<int, 1> c1;
  auto unit = [&](int t, auto par_, auto masked) INLINE {   // P: t & 1
    constexpr int P = decltype(par_)::value;
    std::integral_constant<int, P ^ 1> other;
    auto slot = [&](auto m_) INLINE {
      constexpr int m = decltype(m_)::value;
      if (m == 12)   // they are there; later the compiler's wait for one would be a wait for the transposing reads as well
#pragma unroll
        for (int n = 4; n < KS; n++) asm volatile("" : "+v"(fr[n]));
      if constexpr (m >= 16) {
        if (m == 20) {
          WAIT_LDS(0);
#pragma unroll
          for (int n = 0; n < DT; n++) tie(tf[n]);
          // tile t + 2 has landed (behind it the 4 loads of the next); everyone is done with tile t, and with V of the one after
          asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
        } else if (m < 20) {
          WAIT_LDS(6);
          tie(tf[m & 3]);
        }
      }
      if (m < 8) s = mfma32(fr[m & 7], qf[m & 7], m == 0 ? f32x16{0} : s);
      else if (m < 16) dp = mfma32(fr[m & 7], dof[m & 7], m == 8 ? f32x16{0} : dp);
      else dq[m & 3] = mfma32(value(tf[m & 3]), ds[P][(m & 7) >> 2], dq[m & 3]);
      FENCE();
      if constexpr (m < 8) read_row(m, 1, P ^ 1);
      if constexpr (m >= 12 && m < 20) read_col(std::integral_constant<int, m - 12>{}, par_);
      if constexpr (m >= 20) {
        read_row(2 * (m & 3), 0, P), read_row(2 * (m & 3) + 1, 0, P);
        load(t + 4, m & 3);
      }
      if (P == 0 && m == 10)
#pragma unroll
        for (int n = 0; n < KS; n++) rd.row[n] += t & 2 ? -4 * FW_STAGE : 4 * FW_STAGE;
      if (P == 1 && m == 20)
#pragma unroll
        for (int n = 0; n < KS; n++) rd.tr[n] += t & 2 ? -4 * FW_STAGE : 4 * FW_STAGE;
      vector(m, t + 1, other, masked);
      FENCE();
    };
    each<24>(slot);
  };
  if (ntiles > 0) {
    asm volatile("s_waitcnt vmcnt(12)" ::: "memory");   // tile 0
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int t = 0;
    if (w_live > 0) {
#pragma unroll
      for (int n = 0; n < KS; n++) read_row(n, 0, 0);
#pragma unroll
      for (int n = 0; n < KS; n++) s = mfma32(fr[n], qf[n], n == 0 ? f32x16{0} : s);
#pragma unroll
      for (int n = 0; n < KS; n++) read_row(n, 1, 0);
#pragma unroll
      for (int n = 0; n < KS; n++) dp = mfma32(fr[n], dof[n], n == 0 ? f32x16{0} : dp);
    }
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");   // tile 1
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (w_live > 0) {
#pragma unroll
      for (int n = 0; n < KS; n++) read_row(n, 0, 1);
#pragma unroll
      for (int m = 9; m < 24; m++) vector(m, 0, c0, std::true_type{});
      FENCE();
      for (; t + 1 < w_live && t + 2 < w_full; t += 2) {
        unit(t, c0, std::false_type{});
        unit(t + 1, c1, std::false_type{});
      }
      for (; t + 1 < w_live; t += 2) {   // (behind the last tile one is formed that nobody uses)
        unit(t, c0, std::true_type{});
        unit(t + 1, c1, std::true_type{});
      }
      if (t < w_live) {   // an even tile is left
        auto half = [&](auto ss_) INLINE {
          constexpr int ss = decltype(ss_)::value;
          each<DT>([&](auto n) INLINE { read_col(std::integral_constant<int, DT * ss + decltype(n)::value>{}, c0); });
          WAIT_LDS(0);
#pragma unroll
          for (int n = 0; n < DT; n++) {
            tie(tf[n]);
            dq[n] = mfma32(value(tf[n]), ds[0][ss], dq[n]);
          }
        };
        half(c0);
        half(c1);
      }
    }
    // the other wavefronts' tiles: keep bringing this one's share of them
    for (; t < ntiles; t++) {
      asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int j = 0; j < 4; j++) load(t + 4, j);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  float* patch = reinterpret_cast<float*>(smem) + w4 * 16 * DT * 64;
  __syncthreads();
  if (grp == 1) give(patch, dq, lane);
  __syncthreads();
  if (grp == 1) return;
  take(patch, dq, lane, 1.f, 1.f);
  store_dq_row(p, dq, b, h, qi, g);
}

// dK^T or dV^T of a key, to its row or to the fp32 parts
template <bool PART, bool IS_DK>
__device__ __forceinline__ void store_kv_row(const AttnParams& p, const f32x16 (&acc)[DT], int b, int h, int hk, int key, int g, float* __restrict__ part) {
  if (key >= p.Lk) return;
  if constexpr (PART) {   // [dK | dV][B][Hq][Lk][D] in fp32
    float* dst = part + (IS_DK ? 0 : (int64_t)p.B * p.Hq * p.Lk * D) + (((int64_t)b * p.Hq + h) * p.Lk + key) * D;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        f32x4 w;
#pragma unroll
        for (int e = 0; e < 4; e++) w[e] = acc[dt][4 * a + e];
        *reinterpret_cast<f32x4*>(dst + 32 * dt + 8 * a + 4 * g) = w;
      }
  } else if constexpr (IS_DK) {
    store_dk_row(p, acc, b, hk, key, g);
  } else {
    store_row(static_cast<bf16*>(p.dv) + b * p.sdv.b + hk * p.sdv.h + (int64_t)key * p.sdv.l, acc, 1.f, g);
  }
}

// One of dK and dV of 32 keys per wavefront, over the query tiles of one query head: wavefronts 0 - 3 of a block hold dV of its 128
// keys, 4 - 7 dK.
//   S = Q K^T - lse / scale     dV^T += dO^T P                                              lane = key column
//                               dP = dO V^T - delta     dK^T += Q^T (P o dP)
// Start values, order of the rows and of the sums are those of attn_bwd_dkdv_pipe_kernel, and so are the results, bit for bit, as long as
// that one does not cut its query range: dK and dV do not depend on whether a caller keeps dS.
//
// The two roles are two instances: in one loop with a branch on the role the compiler gives both the registers of both, and spills.
// Each passes the same barriers, one per query tile.
template <bool PART, bool IS_DK>
__device__ __forceinline__ void kv_block(const AttnParams& p, unsigned char* smem, int n0, int h, int b, const bf16* __restrict__ stats,
                                         float* __restrict__ part) {
  constexpr size_t STAGE_BYTES = QS_STAGE * sizeof(bf16);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int hk = h / p.group, wn0 = n0 + (wave & 3) * 32, key = wn0 + i;
  bf16* ring = reinterpret_cast<bf16*>(smem);   // [2][Q tile | dO tile | row values]
  const int t_begin = p.causal ? max(0, n0 - p.off) / ROWS : 0, t_end = (p.Lq + ROWS - 1) / ROWS;
  const int total = max(0, t_end - t_begin);
  TileLoader<D, WAVES, true> lq, lo;
  lq.init(p.sq.l, wave, lane);
  lo.init(p.sdo.l, wave, lane);
  const bf16* qp = static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h;
  const bf16* dop = static_cast<const bf16*>(p.dout) + b * p.sdo.b + h * p.sdo.h;
  const bf16* sp = stats + ((int64_t)b * p.Hq + h) * t_end * 512 + lane * 8;
  auto load = [&](int t, int buf) {
    bf16* st = ring + buf * QS_STAGE;
    lq.load(st, qp, t * ROWS, p.Lq, wave);
    lo.load(st + TILE, dop, t * ROWS, p.Lq, wave);
    if (!IS_DK && wave == 0)
      __builtin_amdgcn_global_load_lds((global_ptr)(sp + (int64_t)t * 512), (lds_ptr)(st + 2 * TILE), 16, 0, 0);
  };
  if (total > 0) load(t_end - 1, 0);

  bf16x8 kf[KS], vf[IS_DK ? KS : 1];
  load_rows(kf, static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h, p.sk.l, key, p.Lk, g);
  if constexpr (IS_DK) load_rows(vf, static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h, p.sv.l, key, p.Lk, g);
  const float c2 = p.scale_log2e;
  Readers<D, true> rd;
  rd.init(ring, g, i);
  f32x16 acc[DT];   // dK^T or dV^T
  clear(acc);

  for (int n = 0; n < total; n++) {
    const int i0 = (t_end - 1 - n) * ROWS;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (n + 1 < total) load(t_end - 2 - n, (n + 1) & 1);
    // every query of the tile comes before every key of this wavefront: nothing to do
    const bool dead = p.causal && i0 + ROWS - 1 + p.off < wn0;
    const float* rv = reinterpret_cast<const float*>(ring + (n & 1) * QS_STAGE + 2 * TILE) + 16 * g;
    auto sub_tile = [&](auto which) {
      __builtin_amdgcn_sched_barrier(0);   // one sub-tile's fragments at a time
      constexpr int mt = decltype(which)::value;
      f32x16 s, dp;
#pragma unroll
      for (int a = 0; a < 4; a++) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(rv + 64 * mt + 4 * a);
#pragma unroll
        for (int e = 0; e < 4; e++) s[4 * a + e] = x[e];
        if constexpr (IS_DK) {
          const f32x4 y = *reinterpret_cast<const f32x4*>(rv + 64 * mt + 32 + 4 * a);
#pragma unroll
          for (int e = 0; e < 4; e++) dp[4 * a + e] = y[e];
        }
      }
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        s = mfma32(row_frag(rd, 2 * mt, ks), kf[ks], s);
        if constexpr (IS_DK) dp = mfma32(row_frag(rd, ROWS + 2 * mt, ks), vf[ks], dp);
      }
      if (p.causal && i0 + p.off < wn0 + 31) {
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (i0 + tile128::acc_tile_row(r, g, mt) + p.off < key) s[r] = -INFINITY;
      }
      bf16x8 pf[2];   // P, or dS
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const float pr = ody_exp2(s[r] * c2);
        pf[r >> 3][r & 7] = (bf16)(IS_DK ? pr * dp[r] : pr);
      }
      bf16x8 f[2];
      auto product = [&](auto slice) {
        constexpr int ss = decltype(slice)::value & 1, hf = decltype(slice)::value >> 1;
        tr_frags<(IS_DK ? 0 : ROWS) + 2 * mt + ss, hf>(f, rd);
#pragma unroll
        for (int dt = 0; dt < 2; dt++) acc[2 * hf + dt] = mfma32(f[dt], pf[ss], acc[2 * hf + dt]);
      };
      product(std::integral_constant<int, 0>{});
      product(std::integral_constant<int, 2>{});
      product(std::integral_constant<int, 1>{});
      product(std::integral_constant<int, 3>{});
    };
    if (!dead) {
      sub_tile(std::integral_constant<int, 0>{});
      sub_tile(std::integral_constant<int, 1>{});
    }
    rd.move((n & 1) ? -(int)STAGE_BYTES : (int)STAGE_BYTES);
  }

  store_kv_row<PART, IS_DK>(p, acc, b, h, hk, key, g, part);
}

// The same with loads three tiles ahead and the vector work of a sub-tile of 32 queries under the products of its neighbours: one call of `unit` forms
// S (and dP) of the sub-tile after and adds this one to dV or dK.  Each role passes the same barriers, one per query tile behind those of the prologue.
template <bool PART, bool IS_DK>
__device__ __forceinline__ void kv_ring_block(const AttnParams& p, unsigned char* smem, int n0, int h, int b, const bf16* __restrict__ stats,
                                              float* __restrict__ part) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int hk = h / p.group, wn0 = n0 + (wave & 3) * 32, key = wn0 + i;
  bf16* ring = reinterpret_cast<bf16*>(smem);   // [4][Q tile | dO tile | row values]
  const int q_tiles = (p.Lq + ROWS - 1) / ROWS, t_top = q_tiles - 1;
  // this block's tiles, last query tile first, and of them those that see a key of this wavefront and those that see all of its keys
  const int total = max(0, q_tiles - (p.causal ? max(0, n0 - p.off) / ROWS : 0));
  int w_total = total, w_full = total;
  if (p.causal) {
    w_total = min(total, max(0, q_tiles - max(0, wn0 - p.off) / ROWS));
    w_full = min(total, max(0, q_tiles - (max(0, wn0 + 31 - p.off) + ROWS - 1) / ROWS));
  }
  const bf16* qp = static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h;
  const bf16* dop = static_cast<const bf16*>(p.dout) + b * p.sdo.b + h * p.sdo.h;
  const bf16* sp = stats + ((int64_t)b * p.Hq + h) * q_tiles * 512;
  // Direct loads of tile n: halves of Q (0, 1) and of dO (2, 3), a quarter of the row values (4; twice).  Rows past the end read zeros, a tile past the end
  // nothing else.
  const int brow = 4 * wave + (lane >> 4), qrow = 2 * (int)p.sq.l, orow = 2 * (int)p.sdo.l;
  auto load = [&](int n, int what) INLINE {
    const int t = t_top - n;
    bf16* st = ring + (n & 3) * QS_STAGE;
    if (what == 4) {
      auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(sp + (int64_t)t * 512), (short)0, n < total ? 1024 : 0, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)(st + 2 * TILE + 128 * (wave & 3)), 4, 256 * (wave & 3) + 4 * lane, 0, 0, 0);
      return;
    }
    const int rows = min(p.Lq - t * ROWS, ROWS), row = what < 2 ? qrow : orow, j = what & 1;
    const bf16* src = (what < 2 ? qp : dop) + (int64_t)(t * ROWS) * (row / 2);
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(src), (short)0, n < total ? (rows - 1) * row + 2 * D : 0, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)(st + (what < 2 ? 0 : TILE) + (8 * j + wave) * 512), 16,
                                             (brow + 32 * j) * row + 16 * ((lane & 15) ^ swz<D>((brow + 32 * j) >> 2)), 0, 0, 0);
  };
  auto all = [&](int n) INLINE {
#pragma unroll
    for (int what = 0; what < 5; what++) load(n, what);
  };
  all(0);
  FENCE();
  bf16x8 kf[KS], vf[IS_DK ? KS : 1];
  fetch_rows(kf, static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h, p.sk.l, key, p.Lk, g);
  if constexpr (IS_DK) fetch_rows(vf, static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h, p.sv.l, key, p.Lk, g);
  FENCE();
  all(1);
  all(2);
  settle_rows(kf, key, p.Lk);
  if constexpr (IS_DK) settle_rows(vf, key, p.Lk);

  const float c2 = p.scale_log2e;
  const int key_off = p.causal ? key - p.off : -(1 << 30);   // the first query that sees this lane's key
  constexpr int NS = IS_DK ? 1 : 2, NT = IS_DK ? DT : 2 * DT;
  f32x16 s[NS], dp, acc[DT];     // S, then P, for dV of either sub-tile of a tile; dP, then dS; dK^T or dV^T
  bf16x8 pf[2][2], fr[KS];       // P or dS of either sub-tile; rows of Q, and for dK then of dO, k-step n
  TrFrag tf[NT];                 // dO^T or Q^T: 16 queries n / DT, columns 32 (n % DT)
  clear(acc);
  Readers<D, true> rd;
  rd.init(ring, g, i);
  // from tile n's place in the ring to the next one's
  auto onward = [&](int n) INLINE { return (n + 1) & 3 ? (int)(QS_STAGE * 2) : -3 * (int)(QS_STAGE * 2); };
  typedef const bf16x8 __attribute__((address_space(3))) * frag_ptr;
  auto read_row = [&](int n, int which, int mt) INLINE { fr[n] = *(frag_ptr)(uintptr_t)(rd.row[n] + 2 * (which * TILE + 2 * mt * D)); };
  auto read_col = [&](auto n_, auto mt_) INLINE {
    constexpr int n = decltype(n_)::value, FIRST = (IS_DK ? 0 : ROWS) + 2 * decltype(mt_)::value + n / DT;
    read_tr<FIRST, 32>(tf[n % NT], rd.tr[2 * (n % DT)], rd.tr[2 * (n % DT) + 1]);
  };
  // a quarter a of a lane's 16 start values of sub-tile mt of tile n
  auto start = [&](int n, int mt, int which, int a, f32x16& x) INLINE {
    const f32x4 v = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(ring + (n & 3) * QS_STAGE + 2 * TILE) + 16 * g + 64 * mt + 32 * which + 4 * a);
#pragma unroll
    for (int e = 0; e < 4; e++) x[4 * a + e] = v[e];
  };
  // The vector work of sub-tile mt of tile n in steps of a product's length from the first product of its S on.  dV: element e becomes P in step 9 + 12 e / 16,
  // the products with it begin in step 24.  dK: P in step 9 + 11 e / 16, dS in step 18 + 6 e / 16, the products in step 40.
  auto vector = [&](int step, int n, auto mt_, auto masked) INLINE {
    constexpr int MT = decltype(mt_)::value, S = IS_DK ? 0 : MT;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      if (IS_DK && 18 + 6 * e / 16 == step) {
        dp[e] = s[S][e] * dp[e];
        if (e & 1) pf[MT][e >> 3][(e & 7) - 1] = (bf16)dp[e - 1], pf[MT][e >> 3][e & 7] = (bf16)dp[e];
      }
      if (9 + (IS_DK ? 11 : 12) * e / 16 == step) {
        const float x = decltype(masked)::value && (t_top - n) * ROWS + tile128::acc_tile_row(e, g, MT) < key_off ? -INFINITY : s[S][e];
        s[S][e] = ody_exp2(x * c2);
        if (!IS_DK && (e & 1)) pf[MT][e >> 3][(e & 7) - 1] = (bf16)s[S][e - 1], pf[MT][e >> 3][e & 7] = (bf16)s[S][e];
      }
    }
  };
  std::integral_constant<int, 0> c0;
  std::integral_constant<int, 1> c1;
  // tile n + 1 has landed (behind it the 5 loads of the next); everyone is done with tile n - 1
  auto turn = [&]() INLINE {
    asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto move = [&](unsigned (&x)[KS], int bytes) INLINE {
#pragma unroll
    for (int n = 0; n < KS; n++) x[n] += bytes;
  };
  auto unit = [&](int n, auto mt_, auto masked) INLINE {
    constexpr int MT = decltype(mt_)::value, NMT = MT ^ 1, S = IS_DK ? 0 : NMT;
    std::integral_constant<int, NMT> nmt;
    const int nn = MT ? n + 1 : n;   // the sub-tile after is in tile nn; behind that, sub-tile MT of tile n + 1
    auto slot = [&](auto m_) INLINE {
      constexpr int m = decltype(m_)::value;
      if constexpr (IS_DK) {
        if (m == 12)   // they are there; later the compiler's wait for one would be a wait for the transposing reads as well
#pragma unroll
          for (int r = 4; r < KS; r++) asm volatile("" : "+v"(fr[r]));
        if (m >= 16 && m < 20) {
          WAIT_LDS(6);
          tie(tf[m & 3]);
        }
        if (m == 20) {
          WAIT_LDS(0);
#pragma unroll
          for (int r = 0; r < DT; r++) tie(tf[r]);
          if (MT == 0) turn();
        }
        if (m < 8) s[0] = mfma32(fr[m & 7], kf[m & 7], s[0]);
        else if (m < 16) dp = mfma32(fr[m & 7], vf[m & 7], dp);
        else acc[m & 3] = mfma32(value(tf[m & 3]), pf[MT][(m & 7) >> 2], acc[m & 3]);
        FENCE();
        if (m < 4) start(nn, NMT, 1, m, dp);
        if constexpr (m < 8) read_row(m, 1, NMT);
        if (MT == 0 && m == 10) move(rd.row, onward(n));
        if constexpr (m >= 12 && m < 20) read_col(std::integral_constant<int, m - 12>{}, mt_);
        if (MT == 1 && m == 20) move(rd.tr, onward(n));
        if constexpr (m >= 20) read_row(2 * (m & 3), 0, MT), read_row(2 * (m & 3) + 1, 0, MT);
        if (MT == 0 && m == 21) load(n + 3, 0), load(n + 3, 1);
        if (MT == 1 && (m == 2 || m == 10 || m == 20)) load(n + 3, m == 2 ? 2 : m == 10 ? 3 : 4);
        vector(m, nn, nmt, masked);
        if (m == 23)
#pragma unroll
          for (int a = 0; a < 4; a++) start(n + 1, MT, 0, a, s[0]);
      } else {
        if (m == 8) {
          WAIT_LDS(0);
#pragma unroll
          for (int r = 0; r < NT; r++) tie(tf[r]);
          if (MT == 0) turn();
        }
        if (m < 8) s[S] = mfma32(fr[m & 7], kf[m & 7], s[S]);
        else acc[m & 3] = mfma32(value(tf[m & 7]), pf[MT][(m & 7) >> 2], acc[m & 3]);
        FENCE();
        if constexpr (m < 8) read_col(m_, mt_);
        if (MT == 1 && m == 8) move(rd.tr, onward(n));
        if constexpr (m >= 8) read_row(m & 7, 0, MT);
        if (MT == 1 && m == 15) move(rd.row, onward(n + 1));
        if (MT == 0 && (m == 10 || m == 13)) load(n + 3, m == 13);
        if (MT == 1 && (m == 2 || m == 6 || m == 10)) load(n + 3, m == 2 ? 2 : m == 6 ? 3 : 4);
        vector(16 + m, n, mt_, masked);
        vector(m, nn, nmt, masked);
        if (m >= 12) start(n + 1, MT, 0, m & 3, s[MT]);
      }
      FENCE();
    };
    each<IS_DK ? 24 : 16>(slot);
  };
  if (total > 0) {
    asm volatile("s_waitcnt vmcnt(10)" ::: "memory");   // the first tile
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int n = 0;
    if (w_total > 0) {
#pragma unroll
      for (int a = 0; a < 4; a++) {
        start(0, 0, 0, a, s[0]);
        if constexpr (IS_DK) start(0, 0, 1, a, dp);
        else start(0, 1, 0, a, s[1]);
      }
#pragma unroll
      for (int r = 0; r < KS; r++) read_row(r, 0, 0);
#pragma unroll
      for (int r = 0; r < KS; r++) s[0] = mfma32(fr[r], kf[r], s[0]);
      if constexpr (IS_DK) {
#pragma unroll
        for (int r = 0; r < KS; r++) read_row(r, 1, 0);
#pragma unroll
        for (int r = 0; r < KS; r++) dp = mfma32(fr[r], vf[r], dp);
      }
#pragma unroll
      for (int r = 0; r < KS; r++) read_row(r, 0, 1);
#pragma unroll
      for (int m = 9; m < (IS_DK ? 24 : 16); m++) vector(m, 0, c0, std::true_type{});
      if constexpr (IS_DK) {
#pragma unroll
        for (int a = 0; a < 4; a++) start(0, 1, 0, a, s[0]);
      } else {
        move(rd.row, onward(0));   // the loop reads rows one tile ahead of columns
      }
      FENCE();
      for (; n + 1 < min(w_total, w_full); n++) {
        unit(n, c0, std::false_type{});
        unit(n, c1, std::false_type{});
      }
      for (; n < w_total; n++) {   // (behind the last tile a sub-tile is formed that nobody uses)
        unit(n, c0, std::true_type{});
        unit(n, c1, std::true_type{});
      }
    }
    // the other wavefronts' tiles: keep bringing this one's share of them
    for (; n < total; n++) {
      turn();
      all(n + 3);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  store_kv_row<PART, IS_DK>(p, acc, b, h, hk, key, g, part);
}

// RING: where rows have tiles enough, dq_ring_block and kv_ring_block.  Bound: a block's longest role, dK, 48 products a tile and wavefront beside dV's 32 (1.75 us
// a tile where these take 1.15; 2.2 before, in waits for transposing reads and for tiles one ahead).
//
// The whole backward behind the pre-pass in one launch.  A rank of key blocks (first keys first: the most query tiles) and a rank of
// query blocks (last queries first) alternate, over all heads, so that what starts last is short on both sides.
template <bool PART, bool RING>
__global__ __launch_bounds__(64 * WAVES, 2) void attn_bwd_short_kernel(const AttnParams p, const bf16* __restrict__ stats,
                                                                   float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const BlockCoord bc = ody_block_coord(p.Hq, p.B);
  const int nkv = (p.Lk + BLOCK_ROWS - 1) / BLOCK_ROWS, nq = (p.Lq + BLOCK_ROWS - 1) / BLOCK_ROWS, both = min(nkv, nq);
  const bool paired = bc.rank < 2 * both;
  const int rank = paired ? bc.rank >> 1 : bc.rank - both;
  if (paired ? bc.rank & 1 : nq > nkv) {
    if constexpr (RING) dq_ring_block(p, smem, (p.causal ? nq - 1 - rank : rank) * BLOCK_ROWS, bc.h, bc.b);
    else dq_block(p, smem, (p.causal ? nq - 1 - rank : rank) * BLOCK_ROWS, bc.h, bc.b);
  } else if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < WAVES / 2) {
    if constexpr (RING) kv_ring_block<PART, false>(p, smem, rank * BLOCK_ROWS, bc.h, bc.b, stats, part);
    else kv_block<PART, false>(p, smem, rank * BLOCK_ROWS, bc.h, bc.b, stats, part);
  } else {
    if constexpr (RING) kv_ring_block<PART, true>(p, smem, rank * BLOCK_ROWS, bc.h, bc.b, stats, part);
    else kv_block<PART, true>(p, smem, rank * BLOCK_ROWS, bc.h, bc.b, stats, part);
  }
}

inline int64_t row_blocks(int B, int L, int H) { return (int64_t)B * H * ((L + BLOCK_ROWS - 1) / BLOCK_ROWS); }

}  // namespace

// The lines were fitted against kernels that the present ones, on both sides, have since replaced.  As they are now, 300 calls of each direction (1 to 64 heads, 64 to
// 8192 rows, a third with other key than query counts) against both kernels for all of them: 1.30 and 1.49 times as fast in the geometric mean as without the kernels
// here, 2.6 and 1.9 % behind the faster one in the mean, and by more than 5 % in 29 and 25 of the 300: forwards of up to 64 blocks from 1024 keys on, which the parts
// keep (1.1 to 1.6 times), backwards that go to the other kernels for their tiles or for their cut query range (1.05 to 1.6).  Here / there, us:
//   Beyond the line in blocks every compute unit has a block of 256 rows, whose tiles serve twice the rows: 32 heads, full, L = 1500: forward
//   52 / 51, backward 167 / 152; causal, L = 3001: 92 / 86, 310 / 285.  Short causal rows leave those blocks a few tiles each, most of them under the
//   mask, so that for them the line of the backward is further out: 4 x 24 heads, L = 820, 133 / 147, 4 x 32 heads, L = 683, 142 / 144, and
//   beyond, 4 x 32 heads, L = 820, 182 / 183; L = 936 220 / 204; with longer rows 2 x 32 heads, L = 1200, 147 / 148, L = 1536 203 / 195.
//   Beyond the line in tiles the other kernels cut the range of the long side into parts, backward, in the ring: 8 heads, full, L = 3000, 182 / 161, 2 heads,
//   causal, L = 5000, 134 / 126; inside it 3 heads, L = 2500, causal 76 / 120, full 77 / 122, 5 heads, L = 3000, full, 101 / 139.  The forward, in the ring: 4 heads,
//   L = 4096, 46 / 47; 2 heads, L = 6000, 63 / 52; 3 heads, L = 8192, 85 / 76, 4 heads 92 / 93; 3 heads, L = 6000, full, 68 / 79; 12 heads, L = 4096, causal, 59 / 79; 6 heads,
//   L = 12 000, 216 / 252.  Up to 64 blocks calls of 1024 keys and more stay with the parts: many keys, 300 queries on 8000, 81 / 60, are the line of 32 tiles' case and not
//   this one's, which no time puts where it is: 8 heads, L = 1024, 19 / 32, 4 heads, L = 1536, 23.7 / 34.8, L = 2048 28 / 36; with fewer keys calls come here (8 heads,
//   L = 1000, 18.9 / 31.6).
// One head, too, below the line: backward of 512 rows, causal, 27 / 68, of 1024 rows 39 / 96; two heads of 512 rows 27 / 68.
bool ody_attn_fwd_short_ok(const AttnParams& p) {
  if (std::max(p.sk.l, p.sv.l) >= tile128::TILE_MAX_STRIDE) return false;   // rows of a tile beyond 32-bit offsets
  const int64_t blocks = row_blocks(p.B, p.Lq, p.Hq), tiles = (p.Lk + ROWS - 1) / ROWS;
  if (blocks <= 64 && p.Lk >= 1024 && ody_attn_fwd_pipe_parts(p.B, p.Lq, p.Lk, p.Hq, p.causal) > 1) return false;
  if (blocks <= 128) return tiles <= 32;
  if (blocks > (p.causal ? 640 : 256)) return false;
  return tiles <= std::min<int64_t>(192, std::max<int64_t>(64, p.causal && blocks <= 256 ? blocks / 2 : 2 * blocks / 3));
}
bool ody_attn_bwd_short_ok(int B, int Lq, int Lk, int Hq, int causal) {
  const int64_t blocks = row_blocks(B, Lq, Hq) + row_blocks(B, Lk, Hq);
  const int rows = std::max(Lq, Lk);
  return blocks <= (causal ? (rows <= 16 * ROWS ? 1536 : 1024) : 512) && rows <= ROWS * (causal || blocks <= 256 ? 56 : 32);
}

int ody_launch_attn_fwd_short(const AttnParams& p, hipStream_t st) {
  const int64_t blocks = row_blocks(p.B, p.Lq, p.Hq);
  // Loop / ring, us: causal, L = 448, 32 heads, 13.5 / 13.7, L = 512 15.5 / 15.0; two blocks a unit L = 1500, 32 heads, 32.9 / 33.5, L = 2048 49.4 / 46.3;
  // full, L = 256, 96 heads, 12.2 / 12.4, L = 331, 64 heads, 13.7 / 13.0, 85 heads 17.0 / 18.1, L = 512, 64 heads, 16.4 / 16.6, L = 1000, 32 heads, 24.7 / 23.4.
  const bool ring = p.Lk >= (p.causal ? (blocks <= 256 ? 512 : 1536) : blocks <= 208 ? 320 : 960);
  auto kern = ring ? &attn_fwd_short_ring_kernel : &attn_fwd_short_kernel;
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), SMEM, "attn_fwd_short")) return rc;
  ODY_LAUNCH("attn_fwd_short", st, kern, dim3((unsigned)row_blocks(p.B, p.Lq, p.Hq)), dim3(64 * WAVES), SMEM, p);
  return ody_check_launch("attn_fwd_short");
}

int ody_launch_attn_bwd_short(const AttnParams& p, const void* stats, float* part, hipStream_t st) {
  const dim3 grid((unsigned)(row_blocks(p.B, p.Lq, p.Hq) + row_blocks(p.B, p.Lk, p.Hq)));
  // Loop / ring, the whole backward, us: causal, L = 331, 21 heads, 22.6 / 22.7, L = 600, 13 heads, 34.9 / 32.6, L = 1000, 8 heads, 45.5 / 40.1; more than one block
  // for a unit: L = 512, 96 heads, 58 / 59, L = 700, 43 heads, 54 / 56, L = 1000, 32 heads, 62 / 60, L = 1500 106 / 101.
  const bool near = std::max(std::max(p.sq.l, p.sdo.l), std::max(p.sk.l, p.sv.l)) < tile128::TILE_MAX_STRIDE;   // 32-bit offsets in a tile
  const bool ring = near && std::max(p.Lq, p.Lk) >= (grid.x <= 256 ? 512 : 960);
  auto kern = ring ? (p.group > 1 ? &attn_bwd_short_kernel<true, true> : &attn_bwd_short_kernel<false, true>)
                   : (p.group > 1 ? &attn_bwd_short_kernel<true, false> : &attn_bwd_short_kernel<false, false>);
  const size_t smem = ring ? 4 * QS_STAGE * sizeof(bf16) : SMEM;
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, "attn_bwd_short")) return rc;
  ODY_LAUNCH("attn_bwd_short", st, kern, grid, dim3(64 * WAVES), smem, p, static_cast<const bf16*>(stats), part);
  return ody_check_launch("attn_bwd_short");
}
