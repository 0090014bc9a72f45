// Flash attention for bf16 and head_dim 64 where there are blocks enough for the whole chip: the arithmetic, tiles and fragments of
// attn_hd64.hip in the order of attn_fwd_pipe.hip and attn_bwd_pipe.hip -- the vector work of one sub-tile under the products of another,
// instead of left to whichever wavefront of a SIMD has some.
//
// Tried and left: 64 rows per wavefront in the backward, one wavefront per SIMD, so that a fragment read from LDS serves two products.  It draws less
// power and takes more cycles.  dQ (304 registers), whole backward with the dQ of attn_hd64.hip / with it, us: 16 heads, L = 8192, causal 481 / 457,
// full 893 / 838, but 4 x 32 heads 3907 / 4016, 32 heads, L = 2048 x 4, 275 / 292.  dK / dV (396 registers), with the one below / with it: 491 / 468,
// 920 / 887, but 3703 / 3732, 279 / 287, 8 heads of the first 308 / 342.
#include <cfloat>
#include <type_traits>
#include "attn_rowtile.h"

namespace {

using namespace rowtile;

constexpr int D = 64, KS = D / 16, DT = D / 32, TILE = ROWS * D;   // elements of a tile: 8 KB
#define FENCE() __builtin_amdgcn_sched_barrier(0)
#define INLINE __attribute__((always_inline))

// Direct loads of one matrix's 64-row tiles, in two halves of one instruction per wavefront each (4 wavefronts).  Rows past the end read
// zeros: they lie beyond the descriptor.
struct Bringer {
  int row_bytes, lane_off;
  __device__ __forceinline__ void init(int64_t stride, int wave, int lane) {
    const int row = 8 * wave + (lane >> 3);
    row_bytes = 2 * (int)stride;
    lane_off = row * row_bytes + 16 * ((lane & 7) ^ swz<D>(row));
  }
  // src: the tile's first row; rows: how many are left from there on; j: half
  __device__ __forceinline__ void load(bf16* tile, const bf16* src, int rows, int j, int wave) const {
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(src), (short)0, (min(rows, ROWS) - 1) * row_bytes + 2 * D, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)(tile + (4 * j + wave) * 512), 16, lane_off + 32 * j * row_bytes, 0, 0, 0);
  }
};

// A transposed fragment (tr_frags) whose reads are still under way: 16 rows from OFF / 128 on, 32 columns by the address pair
struct TrFrag {
  s16x4 lo, hi;
};
template <int FIRST>
__device__ __forceinline__ void read_tr(TrFrag& f, unsigned a0, unsigned a1) {
  asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%4\n\tds_read_b64_tr_b16 %1, %3 offset:%5"
               : "=&v"(f.lo), "=&v"(f.hi)
               : "v"(a0), "v"(a1), "n"(2 * FIRST * D), "n"(2 * (FIRST + 8) * D));
}
// behind the wait for them
__device__ __forceinline__ void tie(TrFrag& f) { asm volatile("" : "+v"(f.lo), "+v"(f.hi)); }
__device__ __forceinline__ bf16x8 value(const TrFrag& f) {
  return concat4(__builtin_bit_cast(bf16x4, f.lo), __builtin_bit_cast(bf16x4, f.hi));
}
#define WAIT_LDS(n) asm volatile("s_waitcnt lgkmcnt(" #n ")" ::: "memory")

// ---------------------------------------------------------------------------------------------------------- forward
//   S^T = K Q^T      O^T += V^T P^T       lane = query column
//
// Bound: the vector pipe of a wavefront's SIMD (exp, bf16 conversion and sums of 64 x 64 scores beside 32 products), so each product has its
// share of it behind, two wavefronts per SIMD, and 64 queries each, so that a fragment read from LDS serves two products.  Before (32 queries,
// three wavefronts per SIMD, attn_hd64.hip) / now, us: 16 heads, L = 8192, causal 179 / 173, full 308 / 265 (1037 TFLOP/s); 24 heads, causal,
// 239 / 219; 4 x 32 heads on 8, causal, 1200 / 1067.
//
// GROUPS = 2: a second set of 4 wavefronts over the same rows, two per SIMD in one block, takes the later half of the tiles; their references, sums
// and O meet in LDS at the end.  For calls with fewer blocks than units can hold two of: 16 heads, L = 8192, causal 160 / 145, L = 4096, full 85 / 73.
constexpr int FW_QT = 2, FW_BM = 32 * FW_QT * 4, FW_SLOTS = 4;

template <int GROUPS>
__global__ __launch_bounds__(256 * GROUPS, 2) void attn_fwd_hd64_pipe_kernel(const AttnParams p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const int wave = wave8 & 3, grp = GROUPS == 1 ? 0 : wave8 >> 2;
  bf16* kring = reinterpret_cast<bf16*>(smem) + grp * 2 * FW_SLOTS * TILE;   // [FW_SLOTS][TILE]
  bf16* vring = kring + FW_SLOTS * TILE;                                     // [FW_SLOTS][TILE]
  const BlockCoord bc = block_coord<GROUPS == 1 ? 0 : 1>(p.Hq, p.B, p.causal);
  const int nqb = gridDim.x / (p.Hq * p.B);
  const int qblk = p.causal ? nqb - 1 - bc.rank : bc.rank;   // heaviest blocks first
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * FW_BM, wq0 = q0 + wave * 32 * FW_QT;

  const int n_end = p.causal ? min(p.Lk, min(q0 + FW_BM, p.Lq) + p.off) : p.Lk;
  const int all_tiles = n_end > 0 ? (n_end + ROWS - 1) / ROWS : 0;
  // this group's share of them: the second one's is not the shorter, for behind the diagonal some of it is left out
  const int t_first = GROUPS == 1 || grp == 0 ? 0 : all_tiles / 2, ntiles = GROUPS == 1 || grp == 1 ? all_tiles : all_tiles / 2;
  // end of those tiles that this wavefront's queries see a key of, and of those that they see whole
  int w_end = ntiles, w_full = p.Lk / ROWS;
  if (p.causal) {
    w_end = min(ntiles, max(t_first, max(0, wq0 + 32 * FW_QT - 1 + p.off + ROWS) / ROWS));
    w_full = min(w_full, max(0, wq0 + p.off + 1) / ROWS);
  }

  Bringer bk, bv;
  bk.init(p.sk.l, wave, lane);
  bv.init(p.sv.l, wave, lane);
  const bf16* kp = static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const bf16* vp = static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h;
  int lk = t_first, lv = t_first;   // the tiles being brought, the last one again where there are no more
  const bf16 *ktp = kp + (int64_t)t_first * (ROWS / 2 * bk.row_bytes), *vtp = vp + (int64_t)t_first * (ROWS / 2 * bv.row_bytes);
  auto load_k = [&](int j) INLINE { bk.load(kring + (lk & (FW_SLOTS - 1)) * TILE, ktp, p.Lk - lk * ROWS, j, wave); };
  auto load_v = [&](int j) INLINE { bv.load(vring + (lv & (FW_SLOTS - 1)) * TILE, vtp, p.Lk - lv * ROWS, j, wave); };
  auto next_k = [&]() INLINE {
    const int to = min(lk + 1, ntiles - 1), step = to - lk;
    lk = to;
    ktp += (int64_t)step * (ROWS / 2 * bk.row_bytes);
  };
  auto next_v = [&]() INLINE {
    const int to = min(lv + 1, ntiles - 1), step = to - lv;
    lv = to;
    vtp += (int64_t)step * (ROWS / 2 * bv.row_bytes);
  };

  bf16x8 qf[FW_QT][KS];
  int lim[FW_QT];   // last key this lane's queries see
#pragma unroll
  for (int qt = 0; qt < FW_QT; qt++) {
    const int qi = wq0 + 32 * qt + i;
    load_rows(qf[qt], static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h, p.sq.l, qi, p.Lq, g);
    lim[qt] = p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1;
  }
  const float c2 = p.scale_log2e;
  f32x16 o[FW_QT][DT], s[2][FW_QT];
  float ref[FW_QT], l4[FW_QT][4];   // a row's reference in log2 units; this lane's partial row sums (four chains: attn_fwd_pipe.hip)
  bf16x8 pb[2][FW_QT][2];
  Readers<D> rd;
  rd.init(kring, g, i);   // rows of K from its row[] on; columns of V from its tr[] + the rings' distance on
  auto score = [&](int kt, int qt, int r, int t) INLINE { return t * ROWS + 32 * kt + acc_row(r, g) > lim[qt] ? -INFINITY : s[kt][qt][r]; };

  // The 32 pairs of elements of P that a turn forms: 0 .. 15 of sub-tile 1 of tile t, then those of sub-tile 0 of tile t + 1; in three steps,
  // each one product behind the one before
  float y[2] = {0.f, 0.f}, x[2] = {0.f, 0.f};
  auto exponents = [&](int e, int t, auto masked) INLINE {
    const int kt = (e & 31) < 16, qt = (e >> 3) & 1, r = 2 * (e & 7), tile = e < 16 ? t : t + 1;
#pragma unroll
    for (int n = 0; n < 2; n++) y[n] = fmaf(decltype(masked)::value ? score(kt, qt, r + n, tile) : s[kt][qt][r + n], c2, -ref[qt]);
  };
  auto take = [&](int e) INLINE {   // pair e: into the row sums and among the operands
    const int kt = (e & 31) < 16, qt = (e >> 3) & 1, r = 2 * (e & 7);
#pragma unroll
    for (int n = 0; n < 2; n++) l4[qt][(r & 3) + n] += x[n], pb[kt][qt][r >> 3][(r & 7) + n] = (bf16)x[n];
  };
  auto weigh = [&](int e, int t, auto masked) INLINE {
    const float x0 = ody_exp2(y[0]), x1 = ody_exp2(y[1]);
    exponents(e + 1, t, masked);
    take(e == 0 ? 31 : e - 1);
    x[0] = x0, x[1] = x1;
  };
  typedef const bf16x8 __attribute__((address_space(3))) * frag_ptr;
  bf16x8 kfr[KS];       // K rows: k-step n
  TrFrag vfr[2 * DT];   // V^T: k-step n >> 1, columns 32 (n & 1)
  auto kslot = [&](int t) INLINE { return (t & (FW_SLOTS - 1)) * TILE * 2; };
  auto read_k = [&](int n, unsigned slot, int kt) INLINE { kfr[n] = *(frag_ptr)(uintptr_t)(rd.row[n] + slot + 2 * 32 * kt * D); };
  auto read_v = [&](int n, unsigned slot, auto kt) INLINE {
    constexpr int KT = decltype(kt)::value;
    const unsigned at = slot + FW_SLOTS * TILE * 2;
    if (n >> 1) read_tr<32 * KT + 16>(vfr[n], rd.tr[2 * (n & 1)] + at, rd.tr[2 * (n & 1) + 1] + at);
    else read_tr<32 * KT>(vfr[n], rd.tr[2 * (n & 1)] + at, rd.tr[2 * (n & 1) + 1] + at);
  };
  // S of sub-tile KT of a tile, and reads of V of sub-tile KT of the one before
  auto s_phase = [&](auto kt, unsigned vslot, int e0, int t, int half, auto masked) INLINE {
    constexpr int KT = decltype(kt)::value;
#pragma unroll
    for (int m = 0; m < 8; m++) {
      const int n = m >> 1, qt = m & 1;
      if (m == 0) WAIT_LDS(2);   // with two reads issued behind: fragments 0 and 1 are there
      if (m == 4) WAIT_LDS(4);
      s[KT][qt] = mfma32(kfr[n], qf[qt][n], n == 0 ? f32x16{0} : s[KT][qt]);
      FENCE();
      if (qt == 1) read_v(n, vslot, kt);
      if (m == 2) load_v(half);
      weigh(e0 + m, t, masked);
      FENCE();
    }
  };
  // O += P V of sub-tile KT, and reads of K of the other sub-tile
  auto pv_phase = [&](auto kt, unsigned kslot, int e0, int t, int half, auto masked) INLINE {
    constexpr int KT = decltype(kt)::value;
#pragma unroll
    for (int m = 0; m < 8; m++) {
      const int n = m >> 1, qt = m & 1;
      if (m == 0) {
        WAIT_LDS(4);
        tie(vfr[0]), tie(vfr[1]);
      }
      if (m == 4) {
        WAIT_LDS(2);
        tie(vfr[2]), tie(vfr[3]);
      }
      o[qt][n & 1] = mfma32(value(vfr[n]), pb[KT][qt][n >> 1], o[qt][n & 1]);
      FENCE();
      if (qt == 1) read_k(n, kslot, KT ^ 1);
      if (m == 2) load_k(half);
      weigh(e0 + m, t, masked);
      FENCE();
    }
  };
  std::integral_constant<int, 0> c0;
  std::integral_constant<int, 1> c1;
  auto turn = [&](int t, auto masked) INLINE {
    s_phase(c0, kslot(t), 0, t, 0, masked);
    pv_phase(c0, kslot(t + 1), 8, t, 1, masked);
    s_phase(c1, kslot(t), 16, t, 1, masked);
    // K tile t + 2 and V tile t + 1 have landed (behind them the 4 loads of the tiles after); everyone is done with K tile t + 1 and V tile t - 1
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    next_k();
    next_v();
    pv_phase(c1, kslot(t + 2), 24, t, 0, masked);
  };

  auto row_sum = [&](int qt) INLINE { return (l4[qt][0] + l4[qt][1]) + (l4[qt][2] + l4[qt][3]); };
  // The reference of a row is the largest score of its first tile (a row that sees any key sees key 0) and stays.
  auto clear_rows = [&]() INLINE {
#pragma unroll
    for (int qt = 0; qt < FW_QT; qt++) {
      clear(o[qt]);
      ref[qt] = -FLT_MAX;   // no score is below it; not minus infinity, from which a masked score would be NaN
      l4[qt][0] = l4[qt][1] = l4[qt][2] = l4[qt][3] = 0.f;
    }
  };
  auto scores = [&](int t) INLINE {
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
      for (int n = 0; n < KS; n++) {
        read_k(n, kslot(t), kt);
#pragma unroll
        for (int qt = 0; qt < FW_QT; qt++) s[kt][qt] = mfma32(kfr[n], qf[qt][n], n == 0 ? f32x16{0} : s[kt][qt]);
      }
  };
  auto largest = [&](int qt, int t) INLINE {   // in log2 units
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
      for (int r = 0; r < 16; r++) mx = fmaxf(mx, score(kt, qt, r, t));
    return half_swap_max(mx) * c2;
  };
  auto products = [&](int t) INLINE {
    auto half = [&](auto kt) INLINE {
#pragma unroll
      for (int n = 0; n < 4; n++) read_v(n, kslot(t), kt);
      WAIT_LDS(0);
#pragma unroll
      for (int n = 0; n < 4; n++) {
        tie(vfr[n]);
#pragma unroll
        for (int qt = 0; qt < FW_QT; qt++) o[qt][n & 1] = mfma32(value(vfr[n]), pb[decltype(kt)::value][qt][n >> 1], o[qt][n & 1]);
      }
    };
    half(c0);
    half(c1);
  };
  clear_rows();
  if (t_first < ntiles) {
    // K tiles t_first .. + 3 and V tiles .. + 2, of the last ones a part: the loop brings the rest
    load_k(0), load_k(1);
#pragma unroll
    for (int a = 0; a < 3; a++) {
      next_k();
      if (a > 0) next_v();
      load_k(0);
      if (a < 2) load_v(0), load_k(1), load_v(1);
    }
    asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int t = t_first;
    if (w_end > t_first) {
      scores(t);
#pragma unroll
      for (int qt = 0; qt < FW_QT; qt++) ref[qt] = fmaxf(ref[qt], largest(qt, t));
#pragma unroll
      for (int e = 16; e < 32; e++) {   // the last pair is left to be taken by the first turn
        exponents(e, t - 1, std::true_type{});
        x[0] = ody_exp2(y[0]), x[1] = ody_exp2(y[1]);
        if (e < 31) take(e);
      }
      exponents(0, t, std::true_type{});
#pragma unroll
      for (int n = 0; n < KS; n++) read_k(n, kslot(t + 1), 0);
      FENCE();
      for (; t + 1 < min(w_end, w_full); t++) turn(t, std::false_type{});
      for (; t + 1 < w_end; t++) turn(t, std::true_type{});
      // the last tile: P of its second half, the products
      take(31);
#pragma unroll
      for (int e = 0; e < 16; e++) {
        exponents(e, t, std::true_type{});
        x[0] = ody_exp2(y[0]), x[1] = ody_exp2(y[1]);
        take(e);
      }
      products(t);
    }
    // the other wavefronts' tiles: keep bringing this one's share of them
    for (; t + 1 < ntiles; t++) {
      load_v(0), load_k(1), load_v(1);
      asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      next_k();
      next_v();
      load_k(0);
    }
  }
  if (GROUPS == 2 && grp == 0 && (all_tiles & 1)) __builtin_amdgcn_s_barrier();   // the second group's one more
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();   // everyone is done with the rings
  {
    // a later score that outgrew its row's reference by more than fp32 holds left a row sum beyond any real one (or a NaN), or,
    // times large values, an infinity in O: the block walks its keys once more with the maximum so far, so that P <= 1
    int* flags = reinterpret_cast<int*>(smem);
    bool beyond = false;
#pragma unroll
    for (int qt = 0; qt < FW_QT; qt++) {
      float zero[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) zero[r & 3] = fmaf(o[qt][dt][r], 0.f, zero[r & 3]);
      beyond |= !((zero[0] + zero[1]) + (zero[2] + zero[3]) == 0.f) || !(half_swap_sum(row_sum(qt)) < 0x1p100f);
    }
    const int mine = __builtin_amdgcn_ballot_w64(beyond) != 0;
    if (lane == 0) flags[wave8] = mine;
    __syncthreads();
    int any = 0;
#pragma unroll
    for (int w = 0; w < 4 * GROUPS; w++) any |= flags[w];
    __syncthreads();
    if (any) {
      clear_rows();
      for (int n = 0; n < (GROUPS == 1 ? all_tiles : (all_tiles + 1) / 2); n++) {
        const int t = t_first + n;
        if (t < ntiles) {
          lk = lv = t;
          ktp = kp + (int64_t)t * ROWS * p.sk.l, vtp = vp + (int64_t)t * ROWS * p.sv.l;
          load_k(0), load_k(1), load_v(0), load_v(1);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (t < w_end) {
          scores(t);
#pragma unroll
          for (int qt = 0; qt < FW_QT; qt++) {
            const float next = fmaxf(ref[qt], largest(qt, t)), alpha = ody_exp2(ref[qt] - next);
            ref[qt] = next;
#pragma unroll
            for (int e = 0; e < 4; e++) l4[qt][e] *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
              for (int r = 0; r < 16; r++) o[qt][dt][r] *= alpha;
          }
#pragma unroll
          for (int e = 0; e < 32; e++) {
            exponents(e, e < 16 ? t : t - 1, std::true_type{});
            x[0] = ody_exp2(y[0]), x[1] = ody_exp2(y[1]);
            take(e);
          }
          products(t);
        }
        __syncthreads();
      }
    }
  }

  auto store = [&](int qt, float l) INLINE {
    const int qi = wq0 + 32 * qt + i;
    l = half_swap_sum(l);
    if (qi >= p.Lq) return;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    store_row(static_cast<bf16*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)qi * p.so.l, o[qt], inv, g);
    if (g == 0) p.lse[((int64_t)b * p.Hq + h) * p.Lq + qi] = l > 0.f ? (ref[qt] + __log2f(l)) * ODY_LN2 : -INFINITY;
  };
  if constexpr (GROUPS == 1) {
#pragma unroll
    for (int qt = 0; qt < FW_QT; qt++) store(qt, row_sum(qt));
  } else {
    // a group hands half of its queries' sums to the other one and finishes the other half
    static_assert(FW_QT == 2 && 2 * 4 * (16 * DT + 2) * 64 * sizeof(float) <= 2 * 2 * FW_SLOTS * TILE * sizeof(bf16), "in the rings");
    float* patches = reinterpret_cast<float*>(smem);
    auto give_half = [&](int qt) INLINE {
      float* patch = patches + (4 * qt + wave) * (16 * DT + 2) * 64;
      give(patch, o[qt], lane);
      patch[16 * DT * 64 + lane] = ref[qt];
      patch[(16 * DT + 1) * 64 + lane] = row_sum(qt);
    };
    auto finish = [&](int qt) INLINE {
      const float* patch = patches + (4 * qt + wave) * (16 * DT + 2) * 64;
      const float ref1 = patch[16 * DT * 64 + lane], next = fmaxf(ref[qt], ref1), a0 = ody_exp2(ref[qt] - next), a1 = ody_exp2(ref1 - next);
      rowtile::take(patch, o[qt], lane, a0, a1);
      ref[qt] = next;
      store(qt, row_sum(qt) * a0 + patch[(16 * DT + 1) * 64 + lane] * a1);
    };
    if (grp == 0) give_half(1);
    else give_half(0);
    __syncthreads();
    if (grp == 0) finish(0);
    else finish(1);
  }
}

// ---------------------------------------------------------------------------------------------------------- backward
//   S = Q K^T - lse / scale     dP = dO V^T - delta     dV^T += dO^T P     dK^T += Q^T (P o dP)      lane = key column
//
// 4 wavefronts of 32 keys, two per SIMD: 216 registers hold the sums of 32 keys, the next sub-tile's fragments and its S and dP; with 64 keys
// they do not.  Bound: the reads from LDS and the matrix pipe alike (16 KB of fragments and 16 products per 32 x 32 sub-tile: 128 cycles of the
// unit's LDS, of which four SIMDs want one each, and 512 of a SIMD's matrix pipe).
// Whole backward before (the same split without the order) / now, us: 16 heads, L = 8192, causal 520 / 472, full 992 / 890; 8 heads of it,
// causal, 386 / 308; 4 x 32 heads, L = 500, full, 57 / 52.  Of it this kernel, with every run of 256 causal blocks reversed, K and V waited for in front of
// the first tiles' loads and an address formed with each read / as it is: 268 / 255, 491 / 483, 152 / 145; 64 heads, L = 512, full, 19.0 / 17.9; 80 heads,
// L = 1000, causal, 39.7 / 36.5.  (With two blocks a unit the last of four runs reversed starts its longest blocks last.)
// PART: fp32 sums of one query head to part [dK | dV][B][Hq][Lk][D]; otherwise every kv head has one.
constexpr int KV_BN = 128, KV_SLOTS = 4;
constexpr int KV_STAGE = 2 * TILE + 2 * 2 * ROWS;   // elements: Q and dO tiles, -lse / scale and -delta of their rows in fp32

template <bool PART>
__global__ __launch_bounds__(256, 2) void attn_bwd_hd64_dkdv_pipe_kernel(const AttnParams p, const float* __restrict__ neg_delta,
                                                                         const float* __restrict__ neg_lse, float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  bf16* ring = reinterpret_cast<bf16*>(smem);   // [KV_SLOTS][KV_STAGE]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const BlockCoord bc = block_coord<2>(p.Hq, p.B, p.causal);   // rank 0 = first key block = most query tiles
  const int b = bc.b, h = bc.h, hk = h / p.group;
  const int n0 = bc.rank * KV_BN, wn0 = n0 + wave * 32, key = wn0 + i;
  const int q_tiles = (p.Lq + ROWS - 1) / ROWS, t_top = q_tiles - 1;
  // this block's tiles, last query tile first, and of them those that see a key of this wavefront and those that see all of its keys
  const int total = max(0, q_tiles - (p.causal ? max(0, n0 - p.off) / ROWS : 0));
  int w_total = total, w_full = total;
  if (p.causal) {
    w_total = min(total, max(0, q_tiles - max(0, wn0 - p.off) / ROWS));
    w_full = min(total, max(0, q_tiles - (max(0, wn0 + 31 - p.off) + ROWS - 1) / ROWS));
  }

  bf16x8 kf[KS], vf[KS];
  fetch_rows(kf, static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h, p.sk.l, key, p.Lk, g);
  fetch_rows(vf, static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h, p.sv.l, key, p.Lk, g);
  const float c2 = p.scale_log2e;

  Bringer bq, bo;
  bq.init(p.sq.l, wave, lane);
  bo.init(p.sdo.l, wave, lane);
  const int64_t head = (int64_t)b * p.Hq + h;
  int lt = 0;   // the tile being brought, the last one again where there are no more
  const bf16* qtp = static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h + (int64_t)t_top * ROWS * p.sq.l;
  const bf16* otp = static_cast<const bf16*>(p.dout) + b * p.sdo.b + h * p.sdo.h + (int64_t)t_top * ROWS * p.sdo.l;
  // wavefronts 0, 2 bring -lse / scale, 1, 3 -delta (zeros for rows past the end: their P is 0)
  const float* values = wave & 1 ? neg_delta + head * p.Lq : neg_lse + head * q_tiles * ROWS;
  const int values_bytes = 4 * (wave & 1 ? p.Lq : q_tiles * ROWS);
  auto load = [&](int part) INLINE {   // 0, 1: halves of Q; 2, 3: of dO; 4: the values
    bf16* st = ring + (lt & (KV_SLOTS - 1)) * KV_STAGE;
    const int row0 = (t_top - lt) * ROWS;
    if (part < 2) bq.load(st, qtp, p.Lq - row0, part, wave);
    else if (part < 4) bo.load(st + TILE, otp, p.Lq - row0, part - 2, wave);
    else {
      auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(values), (short)0, values_bytes, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)(st + 2 * TILE + (wave & 1) * 2 * ROWS), 4, 4 * (row0 + lane), 0, 0, 0);
    }
  };
  auto next = [&]() INLINE {
    const int to = min(lt + 1, total - 1), step = to - lt;
    lt = to;
    qtp -= (int64_t)step * (ROWS / 2 * bq.row_bytes);
    otp -= (int64_t)step * (ROWS / 2 * bo.row_bytes);
  };

  f32x16 dk[DT], dv[DT], s, s_start, dp;   // S, then P; dP, then dS
  clear(dk);
  clear(dv);
  bf16x8 pf[2], dsf[2], pf_next[2], dsf_next[2];
  Readers<D> rd;
  rd.init(ring, g, i);
  const int key_off = p.causal ? key - p.off : -(1 << 30);   // the first query that sees this lane's key
  typedef const bf16x8 __attribute__((address_space(3))) * frag_ptr;
  // from tile it's place in the ring to the next one's
  auto onward = [&](int it) INLINE { return (it + 1) & (KV_SLOTS - 1) ? KV_STAGE * 2 : -(KV_SLOTS - 1) * KV_STAGE * 2; };
  bf16x8 fr[2 * KS];   // Q rows, k-step n; dO rows, k-step n - 4
  TrFrag tf[8];        // n = 2 (2 ss + dt) + which: dO^T (0) or Q^T (1)
  auto read_row = [&](int n, int mt) INLINE {
    fr[n] = *(frag_ptr)(uintptr_t)(rd.row[n & 3] + 2 * ((n >> 2) * ROWS + 32 * mt) * D);
  };
  auto read_col = [&](int n, auto mt_) INLINE {
    constexpr int MT = decltype(mt_)::value;
    const unsigned a0 = rd.tr[2 * ((n >> 1) & 1)], a1 = rd.tr[2 * ((n >> 1) & 1) + 1];
    if (n < 4) {
      if (n & 1) read_tr<32 * MT>(tf[n], a0, a1);
      else read_tr<ROWS + 32 * MT>(tf[n], a0, a1);
    } else {
      if (n & 1) read_tr<32 * MT + 16>(tf[n], a0, a1);
      else read_tr<ROWS + 32 * MT + 16>(tf[n], a0, a1);
    }
  };
  // a quarter a of a lane's 16 start values: rows 8 a + 4 g .. + 3 of sub-tile mt
  auto start_values = [&](int it, int mt, int which, int a, f32x16& x) INLINE {
    const f32x4 v = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(ring + (it & (KV_SLOTS - 1)) * KV_STAGE + 2 * TILE) + which * ROWS +
                                                    32 * mt + 8 * a + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; e++) x[4 * a + e] = v[e];
  };
  auto exponent = [&](int r, int t, int mt, auto masked) INLINE {
    float x = s[r] * c2;
    if (decltype(masked)::value) x = t * ROWS + 32 * mt + acc_row(r, g) < key_off ? -INFINITY : x;   // queries before the key
    s[r] = x;
  };
  auto weight = [&](int r) INLINE { s[r] = ody_exp2(s[r]); };
  auto ds = [&](int r) INLINE { dp[r] *= s[r]; };
  auto pack = [&](bf16x8 (&dst)[2], const f32x16& src, int q) INLINE {
    dst[q >> 2][2 * q & 7] = (bf16)src[2 * q], dst[q >> 2][(2 * q & 7) + 1] = (bf16)src[2 * q + 1];
  };

  // One call: S and dP of the sub-tile after (tile it, sub-tile MT), then dV and dK of this one, 8 products each, the vector work of the former
  // under the later ones.
  auto unit = [&](int it, auto mt_, auto masked) INLINE {
    constexpr int MT = decltype(mt_)::value, NMT = MT ^ 1;
    const int nt = MT ? it + 1 : it, t = t_top - nt;   // the sub-tile after; behind that, sub-tile MT of tile it + 1
#pragma unroll
    for (int m = 0; m < 8; m++) {
      if (m == 0) WAIT_LDS(4);
      if (m == 4) WAIT_LDS(6);
      if (m < 4) s = mfma32(fr[m], kf[m], m == 0 ? s_start : s);
      else dp = mfma32(fr[m], vf[m - 4], dp);
      FENCE();
      if (m < 2) start_values(nt, NMT, 1, 2 * m, dp), start_values(nt, NMT, 1, 2 * m + 1, dp);
      read_col(m, mt_);
      if (m >= 6) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (m == 7) weight(e);
          exponent(4 * (m - 6) + e, t, NMT, masked);
        }
      }
      if (MT == 1 && (m == 2 || m == 5)) load(m == 5);
      FENCE();
    }
#pragma unroll
    for (int m = 0; m < 8; m++) {
      if (m == 0) {
        WAIT_LDS(8);
#pragma unroll
        for (int n = 0; n < 4; n++) tie(tf[n]);
      }
      if (m == 4) {
        WAIT_LDS(8);
#pragma unroll
        for (int n = 4; n < 8; n++) tie(tf[n]);
      }
      const int n = m >> 1;
      if (m & 1) dk[n & 1] = mfma32(value(tf[m]), dsf[n >> 1], dk[n & 1]);
      else dv[n & 1] = mfma32(value(tf[m]), pf[n >> 1], dv[n & 1]);
      FENCE();
      if (MT == 0 && m == 0) {
        // the tile after this one has landed (behind it the 5 loads of the next); everyone is done with the one before this
        asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        next();
      }
      read_row(m, MT);
      if (m < 4) start_values(it + 1, MT, 0, m, s_start);
      if (m <= 2) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          weight(4 * (m + 1) + e);
          if (m < 2) exponent(4 * (m + 2) + e, t, NMT, masked);
        }
      }
      if (m >= 2 && m < 6) {
#pragma unroll
        for (int e = 0; e < 4; e++) ds(4 * (m - 2) + e);
        pack(pf_next, s, 2 * m - 4), pack(pf_next, s, 2 * m - 3);
      }
      if (m >= 3 && m < 7) pack(dsf_next, dp, 2 * m - 6), pack(dsf_next, dp, 2 * m - 5);
      if (MT == 0 && m == 5) load(4);
      if (MT == 1 && (m == 2 || m == 5)) load(2 + (m == 5));
      if (MT == 1 && m == 6)
#pragma unroll
        for (int n = 0; n < KS; n++) rd.tr[n] += onward(it);
      if (MT == 1 && m == 7)
#pragma unroll
        for (int n = 0; n < KS; n++) rd.row[n] += onward(it + 1);
      FENCE();
    }
#pragma unroll
    for (int ss = 0; ss < 2; ss++) pf[ss] = pf_next[ss], dsf[ss] = dsf_next[ss];
  };
  std::integral_constant<int, 0> c0;
  std::integral_constant<int, 1> c1;

  if (total > 0) {
    auto all = [&]() INLINE {
      load(4);
#pragma unroll
      for (int n = 0; n < 4; n++) load(n);
    };
    all();
    next();
    all();
    next();
    all();
    settle_rows(kf, key, p.Lk);   // on their way in front of the tiles
    settle_rows(vf, key, p.Lk);
    asm volatile("s_waitcnt vmcnt(10)" ::: "memory");   // the first tile
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int it = 0;
    if (w_total > 0) {
#pragma unroll
      for (int a = 0; a < 4; a++) {
        start_values(0, 0, 0, a, s_start);
        start_values(0, 0, 1, a, dp);
      }
#pragma unroll
      for (int n = 0; n < 8; n++) read_row(n, 0);
#pragma unroll
      for (int n = 0; n < 4; n++) {
        s = mfma32(fr[n], kf[n], n == 0 ? s_start : s);
        dp = mfma32(fr[4 + n], vf[n], dp);
      }
#pragma unroll
      for (int r = 0; r < 16; r++) {
        exponent(r, t_top, 0, std::true_type{});
        weight(r);
        ds(r);
      }
#pragma unroll
      for (int q = 0; q < 8; q++) {
        pack(pf, s, q);
        pack(dsf, dp, q);
      }
#pragma unroll
      for (int a = 0; a < 4; a++) start_values(0, 1, 0, a, s_start);
#pragma unroll
      for (int n = 0; n < 8; n++) read_row(n, 1);
#pragma unroll
      for (int n = 0; n < KS; n++) rd.row[n] += onward(0);   // the loop reads rows one tile ahead of columns
      FENCE();
      for (; it + 1 < min(w_total, w_full); it++) {
        unit(it, c0, std::false_type{});
        unit(it, c1, std::false_type{});
      }
      for (; it < w_total; it++) {   // (behind the last tile a sub-tile is formed that nobody uses)
        unit(it, c0, std::true_type{});
        unit(it, c1, std::true_type{});
      }
    }
    // the other wavefronts' tiles: keep bringing this one's share of them
    for (; it < total; it++) {
      asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      next();
      all();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  if (key >= p.Lk) return;
  if (PART) {
    float* pk = part + (head * p.Lk + key) * D;
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

//   S^T = K Q^T     dP^T = V dO^T - delta     dQ^T += K^T dS^T       lane = query column
//
// As above, 4 wavefronts of 32 queries, two per SIMD (194 registers).  Bound: power, and the vector pipe (exp, products with P and dP, conversions: 416 cycles
// beside 384 of products per 32 x 32 sub-tile; takes 600), so addresses move once a tile and not with each read.  Counters, 16 heads, L = 8192, full: 1.63 GHz, matrix
// pipe 64 % busy, vector 59 %, LDS 43 %.
// dQ alone, before (the same split without the order, three wavefronts per SIMD) / now, us: 16 heads, L = 8192, causal 212 / 194, full 417 / 370; 8 heads of it,
// causal, 157 / 114; 4 x 32 heads of it 1629 / 1490; 16 heads, L = 4096, causal 83 / 61; on constant inputs, whose clock is not held down, full 348 / 255.
constexpr int DQ_BM = 128, DQ_SLOTS = 4, DQ_STAGE = 2 * TILE;   // K and V tiles

__global__ __launch_bounds__(256, 2) void attn_bwd_hd64_dq_pipe_kernel(const AttnParams p, const float* __restrict__ neg_delta) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  bf16* ring = reinterpret_cast<bf16*>(smem);   // [DQ_SLOTS][K tile | V tile]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, i = lane & 31;
  const BlockCoord bc = block_coord<2>(p.Hq, p.B, p.causal);
  const int nqb = gridDim.x / (p.Hq * p.B);
  const int qblk = p.causal ? nqb - 1 - bc.rank : bc.rank;   // heaviest blocks first
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * DQ_BM, wq0 = q0 + wave * 32, qi = wq0 + i;
  const int n_end = p.causal ? min(p.Lk, min(q0 + DQ_BM, p.Lq) + p.off) : p.Lk;
  // this block's tiles; the sub-tiles with a key that this wavefront sees, their tiles, and those of which all of its queries see all keys
  const int total = max(0, n_end + ROWS - 1) / ROWS;
  int w_subs = max(0, n_end + 31) / 32, w_full = p.Lk / ROWS;
  if (p.causal) {
    w_subs = min(w_subs, max(0, wq0 + 32 + p.off + 31) / 32);
    w_full = min(w_full, max(0, wq0 + 1 + p.off) / ROWS);
  }
  const int w_total = (w_subs + 1) / 2;

  bf16x8 qf[KS], dof[KS];
  fetch_rows(qf, static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h, p.sq.l, qi, p.Lq, g);
  fetch_rows(dof, static_cast<const bf16*>(p.dout) + b * p.sdo.b + h * p.sdo.h, p.sdo.l, qi, p.Lq, g);
  const int64_t head = (int64_t)b * p.Hq + h;
  float lse2 = p.lse[head * p.Lq + min(qi, p.Lq - 1)];
  float nd = neg_delta[head * p.Lq + min(qi, p.Lq - 1)];
  f32x16 start;   // dP starts from -delta: one add less per element
  const int lim = p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1;   // last key this lane's query sees
  const float c2 = p.scale_log2e;

  Bringer bk, bv;
  bk.init(p.sk.l, wave, lane);
  bv.init(p.sv.l, wave, lane);
  int lt = 0;   // the tile being brought, the last one again where there are no more
  const bf16* ktp = static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const bf16* vtp = static_cast<const bf16*>(p.v) + b * p.sv.b + hk * p.sv.h;
  auto load = [&](int part) INLINE {   // 0, 1: halves of K; 2, 3: of V
    bf16* st = ring + (lt & (DQ_SLOTS - 1)) * DQ_STAGE;
    const int rows = p.Lk - lt * ROWS;
    if (part < 2) bk.load(st, ktp, rows, part, wave);
    else bv.load(st + TILE, vtp, rows, part - 2, wave);
  };
  auto next = [&]() INLINE {
    const int to = min(lt + 1, total - 1), step = to - lt;
    lt = to;
    ktp += (int64_t)step * (ROWS / 2 * bk.row_bytes);
    vtp += (int64_t)step * (ROWS / 2 * bv.row_bytes);
  };

  f32x16 dq[DT], s[2], dp[2];   // of either sub-tile of a tile: S, then P; dP, then dS
  clear(dq);
  bf16x8 dsf[2];
  Readers<D> rd;
  rd.init(ring, g, i);
  typedef const bf16x8 __attribute__((address_space(3))) * frag_ptr;
  // from tile it's place in the ring to the next one's
  auto onward = [&](int it) INLINE { return (it + 1) & (DQ_SLOTS - 1) ? DQ_STAGE * 2 : -(DQ_SLOTS - 1) * DQ_STAGE * 2; };
  bf16x8 fr[2 * KS];   // K rows, k-step n; V rows, k-step n - 4
  TrFrag tf[4];        // K^T, n = 2 ss + dt
  auto read_row = [&](int n, int kt) INLINE {
    fr[n] = *(frag_ptr)(uintptr_t)(rd.row[n & 3] + 2 * ((n >> 2) * ROWS + 32 * kt) * D);
  };
  auto read_col = [&](auto n_, auto kt_) INLINE {
    constexpr int n = decltype(n_)::value, KT = decltype(kt_)::value;
    read_tr<32 * KT + 16 * (n >> 1)>(tf[n], rd.tr[2 * (n & 1)], rd.tr[2 * (n & 1) + 1]);
  };
  // The vector work of a sub-tile in 24 steps of a product's length from the first product of its S on: element e becomes P in step
  // 5 + 13 e / 16 (S is there from step 5 on) and dS in step 10 + 10 e / 16 (dP from step 10 on); the products of dQ are steps 20 to 23.
  auto vector = [&](int step, int t, auto kt_, auto masked) INLINE {
    constexpr int KT = decltype(kt_)::value;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      if (10 + 10 * e / 16 == step) {
        dp[KT][e] *= s[KT][e];
        if (e & 1) dsf[e >> 3][e & 7] = (bf16)dp[KT][e], dsf[e >> 3][(e & 7) - 1] = (bf16)dp[KT][e - 1];
      }
      if (5 + 13 * e / 16 == step) {
        float x = fmaf(s[KT][e], c2, -lse2);
        if (decltype(masked)::value) x = t * ROWS + 32 * KT + acc_row(e, g) > lim ? -INFINITY : x;
        s[KT][e] = ody_exp2(x);
      }
    }
  };

  // One call: S and dP of the sub-tile after (tile it, sub-tile KT), then dQ of this one; under them the vector work of both.
  auto unit = [&](int it, auto kt_, auto masked) INLINE {
    constexpr int KT = decltype(kt_)::value, NKT = KT ^ 1;
    const int nt = KT ? it + 1 : it;   // the sub-tile after; behind that, sub-tile KT of tile it + 1
    std::integral_constant<int, NKT> nkt;
#pragma unroll
    for (int m = 0; m < 12; m++) {
      if (m == 8) {
        WAIT_LDS(4);
#pragma unroll
        for (int n = 0; n < 4; n++) tie(tf[n]);
      }
      if (m < 4) s[NKT] = mfma32(fr[m], qf[m], m == 0 ? f32x16{0} : s[NKT]);
      else if (m < 8) dp[NKT] = mfma32(fr[m], dof[m - 4], m == 4 ? start : dp[NKT]);
      else dq[m & 1] = mfma32(value(tf[m - 8]), dsf[(m - 8) >> 1], dq[m & 1]);
      FENCE();
      if (m == 0) read_col(std::integral_constant<int, 0>{}, kt_);
      if (m == 1) read_col(std::integral_constant<int, 1>{}, kt_);
      if (m == 2) read_col(std::integral_constant<int, 2>{}, kt_);
      if (m == 3) read_col(std::integral_constant<int, 3>{}, kt_);
      if (KT == 0 && m == 4) {
        // the tile after this one has landed (behind it the 4 loads of the next); everyone is done with the one before this
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        next();
      }
      if (m >= 4) read_row(m - 4, KT);
      if (KT == 0 && (m == 6 || m == 9)) load(m == 9);
      if (KT == 1 && (m == 1 || m == 5)) load(2 + (m == 5));
      vector(12 + m, it, kt_, masked);
      vector(m, nt, nkt, masked);
      if (KT == 1 && m == 4)
#pragma unroll
        for (int n = 0; n < KS; n++) rd.tr[n] += onward(it);
      if (KT == 1 && m == 11)
#pragma unroll
        for (int n = 0; n < KS; n++) rd.row[n] += onward(it + 1);
      FENCE();
    }
  };
  std::integral_constant<int, 0> c0;
  std::integral_constant<int, 1> c1;

  if (total > 0) {
    auto all = [&]() INLINE {
#pragma unroll
      for (int n = 0; n < 4; n++) load(n);
    };
    all();
    next();
    all();
    next();
    all();
    settle_rows(qf, qi, p.Lq);   // on their way in front of the tiles
    settle_rows(dof, qi, p.Lq);
    asm volatile("" : "+v"(lse2), "+v"(nd));
    lse2 = qi >= p.Lq || lse2 == -INFINITY ? INFINITY : lse2 * ODY_LOG2E;   // past the end, or a query that saw no key: P = 0
#pragma unroll
    for (int r = 0; r < 16; r++) start[r] = nd;
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");   // the first tile
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int it = 0;
    if (w_total > 0) {
#pragma unroll
      for (int n = 0; n < 8; n++) read_row(n, 0);
#pragma unroll
      for (int n = 0; n < 4; n++) {
        s[0] = mfma32(fr[n], qf[n], n == 0 ? f32x16{0} : s[0]);
        dp[0] = mfma32(fr[4 + n], dof[n], n == 0 ? start : dp[0]);
      }
#pragma unroll
      for (int m = 0; m < 12; m++) vector(m, 0, c0, std::true_type{});
#pragma unroll
      for (int n = 0; n < 8; n++) read_row(n, 1);
#pragma unroll
      for (int n = 0; n < KS; n++) rd.row[n] += onward(0);   // the loop reads rows one tile ahead of columns
      FENCE();
      for (; it + 1 < min(w_total, w_full); it++) {
        unit(it, c0, std::false_type{});
        unit(it, c1, std::false_type{});
      }
      for (; it < w_total; it++) {   // (behind the last tile a sub-tile is formed that nobody uses)
        unit(it, c0, std::true_type{});
        if (2 * it + 1 < w_subs) unit(it, c1, std::true_type{});
        else load(2), load(3);
      }
    }
    // the other wavefronts' tiles: keep bringing this one's share of them
    for (; it < total; it++) {
      asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      next();
      all();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  if (qi < p.Lq) store_dq(p, dq, b, h, qi, g);
}

}  // namespace

int ody_launch_attn_fwd_hd64_pipe(const AttnParams& p, int groups, hipStream_t st) {
  const size_t smem = (size_t)groups * 2 * FW_SLOTS * TILE * sizeof(bf16);
  auto kern = groups == 2 ? &attn_fwd_hd64_pipe_kernel<2> : &attn_fwd_hd64_pipe_kernel<1>;
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, "attn_fwd_hd64_pipe")) return rc;
  const int64_t blocks = (int64_t)p.B * p.Hq * ((p.Lq + FW_BM - 1) / FW_BM);
  ODY_LAUNCH("attn_fwd_hd64_pipe", st, kern, dim3((unsigned)blocks), dim3(256 * groups), smem, p);
  return ody_check_launch("attn_fwd_hd64_pipe");
}

int ody_launch_attn_bwd_hd64_dkdv_pipe(const AttnParams& p, const float* neg_delta, const float* neg_lse, float* part, hipStream_t st) {
  constexpr size_t smem = (size_t)KV_SLOTS * KV_STAGE * sizeof(bf16);
  auto kern = part ? &attn_bwd_hd64_dkdv_pipe_kernel<true> : &attn_bwd_hd64_dkdv_pipe_kernel<false>;
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, "attn_bwd_hd64_dkdv_pipe")) return rc;
  const int64_t blocks = (int64_t)p.B * p.Hq * ((p.Lk + KV_BN - 1) / KV_BN);
  ODY_LAUNCH("attn_bwd_hd64_dkdv_pipe", st, kern, dim3((unsigned)blocks), dim3(256), smem, p, neg_delta, neg_lse, part);
  return ody_check_launch("attn_bwd_hd64_dkdv_pipe");
}

int ody_launch_attn_bwd_hd64_dq_pipe(const AttnParams& p, const float* neg_delta, hipStream_t st) {
  constexpr size_t smem = (size_t)DQ_SLOTS * DQ_STAGE * sizeof(bf16);
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(&attn_bwd_hd64_dq_pipe_kernel), smem, "attn_bwd_hd64_dq_pipe")) return rc;
  const int64_t blocks = (int64_t)p.B * p.Hq * ((p.Lq + DQ_BM - 1) / DQ_BM);
  ODY_LAUNCH("attn_bwd_hd64_dq_pipe", st, attn_bwd_hd64_dq_pipe_kernel, dim3((unsigned)blocks), dim3(256), smem, p, neg_delta);
  return ody_check_launch("attn_bwd_hd64_dq_pipe");
}
