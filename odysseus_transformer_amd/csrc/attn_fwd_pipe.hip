// Flash-attention forward, head_dim 128, bf16, on the tile machinery of attn_tile.h.  Query-stationary, computed
// transposed, lane = query column:
//
//      S^T = K Q^T            A: K rows (LDS tile)          B: Q^T (registers)
//      P^T = exp2(S^T c - m)  per-lane reference m, per-lane row sum
//      O^T += V^T P^T         A: V^T (transposed image)     B: P^T = accumulator layout of S^T
//
// A block of 4 wavefronts, one per SIMD with its whole register file: 64 queries each, as two halves that share every fragment read from LDS.
// A turn of the loop forms O^T of tile t and S^T of tile t + 1 in four phases of 16 MFMAs, and under each MFMA one element of P, of the
// sub-tile whose scores are complete and whose turn as an operand is next:
//
//      S^T(t + 1), first 32 keys      P(t), second 32 keys, queries 0 .. 31
//      O^T += P(t), first 32 keys     P(t), second 32 keys, queries 32 .. 63
//      S^T(t + 1), second 32 keys     P(t + 1), first 32 keys, queries 0 .. 31
//      O^T += P(t), second 32 keys    P(t + 1), first 32 keys, queries 32 .. 63
//
// so that matrix and vector pipe are busy at the same time by the order of the instructions and not by what a second wavefront on the SIMD
// happens to do.  Bound: power, behind it issue: an MFMA's 32 cycles hold an exponential (8), three to four other vector instructions, half an
// LDS read and a scalar instruction (4 each).  Against the kernel it replaced (8 wavefronts, two per SIMD, 32 queries each, a tile's S^T, P and
// O^T one after the other), two boxes: 4 heads, L = 32768, causal 976 -> 833 us (constant operands, where power is no bound, 779 -> 633), 32 heads
// on 8, L = 16384: 2040 -> 1740, 4 heads, 8192 queries on 16384 keys 243 -> 211; matrix pipe 56 -> 68 % busy.  What of it is what: the order 6 %,
// an element in three steps, each under another MFMA, 3 %; the direct loads spread over the turn, with few scalar instructions, 4 %; a whole
// phase's fragments in flight, with two waits per phase instead of eight, 3 %.
//
// The reference m of a query is fixed by its first 32 keys (key 0 is among them, and a query that
// sees any key sees key 0): the loop neither tracks maxima nor rescales O.  A later score that
// outgrows the reference by more than fp32 can hold shows up as a row sum that overflowed, or, with large values, as an
// accumulator of O that did; the 256-query block is then flagged and redone by the online-rescaling kernel.
//
// A call with few query blocks (16384 queries are 64 per head; the off-diagonal steps of a zigzag ring have 32) leaves
// compute units idle or, under a causal mask, waiting for the one with the longest block: then every block's key range
// is cut into 2 or 4 parts, one block per (query block, part); each writes its normalised partial result and
// log-sum-exp in fp32 and a small kernel merges the parts with the arithmetic of the ring's block merge.
#include <type_traits>
#include "attn_params.h"
#include "attn_tile.h"

namespace {

using namespace tile128;

constexpr int D = 128, KS = D / 16, DT = D / 32, BN = 64;
constexpr int FW_WAVES = 4, FW_QT = 2, FW_BM = 32 * FW_QT * FW_WAVES, FW_THREADS = 64 * FW_WAVES;
constexpr int FW_SLOTS = 4;                        // of the K ring and of the ring of V^T images
static_assert(FW_WAVES == 4, "the load split and the vmcnt waits assume 4 wavefronts");
#define FENCE() __builtin_amdgcn_sched_barrier(0)
#define INLINE __attribute__((always_inline))

// nsplit > 1: block id = split + nsplit * (the usual id), the block takes part `split` of its tiles; part_out
// [split][B][Lq][Hq][D] and part_lse [split][B][Hq][Lq] in fp32 take the place of p.out / p.lse.  Under a causal mask a
// later part may start beyond the first keys of some of its queries: their reference is then 0 instead of a score,
// which the overflow flag covers like any other reference that turns out too low.
__global__ __launch_bounds__(FW_THREADS, 1) void attn_fwd_pipe_kernel(const AttnParams p, const bf16* __restrict__ vimg,
                                                                  int* __restrict__ bail_flags, int nsplit,
                                                                  float* __restrict__ part_out,
                                                                  float* __restrict__ part_lse) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  bf16* kring = reinterpret_cast<bf16*>(smem_raw);          // [FW_SLOTS][TILE_ELEMS]
  bf16* vring = kring + FW_SLOTS * TILE_ELEMS;              // [FW_SLOTS][IMG_ELEMS]

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5,
            i = lane & 31;
  const int split = blockIdx.x % nsplit;
  const BlockCoord bc = ody_block_coord_of(blockIdx.x / nsplit, p.Hq, p.B);
  const int nqb = gridDim.x / (p.Hq * p.B * nsplit);
  const int qblk = p.causal ? (nqb - 1 - bc.rank) : bc.rank;   // heaviest blocks first
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * FW_BM, wq0 = q0 + wave * 32 * FW_QT;

  const bf16* qp = static_cast<const bf16*>(p.q) + b * p.sq.b + h * p.sq.h;
  const bf16* kp = static_cast<const bf16*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const int kv_tiles = (p.Lk + BN - 1) / BN;
  const bf16* vp = vimg + ((int64_t)b * p.Hkv + hk) * kv_tiles * IMG_ELEMS;

  const int q_hi = min(q0 + FW_BM, p.Lq) - 1;
  int n_end = p.causal ? min(p.Lk, q_hi + p.off + 1) : p.Lk;
  if (n_end < 0) n_end = 0;
  int ntiles = (n_end + BN - 1) / BN;
  int n_full = p.Lk / BN;   // tiles [0, n_full) need no mask for any wavefront of the block
  if (p.causal) n_full = min(n_full, max(0, (q0 + p.off + 1) / BN));
  n_full = min(n_full, ntiles);
  // this block's part of the tiles: [t_first, ntiles)
  int t_first = 0;
  if (nsplit > 1) {
    const int per = (ntiles + nsplit - 1) / nsplit;
    t_first = min(split * per, ntiles);
    ntiles = min(t_first + per, ntiles);
  }
  // end of those that this wavefront's queries see a key of
  int w_end = ntiles;
  if (p.causal) w_end = min(ntiles, max(t_first, (wq0 + 32 * FW_QT - 1 + p.off + BN) / BN));

  // The direct loads of a K tile and of a V^T image, in four quarters of one instruction per wavefront each: `lk` and `lv` are the tiles being
  // brought (the last one again where there are no more).  Buffer loads: behind loads of the flat kind the compiler waits for all LDS reads in
  // flight in front of each use of one.
  if (p.sk.l >= TILE_MAX_STRIDE) {   // beyond a tile's 32-bit offsets: left to the kernel behind
    if (tid == 0) atomicOr(bail_flags + ((int64_t)b * p.Hq + h) * nqb + qblk, 1);
    return;
  }
  const int krow = 2 * (int)p.sk.l;   // bytes
  const int kcol = 16 * (lane & 15), klane = (4 * wave + (lane >> 4)) * krow + kcol, vlane = 1024 * wave + 16 * lane;
  const int last = max(ntiles - 1, 0);   // (a block without tiles brings tile 0 and leaves it)
  int lk = min(t_first, last), lv = lk;
  const bf16* lkp = kp + (int64_t)lk * BN * p.sk.l;
  const bf16* lvp = vp + (int64_t)lk * IMG_ELEMS;
  int k_room = p.Lk - 1 - lk * BN;   // rows behind the tile's first one
  int k_last = min(k_room, BN - 1) * krow + kcol;   // this lane's columns of the tile's last row, which rows past the end re-read
  auto load_k = [&](int j) INLINE {
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(lkp), (short)0, 0x7fffffff, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_ptr)(kring + (lk & (FW_SLOTS - 1)) * TILE_ELEMS + (4 * j + wave) * GROUP_ELEMS), 16,
                                             min(klane + j * 16 * krow, k_last), 0, 0, 0);
  };
  auto load_v = [&](int j) INLINE {
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(lvp), (short)0, IMG_BYTES, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_ptr)(vring + (lv & (FW_SLOTS - 1)) * IMG_ELEMS + (4 * j + wave) * 512), 16,
                                             vlane, 4096 * j, 0, 0);
  };
  auto next_k = [&]() INLINE {
    const int to = min(lk + 1, last), step = to - lk;
    lk = to;
    lkp += (unsigned)(step * (BN / 2 * krow));
    k_room -= step * BN;
    k_last = min(k_room, BN - 1) * krow + kcol;
  };
  auto next_v = [&]() INLINE {
    const int to = min(lv + 1, last), step = to - lv;
    lv = to;
    lvp += step << 13;
  };
  static_assert(IMG_ELEMS == 1 << 13, "the step of next_v");

  // K tiles t_first .. + 3 and V^T images .. + 2, of the last ones a quarter (the loop brings the rest), and the queries behind the first of them: one
  // wait for memory in front of the first products, not one for the queries and another for the tiles, and no branches, with which the compiler
  // loses count of the loads in flight.  Causal, 4 x 24 heads, L = 820: 52.2 -> 50.5 us (backward, alike, 152 -> 146); long rows within 1 %.
#pragma unroll
  for (int j = 0; j < 4; j++) load_k(j);
  FENCE();
  bf16x8 qf[FW_QT][KS];
#pragma unroll
  for (int qt = 0; qt < FW_QT; qt++)
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
      qf[qt][ks] = *reinterpret_cast<const bf16x8*>(qp + (int64_t)min(wq0 + 32 * qt + i, p.Lq - 1) * p.sq.l + 16 * ks + 8 * g);
  FENCE();
#pragma unroll
  for (int a = 0; a < 3; a++) {
    next_k();
    if (a > 0) next_v();
#pragma unroll
    for (int j = 0; j < (a < 2 ? 4 : 1); j++) {
      load_k(j);
      load_v(j);
    }
  }
  FENCE();
#pragma unroll
  for (int qt = 0; qt < FW_QT; qt++)
#pragma unroll
    for (int ks = 0; ks < KS; ks++) asm volatile("" : "+v"(qf[qt][ks]));
  if (wq0 + 32 * FW_QT > p.Lq) {   // rows past the end are zeros
#pragma unroll
    for (int qt = 0; qt < FW_QT; qt++)
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
        if (wq0 + 32 * qt + i >= p.Lq) qf[qt][ks] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  int lim[FW_QT];   // last key this lane's queries see
#pragma unroll
  for (int qt = 0; qt < FW_QT; qt++) lim[qt] = p.causal ? min(p.Lk - 1, wq0 + 32 * qt + i + p.off) : p.Lk - 1;
  const float c2 = p.scale_log2e;
  const int rbase = row_frag_base(g, i), ibase = image_frag_base(g, i);

  f32x16 o[FW_QT][DT];
#pragma unroll
  for (int qt = 0; qt < FW_QT; qt++)
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int r = 0; r < 16; r++) o[qt][dt][r] = 0.f;
  float ref_c[FW_QT] = {0.f, 0.f};          // reference * scale * log2(e); 0 for a query that sees no key
  // this lane's partial row sums in four chains, for the roundings of a sum in order grow with its length: rms error of lse against 64 bits, 4 heads,
  // L = 32768, causal, 6.7e-7 with two chains, 5.4e-7 with four; 32768 keys, full, 8.2e-7 and 6.0e-7.  The time is the same.
  float l4[FW_QT][4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};

  f32x16 s[2][FW_QT];        // [sub-tile][half of the queries]
  bf16x8 pb[2][FW_QT][2];    // P of a sub-tile
  auto score = [&](int kt, int qt, int r, int t) INLINE { return t * BN + acc_tile_row(r, g, kt) > lim[qt] ? -INFINITY : s[kt][qt][r]; };
  // The 64 elements of P that a turn of the loop forms: e = 0 .. 31 of sub-tile 1 of tile t, then those of sub-tile 0 of tile t + 1.  An element
  // takes three steps, each one product behind the one before, so that no instruction waits for its operand: a wavefront issues in order, and
  // what waits holds up the products as well.
  float y = 0.f, x1 = 0.f, x2 = 0.f;   // the exponent of the element due; the two elements before it
  auto exponent = [&](int e, int t, auto masked) INLINE {
    const int kt = (e & 63) < 32, qt = (e >> 4) & 1, r = e & 15, tile = e < 32 ? t : t + 1;
    return fmaf(decltype(masked)::value ? score(kt, qt, r, tile) : s[kt][qt][r], c2, -ref_c[qt]);
  };
  auto take = [&](int e) INLINE {   // element e: into the row sum, and, in pairs, among the operands
    const int kt = (e & 63) < 32, qt = (e >> 4) & 1, r = e & 15;
    l4[qt][r & 3] += x1;
    if (r & 1) pb[kt][qt][r >> 3][(r & 7) - 1] = (bf16)x2, pb[kt][qt][r >> 3][r & 7] = (bf16)x1;
  };
  auto weight = [&](int e, int t, auto masked) INLINE {
    const float x = ody_exp2(y);
    y = exponent(e + 1, t, masked);
    take(e == 0 ? 63 : e - 1);
    x2 = x1, x1 = x;
  };
  constexpr int PF = 8;                   // a phase's fragments; each is loaded again, for the next phase, behind its products
  constexpr int LGKM_4 = 0xc47f;          // s_waitcnt lgkmcnt(4): all but the four reads issued last, i.e. half a phase's fragments are there
  bf16x8 fr[PF];
  auto kfrag = [&](const bf16* Kt, int kt, int n) INLINE { return row_frag(Kt, rbase, n, kt); };                     // n: k-step
  auto vfrag = [&](const bf16* Vi, int kt, int n) INLINE { return image_frag(Vi, ibase, n & 3, n >> 2, kt); };       // n: 4 * ss + dt
  // The four phases of an iteration: 16 MFMAs each, with one element of P formed under each of them.  `fr` holds the first PF fragments of
  // the phase and is left with those of the next one.
  auto s_phase = [&](int kt, const bf16* Vnext, int e0, int t, int load, auto masked) INLINE {
#pragma unroll
    for (int n = 0; n < 8; n++) {
#pragma unroll
      for (int qt = 0; qt < FW_QT; qt++) {
        if ((n & 3) == 0 && qt == 0) __builtin_amdgcn_s_waitcnt(LGKM_4);
        if (n == 0) mfma32_new(s[kt][qt], fr[n % PF], qf[qt][n]);
        else mfma32_onto(s[kt][qt], fr[n % PF], qf[qt][n]);
        FENCE();
        if (n == 2 && qt == 0) load_k(load);
        if (n == 5 && qt == 0) load_v(load);
        if (qt == 1) fr[n % PF] = vfrag(Vnext, kt, n);
        weight(e0 + 2 * n + qt, t, masked);
        FENCE();
      }
    }
  };
  auto pv_phase = [&](int kt, const bf16* Knext, int e0, int t, int load, auto masked) INLINE {
#pragma unroll
    for (int n = 0; n < 8; n++) {
#pragma unroll
      for (int qt = 0; qt < FW_QT; qt++) {
        if ((n & 3) == 0 && qt == 0) __builtin_amdgcn_s_waitcnt(LGKM_4);
        o[qt][n & 3] = mfma32(fr[n % PF], pb[kt][qt][n >> 2], o[qt][n & 3]);
        FENCE();
        if (n == 2 && qt == 0) load_k(load);
        if (n == 5 && qt == 0) load_v(load);
        if (qt == 1) fr[n % PF] = kfrag(Knext, kt ^ 1, n);
        weight(e0 + 2 * n + qt, t, masked);
        FENCE();
      }
    }
  };
  auto kslot = [&](int t) { return kring + (t & (FW_SLOTS - 1)) * TILE_ELEMS; };
  auto vslot = [&](int t) { return vring + (t & (FW_SLOTS - 1)) * IMG_ELEMS; };
  auto turn = [&](int t, auto masked) INLINE {
    s_phase(0, vslot(t), 0, t, 1, masked);
    pv_phase(0, kslot(t + 1), 16, t, 2, masked);
    s_phase(1, vslot(t), 32, t, 3, masked);
    // K tile t + 2 and V^T image t + 1 have landed (behind them the 8 loads of the tiles after); everyone is done with K tile t + 1 and
    // V^T image t - 1
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    next_k();
    next_v();
    pv_phase(1, kslot(t + 2), 48, t, 0, masked);
  };

  if (t_first < ntiles) {
    asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int t = t_first;
    if (t < w_end) {
      // S of the first tile, the references, P of its first half
      const bf16* Kt = kslot(t);
#pragma unroll
      for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int n = 0; n < 8; n++) {
          const bf16x8 f = kfrag(Kt, kt, n);
#pragma unroll
          for (int qt = 0; qt < FW_QT; qt++)
            if (n == 0) mfma32_new(s[kt][qt], f, qf[qt][n]);
            else mfma32_onto(s[kt][qt], f, qf[qt][n]);
        }
      asm volatile("s_nop 15\n\ts_nop 7" : "+v"(s[0][0]), "+v"(s[0][1]), "+v"(s[1][0]), "+v"(s[1][1]));
#pragma unroll
      for (int qt = 0; qt < FW_QT; qt++) {   // the reference: the largest score among the 32 keys of sub-tile 0 (key 0 is one of them)
        float m = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r++) m = fmaxf(m, score(0, qt, r, t));
        m = half_swap_max(m);
        ref_c[qt] = (m != -INFINITY) ? m * c2 : 0.f;
      }
#pragma unroll
      for (int e = 32; e < 64; e++) {   // the last one is left to be taken by the first turn
        x2 = x1, x1 = ody_exp2(exponent(e, t - 1, std::true_type{}));
        if (e < 63) take(e);
      }
      y = exponent(0, t, std::true_type{});
#pragma unroll
      for (int n = 0; n < PF; n++) fr[n] = kfrag(kslot(t + 1), 0, n);
      FENCE();
      for (; t + 1 < min(w_end, n_full); t++) turn(t, std::false_type{});
      for (; t + 1 < w_end; t++) turn(t, std::true_type{});
      // the last tile: P of its second half, the products
      const bf16* Vi = vslot(t);
      take(63);
#pragma unroll
      for (int e = 0; e < 32; e++) {
        x2 = x1, x1 = ody_exp2(exponent(e, t, std::true_type{}));
        take(e);
      }
#pragma unroll
      for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int n = 0; n < 8; n++) {
          const bf16x8 f = vfrag(Vi, kt, n);
#pragma unroll
          for (int qt = 0; qt < FW_QT; qt++) o[qt][n & 3] = mfma32(f, pb[kt][qt][n >> 2], o[qt][n & 3]);
        }
    }
    // the other wavefronts' tiles: keep bringing this one's share of them
    for (; t + 1 < ntiles; t++) {
      for (int j = 1; j < 4; j++) {
        load_k(j);
        load_v(j);
      }
      asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      next_k();
      next_v();
      load_k(0);
      load_v(0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- epilogue
#pragma unroll
  for (int qt = 0; qt < FW_QT; qt++) {
    const int qi = wq0 + 32 * qt + i;
    const float lt = half_swap_sum((l4[qt][0] + l4[qt][1]) + (l4[qt][2] + l4[qt][3]));
    float zero[4] = {0.f, 0.f, 0.f, 0.f};   // 0 times the accumulators of O: 0 unless one of them is not finite
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
      for (int r = 0; r < 16; r++) zero[r & 3] = fmaf(o[qt][dt][r], 0.f, zero[r & 3]);
    const bool finite = (zero[0] + zero[1]) + (zero[2] + zero[3]) == 0.f;
    if (__builtin_amdgcn_ballot_w64(!finite || !(lt < 0x1p100f)) != 0 && lane == 0)
      atomicOr(bail_flags + ((int64_t)b * p.Hq + h) * nqb + qblk, 1);
    if (qi >= p.Lq) continue;
    const float inv = lt > 0.f ? 1.f / lt : 0.f, lse = lt > 0.f ? (ref_c[qt] + __log2f(lt)) * ODY_LN2 : -INFINITY;
    if (nsplit > 1) {   // this part's normalised result and log-sum-exp, for the merge kernel
      float* op = part_out + ((((int64_t)split * p.B + b) * p.Lq + qi) * p.Hq + h) * D;
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int a = 0; a < 4; a++) {
          f32x4 w;
#pragma unroll
          for (int e = 0; e < 4; e++) w[e] = o[qt][dt][4 * a + e] * inv;
          *reinterpret_cast<f32x4*>(op + 32 * dt + 8 * a + 4 * g) = w;
        }
      if (g == 0) part_lse[(((int64_t)split * p.B + b) * p.Hq + h) * p.Lq + qi] = lse;
    } else {
      bf16* op = static_cast<bf16*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)qi * p.so.l;
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int a = 0; a < 4; a++) {
          bf16x4 w;
#pragma unroll
          for (int e = 0; e < 4; e++) w[e] = (bf16)(o[qt][dt][4 * a + e] * inv);
          *reinterpret_cast<bf16x4*>(op + 32 * dt + 8 * a + 4 * g) = w;
        }
      if (g == 0) p.lse[((int64_t)b * p.Hq + h) * p.Lq + qi] = lse;
    }
  }
}

// out, lse of a query from its `nsplit` parts: lse = log sum_s exp(lse_s), out = sum_s exp(lse_s - lse) out_s -- the
// ring merge (decoder/ring.py:30-37 of the reference reaches it through ring_flash_attn) over all parts at once.
// One thread per 4 elements of a (query, head) row.
__global__ __launch_bounds__(256) void attn_fwd_split_merge_kernel(const AttnParams p, int nsplit,
                                                                   const float* __restrict__ part_out,
                                                                   const float* __restrict__ part_lse) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;   // over B * Lq * Hq * D / 4
  const int64_t total = (int64_t)p.B * p.Lq * p.Hq * (D / 4);
  if (idx >= total) return;
  const int d4 = idx % (D / 4);
  const int h = (idx / (D / 4)) % p.Hq;
  const int qi = (idx / ((int64_t)(D / 4) * p.Hq)) % p.Lq;
  const int b = idx / ((int64_t)(D / 4) * p.Hq * p.Lq);
  const int64_t plane_o = (int64_t)p.B * p.Lq * p.Hq * D, plane_l = (int64_t)p.B * p.Hq * p.Lq;
  const int64_t li = ((int64_t)b * p.Hq + h) * p.Lq + qi;
  float m = -INFINITY;
  for (int s = 0; s < nsplit; s++) m = fmaxf(m, part_lse[s * plane_l + li]);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  float wsum = 0.f;
  if (m != -INFINITY) {
    const float* po = part_out + (((int64_t)b * p.Lq + qi) * p.Hq + h) * D + 4 * d4;
    for (int s = 0; s < nsplit; s++) {
      const float w = __expf(part_lse[s * plane_l + li] - m);   // exp(-inf) = 0 for a part that saw no key
      wsum += w;
      acc += w * *reinterpret_cast<const f32x4*>(po + s * plane_o);
    }
  }
  const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
  bf16x4 w;
#pragma unroll
  for (int e = 0; e < 4; e++) w[e] = (bf16)(acc[e] * inv);
  *reinterpret_cast<bf16x4*>(static_cast<bf16*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)qi * p.so.l + 4 * d4) = w;
  if (d4 == 0) p.lse[li] = wsum > 0.f ? m + __logf(wsum) : -INFINITY;
}

inline size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// Parts of a query block's key range.  With fewer blocks than it takes to keep the chip's 256 compute units busy and
// balanced -- one block each when all blocks are equally long (fully visible keys), two each when they are not (under
// a causal mask block i is i + 1 tiles long, and only with a second, lighter block per unit does the heaviest-first
// order even that out) -- the range is cut into 2 or 4 parts of at least 8 tiles (on average, when causal).
int key_splits(int B, int Lq, int Lk, int Hq, bool causal) {
  const int64_t blocks = (int64_t)B * Hq * ((Lq + FW_BM - 1) / FW_BM);
  const int64_t want = causal ? 512 : 256;
  const int tiles = ((causal ? min(Lk, Lq + max(Lk - Lq, 0)) : Lk) + BN - 1) / BN;
  int s = 1;
  while (s < 4 && blocks * s * 2 <= want && tiles >= 16 * s) s *= 2;
  return s;
}

}  // namespace

int ody_attn_fwd_pipe_parts(int B, int Lq, int Lk, int Hq, int causal) { return key_splits(B, Lq, Lk, Hq, causal != 0); }

// workspace: [flags of the 256-query blocks | transposed images of V | fp32 parts of a key-split call: out, lse]
size_t ody_attn_fwd_pipe_workspace(int B, int Lq, int Lk, int Hq, int Hkv, bool with_split) {
  const size_t flags = align256((size_t)B * Hq * ((Lq + FW_BM - 1) / FW_BM) * sizeof(int));
  size_t n = flags + align256(ody_attn_images_bytes(B, Lk, Hkv));
  const int ns = with_split ? max(key_splits(B, Lq, Lk, Hq, false), key_splits(B, Lq, Lk, Hq, true)) : 1;
  if (ns > 1) n += align256((size_t)ns * B * Lq * Hq * D * sizeof(float)) + align256((size_t)ns * B * Hq * Lq * sizeof(float));
  return n;
}

int ody_launch_attn_fwd_pipe(const AttnParams& p, void* workspace, size_t workspace_bytes, hipStream_t st) {
  constexpr size_t smem = (size_t)FW_SLOTS * (TILE_ELEMS + IMG_ELEMS) * sizeof(bf16);
  int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(&attn_fwd_pipe_kernel), smem, "attn_fwd");
  if (rc) return rc;
  const int nqb = (p.Lq + FW_BM - 1) / FW_BM;
  const int nflags = p.B * p.Hq * nqb;
  char* w = static_cast<char*>(workspace);
  int* flags = reinterpret_cast<int*>(w);
  bf16* images = reinterpret_cast<bf16*>(w + align256((size_t)nflags * sizeof(int)));
  rc = ody_launch_attn_images(p.v, p.sv, p.B, p.Lk, p.Hkv, images, flags, nflags, st);
  if (rc) return rc;
  // the key split, where the caller's workspace has room for the parts (the allocation-free entry point's fixed
  // scratch may not)
  int ns = key_splits(p.B, p.Lq, p.Lk, p.Hq, p.causal != 0);
  if (ns > 1 && workspace_bytes < ody_attn_fwd_pipe_workspace(p.B, p.Lq, p.Lk, p.Hq, p.Hkv, true)) ns = 1;
  float* part_out = nullptr;
  float* part_lse = nullptr;
  if (ns > 1) {
    char* parts = w + align256((size_t)nflags * sizeof(int)) + align256(ody_attn_images_bytes(p.B, p.Lk, p.Hkv));
    part_out = reinterpret_cast<float*>(parts);
    part_lse = reinterpret_cast<float*>(parts + align256((size_t)ns * p.B * p.Lq * p.Hq * D * sizeof(float)));
  }
  dim3 grid(nqb * p.Hq * p.B * ns);
  ODY_LAUNCH("attn_fwd_pipe", st, attn_fwd_pipe_kernel, grid, dim3(FW_THREADS), smem, p, images, flags, ns, part_out, part_lse);
  rc = ody_check_launch("attn_fwd_pipe");
  if (rc) return rc;
  if (ns > 1) {
    const int64_t n4 = (int64_t)p.B * p.Lq * p.Hq * (D / 4);
    ODY_LAUNCH("attn_fwd_split_merge", st, attn_fwd_split_merge_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, p, ns,
               part_out, part_lse);
    if ((rc = ody_check_launch("attn_fwd_split_merge"))) return rc;
  }
  return ody_launch_attn_fwd_mfma_flagged(p, flags, FW_BM, st);
}
