// fp32 attention of head_dim 64 (forward and backward) on the bf16 matrix cores: every operand as the sum of three bf16 values (split3.h),
// six products for one.
//
// The fp32 matrix instruction takes 512 cycles for what these six take in 192; what is left is the splitting (6.5 vector instructions per
// element) and LDS traffic.  Streamed tiles of 32 rows are split on their way from registers to LDS, by the wavefronts that share them, and serve
// as row operands and, through the transposing read, as transposed ones (attn_rowtile.h); P and dS are split in registers, where they are
// the next product's operand.  Blocks of 32, 64 or 128 rows (rows_of_block): the more rows share a tile, the less splitting; the fewer, the more
// blocks.
//
// Operands are split times SPLIT_UP, so that the parts hold every bit of the smallest of them too, P and dS included: scores and dP take
// SPLIT_DOWN in the fma that follows them anyway, the results lose their factor where they are stored.  In the forward Q has the factor of K too:
// what is left out of a K below 2^-110 is 2^-134, times a Q below 2^96 nothing that a score's exponential shows.
//
// Results that are not finite (an infinity or NaN in the inputs, operands from 2^96 (Q in the forward) or 2^111 on, sums from 2^96 on) are formed
// again on the fp32 instruction, and so are those of rows whose scores are all that large and negative: what comes out is what it gives.
//
// Before (attn_f32.hip) / here, us: 8 heads, L = 2048, causal: forward 62 / 54, dK and dV 108 / 84, dQ 80 / 62; 16 heads, L = 4096: 387 / 240, 705 / 406,
// 508 / 315 (143 TFLOP/s forward); 219 shapes of 64 to 8192 rows, 2 to 128 heads: 1.20, 1.37 and 1.34 times in the geometric mean.
// 2-norm error against 64 bits, standard normal inputs, out / dQ / dK / dV in 1e-7, before and here: 8 heads, L = 2048, causal 2.1 / 4.6 / 5.6 / 5.2 and
// 1.9 / 3.7 / 4.6 / 4.2; 16 heads, full: 8.3 / 10.4 / 10.3 / 10.1 and 3.0 / 6.4 / 6.4 / 6.1; no output of 14 shapes is further off than before.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>
#include "attn_f32.h"
#include "attn_rowtile.h"
#include "split3.h"

namespace {

using f32tile::F_TILE;
using f32tile::LN2;
using f32tile::TileRegs;
using rowtile::Readers;
using rowtile::acc_row;
using rowtile::row_frag;

constexpr int D = 64, KS = D / 16, DT = D / 32, WAVES = 8;
constexpr int PLANE = F_TILE;                               // rows of a part of a tile, 32 x 64 bf16
constexpr int PARTS_ELEMS = 3 * F_TILE * D;                 // the parts of a tile, 12 KB; the tile in fp32 is smaller
static_assert(PARTS_ELEMS * sizeof(bf16) >= F_TILE * (D + 4) * sizeof(float), "an fp32 tile fits");

// A block is RW wavefronts of 32 rows each, GROUPS = 8 / RW times; group n takes tiles n, n + GROUPS, ...  A group has LDS for the two tiles of a
// turn (RW = 4), or for one after the other (RW = 1: no wavefront waits for another in the loop).
template <int RW>
struct Geo {
  static constexpr int GROUPS = WAVES / RW, ROWS = 32 * RW, LOADERS = 64 * RW;
  static constexpr bool ONE = RW == 1;
  static constexpr int STAGE = (ONE ? 1 : 2) * PARTS_ELEMS, SECOND = ONE ? 0 : 3 * PLANE;   // first row of the second tile's parts
  static constexpr size_t SMEM = GROUPS * STAGE * sizeof(bf16), OWN = RW * PARTS_ELEMS * sizeof(bf16);
  __device__ static __forceinline__ void sync() {
    if constexpr (ONE) wavefront_sync();
    else __syncthreads();
  }
};

// One streamed 32 x 64 tile on its way from memory to LDS: 8 consecutive elements of a row per piece
template <int NT>
struct PartTile {
  static constexpr int N = 4 * D / NT, STEP = 8 * NT / D;   // pieces per thread, rows between them
  static_assert(N * NT == 4 * D, "whole pieces");
  f32x4 v[N][2];
  // Rows past nvalid repeat the last one: their P and dS are zero, which a value that is finite leaves so, and one that is not sends the block to
  // the fp32 instruction.  ZERO, there: they read as zero (on every element of every tile that is an instruction for each).
  // LEAN: one offset of the thread's own for all of its pieces, fewer registers, and a branch.  For the instance that spills (dK and dV, 8 heads,
  // L = 2048: 89 us without, 83 with it; dQ 62.3 and 62.9, 16 heads of 4 x 484 rows 37.2 and 38.4).
  template <bool ZERO, bool LEAN = false>
  __device__ __forceinline__ void fetch(const float* src, int64_t stride, int row0, int nvalid, int tid) {
    const int first = tid / (D / 8), x = tid % (D / 8);
    const int64_t own = (int64_t)first * stride + 8 * x;
#pragma unroll
    for (int n = 0; n < N; n++) {
      const int r = first + n * STEP;
      const float* s;
      if constexpr (LEAN) {
        s = src + (int64_t)(row0 + n * STEP) * stride + own;
        if (nvalid < F_TILE) s -= (int64_t)max(r - nvalid + 1, 0) * stride;
      } else {
        s = src + (int64_t)(row0 + min(r, nvalid - 1)) * stride + 8 * x;
      }
      v[n][0] = *reinterpret_cast<const f32x4*>(s), v[n][1] = *reinterpret_cast<const f32x4*>(s + 4);
      if (ZERO && r >= nvalid) v[n][0] = v[n][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  __device__ __forceinline__ void scale(float mul) {
#pragma unroll
    for (int n = 0; n < N; n++) v[n][0] *= mul, v[n][1] *= mul;
  }
  template <bool UP = true>   // times SPLIT_UP
  __device__ __forceinline__ void put(bf16* dst, int tid) const {   // in parts, [3][32][64], chunks permuted as attn_rowtile.h wants them
#pragma unroll
    for (int n = 0; n < N; n++) {
      const int e = tid + n * NT, r = e / (D / 8), x = e % (D / 8);
      const Split3<8> s(__builtin_shufflevector(v[n][0], v[n][1], 0, 1, 2, 3, 4, 5, 6, 7) * (UP ? SPLIT_UP : 1.f));
#pragma unroll
      for (int p = 0; p < 3; p++) *reinterpret_cast<bf16x8*>(dst + (PLANE * p + r) * D + 8 * (x ^ rowtile::swz<D>(r))) = s.p[p];
    }
  }
  template <bool EXACT, bool UP = true>
  __device__ __forceinline__ void put_as(float* stage, int second, int tid) const {   // as the first or the second tile of a stage
    if constexpr (EXACT) put_f32(stage + second * (F_TILE * (D + 4)), tid);
    else put<UP>(reinterpret_cast<bf16*>(stage) + second * PARTS_ELEMS, tid);
  }
  __device__ __forceinline__ void put_f32(float* dst, int tid) const {
#pragma unroll
    for (int n = 0; n < N; n++) {
      const int e = tid + n * NT, r = e / (D / 8), x = e % (D / 8);
      f32x4* d = reinterpret_cast<f32x4*>(dst + r * (D + 4) + 8 * x);
      d[0] = v[n][0], d[1] = v[n][1];
    }
  }
};

// The parts of a wavefront's 32 rows, times `mul` and SPLIT_UP: lane (g, i) holds row i, k = 16 ks + 8 g .. + 7
__device__ __forceinline__ void load_parts(bf16x8 (&f)[KS][3], const float* base, int64_t stride, int row, bool ok, int g, float mul) {
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    typename FloatVec<8>::type x = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (ok) {
      const f32x4* s = reinterpret_cast<const f32x4*>(base + (int64_t)row * stride + 16 * ks + 8 * g);
      x = __builtin_shufflevector(s[0], s[1], 0, 1, 2, 3, 4, 5, 6, 7);
    }
    const Split3<8> p(x * (mul * SPLIT_UP));
#pragma unroll
    for (int n = 0; n < 3; n++) f[ks][n] = p.p[n];
  }
}

// Result registers 8 H .. 8 H + 7, a k-step of the next product, in parts
template <int H>
__device__ __forceinline__ void parts_of(bf16x8 (&f)[3], const f32x16& s) {
  typename FloatVec<8>::type x;
#pragma unroll
  for (int e = 0; e < 8; e++) x[e] = s[8 * H + e];
  const Split3<8> p(x);
#pragma unroll
  for (int n = 0; n < 3; n++) f[n] = p.p[n];
}

// hi + lo += T F^T for the parts of a tile from row FIRST of the stage on; f(ks, n) is part n of the other operand
template <int FIRST, typename Parts>
__device__ __forceinline__ void tile_times_parts(const Readers<D>& rd, Parts f, f32x16& hi, f32x16& lo) {
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    const bf16x8 a0 = row_frag(rd, FIRST, ks), a1 = row_frag(rd, FIRST + PLANE, ks), a2 = row_frag(rd, FIRST + 2 * PLANE, ks);
    const bf16x8 b0 = f(ks, 0), b1 = f(ks, 1), b2 = f(ks, 2);
    lo = mfma32(a2, b0, lo);
    hi = mfma32(a1, b0, hi);
    lo = mfma32(a0, b2, lo);
    hi = mfma32(a0, b1, hi);
    lo = mfma32(a1, b1, lo);
    hi = mfma32(a0, b0, hi);
  }
}

// Two products of that kind at once, each the other's independent chain; smallest parts first into one accumulator
template <int FA, int FB, typename PartsA, typename PartsB>
__device__ __forceinline__ void tiles_times_parts(const Readers<D>& rd, PartsA fa, f32x16& ca, PartsB fb, f32x16& cb) {
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    const bf16x8 a[3] = {row_frag(rd, FA, ks), row_frag(rd, FA + PLANE, ks), row_frag(rd, FA + 2 * PLANE, ks)};
    const bf16x8 b[3] = {row_frag(rd, FB, ks), row_frag(rd, FB + PLANE, ks), row_frag(rd, FB + 2 * PLANE, ks)};
    const bf16x8 xa[3] = {fa(ks, 0), fa(ks, 1), fa(ks, 2)}, xb[3] = {fb(ks, 0), fb(ks, 1), fb(ks, 2)};
#pragma unroll
    for (int n = 0; n < 6; n++) {
      constexpr int A[6] = {2, 0, 1, 1, 0, 0}, B[6] = {0, 2, 1, 0, 1, 0};
      ca = mfma32(a[A[n]], xa[B[n]], ca);
      cb = mfma32(b[A[n]], xb[B[n]], cb);
    }
  }
}

// acc += T^T W for the parts of a tile and weights in result-register order.  APART: the five smaller products of a tile are summed by
// themselves, so that a long sum is rounded three times a tile and not twelve times.  For the instances with few groups, whose sums are long,
// where there are registers: dV of 32 heads, L = 1500, in 128-row blocks is 5.8e-7 off 64 bits without and 4.0e-7 with it, on the fp32 matrix
// instruction 4.8e-7; in 32-row blocks 4.2e-7 (L = 2048) without it, 5.2e-7 on that instruction.
template <int FIRST, bool APART>
__device__ __forceinline__ void tile_t_times(const Readers<D>& rd, const f32x16& w, f32x16 (&acc)[DT]) {
  f32x16 lo[APART ? DT : 1];
  rowtile::clear(lo);
  auto half = [&](auto which) {
    constexpr int h = decltype(which)::value;
    // the transposed fragments of the three parts, both slices of the head: as rowtile::tr_frags, under one wait
    s16x4 x[12];
    asm volatile("ds_read_b64_tr_b16 %0, %12 offset:%16\n\tds_read_b64_tr_b16 %1, %13 offset:%17\n\t"
                 "ds_read_b64_tr_b16 %2, %14 offset:%16\n\tds_read_b64_tr_b16 %3, %15 offset:%17\n\t"
                 "ds_read_b64_tr_b16 %4, %12 offset:%18\n\tds_read_b64_tr_b16 %5, %13 offset:%19\n\t"
                 "ds_read_b64_tr_b16 %6, %14 offset:%18\n\tds_read_b64_tr_b16 %7, %15 offset:%19\n\t"
                 "ds_read_b64_tr_b16 %8, %12 offset:%20\n\tds_read_b64_tr_b16 %9, %13 offset:%21\n\t"
                 "ds_read_b64_tr_b16 %10, %14 offset:%20\n\tds_read_b64_tr_b16 %11, %15 offset:%21\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(x[4]), "=&v"(x[5]), "=&v"(x[6]), "=&v"(x[7]), "=&v"(x[8]),
                   "=&v"(x[9]), "=&v"(x[10]), "=&v"(x[11])
                 : "v"(rd.tr[0]), "v"(rd.tr[1]), "v"(rd.tr[2]), "v"(rd.tr[3]), "n"(2 * (FIRST + 16 * h) * D), "n"(2 * (FIRST + 16 * h + 8) * D),
                   "n"(2 * (FIRST + PLANE + 16 * h) * D), "n"(2 * (FIRST + PLANE + 16 * h + 8) * D), "n"(2 * (FIRST + 2 * PLANE + 16 * h) * D),
                   "n"(2 * (FIRST + 2 * PLANE + 16 * h + 8) * D)
                 : "memory");
    auto t = [&](int part, int dt) {
      return concat4(__builtin_bit_cast(bf16x4, x[4 * part + 2 * dt]), __builtin_bit_cast(bf16x4, x[4 * part + 2 * dt + 1]));
    };
    bf16x8 b[3];
    parts_of<h>(b, w);
#pragma unroll
    for (int n = 0; n < 6; n++) {   // smallest products first, the two slices of the head in turn
      constexpr int A[6] = {2, 0, 1, 1, 0, 0}, B[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        f32x16& to = APART && n < 5 ? lo[APART ? dt : 0] : acc[dt];
        to = mfma32(t(A[n], dt), b[B[n]], to);
      }
    }
  };
  half(std::integral_constant<int, 0>{});
  half(std::integral_constant<int, 1>{});
  if constexpr (APART) {
#pragma unroll
    for (int dt = 0; dt < DT; dt++) acc[dt] += lo[dt];
  }
}

template <int N>
__device__ __forceinline__ bool all_finite(const f32x16 (&x)[N]) {   // 0 times a value that is not is NaN
  float z[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int n = 0; n < N; n++)
#pragma unroll
    for (int r = 0; r < 16; r++) z[r & 3] = fmaf(x[n][r], 0.f, z[r & 3]);
  return (z[0] + z[1]) + (z[2] + z[3]) == 0.f;
}

// A row whose scores may have left the range that the parts' products hold, 2^96, while their differences are small: NaN, which sends
// the block to the fp32 instruction
__device__ __forceinline__ float in_range(float lse) { return __builtin_fabsf(lse) > 0x1p90f && lse != INFINITY ? __builtin_nanf("") : lse; }

// What the wavefronts exchange at the end, over the stages: a flag each, two rows of 64 values each, the groups' accumulators
constexpr size_t EX_VALUES = 256, EX_ACC = EX_VALUES + 2 * WAVES * 64 * sizeof(float);
__device__ __forceinline__ float* values(unsigned char* smem, int which, int wave) { return reinterpret_cast<float*>(smem + EX_VALUES) + (which * WAVES + wave) * 64; }
// room of the accumulators of group `grp` (from 1 on), wavefront w; N tiles of 32 x 32
template <int RW, int N>
__device__ __forceinline__ float* acc_room(unsigned char* smem, int grp, int w) {
  static_assert(EX_ACC + (size_t)(Geo<RW>::GROUPS - 1) * RW * 16 * N * 64 * sizeof(float) <= Geo<RW>::SMEM + (N > DT ? (RW == 4 ? 1 : 2) * Geo<RW>::OWN : 0), "fits");
  return reinterpret_cast<float*>(smem + EX_ACC) + ((grp - 1) * RW + w) * 16 * N * 64;
}
__device__ __forceinline__ void put_flag(unsigned char* smem, bool x, int wave, int lane) {
  const bool mine = __builtin_amdgcn_ballot_w64(x) != 0;
  if (lane == 0) reinterpret_cast<int*>(smem)[wave] = mine;
}
__device__ __forceinline__ bool any_flag(unsigned char* smem) {
  int any = 0;
#pragma unroll
  for (int w = 0; w < WAVES; w++) any |= reinterpret_cast<int*>(smem)[w];
  return __builtin_amdgcn_readfirstlane(any) != 0;
}

// What the three kernels have in common
template <int RW>
struct Place {
  int tid, lane, wave, i, g, grp, w, gtid;   // gtid: thread of the group
  float* stage;                              // of the group
  __device__ __forceinline__ explicit Place(unsigned char* smem) {
    tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 31, g = lane >> 5;
    grp = wave / RW, w = wave % RW, gtid = w * 64 + lane;
    stage = reinterpret_cast<float*>(smem + grp * Geo<RW>::STAGE * sizeof(bf16));
  }
};

// The block's own rows in parts to LDS, [RW][3][32][64]
template <int RW>
__device__ __forceinline__ void put_own(bf16* dst, const float* base, int64_t stride, int row0, int nrows, float mul, const Place<RW>& at) {
  PartTile<256> own;   // 32 rows by four wavefronts at a time
  for (int n = at.wave >> 2; n < RW; n += 2) {
    if (row0 + 32 * n < nrows) {
      own.fetch<true>(base, stride, row0 + 32 * n, min(32, nrows - row0 - 32 * n), at.tid & 255);
      own.scale(mul);
      own.put(dst + n * PARTS_ELEMS, at.tid & 255);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------- forward
template <int RW>
__global__ __launch_bounds__(64 * WAVES, 2) void attn_fwd_f32_parts_kernel(const AttnParams p) {
  using G = Geo<RW>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const Place<RW> at(smem);
  const int g = at.g, i = at.i;
  const BlockCoord bc = ody_block_coord(p.Hq, p.B);
  const int nqb = gridDim.x / (p.Hq * p.B);
  const int qblk = p.causal ? nqb - 1 - bc.rank : bc.rank;   // heaviest blocks first
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * G::ROWS, wq0 = q0 + at.w * 32, qi = wq0 + i;
  const float* qp = static_cast<const float*>(p.q) + b * p.sq.b + h * p.sq.h;
  const float* kp = static_cast<const float*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const float* vp = static_cast<const float*>(p.v) + b * p.sv.b + hk * p.sv.h;

  // last key this lane's query and the first query of the wavefront see; the key ranges of the block and of the wavefront
  const int lim = p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1;
  const int lim_first = p.causal ? min(p.Lk - 1, wq0 + p.off) : p.Lk - 1;
  const int n_end = max(0, p.causal ? min(p.Lk, min(q0 + G::ROWS, p.Lq) + p.off) : p.Lk);
  const int w_end = wq0 < p.Lq ? max(0, p.causal ? min(p.Lk, min(wq0 + 32, p.Lq) + p.off) : p.Lk) : 0;
  const int ntiles = (n_end + F_TILE - 1) / F_TILE, iters = (ntiles + G::GROUPS - 1) / G::GROUPS;
  if (ntiles == 0) {   // no row sees a key
    if (at.grp == 0 && qi < p.Lq) {
      f32x16 zero[DT];
      rowtile::clear(zero);
      f32tile::store_rows<D>(static_cast<float*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)qi * p.so.l, zero, g, 1.f, false);
      if (g == 0) p.lse[((int64_t)b * p.Hq + h) * p.Lq + qi] = -INFINITY;
    }
    return;
  }
  Readers<D> rd;
  rd.init(reinterpret_cast<bf16*>(at.stage), g, i);

  f32x16 o[DT];
  float m, l, back = 1.f / SPLIT_UP;   // l is the row sum of P times 1 / back, o that of P V times 1 / back^2
  auto walk = [&](auto exact) {
    constexpr bool EXACT = decltype(exact)::value;
    constexpr float DOWN = EXACT ? 1.f : SPLIT_DOWN, UP = EXACT ? 1.f : SPLIT_UP;   // of scores; of P
    bf16x8 qf[KS][3];
    float q32[EXACT ? D / 2 : 1];
    if constexpr (EXACT) f32tile::load_row_frag<D>(q32, qp, p.sq.l, qi, qi < p.Lq, g, p.scale_log2e);
    else load_parts(qf, qp, p.sq.l, qi, qi < p.Lq, g, p.scale_log2e * SPLIT_UP);   // scores come out in the log2 domain
    rowtile::clear(o);
    m = -INFINITY, l = 0.f;
    PartTile<G::LOADERS> kr, vr;
    auto fetch_k = [&](int t) { kr.template fetch<EXACT>(kp, p.sk.l, t * F_TILE, min(F_TILE, p.Lk - t * F_TILE), at.gtid); };
    auto fetch_v = [&](int t) { vr.template fetch<EXACT>(vp, p.sv.l, t * F_TILE, min(F_TILE, p.Lk - t * F_TILE), at.gtid); };
    if (!EXACT && at.grp < ntiles) fetch_k(at.grp), fetch_v(at.grp);
#pragma unroll 1
    for (int it = 0; it < iters; it++) {
      const int t = at.grp + G::GROUPS * it, n0 = t * F_TILE;
      G::sync();
      if (t < ntiles) {
        if (EXACT) fetch_k(t), fetch_v(t);
        kr.template put_as<EXACT, false>(at.stage, 0, at.gtid);
        if (!G::ONE) vr.template put_as<EXACT>(at.stage, 1, at.gtid);
      }
      G::sync();
      if (!EXACT && t + G::GROUPS < ntiles) {
        fetch_k(t + G::GROUPS);
        if (!G::ONE) fetch_v(t + G::GROUPS);
      }
      if (t >= ntiles || n0 >= w_end) continue;

      f32x16 s = {0.f}, s1 = {0.f};
      if constexpr (EXACT) f32tile::tile_times_frag<D>(at.stage, i, g, q32, s, s1);
      else tile_times_parts<0>(rd, [&](int ks, int n) { return qf[ks][n]; }, s, s1);
      s += s1;
      if (n0 + F_TILE - 1 > lim_first) {
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (n0 + acc_row(r, g) > lim) s[r] = -INFINITY;
      }
      float mx = s[0];
#pragma unroll
      for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
      mx = half_swap_max(mx) * DOWN;
      if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {
        const float m_new = fmaxf(m, mx), alpha = m_new == -INFINITY ? 1.f : ody_exp2(m - m_new);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; dt++) o[dt] *= alpha;
      }
      const float m_use = m == -INFINITY ? 0.f : m;
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        s[r] = ody_exp2(fmaf(s[r], DOWN, -m_use)) * UP;
        sum += s[r];
      }
      l += sum;
      if constexpr (G::ONE) {
        G::sync();
        vr.template put_as<EXACT>(at.stage, 0, at.gtid);
        G::sync();
        if (!EXACT && t + G::GROUPS < ntiles) fetch_v(t + G::GROUPS);
      }
      if constexpr (EXACT) f32tile::tile_t_times_regs<D>(at.stage + (G::ONE ? 0 : F_TILE * (D + 4)), i, g, s, o);
      else tile_t_times<G::SECOND, RW != 1>(rd, s, o);
    }
  };
  auto publish = [&]() {
    __syncthreads();   // everyone is done with the stages
    // (a row that sees a key of the group's first tile, and no score that is more than minus infinity)
    const bool lost = qi < p.Lq && at.grp * F_TILE <= lim && m == -INFINITY;
    put_flag(smem, !all_finite(o) || l * 0.f != 0.f || lost, at.wave, at.lane);
    values(smem, 0, at.wave)[at.lane] = m;
    __syncthreads();
  };
  walk(std::false_type{});
  publish();
  if (any_flag(smem)) {
    __syncthreads();
    back = 1.f;
    walk(std::true_type{});
    publish();
  }
  // the groups on a common reference
  float top = m;
#pragma unroll
  for (int n = 0; n < G::GROUPS; n++) top = fmaxf(top, values(smem, 0, n * RW + at.w)[at.lane]);
  if (top == -INFINITY) top = 0.f;
  const float mine = ody_exp2(m - top);
  l *= mine;
#pragma unroll
  for (int dt = 0; dt < DT; dt++) o[dt] *= mine;
  if (at.grp > 0) {
    values(smem, 1, at.wave)[at.lane] = l;
    rowtile::give(acc_room<RW, DT>(smem, at.grp, at.w), o, at.lane);
  }
  __syncthreads();
  if (at.grp != 0) return;
#pragma unroll 1
  for (int n = 1; n < G::GROUPS; n++) {
    l += values(smem, 1, n * RW + at.w)[at.lane];
    rowtile::take(acc_room<RW, DT>(smem, n, at.w), o, at.lane, 1.f, 1.f);
  }
  l = half_swap_sum(l);
  if (qi < p.Lq) {
    f32tile::store_rows<D>(static_cast<float*>(p.out) + b * p.so.b + h * p.so.h + (int64_t)qi * p.so.l, o, g, l > 0.f ? back / l : 0.f, false);
    if (g == 0) p.lse[((int64_t)b * p.Hq + h) * p.Lq + qi] = l > 0.f ? (top + __log2f(l * back)) * LN2 : -INFINITY;
  }
}

// ---------------------------------------------------------------------------------------------------------- dQ
template <int RW>
__global__ __launch_bounds__(64 * WAVES, 2) void attn_bwd_dq_f32_parts_kernel(const AttnParams p) {
  using G = Geo<RW>;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const Place<RW> at(smem);
  const int g = at.g, i = at.i;
  const BlockCoord bc = ody_block_coord(p.Hq, p.B);
  const int nqb = gridDim.x / (p.Hq * p.B);
  const int qblk = p.causal ? nqb - 1 - bc.rank : bc.rank;
  const int h = bc.h, b = bc.b, hk = h / p.group;
  const int q0 = qblk * G::ROWS, wq0 = q0 + at.w * 32, qi = wq0 + i;
  const float* qp = static_cast<const float*>(p.q) + b * p.sq.b + h * p.sq.h;
  const float* dop = static_cast<const float*>(p.dout) + b * p.sdo.b + h * p.sdo.h;
  const float* kp = static_cast<const float*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const float* vp = static_cast<const float*>(p.v) + b * p.sv.b + hk * p.sv.h;

  const int64_t ri = ((int64_t)b * p.Hq + h) * p.Lq + qi;
  const float lse = qi < p.Lq ? p.lse[ri] : -INFINITY;
  const float delta = qi < p.Lq ? p.delta[ri] : 0.f;
  // a query with no visible key (lse = -inf) contributes nothing
  const int lim = lse == -INFINITY ? -1 : (p.causal ? min(p.Lk - 1, qi + p.off) : p.Lk - 1);
  const int n_end = max(0, p.causal ? min(p.Lk, min(q0 + G::ROWS, p.Lq) + p.off) : p.Lk);
  const int w_end = wq0 < p.Lq ? max(0, p.causal ? min(p.Lk, min(wq0 + 32, p.Lq) + p.off) : p.Lk) : 0;
  const int ntiles = (n_end + F_TILE - 1) / F_TILE, iters = (ntiles + G::GROUPS - 1) / G::GROUPS;
  if (ntiles == 0) {   // no row sees a key
    if (at.grp == 0 && qi < p.Lq && !p.accumulate_dq) {
      f32x16 zero[DT];
      rowtile::clear(zero);
      f32tile::store_rows<D>(static_cast<float*>(p.dq) + b * p.sdq.b + h * p.sdq.h + (int64_t)qi * p.sdq.l, zero, g, 1.f, false);
    }
    return;
  }
  Readers<D> rd;
  rd.init(reinterpret_cast<bf16*>(at.stage), g, i);

  Readers<D> drd;   // RW = 1: the parts of dO, common to all wavefronts (in registers they would spill)
  if constexpr (G::ONE) {
    bf16* own = reinterpret_cast<bf16*>(smem + G::SMEM);
    put_own<RW>(own, dop, p.sdo.l, q0, p.Lq, 1.f, at);
    drd.init(own, g, i);
    __syncthreads();
  }
  f32x16 dq[DT];
  float back = SPLIT_DOWN;
  auto walk = [&](auto exact) {
    constexpr bool EXACT = decltype(exact)::value;
    constexpr float DOWN = EXACT ? 1.f : SPLIT_DOWN;
    const float ds_scale = EXACT ? p.scale : p.scale * SPLIT_UP, lse2 = (EXACT ? lse : in_range(lse)) * ODY_LOG2E;
    bf16x8 qf[KS][3], dof[G::ONE ? 1 : KS][3];
    float q32[EXACT ? D / 2 : 1], do32[EXACT ? D / 2 : 1];
    if constexpr (EXACT) {
      f32tile::load_row_frag<D>(q32, qp, p.sq.l, qi, qi < p.Lq, g, p.scale_log2e);
      f32tile::load_row_frag<D>(do32, dop, p.sdo.l, qi, qi < p.Lq, g, 1.f);
    } else {
      load_parts(qf, qp, p.sq.l, qi, qi < p.Lq, g, p.scale_log2e);
      if constexpr (!G::ONE) load_parts(dof, dop, p.sdo.l, qi, qi < p.Lq, g, 1.f);
    }
    rowtile::clear(dq);
    PartTile<G::LOADERS> kr, vr;
    auto fetch_k = [&](int t) { kr.template fetch<EXACT>(kp, p.sk.l, t * F_TILE, min(F_TILE, p.Lk - t * F_TILE), at.gtid); };
    auto fetch_v = [&](int t) { vr.template fetch<EXACT>(vp, p.sv.l, t * F_TILE, min(F_TILE, p.Lk - t * F_TILE), at.gtid); };
    if (!EXACT && at.grp < ntiles) fetch_k(at.grp), fetch_v(at.grp);
#pragma unroll 1
    for (int it = 0; it < iters; it++) {
      const int t = at.grp + G::GROUPS * it, n0 = t * F_TILE;
      f32x16 s = {0.f}, dp = {0.f};   // S^T = K Q^T (log2 domain), dP^T = V dO^T
      G::sync();
      if (t < ntiles) {
        if (EXACT) fetch_k(t), fetch_v(t);
        vr.template put_as<EXACT>(at.stage, G::ONE ? 0 : 1, at.gtid);
        if (!G::ONE) kr.template put_as<EXACT>(at.stage, 0, at.gtid);
      }
      G::sync();
      if (!EXACT && t + G::GROUPS < ntiles) {
        fetch_v(t + G::GROUPS);
        if (!G::ONE) fetch_k(t + G::GROUPS);
      }
      if (t >= ntiles || n0 >= w_end) continue;
      if constexpr (G::ONE) {
        f32x16 more = {0.f};
        if constexpr (EXACT) f32tile::tile_times_frag<D>(at.stage, i, g, do32, dp, more);
        else tile_times_parts<0>(rd, [&](int ks, int n) { return row_frag(drd, PLANE * n, ks); }, dp, more);
        dp += more;
        G::sync();
        kr.template put_as<EXACT>(at.stage, 0, at.gtid);
        G::sync();
        if (!EXACT && t + G::GROUPS < ntiles) fetch_k(t + G::GROUPS);
        more = f32x16{0.f};
        if constexpr (EXACT) f32tile::tile_times_frag<D>(at.stage, i, g, q32, s, more);
        else tile_times_parts<0>(rd, [&](int ks, int n) { return qf[ks][n]; }, s, more);
        s += more;
      } else if constexpr (EXACT) {
        f32tile::tiles_times_frags<D>(at.stage, q32, s, at.stage + F_TILE * (D + 4), do32, dp, i, g);
      } else {
        tiles_times_parts<0, G::SECOND>(rd, [&](int ks, int n) { return qf[ks][n]; }, s, [&](int ks, int n) { return dof[ks][n]; }, dp);
      }
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const float pr = n0 + acc_row(r, g) > lim ? 0.f : ody_exp2(fmaf(s[r], DOWN, -lse2));
        s[r] = pr * fmaf(dp[r], DOWN, -delta) * ds_scale;   // dS^T
      }
      if constexpr (EXACT) f32tile::tile_t_times_regs<D>(at.stage, i, g, s, dq);
      else tile_t_times<0, RW == 4>(rd, s, dq);   // dQ^T += K^T dS^T
    }
  };
  auto publish = [&]() {
    __syncthreads();
    put_flag(smem, !all_finite(dq), at.wave, at.lane);
    if (at.grp > 0) rowtile::give(acc_room<RW, DT>(smem, at.grp, at.w), dq, at.lane);
    __syncthreads();
  };
  walk(std::false_type{});
  publish();
  if (any_flag(smem)) {
    __syncthreads();
    back = 1.f;
    walk(std::true_type{});
    publish();
  }
  if (at.grp != 0) return;
#pragma unroll 1
  for (int n = 1; n < G::GROUPS; n++) rowtile::take(acc_room<RW, DT>(smem, n, at.w), dq, at.lane, 1.f, 1.f);
  if (qi < p.Lq)
    f32tile::store_rows<D>(static_cast<float*>(p.dq) + b * p.sdq.b + h * p.sdq.h + (int64_t)qi * p.sdq.l, dq, g, back, p.accumulate_dq != 0);
}

// ---------------------------------------------------------------------------------------------------------- dK / dV
// The wavefront owns 32 keys; the query tiles of every head of the group are streamed.  The parts of its V rows stay in LDS, and
// those of its K rows too where there is room (in registers, beside both results, 19 to 54 registers spill).
template <int RW>
__global__ __launch_bounds__(64 * WAVES, 2) void attn_bwd_dkdv_f32_parts_kernel(const AttnParams p) {
  using G = Geo<RW>;
  constexpr bool K_IN_LDS = RW != 4;
  constexpr int K_AT = 3 * PLANE * RW;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const Place<RW> at(smem);
  const int g = at.g, i = at.i;
  bf16* vs = reinterpret_cast<bf16*>(smem + G::SMEM);   // [RW][3][32][64], the groups' common V rows
  float* rows = reinterpret_cast<float*>(vs + (K_IN_LDS ? 2 : 1) * RW * PARTS_ELEMS) + at.grp * 2 * F_TILE;   // lse in the log2 domain (+inf: the row contributes nothing), delta
  const BlockCoord bc = ody_block_coord(p.Hkv, p.B);   // with causal masking the first key block is the heaviest
  const int hk = bc.h, b = bc.b;
  const int n0 = bc.rank * G::ROWS, wn0 = n0 + at.w * 32, ki = wn0 + i;
  const float* kp = static_cast<const float*>(p.k) + b * p.sk.b + hk * p.sk.h;
  const float* vp = static_cast<const float*>(p.v) + b * p.sv.b + hk * p.sv.h;

  // first query tile that sees the first key of the block / of the wavefront
  const int i_begin = p.causal ? max(0, n0 - p.off) / F_TILE * F_TILE : 0, w_begin = p.causal ? max(0, wn0 - p.off) : 0;
  // turns over the query tiles of every head of the group
  const int ntq = p.Lq > i_begin ? (p.Lq - i_begin + F_TILE - 1) / F_TILE : 0, turns = ntq * p.group;
  const int iters = (turns + G::GROUPS - 1) / G::GROUPS;
  Readers<D> rd;
  rd.init(reinterpret_cast<bf16*>(at.stage), g, i);

  put_own<RW>(vs, vp, p.sv.l, n0, p.Lk, 1.f, at);
  Readers<D> vrd;   // K's parts lie K_AT rows behind V's
  vrd.init(vs + at.w * PARTS_ELEMS, g, i);
  if constexpr (K_IN_LDS) put_own<RW>(vs + K_AT * D, kp, p.sk.l, n0, p.Lk, p.scale_log2e, at);
  __syncthreads();
  f32x16 dk[DT], dv[DT];
  float back = SPLIT_DOWN;
  auto walk = [&](auto exact) {
    constexpr bool EXACT = decltype(exact)::value;
    constexpr float DOWN = EXACT ? 1.f : SPLIT_DOWN, UP = EXACT ? 1.f : SPLIT_UP;   // of scores and dP; of P, and with it dS
    bf16x8 kf[K_IN_LDS ? 1 : KS][3];
    float k32[EXACT ? D / 2 : 1], v32[EXACT ? D / 2 : 1];
    if constexpr (EXACT) {
      f32tile::load_row_frag<D>(k32, kp, p.sk.l, ki, ki < p.Lk, g, p.scale_log2e);
      f32tile::load_row_frag<D>(v32, vp, p.sv.l, ki, ki < p.Lk, g, 1.f);
    } else if constexpr (!K_IN_LDS) {
      load_parts(kf, kp, p.sk.l, ki, ki < p.Lk, g, p.scale_log2e);
    }
    rowtile::clear(dk);
    rowtile::clear(dv);
    PartTile<G::LOADERS> qr, dor;
    float row = 0.f;   // threads 0 .. 31 of the group carry lse, 32 .. 63 delta of the next tile
    auto fetch_q = [&](int n) {
      const int h = hk * p.group + n / ntq, i0 = i_begin + n % ntq * F_TILE, valid = min(F_TILE, p.Lq - i0);
      qr.template fetch<EXACT, G::ONE>(static_cast<const float*>(p.q) + b * p.sq.b + h * p.sq.h, p.sq.l, i0, valid, at.gtid);
    };
    auto fetch_do = [&](int n) {
      const int h = hk * p.group + n / ntq, i0 = i_begin + n % ntq * F_TILE, valid = min(F_TILE, p.Lq - i0);
      dor.template fetch<EXACT, G::ONE>(static_cast<const float*>(p.dout) + b * p.sdo.b + h * p.sdo.h, p.sdo.l, i0, valid, at.gtid);
      if (at.w == 0) {
        const int64_t r = ((int64_t)b * p.Hq + h) * p.Lq + i0 + min(i, valid - 1);
        const float x = g ? p.delta[r] : p.lse[r];
        row = g ? (i < valid ? x : 0.f) : (i < valid && x != -INFINITY ? (EXACT ? x : in_range(x)) * ODY_LOG2E : INFINITY);
      }
    };
    if (!EXACT && at.grp < turns) fetch_q(at.grp), fetch_do(at.grp);
#pragma unroll 1
    for (int it = 0; it < iters; it++) {
      const int n = at.grp + G::GROUPS * it, i0 = i_begin + n % max(ntq, 1) * F_TILE, next = n + G::GROUPS;
      G::sync();
      if (n < turns) {
        if (EXACT) fetch_q(n), fetch_do(n);
        if (!EXACT && G::ONE) qr.scale(SPLIT_UP);   // once for both times
        qr.template put_as<EXACT, !G::ONE>(at.stage, 0, at.gtid);
        if (!G::ONE) dor.template put_as<EXACT>(at.stage, 1, at.gtid);
        if (at.w == 0) rows[at.lane] = row;
      }
      G::sync();
      if (!EXACT && !G::ONE && next < turns) fetch_q(next), fetch_do(next);
      const bool idle = n >= turns || i0 + F_TILE <= w_begin || wn0 >= p.Lk;
      if (!G::ONE && idle) continue;

      f32x16 s = {0.f}, dp = {0.f};   // S = Q K^T (log2 domain), dP = dO V^T: rows = queries, column = this lane's key
      const int vis = p.causal ? ki - p.off - i0 : -1;   // tile row r is masked iff r < vis
      auto exponentials = [&]() {
#pragma unroll
        for (int a = 0; a < 4; a++) {
          const f32x4 lv = *reinterpret_cast<const f32x4*>(rows + 8 * a + 4 * g);
#pragma unroll
          for (int e = 0; e < 4; e++) s[4 * a + e] = acc_row(4 * a + e, g) < vis ? 0.f : ody_exp2(fmaf(s[4 * a + e], DOWN, -lv[e])) * UP;
        }
      };
      auto gradients = [&]() {   // dS
#pragma unroll
        for (int a = 0; a < 4; a++) {
          const f32x4 dl = *reinterpret_cast<const f32x4*>(rows + F_TILE + 8 * a + 4 * g);
#pragma unroll
          for (int e = 0; e < 4; e++) dp[4 * a + e] = s[4 * a + e] * fmaf(dp[4 * a + e], DOWN, -dl[e]) * p.scale;
        }
      };
      if constexpr (G::ONE) {   // Q, dO, and Q again through the one stage
        if (n >= turns) break;
        f32x16 more = {0.f};
        if constexpr (EXACT) f32tile::tile_times_frag<D>(at.stage, i, g, k32, s, more);
        else tile_times_parts<0>(rd, [&](int ks, int m) { return row_frag(vrd, K_AT + PLANE * m, ks); }, s, more);
        s += more;
        exponentials();
        G::sync();
        dor.template put_as<EXACT>(at.stage, 0, at.gtid);
        G::sync();
        more = f32x16{0.f};
        if constexpr (EXACT) f32tile::tile_times_frag<D>(at.stage, i, g, v32, dp, more);
        else tile_times_parts<0>(rd, [&](int ks, int m) { return row_frag(vrd, PLANE * m, ks); }, dp, more);
        dp += more;
        gradients();
        if (!EXACT && next < turns) fetch_do(next);
        if constexpr (EXACT) f32tile::tile_t_times_regs<D>(at.stage, i, g, s, dv);
        else tile_t_times<0, false>(rd, s, dv);
        G::sync();
        qr.template put_as<EXACT, false>(at.stage, 0, at.gtid);
        G::sync();
        if (!EXACT && next < turns) fetch_q(next);
        if constexpr (EXACT) f32tile::tile_t_times_regs<D>(at.stage, i, g, dp, dk);
        else tile_t_times<0, false>(rd, dp, dk);
      } else {
        if constexpr (EXACT) f32tile::tiles_times_frags<D>(at.stage, k32, s, at.stage + F_TILE * (D + 4), v32, dp, i, g);
        else tiles_times_parts<0, G::SECOND>(rd, [&](int ks, int m) { return K_IN_LDS ? row_frag(vrd, K_AT + PLANE * m, ks) : kf[K_IN_LDS ? 0 : ks][m]; }, s, [&](int ks, int m) { return row_frag(vrd, PLANE * m, ks); }, dp);
        exponentials();
        gradients();
        if constexpr (EXACT) {
          f32tile::tile_t_times_regs<D>(at.stage + F_TILE * (D + 4), i, g, s, dv);
          f32tile::tile_t_times_regs<D>(at.stage, i, g, dp, dk);
        } else {
          tile_t_times<G::SECOND, true>(rd, s, dv);   // dV^T += dO^T P
          tile_t_times<0, true>(rd, dp, dk);          // dK^T += Q^T dS
        }
      }
    }
  };
  auto publish = [&]() {
    __syncthreads();
    put_flag(smem, !all_finite(dk) || !all_finite(dv), at.wave, at.lane);
    if (at.grp > 0) {
      float* room = acc_room<RW, 2 * DT>(smem, at.grp, at.w);
      rowtile::give(room, dk, at.lane);
      rowtile::give(room + 16 * DT * 64, dv, at.lane);
    }
    __syncthreads();
  };
  walk(std::false_type{});
  publish();
  if (any_flag(smem)) {   // (it does not read the own rows in LDS, which the accumulators went over)
    __syncthreads();
    back = 1.f;
    walk(std::true_type{});
    publish();
  }
  if (at.grp != 0) return;
#pragma unroll 1
  for (int n = 1; n < G::GROUPS; n++) {
    const float* room = acc_room<RW, 2 * DT>(smem, n, at.w);
    rowtile::take(room, dk, at.lane, 1.f, 1.f);
    rowtile::take(room + 16 * DT * 64, dv, at.lane, 1.f, 1.f);
  }
  if (ki >= p.Lk) return;
  f32tile::store_rows<D>(static_cast<float*>(p.dk) + b * p.sdk.b + hk * p.sdk.h + (int64_t)ki * p.sdk.l, dk, g, back, false);
  f32tile::store_rows<D>(static_cast<float*>(p.dv) + b * p.sdv.b + hk * p.sdv.h + (int64_t)ki * p.sdv.l, dv, g, back, false);
}

template <int RW>
constexpr size_t dkdv_more() { return (RW == 4 ? 1 : 2) * Geo<RW>::OWN + Geo<RW>::GROUPS * 2 * F_TILE * sizeof(float); }

template <int RW, typename K>
int launch(const char* name, K kern, int rows, int heads, size_t more, const AttnParams& p, hipStream_t st) {
  using G = Geo<RW>;
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), G::SMEM + more, name)) return rc;
  ODY_LAUNCH(name, st, kern, dim3((unsigned)(((int64_t)rows + G::ROWS - 1) / G::ROWS * heads)), dim3(64 * WAVES), G::SMEM + more, p);
  return ody_check_launch(name);
}

// Rows of a block, by the time that the candidates take: us = a * turns + b, where a unit has one block at a time and a block is its
// turns (the groups' longest share of the tiles) and `start` of them for its beginning and end.  Blocks of equal length come in rounds of 256; behind a causal mask,
// longest first, the last ones even the units out to a fifth of the longest.  Fitted to 220 shapes of 64 to 8192 rows, 2 to 128 heads, timed with all
// three: 0.2 to 0.7 % off the best of them in the mean.  us for 32 / 64 / 128 rows, 2 x 16 heads, L = 4096 (1024 blocks of 128), causal: forward 346 / 292 /
// 246, dK and dV 571 / 453 / 413; 8 heads, L = 2048: 55 / 65 / 95, 88 / 100 / 157; 4 x 16 heads, L = 484: 44 / 30 / 32, 65 / 45 / 51.
struct Cost { double start, a, b; };
int rows_of_block(const AttnParams& p, bool own_keys, const Cost (&cost)[3]) {
  const double group = own_keys ? p.group : 1;
  double pairs = (double)p.Lq * p.Lk, longest = own_keys ? p.Lq : p.Lk;
  if (p.causal) {   // a query sees keys up to its own position + off
    pairs = p.off >= 0 ? (double)p.Lq * (p.off + 0.5 * p.Lq) : 0.5 * p.Lk * p.Lk;
    if (own_keys) longest = std::min(p.Lq, p.Lk);
  }
  const int own = own_keys ? p.Lk : p.Lq, heads = p.B * (own_keys ? p.Hkv : p.Hq);
  double best_us = 1e30;
  int best = 32;
  for (int n = 0; n < 3; n++) {
    const int rw = 1 << n, groups = WAVES / rw;
    const double blocks = (double)((own + 32 * rw - 1) / (32 * rw)) * heads;
    const double rows = std::min(longest, pairs / own + (p.causal ? 16.0 * rw : 0.0));   // streamed rows of a block in the mean, of one head
    const double most = std::ceil(std::ceil(longest * group / F_TILE) / groups), mean = std::min(most, rows * group / F_TILE / groups + 0.5);
    const Cost& c = cost[n];
    double turns = most + c.start;
    if (rows >= 0.95 * longest) turns *= std::ceil(blocks / 256);
    else if (blocks > 256) turns = std::max(turns, blocks / 256 * (mean + c.start) + 0.2 * turns);
    if (c.a * turns + c.b < best_us) best_us = c.a * turns + c.b, best = 32 * rw;
  }
  return best;
}

}  // namespace

int ody_launch_attn_fwd_f32_parts(const AttnParams& p, hipStream_t st) {
  static const Cost cost[3] = {{1, 3.95, 3.2}, {1.5, 3.32, 3.3}, {3, 2.73, -1.1}};
  const int rows = rows_of_block(p, false, cost);
  if (rows == 32) return launch<1>("attn_fwd_f32_parts32", &attn_fwd_f32_parts_kernel<1>, p.Lq, p.Hq * p.B, 0, p, st);
  if (rows == 64) return launch<2>("attn_fwd_f32_parts64", &attn_fwd_f32_parts_kernel<2>, p.Lq, p.Hq * p.B, 0, p, st);
  return launch<4>("attn_fwd_f32_parts128", &attn_fwd_f32_parts_kernel<4>, p.Lq, p.Hq * p.B, 0, p, st);
}
int ody_launch_attn_bwd_dq_f32_parts(const AttnParams& p, hipStream_t st) {
  static const Cost cost[3] = {{1, 4.78, 2.4}, {1.5, 4.2, 2.5}, {3, 3.61, -3.2}};
  const int rows = rows_of_block(p, false, cost);
  if (rows == 32) return launch<1>("attn_bwd_dq_f32_parts32", &attn_bwd_dq_f32_parts_kernel<1>, p.Lq, p.Hq * p.B, Geo<1>::OWN, p, st);
  if (rows == 64) return launch<2>("attn_bwd_dq_f32_parts64", &attn_bwd_dq_f32_parts_kernel<2>, p.Lq, p.Hq * p.B, 0, p, st);
  return launch<4>("attn_bwd_dq_f32_parts128", &attn_bwd_dq_f32_parts_kernel<4>, p.Lq, p.Hq * p.B, 0, p, st);
}
int ody_launch_attn_bwd_dkdv_f32_parts(const AttnParams& p, hipStream_t st) {
  static const Cost cost[3] = {{1, 6.34, 1.4}, {2, 5.06, -0.6}, {4, 4.58, -9.1}};
  const int rows = rows_of_block(p, true, cost);
  if (rows == 32) return launch<1>("attn_bwd_dkdv_f32_parts32", &attn_bwd_dkdv_f32_parts_kernel<1>, p.Lk, p.Hkv * p.B, dkdv_more<1>(), p, st);
  if (rows == 64) return launch<2>("attn_bwd_dkdv_f32_parts64", &attn_bwd_dkdv_f32_parts_kernel<2>, p.Lk, p.Hkv * p.B, dkdv_more<2>(), p, st);
  return launch<4>("attn_bwd_dkdv_f32_parts128", &attn_bwd_dkdv_f32_parts_kernel<4>, p.Lk, p.Hkv * p.B, dkdv_more<4>(), p, st);
}
