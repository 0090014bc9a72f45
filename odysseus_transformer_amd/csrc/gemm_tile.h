// The bf16 tile kernel of the dense products (gemm_nt.hip, gemm_nn.hip, gemm_tn.hip instantiate it per operand orientation).
//
// C (M, N) = op(A) . op(B), computed as C^T = op(B)^T . op(A)^T so that a lane ends up with 4 consecutive n of one row.
//
// A block of 8 wavefronts owns BM x BN results and walks K in slabs of 64; two wavefronts share each SIMD.  They form two
// groups (upper and lower half of the rows) that run in anti-phase: while one group multiplies a slab from registers, the
// other reads its fragments of the next one from LDS and issues the global loads of later ones, and a barrier swaps the roles.
// The matrix pipe then always has a wavefront that does nothing but MFMAs.  Operands travel from global memory straight to
// LDS (buffer loads with the LDS bit): no staging registers, no LDS writes, and the loads have a whole slab to land.
//
//   A: two stages; each group loads and reads its own half of the rows, so a stage is free as soon as the group is done with it.
//   B: three stages, loaded by all wavefronts and read by both groups.
//
// LDS layout of an operand tile of W rows (or columns) x 64 k, by its layout in memory:
//   contiguous along K:  [W][64], the eight 16-byte chunks of a row permuted (chunk kc of row r at position kc ^ (r & 7)), read
//                        with 16-byte reads;
//   contiguous along W:  [64][W], the 32-byte column groups of a k row permuted (group x of row k at x ^ g(k)), read with the
//                        transposing read.
// Both are conflict-free for the 16-row fragments of v_mfma_f32_16x16x32_bf16 and are produced by permuting the SOURCE chunk
// of each lane, as a direct load writes its 64 lanes to consecutive LDS addresses.
//
// Rows and columns past the edge re-read the last valid ones and are not stored.  A last slab that K does not fill reads zeros:
// those lanes get an offset beyond the buffer descriptor's range.
//
// A phase is 64 MFMAs, 1024 cycles, and a wavefront issues a transposing read every 17 cycles at best (a 16-byte read of twice the bytes every 20).  The 48 of a
// slab of the TN product, with their addresses and eight loads, made its memory phase the longer one: 1300 to 1500 cycles.  So its group reads the
// fragments of A for the second k-step under the products of the first (each an eighth of the phase ahead of its use; A's stage belongs to the
// group, whereas a stage of B may be refilled by the other group meanwhile), and addresses move by scalars.  TN, TFLOP/s before / here in loops, random
// operands: 22016 x 4096 x 4096 1270 / 1500, 4096 x 11008 x 4096 1270 / 1460, 32000 x 4096 x 4096 1295 / 1500, 4096 x 4096 x 16384 1415 / 1545, 8192^3 1365 /
// 1565, 22016 x 4096 x 1000 1110 / 1250; 1024 x 2816 x 776 11.8 / 9.1 us.  Other numbers of fragments ahead (2, 4, 6, 7 for 8) are 1 to 4 % slower, 1 is 10
// to 20 %.  NN, whose B is read alike, 1.02 to 1.06 of the speed before (to 1.10 where K is short) by the addresses alone.
//
// Bound: the package power limit.  With constant operands the NT instance sustains 2170 TFLOP/s (4096 x 4096 x 11008, 87 % of
// the matrix peak), with random ones 1500; TN 1880 (4096 x 11008 x 4096).  Measured against the kernel it replaced (4 wavefronts, operands staged through
// registers), TFLOP/s in loops of 30 calls and more, 8192^3 / 4096 x 4096 x 11008: NT 1305 -> 1450 / 1347 -> 1520, NN 1283 ->
// 1443 / 1343 -> 1500 (another box: 1565 / 1545, 1506 / 1500; torch.matmul there, NT,
// 1614 / 1600).  A call between two events of its own shows the launch and the clock's way up as well: the second NT product
// 1320 right after idling (torch.matmul 1300 to 1550), 1480 once the card has worked for a second (1470).
#pragma once
#include <type_traits>
#include <utility>
#include "gemm_epi.h"

namespace gemm_tile {

constexpr int BK = 64, THREADS = 512;
constexpr int A_STAGES = 2, B_STAGES = 3;

struct Args {
  const bf16* A;
  const bf16* B;
  bf16* C;
  const bf16* bias;   // EPI_NONE only, may be NULL
  const bf16* add;    // EPI_NONE only, may be NULL: C = add + A B (+ bias), added before the one rounding
  float* part;        // fp32 partial tiles of a call that cuts K, [splits][M][N]
  int M, N, K;
  int64_t lda, ldb, ldc, ld_add;
  int tiles_m, tiles_n;
  int cut, cut_parts; // the last `cut` tiles of the walk are worked on as 2 half or 4 quarter tiles each (256 x 256, K in one range)
  int vec16;          // C (and add) have 16-byte aligned rows
  GemmEpi ep;
};

typedef __attribute__((address_space(3))) void* lds_ptr;
#define ODY_FENCE() __builtin_amdgcn_sched_barrier(0)

constexpr unsigned PAST_END = 0x80000000u;   // beyond every descriptor's range: reads as zero

// column group permutation of a [64][W] tile: the 8 k rows that half a wavefront's transposing read touches (8 q + t, q < 2,
// t < 4) must fall on different 32-byte groups of the 256 bytes that the banks span
template <int W> __device__ __forceinline__ int group_perm(int k) {
  if (W >= 128) return (k & 3) | (((k >> 3) & 1) << 2);
  return ((k >> 1) & 1) | (((k >> 3) & 1) << 1);   // W = 64: two k rows per 256 bytes
}

// The lane, to the compiler a new value each time: what follows from it inside a loop is formed there and takes no registers in between
__device__ __forceinline__ int lane_anew() {
  int x;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(x));
  return x;
}

// One operand's share of the direct loads: W rows (columns) x 64 k per stage, brought by NW wavefronts.  `aim` sets it to a tile; `load` brings
// slab s of K, behind slab s - 1 (KC: any).
//
// Not KC: what changes from slab to slab is scalar, the slab's address; chunks that K does not reach are sorted out behind a branch (`cut`, in front of
// the load of a slab that K fills in part), and not in every load, because the transposing reads leave the memory phase no room.  A slab behind K's end has a
// range of no bytes instead: with `cut` there too, products of one slab, most of whose loads are such, took 1 to 4 % longer than with a mask in every load (TN, us, mask /
// `cut` / range: 32000 x 2048 x 64 35.2 / 36.4 / 35.0, x 24 35.7 / 36.7 / 35.1, 4096 x 4096 x 24 9.9 / 10.1 / 9.8; 1024 x 2816 x 128 5.16 / 4.98 / 4.69; K = 4096 the same).
// KC: slab address and mask anew in every load.  The other form is 1 to 2.5 % slower there (NT, us, this / other: 8192^3 683 / 702, zeros 476 / 487;
// 4096 x 11008 x 4096, zeros, 184 / 188), although it takes fewer instructions.
template <bool KC, int W, int NW>
struct Mover {
  static constexpr int NINS = W / 8 / NW;           // 1 KB instructions per wavefront and stage
  static constexpr int LPR = KC ? 8 : W / 8;        // lanes (16-byte chunks) per tile row
  static constexpr int RPI = 64 / LPR;              // tile rows per instruction
  unsigned v[NINS];                                  // byte offsets of this lane's chunks from the slab's base
  const bf16* base;                                  // first element of the tile's slab 0, or, not KC, of the slab to be loaded next
  int left;                                          // k values from there on

  // row_of(r): operand row of tile row r (KC), or first column of the tile's columns r .. r + 7 (else), clamped to the matrix
  template <typename F>
  __device__ __forceinline__ void aim(int wv, int lane, int64_t ld, const bf16* first, int s, int K, F row_of) {
    base = KC ? first : first + s * (BK * ld), left = KC ? K : K - s * BK;
#pragma unroll
    for (int j = 0; j < NINS; j++) {
      const int r = (wv * NINS + j) * RPI + lane / LPR, p = lane % LPR;
      if (KC) v[j] = (unsigned)(2 * ((int64_t)row_of(r) * ld + 8 * (p ^ (r & 7))));
      else v[j] = (unsigned)(2 * ((int64_t)r * ld + row_of(8 * (p ^ (2 * group_perm<W>(r))))));
    }
  }
  __device__ __forceinline__ bool partial() const { return !KC && (unsigned)(left - 1) < BK - 1; }   // 0 < left < BK
  __device__ __forceinline__ void cut(int wv) {
    if (!partial()) return;
    const int k = wv * NINS * RPI + lane_anew() / LPR;
#pragma unroll
    for (int j = 0; j < NINS; j++)
      if (k + j * RPI >= left) v[j] = PAST_END;
  }
  __device__ __forceinline__ void load(int s, bf16* stage, int wv, int lane, int64_t ld) {
    const bf16* slab = KC ? base + (int64_t)s * BK : base;
    auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(slab), (short)0, KC || left > 0 ? 0x7fffffff : 0, 0x00020000);
#pragma unroll
    for (int j = 0; j < NINS; j++) {
      const unsigned off = !KC || 8 * ((lane & 7) ^ (lane >> 3)) < left - s * BK ? v[j] : PAST_END;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr)(stage + (wv * NINS + j) * 512), 16, (int)off, 0, 0, 0);
    }
    if (!KC) base += BK * ld, left -= BK;
  }
};

// The fragments of NB 16-row blocks of an operand for both k-steps of a slab: lane 16 q + c holds row c, k = 32 ks + 8 q .. + 7.
// Transposing reads are inline assembly: the compiler takes the intrinsic for a possible alias of the direct loads in flight and
// waits for all of them in front of it.  wait() below is what makes their results safe to use.
template <bool KC, int NB>
struct Frags {
  bf16x8 f[2][NB];
};
template <int NB>
struct Frags<false, NB> {
  s16x4 lo[2][NB], hi[2][NB];
};

template <int NB>
__device__ __forceinline__ bf16x8 frag(const Frags<true, NB>& f, int ks, int b) { return f.f[ks][b]; }
template <int NB>
__device__ __forceinline__ bf16x8 frag(const Frags<false, NB>& f, int ks, int b) {
  return concat4(__builtin_bit_cast(bf16x4, f.lo[ks][b]), __builtin_bit_cast(bf16x4, f.hi[ks][b]));
}
// ties a fragment to a point behind the wait for it
template <int NB>
__device__ __forceinline__ void tie(Frags<true, NB>&, int, int) {}
template <int NB>
__device__ __forceinline__ void tie(Frags<false, NB>& f, int ks, int b) {
  asm volatile("" : "+v"(f.lo[ks][b]), "+v"(f.hi[ks][b]));
}

template <int... N, typename F>
__device__ __forceinline__ void each(std::integer_sequence<int, N...>, F f) {
  (f(std::integral_constant<int, N>{}), ...);
}

template <int OFF0, int OFF1>
__device__ __forceinline__ void read_tr(unsigned addr, s16x4& lo, s16x4& hi) {
  asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%3\n\tds_read_b64_tr_b16 %1, %2 offset:%4"
               : "=&v"(lo), "=&v"(hi)
               : "v"(addr), "n"(OFF0), "n"(OFF1));
}

// Consecutive block ids go round-robin over the 8 XCDs, each with its own L2: give every XCD a contiguous range of the n positions.
__device__ __forceinline__ int xcd_position(int id, int n) {
  const int x = id & 7, whole = n >> 3, extra = n & 7;
  return x * whole + min(x, extra) + (id >> 3);
}

// First row and column (in tiles) of the tile at a position of the walk: down M in groups of 8 tiles, so that the tiles in flight share
// panels of both operands
struct TileAt { int m, n; };
__device__ __forceinline__ TileAt tile_at(const Args& p, int pos) {
  constexpr int GROUP = 8;
  const int per_group = GROUP * p.tiles_n, first_m = pos / per_group * GROUP, gsz = min(p.tiles_m - first_m, GROUP);
  return TileAt{first_m + (pos % per_group) % gsz, (pos % per_group) / gsz};
}

constexpr int ROUND = 256;   // blocks of a launch whose blocks take several tiles: one per compute unit

// The BM x BN results from row m0 and column n0 on (n0 / BN = tn), this wavefront's share.
//
// ROUNDS: the block goes on to the tiles ROUND ids further, up to `tiles` of them, without a break: the last slabs of a tile load the first ones
// of the next, and a group stores its results in its memory phase, while the other one multiplies.  A wavefront's patch for them is the part
// of the A stage just read that its own loads fill, so that nobody waits for anybody.  K of three slabs and more.
template <bool A_KC, bool B_KC, int BM, int BN, bool SPLITK, int EPI, bool ROUNDS = false>
__device__ __forceinline__ void gemm_tile_block(const Args& p, int m0, int tn, int tiles = 0) {
  constexpr int WM = BM / 32, WN = BN / 64;      // 16-row blocks per wavefront: rows BM / 2, columns BN / 4
  constexpr int HALF = BM / 2, NH = WN / 2;
  constexpr int AHEAD = A_KC ? 2 * WM : WM;       // fragments of A that the memory phase reads, of two k-steps
  static_assert(EPI == EPI_NONE || !SPLITK, "fused epilogues: one pass over K");
  static_assert(!ROUNDS || ((EPI == EPI_NONE || EPI == EPI_SWIGLU_FWD) && !SPLITK && BM == 256 && BN == 256), "several tiles a block: bf16 bands");
  static_assert((EPI != EPI_SWIGLU_FWD && EPI != EPI_ROPE) || (A_KC && B_KC), "these epilogues belong to the NT product");
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  bf16* As = reinterpret_cast<bf16*>(smem);      // [A_STAGES][2 halves][HALF x 64]
  bf16* Bs = As + A_STAGES * BM * BK;            // [B_STAGES][BN x 64]

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, q = lane >> 4;
  const int wm = wave >> 2, wn = wave & 3;
  int n0 = tn * BN;

  // slabs [s0, s0 + nk) of the K range
  const int slabs = (p.K + BK - 1) / BK;
  int s0 = 0, nk = slabs, k_end = p.K;
  if (SPLITK) {
    const int per = (slabs + (int)gridDim.y - 1) / (int)gridDim.y;
    s0 = blockIdx.y * per;
    nk = max(0, min(slabs - s0, per));
    k_end = min(p.K, (s0 + nk) * BK);
  }

  Mover<A_KC, HALF, 4> ma;
  Mover<B_KC, BN, 8> mb;
  int j0 = EPI == EPI_SWIGLU_FWD ? tn * (BN / 2) : 0;   // first column of h
  auto aim_a = [&](int lane) {
    if (A_KC) ma.aim(wn, lane, p.lda, p.A + (int64_t)m0 * p.lda, s0, p.K, [&](int r) { return min(m0 + wm * HALF + r, p.M - 1) - m0; });
    else ma.aim(wn, lane, p.lda, p.A + m0, s0, k_end, [&](int col) { return min(m0 + wm * HALF + col, p.M - 8) - m0; });
  };
  auto aim_b = [&](int lane) {
    if (EPI == EPI_SWIGLU_FWD)
      mb.aim(wave, lane, p.ldb, p.B, s0, p.K, [&](int r) { return min(j0 + (r & (BN / 2 - 1)), p.ep.I - 1) + (r < BN / 2 ? 0 : p.ep.I); });
    else if (B_KC) mb.aim(wave, lane, p.ldb, p.B + (int64_t)n0 * p.ldb, s0, p.K, [&](int r) { return min(n0 + r, p.N - 1) - n0; });
    else mb.aim(wave, lane, p.ldb, p.B + n0, s0, k_end, [&](int col) { return min(n0 + col, p.N - 8) - n0; });
  };
  aim_a(lane);
  aim_b(lane);
  auto cut = [&] {
    ma.cut(wn);
    mb.cut(wave);
  };
  auto load_a = [&](int kt, int stage) { ma.load(s0 + kt, As + stage * BM * BK + wm * HALF * BK, wn, lane, p.lda); };
  auto load_b = [&](int kt, int slot) { mb.load(s0 + kt, Bs + slot * BN * BK, wave, lane, p.ldb); };

  // tile row (column) of this wavefront's n block b
  auto nblock = [&](int b) {
    if (EPI == EPI_SWIGLU_FWD) return (b / NH) * (BN / 2) + wn * 16 * NH + 16 * (b % NH);      // gate blocks, then their up blocks
    if (EPI == EPI_ROPE) {                                                                      // j blocks of a head, then j + 64
      constexpr int WPH = 4 / (BN / 128);
      return (wn / WPH) * 128 + (b / NH) * 64 + (wn % WPH) * 16 * NH + 16 * (b % NH);
    }
    return wn * 16 * WN + 16 * b;
  };
  const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr)smem;
  const int kc_off = c * BK + 8 * (q ^ (c & 7));                                               // + 64 * row block, ^ 32 for ks = 1
  // byte addresses of the transposing reads, without the stage
  unsigned a_tr[A_KC ? 1 : WM], b_tr[B_KC ? 1 : WN];
  if constexpr (!A_KC) {
    const int at = wm * HALF * BK + (8 * q + (c >> 2)) * HALF + 16 * group_perm<HALF>(8 * q + (c >> 2)) + 4 * (c & 3);
#pragma unroll
    for (int a = 0; a < WM; a++) a_tr[a] = lds0 + 2 * (at ^ (16 * a));
  }
  if constexpr (!B_KC) {
    const int at = A_STAGES * BM * BK + (8 * q + (c >> 2)) * BN + 16 * ((wn * WN) ^ group_perm<BN>(8 * q + (c >> 2))) + 4 * (c & 3);
#pragma unroll
    for (int b = 0; b < WN; b++) b_tr[b] = lds0 + 2 * (at ^ (16 * b));
  }

  f32x4 acc[WM][WN];
  auto clear_acc = [&] {
#pragma unroll
    for (int a = 0; a < WM; a++)
#pragma unroll
      for (int b = 0; b < WN; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear_acc();

  auto store16 = [](bf16* dst, bf16x8 w) {
    typedef unsigned raw_t __attribute__((ext_vector_type(4)));
    __builtin_nontemporal_store(__builtin_bit_cast(raw_t, w), reinterpret_cast<raw_t*>(dst));
  };
  auto rounded = [](f32x4 x) {
    bf16x4 w;
#pragma unroll
    for (int e = 0; e < 4; e++) w[e] = (bf16)x[e];
    return w;
  };

  constexpr int COLS = 16 * WN;
  auto biased = [&](f32x4 x, int b) {
    if (EPI == EPI_NONE && !SPLITK && !ROUNDS && p.bias) {
      const bf16x4 bv = *reinterpret_cast<const bf16x4*>(p.bias + min(n0 + wn * COLS + 16 * b + 4 * q, p.N - 4));
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] += (float)bv[e];
    }
    return x;
  };
  // The results of the tile at m0, tn, through a patch of LDS of 16 T rows that belongs to the wavefront
  auto store_bands = [&](int m0, int tn, bf16* band, auto rows) {
    constexpr int T = decltype(rows)::value;
    const int lane = ROUNDS ? lane_anew() : tid & 63, c = lane & 15, q = lane >> 4;
    const int mw = m0 + wm * HALF, n0 = tn * BN, j0 = tn * (BN / 2);
    constexpr int EP = COLS + 8, CPR = COLS / 8, RPP = 64 / CPR;
#pragma unroll
    for (int a2 = 0; a2 < WM / T; a2++) {
      ODY_FENCE();
      wavefront_sync();
      bf16x4 w[T][WN];
#pragma unroll
      for (int t = 0; t < T; t++) {
        const int m = min(mw + 16 * T * a2 + 16 * t + c, p.M - 1);
        if (EPI == EPI_ROPE && n0 + nblock(0) < p.ep.I) {   // this wavefront's head is a query or key head
#pragma unroll
          for (int b = 0; b < NH; b++) {
            const int j = (nblock(b) & 127) + 4 * q;         // (cos, sin) of frequencies j .. j + 3: 16 bytes of the token's table row
            const bf16x8 cs = *reinterpret_cast<const bf16x8*>(p.ep.aux + (int64_t)m * p.ep.ld_aux + 2 * j);
            f32x4 o1, o2;
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const float co = (float)cs[2 * e], sn = (float)cs[2 * e + 1], x1 = acc[T * a2 + t][b][e], x2 = acc[T * a2 + t][b + NH][e];
              o1[e] = x1 * co - x2 * sn;
              o2[e] = x2 * co + x1 * sn;
            }
            w[t][b] = rounded(o1), w[t][b + NH] = rounded(o2);
          }
        } else {
#pragma unroll
          for (int b = 0; b < WN; b++) w[t][b] = rounded(biased(acc[T * a2 + t][b], b));
        }
#pragma unroll
        for (int b = 0; b < WN; b++) *reinterpret_cast<bf16x4*>(band + (16 * t + c) * EP + 16 * b + 4 * q) = w[t][b];
      }
      wavefront_sync();
#pragma unroll
      for (int pass = 0; pass < 16 * T / RPP; pass++) {
        if (EPI == EPI_SWIGLU_FWD && p.C == nullptr) break;   // only h is wanted
        const int row = pass * RPP + lane / CPR, ch = lane % CPR, m = mw + 16 * T * a2 + row;
        const bf16x8 v = *reinterpret_cast<const bf16x8*>(band + row * EP + 8 * ch);
        const int b = ch >> 1;
        if constexpr (EPI == EPI_SWIGLU_FWD) {
          const int j = j0 + wn * 16 * NH + 16 * (b % NH) + 8 * (ch & 1);
          if (m < p.M && j < p.ep.I) store16(p.C + (int64_t)m * p.ldc + (b / NH) * p.ep.I + j, v);
        } else if constexpr (EPI == EPI_SWIGLU_BWD) {
          const int j = n0 + wn * COLS + 8 * ch;
          if (m < p.M && j < p.N) {
            const bf16* gu = p.ep.aux + (int64_t)m * p.ep.ld_aux + j;
            const bf16x8 gt = *reinterpret_cast<const bf16x8*>(gu), up = *reinterpret_cast<const bf16x8*>(gu + p.ep.I);
            bf16x8 d1, d3;
#pragma unroll
            for (int e = 0; e < 8; e++) {
              const float a1 = (float)gt[e], a3 = (float)up[e], gg = (float)v[e];
              const float sig = 1.f / (1.f + __expf(-a1));
              d1[e] = (bf16)(gg * a3 * sig * (1.f + a1 * (1.f - sig)));
              d3[e] = (bf16)(gg * a1 * sig);
            }
            store16(p.C + (int64_t)m * p.ldc + j, d1);
            store16(p.C + (int64_t)m * p.ldc + p.ep.I + j, d3);
          }
        } else {
          const int n = n0 + nblock(b) + 8 * (ch & 1);
          if (m < p.M && n < p.N) store16(p.C + (int64_t)m * p.ldc + n, v);
        }
      }
      if constexpr (EPI == EPI_SWIGLU_FWD) {
        // h from the rounded values: block b of the first half is the gate of block b of the second
        constexpr int EPH = COLS / 2 + 8, CPH = COLS / 16, RPH = 64 / CPH;
        wavefront_sync();
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
          for (int b = 0; b < NH; b++) {
            bf16x4 hv;
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const float a1 = (float)w[t][b][e], a3 = (float)w[t][b + NH][e];
              hv[e] = (bf16)(a1 / (1.f + __expf(-a1)) * a3);
            }
            *reinterpret_cast<bf16x4*>(band + (16 * t + c) * EPH + 16 * b + 4 * q) = hv;
          }
        wavefront_sync();
#pragma unroll
        for (int pass = 0; pass < (16 * T + RPH - 1) / RPH; pass++) {
          const int row = pass * RPH + lane / CPH, ch = lane % CPH, m = mw + 16 * T * a2 + row, j = j0 + wn * 16 * NH + 8 * ch;
          const bf16x8 v = *reinterpret_cast<const bf16x8*>(band + row * EPH + 8 * ch);
          if (m < p.M && j < p.ep.I) store16(p.ep.out2 + (int64_t)m * p.ep.ld_out2 + j, v);
        }
      }
    }
  };

  if (nk > 0) {
    constexpr int NA = Mover<A_KC, HALF, 4>::NINS, NB = Mover<B_KC, BN, 8>::NINS;
    cut();
    load_b(0, 0);
    load_a(0, 0);
    mb.cut(wave);
    load_b(min(1, nk - 1), 1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(ROUNDS ? 0 : NB) : "memory");
    __builtin_amdgcn_s_barrier();
    if (wm == 1) __builtin_amdgcn_s_barrier();   // the second group runs one phase behind
    int slot = 0, stage = 0;
    // one slab, loading slab `na` of A and slab `nb` of B; STORED: behind a tile's stores, which stand behind all loads issued before
    auto slab = [&](int na, int nb, auto stored) {
      constexpr bool STORED = decltype(stored)::value;
      const bf16* At = As + stage * BM * BK + wm * HALF * BK;
      const bf16* Bt = Bs + slot * BN * BK;
      Frags<A_KC, WM> fa;
      Frags<B_KC, WN> fb;
      [[maybe_unused]] auto read_a = [&](int ks, int a) __attribute__((always_inline)) {
        if constexpr (!A_KC) {
          const unsigned at = a_tr[a] + 2 * stage * BM * BK;
          if (ks == 0) read_tr<0, 8 * HALF>(at, fa.lo[0][a], fa.hi[0][a]);
          else read_tr<64 * HALF, 72 * HALF>(at, fa.lo[1][a], fa.hi[1][a]);
        }
      };
      if (ma.partial() || mb.partial()) cut();
      // ---- memory phase: this slab's fragments; A of the next slab, B of the one after (its stage was read last two phases ago)
      ODY_FENCE();
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        if constexpr (B_KC) {
#pragma unroll
          for (int b = 0; b < WN; b++) fb.f[ks][b] = *reinterpret_cast<const bf16x8*>(Bt + (kc_off ^ (32 * ks)) + nblock(b) * BK);
        } else {
#pragma unroll
          for (int b = 0; b < WN; b++) {
            const unsigned at = b_tr[b] + 2 * slot * BN * BK;
            if (ks == 0) read_tr<0, 8 * BN>(at, fb.lo[0][b], fb.hi[0][b]);
            else read_tr<64 * BN, 72 * BN>(at, fb.lo[1][b], fb.hi[1][b]);
          }
        }
        if constexpr (A_KC) {
#pragma unroll
          for (int a = 0; a < WM; a++) fa.f[ks][a] = *reinterpret_cast<const bf16x8*>(At + (kc_off ^ (32 * ks)) + 16 * a * BK);
        } else {
#pragma unroll
          for (int a = 0; a < WM; a++)
            if (ks * WM + a < AHEAD) read_a(ks, a);
        }
        ODY_FENCE();
        if (ks == 0) load_a(na, stage ^ 1);
        else load_b(nb, slot == 0 ? 2 : slot - 1);
        ODY_FENCE();
      }
      // this wavefront's part of B's next slab has landed (the other group may read it two barriers from here)
      if (STORED) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NA + NB) : "memory");
#pragma unroll
      for (int n = 0; n < AHEAD; n++) tie(fa, n / WM, n % WM);
#pragma unroll
      for (int n = 0; n < 2 * WN; n++) tie(fb, n / WN, n % WN);
      __builtin_amdgcn_s_barrier();
      ODY_FENCE();
      // ---- compute phase
      each(std::make_integer_sequence<int, 2 * WM>{}, [&](auto which) __attribute__((always_inline)) {
        constexpr int n = decltype(which)::value, ks = n / WM, a = n % WM, BEHIND = n + AHEAD < 2 * WM ? AHEAD - 1 : 2 * WM - 1 - n;
        if constexpr (n >= AHEAD) {
          asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(2 * BEHIND) : "memory");   // its two reads are back; those of BEHIND fragments may not be
          tie(fa, ks, a);
          ODY_FENCE();
        }
#pragma unroll
        for (int b = 0; b < WN; b++) {
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(fb, ks, b), frag(fa, ks, a), acc[a][b], 0, 0, 0);   // rows = n, columns = m
          if constexpr (n + AHEAD < 2 * WM)
            if (b == 0) {
              ODY_FENCE();
              read_a((n + AHEAD) / WM, (n + AHEAD) % WM);
              ODY_FENCE();
            }
        }
      });
      ODY_FENCE();
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NB) : "memory");   // A of the next slab has landed
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      slot = slot == 2 ? 0 : slot + 1;
      stage ^= 1;
    };
    // loads past the range repeat its last slab (KC) or fetch nothing: in bounds, and nobody reads them
    if constexpr (!ROUNDS) {
      for (int kt = 0; kt < nk; kt++) slab(min(kt + 1, nk - 1), min(kt + 2, nk - 1), std::false_type{});
    } else {
      for (int id = blockIdx.x;; id += ROUND) {
        const TileAt at = tile_at(p, xcd_position(id, tiles));
        const bool more = id + ROUND < tiles;
        slab(1, 2, std::true_type{});
        for (int kt = 1; kt < nk; kt++) {
          int na = kt + 1, nb = kt + 2;
          if (nb >= nk) {   // the last two slabs
            if (!more) {
              na = nb = nk - 1;
            } else if (na < nk) {
              const TileAt next = tile_at(p, xcd_position(id + ROUND, tiles));
              m0 = next.m * BM, n0 = next.n * BN;
              if (EPI == EPI_SWIGLU_FWD) j0 = next.n * (BN / 2);
              aim_b(lane_anew());
              nb = 0;
            } else {
              aim_a(lane_anew());
              na = 0, nb = 1;
            }
          }
          slab(na, nb, std::false_type{});
        }
        constexpr int OWN = Mover<A_KC, HALF, 4>::NINS * 512;
        static_assert(16 * (COLS + 8) <= OWN, "16 rows fit");
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next tile's first slabs, which the stores would stand behind
        store_bands(at.m * BM, at.n, As + (stage ^ 1) * BM * BK + wm * HALF * BK + wn * OWN, std::integral_constant<int, 1>{});
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        ODY_FENCE();
        if (!more) break;
        clear_acc();
      }
    }
    if (wm == 0) __builtin_amdgcn_s_barrier();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  if constexpr (ROUNDS) return;
  __syncthreads();   // the epilogue reuses the operand stages

  // ---- epilogue.  Lane 16 q + c holds row m = c and columns n = 4 q .. 4 q + 3 of each 16 x 16 block; the blocks leave through a
  // patch of LDS that belongs to the wavefront (its LDS operations complete in order), 32 rows at a time, as 16-byte pieces of
  // rows, by streaming stores: this kernel does not read them again.
  const int mw = m0 + wm * HALF;
  if constexpr (SPLITK) {
    constexpr int EP = COLS + 4, CPR = COLS / 4, RPP = 64 / CPR;
    float* band = reinterpret_cast<float*>(smem) + wave * 32 * EP;
    float* dst = p.part + (int64_t)blockIdx.y * p.M * p.N;
#pragma unroll
    for (int a2 = 0; a2 < WM / 2; a2++) {
      ODY_FENCE();
      wavefront_sync();   // the band before has been read
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int b = 0; b < WN; b++) *reinterpret_cast<f32x4*>(band + (16 * t + c) * EP + 16 * b + 4 * q) = acc[2 * a2 + t][b];
      wavefront_sync();
#pragma unroll
      for (int pass = 0; pass < 32 / RPP; pass++) {
        const int row = pass * RPP + lane / CPR, ch = lane % CPR, m = mw + 32 * a2 + row, n = n0 + wn * COLS + 4 * ch;
        const f32x4 v = *reinterpret_cast<const f32x4*>(band + row * EP + 4 * ch);
        if (m < p.M && n < p.N) *reinterpret_cast<f32x4*>(dst + (int64_t)m * p.N + n) = v;
      }
    }
    return;
  }
  if constexpr (EPI == EPI_NONE) {
    if (!p.vec16) {   // rows of C that 16-byte pieces cannot address
#pragma unroll
      for (int a = 0; a < WM; a++) {
        ODY_FENCE();
        int m = mw + 16 * a + c;
        asm volatile("" : "+v"(m));   // addresses are made here, not all at once in front
#pragma unroll
        for (int b = 0; b < WN; b++) {
          const int n = n0 + wn * COLS + 16 * b + 4 * q;
          if (m >= p.M || n >= p.N) continue;
          f32x4 v = biased(acc[a][b], b);
          if (p.add) {
            const bf16x4 o = *reinterpret_cast<const bf16x4*>(p.add + (int64_t)m * p.ld_add + n);
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] += (float)o[e];
          }
          *reinterpret_cast<bf16x4*>(p.C + (int64_t)m * p.ldc + n) = rounded(v);
        }
      }
      return;
    }
    if (p.add) {   // fp32 bands, so that the sum is rounded once
      constexpr int EP = COLS + 4, CPR = COLS / 8, RPP = 64 / CPR;
      float* band = reinterpret_cast<float*>(smem) + wave * 32 * EP;
#pragma unroll
      for (int a2 = 0; a2 < WM / 2; a2++) {
        ODY_FENCE();
        wavefront_sync();
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
          for (int b = 0; b < WN; b++) *reinterpret_cast<f32x4*>(band + (16 * t + c) * EP + 16 * b + 4 * q) = biased(acc[2 * a2 + t][b], b);
        wavefront_sync();
#pragma unroll
        for (int pass = 0; pass < 32 / RPP; pass++) {
          const int row = pass * RPP + lane / CPR, ch = lane % CPR, m = mw + 32 * a2 + row, n = n0 + wn * COLS + 8 * ch;
          const f32x4 v0 = *reinterpret_cast<const f32x4*>(band + row * EP + 8 * ch);
          const f32x4 v1 = *reinterpret_cast<const f32x4*>(band + row * EP + 8 * ch + 4);
          if (m < p.M && n < p.N) {
            const bf16x8 r = *reinterpret_cast<const bf16x8*>(p.add + (int64_t)m * p.ld_add + n);
            bf16x8 w;
#pragma unroll
            for (int e = 0; e < 4; e++) w[e] = (bf16)(v0[e] + (float)r[e]), w[4 + e] = (bf16)(v1[e] + (float)r[4 + e]);
            store16(p.C + (int64_t)m * p.ldc + n, w);
          }
        }
      }
      return;
    }
  }
  store_bands(m0, tn, reinterpret_cast<bf16*>(smem) + wave * 32 * (COLS + 8), std::integral_constant<int, 2>{});
}
#undef ODY_FENCE

// Block -> tile: first the whole tiles, then, PARTS blocks each, those whose halves or quarters fill a last round better (plan_bf16).  (One kernel for both: 0.3 %
// slower where halves are taken.)
template <bool A_KC, bool B_KC, int BM, int BN, bool SPLITK, int EPI, int PARTS, bool ROUNDS>
__global__ __launch_bounds__(THREADS, BM * BN <= 128 * 128 ? 4 : 2) void gemm_tile_kernel(const Args p) {
  const int whole = p.tiles_m * p.tiles_n - p.cut;
  int pos = ROUNDS && blockIdx.x >= ROUND ? blockIdx.x - ROUND + whole : blockIdx.x, part = 0;
  const bool in_part = BM == 256 && !SPLITK && pos >= whole;
  if (in_part) {
    pos = xcd_position(pos - whole, PARTS * p.cut);
    part = pos % PARTS;
    pos = whole + pos / PARTS;
  } else {
    pos = xcd_position(pos, whole);
  }
  const TileAt at = tile_at(p, pos);
  const int m0 = at.m * BM, tn = at.n;
  if constexpr (BM == 256 && !SPLITK) {
    if (in_part) {
      const int mp = m0 + 128 * (part & 1);
      if (mp >= p.M) return;
      if constexpr (PARTS == 2) {
        gemm_tile_block<A_KC, B_KC, 128, BN, SPLITK, EPI>(p, mp, tn);
      } else {
        const int np = 2 * tn + (part >> 1);
        if (np * (EPI == EPI_SWIGLU_FWD ? BN / 4 : BN / 2) < (EPI == EPI_SWIGLU_FWD ? p.ep.I : p.N))
          gemm_tile_block<A_KC, B_KC, 128, BN / 2, SPLITK, EPI>(p, mp, np);
      }
      return;
    }
  }
  gemm_tile_block<A_KC, B_KC, BM, BN, SPLITK, EPI, ROUNDS>(p, m0, tn, whole);
}

// Whether the blocks take several tiles each (a grid of ROUND blocks): where there are two rounds and more.  A block of one tile waits about
// 4 us for its first slabs and its stores, which nothing hides with one block on a unit; here the matrix cores go on meanwhile.  The same
// sums in the same order.  us before / here: 32768 x 4096 x 512 NT 139 / 118, NN 141 / 121, TN 155 / 136; 4096 x 11008 x 1000 82 / 77, 81 / 76,
// 87 / 82; 22016 x 4096 x 4096 NT 483 / 476, NN 506 / 494, TN 514 / 490; 8192^3 679 / 673, 705 / 692, 714 / 696; 32000 x 4096 x 4096 TN 739 / 716.
// Of the epilogues, SwiGLU's forward gains: gate_up of 16384 tokens (d 4096, I 11008) 2137 / 2086, of 8192 (1024, 5504) 187 / 178.  Those that
// read memory wait in it for the stores before (loads and stores come back in order): the rotation 0.96 to 1.00 of the speed before,
// SwiGLU's backward 0.82 to 0.97, so they keep one tile a block; an addend's fp32 patch is larger than the room there is.
inline bool takes_rounds(const Args& a) { return a.tiles_m * a.tiles_n - a.cut >= 2 * ROUND && a.K > 2 * BK && a.vec16 && !a.bias && !a.add; }

template <bool A_KC, bool B_KC, int BM, int BN, bool SPLITK, int EPI, int PARTS, bool ROUNDS>
int launch_parts(const char* name, const Args& a, int splits, hipStream_t st) {
  constexpr size_t smem = sizeof(bf16) * BK * (A_STAGES * BM + B_STAGES * BN);
  static_assert(smem >= 8 * 32 * (BN / 4 + 4) * sizeof(float), "the fp32 bands fit in the operand stages");
  auto kern = &gemm_tile_kernel<A_KC, B_KC, BM, BN, SPLITK, EPI, PARTS, ROUNDS>;
  if (int rc = ody_allow_dynamic_lds(reinterpret_cast<const void*>(kern), smem, name)) return rc;
  const int whole = a.tiles_m * a.tiles_n - a.cut;
  ODY_LAUNCH(name, st, kern, dim3((ROUNDS ? ROUND : whole) + PARTS * a.cut, splits), dim3(THREADS), smem, a);
  return ody_check_launch(name);
}
template <bool A_KC, bool B_KC, int BM, int BN, bool SPLITK, int EPI>
int launch(const char* name, Args a, int splits, hipStream_t st) {
  a.tiles_m = (a.M + BM - 1) / BM, a.tiles_n = (a.N + BN - 1) / BN;
  if (EPI == EPI_SWIGLU_FWD) a.tiles_n = (a.ep.I + BN / 2 - 1) / (BN / 2);
  if constexpr (BM == 256 && !SPLITK) {
    if constexpr ((EPI == EPI_NONE || EPI == EPI_SWIGLU_FWD) && BN == 256)
      if (takes_rounds(a)) {
        if (a.cut_parts == 4) return launch_parts<A_KC, B_KC, BM, BN, SPLITK, EPI, 4, true>(name, a, splits, st);
        return launch_parts<A_KC, B_KC, BM, BN, SPLITK, EPI, 2, true>(name, a, splits, st);
      }
    if (a.cut_parts == 4) return launch_parts<A_KC, B_KC, BM, BN, SPLITK, EPI, 4, false>(name, a, splits, st);
  }
  return launch_parts<A_KC, B_KC, BM, BN, SPLITK, EPI, 2, false>(name, a, splits, st);
}

}  // namespace gemm_tile

// one per orientation: tile BM x BN, K cut into `splits` ranges (EPI_NONE only, partials to a.part)
int ody_launch_gemm_nt(int epi, int BM, int BN, int splits, const gemm_tile::Args& a, hipStream_t st);
int ody_launch_gemm_nn(int epi, int BM, int BN, int splits, const gemm_tile::Args& a, hipStream_t st);
int ody_launch_gemm_tn(int BM, int BN, int splits, const gemm_tile::Args& a, hipStream_t st);
