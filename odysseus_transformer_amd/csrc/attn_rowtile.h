// Row tiles of the attention kernels that read both kinds of operand from one tile (attn_hd64.hip, attn_short.hip): 64 rows of D
// elements in LDS, filled by direct loads, read in rows with 16-byte reads and, where a product contracts over the row index, with the
// transposing read.  No images, so no pass over the operands before the kernel.
//
// QUADS: the rows of an operand are taken in the order of attn_tile.h (row 4 (i & 15) + (i >> 4) + 2 kt of the tile for row i of sub-tile kt),
// for a kernel whose sums must come out like those of the kernels over images, bit for bit.
//
// A row is D / 8 chunks of 16 bytes; chunk c of row r sits at position c ^ swz(r).  The permutation is applied to the source chunk of
// each lane, as a direct load writes its lanes to consecutive addresses.  Conflict-free for both kinds of read:
//   D = 64   swz(r) = bits 3, 2, 1 of r in bits 0, 1, 2.  The 16 rows that a 16-byte read serves together (attn_tile.h) have pairwise
//            different (r & 1, swz), and of the four rows of a transposing read those two that share a 128-byte half differ in bit 2 of
//            swz.
//   D = 128  swz(r) = bits 1, 0 of r in bits 3, 2 and bits 3, 2 in bits 1, 0.  The 16 rows have 16 different swz, and the four rows of a
//            transposing read lie in the four 64-byte quarters of a row.  With QUADS the same of r >> 2: the 16 rows are 4 apart.
#pragma once
#include "attn_params.h"
#include "attn_tile.h"

namespace rowtile {

constexpr int ROWS = 64;   // of a tile
typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __attribute__((address_space(1))) const void* global_ptr;

// Blocks heaviest first, all (head, batch) pairs of a rank together (ody_block_coord), and under a causal mask every other run
// of 256 blocks with its ranks reversed: the three or four blocks that share a compute unit then add up to about the same
// length.  In plain order the units with the first blocks of every run got 320 tiles where the mean was 260 (forward of 16 heads,
// L = 8192: 182 us, 158 this way).
// RUNS: so many runs of 256 are on the units from the start, and only among them ranks are reversed; what follows goes to whichever unit is done first,
// longest first (0: all may share a unit).
template <int RUNS = 0>
__device__ __forceinline__ BlockCoord block_coord(int H, int B, int causal) {
  BlockCoord c = ody_block_coord(H, B);
  const int ranks = gridDim.x / (H * B), run = max(1, 256 / (H * B)), n = c.rank / run;
  if (causal && (n & 1) && (RUNS == 0 || n < RUNS) && (n + 1) * run <= ranks) c.rank = n * run + run - 1 - c.rank % run;
  return c;
}

template <int D>
__device__ __forceinline__ int swz(int r) {
  if constexpr (D == 64) return ((r & 2) << 1) | ((r & 4) >> 1) | ((r & 8) >> 3);
  else return ((r & 3) << 2) | ((r >> 2) & 3);
}

// Fragment reads go by LDS byte addresses: what depends on the lane and the stage sits in D / 8 registers that move from stage to
// stage, the rest is in the offset field of the instruction.
template <int D, bool QUADS = false>
struct Readers {
  static_assert(D == 128 || !QUADS, "attn_tile.h is for head_dim 128");
  static constexpr int KS = D / 16, NT = D / 16;
  unsigned row[KS], tr[NT];
  __device__ __forceinline__ void init(const bf16* stage, int g, int i) {
    const unsigned a = (unsigned)(uintptr_t)(lds_ptr)const_cast<bf16*>(stage);
    const int rb = (QUADS ? 4 * (i & 15) + (i >> 4) : i) * D + 8 * (g ^ swz<D>(i));
#pragma unroll
    for (int ks = 0; ks < KS; ks++) row[ks] = a + 2 * (rb ^ (16 * ks));
    // tr[2 dt + n], without the distance of n = 1: rows 8 n + 4 g + t (QUADS: 32 n + 16 g + 4 t), columns 32 dt + 16 (i >> 4) + 4 (i & 3) .. + 3
    const int t = (i & 15) >> 2, c = 2 * (i >> 4) + ((i & 3) >> 1);
    const int tb = (QUADS ? 4 : 1) * (4 * g + t) * D + 8 * (c ^ swz<D>(4 * g + t)) + 4 * (i & 1);
#pragma unroll
    for (int n = 0; n < NT; n++) tr[n] = a + 2 * (tb ^ (8 * ((4 * (n >> 1)) ^ swz<D>(8 * (n & 1)))));
  }
  __device__ __forceinline__ void move(int bytes) {
#pragma unroll
    for (int n = 0; n < KS; n++) row[n] += bytes, tr[n] += bytes;
  }
};
// A operand, rows first .. first + 31 behind the stage's start (QUADS: first = the tile's + 2 kt): lane (g, i) holds row i, k = 16 ks + 8 g .. + 7
template <int D, bool QUADS>
__device__ __forceinline__ bf16x8 row_frag(const Readers<D, QUADS>& r, int first, int ks) {
  typedef const bf16x8 __attribute__((address_space(3))) * frag_ptr;
  return *(frag_ptr)(uintptr_t)(r.row[ks] + 2 * first * D);
}
// A operands of the transposed tile, 16 rows from FIRST on, columns 64 HALF .. 64 HALF + 63: lane (g, i) of f[dt] holds column
// 64 HALF + 32 dt + i, and k element e is row FIRST + 8 (e >> 2) + 4 g + (e & 3) (QUADS: FIRST + 32 (e >> 2) + 16 g + 4 (e & 3)) -- the order in which accumulators hold their rows, so
// that P and dS go from accumulator to B operand in place.  The reads and the wait for them are one piece of assembly: behind the
// intrinsic the compiler waits for every direct load in flight, as for possible writers of what is read here.
template <int FIRST, int HALF, int D, bool QUADS>
__device__ __forceinline__ void tr_frags(bf16x8 (&f)[2], const Readers<D, QUADS>& r) {
  s16x4 x0, x1, y0, y1;
  asm volatile("ds_read_b64_tr_b16 %0, %4 offset:%8\n\tds_read_b64_tr_b16 %1, %5 offset:%9\n\t"
               "ds_read_b64_tr_b16 %2, %6 offset:%8\n\tds_read_b64_tr_b16 %3, %7 offset:%9\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(x0), "=&v"(x1), "=&v"(y0), "=&v"(y1)
               : "v"(r.tr[4 * HALF]), "v"(r.tr[4 * HALF + 1]), "v"(r.tr[4 * HALF + 2]), "v"(r.tr[4 * HALF + 3]), "n"(2 * FIRST * D),
                 "n"(2 * (FIRST + (QUADS ? 32 : 8)) * D)
               : "memory");
  f[0] = concat4(__builtin_bit_cast(bf16x4, x0), __builtin_bit_cast(bf16x4, x1));
  f[1] = concat4(__builtin_bit_cast(bf16x4, y0), __builtin_bit_cast(bf16x4, y1));
}
// row of accumulator register r
__device__ __forceinline__ int acc_row(int r, int g) { return 8 * (r >> 2) + 4 * g + (r & 3); }

// Direct loads of 64-row tiles of one matrix by WAVES wavefronts: an instruction brings 512 / D rows.  Rows at or beyond nrows
// re-read the last one (finite filler that the caller masks); tiles start below nrows.
template <int D, int WAVES, bool QUADS = false>
struct TileLoader {
  static constexpr int LANES = D / 8, PER = 64 / LANES, STEP = PER * WAVES, STEPS = ROWS / STEP;
  static_assert(QUADS ? STEP == 32 : STEP % 16 == 0, "swz of the rows of the other steps");
  int64_t off, stride;   // of this lane's row in the first instruction; row stride
  int row, col;
  __device__ __forceinline__ void init(int64_t s, int w, int lane) {
    row = PER * w + lane / LANES;
    col = 8 * ((lane % LANES) ^ swz<D>(QUADS ? row >> 2 : row));   // swz looks at its argument modulo 16
    off = (int64_t)row * s + (QUADS ? 0 : col);
    stride = s;
  }
  // base: the matrix of this (batch, head), uniform
  __device__ __forceinline__ void load(bf16* tile, const bf16* base, int row0, int nrows, int w) const {
#pragma unroll
    for (int j = 0; j < STEPS; j++) {
      const bf16* src = base + (int64_t)(row0 + STEP * j) * stride + off + (QUADS ? col ^ (8 * swz<D>(STEP * j >> 2)) : 0);
      if (row0 + ROWS > nrows) src += (int64_t)min(nrows - 1 - row0 - STEP * j - row, 0) * stride;
      __builtin_amdgcn_global_load_lds((global_ptr)src, (lds_ptr)(tile + (WAVES * j + w) * 512), 16, 0, 0);
    }
  }
};

// The 32 rows of a wavefront as B operands: lane (g, i) holds row `row`, k = 16 ks + 8 g .. + 7; zero beyond nrows
template <int KS>
__device__ __forceinline__ void load_rows(bf16x8 (&f)[KS], const bf16* base, int64_t stride, int row, int nrows, int g) {
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    f[ks] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
    if (row < nrows) f[ks] = *reinterpret_cast<const bf16x8*>(base + (int64_t)row * stride + 16 * ks + 8 * g);
  }
  // arrived before the loop: left pending, the wait for them would land on a use inside it, as a wait for the tile loads too
#pragma unroll
  for (int ks = 0; ks < KS; ks++) asm volatile("" : "+v"(f[ks]));
}
// The same in two steps, with the loads of the first tiles between them: one latency in front of the loop instead of two.  (Without a branch
// around the loads, at whose end the compiler waits.)
template <int KS>
__device__ __forceinline__ void fetch_rows(bf16x8 (&f)[KS], const bf16* base, int64_t stride, int row, int nrows, int g) {
  const bf16* src = base + (int64_t)min(row, nrows - 1) * stride + 8 * g;
#pragma unroll
  for (int ks = 0; ks < KS; ks++) f[ks] = *reinterpret_cast<const bf16x8*>(src + 16 * ks);
}
template <int KS>
__device__ __forceinline__ void settle_rows(bf16x8 (&f)[KS], int row, int nrows) {
#pragma unroll
  for (int ks = 0; ks < KS; ks++) asm volatile("" : "+v"(f[ks]));
  if (row >= nrows)
#pragma unroll
    for (int ks = 0; ks < KS; ks++) f[ks] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
}

template <int DT>
__device__ __forceinline__ void clear(f32x16 (&x)[DT]) {
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) x[dt][r] = 0.f;
}

// accumulators of the second group to LDS, and back into the first (dst [register][lane] of this wavefront)
template <int DT>
__device__ __forceinline__ void give(float* patch, const f32x16 (&x)[DT], int lane) {
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) patch[(16 * dt + r) * 64 + lane] = x[dt][r];
}
template <int DT>
__device__ __forceinline__ void take(const float* patch, f32x16 (&x)[DT], int lane, float mine, float theirs) {
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) x[dt][r] = x[dt][r] * mine + patch[(16 * dt + r) * 64 + lane] * theirs;
}

// D accumulator columns of one row -> bf16 row
template <int DT>
__device__ __forceinline__ void store_row(bf16* dst, const f32x16 (&x)[DT], float scale, int g) {
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int a = 0; a < 4; a++) {
      bf16x4 w;
#pragma unroll
      for (int e = 0; e < 4; e++) w[e] = (bf16)(x[dt][4 * a + e] * scale);
      *reinterpret_cast<bf16x4*>(dst + 32 * dt + 8 * a + 4 * g) = w;
    }
}

// dQ^T of one query of a head of 64 (attn_store.h has that of 128) -> row qi of dq: scaled, then added to an fp32 or bf16 destination, or stored
__device__ __forceinline__ void store_dq(const AttnParams& p, const f32x16 (&dq)[2], int b, int h, int qi, int g) {
  const int64_t at = b * p.sdq.b + h * p.sdq.h + (int64_t)qi * p.sdq.l;
  if (p.dq_f32) {   // the running dq of a ring step: exact accumulation over the key blocks
    float* dst = static_cast<float*>(p.dq) + at;
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        f32x4* x = reinterpret_cast<f32x4*>(dst + 32 * dt + 8 * a + 4 * g);
        f32x4 w = {0.f, 0.f, 0.f, 0.f};
        if (p.accumulate_dq) w = *x;
#pragma unroll
        for (int e = 0; e < 4; e++) w[e] += dq[dt][4 * a + e] * p.scale;
        *x = w;
      }
  } else if (p.accumulate_dq) {
    bf16* dst = static_cast<bf16*>(p.dq) + at;
#pragma unroll
    for (int dt = 0; dt < 2; dt++)
#pragma unroll
      for (int a = 0; a < 4; a++) {
        bf16x4* x = reinterpret_cast<bf16x4*>(dst + 32 * dt + 8 * a + 4 * g);
        const bf16x4 old = *x;
        bf16x4 w;
#pragma unroll
        for (int e = 0; e < 4; e++) w[e] = (bf16)(dq[dt][4 * a + e] * p.scale + (float)old[e]);
        *x = w;
      }
  } else {
    store_row(static_cast<bf16*>(p.dq) + at, dq, p.scale, g);
  }
}

}  // namespace rowtile
