// Tile engine on the bf16 matrix cores with float32 results (gfx950, CDNA4, wave64).
//
// One workgroup of 256 threads (4 waves, 2x2) computes a 128x128 tile of
//     C[m][n] = sum_k  P(k, m) * Q(k, n)          k in [kbeg, kend)
// The fp32 matrix instructions of this chip run at 157 TFLOP/s, the bf16 ones at 2500.  A
// float32 is the exact sum of three bf16 numbers (8 + 8 + 8 significant bits, each the
// rounded rest of the ones before), x = h + m + l, so a product of two floats is nine
// products of bf16 numbers, each exact in float32:
//     x y = h h' + (h m' + m h') + (h l' + m m' + l h') + [m l' + l m' + l l'].
// (An element below 2^-109, 1.5e-33, is that sum only down to 2^-133, the smallest bf16 number: it
// enters rounded to a multiple of that, so that a product with a large factor keeps 2^-134 / |x|
// instead of 2^-24.)
// The bracket is at most 2^-25 and on average 2^-26 of x y, below the rounding of one float32
// accumulation, and is left out (on 64-wide tiles its last term only); the others run as
// v_mfma_f32_32x32x16_bf16.  The leading
// products and the five corrections have accumulators of their own: the leading ones are
// rounded once per 16 reduction steps, the corrections are 2^-8 of them, and the two are
// added at the end.  Measured against float64 on one 32x32 tile (relative 2-norm, this
// engine / v_mfma_f32_32x32x2_f32 on the same data):
//     N(0,1):           K = 128  6.3e-8 / 2.2e-7    K = 4096  4.0e-7 / 1.1e-6    K = 65536  1.7e-6 / 4.6e-6
//     max(0, N(0,1)):   K = 128  4.4e-8 / 8.6e-8    K = 4096  3.2e-7 / 5.0e-7    K = 65536  1.4e-6 / 2.0e-6
// and a factor of N(0,1) (either engine): K = 1  2.6e-8 / 2.5e-8, worst element 1.7 / 1.0 times 2^-24;
// 2  2.6e-8 / 3.1e-8;  4  2.7e-8 / 4.0e-8;  16  3.3e-8 / 7.3e-8;  53  4.7e-8 / 1.3e-7
// (with all six products in one accumulator the errors are those of the fp32 instruction,
// and sums of positive terms drift by -1.3e-6 at K = 65536: the accumulation inside the
// instruction rounds down.)
//
// A 64x64 sub-tile per wave takes 24 matrix instructions (768 cycles) per 16 reduction
// steps where the fp32 instruction takes 2048 cycles.  The operands are split on their way
// into LDS, once per workgroup; that is 5.5 vector instructions per element, which run
// beside the matrix instructions of the other wave on the SIMD.
#pragma once
#include "gemm_core.h"

namespace kfac {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) char lds_c;
typedef __attribute__((address_space(3))) unsigned lds_u;
typedef __attribute__((address_space(3))) v4u lds_u4;
typedef __attribute__((address_space(3))) v2u lds_u2;

// LDS of one operand chunk (16 reduction steps): three planes (h, m, l), each with the 16-byte
// groups of 8 consecutive k of all rows, the two groups of a row in two halves:
//     plane * PLANE + (k / 8) * HALF + row * 16 + (k % 8) * 2
// A fragment of the matrix instruction (lane: row = lane % 32, k = 8 * (lane / 32) + 0..7) is
// one ds_read_b128.  The halves are 64 bytes further apart than their size, which leaves a wave that
// writes 8-byte pieces of both at once without bank conflicts (counters: none in the products of
// both operand layouts; 128 bytes: a third of the LDS cycles of the one that writes 8-byte
// pieces, and of the step tiles of inverse.hip, whose inversion of 3500^2 takes 1160 us, not 1084).
template <int ROWS>
struct SplitChunk {
  static constexpr int HALF = ROWS * 16 + 64;
  static constexpr int PLANE = 2 * HALF;
  static constexpr int BYTES = 3 * PLANE;
};

// The 32x32 blocks of a tile that one wave computes, and from which fragment rows (of 32) of the
// operands.  TM x TN: the tile; NT: its threads; NB blocks a wave, block B = fragment row a(B) of P
// against row b(B) of Q (SAME: of P: a diagonal tile of a symmetric product, of which only P is
// staged); PF / QF fragment rows a wave.  PRODUCTS: how many of the nine partial products are taken;
// SCALE: what elements are multiplied with before they are split (a power of two).
// SplitTile: four waves, each a 64x64 quadrant of 128x128.
struct SplitTile {
  static constexpr int TM = 128, TN = 128, NT = 256, NB = 4, PF = 2, QF = 2;
  static constexpr int PRODUCTS = 6;
  static constexpr float SCALE = 1.f;
  static constexpr bool SAME = false;
  static constexpr int a(int B) { return B >> 1; }
  static constexpr int b(int B) { return B & 1; }
};
// SplitDiag: a 128x128 diagonal tile is symmetric itself; its blocks on and above the diagonal
// (10 of 16) are dealt to the four waves three at a time, as products of three fragment rows
// r0, r1, r2 of the one operand:
//     block 0 = (r0, r1)    block 1 = (r0, r2)    block 2 = (r1, r1)
//   waves 0 / 1: r = (0, 1, 0) / (2, 3, 2), the three blocks of a diagonal quadrant;
//   waves 2 / 3: r = (0, 2, 3) / (1, 2, 3), a row of the quadrant above the diagonal (their block 2
//   repeats one of wave 1's and is not stored).
// Every wave runs the same code, and the tile is done in three quarters of the time.
struct SplitDiag {
  static constexpr int TM = 128, TN = 128, NT = 256, NB = 3, PF = 3, QF = 0;
  static constexpr int PRODUCTS = 6;
  static constexpr float SCALE = 1.f;
  static constexpr bool SAME = true;
  static constexpr int a(int B) { return B == 2 ? 1 : 0; }
  static constexpr int b(int B) { return B == 1 ? 2 : 1; }
};
// SmallTile, SmallDiag: 64x64, a block on each of four waves (of a diagonal tile three blocks are
// stored).  A chunk is short work for a wave (6 matrix instructions), so what bounds these is the barrier and
// the loads of each chunk, and workgroups in flight hide them: five to a CU at 100 registers.  (One wave
// with the four blocks does with two thirds of the LDS reads, but needs 330 registers.)  On the fp32
// matrix instructions, a wave to a tile, / here with six partial products / here: output gradients of 32 images of
// 64x112x112 68 / 41 / 44 us, 128x56x56 54 / 35 / 38, six layers of 64x56x56 82 / 44 / 50, of 160x13x13
// 22 / 14.7 / 15.1; 3x3 inputs of 64x56x56, three layers, 485 / 326 / 357, the 3x224x224 of a 7x7 stem 262 / 160 /
// 171; 4096 rows of 100 26 / 10.8 / 11.0.  (What the two more products cost is what makes every sum as good as
// the fp32 instructions' own, see split_blocks; the scale costs nothing.)
constexpr float SMALL_SCALE = 16777216.f;       // 2^24
struct SmallTile {
  static constexpr int TM = 64, TN = 64, NT = 256, NB = 1, PF = 1, QF = 1;
  static constexpr int PRODUCTS = 8;
  static constexpr float SCALE = SMALL_SCALE;
  static constexpr bool SAME = false;
  static constexpr int a(int) { return 0; }
  static constexpr int b(int) { return 0; }
};
struct SmallDiag {
  static constexpr int TM = 64, TN = 64, NT = 256, NB = 1, PF = 2, QF = 0;
  static constexpr int PRODUCTS = 8;
  static constexpr float SCALE = SMALL_SCALE;
  static constexpr bool SAME = true;
  static constexpr int a(int) { return 0; }
  static constexpr int b(int) { return 1; }
};

// tiles 64 W wide
template <int W>
struct SplitCfg {
  static constexpr int TS = 64 * W;
  static constexpr int NT = NTHREADS;
  static constexpr int STAGE = 2 * SplitChunk<TS>::BYTES;
  static constexpr int VOTES = 2 * STAGE;                // a word per wave (split_blocks)
  static constexpr int SMEM_BYTES = VOTES + 4 * (NT / 64);
};

__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  v2bf r;
  r[0] = (__bf16)a;
  r[1] = (__bf16)b;
  return __builtin_bit_cast(unsigned, r);
}
__device__ __forceinline__ float bf16_lo(unsigned p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float bf16_hi(unsigned p) {
  return __builtin_bit_cast(float, p & 0xffff0000u);
}
// two floats -> their h, m and l parts, packed
__device__ __forceinline__ void split_pair(float a, float b, unsigned& h, unsigned& m, unsigned& l) {
  h = pack_bf16(a, b);
  asm("" : "+v"(h));       // (or the low half would be converted a second time)
  const float ra = a - bf16_lo(h), rb = b - bf16_hi(h);
  m = pack_bf16(ra, rb);
  asm("" : "+v"(m));
  l = pack_bf16(ra - bf16_lo(m), rb - bf16_hi(m));
}

// Leading sums + corrections.  An infinite element has no rest (inf - inf): where the corrections
// are not finite the leading sum is the result, infinite with its sign as a float32 sum's, and
// NaN only where that is.  (Finite elements that round to an infinite leading part: split_blocks.)
__device__ __forceinline__ void add_corrections(v16f& acc, const v16f& cor) {
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] += __builtin_isfinite(cor[i]) ? cor[i] : 0.f;
}

// the element at `off` (per lane, range-checked) + `at` (the same for all lanes)
__device__ __forceinline__ float buffer_load_at(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned at) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, (int)at, 0));
}

// ---------------------------------------------------------------------------
// global -> registers -> LDS, one chunk of an operand.  Two chunks are in flight (SET): a
// chunk is fetched two steps ahead of its use, split and stored one step ahead, in PIECES of
// two elements that the tile loop deals out between its matrix instructions.
// ---------------------------------------------------------------------------
// How four consecutive k of an MK operand lie in memory (`kruns`):
//   K_FLAT   always next to each other (a matrix row)
//   K_RUNS   in runs of at least 4 if `runs()`: `KRun run(k)` gives the offset of k, how many
//            elements its run still holds (itself included) and the offset of the next run;
//            `quads()`: all runs are multiples of 4 long
//            `padded()`: a run takes up a multiple of 4 of the reduction index, of which the last
//            up to three are no elements (of value 0)
//   K_ANY    anywhere (one offset per element)
enum { K_FLAT = 0, K_RUNS = 1, K_ANY = 2 };
struct KRun {
  unsigned off, next;
  int len;
};
// What a tile's chunks inside the k range may assume (`fast`): nothing; four consecutive k of an
// operand are one 16-byte load; or, in padded runs, one load that for the last four of a run
// is moved back to the run's end, so that it brings elements of the group before once more:
// the first `cut` of it, which count as 0.  (Within a group the k are then in another order, the
// same one in both operands.)
// A run that is no multiple of 4 without padding has groups across its end, and lanes that
// load element by element, and such a chunk waits for its own loads: 99 / 100 / 69 TFLOP/s for
// 2048 channels of 13x13 / 25x25 / 7 positions where 14x14 reach 155; padded 144 / 145 / 130.
enum { ANY_K = 0, FAST_K = 1, PADDED_K = 2 };

// Index positions of a run of `run` elements: a multiple of 4 wherever a group of 4 fits into it.
// (A run of 5 is 60 % more work and still faster, as correlations and as products: 8 images of 600x3x3 /
// 32 of 512x3x3 / 2048x7x7 / 384x55x55 unpadded 21.2 / 24.1 / 71.3 / 122.7 us, padded 18.3 / 19.0 /
// 64.4 / 108.2; correlations of 512 channels of 7x7, rows of 5,
// 211 us unpadded, 201 padded; 9x9, rows of 7, 265 / 234; 128 channels of 56x56, rows of 54,
// 527 / 489; 28x28, rows of 26, 177 / 170.)
__host__ __device__ inline int padded_run(int run) {
  const int up = (run + 3) & ~3;
  return run >= 4 ? up : run;
}

// an operand that may lie in padded runs
template <class OP, class = void>
struct has_padded_runs : std::false_type {};
template <class OP>
struct has_padded_runs<OP, std::enable_if_t<OP::pads_runs>> : std::true_type {};

template <class OP, int ROWS, int NT, int LAYOUT = OP::layout>
struct SplitStager;

// Consecutive m contiguous: a thread takes 8 consecutive k of one column (4 where there are more
// threads than that).
template <class OP, int ROWS, int NT>
struct SplitStager<OP, ROWS, NT, KM> {
  static constexpr int KPT = ROWS * 2 >= NT ? 8 : 4;
  static constexpr int NI = ROWS * (16 / KPT) / NT;
  static constexpr int PIECES = KPT / 2 * NI;
  static_assert(ROWS * (16 / KPT) % NT == 0 && ROWS % 64 == 0, "a wave's lanes share their k");
  typedef unsigned Part __attribute__((ext_vector_type(KPT / 2)));
  typename OP::MS ms[NI];
  float regs[2][NI][KPT];
  unsigned ones[2];          // bit KPT i + j: element j of column i is the constant 1
  Part ph, pm, pl;           // the column being split

  static __device__ __forceinline__ int tid() { return threadIdx.x & (NT - 1); }
  static __device__ __forceinline__ int kgroup(int i) {
    return __builtin_amdgcn_readfirstlane((tid() + NT * i) / ROWS);
  }
  // the tile lies inside the columns that are plain memory
  static __device__ __forceinline__ int fast(const OP& op, int m0) {
    return op.vec_cols() == op.M || m0 + ROWS <= op.vec_cols() ? FAST_K : ANY_K;
  }
  __device__ __forceinline__ void init(const OP& op, int m0) {
#pragma unroll
    for (int i = 0; i < NI; ++i) ms[i] = op.mstate(m0 + ((tid() + NT * i) & (ROWS - 1)));
  }
  template <int SET, class OTHER>
  __device__ __forceinline__ void take_k(const OP&, const OP&, const OTHER&) {}
  // a chunk inside the k range of a `fast` tile, load by load
  static constexpr int LOADS = KPT * NI;
  template <int SET, int LOAD, int MODE, bool KNOWN>
  __device__ __forceinline__ void fetch_load(const OP& op, int k0) {
    constexpr int i = LOAD / KPT, j = LOAD % KPT;
    regs[SET][i][j] = buffer_load_at(op.rsrc(), ms[i].off, (k0 + KPT * kgroup(i) + j) * op.kstride());
  }
  // any chunk
  template <int SET>
  __device__ __forceinline__ void fetch(const OP& op, int k0, int kend) {
    unsigned one = 0;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int k = k0 + KPT * kgroup(i);
#pragma unroll
      for (int j = 0; j < KPT; ++j) {
        // (k is the same for all lanes: its offset is a scalar)
        const bool in = k + j < kend;
        const unsigned at = in ? (k + j) : 0;
        regs[SET][i][j] = buffer_load_at(op.rsrc(), in ? ms[i].off : INV_M, at * op.kstride());
        if (op.second())
          regs[SET][i][j] += buffer_load_at(op.rsrc2(), in ? ms[i].off2 : INV_M, at * 4u);
        one |= (unsigned)(op.is_one(ms[i]) && in) << (KPT * i + j);
      }
    }
    ones[SET] = one;
  }
  // the elements as they are (fp32_tile): rows of LDS_MK floats
  __device__ __forceinline__ void commit_plain(lds_f* chunk) {
    static_assert(KPT == 4, "one 16-byte store a column");
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      v4f v;
#pragma unroll
      for (int j = 0; j < KPT; ++j) {
        v[j] = ((ones[0] >> (KPT * i + j)) & 1u) ? 1.f : regs[0][i][j];
        if (squares_elements<OP>::value) v[j] *= v[j];
      }
      *(lds_f4*)(chunk + ((tid() + NT * i) & (ROWS - 1)) * LDS_MK + KPT * kgroup(i)) = v;
    }
  }
  template <int SET, int PIECE, int MODE, bool SCALED = false>
  __device__ __forceinline__ void commit(lds_c* chunk, float scale = 1.f) {
    typedef SplitChunk<ROWS> L;
    constexpr int i = PIECE / (KPT / 2), j = PIECE % (KPT / 2);
    float v[2] = {regs[SET][i][2 * j], regs[SET][i][2 * j + 1]};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (MODE == ANY_K) v[e] = ((ones[SET] >> (KPT * i + 2 * j + e)) & 1u) ? 1.f : v[e];
      if (squares_elements<OP>::value) v[e] *= v[e];
      if (SCALED) v[e] *= scale;
    }
    unsigned h, m, l;
    split_pair(v[0], v[1], h, m, l);
    ph[j] = h;
    pm[j] = m;
    pl[j] = l;
    if (j == KPT / 2 - 1) {
      typedef __attribute__((address_space(3))) Part lds_part;
      const int k = KPT * kgroup(i);
      lds_c* const at = chunk + k / 8 * L::HALF + ((tid() + NT * i) & (ROWS - 1)) * 16 + k % 8 * 2;
      *(lds_part*)at = ph;
      *(lds_part*)(at + L::PLANE) = pm;
      *(lds_part*)(at + 2 * L::PLANE) = pl;
    }
  }
};

// Consecutive k contiguous: a thread takes 4 consecutive k of NI rows.
template <class OP, int ROWS, int NT>
struct SplitStager<OP, ROWS, NT, MK> {
  static constexpr int NI = ROWS * 4 / NT;
  static constexpr int PIECES = 2 * NI;
  static constexpr int STEP = NT / 4;
  typename OP::MS ms[NI];
  v4f regs[2][NI];
  unsigned ones;             // bit i: row i is the row of ones (K_ANY operands)
  unsigned kin[2];           // bit j: element j lies inside the k range (where `ones` matters)
  v2u ph, pm, pl;            // the row being split

  static __device__ __forceinline__ int tid() { return threadIdx.x & (NT - 1); }
  static __device__ __forceinline__ int fast(const OP& op, int) {
    if constexpr (OP::kruns == K_RUNS) return op.quads() ? FAST_K : op.padded() ? PADDED_K : ANY_K;
    return OP::kruns == K_FLAT ? FAST_K : ANY_K;
  }
  __device__ __forceinline__ void init(const OP& op, int m0) {
    ones = 0;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      ms[i] = op.mstate(m0 + (tid() >> 2) + STEP * i);
      if (OP::kruns == K_ANY) ones |= (unsigned)op.is_one(ms[i]) << i;
    }
  }
  static constexpr int LOADS = NI;
  unsigned koff;             // of the chunk being fetched by fetch_load
  int cut[2];                // PADDED_K: elements of the group that count as 0
  // the k of the other operand's chunk
  template <int SET, class OTHER>
  __device__ __forceinline__ void take_k(const OP& op, const OP& other, const OTHER& o) {
    koff = o.koff + op.k_shift(other);
    cut[SET] = o.cut[SET];
  }
  template <int SET, int LOAD, int MODE, bool KNOWN>
  __device__ __forceinline__ void fetch_load(const OP& op, int k0) {
    const int k = k0 + 4 * (tid() & 3);
    if (LOAD == 0 && !KNOWN) {
      if constexpr (OP::kruns == K_RUNS) {
        const KRun run = op.run(k);
        koff = run.off;
        if (MODE == PADDED_K) {
          cut[SET] = max(0, 4 - run.len);
          koff -= 4u * cut[SET];
        }
      } else {
        koff = op.kstate(k, true).off;
      }
    }
    regs[SET][LOAD] = buffer_load4(op.rsrc(), ms[LOAD].off + koff);
  }
  template <int SET>
  __device__ __forceinline__ void fetch(const OP& op, int k0, int kend) {
    const __amdgpu_buffer_rsrc_t rs = op.rsrc();
    const int k = k0 + 4 * (tid() & 3);
    cut[SET] = 0;
    if constexpr (OP::kruns == K_RUNS) {
      if (op.runs()) {
        const KRun run = op.run(k);
        const bool whole = run.len >= 4 && k + 4 <= kend;
        if (__builtin_amdgcn_ballot_w64(!whole) == 0) {
#pragma unroll
          for (int i = 0; i < NI; ++i) regs[SET][i] = buffer_load4(rs, ms[i].off + run.off);
        } else if (whole) {
#pragma unroll
          for (int i = 0; i < NI; ++i) regs[SET][i] = buffer_load4(rs, ms[i].off + run.off);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const unsigned off = j < run.len ? run.off + 4 * j : run.next + 4 * (j - run.len);
            const unsigned ko = k + j < kend ? off : INV_K;
#pragma unroll
            for (int i = 0; i < NI; ++i) regs[SET][i][j] = buffer_load(rs, ms[i].off + ko);
          }
        }
        return;
      }
    }
    unsigned in = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const typename OP::KS ks = op.kstate(k + j, k + j < kend);
      in |= (unsigned)(k + j < kend) << j;
#pragma unroll
      for (int i = 0; i < NI; ++i) regs[SET][i][j] = buffer_load(rs, op.off(ms[i], ks));
    }
    kin[SET] = in;
  }
  __device__ __forceinline__ void commit_plain(lds_f* chunk) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      v4f v = regs[0][i];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (OP::kruns == K_ANY) v[j] = ((ones >> i) & (kin[0] >> j) & 1u) ? 1.f : v[j];
        if (squares_elements<OP>::value) v[j] *= v[j];
      }
      *(lds_f4*)(chunk + ((tid() >> 2) + STEP * i) * LDS_MK + 4 * (tid() & 3)) = v;
    }
  }
  template <int SET, int PIECE, int MODE, bool SCALED = false>
  __device__ __forceinline__ void commit(lds_c* chunk, float scale = 1.f) {
    typedef SplitChunk<ROWS> L;
    constexpr int i = PIECE / 2, j = PIECE % 2;
    float v[2] = {regs[SET][i][2 * j], regs[SET][i][2 * j + 1]};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (MODE == PADDED_K && 2 * j + e < 3) v[e] = cut[SET] > 2 * j + e ? 0.f : v[e];
      if (OP::kruns == K_ANY) v[e] = ((ones >> i) & (kin[SET] >> (2 * j + e)) & 1u) ? 1.f : v[e];
      if (squares_elements<OP>::value) v[e] *= v[e];
      if (SCALED) v[e] *= scale;
    }
    unsigned h, m, l;
    split_pair(v[0], v[1], h, m, l);
    ph[j] = h;
    pm[j] = m;
    pl[j] = l;
    if (j == 1) {
      lds_c* const at = chunk + ((tid() >> 1) & 1) * L::HALF + ((tid() >> 2) + STEP * i) * 16 +
                        (tid() & 1) * 8;
      *(lds_u2*)at = ph;
      *(lds_u2*)(at + L::PLANE) = pm;
      *(lds_u2*)(at + 2 * L::PLANE) = pl;
    }
  }
};

template <int ROWS>
__device__ __forceinline__ v8bf load_frag(const lds_c* chunk, int row0, int lane, int plane) {
  typedef SplitChunk<ROWS> L;
  const lds_c* const at = chunk + plane * L::PLANE + (lane >> 5) * L::HALF + (row0 + (lane & 31)) * 16;
  return __builtin_bit_cast(v8bf, *(const lds_u4*)at);
}

template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

struct SplitTri {
  int r[3];
  bool last;           // block 2 is this wave's to store
};
__device__ __forceinline__ SplitTri split_tri(int wave) {
  if (wave == 0) return SplitTri{{0, 1, 0}, true};
  if (wave == 1) return SplitTri{{2, 3, 2}, true};
  return SplitTri{{wave - 2, 2, 3}, false};
}

// fragments of one chunk: [h, m, l][row]
template <class TILE>
struct SplitFrags {
  v8bf p[3][TILE::PF];
  v8bf q[3][TILE::QF > 0 ? TILE::QF : 1];
};

// product PR for block B, in the order h h', h m', m h', m m', (m l', l m',) h l', l h': the last two leave
// m's registers to the next chunk
template <class TILE, int PR, int B>
__device__ __forceinline__ void split_product(const SplitFrags<TILE>& fr, v16f& sum) {
  constexpr int LAST = PR - (TILE::PRODUCTS - 2);
  constexpr int PA = LAST == 0 ? 0 : LAST == 1 ? 2 : PR < 4 ? PR >> 1 : PR == 4 ? 1 : 2;
  constexpr int PB = LAST == 0 ? 2 : LAST == 1 ? 0 : PR < 4 ? PR & 1 : PR == 4 ? 2 : 1;
  const v8bf a = fr.p[PA][TILE::a(B)];
  v8bf b;
  if constexpr (TILE::SAME) b = fr.p[PB][TILE::b(B)];
  else b = fr.q[PB][TILE::b(B)];
  sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, sum, 0, 0, 0);
}

// the fragment rows of a wave, as rows of the tile
struct SplitRows {
  int p[3], q[2];
};

// Accumulates C = P Q over [kbeg, kend) into the wave's blocks (leading products in acc, the
// corrections in cor).
template <class C, int MODE, class OPP, class OPQ>
__device__ __forceinline__ void split_tile_loop(const OPP& P, const OPQ& Q, int m0, int n0, int kbeg,
                                                int kend, lds_c* sm, const SplitRows& rows,
                                                v16f (&acc)[C::NB], v16f (&cor)[C::NB]) {
  constexpr bool TRI = C::SAME;
  constexpr int STAGE = SplitCfg<C::TM / 64>::STAGE;
  constexpr int QOFF = SplitChunk<C::TM>::BYTES;
  constexpr int NB = C::NB;
  const int lane = threadIdx.x & 63;
  typedef SplitStager<OPP, C::TM, C::NT> SP;
  typedef SplitStager<OPQ, C::TN, C::NT> SQ;
  SP sp;
  SQ sq;
  sp.init(P, m0);
  if (!TRI) sq.init(Q, n0);
  const int nchunks = (kend - kbeg + KC - 1) / KC;
  const int nfull = (kend - kbeg) / KC;
  if (nchunks <= 0) return;
  auto fetch = [&](auto set_, int c) {
    constexpr int SET = decltype(set_)::value;
    sp.template fetch<SET>(P, kbeg + c * KC, kend);
    if (!TRI) sq.template fetch<SET>(Q, kbeg + c * KC, kend);
  };
  constexpr int LOADS = SP::LOADS + (TRI ? 0 : SQ::LOADS);
  auto fetch_load = [&](auto set_, auto load_, int c) {
    constexpr int SET = decltype(set_)::value, X = decltype(load_)::value;
    if constexpr (X < SP::LOADS)
      sp.template fetch_load<SET, X, MODE, false>(P, kbeg + c * KC);
    else {
      // (two operands in runs have the same ones: one division for both)
      constexpr bool known = has_padded_runs<OPP>::value && std::is_same<OPP, OPQ>::value &&
                             MODE != ANY_K && C::TM == C::TN;
      if constexpr (known && X == SP::LOADS) sq.template take_k<SET>(Q, P, sp);
      sq.template fetch_load<SET, X - SP::LOADS, MODE, known>(Q, kbeg + c * KC);
    }
  };
  constexpr int PIECES = SP::PIECES + (TRI ? 0 : SQ::PIECES);
  auto commit = [&](auto set_, auto piece_, lds_c* stage) {
    constexpr int SET = decltype(set_)::value, X = decltype(piece_)::value;
    if constexpr (X < SP::PIECES)
      sp.template commit<SET, X, MODE, C::SCALE != 1.f>(stage, C::SCALE);
    else
      sq.template commit<SET, X - SP::PIECES, MODE, C::SCALE != 1.f>(stage + QOFF, C::SCALE);
  };
  SplitFrags<C> fr[2];
  auto load_frags = [&](auto set_, auto plane_) {
    constexpr int SET = decltype(set_)::value, PL = decltype(plane_)::value;
    const lds_c* const tp = sm + SET * STAGE;
#pragma unroll
    for (int i = 0; i < C::PF; ++i) fr[SET].p[PL][i] = load_frag<C::TM>(tp, rows.p[i], lane, PL);
#pragma unroll
    for (int i = 0; i < C::QF; ++i) fr[SET].q[PL][i] = load_frag<C::TN>(tp + QOFF, rows.q[i], lane, PL);
  };
  constexpr std::integral_constant<int, 0> S0{};
  constexpr std::integral_constant<int, 1> S1{};
  // (chunks past the end are fetched like the others: their elements lie outside the k
  // range and cost no memory access, and the number of loads in flight is the same on every
  // path, so that a commit waits for its own chunk only)
  fetch(S0, 0);
  fetch(S1, 1);
  static_for<PIECES>([&](auto x) { commit(S0, x, sm); });
  __syncthreads();
  load_frags(S0, std::integral_constant<int, 0>{});

  // One chunk.  Its leading planes are in registers already; the loads of chunk c + 2 and the
  // pieces of chunk c + 1 are dealt out between the matrix instructions of all but two
  // products; then the workgroup meets (chunk c has been read and chunk c + 1 written by
  // every wave), and the leading planes of chunk c + 1 come in under the last two products.
  auto step = [&](auto set_, auto full_, int c) {
    constexpr int SET = decltype(set_)::value;
    constexpr bool FULL = decltype(full_)::value;
    lds_c* const next = sm + (SET ^ 1) * STAGE;
    load_frags(set_, std::integral_constant<int, 1>{});
    load_frags(set_, std::integral_constant<int, 2>{});
    if (!FULL) fetch(set_, c + 2);
    __builtin_amdgcn_sched_barrier(0);
    static_for<C::PRODUCTS>([&](auto prod_) {
      constexpr int PR = decltype(prod_)::value;
      if constexpr (PR == C::PRODUCTS - 2) {
        __syncthreads();
        load_frags(std::integral_constant<int, SET ^ 1>{}, std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);
      }
      static_for<NB>([&](auto blk_) {
        constexpr int B = decltype(blk_)::value;
        constexpr int IDX = PR * NB + B;
        split_product<C, PR, B>(fr[SET], PR == 0 ? acc[B] : cor[B]);
        if constexpr (PR < C::PRODUCTS - 2) {
          constexpr int LAST = (C::PRODUCTS - 2) * NB;
          constexpr int l0 = IDX * LOADS / LAST, l1 = (IDX + 1) * LOADS / LAST;
          if constexpr (FULL)
            static_for<l1 - l0>([&](auto x) {
              fetch_load(set_, std::integral_constant<int, l0 + decltype(x)::value>{}, c + 2);
            });
          constexpr int p0 = IDX * PIECES / LAST, p1 = (IDX + 1) * PIECES / LAST;
          static_for<p1 - p0>([&](auto x) {
            commit(std::integral_constant<int, SET ^ 1>{},
                   std::integral_constant<int, p0 + decltype(x)::value>{}, next);
          });
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    });
  };
  constexpr std::false_type ANY{};
  int c = 0;
  if (MODE != ANY_K) {
    constexpr std::true_type FULL{};
    for (; c + 3 < nfull; c += 2) {       // (chunks c + 2 and c + 3 lie inside the range)
      step(S0, FULL, c);
      step(S1, FULL, c + 1);
    }
  }
  for (; c < nchunks; c += 2) {           // (a chunk past the end adds zeros)
    step(S0, ANY, c);
    step(S1, ANY, c + 1);
  }
}

// The same in a rolled loop, one chunk after the other, the loads of the next one in flight under
// the products of this one, with every element multiplied by `scale`.  For reductions of up to
// SHORT_K steps: such a tile is a chain of latencies, instruction fetches among them, and this
// loop has a third of the code and no chunk past the end.  Factor of 16 rows of 300 / 48 of 1000 /
// 8 of 5000: 12.1 / 15.7 / 57.5 us by the loop above, 9.8 / 14.1 / 52.7 by this one (9.4 / 13.3 /
// 51.8 on the fp32 tile engine); 64 rows of 512: 16.1 / 16.7.
constexpr int SHORT_K = 48;
template <class C, class OPP, class OPQ>
__device__ __forceinline__ void split_tile_rolled(const OPP& P, const OPQ& Q, int m0, int n0, int kbeg,
                                                  int kend, lds_c* sm, const SplitRows& rows, float scale,
                                                  v16f (&acc)[C::NB], v16f (&cor)[C::NB]) {
  constexpr bool TRI = C::SAME;
  constexpr int STAGE = SplitCfg<C::TM / 64>::STAGE;
  constexpr int QOFF = SplitChunk<C::TM>::BYTES;
  const int lane = threadIdx.x & 63;
  typedef SplitStager<OPP, C::TM, C::NT> SP;
  typedef SplitStager<OPQ, C::TN, C::NT> SQ;
  SP sp;
  SQ sq;
  sp.init(P, m0);
  if (!TRI) sq.init(Q, n0);
  sp.template fetch<0>(P, kbeg, kend);
  if (!TRI) sq.template fetch<0>(Q, kbeg, kend);
  int stage = 0;
#pragma unroll 1
  for (int k0 = kbeg; k0 < kend; k0 += KC) {
    lds_c* const at = sm + stage;
    stage ^= STAGE;
    static_for<SP::PIECES>(
        [&](auto x) { sp.template commit<0, decltype(x)::value, ANY_K, true>(at, scale); });
    if (!TRI)
      static_for<SQ::PIECES>(
          [&](auto x) { sq.template commit<0, decltype(x)::value, ANY_K, true>(at + QOFF, scale); });
    if (k0 + KC < kend) {
      sp.template fetch<0>(P, k0 + KC, kend);
      if (!TRI) sq.template fetch<0>(Q, k0 + KC, kend);
    }
    __syncthreads();       // (every wave is done with the chunk before this one: its stage is free)
    SplitFrags<C> fr;
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) {
#pragma unroll
      for (int i = 0; i < C::PF; ++i) fr.p[pl][i] = load_frag<C::TM>(at, rows.p[i], lane, pl);
#pragma unroll
      for (int i = 0; i < C::QF; ++i) fr.q[pl][i] = load_frag<C::TN>(at + QOFF, rows.q[i], lane, pl);
    }
    static_for<C::PRODUCTS>([&](auto prod_) {
      constexpr int PR = decltype(prod_)::value;
      static_for<C::NB>([&](auto blk_) {
        constexpr int B = decltype(blk_)::value;
        split_product<C, PR, B>(fr, PR == 0 ? acc[B] : cor[B]);
      });
    });
  }
}

// The same on the fp32 instructions (64-wide tiles): what leaves the range of the split elements.
template <class C, class OPP, class OPQ>
__device__ __forceinline__ void fp32_tile(const OPP& P, const OPQ& Q, int m0, int n0, int kbeg, int kend,
                                          lds_c* sm, const SplitRows& rows, v16f& acc) {
  static_assert(C::NB == 1 && C::TM * LDS_MK * 4 <= SplitChunk<C::TM>::BYTES, "one block a wave, 64-wide chunks");
  constexpr bool SAME = C::SAME;
  constexpr int STAGE = SplitCfg<C::TM / 64>::STAGE;
  constexpr int QOFF = SAME ? 0 : SplitChunk<C::TM>::BYTES;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  SplitStager<OPP, C::TM, C::NT> sp;
  SplitStager<OPQ, C::TN, C::NT> sq;
  sp.init(P, m0);
  if (!SAME) sq.init(Q, n0);
  int stage = 0;
#pragma unroll 1
  for (int k0 = kbeg; k0 < kend; k0 += KC) {
    lds_c* const at = sm + stage;
    stage ^= STAGE;
    sp.template fetch<0>(P, k0, kend);
    if (!SAME) sq.template fetch<0>(Q, k0, kend);
    sp.commit_plain((lds_f*)at);
    if (!SAME) sq.commit_plain((lds_f*)(at + QOFF));
    __syncthreads();       // (every wave is done with the chunk before this one: its stage is free)
    const lds_f* const pa = (const lds_f*)at + (rows.p[0] + r) * LDS_MK + 4 * h;
    const lds_f* const pb = (const lds_f*)(at + QOFF) + ((SAME ? rows.p[1] : rows.q[0]) + r) * LDS_MK + 4 * h;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const v4f a = *(const lds_f4*)(pa + 8 * j), b = *(const lds_f4*)(pb + 8 * j);
#pragma unroll
      for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], b[s], acc, 0, 0, 0);
    }
  }
}

// The sum of a wave's blocks over [kbeg, kend), in acc.
// A finite element beyond the largest bf16 number (3.3895e38) rounds to an infinite leading part,
// and every sum that it enters comes out as inf or NaN; and leading parts that are rounded up have
// an infinite sum where the elements' own is still finite (above 0.992 of the largest float32:
// the square of 2^64 - 2^54).  So a tile with a sum that is not finite is computed once more
// from halves of the elements, and the sums taken four times: what is finite then, is what a
// float32 sum gives, and what is not, is not there either.  (Half of an element is exact, but for
// a last bit of 2^-149.)  The waves vote across the barrier that ends a tile anyway.
// The 64-wide tiles are as good as fp32 instructions, which they replaced, at every element:
//   they take the two largest of the partial products left out as well.  In sums of one or few terms
//   those are as large as a float32 sum's own rounding (a single product is off by up to 1.7 half units in the
//   last place without them, 1.0 with them);
//   elements are multiplied by 2^24 before they are split, so that those below 2^-109 keep all their bits (to the
//   last one of the smallest float32, 2^-149), and the sums by 2^-48;
//   a tile with a sum that is then not finite, with an element from 2^104 or a sum from 2^80 on, that is,
//   is computed once more by the fp32 instructions.
template <class C, class OPP, class OPQ>
__device__ __forceinline__ void split_blocks(const OPP& P, const OPQ& Q, int m0, int n0, int kbeg,
                                             int kend, float* smem, const SplitRows& rows,
                                             v16f (&acc)[C::NB]) {
  constexpr bool TRI = C::SAME;
  constexpr int NB = C::NB;
  v16f cor[NB];
  lds_c* const sm = (lds_c*)smem;
  lds_u* const votes = (lds_u*)(sm + SplitCfg<C::TM / 64>::VOTES);
  const int wave = (int)(threadIdx.x & (C::NT - 1)) >> 6;
  // (uniform per workgroup; operands in padded runs are two of a kind)
  const int mode = SplitStager<OPP, C::TM, C::NT>::fast(P, m0);
  const int qmode = TRI ? mode : SplitStager<OPQ, C::TN, C::NT>::fast(Q, n0);
  auto clear = [&]() {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[b][i] = cor[b][i] = 0.f;
  };
  clear();
  if (kend <= kbeg) return;
  if (kend - kbeg <= SHORT_K) {
    split_tile_rolled<C>(P, Q, m0, n0, kbeg, kend, sm, rows, C::SCALE, acc, cor);
  } else if (mode == FAST_K && qmode == FAST_K) {
    split_tile_loop<C, FAST_K>(P, Q, m0, n0, kbeg, kend, sm, rows, acc, cor);
  } else if (has_padded_runs<OPP>::value && mode == PADDED_K) {
    if constexpr (has_padded_runs<OPP>::value)
      split_tile_loop<C, PADDED_K>(P, Q, m0, n0, kbeg, kend, sm, rows, acc, cor);
  } else {
    split_tile_loop<C, ANY_K>(P, Q, m0, n0, kbeg, kend, sm, rows, acc, cor);
  }
  // (0 times a sum that is not finite is NaN; the third part of an element with an infinite leading
  // part is NaN, and so are all the corrections that it enters)
  float probe = 0.f;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      acc[b][i] += cor[b][i];
      probe = fmaf(acc[b][i], 0.f, probe);
    }
  votes[wave] = __builtin_amdgcn_ballot_w64(probe != 0.f) != 0;
  __syncthreads();           // (and the next tile of this workgroup may overwrite the stages)
  unsigned any = 0;
#pragma unroll
  for (int w = 0; w < C::NT / 64; ++w) any |= votes[w];
  const bool again = __builtin_expect(__builtin_amdgcn_readfirstlane((int)any) != 0, 0);
  if constexpr (NB == 1) {
    if (again) {
      clear();
      fp32_tile<C>(P, Q, m0, n0, kbeg, kend, sm, rows, acc[0]);
      __syncthreads();
    } else {
      acc[0] *= 1.f / (C::SCALE * C::SCALE);
    }
  } else if (again) {
    clear();
    split_tile_rolled<C>(P, Q, m0, n0, kbeg, kend, sm, rows, 0.5f, acc, cor);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      add_corrections(acc[b], cor[b]);
      acc[b] *= 4.f;
    }
    __syncthreads();
  }
}

// The 32x32 blocks of a wave, rows from `row0`, columns from `col0`, through the epilogue.
// `what`: nothing (the block is another wave's), the block or, for a block on the diagonal, its upper
// triangle.  (The two orders in which the corrections h m' and m h' are added round differently, so that
// only one triangle of such a block is used: the result is symmetric to the bit.)
enum { BLK_NONE = 0, BLK_PLAIN = 1, BLK_UPPER = 2 };
template <int NB, class EPI>
__device__ __forceinline__ void store_blocks(const v16f (&acc)[NB], const int (&row0)[NB],
                                             const int (&col0)[NB], const int (&what)[NB],
                                             const EPI& epi) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 31, h = lane >> 5;
  auto row_of = [&](int b, int i) { return row0[b] + 8 * (i >> 2) + 4 * h + (i & 3); };
  auto put = [&](int b, auto&& element) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = row_of(b, i), col = col0[b] + r;
      if (what[b] != BLK_UPPER || row <= col) element(i, row, col);
    }
  };
  if constexpr (reading_epilogue<EPI>::value) {
    // C = alpha*acc + beta*C_old: the old values of two blocks are loaded ahead of the stores.
    // Interleaved load/store pairs would each wait for their own load (a store to C may alias
    // the next load of C, so the compiler keeps them in order).
    if (epi.reads()) {
#pragma unroll
      for (int b0 = 0; b0 < NB; b0 += 2) {
        float old[2][16];
#pragma unroll
        for (int b = b0; b < b0 + 2 && b < NB; ++b)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            old[b - b0][i] = what[b] != BLK_NONE ? epi.fetch(row_of(b, i), col0[b] + r) : 0.f;
#pragma unroll
        for (int b = b0; b < b0 + 2 && b < NB; ++b)
          if (what[b] != BLK_NONE)
            put(b, [&](int i, int row, int col) { epi.store_with(row, col, acc[b][i], old[b - b0][i]); });
      }
      return;
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b)
    if (what[b] != BLK_NONE)
      put(b, [&](int i, int row, int col) { epi.store(row, col, acc[b][i]); });
}

// An epilogue with value() and put() can have the images of a tile's blocks across the diagonal stored as well.
template <class T, class = void>
struct imaging_epilogue : std::false_type {};
template <class T>
struct imaging_epilogue<T, std::void_t<decltype(std::declval<const T&>().put(0, 0, 0.f))>> : std::true_type {};

// store_blocks, with the image of every block.  It goes through the wave's own piece of LDS (`smem`, free again when
// the sums are done; the workgroup's last use of it), a block at a time, and to memory by its rows: from the
// registers it is written by 4-byte pieces of 64 rows at a time.  The old values of all blocks are in flight
// together (they are symmetric like the new ones).  Bound by memory, 16 bytes an element of the triangle.  Running
// average of a factor, us with the images from the registers / here: 256 rows of 9216 285 / 244 (2.8 TB/s), of 4096
// 83 / 68, 64 rows of 4096 59 / 44 (3.0 TB/s), 32 of 2048 23.7 / 19.7, 16 of 1000 18.9 / 16.9; 256 of 2048 38.4 / 38.8.
constexpr int IMAGE_LD = 33;
static_assert(NTHREADS / 64 * 32 * IMAGE_LD * 4 <= SplitCfg<2>::VOTES, "the images lie where the tile's chunks were");
template <int NB, class EPI>
__device__ __forceinline__ void store_images(const v16f (&acc)[NB], const int (&row0)[NB],
                                             const int (&col0)[NB], const int (&what)[NB], float* smem,
                                             const EPI& epi) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 31, h = lane >> 5;
  lds_f* const t = (lds_f*)smem + ((int)(threadIdx.x & (NTHREADS - 1)) >> 6) * 32 * IMAGE_LD;
  float old[NB][16];
  bool reads = false;
  if constexpr (reading_epilogue<EPI>::value) {
    reads = epi.reads();
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        old[b][i] = reads && what[b] != BLK_NONE
                        ? epi.fetch(row0[b] + 8 * (i >> 2) + 4 * h + (i & 3), col0[b] + r) : 0.f;
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (what[b] == BLK_NONE) continue;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 8 * (i >> 2) + 4 * h + (i & 3);
      float o = epi.value(acc[b][i]);
      if constexpr (reading_epilogue<EPI>::value) o = reads ? epi.value(acc[b][i], old[b][i]) : o;
      if (what[b] != BLK_UPPER || row <= r) epi.put(row0[b] + row, col0[b] + r, o);
      t[r * IMAGE_LD + row] = o;
    }
    // (other lanes' values: a wave's accesses to LDS are done in order)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 2 * i + h;         // of the image
      const float o = t[row * IMAGE_LD + r];
      if (what[b] != BLK_UPPER || r < row) epi.put(col0[b] + row, row0[b] + r, o);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

// A 64-wide tile with mirror images, a 32x32 block on each of four waves, through LDS (`smem`, free again when the sums
// are done; the workgroup's last use of it): from the registers an image would be written by 4-byte pieces
// of 64 rows at a time.  Results go there once (`old` values are read, and `epi` applied, for the blocks on and above
// the diagonal only), and come back row by row.  TRI: a diagonal tile, whose upper triangle is the result.
// Factor of 16 rows of 64 / 64 of 64 / 128 of 100: 7.2 / 8.4 / 9.5 us from the registers, 4.5 / 5.8 / 8.2 here
// (on the fp32 instructions, whose diagonal blocks need no image, 5.4 / 7.8 / 24.1).
constexpr int SMALL_LD = 65;
static_assert(64 * SMALL_LD * 4 <= SplitCfg<1>::VOTES, "the result of a 64-wide tile lies where its chunks were");
template <bool TRI, class EPI>
__device__ __forceinline__ void store_small(const v16f& acc, int m0, int n0, int wm, int wn, float* smem,
                                            const EPI& epi) {
  lds_f* const t = (lds_f*)smem;
  const int lane = threadIdx.x & 63;
  const int row0 = wm + 4 * (lane >> 5), col = wn + (lane & 31);
  if (!TRI || wm <= wn) {
    float old[16];
    bool reads = false;
    if constexpr (reading_epilogue<EPI>::value) {
      reads = epi.reads();
#pragma unroll
      for (int i = 0; i < 16; ++i)
        old[i] = reads ? epi.fetch(m0 + row0 + 8 * (i >> 2) + (i & 3), n0 + col) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = row0 + 8 * (i >> 2) + (i & 3);
      float o = epi.value(acc[i]);
      if constexpr (reading_epilogue<EPI>::value) o = reads ? epi.value(acc[i], old[i]) : o;
      t[row * SMALL_LD + col] = o;
      if (!TRI) epi.put(m0 + row, n0 + col, o);
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    // row r of the tile (TRI), or of its image
    const int r = (int)(threadIdx.x >> 6) + 4 * i, c = lane;
    if (TRI) epi.put(m0 + r, n0 + c, t[min(r, c) * SMALL_LD + max(r, c)]);
    else epi.put(n0 + r, m0 + c, t[c * SMALL_LD + r]);
  }
}

// a tile of a product of two operands, 64 W wide
template <int W, class OPP, class OPQ, class STORE>
__device__ __forceinline__ void split_tile_full(const OPP& P, const OPQ& Q, int m0, int n0, int kbeg,
                                                int kend, float* smem, const STORE& store) {
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x & (SplitCfg<W>::NT - 1)) >> 6);
  const int wm = (wave >> 1) * 32 * W, wn = (wave & 1) * 32 * W;
  if constexpr (W == 1) {
    v16f acc[1];
    split_blocks<SmallTile>(P, Q, m0, n0, kbeg, kend, smem, SplitRows{{wm}, {wn}}, acc);
    const int row0[1] = {m0 + wm}, col0[1] = {n0 + wn}, what[1] = {BLK_PLAIN};
    store([&](const auto& epi) {
      if (epi.mirror) store_small<false>(acc[0], m0, n0, wm, wn, smem, epi);
      else store_blocks<1>(acc, row0, col0, what, epi);
    });
  } else {
    v16f acc[4];
    split_blocks<SplitTile>(P, Q, m0, n0, kbeg, kend, smem, SplitRows{{wm, wm + 32}, {wn, wn + 32}}, acc);
    const int row0[4] = {m0 + wm, m0 + wm, m0 + wm + 32, m0 + wm + 32};
    const int col0[4] = {n0 + wn, n0 + wn + 32, n0 + wn, n0 + wn + 32};
    const int what[4] = {BLK_PLAIN, BLK_PLAIN, BLK_PLAIN, BLK_PLAIN};
    store([&](const auto& epi) {
      if constexpr (imaging_epilogue<std::decay_t<decltype(epi)>>::value) {
        if (epi.mirror) {
          store_images<4>(acc, row0, col0, what, smem, epi);
          return;
        }
      }
      store_blocks<4>(acc, row0, col0, what, epi);
    });
  }
}

// a diagonal tile of a symmetric product: with `both`, the blocks above its diagonal are stored
// at their mirror positions too
template <int W, class OP, class STORE>
__device__ __forceinline__ void split_tile_tri(const OP& P, int m0, int kbeg, int kend, float* smem,
                                               bool both, const STORE& store) {
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x & (SplitCfg<W>::NT - 1)) >> 6);
  if constexpr (W == 1) {
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    v16f acc[1];
    split_blocks<SmallDiag>(P, P, m0, m0, kbeg, kend, smem, SplitRows{{wm, wn}, {}}, acc);
    // (both triangles, always)
    store([&](const auto& epi) { store_small<true>(acc[0], m0, m0, wm, wn, smem, epi); });
  } else {
    const SplitTri t = split_tri(wave);
    const int r0 = 32 * t.r[0], r1 = 32 * t.r[1], r2 = 32 * t.r[2];
    v16f acc[3];
    split_blocks<SplitDiag>(P, P, m0, m0, kbeg, kend, smem, SplitRows{{r0, r1, r2}, {}}, acc);
    const int row0[3] = {m0 + r0, m0 + r0, m0 + r1};
    const int col0[3] = {m0 + r1, m0 + r2, m0 + r1};
    const int what[3] = {BLK_PLAIN, t.r[0] == t.r[2] ? BLK_UPPER : BLK_PLAIN, t.last ? BLK_UPPER : BLK_NONE};
    store([&](const auto& epi) {
      if constexpr (imaging_epilogue<std::decay_t<decltype(epi)>>::value) {
        if (both) {
          store_images<3>(acc, row0, col0, what, smem, epi);
          return;
        }
      }
      store_blocks<3>(acc, row0, col0, what, epi);
    });
  }
}

// The tile (m0, n0) of the product, 128x128 on 256 threads; `same`: P and Q describe the same
// columns (a diagonal tile of a symmetric product, of which, without `both`, the 32x32 blocks
// below the diagonal are not written).
template <class OPP, class OPQ, class EPI>
__device__ __forceinline__ void split_tile(const OPP& P, const OPQ& Q, int m0, int n0, int kbeg,
                                           int kend, bool same, const EPI& epi, float* smem,
                                           bool both = true) {
  auto store = [&](auto&& put) { put(epi); };
  if constexpr (std::is_same<OPP, OPQ>::value) {
    if (same) {
      split_tile_tri<2>(P, m0, kbeg, kend, smem, both, store);
      return;
    }
  }
  split_tile_full<2>(P, Q, m0, n0, kbeg, kend, smem, store);
}

}  // namespace kfac
