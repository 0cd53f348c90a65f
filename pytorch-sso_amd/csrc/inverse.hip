// Batched damped SPD inverse:  dst_i = (src_i + damp_i * I)^-1  for a whole set
// of matrices of different sizes in one sequence of launches.
//
//   1. copy the upper triangle of src into dst and add damp to the diagonal
//      (damp is either given, or computed on the device from the traces of a
//      pair of Kronecker factors: the pi-damping split);
//   2. blocked right-looking Cholesky  S = U^T U  (upper, in place in dst) with
//      128-wide panels: one workgroup factors AND inverts the 128x128 diagonal
//      block in LDS; the row panel is a product with that small inverse; the
//      trailing update is a symmetric rank-128 product on the MFMA tile engine.
//      Panels are grouped: the rows of the current group receive each panel's
//      update in the launch that factors the next diagonal block (that block's
//      workgroup applies it to its own tile first, tile workgroups to the rest,
//      so that the chip is not idle while the latency-bound block is factored:
//      two launches per panel), the rows beyond the group receive the whole group
//      in one deeper product;
//   3. Y = U^-1 by recursive doubling over the 128-blocks:
//      Y12 = -Y11 * U12 * Y22, two MFMA products per level, log2(n/128) levels
//      (without the last one for a factor that may stay in two halves, see half_cut);
//   4. dst = Y Y^T on the MFMA tile engine (upper tiles, mirrored).
//   Batches whose tiles fit beside a diagonal block have steps 3 and 4 done by the launches of
//   step 2 (the sweep, potrf_step_kernel).
//
// Every launch covers all matrices that still have work at that step (matrices
// are processed in descending size order so the active ones form a prefix),
// so small factors ride along with the large ones instead of getting a launch
// sequence each.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <vector>

#include "common.h"
#include "diag_schedule.h"
#include "operands.h"

namespace kfac {

struct MatDesc {
  const float* src;
  float* U;      // Cholesky factor, then the inverse: dst (the workspace slot when only Y is wanted)
  float* Y;      // inverse of the Cholesky factor, n*n: the workspace slot, or the caller's
                 // buffer when Y itself is the result
  int n;
  int T;         // number of 128-blocks
  float damp;    // given damping, or sqrt(damping) in pi mode
  int partner;   // -1: damp is final; else index of the other factor of the pair
  int is_a;      // pi mode: 1 -> damp*pi, 0 -> damp/pi
  int out;       // position in the caller's info array
  float trace;
  int rev;       // 1: the work matrix is src with rows and columns reversed (see run_batched)
  float* W;      // rev only: receives the upper Cholesky factor of the inverse, else nullptr
  int noinv;     // 1: the explicit inverse is not wanted, Y is the result (Y Y^T = inverse)
  int cut;       // > 0 (with noinv): Y is left in two halves, cut in front of this block
};

constexpr int SETUP_CHUNK = 48;
struct DescChunk {
  MatDesc d[SETUP_CHUNK];
};

__global__ void inv_setup_kernel(DescChunk chunk, MatDesc* table, int offset, int count) {
  const int i = threadIdx.x;
  if (i < count) table[offset + i] = chunk.d[i];
}

// the same, with the trace of src (one workgroup per matrix)
__global__ __launch_bounds__(256) void inv_trace_kernel(const DescChunk chunk, MatDesc* table, int offset) {
  __shared__ float red[256];
  MatDesc m = chunk.d[blockIdx.x];
  const int n = m.n;
  float s = 0.f;
  for (int i = threadIdx.x; i < n; i += 256) s += m.src[(size_t)i * n + i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    m.trace = red[0];
    table[offset + blockIdx.x] = m;
  }
}

__device__ __forceinline__ float effective_damp(const MatDesc* table, const MatDesc& m) {
  if (m.partner < 0) return m.damp;
  const MatDesc& o = table[m.partner];
  const float ta = m.is_a ? m.trace / m.n : o.trace / o.n;
  const float tg = m.is_a ? o.trace / o.n : m.trace / m.n;
  const float pi = sqrtf(ta / tg);
  return m.is_a ? m.damp * pi : m.damp / pi;
}

// U = upper tiles of (src + damp I); also clears info.  A workgroup copies a quarter of a tile,
// in two rounds: a whole tile, in eight, left the copy of a few matrices waiting for
// eight round trips to memory (four 1000^2 ones: 18.7 -> 9.1 us).
constexpr int COPY_PARTS = 4;
__global__ __launch_bounds__(256) void inv_copy_damp_kernel(const MatDesc* table, int* info,
                                                            const WorkList wl) {
  int mat, local;
  work_find(wl, mat, local);
  const MatDesc m = table[mat];
  if (local == 0 && threadIdx.x == 0) info[m.out] = 0;
  int bi, bj;
  upper_tile(local / COPY_PARTS, m.T, bi, bj);
  const float damp = effective_damp(table, m);
  const int n = m.n;
  // 8 loads in flight per thread, then 8 stores
  constexpr int PART = BM * BN / COPY_PARTS;
  const int first = local % COPY_PARTS * PART;
  for (int e0 = first + threadIdx.x; e0 < first + PART; e0 += 256 * 8) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int e = e0 + 256 * k;
      const int row = bi * BM + (e >> 7);
      const int col = bj * BN + (e & 127);
      const size_t at = m.rev ? (size_t)(n - 1 - row) * n + (n - 1 - col) : (size_t)row * n + col;
      v[k] = (row < n && col < n) ? m.src[at] : 0.f;
      if (row == col) v[k] += damp;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int e = e0 + 256 * k;
      const int row = bi * BM + (e >> 7);
      const int col = bj * BN + (e & 127);
      if (row < n && col < n) m.U[(size_t)row * n + col] = v[k];
    }
  }
}

// ---------------------------------------------------------------------------
// 128x128 diagonal block: Cholesky (upper) and its inverse, in LDS.
// ---------------------------------------------------------------------------
constexpr int DB = 128;          // diagonal block size
constexpr int DLD = DB + 4;      // LDS leading dimension (rows of 16-byte pieces)
// S and Z; what the steps of the strips leave; the A operands of one strip; marks by strip and block
// column, and of the waves that applied a pending panel; write items taken
constexpr int DIAG_STEPS = 4 * 16 * 4;
constexpr int DIAG_OPS = 16 * 64;
constexpr int DIAG_MARKS = 4 * 8 * 8;
static_assert(PENDING_WAVES <= 16, "a mark for each");
constexpr int DIAG_SMEM_BYTES = (2 * DB * DLD + DIAG_STEPS + DIAG_OPS + DIAG_MARKS + 4) * (int)sizeof(float);

__device__ __forceinline__ float lane_value(float v, int src_lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), src_lane));
}

// One wave: acc(32x32) = sum_{k<K} A(k, i) * B(k, j) with operands in LDS,
//   A(k, i) = a[k*a_ks + i*a_is],  B(k, j) = b[k*b_ks + j*b_js]   (K a multiple of 32).
// Result element t of lane (r, h): row 8*(t/4) + 4h + t%4, column r.
__device__ __forceinline__ v16f lds_mma32(const lds_f* a, int a_ks, int a_is, const lds_f* b,
                                          int b_ks, int b_js, int K) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 31, h = lane >> 5;
  v16f acc;
#pragma unroll
  for (int t = 0; t < 16; ++t) acc[t] = 0.f;
  const lds_f* pa = a + h * a_ks + r * a_is;
  const lds_f* pb = b + h * b_ks + r * b_js;
  // 32 deep at a time: the 32 operand reads of a slice are issued together, and those of the
  // next slice before the 16 MFMAs of this one
  float av[16], bv[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    av[i] = pa[2 * i * a_ks];
    bv[i] = pb[2 * i * b_ks];
  }
  for (int k0 = 0; k0 < K; k0 += 32) {
    float an[16], bn[16];
    if (k0 + 32 < K) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        an[i] = pa[(k0 + 32 + 2 * i) * a_ks];
        bn[i] = pb[(k0 + 32 + 2 * i) * b_ks];
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], bv[i], acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      av[i] = an[i];
      bv[i] = bn[i];
    }
  }
  return acc;
}

// The elimination of a 32-row strip, two rows per step, on 32x32 blocks that live in the
// accumulator registers of v_mfma_f32_32x32x2_f32: element t of lane (r = lane & 31,
// h = lane >> 5) is (row 8*(t/4) + 4*h + t%4, column r), so row c of a block is ONE register
// (index 4*(c/8) + c%4) in the 32 lanes of half (c/4)%2, lane = column, and rows c, c+1
// (c even) are neighbouring registers in the same half.
//   L: the diagonal leaf, a full symmetric 32x32 block (Schur complement of the rows above),
//      held by the wave that leads the strip;
//   P: the same rows of another 32 columns (a block of the row panel, or of [ . | identity]),
//      held by a wave that follows.
// A step finishes rows c and c+1:  with the 2x2 pivot block [p00 p01; p01 p11] of L,
//   w0 = L[c] / sqrt(p00),  u01 = p01 / sqrt(p00),  w1 = (L[c+1] - u01 w0) / sqrt(p11 - u01^2)
// are rows c, c+1 of U (the same combination y0, y1 of P's rows: those rows of the second
// block), and the rows below get  X[i][j] -= w0[i] y0[j] + w1[i] y1[j]  as ONE rank-2 matrix
// instruction per block: its reduction slot 0 is the lanes 0-31 of the operand registers,
// slot 1 the lanes 32-63, so (w0 | w1) in the two halves of one register is the B operand
// (lane = column j) and, negated and zeroed in the lanes i <= c+1, the A operand (lane = row
// i; by the symmetry of L its rows are its columns).  Both rows live in one half, so one
// v_permlane32_swap moves the second into the other half; apart from that and the three
// pivot entries (v_readlane) no value changes lanes.  The chain from step to step is
//   matrix instruction -> pivots -> two 1/sqrt -> w1 -> swap -> matrix instruction.
// The leading wave does that and nothing else.  It leaves the finished rows in LDS, straight
// from the operand register, its A operand, and behind them the two 1/sqrt, u01 and a mark; the waves
// that follow read them, two steps ahead of their use, and end a few steps behind it.
// (One wave with the leaf and a second block took 280-400 cycles a step: the second block's
// instructions are not hidden behind the matrix instruction of the same wave.  Measured on one
// wave: the leading step 170, 210 with what it leaves as one 16-byte store, 186 as it is; the
// following one 122, and 190 with a matrix instruction of another accumulator in it.)
// LDS serves the requests of a wave in order, so whoever sees the mark sees the rows.
// Below its diagonal U_qq is left with rounding noise; whoever copies it out writes zeros instead.
// `pmin`, `piv`: the smallest pivot so far and all 32 of them, for the caller's check.
// With P = rows of the panel the strip ends as U[q][*] = U_qq^-T A[q][*] without a
// triangular solve; with P = [pending | identity] as the rows of U^-T.
template <int H>
__device__ __forceinline__ float pair_operand(float x0, float x1) {
  // both valid in the lanes of half H -> x0 in lanes 0-31, x1 in lanes 32-63
  // (the instruction swaps lanes 32-63 of its first register with lanes 0-31 of its second)
  const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x0),
                                                   __builtin_bit_cast(unsigned, x1), false, false);
  return __builtin_bit_cast(float, H ? sw[1] : sw[0]);
}

// What a step leaves for the waves that follow: {1/sqrt of its two pivots}, {u01, mark}, the mark
// behind everything else (volatile: in this order, and the loads in front of what they guard)
typedef float v2f __attribute__((ext_vector_type(2)));
typedef volatile __attribute__((address_space(3))) float lds_vf;
typedef volatile __attribute__((address_space(3))) v2f lds_vf2;

template <int C>
__device__ __forceinline__ void lead_from(v16f& L, lds_vf* rows, lds_vf* ops, lds_vf2* steps, int r,
                                          float& pmin, float (&piv)[32]) {
  if constexpr (C < 32) {
    constexpr int T = 4 * (C >> 3) + (C & 3), H = (C >> 2) & 1;
    const float v0 = L[T], v1 = L[T + 1];
    const float p00 = lane_value(v0, 32 * H + C);
    const float p01 = lane_value(v0, 32 * H + C + 1);
    const float p11 = lane_value(v1, 32 * H + C + 1);
    const float r0 = __builtin_amdgcn_rsqf(p00);
    const float u01 = p01 * r0;
    const float d = fmaf(-u01, u01, p11);
    const float r1 = __builtin_amdgcn_rsqf(d);
    const float w0 = v0 * r0;
    const float w1 = fmaf(-u01, w0, v1) * r1;
    const float xb = pair_operand<H>(w0, w1);
    const float xa = r > C + 1 ? -xb : 0.f;
    if (C < 30) L = __builtin_amdgcn_mfma_f32_32x32x2f32(xa, xb, L, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    // (the operand register holds row C in the lanes 0-31 and row C+1 in the lanes 32-63: one
    // store writes both, the pointer carries the lane's row and column)
    rows[C * DLD] = xb;
    ops[C / 2 * 64] = xa;
    steps[C] = v2f{r0, r1};
    steps[C + 1] = v2f{u01, 1.f};
    pmin = fminf(fminf(pmin, p00), d);
    piv[C] = p00;
    piv[C + 1] = d;
    __builtin_amdgcn_sched_barrier(0);
    lead_from<C + 2>(L, rows, ops, steps, r, pmin, piv);
  }
}

__device__ __forceinline__ bool is_marked(float mark) {
  return __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, mark)) != 0;
}

// What a following wave reads of two steps: the mark of the later one first
struct TwoSteps {
  v2f m1, s1, m0, s0;
  float x0, x1;
  __device__ __forceinline__ void read(const lds_vf* ops, const lds_vf2* steps) {
    m1 = steps[3];
    s1 = steps[2];
    m0 = steps[1];
    s0 = steps[0];
    x0 = ops[0];
    x1 = ops[64];
  }
  __device__ __forceinline__ bool ready() const { return is_marked(m1[1]); }
};

template <int C>
__device__ __forceinline__ void follow_step(v16f& P, const v2f& s, float u01, float x, lds_vf* rows) {
  constexpr int T = 4 * (C >> 3) + (C & 3), H = (C >> 2) & 1;
  const float y0 = P[T] * s[0];
  const float y1 = fmaf(-u01, y0, P[T + 1]) * s[1];
  const float pb = pair_operand<H>(y0, y1);
  if (C < 30) P = __builtin_amdgcn_mfma_f32_32x32x2f32(x, pb, P, 0, 0, 0);
  __builtin_amdgcn_sched_barrier(0);
  rows[C * DLD] = pb;
}

// `ops`, `steps`: the strip's; `rows`: where the rows of P go (the pointer carries the lane's row and
// column); `marks`: one for every two of its steps
template <int C>
__device__ __forceinline__ void follow_from(v16f& P, TwoSteps t, const lds_vf* ops,
                                            const lds_vf2* steps, lds_vf* rows, lds_vf* marks) {
  if constexpr (C < 32) {
    // (the leading wave takes all its steps whatever it finds, and waits for nobody)
    if (__builtin_expect(!t.ready(), 0)) {
      do t.read(ops + C / 2 * 64, steps + C);
      while (!t.ready());
    }
    // (a register of a load in flight that nobody uses would be given to the next load, which then
    // waits for the first)
    asm volatile("" :: "v"(t.m0));
    TwoSteps tn = t;
    if constexpr (C < 28) tn.read(ops + (C + 4) / 2 * 64, steps + C + 4);
    __builtin_amdgcn_sched_barrier(0);
    follow_step<C>(P, t.s0, t.m0[0], t.x0, rows);
    follow_step<C + 2>(P, t.s1, t.m1[0], t.x1, rows);
    marks[C / 4] = 1.f;
    __builtin_amdgcn_sched_barrier(0);
    follow_from<C + 4>(P, tn, ops, steps, rows, marks);
  }
}

// What strip q takes from a block of a strip below,  A^T B  with A and B blocks of strip q, while the
// waves that make their rows are at it: `a`, `b` (with the lane's row and column), two steps at a
// time behind their marks.  Those waves end, see follow_from.
struct Rows {
  const lds_vf *a, *b;
  const lds_vf *mark_a, *mark_b;
};
// One such product, or (TWO) two at a time.  The marks are read as one value, by lane, and tested
// at once.
template <bool TWO>
__device__ __forceinline__ void collect(v16f& N, const Rows r0, v16f& M, const Rows r1) {
  const lds_vf* mark = threadIdx.x & 1 ? r0.mark_b : r0.mark_a;
  if (TWO && (threadIdx.x & 2)) mark = threadIdx.x & 1 ? r1.mark_b : r1.mark_a;
  struct Step {
    float mark, a0, a1, b0, b1, c0, c1, d0, d1;
  };
  auto read = [&](int k) {
    Step x;
    const int at = 4 * k * DLD;
    x.mark = mark[k];
    x.a0 = r0.a[at];
    x.b0 = r0.b[at];
    x.a1 = r0.a[at + 2 * DLD];
    x.b1 = r0.b[at + 2 * DLD];
    x.c0 = x.c1 = x.d0 = x.d1 = 0.f;
    if (TWO) {
      x.c0 = r1.a[at];
      x.d0 = r1.b[at];
      x.c1 = r1.a[at + 2 * DLD];
      x.d1 = r1.b[at + 2 * DLD];
    }
    return x;
  };
  auto ready = [&](const Step& x) { return __builtin_amdgcn_ballot_w64(__builtin_bit_cast(int, x.mark) == 0) == 0; };
  Step t = read(0);
#pragma unroll
  for (int e = 0; e < 16; ++e) N[e] = 0.f;
  if (TWO) M = N;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (__builtin_expect(!ready(t), 0)) {
      do t = read(k);
      while (!ready(t));
    }
    const Step n = k < 7 ? read(k + 1) : t;
    __builtin_amdgcn_sched_barrier(0);
    N = __builtin_amdgcn_mfma_f32_32x32x2f32(t.a0, t.b0, N, 0, 0, 0);
    if (TWO) M = __builtin_amdgcn_mfma_f32_32x32x2f32(t.c0, t.d0, M, 0, 0, 0);
    N = __builtin_amdgcn_mfma_f32_32x32x2f32(t.a1, t.b1, N, 0, 0, 0);
    if (TWO) M = __builtin_amdgcn_mfma_f32_32x32x2f32(t.c1, t.d1, M, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    t = n;
  }
}

// Factors and inverts diagonal block p of matrix m: one workgroup of DIAG_THREADS threads
// (12 waves) with DIAG_SMEM_BYTES of LDS at dsm: S, the block (upper triangle and the whole
// diagonal 32-blocks; finished rows of U replace it strip by strip), and Z, the rows of
// U_pp^-T.
// Four strips of 32 rows, one barrier behind each.  Strip q has its leaf and four further blocks of
// the same rows: the blocks of the row panel to the right of the leaf, and the blocks of the
// same rows of Z (the last one starting as the identity).  The inverse Y_pp = Z^T is complete
// when the last strip is: no back substitution, no doubling.  What a strip takes from the rows
// below it goes
//   to strip q+1 while strip q is eliminated, by the waves that then have those blocks (COLLECT);
//   to the rows further down, in LDS, by the helping waves, in the strip before those rows' own.
// The finished rows of strip q are written to memory during strip q+1, by the collecting waves before they
// collect, in the last strip by those without a block.
// Bound by latency and, in the strips, by the issue of a SIMD's matrix core and vector unit, which take
// turns: the steps of a strip take the leading wave 200 cycles each where nothing else is on its
// SIMD.  One block alone 17.5 -> 15.8 us, with the pending panel 22.1 -> 19.5, the inverse of a 2305^2 matrix
// and its Cholesky factor 1166 -> 1075 (with the helping waves and the writes at the end of the strip that they
// belong to); before that 21.0 -> 17.1 and 26.1 -> 21.2 (four waves that each
// held the leaf and a second block, three barriers a strip, the pending panel on the fp32 instructions, 4-byte
// accesses to memory); the inverse of a 2305^2 matrix and its Cholesky factor 1333 -> 1160 us.
constexpr int DIAG_THREADS = 64 * DIAG_WAVES;
typedef SplitChunk<DB> PendingGroup;                       // (HALF: 8 k of 128 columns)
constexpr int PENDING_PLANE = 8 * PendingGroup::HALF;      // 64 k
static_assert(3 * PENDING_PLANE <= (DB - PENDING_ROW0) * DLD * (int)sizeof(float), "half of W lives in the LDS of Z");

// `pending`: the row panel above (block row p-1) has not been applied to this block yet
// (the launch that holds this workgroup applies it to the rest of block row p meanwhile).
__device__ __forceinline__ void diag_block(const MatDesc& m, int p, int* info, float* dsm,
                                           bool pending) {
  lds_f* const S = (lds_f*)dsm;
  lds_f* const Z = S + DB * DLD;
  lds_f* const steps = Z + DB * DLD;
  lds_f* const ops = steps + DIAG_STEPS;
  lds_f* const marks = ops + DIAG_OPS;
  typedef __attribute__((address_space(3))) int lds_i;
  lds_i* const taken = (lds_i*)(marks + DIAG_MARKS);
  const int n = m.n;
  const int r0 = p * DB;
  const int nb = min(DB, n - r0);
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);     // (provably uniform: scalar branches)
  const int lane = t & 63;
  const int r = lane & 31, h = lane >> 5;
  if (t < DIAG_STEPS) steps[t] = 0.f;
  if (t < DIAG_MARKS) marks[t] = 0.f;
  if (t == 0) *taken = 0;

  // pending: W, tile (p-1, p) of U, all of its 128 rows, in the same round trip as the block; 8
  // consecutive k of one column a piece, wave by wave
  constexpr int WGROUPS = (DB * DB / 8 + DIAG_THREADS - 1) / DIAG_THREADS;
  float w[WGROUPS][8];
  auto wgroup = [&](int g) { return (wave >> 1) + DIAG_THREADS / DB * g; };      // of 8 k

  // load the upper triangle, by 32-blocks; pad with the identity up to 128.  All loads of a thread
  // are issued before the first is used: one memory round trip for the block.  (What lies
  // below the diagonal inside a diagonal 32-block is nobody's value and stays unread.)
  {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(m.U + (size_t)r0 * n + r0);
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(m.U + ((size_t)r0 - DB) * n + r0);
    constexpr int ROWS = DIAG_THREADS / 32, PER = (DB + ROWS - 1) / ROWS;
    const int j = 4 * (t & 31);
    v4f v[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = u * ROWS + (t >> 5);
      const unsigned at = (unsigned)(i * n + j) * 4u;
      const bool in = i < nb && j >= (i & ~31);
      if (nb - j >= 4 || nb <= j) {
        v[u] = buffer_load4(rs, in && j < nb ? at : INV_M);
      } else {
        // (the last columns of the matrix: nothing is read behind its end)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[u][e] = buffer_load(rs, in && j + e < nb ? at + 4 * e : INV_M);
      }
    }
    if (pending) {
      const unsigned col = t % DB < nb ? 4u * (t % DB) : INV_M;
#pragma unroll
      for (int g = 0; g < WGROUPS; ++g)
#pragma unroll
        for (int k = 0; k < 8; ++k)
          w[g][k] = buffer_load_at(ra, wgroup(g) < DB / 8 ? col : INV_M, 4u * n * (8 * wgroup(g) + k));
    }
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = u * ROWS + (t >> 5);
      if (i >= DB) break;
      if (i >= nb) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[u][e] = i == j + e ? 1.f : 0.f;
      }
      *(lds_f4*)(S + i * DLD + j) = v[u];
    }
  }
  // S -= W^T W, split into bf16 parts as in gemm_split.h, half of the reduction after the other in
  // the LDS of Z, a 32x32 block of S on each of ten waves; no barrier behind it but the one that ends the
  // first strip: pending_row etc. say why.
  // (Eight of the nine partial products, as good as the fp32 instructions.  The ends of the range do
  // not matter here: W is part of a Cholesky factor, so the sum of the squares of a column is at most the
  // diagonal entry below it.  No element is above 2^64; what one below 2^-108 loses, 2^-133 times the
  // other column, is below the rounding 2^-24 sqrt(S_ii S_jj) of the entry it goes to wherever S_ii is a
  // float32 that is not zero; and halves of the elements keep leading sums finite that are rounded up from
  // near the largest float32.)
  if (pending) {
    v16f acc, cor;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = cor[e] = 0.f;
    // (behind the first rows of Z, which the first strip writes)
    lds_c* const planes = (lds_c*)(Z + PENDING_ROW0 * DLD);
    const int bi = pending_row(wave), bj = pending_col(wave);
    v4u ph[WGROUPS], pm[WGROUPS], pl[WGROUPS];
    // the pieces of one half of the reduction, split (the second half's under the first's products)
    auto split_half = [&](int half) {
#pragma unroll
      for (int g = 0; g < WGROUPS; ++g) {
        if (wgroup(g) >> 3 != half) continue;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          unsigned x, y, z;
          split_pair(0.5f * w[g][2 * k], 0.5f * w[g][2 * k + 1], x, y, z);
          ph[g][k] = x;
          pm[g][k] = y;
          pl[g][k] = z;
        }
      }
    };
    if (wave < 4) __builtin_amdgcn_s_setprio(3);
    split_half(0);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (half) __syncthreads();          // (the first half has been read)
#pragma unroll
      for (int g = 0; g < WGROUPS; ++g) {
        if (wgroup(g) >> 3 != half) continue;
        lds_c* const at = planes + (wgroup(g) & 7) * PendingGroup::HALF + (t % DB) * 16;
        *(lds_u4*)at = ph[g];
        *(lds_u4*)(at + PENDING_PLANE) = pm[g];
        *(lds_u4*)(at + 2 * PENDING_PLANE) = pl[g];
      }
      __syncthreads();
      if (wave < PENDING_WAVES) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          v8bf a[3], b[3];
#pragma unroll
          for (int part = 0; part < 3; ++part) {
            const lds_c* const at = planes + part * PENDING_PLANE + (2 * ks + h) * PendingGroup::HALF + r * 16;
            a[part] = __builtin_bit_cast(v8bf, *(const lds_u4*)(at + 32 * bi * 16));
            b[part] = __builtin_bit_cast(v8bf, *(const lds_u4*)(at + 32 * bj * 16));
          }
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
          cor = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], cor, 0, 0, 0);
          cor = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], cor, 0, 0, 0);
          cor = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], cor, 0, 0, 0);
          cor = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[2], cor, 0, 0, 0);
          cor = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[0], cor, 0, 0, 0);
          cor = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[2], cor, 0, 0, 0);
          cor = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[1], cor, 0, 0, 0);
        }
      }
      if (half == 0) split_half(1);
    }
    if (wave < PENDING_WAVES) {
      add_corrections(acc, cor);
      lds_f* const at = S + (32 * bi + 4 * h) * DLD + 32 * bj + r;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        lds_f* const s = at + (8 * (e >> 2) + (e & 3)) * DLD;
        *s = fmaf(-4.f, acc[e], *s);
      }
    }
  } else {
    __syncthreads();
  }
  v16f N;              // what the strip above takes from this wave's block
#pragma unroll
  for (int e = 0; e < 16; ++e) N[e] = 0.f;

  typedef __attribute__((address_space(1))) float global_f;
  typedef __attribute__((address_space(1), aligned(4))) v4f global_f4;
  global_f* const gU = (global_f*)(m.U + (size_t)r0 * n + r0);
  global_f* const gY = (global_f*)(m.Y + (size_t)r0 * n + r0);
  // rows [32 qs, 32 qs + 32) of U and the same columns of Y = Z^T, a sixteenth of them
  constexpr int WRITE_ITEMS = 16;
  auto write_item = [&](int qs, int item) {
    const int e = 64 * item + lane;
    const int iu = 32 * qs + (e >> 5), ju = 4 * (e & 31);      // U[iu][ju ...]
    const int iy = e >> 3, jy = 32 * qs + 4 * (e & 7);         // Y[iy][jy ...] = Z[jy ...][iy]
    v4f u = *(const lds_f4*)(S + iu * DLD + ju), y;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      y[i] = Z[(jy + i) * DLD + iy];
      u[i] = iu <= ju + i ? u[i] : 0.f;
      y[i] = iy <= jy + i ? y[i] : 0.f;
    }
    auto put = [&](global_f* row, int col, const v4f& x) {
      if (col + 4 <= nb) {
        *(global_f4*)(row + col) = x;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (col + i < nb) row[col + i] = x[i];
      }
    };
    if (iu < nb) put(gU + iu * n, ju, u);
    if (iy < nb) put(gY + iy * n, jy, y);
  };

  const int nq = (nb + 31) / 32;
  // Element (8*(e/4) + 4h + e%4, r) of block (i, col) of S, or of Z
  auto block_at = [&](bool in_s, int i, int col) {
    return (in_s ? S : Z) + (32 * i + 4 * h) * DLD + 32 * col + r;
  };
  for (int q = 0; q < nq; ++q) {
    const int c0 = 32 * q;
    const unsigned long long roles = q == 0 ? STRIP_ROLES[0] : q == 1 ? STRIP_ROLES[1]
                                   : q == 2 ? STRIP_ROLES[2] : STRIP_ROLES[3];
    const int code = (int)(roles >> (5 * wave)) & 31;
    const int c = code & 7;
    const bool in_s = c < 4;
    const bool there = in_s ? c < nq : c - 4 <= q;        // (a matrix may end in this block)
    // first row of a strip (of this one) in block column k, with the lane's row and column
    auto rows_in = [&](int strip, int k) {
      return (lds_vf*)((k < 4 ? S : Z) + (32 * strip + h) * DLD + 32 * (k & 3) + r);
    };
    auto marks_in = [&](int strip, int k) { return (lds_vf*)(marks + (8 * strip + k) * 8); };
    auto rows_at = [&](int k) { return rows_in(q, k); };
    auto marks_at = [&](int k) { return marks_in(q, k); };
    lds_vf2* const step = (lds_vf2*)(steps + 64 * q);
    lds_vf* const op = (lds_vf*)(ops + lane);
    if (code == 1) {
      __builtin_amdgcn_s_setprio(3);
      // (the lane's column made opaque, so that the lane masks derived from it are computed
      // where they are used instead of being kept, and spilled, across the loop over the strips)
      int rr = r;
      asm volatile("" : "+v"(rr));
      v16f L;
      // (the leaf in full, what lies below its diagonal from above it)
      const lds_f* const src = S + c0 * DLD + c0;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = 8 * (e >> 2) + 4 * h + (e & 3);
        L[e] = src[row <= rr ? row * DLD + rr : rr * DLD + row] - N[e];
      }
      float pmin = 1.f, piv[32];
      lead_from<0>(L, rows_at(q), op, step, rr, pmin, piv);
      // LAPACK's info: the first pivot that is not positive.  A NaN anywhere in the leaf
      // reaches a pivot and from there every later one, so the last pivot stands for them.
      if (!(pmin > 0.f) || !(piv[31] > 0.f)) {
        int bad = 0;
#pragma unroll
        for (int i = 31; i >= 0; --i)
          if (!(piv[i] > 0.f)) bad = r0 + c0 + i + 1;
        int* const out = info + m.out;
        if (lane == 0 && *out == 0) *out = bad;
      }
    } else if (code >= 16) {
      __builtin_amdgcn_s_setprio(1);
      // the rows of the strip above to memory first, a quarter each: what is to be collected comes later
      if (q > 0) {
#pragma unroll
        for (int k = 0; k < 4; ++k) write_item(q - 1, 4 * (c - q - 1) + k);
      }
      const Rows from{rows_at(q + 1), rows_at(c), marks_at(q + 1), marks_at(c)};
      if (there && q + 1 < nq) collect<false>(N, from, N, from);
    } else if (code >= 8) {
      __builtin_amdgcn_s_setprio(2);
      if (there) {
        v16f P;
        if (!in_s && c - 4 == q) {
#pragma unroll
          for (int e = 0; e < 16; ++e) P[e] = 8 * (e >> 2) + 4 * h + (e & 3) == r ? 1.f : 0.f;
        } else {
          // (a block of Z below the diagonal starts at zero: the strip of its column is the
          // first to update it, and finds it uninitialised)
          const bool fresh = !in_s && c - 4 == q - 1;
          const lds_f* const src = block_at(in_s, q, c & 3);
#pragma unroll
          for (int e = 0; e < 16; ++e)
            P[e] = (fresh ? 0.f : src[(8 * (e >> 2) + (e & 3)) * DLD]) - N[e];
        }
        TwoSteps none;
        none.m1 = none.s1 = none.m0 = none.s0 = v2f{0.f, 0.f};
        none.x0 = none.x1 = 0.f;
        follow_from<0>(P, none, op, step, rows_at(c), marks_at(c));
      }
    } else if (code >= 2) {
      __builtin_amdgcn_s_setprio(0);
      // what the strips above this one take from a block of the next one (their rows are all there)
      int i = 0, col = 0;
      if (q > 0)
        helped_blocks(q - 1, nq, code - 2, [&](int row, int c) {
          i = row == q + 1 ? row : i;
          col = row == q + 1 ? c : col;
        });
      auto rows_of = [&](int strip) {
        return Rows{rows_in(strip, i), rows_in(strip, col), marks_in(strip, i), marks_in(strip, col)};
      };
      auto apply = [&](const v16f& x) {
        lds_f* const at = block_at(col < 4, i, col & 3);
        // (a block of Z below the diagonal starts at zero, and finds it uninitialised)
        float old[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) old[e] = col < 4 ? at[(8 * (e >> 2) + (e & 3)) * DLD] : 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) at[(8 * (e >> 2) + (e & 3)) * DLD] = old[e] - x[e];
      };
      if (i > 0 && helped_from(col) < q - 1) {
        v16f x, y;
        collect<true>(x, rows_of(q - 1), y, rows_of(q - 2));
        x += y;
        apply(x);
      } else if (i > 0) {
        v16f x;
        collect<false>(x, rows_of(q - 1), x, rows_of(q - 1));
        apply(x);
      }
    }
    // (in the last strip of a whole block, which nobody collects from, by the waves without a block)
    if (q == 3 && code < 8 && code != 1) {
      for (;;) {
        int item = 0;
        if (lane == 0)
          item = __hip_atomic_fetch_add(taken, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        item = __builtin_amdgcn_readfirstlane(item);
        if (item >= WRITE_ITEMS) break;
        write_item(q - 1, item);
      }
    }
    __syncthreads();
  }
  __builtin_amdgcn_s_setprio(0);
  for (int item = wave; item < WRITE_ITEMS; item += DIAG_THREADS / 64) write_item(nq - 1, item);
}

__global__ __launch_bounds__(DIAG_THREADS) void potrf_diag_kernel(const MatDesc* table, int p,
                                                                   int* info) {
  extern __shared__ __attribute__((aligned(16))) float dsm[];
  diag_block(table[blockIdx.x], p, info, dsm, false);
}

// row panel of the blocked Cholesky: U[p, j] = Ypp^T * A[p, j], j > p
__global__ __launch_bounds__(NTHREADS, 2) void potrf_panel_kernel(const MatDesc* table, int p,
                                                               const WorkList wl) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  int mat, local;
  work_find(wl, mat, local);
  const MatDesc m = table[mat];
  const int bj = p + 1 + local;
  if (bj >= m.T) return;
  const int n = m.n;
  const int r0 = p * DB;
  DenseKM P{m.Y + (size_t)r0 * n + r0, nullptr, n, DB, 0};
  DenseKM Q{m.U + (size_t)r0 * n, nullptr, n, n, 0};
  EpiStore epi{m.U + (size_t)r0 * n, n, DB, n, 1.f, 0.f, false};
  split_tile(P, Q, 0, bj * BN, 0, DB, false, epi, smem);
}

// Tile (bi <= bj) number `local` of the trailing update of block rows [row_lo, row_hi).
__device__ __forceinline__ bool trail_tile(int T, int row_lo, int row_hi, int local, int& bi,
                                           int& bj) {
  const int hi = min(row_hi, T);
  if (row_lo >= hi) return false;
  if (row_hi >= T) {
    // all remaining rows: walk the upper triangle of the (T - row_lo)^2 block grid
    const int Tr = T - row_lo;
    if (local >= Tr * (Tr + 1) / 2) return false;
    upper_tile(xcd_remap(local, Tr * (Tr + 1) / 2), Tr, bi, bj);
    bi += row_lo;
    bj += row_lo;
    return true;
  }
  // a few rows: rectangular walk, tiles left of the diagonal exit
  const int width = T - row_lo;
  const int rr = local / width;
  bi = row_lo + rr;
  bj = row_lo + (local - rr * width);
  return bi < hi && bj >= bi;
}

// trailing update with the block rows [kb0, kb0 + nk) of U:
//   A[i, j] -= sum_k U[k, i]^T U[k, j]   for block rows row_lo <= i < row_hi, j >= i.
// The Cholesky runs in groups of GROUP_BLOCKS diagonal blocks: inside a group each step
// updates only the remaining rows of that group (nk = 1), and the rows beyond it receive
// the whole group at once (nk = GROUP_BLOCKS), which cuts the read-modify-write passes over
// the trailing matrix by that factor (a rank-128 update of a large trailing matrix is
// bound by memory traffic, not by the matrix cores).  Taller groups cost the factors of a ResNet-50
// more than they bring to larger matrices (height 4 / 6 / 8: 4.67 / 4.83 / 4.88 ms; 9217 / 4097 / 4097
// and smaller 9.35 / 9.21 / 9.45), and accuracy: on the fp32 tile engine the error of the
// inverse of a 9217^2 factor with condition number 9e2 grew from 2.2e-5 (height 1) over
// 5.2e-5 (4; scipy's float32 LU inverse: 4.7e-5) to 1.0e-4 (16), because a deeper product
// accumulates more terms before it meets the entry it nearly cancels.
constexpr int GROUP_BLOCKS = 4;
// The last TAIL_BLOCKS diagonal blocks of the largest matrices form one group: the deeper
// update of the rows beyond a group is a launch that lasts as long as one 512-deep tile
// however few tiles it has, while the rank-128 updates of a short trailing matrix
// fit beside the next diagonal block.  16 / 24 / 32 / 40: the factors of a ResNet-50 4.60 / 4.67 /
// 4.96 / 5.42 ms, matrices of 9217 / 4097 / 4097 and smaller 9.38 / 9.35 / 9.25 / 9.28, the Cholesky factor of
// 3500^2 0.94 / 0.89 / 0.87 / 0.87.
constexpr int TAIL_BLOCKS = 24;

__global__ __launch_bounds__(NTHREADS, 2) void potrf_trail_kernel(const MatDesc* table, int kb0,
                                                               int nk, int row_lo, int row_hi,
                                                               const WorkList wl) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  int mat, local;
  work_find(wl, mat, local);
  const MatDesc m = table[mat];
  int bi, bj;
  if (!trail_tile(m.T, row_lo, row_hi, local, bi, bj)) return;
  const int n = m.n;
  DenseKM P{m.U + (size_t)kb0 * DB * n, nullptr, n, n, 0};
  EpiStore epi{m.U, n, n, n, -1.f, 1.f, false};
  // (nobody reads U below its diagonal)
  split_tile(P, P, bi * BM, bj * BN, 0, nk * DB, bi == bj, epi, smem, false);
}

// One 128x128 tile of a rank-128 update beside a diagonal block, by the first 8 waves of the
// workgroup (64x32 per wave):  C[m][n] = beta C + sign * sum_k P(k, m) Q(k, n), k < depth <= 128.
// Such a tile is alone on its compute unit (the launch carries the diagonal block's LDS), so
// it is a chain of latencies: memory -> split -> LDS -> matrix instructions -> memory.  The
// operands come in two halves of 64 k, split into bf16 parts as in gemm_split.h; the whole
// first half is in flight at once, the second under the products of the first, and C's old
// values under those of the second.  A workgroup takes one tile after the other.
// Bound by memory where every unit has one: 128 KB of C and up to 128 KB of operands per tile,
// 11 us each with 510 tiles in a launch (the fp32 tile engine, three tiles to a workgroup:
// 19 us).  Inverse of a 2900^2 / 3500^2 / 4600^2 matrix 1121 -> 920 / 1367 -> 1124 /
// 2177 -> 1922 us, and 2.5 times closer to float64 (6.7e-5 -> 2.7e-5 at 2900).
// PMK / QMK: the operand has consecutive k next to each other (P(k, m) = p[m n + k]) instead of
// consecutive m (p[k n + m]).
// `fresh`: there are no old values (OLD false: known at compile time).
// `upper`: only elements on and above the diagonal of C are stored, with `mirror` at their
// mirror positions too (a tile on the diagonal is symmetric except for rounding).
constexpr int STEP_THREADS = 512;
typedef SplitChunk<128> StepGroup;                  // (HALF: 8 k of 128 rows)
constexpr int STEP_PLANE = 8 * StepGroup::HALF;     // 64 k
constexpr int STEP_OPERAND = 3 * STEP_PLANE;
static_assert(2 * STEP_OPERAND <= DIAG_SMEM_BYTES, "a tile lives in the diagonal block's LDS");

template <bool MKL>
struct StepOperand {
  const float* p;
  int n, m0, depth;
  float v[16];
  // k in [64 half, 64 half + 64): 16 elements per thread
  __device__ __forceinline__ void load(int half) {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(p);
    const int t = threadIdx.x;
    if constexpr (MKL) {
      const int k = 64 * half + 4 * (t & 15);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + (t >> 4) + 32 * i;
        const unsigned off = (unsigned)(m * n + k) * 4u;
        if (depth == DB) {
          const v4f x = buffer_load4(rs, m < n ? off : INV_M);
#pragma unroll
          for (int j = 0; j < 4; ++j) v[4 * i + j] = x[j];
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            v[4 * i + j] = buffer_load(rs, m < n && k + j < depth ? off + 4 * j : INV_M);
        }
      }
    } else {
      const int m = m0 + (t & 127);
      const int k = 64 * half + 8 * __builtin_amdgcn_readfirstlane(t >> 7);
      const unsigned off = m < n ? (unsigned)m * 4u : INV_M;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          // (no branch around the load: what is done with its value would move in there, and wait for it)
          const int at = k + 32 * i + j;
          const bool in = depth == DB || at < depth;
          v[8 * i + j] = buffer_load_at(rs, in ? off : INV_M, in ? (unsigned)(at * n) * 4u : 0u);
        }
    }
  }
  // (SCALED: multiplied by SMALL_SCALE)
  template <bool SCALED>
  __device__ __forceinline__ void commit(lds_c* at) {
    const int t = threadIdx.x;
    const float f = SCALED ? SMALL_SCALE : 1.f;
    if constexpr (MKL) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v2u h, m, l;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          unsigned a, b, c;
          split_pair(v[4 * i + 2 * j] * f, v[4 * i + 2 * j + 1] * f, a, b, c);
          h[j] = a;
          m[j] = b;
          l[j] = c;
        }
        lds_c* const o = at + ((t & 15) >> 1) * StepGroup::HALF + ((t >> 4) + 32 * i) * 16 + (t & 1) * 8;
        *(lds_u2*)o = h;
        *(lds_u2*)(o + STEP_PLANE) = m;
        *(lds_u2*)(o + 2 * STEP_PLANE) = l;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        v4u h, m, l;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          unsigned a, b, c;
          split_pair(v[8 * i + 2 * j] * f, v[8 * i + 2 * j + 1] * f, a, b, c);
          h[j] = a;
          m[j] = b;
          l[j] = c;
        }
        lds_c* const o = at + ((t >> 7) + 4 * i) * StepGroup::HALF + (t & 127) * 16;
        *(lds_u4*)o = h;
        *(lds_u4*)(o + STEP_PLANE) = m;
        *(lds_u4*)(o + 2 * STEP_PLANE) = l;
        if (SCALED) __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
};

// Without old values (the row panels) a tile is as good as the fp32 instructions that it replaces, as a 64-wide one
// of gemm_split.h is and in the same ways: eight of the nine partial products, elements multiplied by
// 2^24 before they are split, and where a sum is then not finite, the tile on the fp32 instructions.
constexpr int STEP_VOTES = 2 * STEP_OPERAND;        // a word per wave

// C[m][n] of a wave's two 32x32 blocks at (m0, n0) and (m0 + 32, n0), k < depth, straight from memory
// (consecutive m and n)
__device__ __forceinline__ void step_fp32(const float* p, const float* q, int n, int m0, int n0, int depth,
                                          v16f (&acc)[2]) {
  const __amdgpu_buffer_rsrc_t rp = make_rsrc(p), rq = make_rsrc(q);
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;
#pragma unroll 1
  for (int k0 = 0; k0 < DB; k0 += 2) {
    const int k = k0 + h;
    const unsigned row = (unsigned)(k * n) * 4u;
    const float b = buffer_load(rq, k < depth && n0 + r < n ? row + 4u * (n0 + r) : INV_M);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int m = m0 + 32 * i + r;
      const float a = buffer_load(rp, k < depth && m < n ? row + 4u * m : INV_M);
      acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[i], 0, 0, 0);
    }
  }
}

template <bool PMK, bool QMK, bool OLD = true>
__device__ __forceinline__ void step_tile(const float* p, const float* q, float* C, int n, int m0,
                                          int n0, int depth, float sign, bool fresh, bool upper,
                                          bool mirror, lds_c* sm) {
  StepOperand<PMK> P{p, n, m0, depth};
  StepOperand<QMK> Q{q, n, n0, depth};
  lds_c* const sq = sm + STEP_OPERAND;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wm = (wave & 1) * 64, wn = (wave >> 1) * 32;
  v16f acc[2], cor[2];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[b][e] = cor[b][e] = 0.f;
  auto products = [&]() {
#pragma unroll 1
    for (int ks = 0; ks < 4; ++ks) {
      v8bf a[3][2], b[3];
      const lds_c* const at = sm + (2 * ks + h) * StepGroup::HALF + r * 16;
      auto load_a = [&](int i) {
#pragma unroll
        for (int pl = 0; pl < 3; ++pl)
          a[pl][i] = __builtin_bit_cast(v8bf, *(const lds_u4*)(at + pl * STEP_PLANE + (wm + 32 * i) * 16));
      };
#pragma unroll
      for (int pl = 0; pl < 3; ++pl)
        b[pl] = __builtin_bit_cast(v8bf, *(const lds_u4*)(at + pl * STEP_PLANE + STEP_OPERAND + wn * 16));
      load_a(0);
      if (OLD) load_a(1);
      auto product = [&](auto prod_, int i) {
        constexpr int PR = decltype(prod_)::value;
        constexpr int PA = PR == 2 || PR == 3 || PR == 6 ? 1 : PR == 5 || PR == 7 ? 2 : 0;
        constexpr int PB = PR == 1 || PR == 3 || PR == 7 ? 1 : PR == 4 || PR == 6 ? 2 : 0;
        v16f& x = PR == 0 ? acc[i] : cor[i];
        x = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[PA][i], b[PB], x, 0, 0, 0);
      };
      if constexpr (OLD) {
        static_for<6>([&](auto prod_) {
          product(prod_, 0);
          product(prod_, 1);
        });
      } else {
        // (one block after the other: the operands of both, eight products each, do not fit beside the half in flight)
        static_for<8>([&](auto prod_) { product(prod_, 0); });
        __builtin_amdgcn_sched_barrier(0);
        load_a(1);
        static_for<8>([&](auto prod_) { product(prod_, 1); });
      }
    }
  };
  P.load(0);
  Q.load(0);
  P.template commit<!OLD>(sm);
  Q.template commit<!OLD>(sq);
  P.load(1);
  Q.load(1);
  __syncthreads();
  products();
  __syncthreads();
  P.template commit<!OLD>(sm);
  Q.template commit<!OLD>(sq);
  const __amdgpu_buffer_rsrc_t rc = make_rsrc(C);
  const int col = n0 + wn + r;
  float old[2][16];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int row = m0 + wm + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
      const bool in = !fresh && row < n && col < n && (!upper || row <= col);
      old[i][e] = OLD ? buffer_load(rc, in ? (unsigned)(row * n + col) * 4u : INV_M) : 0.f;
    }
  __syncthreads();
  products();
  if constexpr (!OLD) {
    static_assert(!PMK && !QMK, "step_fp32 reads consecutive m and n");
    float probe = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[i][e] += cor[i][e];
        probe = fmaf(acc[i][e], 0.f, probe);
      }
    lds_u* const votes = (lds_u*)(sm + STEP_VOTES);
    votes[wave] = __builtin_amdgcn_ballot_w64(probe != 0.f) != 0;
    __syncthreads();
    unsigned any = 0;
#pragma unroll
    for (int w = 0; w < STEP_THREADS / 64; ++w) any |= votes[w];
    if (__builtin_expect(__builtin_amdgcn_readfirstlane((int)any) != 0, 0)) {
      step_fp32(p, q, n, m0 + wm, n0 + wn, depth, acc);
      __syncthreads();     // (a panel overwrites its own operand)
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i] *= 1.f / (SMALL_SCALE * SMALL_SCALE);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (OLD) add_corrections(acc[i], cor[i]);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int row = m0 + wm + 32 * i + 8 * (e >> 2) + 4 * h + (e & 3);
      if (row < n && col < n && (!upper || row <= col)) {
        const float v = fmaf(sign, acc[i][e], old[i][e]);
        C[(size_t)row * n + col] = v;
        if (mirror && row < col) C[(size_t)col * n + row] = v;
      }
    }
  }
  __syncthreads();       // (the next tile overwrites the operands)
}

// Diagonal blocks p and, beside them, the part of panel p-1's update that nothing needs
// before the next row panel:   A[i,j] -= U[p-1,i]^T U[p-1,j]   for block rows
// row_lo <= i < row_hi (row_lo = p + 1: row p got its update in a launch of its own).
// The first `ndiag` workgroups take one diagonal block each (potrf_diag_kernel's work).  The
// launch carries the diagonal block's LDS, so one workgroup runs per CU: the others use the
// CUs that the few diagonal blocks leave idle, for about as long as a diagonal block takes,
// and where there are more tiles than such CUs they walk the list of tiles.
//
// SWEEP: the whole inversion rides in these launches (see use_sweep).  With Z = U^-T, whose
// rows obey  Z[i] = Y_ii^T (I[i] - sum_{k < i} U[k,i]^T Z[k]),  and X = Z^T Z the inverse, the
// launch of diagonal block p applies block row k = p - 1 of U and Z to everything:
//   A[i,j] -= U[k,i]^T U[k,j]   p <= i <= j        (T - p)(T - p + 1) / 2 tiles
//   Z[i,j] -= U[k,i]^T Z[k,j]   p <= i, j <= k     (T - p) p
//   X[i,j] += Z[k,i]^T Z[k,j]   i <= j <= k        p (p + 1) / 2
// about T^2 / 2 tiles at every p, and the launch of p = T finishes X.  A finished row of Z lies
// in column k of Y (Y = Z^T), a pending one below Y's diagonal; X grows in the columns of U
// that no later step reads.
__host__ __device__ inline int sweep_items(int T, int p, bool x) {
  if (p > T) return 0;
  const int Tr = T - p;
  return Tr * (Tr + 1) / 2 + Tr * p + (x ? p * (p + 1) / 2 : 0);
}

__device__ __forceinline__ void sweep_tile(const MatDesc& m, int p, int local, lds_c* sm) {
  const int n = m.n, Tr = m.T - p, k0 = (p - 1) * DB;
  const int nA = Tr * (Tr + 1) / 2;
  const float* const uk = m.U + (size_t)k0 * n;
  const float* const zk = m.Y + k0;
  int bi, bj;
  if (local < nA) {
    upper_tile(xcd_remap(local, nA), Tr, bi, bj);
    if (bj == 0) return;                     // tile (p, p): the diagonal block's own workgroup
    bi += p;
    bj += p;
    step_tile<false, false>(uk, uk, m.U, n, bi * BM, bj * BN, DB, -1.f, false, true, false, sm);
  } else if (local < nA + Tr * p) {
    const int at = xcd_remap(local - nA, Tr * p);
    bi = at / p;
    bj = at - bi * p;
    bi += p;
    // (column p - 1 of these rows meets its first update: what lies there is not a value yet)
    step_tile<false, true>(uk, zk, m.Y, n, bi * BM, bj * BN, DB, -1.f, bj == p - 1, false, false, sm);
  } else {
    upper_tile(xcd_remap(local - nA - Tr * p, p * (p + 1) / 2), p, bi, bj);
    step_tile<true, true>(zk, zk, m.U, n, bi * BM, bj * BN, min(DB, n - k0), 1.f, bj == p - 1, true,
                          p == m.T, sm);
  }
}

template <bool SWEEP>
__global__ __launch_bounds__(DIAG_THREADS) void potrf_step_kernel(const MatDesc* table, int p,
                                                                   int* info, int ndiag,
                                                                   int row_lo, int row_hi,
                                                                   const WorkList wl) {
  extern __shared__ __attribute__((aligned(16))) float dsm[];
  if ((int)blockIdx.x < ndiag) {
    diag_block(table[blockIdx.x], p, info, dsm, true);
    return;
  }
  if (threadIdx.x >= STEP_THREADS) return;     // (a wave that has returned no longer counts)
  const int total = wl.cum[wl.n];
  for (int item = (int)blockIdx.x - ndiag; item < total; item += (int)gridDim.x - ndiag) {
    int mat, local, bi, bj;
    work_find_item(wl, item, mat, local);
    const MatDesc m = table[mat];
    if constexpr (SWEEP) {
      sweep_tile(m, p, local, (lds_c*)dsm);
    } else {
      if (!trail_tile(m.T, row_lo, row_hi, local, bi, bj)) continue;
      if (bj == p) continue;                   // tile (p, p): the diagonal block's own workgroup
      const float* const uk = m.U + (size_t)(p - 1) * DB * m.n;
      step_tile<false, false>(uk, uk, m.U, m.n, bi * BM, bj * BN, DB, -1.f, false, true, false,
                              (lds_c*)dsm);
    }
  }
}

// Workgroups of a step launch behind its `nd` diagonal blocks: one per tile, at most one per
// compute unit.
constexpr int STEP_CUS = 256;
static int step_workgroups(int nd, int tiles) { return std::min(tiles, std::max(STEP_CUS - nd, 64)); }

// The row panel for launches of few tiles: the same 128x128x128 product as a tile beside a diagonal
// block, one workgroup of 8 waves to a tile.  Alone it is a chain of latencies (93 tiles 12.7 us, 15.8
// with 16 waves on the fp32 matrix instructions and both operands whole in LDS, and since then 66 tiles 10.6 ->
// 11.8 for eight partial products instead of six and the vote); beside the launches of
// another stream what counts is that it fits into what one workgroup of the tile engine leaves: 99 KiB
// of LDS and 128 registers, where 128 KiB had to wait for an empty compute unit, that is until the other
// launch had handed out its last tile.
constexpr int FINE_THREADS = STEP_THREADS;
constexpr int FINE_SMEM_BYTES = STEP_VOTES + 4 * (FINE_THREADS / 64);
static_assert(FINE_SMEM_BYTES + SplitCfg<2>::SMEM_BYTES <= 160 * 1024, "fits beside a workgroup of the tile engine");
constexpr int FINE_MAX_TILES = 256;      // one workgroup per CU

// Tile `local` of row panel p.  U[p,j] = Y_pp^T A[p,j] in place for j > p, and in a sweep, after
// those T - p - 1 tiles, the finished row p of Z for j < p: Z[p,j] = Y_pp^T (pending row), read
// below the diagonal of Y and stored transposed above it.
struct PanelTile {
  const float* q;      // right-hand operand (row k at q + k n), `cols` columns wide
  float* c;            // where the result goes: U[p,j], or Y[j,p]
  int rows, cols;      // of the tile (rows: also the depth of the reduction)
  bool z;
};
__device__ __forceinline__ bool panel_tile(const MatDesc& m, int p, int local, PanelTile& t) {
  const int n = m.n, right = m.T - p - 1;
  t.z = local >= right;
  if (!t.z) {
    const int bj = p + 1 + local;
    t.q = t.c = m.U + (size_t)p * DB * n + bj * DB;
    t.rows = DB;
    t.cols = min(DB, n - bj * DB);
    return true;
  }
  const int bj = local - right;
  if (bj >= p) return false;
  t.q = m.Y + (size_t)p * DB * n + bj * DB;
  t.c = m.Y + (size_t)bj * DB * n + p * DB;
  t.rows = min(DB, n - p * DB);
  t.cols = DB;
  return true;
}

__global__ __launch_bounds__(FINE_THREADS, 4) void potrf_fine_kernel(const MatDesc* table, int p,
                                                                     const WorkList wl) {
  extern __shared__ __attribute__((aligned(16))) float fsm[];
  int mat, local;
  work_find(wl, mat, local);
  const MatDesc m = table[mat];
  const int n = m.n, row0 = p * DB, right = m.T - p - 1;
  const float* const y = m.Y + (size_t)row0 * n;
  if (local < right) {
    step_tile<false, false, false>(y, m.U + (size_t)row0 * n, m.U, n, row0, (p + 1 + local) * BM, DB,
                                   1.f, true, false, false, (lds_c*)fsm);
  } else if (local - right < p) {
    // (the transposed result comes from the exchanged operands)
    step_tile<false, false, false>(y, y, m.Y, n, (local - right) * BM, row0, min(DB, n - row0), 1.f,
                                   true, false, false, (lds_c*)fsm);
  }
}

// The same product for launches of very few tiles (at most SUB_MAX_TILES): every tile is
// dealt to four workgroups, so that four CUs' matrix cores work on it.  The row panel
// overwrites its own right-hand operand, so the pieces must not share columns: four
// 128x32 column strips, four 32x32 blocks each.  8 waves: the blocks' reductions, 32 to 128 deep
// since Y_pp is triangular, are cut at 64 k, and the two parts of the longer ones are added through
// LDS.  (All of them 128 deep, a half to a wave: 1153 us where this takes 1144, inverse and Cholesky
// factor of 2305^2.)
constexpr int SUB_THREADS = 512;
constexpr int SUB_SMEM_BYTES = DB * (128 + 32) * (int)sizeof(float);
// (32 instead of 64: inverse of 4600^2 1856 / 1976 us, three of 2305^2 1012 / 1064)
constexpr int SUB_MAX_TILES = 64;        // 4 workgroups per tile, one workgroup per CU

__global__ __launch_bounds__(SUB_THREADS) void potrf_sub_kernel(const MatDesc* table, int p,
                                                                const WorkList wl) {
  constexpr int WP = 128, WQ = 32;
  extern __shared__ __attribute__((aligned(16))) float fsm[];
  lds_f* const tp = (lds_f*)fsm;
  lds_f* const tq = tp + DB * WP;
  int mat, item;
  work_find(wl, mat, item);
  const int local = item >> 2, sj = item & 3;
  const MatDesc m = table[mat];
  const int n = m.n;
  PanelTile pt;
  if (!panel_tile(m, p, local, pt)) return;
  const float* P = m.Y + (size_t)p * DB * n + p * DB;
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const int r = lane & 31, h = lane >> 5;
  // block row br (k < 32 (br + 1): Y_pp is zero below its diagonal) and the wave's part of its
  // reduction; waves w and w + 4 share a SIMD, so no SIMD has more than 96 k
  // (a digit per wave: br = 3 3 2 1 0 2 - -, kbeg = 0 64 0 0 0 64 - -, kn = 64 64 64 64 32 32 0 0)
  const int br = (0x00201233 >> (4 * wave)) & 15, kbeg = ((0x22 >> wave) & 1) * 64,
            kn = ((0x00112222 >> (4 * wave)) & 15) * 32;
  const int row0 = 32 * br, col0 = WQ * sj;         // of this wave's block in the tile (U[p,j])

  const __amdgpu_buffer_rsrc_t rp = make_rsrc(P), rq = make_rsrc(pt.q);
  float vp[WP / 4], vq[WQ / 4];
#pragma unroll
  for (int i = 0; i < WP / 4; ++i) {
    const int idx = t + SUB_THREADS * i;
    const int k = idx / WP, col = idx % WP;
    vp[i] = buffer_load(rp, k <= (col | 31) && k < pt.rows && col < pt.rows ? (unsigned)(k * n + col) * 4u : INV_M);
  }
#pragma unroll
  for (int i = 0; i < WQ / 4; ++i) {
    const int idx = t + SUB_THREADS * i;
    const int k = idx / WQ, col = WQ * sj + idx % WQ;
    vq[i] = buffer_load(rq, k < pt.rows && col < pt.cols ? (unsigned)(k * n + col) * 4u : INV_M);
  }
#pragma unroll
  for (int i = 0; i < WP / 4; ++i) tp[t + SUB_THREADS * i] = vp[i];
#pragma unroll
  for (int i = 0; i < WQ / 4; ++i) tq[t + SUB_THREADS * i] = vq[i];
  __syncthreads();
  const lds_f* const bp = tp + kbeg * WP + row0;
  const lds_f* const bq = tq + kbeg * WQ;
  // (the transposed result comes from the exchanged operands: rows j, and lanes along i)
  v16f acc;
  if (kn > 0) acc = lds_mma32(pt.z ? bq : bp, pt.z ? WQ : WP, 1, pt.z ? bp : bq, pt.z ? WP : WQ, 1, kn);
  __syncthreads();
  // the second parts of the reduction travel through LDS (the operands are spent)
  lds_f* const red = tp + br * 1024;
  if (kbeg > 0) {
#pragma unroll
    for (int e = 0; e < 16; ++e) red[e * 64 + lane] = acc[e];
  }
  __syncthreads();
  if (kbeg == 0 && kn > 0) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int at = 8 * (e >> 2) + 4 * h + (e & 3);
      const int row = (pt.z ? col0 : row0) + at, col = (pt.z ? row0 : col0) + r;
      const float v = br >= 2 ? acc[e] + red[e * 64 + lane] : acc[e];
      if (row < (pt.z ? pt.cols : pt.rows) && col < (pt.z ? pt.rows : pt.cols))
        pt.c[(size_t)row * n + col] = v;
    }
  }
}

// ---- Y = U^-1 by balanced recursive halving over the 128-blocks ---------------
// Depth d cuts the T blocks of a matrix into 2^d nearly equal segments
// (boundaries floor(j*T/2^d)); the merge of the two children X1, X2 of a
// depth-d segment computes  Y12 = -Y11 * U12 * Y22, one tile per pair of a block of
// X1 and a block of X2.  A launch walks the tiles of all merges of its depth.
struct MergeTile {
  int X1, b1, X2, b2, it, jt;
  bool valid;
};

struct Segment {
  int p0, mid, p1;
  __host__ __device__ int tiles() const { return (mid - p0) * (p1 - mid); }
};

__host__ __device__ inline Segment segment(int P, int depth, int T) {
  Segment s;
  s.p0 = (int)(((long)P * T) >> depth);
  s.p1 = (int)(((long)(P + 1) * T) >> depth);
  s.mid = (int)(((long)(2 * P + 1) * T) >> (depth + 1));
  return s;
}

__host__ __device__ inline int merge_tiles(int T, int depth) {
  int total = 0;
  for (int P = 0; P < (1 << depth); ++P) total += segment(P, depth, T).tiles();
  return total;
}

// Tile `local` of the merges at `depth`, longest reduction first: a launch lasts at least
// as long as its longest tile (up to T/2 blocks on ONE compute unit, shared with another
// workgroup), so those start first and the launch ends on its one-block tiles.  The
// reduction of the first product grows with the column of the tile (`fast` = column, the
// tiles of a column share the Y22 panel), that of the second shrinks with the row (`fast`
// = row, its tiles share the Y11 panel).  The halves of all segments of a depth differ by
// at most one block, so rank r (0 = longest) holds one tile per `slow` index of every
// segment, except the last rank, which only the longer segments have.
__device__ __forceinline__ MergeTile merge_tile(const MatDesc& m, int depth, int local,
                                                bool by_column) {
  MergeTile t;
  t.valid = false;
  const int T = m.T, nseg = 1 << depth;
  int fmax = 0, s_all = 0, s_top = 0;
  for (int P = 0; P < nseg; ++P) {
    const Segment sg = segment(P, depth, T);
    const int rows = sg.mid - sg.p0, cols = sg.p1 - sg.mid;
    const int f = by_column ? rows : cols, sl = by_column ? cols : rows;
    if (f == 0 || sl == 0) continue;
    if (f > fmax) { fmax = f; s_top = 0; }
    if (f == fmax) s_top += sl;
    s_all += sl;
  }
  if (fmax == 0) return t;
  const int full = (fmax - 1) * s_all;
  if (local >= full + s_top) return t;
  int r, q;
  if (local < full) {
    r = local / s_all;
    q = local - r * s_all;
  } else {
    r = fmax - 1;
    q = local - full;
  }
  for (int P = 0; P < nseg; ++P) {
    const Segment sg = segment(P, depth, T);
    const int rows = sg.mid - sg.p0, cols = sg.p1 - sg.mid;
    const int f = by_column ? rows : cols, sl = by_column ? cols : rows;
    if (f == 0 || sl == 0 || f <= r) continue;
    if (q >= sl) { q -= sl; continue; }
    if (by_column) {
      t.it = r;
      t.jt = q;
    } else {
      t.it = q;
      t.jt = f - 1 - r;
    }
    t.X1 = sg.p0 * DB;
    t.b1 = rows * DB;
    t.X2 = sg.mid * DB;
    t.b2 = min(cols * DB, m.n - t.X2);
    t.valid = true;
    return t;
  }
  return t;
}

// first product:  W^T[j][i] = sum_{k <= j} Y22[k][j] * U12[i][k], stored at
// Y[X2 rows][X1 cols] (the unused lower triangle of Y)
__global__ __launch_bounds__(NTHREADS, 2) void trtri_w_kernel(const MatDesc* table, int depth,
                                                           const WorkList wl) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  int mat, local;
  work_find(wl, mat, local);
  const MatDesc m = table[mat];
  const MergeTile t = merge_tile(m, depth, local, false);
  if (!t.valid) return;
  const int n = m.n;
  DenseKM P{m.Y + (size_t)t.X2 * n + t.X2, nullptr, n, t.b2, 0};
  DenseMK Q{m.U + (size_t)t.X1 * n + t.X2, n, t.b1};
  EpiStore epi{m.Y + (size_t)t.X2 * n + t.X1, n, t.b2, t.b1, 1.f, 0.f, false};
  split_tile(P, Q, t.jt * BM, t.it * BN, 0, min(t.b2, (t.jt + 1) * DB), false, epi, smem);
}

// second product:  Y12[i][j] = - sum_{k >= i} Y11[i][k] * W^T[j][k]
__global__ __launch_bounds__(NTHREADS, 2) void trtri_y_kernel(const MatDesc* table, int depth,
                                                           const WorkList wl) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  int mat, local;
  work_find(wl, mat, local);
  const MatDesc m = table[mat];
  const MergeTile t = merge_tile(m, depth, local, true);
  if (!t.valid) return;
  const int n = m.n;
  DenseMK P{m.Y + (size_t)t.X1 * n + t.X1, n, t.b1};
  DenseMK Q{m.Y + (size_t)t.X2 * n + t.X1, n, t.b2};
  EpiStore epi{m.Y + (size_t)t.X1 * n + t.X2, n, t.b1, t.b2, -1.f, 0.f, false};
  split_tile(P, Q, t.it * BM, t.jt * BN, t.it * DB, t.b1, false, epi, smem);
}

// Which upper tile (bi <= bj) of Y Y^T a workgroup takes.  The tiles of a column bj all
// reduce over k >= bj*128 (same length) and share the operand panel Y[bj rows], and the
// work of a column, (bj + 1) * (T - bj), varies smoothly with bj.  Workgroups go to the
// 8 XCDs (one L2 each) in turn by dispatch index, so XCD x is given the columns
// bj = x, x + 8, ... (equal work within 3 %, a panel is read by one L2 only), first
// column (longest reduction) first.  The classes differ a little in tile count while every
// XCD gets the same number of workgroups: the surplus tiles of a class, which are its
// shortest, go to the workgroups that the smaller classes leave without a tile.
__device__ __forceinline__ int column_class_size(int T, int x) {
  if (x > T - 1) return 0;
  const int c = (T - 1 - x) / 8 + 1;
  return c * (x + 1) + 4 * c * (c - 1);
}

__device__ __forceinline__ void column_class_tile(int x, int t, int& bi, int& bj) {
  bj = x;
  while (t >= bj + 1) {
    t -= bj + 1;
    bj += 8;
  }
  bi = t;
}

__device__ __forceinline__ void lauum_tile(int T, int local, int& bi, int& bj) {
  const int ntiles = T * (T + 1) / 2;
  const int g = (int)blockIdx.x;
  const int x = g & 7;
  const int s8 = (g - local) & 7;                  // where the matrix starts in the grid, mod 8
  int deficit_before = 0, slots_x = 0, size_x = 0, first_x = 0;
  int slots[8], size[8];
#pragma unroll
  for (int y = 0; y < 8; ++y) {
    const int first = (y - s8 + 8) & 7;            // first workgroup of this matrix on XCD y
    slots[y] = max(0, (ntiles - first + 7) / 8);
    size[y] = column_class_size(T, y);
    if (y == x) {
      slots_x = slots[y];
      size_x = size[y];
      first_x = first;
    }
  }
  const int t = (local - first_x) / 8;
  if (t < size_x) {
    column_class_tile(x, t, bi, bj);
    return;
  }
#pragma unroll
  for (int y = 0; y < 8; ++y)
    if (y < x) deficit_before += max(0, slots[y] - size[y]);
  int r = deficit_before + (t - size_x);           // rank among the tiles without a workgroup
  (void)slots_x;
#pragma unroll
  for (int z = 0; z < 8; ++z) {
    const int excess = max(0, size[z] - slots[z]);
    if (r >= 0 && r < excess) {
      column_class_tile(z, slots[z] + r, bi, bj);
      return;
    }
    r -= excess;
  }
  bi = bj = 0;       // not reached: the classes hold exactly ntiles tiles
}

// C[f(row)][f(col)] = v (and, by put(), its mirror image), f(i) = base + sign * i: the identity, or the
// reversal i -> n - 1 - i that undoes the reversed read of a matrix factored back to front
struct EpiSymFlip {
  float* C;
  int n, base, sign;
  bool mirror;
  __device__ __forceinline__ float value(float v) const { return v; }
  __device__ __forceinline__ void put(int row, int col, float o) const {
    if (row < n && col < n) C[(size_t)(base + sign * row) * n + base + sign * col] = o;
  }
  __device__ __forceinline__ void store(int row, int col, float v) const { put(row, col, v); }
};

// dst = Y Y^T over the upper tiles (k >= the later block), mirrored
__global__ __launch_bounds__(NTHREADS, 2) void lauum_kernel(const MatDesc* table, const WorkList wl) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  int mat, local;
  work_find(wl, mat, local);
  const MatDesc m = table[mat];
  if (m.noinv) return;
  int bi, bj;
  lauum_tile(m.T, local, bi, bj);
  const int n = m.n;
  DenseMK P{m.Y, n, n};
  EpiSymFlip epi{m.U, n, m.rev ? n - 1 : 0, m.rev ? -1 : 1, bi != bj};
  split_tile(P, P, bi * BM, bj * BN, bj * DB, n, bi == bj, epi, smem);
}

// W = J Y^T J (J = reversal) for the matrices factored back to front: with S = J X J = R^T R
// and Y = R^-1, X^-1 = J Y Y^T J = W^T W and W is upper triangular with a positive diagonal,
// i.e. the upper Cholesky factor of X^-1, read off the triangular inverse instead of being
// computed by a second factorisation.  W[i][j] = Y[n-1-j][n-1-i] for j >= i, 0 below;
// 64 x 64 tiles through LDS so that reads and writes are both row-contiguous.
__global__ __launch_bounds__(256) void std_from_inverse_factor_kernel(const MatDesc* table,
                                                                      const WorkList wl) {
  __shared__ float tile[64][65];
  int mat, local;
  work_find(wl, mat, local);
  const MatDesc m = table[mat];
  if (m.W == nullptr) return;
  const int n = m.n;
  const int T64 = (n + 63) / 64;
  const int ti = local / T64, tj = local - ti * T64;       // tile of W: rows ti, columns tj
  const int i0 = ti * 64, j0 = tj * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  if (tj >= ti) {
    // source element for W[i0 + a][j0 + b] is Y[n-1-j0-b][n-1-i0-a]: lanes run along a
    for (int b = ty; b < 64; b += 4) {
      const int r = n - 1 - j0 - b, c = n - 1 - i0 - tx;
      tile[b][tx] = (r >= 0 && c >= 0 && c >= r) ? m.Y[(size_t)r * n + c] : 0.f;
    }
  }
  __syncthreads();
  for (int a = ty; a < 64; a += 4) {
    const int i = i0 + a, j = j0 + tx;
    if (i < n && j < n) m.W[(size_t)i * n + j] = (tj >= ti && j >= i) ? tile[tx][a] : 0.f;
  }
}

// Two halves.  The last merge of the triangular inverse, Y12 = -Y11 U12 Y22 at depth 0, is n^3/4
// of its n^3/3 multiply-adds; whoever applies Y to a matrix can do without it and use U12 as it is,
//   V Y = [V1 Y11, (V2 - (V1 Y11) U12) Y22],
// at the cost of applying Y.  Such a factor holds Y11, Y22 and, in the place of Y12, U12.
static int half_cut(int T) { return T >> 1; }       // (segment(0, 0, T).mid)

// zero the strictly lower triangle of a triangular result: of U for every matrix
// (Cholesky-factor output), or, with `of_y`, of Y for the matrices whose result Y is (whose
// U12 comes to Y here where it is left in two halves)
__global__ __launch_bounds__(256) void zero_lower_kernel(const MatDesc* table, int of_y,
                                                         const WorkList wl) {
  int mat, local;
  work_find(wl, mat, local);
  const MatDesc m = table[mat];
  if (of_y && !m.noinv) return;
  float* const X = of_y ? m.Y : m.U;
  const int n = m.n;
  const int T = m.T;
  const int bi = local / T, bj = local - bi * T;
  if (bj > bi) {
    if (!of_y || bi >= m.cut || bj < m.cut) return;
    // 16 loads in flight, then 16 stores
    const float* const from = m.U;
    for (int e0 = threadIdx.x; e0 < BM * BN; e0 += 256 * 16) {
      float v[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int e = e0 + 256 * k, row = bi * BM + (e >> 7), col = bj * BN + (e & 127);
        v[k] = col < n ? from[(size_t)row * n + col] : 0.f;
      }
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int e = e0 + 256 * k, row = bi * BM + (e >> 7), col = bj * BN + (e & 127);
        if (col < n) X[(size_t)row * n + col] = v[k];
      }
    }
    return;
  }
  for (int e = threadIdx.x; e < BM * BN; e += 256) {
    const int row = bi * BM + (e >> 7);
    const int col = bj * BN + (e & 127);
    if (row < n && col < n && col < row) X[(size_t)row * n + col] = 0.f;
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

struct HostMat {
  const float* src;
  float* dst;
  int n;
  float damp;
  int partner;   // index in caller order, or -1
  int is_a;
  int out;
  float* std = nullptr;   // non-null: factor back to front and also deliver the upper
                          // Cholesky factor W of the inverse (W^T W = inverse; the posterior
                          // std of Noisy K-FAC)
  float* fac = nullptr;   // non-null (then dst and std are null): deliver the inverse as its
                          // triangular factor only, Y upper with Y Y^T = inverse
  int halves = 0;         // with fac: 1 it may be left in two halves, 2 it has to be
};

static size_t inverse_workspace_bytes(const std::vector<int>& dims) {
  size_t bytes = align256(dims.size() * sizeof(MatDesc));
  for (int n : dims) bytes += align256((size_t)n * n * sizeof(float));
  return bytes;
}

enum { MODE_INVERSE = 0, MODE_CHOLESKY = 1 };

// The sweep (SWEEP of potrf_step_kernel) or, after the factorisation, the recursive triangular
// inverse and Y Y^T.  The sweep has two launches per 128 columns and nothing after them, but its
// products are 128 deep and read and write their results every time; the recursive one adds
// 2 log2(T) + 1 launches, each as long as its longest tile, of deep products.  So the line
// lies where the tiles of a step, about T^2 / 2 per matrix, no longer fit beside a diagonal block:
// three per compute unit.  Recursive / sweep, one matrix of n rows, us (same step tiles):
//     300: 140 / 102   1000: 401 / 263   2305: 940 / 611   3500 (406 tiles): 1408 / 1075
//     4600 (666): 2001 / 1856;   three of 2305 (570): 1042 / 1012;   five of 2200 (855): 1189 / 1265
//     the layers of a ResNet-50 (several thousand): 4.67 / 7.32 ms
// (between 600 and 765 tiles several matrices are better off without: four of 2305 (760) 1191 / 1276,
// twenty of 1000 (720) 569 / 609; one of 4600 is not.)
// (a matrix of one block has no panels: Y Y^T by its own kernel, 70 us instead of 75.)
constexpr long SWEEP_MAX_TILES = 3 * 255;
static bool use_sweep(const std::vector<int>& Ts) {
  long tiles = 0;
  int longest = 0;
  for (int T : Ts) {
    tiles += (long)T * (T + 1) / 2;
    longest = std::max(longest, T);
  }
  return longest > 1 && tiles <= SWEEP_MAX_TILES;
}

static int run_batched(std::vector<HostMat>& mats, int mode, int* info, void* workspace,
                       size_t workspace_bytes, hipStream_t stream) {
  const int nmat = (int)mats.size();
  if (nmat == 0) return KFAC_OK;
  std::vector<int> dims(nmat);
  for (int i = 0; i < nmat; ++i) dims[i] = mats[i].n;
  if (workspace == nullptr || workspace_bytes < inverse_workspace_bytes(dims))
    return KFAC_ERR_WORKSPACE;

  // kernels that need more than the default 64 KiB of LDS (registered once per process)
  if (!enable_large_lds((const void*)potrf_diag_kernel, DIAG_SMEM_BYTES) ||
      !enable_large_lds((const void*)potrf_step_kernel<false>, DIAG_SMEM_BYTES) ||
      !enable_large_lds((const void*)potrf_step_kernel<true>, DIAG_SMEM_BYTES) ||
      !enable_large_lds((const void*)potrf_fine_kernel, FINE_SMEM_BYTES) ||
      !enable_large_lds((const void*)potrf_sub_kernel, SUB_SMEM_BYTES))
    return KFAC_ERR_LAUNCH;

  // descending size order; remember where each caller index went
  std::vector<int> order(nmat);
  for (int i = 0; i < nmat; ++i) order[i] = i;
  std::stable_sort(order.begin(), order.end(),
                   [&](int a, int b) { return mats[a].n > mats[b].n; });
  std::vector<int> pos(nmat);
  for (int s = 0; s < nmat; ++s) pos[order[s]] = s;

  MatDesc* table = (MatDesc*)workspace;
  char* ybase = (char*)workspace + align256(nmat * sizeof(MatDesc));
  size_t yoff = 0;
  std::vector<int> Ts(nmat), cuts(nmat);
  for (int s = 0; s < nmat; ++s) Ts[s] = cdiv(mats[order[s]].n, DB);
  const int Tmax = Ts[0];
  bool any_cut = false;
  for (int s = 0; s < nmat; ++s) any_cut |= mats[order[s]].halves == 2;
  const bool sweep = mode == MODE_INVERSE && !any_cut && use_sweep(Ts);
  bool any_pi = false;
  for (auto& h : mats) any_pi |= h.partner >= 0;
  for (int s0 = 0; s0 < nmat; s0 += SETUP_CHUNK) {
    DescChunk chunk;
    const int cnt = std::min(SETUP_CHUNK, nmat - s0);
    for (int k = 0; k < cnt; ++k) {
      const HostMat& h = mats[order[s0 + k]];
      MatDesc& d = chunk.d[k];
      d.src = h.src;
      // the slot of the workspace holds Y, or, when Y goes straight to the caller, the
      // Cholesky factor that nobody asked for
      d.noinv = h.fac != nullptr;
      d.cut = d.noinv && h.halves && !sweep ? half_cut(cdiv(h.n, DB)) : 0;
      d.U = d.noinv ? (float*)(ybase + yoff) : h.dst;
      d.Y = d.noinv ? h.fac : (float*)(ybase + yoff);
      yoff += align256((size_t)h.n * h.n * sizeof(float));
      d.n = h.n;
      d.T = cdiv(h.n, DB);
      d.damp = h.damp;
      d.partner = h.partner < 0 ? -1 : pos[h.partner];
      d.is_a = h.is_a;
      d.out = h.out;
      d.trace = 0.f;
      d.rev = h.std != nullptr;
      d.W = h.std;
      cuts[s0 + k] = d.cut;
    }
    if (any_pi)
      hipLaunchKernelGGL(inv_trace_kernel, dim3(cnt), dim3(256), 0, stream, chunk, table, s0);
    else
      hipLaunchKernelGGL(inv_setup_kernel, dim3(1), dim3(SETUP_CHUNK), 0, stream, chunk, table, s0, cnt);
  }
  auto active = [&](int minT) {   // matrices with T >= minT (a prefix of the sorted table)
    int c = 0;
    while (c < nmat && Ts[c] >= minT) ++c;
    return c;
  };

  // Runs `launch(worklist)` over the first `count` matrices of the sorted table,
  // WL_MAX at a time, with items(s) work items for the matrix at position s; matrices
  // without items are skipped at the ends and cost nothing in between.
  auto for_matrices = [&](int count, auto&& items, auto&& launch) {
    for (int s0 = 0; s0 < count; s0 += WL_MAX) {
      WorkList wl;
      wl.first = s0;
      wl.n = std::min(WL_MAX, count - s0);
      wl.cum[0] = 0;
      for (int i = 0; i < wl.n; ++i) wl.cum[i + 1] = wl.cum[i] + std::max(0, (int)items(s0 + i));
      for (int i = wl.n + 1; i <= WL_MAX; ++i) wl.cum[i] = wl.cum[wl.n];
      if (wl.cum[wl.n] > 0) launch(wl, wl.cum[wl.n]);
    }
  };

  // ... with items(T) work items for a matrix of T blocks
  auto for_worklists = [&](int count, auto&& items, auto&& launch) {
    for_matrices(count, [&](int s) { return items(Ts[s]); }, launch);
  };

  for_worklists(nmat, [](int T) { return COPY_PARTS * T * (T + 1) / 2; },
                [&](const WorkList& wl, int grid) {
    hipLaunchKernelGGL(inv_copy_damp_kernel, dim3(grid), dim3(256), 0, stream, table, info, wl);
  });

  // (a matrix factored back to front is written back through a reversal: its Y Y^T comes after)
  auto sweep_x = [&](int s) {
    const HostMat& h = mats[order[s]];
    return h.fac == nullptr && h.std == nullptr;
  };
  for (int p = 0; sweep && p <= Tmax; ++p) {
    const int na = active(p + 1);
    if (p == 0) {
      hipLaunchKernelGGL(potrf_diag_kernel, dim3(na), dim3(DIAG_THREADS), DIAG_SMEM_BYTES, stream,
                         table, p, info);
    } else {
      bool first = true;
      for_matrices(active(p), [&](int s) { return sweep_items(Ts[s], p, sweep_x(s)); },
                   [&](const WorkList& wl, int grid) {
        const int nd = first ? na : 0;
        first = false;
        hipLaunchKernelGGL(potrf_step_kernel<true>, dim3(nd + step_workgroups(nd, grid)),
                           dim3(DIAG_THREADS), DIAG_SMEM_BYTES, stream, table, p, info, nd, p, Tmax,
                           wl);
      });
    }
    int panels = 0;
    auto panel_items = [&](int T) { return T > p ? T - 1 : 0; };
    for (int s = 0; s < na; ++s) panels += panel_items(Ts[s]);
    if (panels <= SUB_MAX_TILES)
      for_worklists(na, [&](int T) { return 4 * panel_items(T); }, [&](const WorkList& wl, int grid) {
        hipLaunchKernelGGL(potrf_sub_kernel, dim3(grid), dim3(SUB_THREADS), SUB_SMEM_BYTES, stream,
                           table, p, wl);
      });
    else
      for_worklists(na, panel_items, [&](const WorkList& wl, int grid) {
        hipLaunchKernelGGL(potrf_fine_kernel, dim3(grid), dim3(FINE_THREADS), FINE_SMEM_BYTES,
                           stream, table, p, wl);
      });
  }
  for (int P0 = 0, Pend = 0; !sweep && P0 < Tmax; P0 = Pend) {
    Pend = Tmax - P0 <= TAIL_BLOCKS ? Tmax : std::min(P0 + GROUP_BLOCKS, Tmax);
    auto total_items = [&](int count, auto&& items) {
      long sum = 0;
      for (int i = 0; i < count; ++i) sum += std::max(0, (int)items(Ts[i]));
      return sum;
    };
    for (int p = P0; p < Pend; ++p) {
      const int na = active(p + 1);
      // diagonal block p; from the group's second block on it first takes panel p-1's update
      // itself, and the same launch holds the tiles that apply that panel to the other rows
      // of the group (block row p first: the next row panel needs it; nothing else needs any
      // of them before the next launch)
      auto rest_items = [&](int T) {
        const int Tr = T - p;          // (all remaining rows: the upper triangle of tiles)
        return Pend >= T ? Tr * (Tr + 1) / 2 : (Pend - p) * Tr;
      };
      if (p == P0) {
        hipLaunchKernelGGL(potrf_diag_kernel, dim3(na), dim3(DIAG_THREADS), DIAG_SMEM_BYTES, stream,
                           table, p, info);
      } else {
        bool first = true;
        for_worklists(na, rest_items, [&](const WorkList& wl, int grid) {
          const int nd = first ? na : 0;
          first = false;
          hipLaunchKernelGGL(potrf_step_kernel<false>, dim3(nd + step_workgroups(nd, grid)),
                             dim3(DIAG_THREADS), DIAG_SMEM_BYTES, stream, table, p, info, nd, p,
                             Pend, wl);
        });
      }
      const int nb = active(p + 2);
      if (nb == 0) continue;
      auto panel_items = [&](int T) { return T - p - 1; };
      if (total_items(nb, panel_items) <= SUB_MAX_TILES) {
        for_worklists(nb, [&](int T) { return 4 * std::max(0, panel_items(T)); },
                      [&](const WorkList& wl, int grid) {
                        hipLaunchKernelGGL(potrf_sub_kernel, dim3(grid), dim3(SUB_THREADS),
                                           SUB_SMEM_BYTES, stream, table, p, wl);
                      });
      } else
      for_worklists(nb, panel_items, [&](const WorkList& wl, int grid) {
        if (grid <= FINE_MAX_TILES)
          hipLaunchKernelGGL(potrf_fine_kernel, dim3(grid), dim3(FINE_THREADS), FINE_SMEM_BYTES,
                             stream, table, p, wl);
        else
          KFAC_LAUNCH_TILE2(potrf_panel_kernel, dim3(grid), stream, table, p, wl);
      });
    }
    const int nc = active(Pend + 1);
    if (Pend < Tmax && nc > 0) {
      for_worklists(nc, [&](int T) { const int Tr = T - Pend; return Tr * (Tr + 1) / 2; },
                    [&](const WorkList& wl, int grid) {
                      KFAC_LAUNCH_TILE2(potrf_trail_kernel, dim3(grid), stream, table, P0,
                                        Pend - P0, Pend, Tmax, wl);
                    });
    }
  }
  if (mode == MODE_CHOLESKY) {
    for_worklists(nmat, [](int T) { return T * T; }, [&](const WorkList& wl, int grid) {
      hipLaunchKernelGGL(zero_lower_kernel, dim3(grid), dim3(256), 0, stream, table, 0, wl);
    });
    return launch_status();
  }
  if (Tmax > 1 && !sweep) {
    int D = 0;
    while ((1 << D) < Tmax) ++D;
    const int na = active(2);
    for (int depth = D - 1; depth >= 0 && na > 0; --depth) {
      // matrices with fewer than 2^depth blocks have no merge this deep, those left in two halves
      // not the last one
      auto pairs = [&](int s) {
        return (1 << depth) < Ts[s] && (depth > 0 || cuts[s] == 0) ? merge_tiles(Ts[s], depth) : 0;
      };
      for_matrices(na, pairs, [&](const WorkList& wl, int grid) {
        KFAC_LAUNCH_TILE2(trtri_w_kernel, dim3(grid), stream, table, depth, wl);
      });
      for_matrices(na, pairs, [&](const WorkList& wl, int grid) {
        KFAC_LAUNCH_TILE2(trtri_y_kernel, dim3(grid), stream, table, depth, wl);
      });
    }
  }
  bool any_inv = false, any_std = false, any_fac = false;
  for (auto& h : mats) {
    any_inv |= h.dst != nullptr;
    any_std |= h.std != nullptr;
    any_fac |= h.fac != nullptr;
  }
  if (any_inv)      // (in a sweep, those of its matrices that it did not finish)
    for_matrices(nmat, [&](int s) { return sweep && sweep_x(s) ? 0 : Ts[s] * (Ts[s] + 1) / 2; },
                 [&](const WorkList& wl, int grid) {
      KFAC_LAUNCH_TILE2(lauum_kernel, dim3(grid), stream, table, wl);
    });
  if (any_fac)   // the triangular inversion kept intermediate products below the diagonal
    for_worklists(nmat, [](int T) { return T * T; }, [&](const WorkList& wl, int grid) {
      hipLaunchKernelGGL(zero_lower_kernel, dim3(grid), dim3(256), 0, stream, table, 1, wl);
    });
  if (any_std) {
    // (items per matrix: its 64 x 64 tiles; Ts holds 128-blocks, so 4 T^2 covers them)
    for_worklists(nmat, [](int T) { return 4 * T * T; }, [&](const WorkList& wl, int grid) {
      hipLaunchKernelGGL(std_from_inverse_factor_kernel, dim3(grid), dim3(256), 0, stream, table,
                         wl);
    });
  }
  return launch_status();
}

// ---------------------------------------------------------------------------
// Scratch for the entry point that allocates nothing: one array in device memory,
// part of the code object, so every GPU this library runs on holds its own copy at
// its own address until the process ends.  In host code the name `scratch` is only a
// handle for hipGetSymbolAddress; kernels and memory calls get the address it returns.
// ---------------------------------------------------------------------------
constexpr size_t STATIC_SCRATCH_BYTES = (size_t)8 << 20;
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

constexpr int SCRATCH_MAX_DEVICES = 64;
static std::atomic<void*> scratch_ptr[SCRATCH_MAX_DEVICES];   // address on each device, once known

// Device address of `scratch` on the current device (looked up on the first call on that
// device); nullptr on failure.
static void* static_scratch() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SCRATCH_MAX_DEVICES) return nullptr;
  void* ptr = scratch_ptr[dev].load(std::memory_order_acquire);
  if (ptr != nullptr) return ptr;
  if (hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr)
    return nullptr;
  scratch_ptr[dev].store(ptr, std::memory_order_release);
  return ptr;
}

// Calls that share the array are put in order: each call records an event behind its last
// kernel, and the next call on that device makes its stream wait for it first (a no-op for
// the single-stream caller).  The events are created on a device's first call.  A stream
// under graph capture takes no part: an event recorded outside a capture cannot be waited
// for inside one, and inside a graph the graph's own order applies.
static std::mutex scratch_mutex;
static hipEvent_t scratch_done[SCRATCH_MAX_DEVICES];    // (never destroyed: no teardown order)
static bool scratch_done_set[SCRATCH_MAX_DEVICES];

static bool stream_is_capturing(hipStream_t stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &st) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return st != hipStreamCaptureStatusNone;
}

}  // namespace kfac

using namespace kfac;

extern "C" {

size_t kfac_static_workspace_bytes(void) { return STATIC_SCRATCH_BYTES; }

int kfac_damped_inverse_batched_static(int count, const int* dims, const float* const* src,
                                       const float* damp, float* const* dst, int* info,
                                       void* stream) {
  if (count < 0 || (count > 0 && (!dims || !src || !dst || !info))) return KFAC_ERR_ARG;
  std::vector<HostMat> mats(count);
  std::vector<int> d(count);
  for (int i = 0; i < count; ++i) {
    if (dims[i] <= 0 || dims[i] > 16384 || !src[i] || !dst[i] || src[i] == dst[i])
      return KFAC_ERR_ARG;
    mats[i] = HostMat{src[i], dst[i], dims[i], damp ? damp[i] : 0.f, -1, 0, i};
    d[i] = dims[i];
  }
  if (count == 0) return KFAC_OK;
  if (inverse_workspace_bytes(d) > STATIC_SCRATCH_BYTES) return KFAC_ERR_TOO_LARGE;
  void* ptr = static_scratch();
  if (ptr == nullptr) return KFAC_ERR_LAUNCH;
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SCRATCH_MAX_DEVICES) return KFAC_ERR_LAUNCH;
  hipStream_t st = (hipStream_t)stream;
  std::lock_guard<std::mutex> order(scratch_mutex);
  const bool ordered = !stream_is_capturing(st);
  if (ordered) {
    if (!scratch_done_set[dev]) {
      if (hipEventCreateWithFlags(&scratch_done[dev], hipEventDisableTiming) != hipSuccess)
        return KFAC_ERR_LAUNCH;
      scratch_done_set[dev] = true;
    } else if (hipStreamWaitEvent(st, scratch_done[dev], 0) != hipSuccess) {
      return KFAC_ERR_LAUNCH;
    }
  }
  const int status = run_batched(mats, MODE_INVERSE, info, ptr, STATIC_SCRATCH_BYTES, st);
  if (ordered && hipEventRecord(scratch_done[dev], st) != hipSuccess) return KFAC_ERR_LAUNCH;
  return status;
}

double kfac_inverse_executed_flops(int count, const int* dims, const int* factored) {
  if (count <= 0 || !dims) return 0.;
  const double B = 2. * DB * DB * DB;       // one 128-deep step of a 128 x 128 tile
  // diagonal block: per strip 15 rank-2 steps of five blocks, the updates by finished strips
  // (20 blocks, 32 deep), the pending panel (10 blocks, 128 deep)
  const double diag = 4096. * (4 * 75 + 20 * 16 + 10 * 64);
  double total = 0.;
  std::vector<int> Ts(count);
  for (int i = 0; i < count; ++i) Ts[i] = cdiv(dims[i], DB);
  if (use_sweep(Ts)) {
    for (int i = 0; i < count; ++i) {
      const int T = Ts[i];
      total += T * diag + B * T * (T - 1);      // diagonal blocks; row panels of U and Z
      for (int p = 1; p <= T; ++p)              // (tile (p, p) is the diagonal block's)
        total += B * (sweep_items(T, p, !(factored && factored[i])) - (p < T ? 1 : 0));
    }
    return total;
  }
  for (int i = 0; i < count; ++i) {
    const double T = Ts[i];
    // Cholesky: row panels, trailing updates (whole diagonal tiles)
    total += T * diag + B * (T * (T - 1) / 2 + (T - 1) * T * (T + 1) / 6);
    // triangular inverse: per merge of r x c blocks, W tiles reduce over 1..c blocks,
    // Y tiles over r..1
    const int Ti = (int)T;
    int D = 0;
    while ((1 << D) < Ti) ++D;
    for (int depth = factored && factored[i] == 2 ? 1 : 0; depth < D; ++depth)
      for (int P = 0; P < (1 << depth); ++P) {
        const Segment sg = segment(P, depth, Ti);
        const double r = sg.mid - sg.p0, c = sg.p1 - sg.mid;
        total += B * (r * c * (c + 1) / 2 + c * r * (r + 1) / 2);
      }
    // Y Y^T where the explicit inverse is formed: tile (bi <= bj) reduces over T - bj blocks
    if (!(factored && factored[i]))
      for (int bj = 0; bj < Ti; ++bj) total += B * (bj + 1.) * (T - bj);
  }
  return total;
}

size_t kfac_inverse_workspace_bytes(int count, const int* dims) {
  if (count <= 0 || !dims) return 0;
  std::vector<int> d(dims, dims + count);
  for (int n : d)
    if (n <= 0) return 0;
  return inverse_workspace_bytes(d);
}

int kfac_damped_inverse_batched(int count, const int* dims, const float* const* src,
                                const float* damp, float* const* dst, int* info,
                                void* workspace, size_t workspace_bytes, void* stream) {
  if (count < 0 || (count > 0 && (!dims || !src || !dst || !info))) return KFAC_ERR_ARG;
  std::vector<HostMat> mats(count);
  for (int i = 0; i < count; ++i) {
    if (dims[i] <= 0 || dims[i] > 16384 || !src[i] || !dst[i] || src[i] == dst[i])
      return KFAC_ERR_ARG;
    mats[i] = HostMat{src[i], dst[i], dims[i], damp ? damp[i] : 0.f, -1, 0, i};
  }
  return run_batched(mats, MODE_INVERSE, info, workspace, workspace_bytes, (hipStream_t)stream);
}

int kfac_pi_damped_inverse_batched(int layers, const int* dA, const int* dG,
                                   const float* const* A, const float* const* G,
                                   const float* damping, float* const* Ainv, float* const* Ginv,
                                   int* info, void* workspace, size_t workspace_bytes,
                                   void* stream) {
  if (layers < 0 || (layers > 0 && (!dA || !dG || !A || !G || !damping || !Ainv || !Ginv || !info)))
    return KFAC_ERR_ARG;
  std::vector<HostMat> mats(2 * layers);
  for (int l = 0; l < layers; ++l) {
    if (dA[l] <= 0 || dG[l] <= 0 || dA[l] > 16384 || dG[l] > 16384 || !A[l] || !G[l] ||
        !Ainv[l] || !Ginv[l] || A[l] == Ainv[l] || G[l] == Ginv[l] || !(damping[l] >= 0.f))
      return KFAC_ERR_ARG;
    const float r = sqrtf(damping[l]);
    mats[2 * l] = HostMat{A[l], Ainv[l], dA[l], r, 2 * l + 1, 1, 2 * l};
    mats[2 * l + 1] = HostMat{G[l], Ginv[l], dG[l], r, 2 * l, 0, 2 * l + 1};
  }
  return run_batched(mats, MODE_INVERSE, info, workspace, workspace_bytes, (hipStream_t)stream);
}

int kfac_pi_damped_inverse_std_batched(int layers, const int* dA, const int* dG,
                                       const float* const* A, const float* const* G,
                                       const float* damping, float* const* Ainv,
                                       float* const* Ginv, float* const* Astd,
                                       float* const* Gstd, int* info, void* workspace,
                                       size_t workspace_bytes, void* stream) {
  if (layers < 0 || (layers > 0 && (!dA || !dG || !A || !G || !damping || !Ainv || !Ginv ||
                                    !Astd || !Gstd || !info)))
    return KFAC_ERR_ARG;
  std::vector<HostMat> mats(2 * layers);
  for (int l = 0; l < layers; ++l) {
    if (dA[l] <= 0 || dG[l] <= 0 || dA[l] > 16384 || dG[l] > 16384 || !A[l] || !G[l] ||
        !Ainv[l] || !Ginv[l] || A[l] == Ainv[l] || G[l] == Ginv[l] || !(damping[l] >= 0.f))
      return KFAC_ERR_ARG;
    if (Astd[l] && (Astd[l] == Ainv[l] || Astd[l] == A[l])) return KFAC_ERR_ARG;
    if (Gstd[l] && (Gstd[l] == Ginv[l] || Gstd[l] == G[l])) return KFAC_ERR_ARG;
    const float r = sqrtf(damping[l]);
    mats[2 * l] = HostMat{A[l], Ainv[l], dA[l], r, 2 * l + 1, 1, 2 * l, Astd[l]};
    mats[2 * l + 1] = HostMat{G[l], Ginv[l], dG[l], r, 2 * l, 0, 2 * l + 1, Gstd[l]};
  }
  return run_batched(mats, MODE_INVERSE, info, workspace, workspace_bytes, (hipStream_t)stream);
}

// A_halves: NULL, or which factors of A may (1) or have to (2) be left in two halves; on return, which are
static int factored_batched(int layers, const int* dA, const int* dG, const float* const* A,
                            const float* const* G, const float* damping, float* const* Ainv,
                            float* const* Ginv, float* const* Afac, float* const* Gfac, int* A_halves,
                            int* info, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (layers < 0 || (layers > 0 && (!dA || !dG || !A || !G || !damping || !Ainv || !Ginv ||
                                    !Afac || !Gfac || !info)))
    return KFAC_ERR_ARG;
  std::vector<HostMat> mats(2 * layers);
  std::vector<int> Ts(2 * layers);
  bool any_cut = false;
  for (int l = 0; l < layers; ++l) {
    if (dA[l] <= 0 || dG[l] <= 0 || dA[l] > 16384 || dG[l] > 16384 || !A[l] || !G[l] ||
        !(damping[l] >= 0.f))
      return KFAC_ERR_ARG;
    // per matrix exactly one of the two forms, never on top of its input
    if ((Ainv[l] == nullptr) == (Afac[l] == nullptr) || (Ginv[l] == nullptr) == (Gfac[l] == nullptr))
      return KFAC_ERR_ARG;
    if (Ainv[l] == A[l] || Afac[l] == A[l] || Ginv[l] == G[l] || Gfac[l] == G[l])
      return KFAC_ERR_ARG;
    const float r = sqrtf(damping[l]);
    mats[2 * l] = HostMat{A[l], Ainv[l], dA[l], r, 2 * l + 1, 1, 2 * l, nullptr, Afac[l],
                          A_halves && Afac[l] && half_cut(cdiv(dA[l], DB)) > 0 ? A_halves[l] : 0};
    any_cut |= mats[2 * l].halves == 2;
    mats[2 * l + 1] = HostMat{G[l], Ginv[l], dG[l], r, 2 * l, 0, 2 * l + 1, nullptr, Gfac[l]};
    Ts[2 * l] = cdiv(dA[l], DB);
    Ts[2 * l + 1] = cdiv(dG[l], DB);
  }
  // (the sweep has whole factors at no extra cost)
  const bool whole = !any_cut && use_sweep(Ts);
  for (int l = 0; A_halves && l < layers; ++l) A_halves[l] = mats[2 * l].halves && !whole;
  return run_batched(mats, MODE_INVERSE, info, workspace, workspace_bytes, stream);
}

int kfac_pi_damped_inverse_factored_batched(int layers, const int* dA, const int* dG,
                                            const float* const* A, const float* const* G,
                                            const float* damping, float* const* Ainv,
                                            float* const* Ginv, float* const* Afac,
                                            float* const* Gfac, int* info, void* workspace,
                                            size_t workspace_bytes, void* stream) {
  return factored_batched(layers, dA, dG, A, G, damping, Ainv, Ginv, Afac, Gfac, nullptr, info,
                          workspace, workspace_bytes, (hipStream_t)stream);
}

int kfac_pi_damped_inverse_halves_batched(int layers, const int* dA, const int* dG,
                                          const float* const* A, const float* const* G,
                                          const float* damping, float* const* Ainv,
                                          float* const* Ginv, float* const* Afac,
                                          float* const* Gfac, int* A_halves, int* info,
                                          void* workspace, size_t workspace_bytes, void* stream) {
  if (layers > 0 && !A_halves) return KFAC_ERR_ARG;
  return factored_batched(layers, dA, dG, A, G, damping, Ainv, Ginv, Afac, Gfac, A_halves, info,
                          workspace, workspace_bytes, (hipStream_t)stream);
}

size_t kfac_factor_complete_workspace_bytes(int count) {
  return count > 0 ? align256((size_t)count * sizeof(MatDesc)) : 0;
}

int kfac_factor_complete_batched(int count, const int* dims, float* const* factors,
                                 void* workspace, size_t workspace_bytes, void* stream_) {
  if (count < 0 || (count > 0 && (!dims || !factors))) return KFAC_ERR_ARG;
  if (count == 0) return KFAC_OK;
  if (!workspace || workspace_bytes < kfac_factor_complete_workspace_bytes(count))
    return KFAC_ERR_WORKSPACE;
  for (int i = 0; i < count; ++i)
    if (dims[i] <= 0 || dims[i] > 16384 || !factors[i]) return KFAC_ERR_ARG;
  hipStream_t stream = (hipStream_t)stream_;
  MatDesc* const table = (MatDesc*)workspace;
  for (int s0 = 0; s0 < count; s0 += SETUP_CHUNK) {
    DescChunk chunk{};
    const int cnt = std::min(SETUP_CHUNK, count - s0);
    for (int k = 0; k < cnt; ++k) {
      MatDesc& d = chunk.d[k];
      d.U = d.Y = factors[s0 + k];         // (the merge leaves W below the diagonal, and U12 is read before Y12 is written)
      d.n = dims[s0 + k];
      d.T = cdiv(d.n, DB);
      d.partner = -1;
      d.noinv = 1;
    }
    hipLaunchKernelGGL(inv_setup_kernel, dim3(1), dim3(SETUP_CHUNK), 0, stream, chunk, table, s0, cnt);
  }
  for (int s0 = 0; s0 < count; s0 += WL_MAX) {
    auto list = [&](auto&& items) {
      WorkList wl;
      wl.first = s0;
      wl.n = std::min(WL_MAX, count - s0);
      wl.cum[0] = 0;
      for (int i = 0; i < wl.n; ++i) wl.cum[i + 1] = wl.cum[i] + items(cdiv(dims[s0 + i], DB));
      for (int i = wl.n + 1; i <= WL_MAX; ++i) wl.cum[i] = wl.cum[wl.n];
      return wl;
    };
    const WorkList merges = list([](int T) { return T > 1 ? merge_tiles(T, 0) : 0; });
    const WorkList tiles = list([](int T) { return T * T; });
    if (merges.cum[merges.n] == 0) continue;
    KFAC_LAUNCH_TILE2(trtri_w_kernel, dim3(merges.cum[merges.n]), stream, table, 0, merges);
    KFAC_LAUNCH_TILE2(trtri_y_kernel, dim3(merges.cum[merges.n]), stream, table, 0, merges);
    hipLaunchKernelGGL(zero_lower_kernel, dim3(tiles.cum[tiles.n]), dim3(256), 0, stream, table, 1,
                       tiles);
  }
  return launch_status();
}

int kfac_cholesky_upper_batched(int count, const int* dims, const float* const* src,
                                float* const* dst, int* info, void* workspace,
                                size_t workspace_bytes, void* stream) {
  if (count < 0 || (count > 0 && (!dims || !src || !dst || !info))) return KFAC_ERR_ARG;
  std::vector<HostMat> mats(count);
  for (int i = 0; i < count; ++i) {
    if (dims[i] <= 0 || dims[i] > 16384 || !src[i] || !dst[i] || src[i] == dst[i])
      return KFAC_ERR_ARG;
    mats[i] = HostMat{src[i], dst[i], dims[i], 0.f, -1, 0, i};
  }
  return run_batched(mats, MODE_CHOLESKY, info, workspace, workspace_bytes, (hipStream_t)stream);
}

}  // extern "C"
