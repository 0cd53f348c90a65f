// fp32 MFMA tile engine for gfx950 (CDNA4, wave64), and what it shares with the engine on the bf16
// matrix cores (gemm_split.h), on which all products run but the per-sample gradients of a convolution.
//
// One workgroup of 256 threads (4 waves, 2x2) computes a 128x128 tile of
//     C[m][n] = sum_k  P(k, m) * Q(k, n)          k in [kbeg, kend)
// with v_mfma_f32_32x32x2_f32.  Each wave owns a 64x64 sub-tile (2x2 MFMA
// blocks, 64 accumulator registers).  Operands are described by functors that
// map (k, m) to a global-memory element, so the same engine serves matrices and the implicit
// im2col of a convolution, without ever materialising a transposed,
// concatenated or unfolded copy.
//
// Operand functor contract (details in operands.h):
//   static constexpr int layout;      KM: consecutive m are contiguous in memory
//                                     MK: consecutive k are contiguous in memory
//   MS mstate(int m) / KS kstate(int k, bool valid): per-index precomputation
//   unsigned off(MS, KS): byte offset for a raw buffer load; an element outside
//                         the operand gets an offset beyond the buffer and reads 0
// This engine takes MK operands: a chunk lies in LDS as lds[m][KC+4] and the MFMA lanes read
// ds_read_b128.  Within a chunk the k values are consumed in the order
//   step (j,s), lane half h  ->  k = 8j + 4h + s
// for both operands, which is a permutation of the reduction index and so does
// not change the product.
#pragma once
#include <type_traits>
#include <hip/hip_runtime.h>

namespace kfac {

constexpr int BM = 128;          // tile rows
constexpr int BN = 128;          // tile cols
constexpr int NTHREADS = 256;
constexpr int KC = 16;           // reduction depth per LDS stage, of either engine

enum { KM = 0, MK = 1 };

__host__ __device__ inline int tiles128(int d) { return (d + BM - 1) / BM; }

typedef float v16f __attribute__((ext_vector_type(16)));

// LDS pointers carry their address space explicitly: through a generic pointer
// the compiler emits FLAT loads/stores, whose completion is counted together
// with global loads, and the wait before the MFMAs would then also wait for the
// prefetch of the next chunk.
typedef __attribute__((address_space(3))) float lds_f;
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4f lds_f4;

// Division of an index below 2^31 by a divisor fixed per launch, as a multiply
// and a shift: with l = ceil(log2 d) and m = ceil(2^(31+l) / d) (which fits 32
// bits), floor(n / d) == (n * m) >> (31 + l) for every n < 2^31.  The operand
// functors turn a reduction index into (image, row, column) once per thread and
// chunk; a hardware-less integer division there costs about 40 instructions.
struct FastDiv {
  unsigned m, sh;
  FastDiv() = default;
  __host__ __device__ explicit FastDiv(unsigned d) {
    unsigned l = 0;
    while ((1ull << l) < d) ++l;
    sh = 31 + l;
    m = (unsigned)(((1ull << sh) + d - 1) / d);
  }
  __host__ __device__ __forceinline__ int div(int n) const {
    return (int)(((unsigned long long)(unsigned)n * m) >> sh);
  }
};

// ---- raw buffer addressing (see the operand contract in operands.h) ----------
constexpr unsigned INV_M = 0x80000000u;
constexpr unsigned INV_K = 0x40000000u;
constexpr long MAX_OPERAND_BYTES = 1L << 30;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const float* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, (int)MAX_OPERAND_BYTES,
                                           0x00020000);
}
__device__ __forceinline__ float buffer_load(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}
typedef unsigned v4u __attribute__((ext_vector_type(4)));
// four consecutive elements (dword-aligned); the range check covers the group as a whole
__device__ __forceinline__ v4f buffer_load4(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}

// An operand type with `static constexpr bool square = true` has its elements
// squared on the way into LDS (diagonal curvature: sums of squared gradients).
template <class T, class = void>
struct squares_elements : std::false_type {};
template <class T>
struct squares_elements<T, std::void_t<decltype(T::square)>> : std::bool_constant<T::square> {};

// An epilogue with `static constexpr bool reads_output = true` offers
// reads() / fetch(row, col) / store_with(row, col, v, old) next to store().
template <class T, class = void>
struct reading_epilogue : std::false_type {};
template <class T>
struct reading_epilogue<T, std::void_t<decltype(T::reads_output)>>
    : std::bool_constant<T::reads_output> {};

// ---------------------------------------------------------------------------
// global -> register -> LDS staging of one operand chunk (KC x ROWS elements)
// ---------------------------------------------------------------------------
constexpr int LDS_MK = KC + 4;                       // padded row of a chunk (conflict-free b128)
constexpr int CHUNK_FLOATS = LDS_MK * BM;
constexpr int SMEM_FLOATS = 4 * CHUNK_FLOATS;        // two stages of two operands, 40 KiB

template <class OP, int ROWS>
struct Stager {
  static_assert(OP::layout == MK, "this engine stages rows of consecutive k");
  static constexpr int CNT = KC * ROWS / NTHREADS;   // elements per thread
  static constexpr int MSTEP = NTHREADS / KC;        // rows per sweep
  typename OP::MS ms[CNT];
  float regs[CNT];
  unsigned onebits;    // element i is the constant 1 (and inside the k range)

  __device__ __forceinline__ void init(const OP& op, int m0) {
#pragma unroll
    for (int i = 0; i < CNT; ++i) ms[i] = op.mstate(m0 + (int)threadIdx.x / KC + MSTEP * i);
    onebits = 0;
  }

  // Issue the buffer loads of one chunk.  Elements outside the operand or the
  // k range come back as 0 from the hardware's range check; the loaded values
  // are not touched until commit, so nothing here waits on memory.
  __device__ __forceinline__ void fetch(const OP& op, int k0, int kend) {
    const __amdgpu_buffer_rsrc_t rs = op.rsrc();
    unsigned oneb = 0;
    const int k = k0 + (int)threadIdx.x % KC;
    const bool kin = k < kend;
    const typename OP::KS ks = op.kstate(k, kin);
#pragma unroll
    for (int i = 0; i < CNT; ++i) {
      regs[i] = buffer_load(rs, op.off(ms[i], ks));
      oneb |= (unsigned)(op.is_one(ms[i]) && kin) << i;
    }
    onebits = oneb;
  }

  __device__ __forceinline__ void commit(lds_f* tile) const {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < CNT; ++i)
      tile[(t / KC + MSTEP * i) * LDS_MK + t % KC] = ((onebits >> i) & 1u) ? 1.f : regs[i];
  }
};

// fragments of one operand for the 8 MFMA steps of a staged chunk: f[sub][4j+s]
__device__ __forceinline__ void load_frags(const lds_f* tile, int base, int r, int h,
                                           float (&f)[2][8]) {
#pragma unroll
  for (int sub = 0; sub < 2; ++sub)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const v4f v = *(const lds_f4*)(&tile[(base + 32 * sub + r) * LDS_MK + 8 * j + 4 * h]);
      f[sub][4 * j + 0] = v.x;
      f[sub][4 * j + 1] = v.y;
      f[sub][4 * j + 2] = v.z;
      f[sub][4 * j + 3] = v.w;
    }
}

// Position in C of accumulator element i of block (a, b) of the calling thread.
__device__ __forceinline__ void acc_coords(int m0, int n0, int a, int b, int i, int& row,
                                           int& col) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  row = m0 + (wave >> 1) * 64 + 32 * a + 8 * (i >> 2) + 4 * h + (i & 3);
  col = n0 + (wave & 1) * 64 + 32 * b + r;
}

// The MFMAs of k-steps [S0, S1) of a chunk.
template <int S0, int S1>
__device__ __forceinline__ void mma_slice(const float (&fa)[2][8], const float (&fb)[2][8],
                                          v16f (&acc)[2][2]) {
#pragma unroll
  for (int s = S0; s < S1; ++s)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[a][s], fb[b][s], acc[a][b], 0, 0, 0);
}

// ---------------------------------------------------------------------------
// The tile engine.  EPI::store_at((a*2 + b)*16 + i, value) receives every accumulator of the
// calling thread, in order (acc_coords gives its position).
// ---------------------------------------------------------------------------
template <class OPP, class OPQ, class EPI>
__device__ __forceinline__ void gemm_tile(const OPP& P, const OPQ& Q, int m0, int n0, int kbeg,
                                          int kend, EPI& epi, float* smem) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int r = lane & 31;
  const int h = lane >> 5;
  const int wm = (wave >> 1) * 64;
  const int wn = (wave & 1) * 64;

  v16f acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;

  Stager<OPP, BM> sp;
  Stager<OPQ, BN> sq;
  sp.init(P, m0);
  sq.init(Q, n0);

  lds_f* const sm = (lds_f*)smem;
  constexpr int STAGE = 2 * CHUNK_FLOATS;

  const int nchunks = (kend - kbeg + KC - 1) / KC;
  if (nchunks > 0) {
    sp.fetch(P, kbeg, kend);
    sq.fetch(Q, kbeg, kend);
    sp.commit(sm);
    sq.commit(sm + CHUNK_FLOATS);
  }
  __syncthreads();

  for (int c = 0; c < nchunks; ++c) {
    const int cur = c & 1;
    const bool more = (c + 1) < nchunks;
    if (more) {
      sp.fetch(P, kbeg + (c + 1) * KC, kend);
      sq.fetch(Q, kbeg + (c + 1) * KC, kend);
    }
    const lds_f* const tpc = sm + cur * STAGE;
    lds_f* const tpn = sm + (cur ^ 1) * STAGE;
    float fa[2][8], fb[2][8];
    load_frags(tpc, wm, r, h, fa);
    load_frags(tpc + CHUNK_FLOATS, wn, r, h, fb);
    // The LDS writes of the NEXT chunk are issued between the MFMAs, so that they (and the
    // wait for the global loads that feed them) sit in their shadow instead of in
    // front of the barrier.
    mma_slice<0, 4>(fa, fb, acc);
    if (more) {
      sp.commit(tpn);
      sq.commit(tpn + CHUNK_FLOATS);
    }
    mma_slice<4, 8>(fa, fb, acc);
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) epi.store_at((a * 2 + b) * 16 + i, acc[a][b][i]);
}

// ---------------------------------------------------------------------------
// A tile whose reduction was cut into `nparts` pieces, each computed by a workgroup of its
// own that stored its raw 128x128 partial (EpiPartial) at parts + piece * 128 * 128: a
// workgroup of a LATER launch adds the pieces up in order and hands every element to the
// epilogue.  (Finishing in the same launch, by the piece that arrives last, was measured:
// the device-wide fences it needs write back and invalidate the whole L2 of an XCD each
// time, and the operand panels that the other workgroups share through that L2 with them.)
// ---------------------------------------------------------------------------
// (`stride`: floats from one piece of the tile to the next)
template <class EPI>
__device__ __forceinline__ void splitk_sum(const float* parts, int nparts, int m0, int n0,
                                           const EPI& epi, size_t stride = BM * BN) {
  constexpr int TILE = BM * BN;
  constexpr int PER_THREAD = TILE / 4 / NTHREADS;      // float4 groups per thread: 16
  // piece by piece, the 16 loads of a thread in flight together
  v4f acc[PER_THREAD];
#pragma unroll
  for (int i = 0; i < PER_THREAD; ++i)
    acc[i] = *reinterpret_cast<const v4f*>(parts + 4 * ((int)threadIdx.x + NTHREADS * i));
  for (int q = 1; q < nparts; ++q) {
    const float* p = parts + (size_t)q * stride;
    v4f v[PER_THREAD];
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i)
      v[i] = *reinterpret_cast<const v4f*>(p + 4 * ((int)threadIdx.x + NTHREADS * i));
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) acc[i] += v[i];
  }
#pragma unroll
  for (int i = 0; i < PER_THREAD; ++i) {
    const int e = 4 * ((int)threadIdx.x + NTHREADS * i);
    const int row = m0 + (e >> 7), col = n0 + (e & (BN - 1));
    epi.store(row, col, acc[i].x);
    epi.store(row, col + 1, acc[i].y);
    epi.store(row, col + 2, acc[i].z);
    epi.store(row, col + 3, acc[i].w);
  }
}

// Workgroups are handed to the 8 XCDs round-robin in dispatch order, and each
// XCD has its own L2.  This maps the dispatch index `id` of a 1-D problem of
// `total` work items so that every XCD walks a CONTIGUOUS range of items:
// neighbouring tiles, which share operand panels, then hit the same L2.
__device__ __forceinline__ int xcd_remap(int id, int total) {
  const int x = id & 7, q = total >> 3, r = total & 7;
  const int base = x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q;
  return base + (id >> 3);
}

// Workgroups go to the 8 XCDs round-robin by dispatch index g.  The n items of one
// product occupy the dispatch indices [c0, c0 + n); this permutation of [0, n) gives
// every XCD a contiguous run of them.
__device__ __forceinline__ int xcd_remap_range(int g, int c0, int n) {
  const int s = c0 & 7;
  const int v = g - c0 + s;        // index in a virtual range that starts at a multiple of 8
  const int x = v & 7;
  const int tv = n + s;
  int base = 0;
#pragma unroll
  for (int y = 0; y < 8; ++y) {
    const int cnt = ((tv - y + 7) >> 3) - (y < s ? 1 : 0);
    base += y < x ? cnt : 0;
  }
  return base + (v >> 3) - (x < s ? 1 : 0);
}


// Batched launches (one for many matrices or layers of different sizes) use a 1-D
// grid of exactly the workgroups needed: cum[i] is the first work item of the i-th
// listed matrix (table index first + i), cum[n] the grid size.  (A rectangular grid
// "largest tile count x matrices" would start tens of thousands of workgroups
// that only find out that their matrix is too small.)
constexpr int WL_MAX = 128;
struct WorkList {
  int n, first;
  int cum[WL_MAX + 1];
};

// matrix (table index) and local work item of work item `item` of the list
__device__ __forceinline__ void work_find_item(const WorkList& wl, int item, int& mat,
                                               int& local) {
  int lo = 0, hi = wl.n;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (wl.cum[mid] <= item) lo = mid; else hi = mid;
  }
  mat = wl.first + lo;
  local = item - wl.cum[lo];
}

// ... of the calling workgroup, in a launch whose grid is the list
__device__ __forceinline__ void work_find(const WorkList& wl, int& mat, int& local) {
  work_find_item(wl, (int)blockIdx.x, mat, local);
}

// tile index t (0-based, row-major over the upper triangle incl. diagonal of a
// T x T block grid) -> (bi, bj), bi <= bj
__device__ __forceinline__ void upper_tile(int t, int T, int& bi, int& bj) {
  int i = 0;
  int rowlen = T;
  // closed form guess then fix-up (T is at most a few hundred)
  const float fT = 2.f * T + 1.f;
  i = (int)((fT - sqrtf(fT * fT - 8.f * (float)t)) * 0.5f);
  if (i < 0) i = 0;
  if (i > T - 1) i = T - 1;
  // start(i) = i*T - i*(i-1)/2
  while (i > 0 && (i * T - (i * (i - 1)) / 2) > t) --i;
  while (i + 1 < T && ((i + 1) * T - ((i + 1) * i) / 2) <= t) ++i;
  (void)rowlen;
  bi = i;
  bj = i + (t - (i * T - (i * (i - 1)) / 2));
}

}  // namespace kfac
