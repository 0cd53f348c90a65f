// Host-side helpers shared by the C-ABI translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/kfac_hip.h"

namespace kfac {

inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// Dynamic LDS sizes are registered once per kernel (required above 64 KiB, as
// for the 138 KiB of the diagonal-block kernel; harmless below).
bool enable_large_lds(const void* kernel, int bytes);

#define KFAC_LAUNCH_TILE2(kernel, grid, stream, ...)                                         \
  do {                                                                                       \
    constexpr int lds_bytes_ = kfac::SplitCfg<2>::SMEM_BYTES;                           \
    if (kfac::enable_large_lds((const void*)(kernel), lds_bytes_))                           \
      hipLaunchKernelGGL((kernel), (grid), dim3(kfac::NTHREADS), lds_bytes_, (stream),       \
                         __VA_ARGS__);                                                       \
  } while (0)

// A factor of a stride-1, bias-free Conv2d by spatial correlations
// (factor_conv_taps.hip).  conv_a_taps returns -1 when the geometry is not
// covered; the caller then uses the im2col kernel.
bool conv_a_taps_applicable(int c, int kh, int kw, int sh, int sw, int add_bias);
size_t conv_a_taps_workspace(int n, int c, int H, int W, int kh, int kw, int ph, int pw, int dh,
                             int dw);
double conv_a_taps_executed_flops(int n, int c, int H, int W, int kh, int kw, int ph, int pw,
                                  int dh, int dw);   // 0 when the geometry is not covered
int conv_a_taps(const float* x, int n, int c, int H, int W, int kh, int kw, int ph, int pw, int dh,
                int dw, float alpha, float beta, const float* A_prev, float* A, void* workspace,
                size_t workspace_bytes, hipStream_t stream);

// Copies a small host table to device memory at `dev` (4-byte aligned, `bytes` rounded up to
// a multiple of 4 are written) as kernel arguments of a few tiny launches on `stream`: no
// hipMemcpy, so the caller stays capturable and never waits for the device.  The host
// memory may be reused as soon as this returns.
void upload_table(const void* host, size_t bytes, void* dev, hipStream_t stream);

// The stride-1 k x k input factors of several layers at once (factor_conv_taps.hip): every
// geometry must be one that conv_a_taps covers (conv_a_taps_workspace(...) > 0).
struct TapsJob {
  const float* x;
  int n, c, H, W, kh, kw, ph, pw, dh, dw;
  float alpha, beta;
  const float* A_prev;
  float* A;
};
size_t conv_a_taps_grouped_workspace(int count, const TapsJob* jobs);
double conv_a_taps_grouped_executed_flops(int count, const TapsJob* jobs);
int conv_a_taps_grouped(int count, const TapsJob* jobs, void* workspace, size_t workspace_bytes,
                        hipStream_t stream);

// Blocks per piece of the cut reductions of a launch of 128x128 tiles (0: none is cut).
// `work` = sum over the tiles of their reduction length in blocks, `longest` = the longest
// of them: with the work spread evenly over the chip's resident workgroups (2 per CU) the
// launch would last work / 512 block times, and it cannot end before its longest tile does
// (which shares its compute unit with another workgroup until the launch thins out).
// Where the longest tile is the longer of the two, reductions are cut into pieces that are
// work items of the same launch and store raw partial tiles; a short launch afterwards adds
// the pieces of every cut tile up in order (splitk_sum).
// MIN_PIECE_BLOCKS: a shorter piece writes and reads its partial for too little work.
// Preconditioning of a 784-1000-1000-10 network / a conv net (1600, 3201) / slim and full
// ResNet-50 with pieces of at least 1, 2, 3, 4 blocks: 207 176 172 187 / 252 219 185 194 /
// 565 562 540 538 / 988 992 992 995 us (4 blocks and work / 768: 192 / 195 / 546 / 1113).
constexpr int MIN_PIECE_BLOCKS = 3;
constexpr int RESIDENT_TILES = 512;
inline int piece_blocks(long work, int longest) {
  const long even = work / RESIDENT_TILES + 1;
  if (longest <= MIN_PIECE_BLOCKS || 3 * (long)longest <= 4 * even) return 0;
  const long pb = even / 2 > MIN_PIECE_BLOCKS ? even / 2 : MIN_PIECE_BLOCKS;
  return pb >= longest ? 0 : (int)pb;
}

// Chunks per item of a launch of factor products that hold `units` (tile, chunk) pairs, on tiles
// 64 w wide: `dflt` where the launch holds plenty of items at that length, shorter items where it
// would not fill the chip.  128-wide tiles: 1.5 times (output gradients of 32 images of 2048x7x7 /
// 1024x13x13 / 256x56x56 in 1.5 / 2 / 3 rounds: 79 / 87 / 98, 69 / 73 / 82, 73 / 78 / 91 us), or once
// where that would take items of less than 8 chunks (a strided pointwise layer, 256 rows, 588 items
// of 8 chunks 64 us, one round of 10 chunks 54).  64-wide tiles: once, with as many items as are resident
// (`resident_small`: five workgroups per CU; correlations, whose strips are short items, six).
// Output gradients of 32 images of 64x112x112 / six of 64x56x56 / 128x56x56 with 768, 1280, 1536 and
// 4096 items: 39 41 46 60 / 43 45 49 68 / 31 35 36 39 us; 3x3 inputs of 64x56x56, one layer / three, in
// 1280, 1536, 4096: 142 135 166 / 334 323 319; the stem of a ResNet-50 with 768 ... 4096: 181 168 162 170.
constexpr double RESIDENT_SMALL = 1280., RESIDENT_SMALL_CORR = 1536.;
inline long group_item_chunks(int w, double units, long dflt, double resident_small = RESIDENT_SMALL) {
  const double resident = w == 1 ? resident_small : RESIDENT_TILES;
  long t = (long)(units / ((w == 1 ? 1. : 1.5) * resident));
  if (t < 8) t = w == 1 ? 8 : std::max(8L, (long)(units / resident) + 1);
  return std::min(t, dflt);
}

// Tiles' worth of MFMA work in the T(T+1)/2 upper tiles of a symmetric product with T tiles
// per side, 64 w wide: of the 32x32 blocks of a diagonal tile the four waves compute 12 of 16 where it is
// 128 wide (three each, split_tile_tri), all four where it is 64 wide.
inline double syrk_tile_units(int T, int w) {
  return (double)T * (T - 1) / 2 + T * (w == 1 ? 1. : 3. / 4.);
}

inline int launch_status() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? KFAC_OK : KFAC_ERR_LAUNCH;
}

}  // namespace kfac
