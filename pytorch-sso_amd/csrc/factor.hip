// Kronecker factor builders: symmetric products  C = alpha * P^T P + beta * C
// over the upper-triangular 128x128 tiles of C, mirrored in the epilogue.
#include "common.h"
#include "operands.h"
#include "syrk_reduce.h"

#include <string.h>

#include <atomic>

namespace kfac {

// Which kernels already had their dynamic-LDS limit raised, per device.  A fixed table
// of atomics: trivially destructible, so nothing of this library runs at process exit
// (objects with destructors in a shared library are torn down in an order that other
// libraries' exit handlers do not expect).
bool enable_large_lds(const void* kernel, int bytes) {
  constexpr int MAX_DEVICES = 64, CAP = 96;
  static std::atomic<const void*> done[MAX_DEVICES][CAP];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  if (dev >= 0 && dev < MAX_DEVICES) {
    for (int i = 0; i < CAP; ++i) {
      const void* k = done[dev][i].load(std::memory_order_acquire);
      if (k == kernel) return true;
      if (k != nullptr) continue;
      if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) !=
          hipSuccess)
        return false;
      // publish in the first free slot from here on (two threads setting the attribute
      // of one kernel at the same time both succeed; a duplicate entry is harmless)
      for (; i < CAP; ++i) {
        const void* expected = nullptr;
        if (done[dev][i].compare_exchange_strong(expected, kernel, std::memory_order_acq_rel) ||
            expected == kernel)
          break;
      }
      return true;
    }
  }
  // table full or device index out of its range: set the attribute on every call
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) ==
         hipSuccess;
}

// WORDS: what a launch carries as arguments, four to a thread
template <int WORDS>
struct UploadChunk {
  uint4 w[WORDS / 4];
};
template <int WORDS>
__global__ __launch_bounds__(WORDS / 4) void upload_kernel(const UploadChunk<WORDS> chunk, unsigned* dst, int words) {
  const uint4 v = chunk.w[threadIdx.x];
  const int i = 4 * threadIdx.x;
  if (i < words) dst[i] = v.x;
  if (i + 1 < words) dst[i + 1] = v.y;
  if (i + 2 < words) dst[i + 2] = v.z;
  if (i + 3 < words) dst[i + 3] = v.w;
}
template <int WORDS>
static void upload_chunk(const char* host, size_t bytes, unsigned* dst, hipStream_t stream) {
  UploadChunk<WORDS> c;
  const size_t words = (bytes + 3) / 4;
  ((unsigned*)c.w)[words - 1] = 0;
  memcpy(c.w, host, bytes);
  hipLaunchKernelGGL(upload_kernel<WORDS>, dim3(1), dim3(WORDS / 4), 0, stream, c, dst, (int)words);
}

// 15 KiB a launch, as few launches as that takes, and 3.75 KiB where that is enough.  One behind the other the
// launches take what the host needs for them: with 1 / 3 / 3.75 / 7.5 / 15 KiB of arguments 2.8 / 2.9 / 3.0 / 3.2 / 3.6 us
// (the kernel itself 1.3 to 1.8).  The tables of a ResNet-50 are 26 launches of 3.75 KiB or 13 (a step with old inverses,
// from an idle device, 6026 -> 5937 us).
constexpr int UPLOAD_SMALL = 960, UPLOAD_WORDS = 3840;
void upload_table(const void* host, size_t bytes, void* dev, hipStream_t stream) {
  for (size_t at = 0; at < bytes; at += UPLOAD_WORDS * 4) {
    const size_t n = std::min(bytes - at, (size_t)UPLOAD_WORDS * 4);
    if (n <= UPLOAD_SMALL * 4)
      upload_chunk<UPLOAD_SMALL>((const char*)host + at, n, (unsigned*)((char*)dev + at), stream);
    else
      upload_chunk<UPLOAD_WORDS>((const char*)host + at, n, (unsigned*)((char*)dev + at), stream);
  }
}

// Tile configuration and k-split of a symmetric d x d product reduced over K:
// 64-wide tiles for small factors (a 128-wide tile would be mostly padding), 128-wide
// tiles otherwise; enough k-splits to fill the chip, each split at least 128 deep.
struct SyrkPlan {
  int w;        // 1 -> 64x64 tiles, 2 -> 128x128
  int ts;       // tile size
  int T;        // tiles per side
  int ntiles;   // upper-triangular tiles
  int splits;
  int cps;      // chunks (of KC) per split
};

static SyrkPlan plan_syrk(int d, long K) {
  SyrkPlan p;
  // 64-wide tiles up to 192 rows, and to 256 where the reduction is short: of 200 rows over 4096 / 16384 /
  // 32768 / 60000 / 100000 terms 13.8 / 24.7 / 34.1 / 51.1 / 74.1 us, on 128-wide tiles 18.4 / 26.9 / 31.2 / 40.7 /
  // 55.6; of 256 over the same 14.2 / 25.8 / 34.9 / 55.2 / 80.4 and 19.0 / 28.8 / 35.0 / 46.2 / 62.4.
  p.w = d <= 192 || (d <= 256 && K <= 24576) ? 1 : 2;
  p.ts = 64 * p.w;
  p.T = cdiv(d, p.ts);
  p.ntiles = p.T * (p.T + 1) / 2;
  const long nchunks = (K + KC - 1) / KC;
  // (64-wide: 32 images of 64x112x112 in 1280 / 1536 / 2048 workgroups 39.5 / 42.7 / 46.4 us, of the
  // 3x224x224 of a 7x7 stem 244 / 222 / 221)
  const long target = p.w == 1 ? 1536 : 512;
  long splits = target / p.ntiles;
  if (splits < 1) splits = 1;
  const long min_chunks = 128 / KC;      // each split at least 128 deep
  const long max_splits = nchunks / min_chunks > 0 ? nchunks / min_chunks : 1;
  if (splits > max_splits) splits = max_splits;
  long cps = (nchunks + splits - 1) / splits;
  if (cps < 1) cps = 1;
  splits = (nchunks + cps - 1) / cps;
  if (splits < 1) splits = 1;
  if (p.w == 2) {
    // Two workgroups per CU are resident and share its matrix cores; one that is left alone, the last
    // of an odd number, takes 1.5 times its share.  So the launch takes (workgroups on the fullest
    // CU, and a half if they are odd) x (chunks per split): more splits than fit at once take
    // time off some products and add to others.  Every extra split costs one more partial tile
    // written and read (the last term, in chunk times).  8192 rows of 1600 / 2176 in 5 / 3 splits
    // (2 workgroups on the fullest CU) 137 / 224 us, in 8 / 5 (3) 153 / 243; of 2304 / 2432 in 2 splits
    // (2) 286 / 297, in 4 (3) 264 / 272.
    const int ncu = 256;
    auto cost = [&](long s, long c) {
      const int on_one = cdiv((int)(s * p.ntiles), ncu);
      return (on_one + on_one % 2 * 0.5) * (c + 3) + (s > 1 ? 0.035 * s * p.ntiles : 0.);
    };
    double best = cost(splits, cps);
    long best_s = splits, best_cps = cps;
    for (long s = splits + 1; s <= max_splits && s * p.ntiles <= 3 * ncu; ++s) {
      const long c = (nchunks + s - 1) / s;
      if ((nchunks + c - 1) / c != s) continue;
      if (cost(s, c) < best) {
        best = cost(s, c);
        best_s = s;
        best_cps = c;
      }
    }
    splits = best_s;
    cps = best_cps;
  }
  p.splits = (int)splits;
  p.cps = (int)cps;
  return p;
}

// The plan of `terms` terms carried over to the `positions` that they take up: no more splits,
// so that the scratch is that of kfac_factor_workspace_bytes(d, terms).
static SyrkPlan stretch_plan(SyrkPlan p, int64_t positions) {
  const long nchunks = (long)((positions + KC - 1) / KC);
  p.cps = (int)((nchunks + p.splits - 1) / p.splits);
  p.splits = (int)((nchunks + p.cps - 1) / p.cps);
  return p;
}

template <class OP, int W>
__global__ __launch_bounds__(256, W == 2 ? 2 : 3) void syrk_kernel(OP op, int d, int K, int T, int ntiles,
                                                          int splits, int chunks_per_split,
                                                          float* C, const float* Cin,
                                                          float alpha, float beta, float* ws) {
  constexpr int TS = 64 * W;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  // work item = (split, tile), tile fastest: the tiles of one split read the
  // same rows of the input, so they are kept on one XCD
  const int item = xcd_remap(blockIdx.y * ntiles + blockIdx.x, ntiles * splits);
  const int tile = item % ntiles;
  const int split = item / ntiles;
  int bi, bj;
  upper_tile(tile, T, bi, bj);
  const int kbeg = split * chunks_per_split * KC;
  int kend = kbeg + chunks_per_split * KC;
  if (kend > K) kend = K;
  const EpiStore whole{C, d, d, d, alpha, beta, bi != bj, Cin};
  const EpiPartial part{ws + ((size_t)split * ntiles + tile) * (TS * TS), bi * TS, bj * TS, d, d, TS};
  syrk_tile<W>(op, bi, bj, kbeg, kend, splits == 1, whole, part, smem);
}

template <int TS>
__global__ __launch_bounds__(256) void syrk_reduce_kernel(const float* ws, int d, int T,
                                                           int ntiles, int splits, float* C,
                                                           const float* Cin, float alpha,
                                                           float beta) {
  syrk_reduce_many<TS>(ws, d, T, ntiles, splits, C, Cin, alpha, beta, blockIdx.x, blockIdx.y);
}

template <int TS>
__global__ __launch_bounds__(256) void syrk_reduce_tile_kernel(const float* ws, int d, int T,
                                                                int ntiles, int splits, float* C,
                                                                const float* Cin, float alpha,
                                                                float beta) {
  syrk_reduce_tile<TS>(ws, d, T, ntiles, splits, C, Cin, alpha, beta, blockIdx.x, blockIdx.y,
                       blockIdx.z);
}

template <class OP, int W>
static void launch_syrk_cfg(const OP& op, const SyrkPlan& p, int d, int64_t K, float alpha,
                            float beta, const float* Cin, float* C, void* workspace,
                            hipStream_t stream) {
  constexpr int TS = 64 * W;
  constexpr int lds_bytes = syrk_lds_bytes<W>();
  if (!enable_large_lds((const void*)syrk_kernel<OP, W>, lds_bytes)) return;
  hipLaunchKernelGGL((syrk_kernel<OP, W>), dim3(p.ntiles, p.splits), dim3(256), lds_bytes,
                     stream, op, d, (int)K, p.T, p.ntiles, p.splits, p.cps, C, Cin, alpha, beta,
                     (float*)workspace);
  if (p.splits > 16) {
    hipLaunchKernelGGL((syrk_reduce_kernel<TS>), dim3(p.ntiles, TS * (TS / 64)), dim3(256), 0,
                       stream, (const float*)workspace, d, p.T, p.ntiles, p.splits, C, Cin, alpha,
                       beta);
  } else if (p.splits > 1) {
    hipLaunchKernelGGL((syrk_reduce_tile_kernel<TS>), dim3(p.ntiles, TS / 32, TS / 64), dim3(256),
                       0, stream, (const float*)workspace, d, p.T, p.ntiles, p.splits, C, Cin,
                       alpha, beta);
  }
}

// `terms` terms at `K` index positions
template <class OP>
static int launch_syrk(const OP& op, int d, int64_t terms, int64_t K, float alpha, float beta,
                       const float* Cin, float* C, void* workspace, size_t workspace_bytes,
                       hipStream_t stream) {
  const SyrkPlan p = stretch_plan(plan_syrk(d, (long)terms), K);
  if (p.splits > 1) {
    const size_t need = (size_t)p.splits * p.ntiles * p.ts * p.ts * sizeof(float);
    if (workspace == nullptr || workspace_bytes < need) return KFAC_ERR_WORKSPACE;
  }
  if (p.w == 1)
    launch_syrk_cfg<OP, 1>(op, p, d, K, alpha, beta, Cin, C, workspace, stream);
  else
    launch_syrk_cfg<OP, 2>(op, p, d, K, alpha, beta, Cin, C, workspace, stream);
  return launch_status();
}

}  // namespace kfac

using namespace kfac;

extern "C" {

int kfac_abi_version(void) { return 2; }

size_t kfac_factor_workspace_bytes(int d, int64_t K) {
  if (d <= 0 || K <= 0) return 0;
  const SyrkPlan p = plan_syrk(d, (long)K);
  return p.splits > 1 ? (size_t)p.splits * p.ntiles * p.ts * p.ts * sizeof(float) : 0;
}

// Operand offsets are 30-bit byte offsets: an input larger than 1 GiB is consumed
// in slices along its leading dimension, each slice accumulating into C.
static int64_t slice_len(int64_t total, int64_t elems_per_unit) {
  const int64_t max_units = (MAX_OPERAND_BYTES / 4) / elems_per_unit;
  return max_units < 1 ? 0 : (total < max_units ? total : max_units);
}

// MFMA flops one launch_syrk executes: every (tile, split) workgroup runs whole chunks of
// KC reduction steps on a full ts x ts tile (padding and the k tail included); a diagonal
// tile leaves out its 32x32 blocks below the diagonal.
static double syrk_executed_flops(int d, int64_t terms, int64_t K) {
  const SyrkPlan p = plan_syrk(d, (long)terms);
  const double chunks = (double)((K + KC - 1) / KC);
  return syrk_tile_units(p.T, p.w) * chunks * KC * 2.0 * p.ts * p.ts;
}

double kfac_factor_executed_flops(int d, int64_t K) {
  if (d <= 0 || K <= 0) return 0.;
  return syrk_executed_flops(d, K, K);
}

double kfac_factor_conv_a_executed_flops(int n, int c, int H, int W, int kh, int kw, int sh,
                                         int sw, int ph, int pw, int dh, int dw, int add_bias) {
  if (n <= 0 || c <= 0 || H <= 0 || W <= 0 || kh <= 0 || kw <= 0 || sh <= 0 || sw <= 0 ||
      ph < 0 || pw < 0 || dh <= 0 || dw <= 0)
    return 0.;
  const int OH = (H + 2 * ph - dh * (kh - 1) - 1) / sh + 1;
  const int OW = (W + 2 * pw - dw * (kw - 1) - 1) / sw + 1;
  if (OH <= 0 || OW <= 0) return 0.;
  const int64_t image = (int64_t)c * H * W;
  const int64_t step = slice_len(n, image);
  if (step == 0) return 0.;
  const int d = c * kh * kw + (add_bias ? 1 : 0);
  double total = 0.;
  for (int64_t n0 = 0; n0 < n; n0 += step) {
    const int cnt = (int)(n - n0 < step ? n - n0 : step);
    if (kh == 1 && kw == 1 && sh == 1 && sw == 1 && ph == 0 && pw == 0 && !add_bias) {
      const int64_t terms = (int64_t)cnt * H * W;
      total += syrk_executed_flops(d, terms, (int64_t)cnt * padded_run(H * W));
      continue;
    }
    if (conv_a_taps_applicable(c, kh, kw, sh, sw, add_bias)) {
      const double t = conv_a_taps_executed_flops(cnt, c, H, W, kh, kw, ph, pw, dh, dw);
      if (t > 0.) {
        total += t;
        continue;
      }
    }
    const int64_t terms = (int64_t)cnt * OH * OW;
    total += syrk_executed_flops(d, terms, terms);
  }
  return total;
}

size_t kfac_factor_conv_a_workspace_bytes(int n, int c, int H, int W, int kh, int kw, int sh,
                                          int sw, int ph, int pw, int dh, int dw, int add_bias) {
  if (n <= 0 || c <= 0 || H <= 0 || W <= 0 || kh <= 0 || kw <= 0 || sh <= 0 || sw <= 0 ||
      ph < 0 || pw < 0 || dh <= 0 || dw <= 0)
    return 0;
  const int OH = (H + 2 * ph - dh * (kh - 1) - 1) / sh + 1;
  const int OW = (W + 2 * pw - dw * (kw - 1) - 1) / sw + 1;
  if (OH <= 0 || OW <= 0) return 0;
  const int64_t image = (int64_t)c * H * W;
  const int64_t step = slice_len(n, image);
  if (step == 0) return 0;
  const int d = c * kh * kw + (add_bias ? 1 : 0);
  size_t need = kfac_factor_workspace_bytes(d, step * OH * OW);
  if (conv_a_taps_applicable(c, kh, kw, sh, sw, add_bias)) {
    const size_t t = conv_a_taps_workspace((int)step, c, H, W, kh, kw, ph, pw, dh, dw);
    if (t > need) need = t;
    if (n % step) {
      const size_t t2 = conv_a_taps_workspace((int)(n % step), c, H, W, kh, kw, ph, pw, dh, dw);
      if (t2 > need) need = t2;
    }
  }
  return need;
}

int kfac_factor_linear(const float* x, int64_t rows, int f, int64_t ldx, int add_bias,
                       float alpha, float beta, const float* C_prev, float* C, void* workspace,
                       size_t workspace_bytes, void* stream) {
  if (!x || !C || rows <= 0 || f <= 0 || ldx < f) return KFAC_ERR_ARG;
  const int d = f + (add_bias ? 1 : 0);
  if ((int64_t)d * d * 4 > MAX_OPERAND_BYTES) return KFAC_ERR_ARG;
  const int64_t step = slice_len(rows, ldx);
  if (step == 0) return KFAC_ERR_ARG;
  for (int64_t r0 = 0; r0 < rows; r0 += step) {
    const int64_t cnt = rows - r0 < step ? rows - r0 : step;
    DenseKM op{x + r0 * ldx, nullptr, (int)ldx, d, add_bias ? 1 : 0};
    const int st = launch_syrk(op, d, cnt, cnt, alpha, r0 == 0 ? beta : 1.f,
                               r0 == 0 ? C_prev : nullptr, C, workspace, workspace_bytes,
                               (hipStream_t)stream);
    if (st != KFAC_OK) return st;
  }
  return KFAC_OK;
}

int kfac_factor_conv_a(const float* x, int n, int c, int H, int W, int kh, int kw, int sh, int sw,
                       int ph, int pw, int dh, int dw, int add_bias, float alpha, float beta,
                       const float* C_prev, float* C, void* workspace, size_t workspace_bytes,
                       void* stream) {
  if (!x || !C || n <= 0 || c <= 0 || H <= 0 || W <= 0 || kh <= 0 || kw <= 0 || sh <= 0 ||
      sw <= 0 || ph < 0 || pw < 0 || dh <= 0 || dw <= 0)
    return KFAC_ERR_ARG;
  if (H >= 16384 || W >= 16384 || kh * dh >= 16384 || kw * dw >= 16384) return KFAC_ERR_ARG;
  const int OH = (H + 2 * ph - dh * (kh - 1) - 1) / sh + 1;
  const int OW = (W + 2 * pw - dw * (kw - 1) - 1) / sw + 1;
  if (OH <= 0 || OW <= 0) return KFAC_ERR_ARG;
  const int64_t dd = (int64_t)c * kh * kw + (add_bias ? 1 : 0);
  if (dd * dd * 4 > MAX_OPERAND_BYTES) return KFAC_ERR_ARG;
  const int d = (int)dd;
  const int64_t image = (int64_t)c * H * W;
  const int64_t step = slice_len(n, image);   // (offsets into the padding are never used)
  if (step == 0) return KFAC_ERR_ARG;
  for (int64_t n0 = 0; n0 < n; n0 += step) {
    const int cnt = (int)(n - n0 < step ? n - n0 : step);
    const float bslice = n0 == 0 ? beta : 1.f;
    const float* prev = n0 == 0 ? C_prev : nullptr;
    if (kh == 1 && kw == 1 && sh == 1 && sw == 1 && ph == 0 && pw == 0 && !add_bias) {
      // a pointwise convolution: M is the input itself, viewed as [c, n*H*W]
      const int64_t terms = (int64_t)cnt * H * W;
      const int positions = padded_run(H * W);
      ConvG op{x + n0 * image, c, H * W, positions};
      const int st = launch_syrk(op, d, terms, (int64_t)cnt * positions, alpha, bslice, prev, C,
                                 workspace, workspace_bytes, (hipStream_t)stream);
      if (st != KFAC_OK) return st;
      continue;
    }
    if (conv_a_taps_applicable(c, kh, kw, sh, sw, add_bias)) {
      const int st = conv_a_taps(x + n0 * image, cnt, c, H, W, kh, kw, ph, pw, dh, dw, alpha,
                                 bslice, prev, C, workspace, workspace_bytes, (hipStream_t)stream);
      if (st == KFAC_OK) continue;
      if (st != -1) return st;
    }
    ConvA op{x + n0 * image, c, H, W, kh, kw, sh, sw, ph, pw, dh, dw, OH, OW, d, add_bias ? 1 : 0};
    const int64_t terms = (int64_t)cnt * OH * OW;
    const int st = launch_syrk(op, d, terms, terms, alpha, bslice, prev, C, workspace,
                               workspace_bytes, (hipStream_t)stream);
    if (st != KFAC_OK) return st;
  }
  return KFAC_OK;
}

int kfac_factor_conv_g(const float* g, int n, int c, int h, int w, float alpha, float beta,
                       const float* C_prev, float* C, void* workspace, size_t workspace_bytes,
                       void* stream) {
  if (!g || !C || n <= 0 || c <= 0 || h <= 0 || w <= 0) return KFAC_ERR_ARG;
  if ((int64_t)c * c * 4 > MAX_OPERAND_BYTES) return KFAC_ERR_ARG;
  const int64_t image = (int64_t)c * h * w;
  const int64_t step = slice_len(n, image);
  if (step == 0) return KFAC_ERR_ARG;
  for (int64_t n0 = 0; n0 < n; n0 += step) {
    const int cnt = (int)(n - n0 < step ? n - n0 : step);
    const int64_t terms = (int64_t)cnt * h * w;
    const int positions = padded_run(h * w);
    ConvG op{g + n0 * image, c, h * w, positions};
    const int st = launch_syrk(op, c, terms, (int64_t)cnt * positions, alpha, n0 == 0 ? beta : 1.f,
                               n0 == 0 ? C_prev : nullptr, C, workspace, workspace_bytes,
                               (hipStream_t)stream);
    if (st != KFAC_OK) return st;
  }
  return KFAC_OK;
}

}  // extern "C"
