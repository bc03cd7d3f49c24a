// C ABI for the matmul family: operand classification, kernel choice, launches.
#include <algorithm>
#include <cmath>

#include "gemm_16bit_small.h"
#include "gemm_f32_direct.h"
#include "gemm_impl.h"
#include "mg_deferred.h"
#include "mg_rows.h"

namespace mg {

static bool mult4(int64_t v) { return (v & 3) == 0; }

// Sums the (splits, batch, M, N) partial products of an fp32 product split along K.
static int launch_f32_splitk_reduce(const GemmArgs& g, const float* partial, int splits, hipStream_t stream) {
  const int64_t numel = g.batch * g.M * g.N;
  const unsigned blocks = static_cast<unsigned>(ceil_div(numel, 1024));  // four outputs per thread
  const float* bias = static_cast<const float*>(g.bias);
  if (bias)
    hipLaunchKernelGGL((gemm_splitk_reduce_kernel<float, true>), dim3(blocks), dim3(256), 0, stream, partial, bias,
                       static_cast<float*>(g.c), numel, numel, splits, static_cast<int>(g.N), epilogue_of<float>(g));
  else
    hipLaunchKernelGGL((gemm_splitk_reduce_kernel<float, false>), dim3(blocks), dim3(256), 0, stream, partial, bias,
                       static_cast<float*>(g.c), numel, numel, splits, static_cast<int>(g.N), epilogue_of<float>(g));
  MG_LAUNCH_CHECK();
  return MG_OK;
}

template <bool A_KC, bool B_KC, int TS>
static int launch_f32_pipe(const GemmArgs& g, hipStream_t stream) {
  const int tiles_m = static_cast<int>(ceil_div(g.M, TS));
  const int tiles_n = static_cast<int>(ceil_div(g.N, TS));
  const int64_t blocks = static_cast<int64_t>(tiles_m) * tiles_n * g.batch;
  if (blocks > 0x7fffffffLL) return fail(MG_ERR_INVALID, "matmul: too many output tiles");
  const int64_t lda = A_KC ? g.sam : g.sak;
  const int64_t ldb = B_KC ? g.sbn : g.sbk;
  const float* a = static_cast<const float*>(g.a);
  const float* b = static_cast<const float*>(g.b);
  const float* bias = static_cast<const float*>(g.bias);
  float* c = static_cast<float*>(g.c);
  const int M = static_cast<int>(g.M), N = static_cast<int>(g.N), K = static_cast<int>(g.K);
  const int batches = static_cast<int>(g.batch);
  // An output with fewer tiles than CUs (a 10-class head: 2048 x 10 from K = 4096 is 16
  // tiles) is split along K so that the device is filled; the partial tiles are summed in a
  // fixed order by the same reduction the 16-bit path uses.
  const int64_t cus = device_info().cu_count;
  int splits = 1;
  if (blocks < cus && g.K >= 1024) {
    splits = static_cast<int>(ceil_div(env_int("MOGRAD_HIP_GEMM_SPLITK_WG_PER_CU", 2) * cus, blocks));
    const int max_splits = static_cast<int>(g.K / env_int("MOGRAD_HIP_GEMM_SPLITK_MIN_K", 256));
    if (splits > max_splits) splits = max_splits;
    if (splits > 64) splits = 64;
  }
  if (splits > 1) {
    const int k_per_split = static_cast<int>(ceil_div(ceil_div(g.K, splits), kGemmBK) * kGemmBK);
    splits = static_cast<int>(ceil_div(g.K, k_per_split));
    const int64_t numel = g.batch * g.M * g.N;
    Scratch partial;
    MG_TRY(partial.take(static_cast<int64_t>(splits) * numel * static_cast<int64_t>(sizeof(float))));
    const int64_t work = blocks * splits;
    hipLaunchKernelGGL((gemm_f32_pipe_kernel<A_KC, B_KC, false, true, TS>), dim3(static_cast<unsigned>(work)),
                       dim3(kGemmThreads), 0, stream, a, b, bias, c, partial.as<float>(), M, N, K, lda, ldb, g.N, g.bsa,
                       g.bsb, g.M * g.N, tiles_m, tiles_n, batches, k_per_split, static_cast<int>(work),
                       GemmEpilogue<float>{nullptr, nullptr, 0});
    MG_LAUNCH_CHECK();
    return launch_f32_splitk_reduce(g, partial.as<float>(), splits, stream);
  }
  // The workgroups that are resident at once walk a larger problem.
  int64_t grid = (TS == 128 ? 2 : 4) * cus * env_int("MOGRAD_HIP_GEMM_F32_ROUNDS", 1);
  if (grid > blocks || env_int("MOGRAD_HIP_GEMM_F32_ROUNDS", 1) == 0) grid = blocks;
  float* no_partial = nullptr;
  if (bias)
    hipLaunchKernelGGL((gemm_f32_pipe_kernel<A_KC, B_KC, true, false, TS>), dim3(static_cast<unsigned>(grid)),
                       dim3(kGemmThreads), 0, stream, a, b, bias, c, no_partial, M, N, K, lda, ldb, g.N, g.bsa, g.bsb,
                       g.M * g.N, tiles_m, tiles_n, batches, K, static_cast<int>(blocks), epilogue_of<float>(g));
  else
    hipLaunchKernelGGL((gemm_f32_pipe_kernel<A_KC, B_KC, false, false, TS>), dim3(static_cast<unsigned>(grid)),
                       dim3(kGemmThreads), 0, stream, a, b, bias, c, no_partial, M, N, K, lda, ldb, g.N, g.bsa, g.bsb,
                       g.M * g.N, tiles_m, tiles_n, batches, K, static_cast<int>(blocks), epilogue_of<float>(g));
  MG_LAUNCH_CHECK();
  return MG_OK;
}

// dst (batch, rows, cols_to) = src (batch, rows, cols) with zero columns appended: the image of an
// operand that the copying kernels can read 16 bytes at a time.  cols_to is a whole number of
// 16-byte chunks and dst aligned to them; src may lie anywhere.  One thread per chunk; up to three arrays
// per launch.  Bound by its bytes, or by the launch for small arrays.
template <typename T>
struct PadJob {
  const T* src;
  T* dst;
  int64_t ld, batch_stride, chunks;  // chunks: of the whole array
  int rows, cols, cols_to;
};
template <typename T>
struct PadJobs {
  PadJob<T> job[3];
  int block_end[3];
};
template <typename T>
__global__ __launch_bounds__(256) void pad_columns_kernel(PadJobs<T> jobs) {
  const int b = blockIdx.x;
  const int which = b < jobs.block_end[0] ? 0 : b < jobs.block_end[1] ? 1 : 2;
  const PadJob<T>& j = jobs.job[which];
  const int64_t i = static_cast<int64_t>(b - (which ? jobs.block_end[which - 1] : 0)) * 256 + threadIdx.x;
  if (i >= j.chunks) return;
  constexpr int E = 16 / sizeof(T);
  const int per_row = j.cols_to / E;
  const int64_t row = i / per_row;
  const int c0 = static_cast<int>(i - row * per_row) * E;
  const T* src = j.src + row / j.rows * j.batch_stride + row % j.rows * j.ld + c0;
  reinterpret_cast<uint4*>(j.dst)[i] = gemm_gather_chunk(src, j.cols - c0);
}

// Collects the operands of one product that need such an image and makes them in one launch.
template <typename T>
struct PadCopies {
  PadJobs<T> jobs{};
  Scratch mem[3];
  int count = 0;
  int64_t blocks = 0;
  // The image of `src`, whose rows then lie `*ld` apart and batches `*batch_stride`.
  int add(const void** src, int64_t batch, int64_t rows, int64_t cols, int64_t* ld, int64_t* batch_stride) {
    constexpr int E = 16 / sizeof(T);
    // (long rows: whole cache lines, see deep_16bit_us)
    const int64_t unit = sizeof(T) == 2 && cols >= 2048 ? 64 : E, to = ceil_div(cols, unit) * unit;
    const int64_t images = *batch_stride == 0 ? 1 : batch;
    MG_TRY(mem[count].take(images * rows * to * static_cast<int64_t>(sizeof(T))));
    PadJob<T>& j = jobs.job[count];
    j = PadJob<T>{static_cast<const T*>(*src), mem[count].template as<T>(), *ld, *batch_stride, images * rows * (to / E),
                  static_cast<int>(rows), static_cast<int>(cols), static_cast<int>(to)};
    blocks += ceil_div(j.chunks, 256);
    for (int i = count; i < 3; ++i) jobs.block_end[i] = static_cast<int>(blocks);
    ++count;
    *src = j.dst;
    *ld = to;
    *batch_stride = images == 1 ? 0 : rows * to;
    return MG_OK;
  }
  int launch(hipStream_t stream) {
    if (count == 0 || blocks == 0) return MG_OK;
    if (blocks > 0x7fffffffLL) return fail(MG_ERR_INVALID, "matmul: operand too large");
    hipLaunchKernelGGL((pad_columns_kernel<T>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, jobs);
    MG_LAUNCH_CHECK();
    return MG_OK;
  }
};

// Outputs of one tile column (or row) of 16 take gemm_f32_direct_kernel's 16 x 16 tiles, others its
// 32 x 32 ones; four waves along k in either.
static int f32_direct_tile(int64_t M, int64_t N) { return std::min(M, N) <= 16 ? 16 : 32; }

template <bool A_KC, bool B_KC>
static int launch_f32_direct(const GemmArgs& g, hipStream_t stream) {
  const int tile = f32_direct_tile(g.M, g.N);
  const int64_t tiles_m = ceil_div(g.M, tile), tiles_n = ceil_div(g.N, tile);
  const int64_t blocks = tiles_m * tiles_n * g.batch;
  // K ranges: enough for a workgroup per CU, each with at least 256 of K.
  int splits = static_cast<int>(std::max<int64_t>(
      1, std::min({ceil_div(device_info().cu_count, blocks), g.K / env_int("MOGRAD_HIP_GEMM_SPLITK_MIN_K", 256),
                   static_cast<int64_t>(64)})));
  const int k_per_split = static_cast<int>(ceil_div(ceil_div(g.K, splits), 64) * 64);
  splits = static_cast<int>(ceil_div(g.K, k_per_split));
  if (blocks * splits > 0x7fffffffLL) return fail(MG_ERR_INVALID, "matmul: too many output tiles");
  Scratch partial;
  if (splits > 1) MG_TRY(partial.take(splits * g.batch * g.M * g.N * static_cast<int64_t>(sizeof(float))));
  const Gemm32Problem pr{static_cast<const float*>(g.a), static_cast<const float*>(g.b), static_cast<const float*>(g.bias),
                         static_cast<float*>(g.c), partial.as<float>(), static_cast<int>(g.M), static_cast<int>(g.N),
                         static_cast<int>(g.K), A_KC ? g.sam : g.sak, B_KC ? g.sbn : g.sbk, g.N, g.bsa, g.bsb, g.M * g.N,
                         static_cast<int>(tiles_m), static_cast<int>(tiles_n), static_cast<int>(g.batch), k_per_split,
                         splits, epilogue_of<float>(g)};
  const dim3 grid(static_cast<unsigned>(blocks * splits));
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, pr); };
  if (splits == 1) {
    if (tile == 16) launch(gemm_f32_direct_kernel<A_KC, B_KC, 16, false>);
    else launch(gemm_f32_direct_kernel<A_KC, B_KC, 32, false>);
    MG_LAUNCH_CHECK();
    return MG_OK;
  }
  if (tile == 16) launch(gemm_f32_direct_kernel<A_KC, B_KC, 16, true>);
  else launch(gemm_f32_direct_kernel<A_KC, B_KC, 32, true>);
  MG_LAUNCH_CHECK();
  return launch_f32_splitk_reduce(g, partial.as<float>(), splits, stream);
}

static bool mult8(int64_t v) { return (v & 7) == 0; }
// Into how many K ranges a 16-bit product of `blocks` output tiles is split (1: not at all):
// enough for `wg_per_cu` workgroups per CU, each with at least 256 of K.
static int splitk_16bit_splits(int64_t blocks, int64_t K, int wg_per_cu) {
  const int64_t cus = device_info().cu_count;
  if (blocks >= cus || K < 1024) return 1;
  int splits = static_cast<int>(ceil_div(wg_per_cu * cus, blocks));
  const int max_splits = static_cast<int>(K / env_int("MOGRAD_HIP_GEMM_SPLITK_MIN_K", 256));
  if (splits > max_splits) splits = max_splits;
  if (splits > 64) splits = 64;
  return splits < 1 ? 1 : splits;
}

// What a 16-bit product costs, in us, in workgroups of one kind of tile: `items` of them (K ranges included),
// each `steps` k-steps of 64.  A CU holds two workgroups of 128-row tiles, whose steps take 0.85 us (128 x
// 128) and 1.1 us (128 x 192) for the pair, 0.46 and 0.69 us where there is one at the end; 0.52 us where no CU has more than one
// 128 x 128 tile, whose steps then wait for weights that no cache holds ((700, 1536) <- 1536: 16.6 us, 12.9 with
// 64 x 64 tiles; (512, 3072) <- 1024 13.2, 11.5; (4096, 384) <- 1536 17.1, 14.9); a 256 x 256 tile, alone
// on its CU, 1.47 us (1.3 where CUs stay idle) and 1.5 us until its first MFMA.  `split_lines`: rows of a k-contiguous operand that do not start on
// cache lines, so that every 128 bytes of a copy are two lines, long enough to matter ((13037, 680) <- 7288: 177 us with 128 x 192
// tiles, 147 with 256 x 256 ones).  The launch, the last epilogue and writing the result, which the tiles of a round do
// together, come on top.  (From 40 products of 2048 to 32768 rows, 64 to 8192 columns and K 64 to 7288, most within 10 %; over 339
// of 32 to 16384 rows with weights from memory the choice is 0.2 % slower than the best kind of tile of each, five of them more than 5 %.)
static double deep_16bit_us(Gemm16Tile tile, double items, double steps, bool split_lines, double cus) {
  const double per_cu = std::ceil(items / cus);
  if (tile == kTile256) return 4.0 + per_cu * ((items < 0.75 * cus ? 1.3 : 1.47) * steps + 1.5);
  const double pairs = std::floor(per_cu / 2), odd = per_cu - 2 * pairs, f = split_lines ? 1.3 : 1.0;
  if (tile == kTile128) return 3.6 + f * steps * (0.85 * pairs + (pairs == 0 ? 0.52 : 0.46) * odd);
  // (alone on its CU a 128 x 192 tile's ends stand in the open: (8192, 384 <- 128) 6.3 us, 5.2 with 128 x 128)
  return 3.6 + f * steps * (1.1 * pairs + 0.69 * odd) + (pairs == 0 ? 0.7 : 0.0);
}
static double partials_us(double values) { return 2.6 + values * 8.0 / 3.5e6; }

// Which tiles a 16-bit product is done fastest with, and in how many K ranges.  kSmall: the 64 x 64 tiles of
// gemm_16bit_small.h, whose estimate (3.4 us for a launch and its ends, 0.24 us per step for each
// workgroup that a CU has to walk) comes from 80 products of 64 to 16384 rows, 64 to 3768 columns and K 64 to 16384.
constexpr int kSmall = 4;
struct Choice16 {
  int tile;
  int splits;
  double us = 1e30;
};
static Choice16 small_16bit(int64_t M, int64_t N, int64_t K, int64_t batch, double no_more_than = 1e30) {
  const double cus = device_info().cu_count, steps = std::ceil(static_cast<double>(K) / kG16BK);
  const double out = static_cast<double>(M) * N * batch * 2.0 / 5e6, tiles = static_cast<double>(ceil_div(M, kSmallT) * ceil_div(N, kSmallT) * batch);
  const int64_t most = std::max<int64_t>(1, std::min<int64_t>(64, K / env_int("MOGRAD_HIP_GEMM_SPLITK_MIN_K", 256)));
  Choice16 best{kSmall, 1};
  for (int s = 1; s <= 16 && (s == 1 || (s <= most && tiles * s <= 2 * cus && steps >= 4 * s)); ++s) {
    const double sums = s > 1 ? partials_us(tiles * s * kSmallT * kSmallT) : 0.0;
    if (sums >= std::min(best.us, no_more_than)) break;
    const double us = 3.4 + out + std::ceil(steps / s) * 0.24 * std::ceil(tiles * s / cus) + sums;
    if (us < best.us) best = Choice16{kSmall, s, us};
  }
  return best;
}
// (A search stops where the partial tiles alone, which grow with the ranges, cost more than the best form so far:
// every call makes this choice, (512, 512) <- 65536 from 71 estimates.)
static Choice16 choose_16bit(int64_t M, int64_t N, int64_t K, int64_t batch, bool split_lines) {
  const double cus = device_info().cu_count, steps = std::ceil(static_cast<double>(K) / kG16BK);
  const double out = static_cast<double>(M) * N * batch * 2.0 / 5e6;  // (rows off the 16-byte chunks: 0.8 us more in the larger tiles)
  const int64_t most = std::max<int64_t>(1, std::min<int64_t>(64, K / env_int("MOGRAD_HIP_GEMM_SPLITK_MIN_K", 256)));
  auto tiles_of = [&](int m, int n) { return static_cast<double>(ceil_div(M, m) * ceil_div(N, n) * batch); };
  Choice16 best{kTile128, 1};
  if (env_str("MOGRAD_HIP_GEMM_SPLITK_WG_PER_CU")) {
    best.splits = splitk_16bit_splits(static_cast<int64_t>(tiles_of(kGemmBM, kGemmBN)), K,
                                      env_int("MOGRAD_HIP_GEMM_SPLITK_WG_PER_CU", 2));
    return best;
  }
  auto offer = [&](int tile, int splits, double us) {
    if (us < best.us) best = Choice16{tile, splits, us};
  };
  for (int t = kTile128; t <= kTile256; ++t) {
    const double tiles = tiles_of(kGemm16TileM[t], kGemm16TileN[t]);
    for (int s = 1; s <= (t == kTile256 ? 1 : most); ++s) {
      const double sums = s > 1 ? partials_us(tiles * s * kGemm16TileM[t] * kGemm16TileN[t]) : 0.0;
      if (s > 1 && (tiles * (s - 1) >= 2 * cus || sums >= best.us)) break;
      const double us = deep_16bit_us(static_cast<Gemm16Tile>(t), tiles * s, std::ceil(steps / s), split_lines, cus);
      offer(t, s, us + out + (N % 8 ? 0.8 : 0.0) + sums);
    }
  }
  const Choice16 small = small_16bit(M, N, K, batch, best.us);
  return small.us < best.us ? small : best;
}
// The K range of one workgroup, a multiple of the k-step, and the number of ranges that leaves.
static int splitk_16bit_range(int64_t K, int* splits) {
  const int k_per_split = static_cast<int>(ceil_div(ceil_div(K, *splits), kG16BK) * kG16BK);
  *splits = static_cast<int>(ceil_div(K, k_per_split));
  return k_per_split;
}

// Sums the K ranges of a 16-bit product's partial tiles (gemm16_partial_floats) into C, or leaves that to
// mg_finish_deferred (same code, same order).
template <typename T>
static int launch_16bit_splitk_reduce(const GemmArgs& g, Scratch& partial_mem, int splits, hipStream_t stream) {
  const float* const partial = partial_mem.as<float>();
  const int64_t slice = gemm16_partial_floats(g.M, g.N, g.batch, 1);
  if (slice / 1024 > 0x7fffffffLL) return fail(MG_ERR_INVALID, "matmul: too many output tiles");
  if (g.deferred) {
    DeferredList* dl = deferred_current();
    dl->push(kDeferSplitK, partial, g.c, slice, static_cast<int>(g.M), static_cast<int>(g.N), splits, ceil_div(slice / 4, 1024));
    dl->hold(partial_mem);
    return MG_OK;
  }
  const unsigned blocks = static_cast<unsigned>(slice / 1024);  // whole tiles: four outputs per thread
  const T* bias = static_cast<const T*>(g.bias);
  T* c = static_cast<T*>(g.c);
  const int N = static_cast<int>(g.N), M = static_cast<int>(g.M), tiles_n = static_cast<int>(ceil_div(g.N, kGemmBN));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, stream, partial, bias, c, slice, slice, splits, N,
                       epilogue_of<T>(g), M, tiles_n);
  };
  if (bias) launch(gemm_splitk_reduce_kernel<T, true, true>);
  else launch(gemm_splitk_reduce_kernel<T, false, true>);
  MG_LAUNCH_CHECK();
  return MG_OK;
}

// ANY: operands of any alignment, at least 8 elements along the axis that each is contiguous along.
template <typename T, bool A_KC, bool B_KC, bool ANY = false>
static int launch_16bit_small(const GemmArgs& g, int splits, hipStream_t stream) {
  const int64_t tiles_m = ceil_div(g.M, kSmallT), tiles_n = ceil_div(g.N, kSmallT), tiles = tiles_m * tiles_n;
  const int k_per_split = splitk_16bit_range(g.K, &splits);
  const int64_t grid = splits > 1 ? gemm_split_grid(tiles, splits, g.batch) : tiles * g.batch;
  if (grid > 0x7fffffffLL) return fail(MG_ERR_INVALID, "matmul: too many output tiles");
  Scratch partial;
  if (splits > 1)
    MG_TRY(partial.take(gemm16_partial_floats(g.M, g.N, g.batch, splits) * static_cast<int64_t>(sizeof(float))));
  Gemm16Problem<T> pr{static_cast<const T*>(g.a), static_cast<const T*>(g.b), static_cast<const T*>(g.bias),
                      static_cast<T*>(g.c), partial.as<float>(), static_cast<int>(g.M), static_cast<int>(g.N),
                      static_cast<int>(g.K), A_KC ? g.sam : g.sak, B_KC ? g.sbn : g.sbk, g.N, g.bsa, g.bsb,
                      g.M * g.N, static_cast<int>(tiles_m), static_cast<int>(tiles_n), k_per_split, splits,
                      static_cast<int>(g.batch), epilogue_of<T>(g)};
  gemm16_gradient(g, pr);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream, pr);
  };
  if (splits > 1) launch(gemm_16bit_small_kernel<T, A_KC, B_KC, false, true, ANY>);
  else if (g.bias) launch(gemm_16bit_small_kernel<T, A_KC, B_KC, true, false, ANY>);
  else launch(gemm_16bit_small_kernel<T, A_KC, B_KC, false, false, ANY>);
  MG_LAUNCH_CHECK();
  return splits > 1 ? launch_16bit_splitk_reduce<T>(g, partial, splits, stream) : MG_OK;
}

// Operands whose tiles cannot be copied straight into LDS (see dispatch_16bit): the register-staged kernel.
template <typename T, bool A_KC, bool B_KC>
static int launch_16bit_staged(const GemmArgs& g, int splits, hipStream_t stream) {
  const int tiles_m = static_cast<int>(ceil_div(g.M, kGemmBM)), tiles_n = static_cast<int>(ceil_div(g.N, kGemmBN));
  const int64_t tiles = static_cast<int64_t>(tiles_m) * tiles_n;
  const int k_per_split = splits > 1 ? splitk_16bit_range(g.K, &splits) : static_cast<int>(g.K);
  const int64_t grid = splits > 1 ? gemm_split_grid(tiles, splits, g.batch) : tiles * g.batch;
  if (grid > 0x7fffffffLL) return fail(MG_ERR_INVALID, "matmul: too many output tiles");
  Scratch partial;
  if (splits > 1)
    MG_TRY(partial.take(gemm16_partial_floats(g.M, g.N, g.batch, splits) * static_cast<int64_t>(sizeof(float))));
  auto launch = [&](auto kernel, GemmEpilogue<T> ep, auto* c) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kGemmThreads), 0, stream, static_cast<const T*>(g.a),
                       static_cast<const T*>(g.b), static_cast<const T*>(g.bias), c, partial.as<float>(),
                       static_cast<int>(g.M), static_cast<int>(g.N), static_cast<int>(g.K), A_KC ? g.sam : g.sak,
                       B_KC ? g.sbn : g.sbk, g.N, g.bsa, g.bsb, g.M * g.N, tiles_m, tiles_n, k_per_split, splits,
                       static_cast<int>(g.batch), ep);
  };
  T* const c = static_cast<T*>(g.c);
  if (splits > 1) {
    launch(gemm_16bit_mfma_kernel<T, A_KC, B_KC, false, true>, GemmEpilogue<T>{nullptr, nullptr, 0}, c);
  } else if (g.c_f32) {
    if constexpr (!A_KC && !B_KC)
      launch(gemm_16bit_mfma_kernel<T, A_KC, B_KC, false, false, float>, epilogue_of<T>(g), static_cast<float*>(g.c));
  } else if (g.bias) {
    launch(gemm_16bit_mfma_kernel<T, A_KC, B_KC, true, false>, epilogue_of<T>(g), c);
  } else {
    launch(gemm_16bit_mfma_kernel<T, A_KC, B_KC, false, false>, epilogue_of<T>(g), c);
  }
  MG_LAUNCH_CHECK();
  return splits > 1 ? launch_16bit_splitk_reduce<T>(g, partial, splits, stream) : MG_OK;
}

// 16-bit MFMA path, split along K where the output has too few tiles to fill the device (dW of a narrow
// layer: reduction over thousands of rows into a small matrix).  `wide`: operands on 16-byte chunks.
// MOGRAD_HIP_GEMM16_PIPE overrides the choice of tiles: 0 the register-staged kernel, 64 the 64 x 64 tiles,
// 1 to 1999 the 128 x 128, 2xxx the 128 x 192, 4xxx the 256 x 256 ones.  (The K ranges are
// chosen with the tiles; a kernel that is asked for takes the same ones.)
template <typename T, bool A_KC, bool B_KC>
static int launch_16bit(const GemmArgs& g, bool wide, hipStream_t stream) {
  const int64_t tiles128 = ceil_div(g.M, kGemmBM) * ceil_div(g.N, kGemmBN) * g.batch;
  const int64_t lda = A_KC ? g.sam : g.sak, ldb = B_KC ? g.sbn : g.sbk;
  if (g.c_f32 && (A_KC || B_KC)) return fail(MG_ERR_UNSUPPORTED, "matmul: no kernel for an fp32 result of this layout");
  if (!wide)
    return launch_16bit_staged<T, A_KC, B_KC>(
        g, splitk_16bit_splits(tiles128, g.K, env_int("MOGRAD_HIP_GEMM_SPLITK_WG_PER_CU", 2)), stream);
  Choice16 choice = choose_16bit(g.M, g.N, g.K, g.batch, g.K >= 1024 && ((A_KC && lda % 64 != 0) || (B_KC && ldb % 64 != 0)));
  if (const int64_t pipe = env_int("MOGRAD_HIP_GEMM16_PIPE", -1); pipe >= 0) {
    choice.tile = pipe == 0 ? -1 : pipe == 64 ? kSmall : pipe < 2000 ? kTile128 : pipe < 4000 ? kTile192 : kTile256;
    if (choice.tile == kTile256 && choice.splits > 1) choice.tile = kTile128;
  }
  if (choice.tile == kSmall) return launch_16bit_small<T, A_KC, B_KC>(g, choice.splits, stream);
  if (choice.tile < 0 || std::max(lda, ldb) > kGemmDeepMaxLd) return launch_16bit_staged<T, A_KC, B_KC>(g, choice.splits, stream);
  int splits = choice.splits;
  const int k_per_split = splits > 1 ? splitk_16bit_range(g.K, &splits) : static_cast<int>(g.K);
  Scratch partial;  // whole 128 x 128 tiles in accumulator order; the reduction maps them back onto the output
  if (splits > 1)
    MG_TRY(partial.take(gemm16_partial_floats(g.M, g.N, g.batch, splits) * static_cast<int64_t>(sizeof(float))));
  MG_TRY(launch_16bit_deep<T>(g, static_cast<Gemm16Tile>(choice.tile), splits, k_per_split, partial.as<float>(), stream));
  return splits > 1 ? launch_16bit_splitk_reduce<T>(g, partial, splits, stream) : MG_OK;
}

static bool generic_grid_fits(const GemmArgs& g) { return ceil_div(g.M, 64) <= 65535 && g.batch <= 65535; }

// fp32 products whose operands are each contiguous along one axis.
//   tiles copied into LDS, 128 x 128 where every CU gets one and the last round of them is not so
//   empty that 64 x 64 ones, 6 % slower in themselves, are done first ((8000, 600) <- 900, 315 large
//   tiles: 126 us against 89; (1390, 3016) <- 576: 80 against 58; (4096, 1024) <- 1024 74 against 81);
//   64 x 64 down to one for every second CU ((2048, 768) <- 768: 31 us against 55 with
//   128 x 128 and 42 straight from memory), fewer where a long reduction can be split as well
//   ((480, 160) <- 11200: 35 against 51);
//   operands that do not lie on 16-byte chunks are copied to rows that do, which takes a tile
//   per CU to pay ((1999, 1001) <- 767: 44 us against 59; (2587, 256) <- 256: 14 against 10);
//   everything smaller straight from memory (gemm_f32_direct.h).
// MOGRAD_HIP_GEMM_F32_TILE = 32 | 64 | 128 overrides the choice (32: straight from memory).
static int dispatch_f32(const GemmArgs& g_in, hipStream_t stream, bool* handled) {
  GemmArgs g = g_in;
  const bool a_kc = g.sak == 1, b_kc = g.sbk == 1;
  const int64_t cus = device_info().cu_count;
  const int64_t blocks128 = ceil_div(g.M, 128) * ceil_div(g.N, 128) * g.batch;
  const int64_t blocks64 = ceil_div(g.M, 64) * ceil_div(g.N, 64) * g.batch;
  const bool a_wide = (a_kc ? mult4(g.sam) && mult4(g.K) : mult4(g.sak) && mult4(g.M)) && mult4(g.bsa) && aligned16(g.a);
  const bool b_wide = (b_kc ? mult4(g.sbn) && mult4(g.K) : mult4(g.sbk) && mult4(g.N)) && mult4(g.bsb) && aligned16(g.b);
  const bool wide = a_wide && b_wide;
  // Next to no reduction and a large output (the dX of a 10-class head): neither the copies nor the
  // fragments have anything to reuse, and the plain kernel's stores are the widest.  For one of its
  // k-steps of 16 that holds whatever the alignment ((2048, 4096) <- 16: 13.0 us against 14.7 with 64 x 64
  // tiles and 15.7 with 128 x 128; 8192 x 8192 68, 81, 90), for two only against operands that would have to be
  // copied first (<- 20: 18.5, 14.9, 16.0; 94, 85, 91).  Its grid ends at 65535 batches.
  const bool plain = g.K < 32 && blocks64 >= cus && (g.K <= kGenericBK || !wide) && generic_grid_fits(g);
  *handled = !plain;
  if (plain) return MG_OK;
  const bool use64 = wide ? 2 * blocks64 >= cus || (8 * blocks64 >= cus && g.K >= 1024) ||
                                (g.K >= 4096 && 2.0 * g.batch * g.M * g.N * g.K >= 4e8)
                          : blocks64 >= cus;
  const bool use128 = blocks128 >= cus && g.K >= 32 && 4.0 * ceil_div(blocks128, cus) <= 1.06 * ceil_div(blocks64, cus);
  const int tile = env_int("MOGRAD_HIP_GEMM_F32_TILE", use128 ? 128 : use64 ? 64 : 32);
  if (tile == 32) {
    if (a_kc && b_kc) return launch_f32_direct<true, true>(g, stream);
    if (a_kc) return launch_f32_direct<true, false>(g, stream);
    if (b_kc) return launch_f32_direct<false, true>(g, stream);
    return launch_f32_direct<false, false>(g, stream);
  }
  PadCopies<float> pad;
  if (!a_wide) {
    if (a_kc) MG_TRY(pad.add(&g.a, g.batch, g.M, g.K, &g.sam, &g.bsa));
    else MG_TRY(pad.add(&g.a, g.batch, g.K, g.M, &g.sak, &g.bsa));
  }
  if (!b_wide) {
    if (b_kc) MG_TRY(pad.add(&g.b, g.batch, g.N, g.K, &g.sbn, &g.bsb));
    else MG_TRY(pad.add(&g.b, g.batch, g.K, g.N, &g.sbk, &g.bsb));
  }
  MG_TRY(pad.launch(stream));
#define MG_F32_PIPE(TS_)                                                       \
  do {                                                                         \
    if (a_kc && b_kc) return launch_f32_pipe<true, true, TS_>(g, stream);      \
    if (a_kc) return launch_f32_pipe<true, false, TS_>(g, stream);             \
    if (b_kc) return launch_f32_pipe<false, true, TS_>(g, stream);             \
    return launch_f32_pipe<false, false, TS_>(g, stream);                      \
  } while (0)
  if (tile == 64) MG_F32_PIPE(64);
  MG_F32_PIPE(128);
#undef MG_F32_PIPE
}

// Two k-contiguous 16-bit operands off the 16-byte chunks, in us: in place in 64 x 64 tiles that are staged through registers
// (0.43 us a step where a workgroup has its CU, 0.35 for each of several), and in the ragged variant's 128 x 128 ones.  From 1500
// products of 16 to 32768 rows and up to 8192 columns and K, within a tenth for most.
static double any_16bit_us(const GemmArgs& g, int splits, double cus) {
  const double tiles = static_cast<double>(g.batch * ceil_div(g.M, kSmallT) * ceil_div(g.N, kSmallT)) * splits, rounds = std::ceil(tiles / cus);
  return 3.4 + static_cast<double>(g.batch * g.M * g.N) / 2.5e6 + std::ceil(static_cast<double>(g.K) / kG16BK / splits) * (rounds == 1 ? 0.43 : 0.35 * rounds) +
         (splits > 1 ? partials_us(tiles * kSmallT * kSmallT) : 0.0);
}
static double ragged_16bit_us(const GemmArgs& g, double cus) {
  const int64_t tiles = g.batch * ceil_div(g.M, kGemmBM) * ceil_div(g.N, kGemmBN);
  int splits = splitk_16bit_splits(tiles, g.K, 2);
  const int k_per_split = splitk_16bit_range(g.K, &splits);
  const double items = static_cast<double>(tiles) * splits, per_cu = std::ceil(items / cus), pairs = std::floor(per_cu / 2), odd = per_cu - 2 * pairs;
  return 7.3 + static_cast<double>(g.batch * g.M * g.N) / 2.5e6 + k_per_split / kG16BK * (1.44 * pairs + (pairs == 0 ? 1.0 : 0.64) * odd) +
         (splits > 1 ? items * kGemmBM * kGemmBN * 5.0 / 3.5e6 : 0.0);
}

template <typename T>
static int dispatch_16bit(const GemmArgs& g_in, hipStream_t stream, bool* handled) {
  *handled = false;
  GemmArgs g = g_in;
  if (g.K <= 0) return MG_OK;
  // Each operand must be contiguous along k or along its other axis.  When leading
  // dimensions, extents and addresses are all multiples of 8 elements the tiles are copied
  // straight into LDS; otherwise they are staged through registers (the ragged variant), or,
  // where the product is long enough to pay for it, the operand is copied to rows that are.
  const bool a_mc = g.sam == 1;
  const bool b_nc = g.sbn == 1;
  // (fp32 weight gradients have kernels for dW's own layout alone, also where a width of 1 makes it both)
  const bool a_kc = g.sak == 1 && !(g.c_f32 && a_mc);
  const bool b_kc = g.sbk == 1 && !(g.c_f32 && b_nc);
  if (!((a_kc || a_mc) && (b_kc || b_nc))) return MG_OK;
  const bool a_wide = (a_kc ? mult8(g.sam) && mult8(g.K) : mult8(g.sak) && mult8(g.M)) && aligned16(g.a) && mult8(g.bsa);
  const bool b_wide = (b_kc ? mult8(g.sbn) && mult8(g.K) : mult8(g.sbk) && mult8(g.N)) && aligned16(g.b) && mult8(g.bsb);
  *handled = true;
  bool wide = a_wide && b_wide;
  PadCopies<T> pad;
  // The copy costs a launch and two passes over the operand, the ragged variant its slower staging:
  // two k-contiguous operands are as fast through it up to some 20 GFLOP ((2048, 1000) <- 1001:
  // 19.9 us against 23.7; (4000, 4001) <- 1025: 68 against 66), the transposing layouts only at a
  // few k-steps ((1999, 767) <- 1001: 51 against 28 us; (16384, 384) <- 65: 9 against 11).
  const bool copy_pays = a_kc && b_kc ? 2.0 * g.batch * g.M * g.N * g.K >= 2e10 : g.K >= 128;
  // 64 x 64 tiles that are staged through registers, whose steps take a third longer than copied ones, where they are done before
  // either: us of the routes before | now, (2048, 1000 <- 1001) 20.7 | 15.1, (700, 701 <- 703) 21.0 | 8.5, (300, 3001 <- 517) 15.1 | 7.4,
  // (5000, 333 <- 777) 21.1 | 12.9, (200, 8001 <- 1023) 28.4 | 15.6, (77, 164 <- 1681) 11.2 | 8.2.
  const int64_t pipe = env_int("MOGRAD_HIP_GEMM16_PIPE", -1);
  // (Of the transposing layouts short reductions stay with the ragged variant: (16, 4097 <- 4097) backward 44 | 54.)
  if (!wide && (a_kc ? g.K : g.M) >= 8 && (b_kc ? g.K : g.N) >= 8 && ((a_kc && b_kc) || g.K >= 128) && !env_str("MOGRAD_HIP_GEMM16_PAD") && (pipe == -1 || pipe == 64)) {
    const Choice16 small = small_16bit(g.M, g.N, g.K, g.batch);
    // (Up to three tiles to a CU: (700, 4400 <- 77) 8.8 | 8.3, 759 tiles; (1000, 4000 <- 141) 10.0 | 10.8, 1008; (966, 5920 <- 141)
    // 12.5 | 15.8, 1488.)
    const bool few = g.batch * ceil_div(g.M, 64) * ceil_div(g.N, 64) <= 3 * static_cast<int64_t>(device_info().cu_count);
    // (Long K in few tiles: the ragged variant's K ranges, (211, 2613 <- 4293) 23.7 | 33.9, (4430, 105 <- 3721) 23.0 | 30.2.)
    const double cus = device_info().cu_count;
    const bool ragged = a_kc && b_kc && !copy_pays && any_16bit_us(g, small.splits, cus) > ragged_16bit_us(g, cus);
    if (pipe == 64 || (few && !ragged && 1.35 * small.us <= choose_16bit(g.M, g.N, g.K, g.batch, false).us + 7.0)) {
      if (a_kc && b_kc) return launch_16bit_small<T, true, true, true>(g, small.splits, stream);
      if (a_kc) return launch_16bit_small<T, true, false, true>(g, small.splits, stream);
      if (b_kc) return launch_16bit_small<T, false, true, true>(g, small.splits, stream);
      return launch_16bit_small<T, false, false, true>(g, small.splits, stream);
    }
  }
  if (!wide && env_int("MOGRAD_HIP_GEMM16_PAD", copy_pays) != 0) {
    if (!a_wide) {
      if (a_kc) MG_TRY(pad.add(&g.a, g.batch, g.M, g.K, &g.sam, &g.bsa));
      else MG_TRY(pad.add(&g.a, g.batch, g.K, g.M, &g.sak, &g.bsa));
    }
    if (!b_wide) {
      if (b_kc) MG_TRY(pad.add(&g.b, g.batch, g.N, g.K, &g.sbn, &g.bsb));
      else MG_TRY(pad.add(&g.b, g.batch, g.K, g.N, &g.sbk, &g.bsb));
    }
    MG_TRY(pad.launch(stream));
    wide = true;
  }
  if (a_kc && b_kc) return launch_16bit<T, true, true>(g, wide, stream);
  if (a_kc) return launch_16bit<T, true, false>(g, wide, stream);
  if (b_kc) return launch_16bit<T, false, true>(g, wide, stream);
  return launch_16bit<T, false, false>(g, wide, stream);
}

template <typename T>
static int launch_generic(const GemmArgs& g, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>(ceil_div(g.N, 64)), static_cast<unsigned>(ceil_div(g.M, 64)),
                  static_cast<unsigned>(g.batch));
  if (!generic_grid_fits(g)) return fail(MG_ERR_INVALID, "matmul: shape exceeds the generic kernel's grid");
  const T* a = static_cast<const T*>(g.a);
  const T* b = static_cast<const T*>(g.b);
  const T* bias = static_cast<const T*>(g.bias);
  T* c = static_cast<T*>(g.c);
  if constexpr (sizeof(T) == 2) {
    if (g.c_f32) {
      hipLaunchKernelGGL((gemm_generic_kernel<T, false, float>), grid, dim3(256), 0, stream, a, b, bias, static_cast<float*>(g.c),
                         static_cast<int>(g.M), static_cast<int>(g.N), static_cast<int>(g.K), g.sam, g.sak, g.sbk, g.sbn, g.N,
                         g.bsa, g.bsb, g.M * g.N, epilogue_of<T>(g));
      MG_LAUNCH_CHECK();
      return MG_OK;
    }
  }
  if (bias)
    hipLaunchKernelGGL((gemm_generic_kernel<T, true>), grid, dim3(256), 0, stream, a, b, bias, c, static_cast<int>(g.M),
                       static_cast<int>(g.N), static_cast<int>(g.K), g.sam, g.sak, g.sbk, g.sbn, g.N, g.bsa, g.bsb,
                       g.M * g.N, epilogue_of<T>(g));
  else
    hipLaunchKernelGGL((gemm_generic_kernel<T, false>), grid, dim3(256), 0, stream, a, b, bias, c, static_cast<int>(g.M),
                       static_cast<int>(g.N), static_cast<int>(g.K), g.sam, g.sak, g.sbk, g.sbn, g.N, g.bsa, g.bsb,
                       g.M * g.N, epilogue_of<T>(g));
  MG_LAUNCH_CHECK();
  return MG_OK;
}

// Rows of at most this many of an fp32 operand without a unit stride are copied k-contiguous.
constexpr int64_t kThinRows = 128;

int gemm_dispatch(const char* who, const GemmArgs& g_in, hipStream_t stream) {
  GemmArgs g = g_in;
  if (!is_float_dtype(g.dtype)) return fail(MG_ERR_INVALID, "%s: unsupported dtype %s", who, dtype_name(g.dtype));
  if (g.batch < 0 || g.M < 0 || g.N < 0 || g.K < 0 || g.M > 0x7fffffffLL || g.N > 0x7fffffffLL || g.K > 0x7fffffffLL)
    return fail(MG_ERR_INVALID, "%s: bad shape batch=%lld M=%lld N=%lld K=%lld", who, static_cast<long long>(g.batch),
                static_cast<long long>(g.M), static_cast<long long>(g.N), static_cast<long long>(g.K));
  if (g.batch == 0 || g.M == 0 || g.N == 0) return MG_OK;
  if (!g.a || !g.b || !g.c) return fail(MG_ERR_INVALID, "%s: null pointer argument", who);

  // A thin fp32 operand that is contiguous along neither axis (every second column of a table) would leave
  // the whole product to the plain kernel, which walks a long K in few workgroups: it is copied first, a
  // small fraction of the other operand's bytes.
  Scratch a_copy, b_copy;
  if (g.dtype == MG_F32 && g.K >= 512) {
    const bool a_unit = g.sak == 1 || g.sam == 1, b_unit = g.sbk == 1 || g.sbn == 1;
    const bool a_thin = g.M <= kThinRows, b_thin = g.N <= kThinRows;
    auto copy = [&](Scratch& mem, const void** src, int64_t rows, int64_t* row_stride, int64_t* k_stride, int64_t* batch_stride) -> int {
      const int64_t images = *batch_stride == 0 ? 1 : g.batch;
      MG_TRY(mem.take(images * rows * g.K * static_cast<int64_t>(sizeof(float))));
      const int64_t shape[3] = {images, rows, g.K}, strides[3] = {*batch_stride, *row_stride, *k_stride};
      MG_TRY(mg_contiguous(*src, mem.as<float>(), 3, shape, strides, MG_F32, stream));
      *src = mem.as<float>();
      *row_stride = g.K, *k_stride = 1, *batch_stride = images == 1 ? 0 : rows * g.K;
      return MG_OK;
    };
    if (!a_unit && a_thin && (b_unit || b_thin)) MG_TRY(copy(a_copy, &g.a, g.M, &g.sam, &g.sak, &g.bsa));
    if (!b_unit && b_thin && (a_unit || a_thin)) MG_TRY(copy(b_copy, &g.b, g.N, &g.sbn, &g.sbk, &g.bsb));
  }
  if (g.dtype == MG_F32 && g.K > 0 && (g.sak == 1 || g.sam == 1) && (g.sbk == 1 || g.sbn == 1)) {
    bool handled = false;
    const int rc = dispatch_f32(g, stream, &handled);
    if (handled || rc != MG_OK) return rc;
  }
  if (g.dtype != MG_F32) {
    bool handled = false;
    const int rc = g.dtype == MG_BF16 ? dispatch_16bit<bf16_t>(g, stream, &handled)
                                      : dispatch_16bit<f16_t>(g, stream, &handled);
    if (handled || rc != MG_OK) return rc;
  }
  switch (g.dtype) {
    case MG_F32: return launch_generic<float>(g, stream);
    case MG_F16: return launch_generic<f16_t>(g, stream);
    default: return launch_generic<bf16_t>(g, stream);
  }
}

int colsum_dispatch(const void* a, void* dst, int64_t outer, int64_t reduce, int64_t inner, int dtype,
                    hipStream_t stream, bool dst_f32 = false);  // reduce.hip
int ln_bwd(const void* dy, const void* x, const void* gamma, const float* mean, const float* rstd, const void* residual,
           void* dx, void* dgamma, void* dbeta, int64_t rows, int64_t cols, float eps, int dtype,
           mg_stream stream);  // layer_norm.hip

// dX (M,K) = dY (M,N) W (N,K) and dW (N,K) = dY^T X of a 16-bit Linear layer in one launch
// (linear_bwd_16bit_kernel), dW split along the rows.  dW comes out bit for bit
// as from its own launch with the same number of K ranges, and so does dX unless its own launch would split it along N (fewer
// dX tiles than CUs): here dX is never split, the dW workgroups fill the device.
// *done = false: not such a shape, nothing launched.
// MOGRAD_HIP_LINEAR_BWD_ONE_LAUNCH=0 switches it off (benchmarks, tests of the equivalence).
// With `ln`, the launch's dX tiles continue as the backward of the LayerNorm whose output X is:
// `dx` then receives that LayerNorm's input gradient (added to
// what it holds when dx_accumulate), dY W itself is not stored, and the LayerNorm's dgamma and
// dbeta follow from one partial row per tile of 128 rows.  Only for the 128 x 384 tiles of a
// 384-wide input (K == 384); otherwise *done stays false.
struct LinearBwdLayerNorm {
  const void* x;       // the LayerNorm's input (M, K)
  const void* gamma;   // (K)
  const float* mean;   // (M)
  const float* rstd;
  void* dgamma;        // (K)
  void* dbeta;
};

// Inputs of 384 columns can take 128 x 384 output tiles, which hold whole rows of dX (eight waves, one workgroup
// per CU): taken for the LayerNorm backward that continues in them, when those tiles leave CUs free for dW's K ranges and
// the layer is wide enough.  dW's K ranges are then those of that launch, with and without the LayerNorm.
// MOGRAD_HIP_LINEAR_BWD_WIDE=0: as any other width, with the K ranges that dW has in a launch of its own.
static bool wide_linear_bwd(int64_t M, int64_t N, int64_t K) {
  return K == kGemm16TileN[kTileWide] && ceil_div(M, kGemmBM) < device_info().cu_count && N >= 768 &&
         env_int("MOGRAD_HIP_LINEAR_BWD_WIDE", 1) != 0;
}

// How the backward of a 16-bit layer goes out: in one launch, with which tiles and dW in how many K ranges, or in a
// launch for each product (tile < 0).  The least of these estimates, in us, is taken:
//   64 x 64 tiles (gemm_16bit_small.h): the longest chain of k-steps (of 64) in one workgroup, 0.217 us a step, dW's and
//     dX's together by 0.68 where they share CUs, dW's a fifth longer with db; the steps of all workgroups dealt over the
//     CUs, 0.192 us each, a sixth more where rows do not start on cache lines; of the two the longer, and a quarter of the
//     other.  What is read and written of X and W; K ranges 1.6 us and 0.0096 us a tile.
//   128-row tiles: chain and load as in deep_16bit_us, a chain's steps between the two figures there (it shares its
//     CU for a part of its life), by 0.84 in this launch, 1.02 where rows do not start on cache lines.  128 x 384 tiles,
//     which carry a LayerNorm's backward: 1.5 us a step, against a launch of its own for that (from 30 layers of
//     1024 to 32000 rows, 10 %).
//   a launch for each product, and 7 us of one or two more for the sum of dY's rows.  Off the 16-byte chunks dW is the
//     register-staged kernel's, 5 us more: (114, 1771 <- 384) 20 us against 12.
// Fitted to what the choice costs over 390 layers, each by every route and 1 to 32 K ranges, fp32 gradients with deferred
// sums and 16-bit ones at once, caches warm and cold: a third of 64 to 16384 rows and any widths from 64 to 4608, a third as
// in transformer blocks of 64 to 2048 tokens, a third of 2048 to 20000.  On 300 others the route taken is 1.6 to 2.4,
// 0.2 to 1.4 and 2.7 to 3.0 % slower than each one's best.  So (320, 3072 <- 768) with db is one launch, 19.4 us
// against 26.6, (320, 1536 <- 6144) without is two, 29.0 against 33.2, and (1999, 1001 <- 768) takes 64 x 64 tiles, 22.7
// against 26.5.  The type of the gradients is not part of it: fp32 and 16-bit ones, deferred or not, come from the same sums.
// A range has at least 256 rows (64 x 64 tiles: 128).  MOGRAD_HIP_LINEAR_BWD_SMALL = 0 | 1 and MOGRAD_HIP_LINEAR_BWD_SPLITS override the choice.
static Choice16 choose_linear_bwd(int64_t M, int64_t N, int64_t K, bool with_dx, bool with_db) {
  const double cus = device_info().cu_count;
  const double steps_w = static_cast<double>(ceil_div(M, kG16BK)), steps_x = static_cast<double>(ceil_div(N, kG16BK));
  const double x_mb = static_cast<double>(M) * K * 2.0 / 1e6, w_mb = static_cast<double>(N) * K * 2.0 / 1e6;
  const bool on_lines = N % 64 == 0 && K % 64 == 0;  // rows that start on cache lines
  Choice16 small{kSmall, 1};
  {
    const double tiles_k = static_cast<double>(ceil_div(K, kSmallT));
    const double tiles_w = steps_x * tiles_k, tiles_x = with_dx ? steps_w * tiles_k : 0.0, chain_x = with_dx ? steps_x : 0.0;
    const double step = on_lines ? 0.192 : 0.225;
    for (int s = 1; s <= 32 && (s == 1 || M >= 128 * s); ++s) {
      if (s > 1 && 5.0 + tiles_w * s * 0.0096 >= small.us) break;
      const double len = std::ceil(steps_w / s), chain_w = with_db ? 1.22 * len : len;
      const double both = tiles_w * s + tiles_x > cus ? 0.68 * (chain_w + chain_x) : 0.0;
      const double chain = 0.217 * std::max({chain_w, chain_x, both});
      const double load = step * (tiles_w * s * len + tiles_x * steps_x) / cus;
      const double t = 3.4 + std::max(chain, load) + 0.25 * std::min(chain, load) +
                       (with_dx ? 0.38 * x_mb + 0.72 * w_mb : 0.43 * w_mb) + (s > 1 ? 1.6 + tiles_w * s * 0.0096 : 0.0);
      if (t < small.us) small.us = t, small.splits = s;
    }
    small.splits = static_cast<int>(env_int("MOGRAD_HIP_LINEAR_BWD_SPLITS", small.splits));
  }
  Choice16 deep{-1, 1};
  const int most = static_cast<int>(std::min<int64_t>(64, M / 256));
  auto offer = [&](Gemm16Tile t, int s) {  // false: more ranges are not worth a look
    const double tiles_k = static_cast<double>(ceil_div(K, kGemm16TileN[t]));
    const double tiles_w = static_cast<double>(ceil_div(N, kGemmBM)) * tiles_k * s, tiles_x = static_cast<double>(ceil_div(M, kGemmBM)) * tiles_k;
    const double len = std::ceil(steps_w / s), pair = t == kTile192 ? 1.1 : t == kTileWide ? 1.5 : 0.85, one = t == kTile192 ? 0.69 : t == kTileWide ? 1.5 : 0.46;
    const double slots = t == kTileWide ? cus : 2 * cus, sums = partials_us(tiles_w * kGemmBM * kGemm16TileN[t]);
    if (sums >= deep.us) return false;
    const double load = (tiles_w * len + tiles_x * steps_x) / slots * pair;
    const double chain = std::max(len, steps_x) * 0.5 * (pair + one);
    const double walk = std::max(load, chain) + (tiles_w + tiles_x > slots ? 0.5 * std::min(len, steps_x) * pair : 0.0);
    const double us = (t == kTileWide ? 4.0 + walk : 4.4 + (on_lines ? 0.84 : 1.02) * walk) + x_mb / 5.0 + sums;
    if (us < deep.us) deep = Choice16{t, s, us};
    return true;
  };
  const bool wide = wide_linear_bwd(M, N, K);
  const int64_t only = env_int("MOGRAD_HIP_LINEAR_BWD_TILE", 0);  // 128 | 192
  if (!with_dx || ceil_div(N, kGemmBM) * ceil_div(K, kGemmBN) >= cus) {  // dW fills the device unsplit: a launch for each product
  } else if (env_str("MOGRAD_HIP_LINEAR_BWD_WIDE") && env_int("MOGRAD_HIP_LINEAR_BWD_WIDE", 1) == 0) {
    const Gemm16Tile t = K % 192 == 0 ? kTile192 : kTile128;
    const int s = splitk_16bit_splits(ceil_div(N, kGemmBM) * ceil_div(K, kGemmBN), M, 1);
    if (s > 1) offer(t, s);
  } else if (wide) {
    for (int s = 2; s <= most && offer(kTileWide, s); ++s) {
    }
  } else {
    for (int s = 2; s <= most && only != 192 && offer(kTile128, s); ++s) {
    }
    for (int s = 2; s <= most && only != 128 && offer(kTile192, s); ++s) {
    }
  }
  if (deep.tile < 0 || (!wide && only == 0 && !env_str("MOGRAD_HIP_LINEAR_BWD_WIDE"))) {
    double apart = choose_16bit(N, K, M, 1, false).us + (with_db ? 7.0 : 0.0) + (mult8(N) && mult8(K) ? 0.0 : 5.0);
    if (with_dx) apart += choose_16bit(M, K, N, 1, N >= 1024 && N % 64 != 0).us;
    if (apart < deep.us) deep = Choice16{-1, 1, apart};
  }
  const bool is_small = small.us + (deep.tile == kTileWide ? std::max(6.0, 3.0 + x_mb) : 0.0) <= deep.us;
  // (A choice of the larger tiles' form is also one for them.)
  return env_int("MOGRAD_HIP_LINEAR_BWD_SMALL", is_small && !env_str("MOGRAD_HIP_LINEAR_BWD_WIDE")) != 0 ? small : deep;
}

template <typename T>
static int linear_bwd_one_launch(const void* dy, const void* x, const void* w, void* dx, void* dw, void* db, int64_t M,
                                 int64_t N, int64_t K, const void* relu_mask, bool dx_accumulate, hipStream_t stream,
                                 bool* done, bool* db_done, const LinearBwdLayerNorm* ln) {
  *done = false;
  *db_done = false;
  if (env_int("MOGRAD_HIP_LINEAR_BWD_ONE_LAUNCH", 1) == 0 || env_str("MOGRAD_HIP_GEMM16_PIPE")) return MG_OK;
  if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL) return MG_OK;
  // Widths that are no multiple of 8 (a 65-symbol vocabulary): rows of dY, or of X and W, start
  // at odd addresses, which the copies into LDS cannot take.  Those arrays are first copied to
  // rows of the next multiple of 8, zeros behind (`pads` below); dX, dW and db keep their shape.
  const bool pad_n = !mult8(N) || !aligned16(dy), pad_k = !mult8(K) || !aligned16(x) || (dx && !aligned16(w));
  const int64_t cus = device_info().cu_count;
  const Choice16 choice = choose_linear_bwd(M, N, K, dx != nullptr, db != nullptr);
  if (choice.tile < 0) return MG_OK;
  // 64 x 64 tiles read arrays that are at least 8 wide from wherever they start.  That saves the copies, a launch of 2.4 us and
  // their bytes, and makes the steps of the longer of the two walks longer: dX's over N by 0.1 us a step, 0.2 where its last tile
  // of columns is cut off, dW's over M by 0.22, by 0.15 of what the copies of X and W leave of that.  With the copies | without,
  // (64, 1001 <- 192) 9.7 | 8.8, (64, 2601 <- 192) 15.9 | 17.3, (64, 1001 <- 200) 10.0 | 10.3, (64, 2601 <- 200) 15.9 | 21.2;
  // (406, 1832 <- 83) 14.0 | 17.0, (675, 149 <- 2391) 15.4 | 12.6, (700, 701 <- 703) 14.1 | 11.8; (2587, 101 <- 256) 12.7 | 11.1,
  // (1481, 299 <- 1088) 16.1 | 19.2, (1344, 77 <- 2240) 13.8 | 16.2.  Longer products are faster with the copies ((1999, 1001 <- 768)
  // 22.3 | 24.5; (300, 3001 <- 517) 24.9 | 30.4).  Over 3400 layers of 16 to 8192 rows and 16 to 4096 columns this takes 0.4 % more
  // time than the better of the two for each, the copies always 20 %.  MOGRAD_HIP_LINEAR_BWD_ANY = 0 | 1 overrides it.
  const double longer_x = !dx ? 0.0 : (K % 64 == 0 ? 0.1 : 0.2) * static_cast<double>(ceil_div(N, 64));
  const double longer_w = (pad_k ? 0.15 : 0.22) * static_cast<double>(ceil_div(ceil_div(M, 64), std::max(choice.splits, 1)));
  const double copied = (pad_n ? static_cast<double>(M) * N : 0.0) + (pad_k ? static_cast<double>(K) * (dx ? M + N : M) : 0.0);
  const bool any_pays = choice.us <= 15.0 && std::max(longer_x, longer_w) <= 2.4 + 4.0 * copied / 3.7e6;
  const bool any = choice.tile == kSmall && (pad_n || pad_k) && N >= 8 && K >= 8 && !env_str("MOGRAD_HIP_GEMM16_PAD") &&
                   env_int("MOGRAD_HIP_LINEAR_BWD_ANY", any_pays) != 0;
  const bool small = choice.tile == kSmall, wide = choice.tile == kTileWide;
  if (ln && (!wide || relu_mask || pad_n || pad_k || !aligned16(ln->x) || !aligned16(ln->gamma) || !aligned16(dx))) return MG_OK;
  // (without the LayerNorm the same K ranges in 128 x 192 tiles, two workgroups per CU)
  const Gemm16Tile deep = wide && !ln ? kTile192 : static_cast<Gemm16Tile>(small ? kTile128 : choice.tile);
  const int tile = small ? kSmallT : kGemmBM;  // rows of an output tile
  const int tiles_kk = static_cast<int>(ceil_div(K, small ? kSmallT : kGemm16TileN[deep]));
  const int w_tiles_m = static_cast<int>(ceil_div(N, tile));
  const int64_t w_tiles = static_cast<int64_t>(w_tiles_m) * tiles_kk;
  const int x_tiles_m = static_cast<int>(ceil_div(M, tile));
  const int64_t x_tiles = dx ? static_cast<int64_t>(x_tiles_m) * tiles_kk : 0;  // (a first layer's dX is not wanted)
  int splits = choice.splits;
  const bool split_sums = splits > 1 || !small;
  const int k_per_split = splits > 1 ? splitk_16bit_range(M, &splits) : static_cast<int>(M);
  const int64_t n_dw = split_sums ? gemm_split_grid(w_tiles, splits, 1) : w_tiles;
  if (n_dw + x_tiles > 0x7fffffffLL) return MG_OK;

  int64_t ldy = N, ldx = K, ldw = K;
  if (!small && std::max(N, K) + 8 > kGemmDeepMaxLd) return MG_OK;
  PadCopies<T> pads;
  int64_t no_batch = 0;
  if (pad_n && !any) MG_TRY(pads.add(&dy, 1, M, N, &ldy, &no_batch));
  if (pad_k && !any) {
    MG_TRY(pads.add(&x, 1, M, K, &ldx, &no_batch));
    if (dx) MG_TRY(pads.add(&w, 1, N, K, &ldw, &no_batch));
  }
  MG_TRY(pads.launch(stream));

  Scratch partial;
  const int64_t numel = N * K;
  const int64_t slice = gemm16_partial_floats(N, K, 1, 1);  // whole tiles per K range
  if (split_sums) MG_TRY(partial.take(static_cast<int64_t>(splits) * slice * static_cast<int64_t>(sizeof(float))));
  const T* dyt = static_cast<const T*>(dy);
  const Gemm16Problem<T> pw{dyt, static_cast<const T*>(x), nullptr, static_cast<T*>(dw), partial.as<float>(),
                            static_cast<int>(N), static_cast<int>(K), static_cast<int>(M),
                            ldy, ldx, K, 0, 0, numel, w_tiles_m, tiles_kk, k_per_split, splits, 1,
                            GemmEpilogue<T>{nullptr, nullptr, 0}};
  const Gemm16Problem<T> px{dyt, static_cast<const T*>(w), nullptr, static_cast<T*>(dx), nullptr,
                            static_cast<int>(M), static_cast<int>(K), static_cast<int>(N),
                            ldy, ldw, K, 0, 0, M * K, x_tiles_m, tiles_kk, static_cast<int>(N), 1, 1,
                            GemmEpilogue<T>{dx_accumulate ? static_cast<const T*>(dx) : nullptr,
                                            static_cast<const T*>(relu_mask), 0}};
  // The bias gradient rides along: the dW workgroups of the first tile column sum the dY
  // tiles they hold over their K range, and the finishing kernel adds the ranges.  No second
  // pass over dY: (16384, 1536 <- 384) with db 71 -> 60.5 us against dX, dW and a separate
  // mg_sum_axis.  MOGRAD_HIP_LINEAR_BWD_BIAS_IN_LAUNCH=0: the separate column sum.
  Gemm16Problem<T> pw2 = pw;
  DeferredList* const dl = deferred_current();
  pw2.partial_stream = dl != nullptr && env_int("MOGRAD_HIP_DEFER_NT_STORE", 1) != 0;  // see gemm16_gradient
  Scratch db_part;
  int groups = 0;
  const bool db_here = db && env_int("MOGRAD_HIP_LINEAR_BWD_BIAS_IN_LAUNCH", 1) != 0;
  auto launch_small = [&](auto aligned, auto ragged) {
    hipLaunchKernelGGL((any ? ragged : aligned), dim3(static_cast<unsigned>(n_dw + x_tiles)), dim3(kGemmThreads), 0, stream, pw2, px,
                       static_cast<int>(n_dw));
  };
  if (!split_sums) {
    // nothing to sum: where the gradients are wanted in fp32 they are written so here
    if (dl && dl->out_dtype == MG_F32) {
      pw2.c32 = static_cast<float*>(dw);
      if (db_here) pw2.colsum32 = static_cast<float*>(db);
    } else if (db_here) {
      pw2.colsum = static_cast<T*>(db);
    }
    launch_small(linear_bwd_small_16bit_kernel<T, false, false>, linear_bwd_small_16bit_kernel<T, false, true>);
    MG_LAUNCH_CHECK();
    *db_done = db_here;
    *done = true;
    return MG_OK;
  }
  if (db_here) {
    groups = splits;
    MG_TRY(db_part.take(static_cast<int64_t>(groups) * N * static_cast<int64_t>(sizeof(float))));
    pw2.colsum_part = db_part.as<float>();
  }
  Scratch ln_part_g, ln_part_b;
  if (ln) {
    MG_TRY(ln_part_g.take(static_cast<int64_t>(x_tiles_m) * K * static_cast<int64_t>(sizeof(float))));
    MG_TRY(ln_part_b.take(static_cast<int64_t>(x_tiles_m) * K * static_cast<int64_t>(sizeof(float))));
    Gemm16Problem<T> px2 = px;
    px2.ln = Gemm16LayerNormBwd<T>{static_cast<const T*>(ln->x), static_cast<const T*>(ln->gamma), ln->mean, ln->rstd,
                                   ln_part_g.as<float>(), ln_part_b.as<float>()};
    MG_TRY(launch_linear_bwd_deep<T>(pw2, px2, kTileWide, n_dw, x_tiles, stream));
  } else if (small) {
    launch_small(linear_bwd_small_16bit_kernel<T, true, false>, linear_bwd_small_16bit_kernel<T, true, true>);
    MG_LAUNCH_CHECK();
  } else {
    MG_TRY(launch_linear_bwd_deep<T>(pw2, px, deep, n_dw, x_tiles, stream));
  }
  if (ln) {  // the tiles' partial rows of dgamma / dbeta: summed now, or left on the deferred list
    reduce_partials_or_defer<T>(ln_part_g, static_cast<T*>(ln->dgamma), &ln_part_b, static_cast<T*>(ln->dbeta), x_tiles_m,
                                K, static_cast<int>(cus), stream);
    MG_LAUNCH_CHECK();
  }
  const int dw_blocks = static_cast<int>(slice / 1024);  // 256 threads, four consecutive partial values each
  const int db_blocks = groups > 0 ? static_cast<int>(ceil_div(N, 64)) : 0;
  if (dl) {
    // The sums of the K ranges are left to mg_finish_deferred (same code, same order).
    dl->push(kDeferSplitK, partial.as<float>(), dw, slice, static_cast<int>(N), static_cast<int>(K), splits,
             ceil_div(slice / 4, 1024));
    dl->hold(partial);
    if (groups > 0) {
      dl->push(kDeferBiasRows, db_part.as<float>(), db, 0, 0, static_cast<int>(N), groups, ceil_div(db_blocks, 4));
      dl->hold(db_part);
    }
    *db_done = groups > 0;
    *done = true;
    return MG_OK;
  }
  hipLaunchKernelGGL((linear_bwd_finish_kernel<T>), dim3(static_cast<unsigned>(dw_blocks + db_blocks)), dim3(256), 0,
                     stream, partial.as<float>(), static_cast<T*>(dw), static_cast<int>(N), slice, splits,
                     static_cast<int>(K), dw_blocks, db_part.as<float>(), static_cast<T*>(db), groups,
                     static_cast<int>(N));
  MG_LAUNCH_CHECK();
  *db_done = groups > 0;
  *done = true;
  return MG_OK;
}

// The same for an fp32 layer small enough for gemm_f32_direct_kernel's tiles: dX, dW and db in one
// launch, dW split along the rows only when its tiles leave CUs idle and there are rows enough
// (then a finishing launch follows, or the sum is deferred).  Up to 2 GFLOP for both products: below
// that the launches saved and the filled device outweigh the direct kernel's lower rate.
// MOGRAD_HIP_LINEAR_BWD_ONE_LAUNCH=0 switches it off.
static int linear_bwd_f32_one_launch(const void* dy, const void* x, const void* w, void* dx, void* dw, void* db, int64_t M,
                                     int64_t N, int64_t K, const void* relu_mask, bool dx_accumulate, hipStream_t stream,
                                     bool* done, bool* db_done) {
  *done = false;
  *db_done = false;
  if (env_int("MOGRAD_HIP_LINEAR_BWD_ONE_LAUNCH", 1) == 0) return MG_OK;
  if (M <= 0 || N <= 0 || K <= 0 || (dx ? 4.0 : 2.0) * M * N * K > 1e6 * env_int("MOGRAD_HIP_LINEAR_BWD_F32_MFLOP", 2000)) return MG_OK;
  if (M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL) return MG_OK;
  constexpr int kTile = 32;
  const int64_t tiles_m = ceil_div(M, kTile), tiles_n = ceil_div(N, kTile), tiles_k = ceil_div(K, kTile);
  const int64_t x_blocks = dx ? tiles_m * tiles_k : 0, w_blocks = tiles_n * tiles_k;
  // a large dX with next to no reduction (a 10-class head): see dispatch_f32
  if (N < 32 && x_blocks >= 4 * device_info().cu_count) return MG_OK;
  int splits = static_cast<int>(
      std::max<int64_t>(1, std::min({ceil_div(device_info().cu_count, w_blocks), M / 256, static_cast<int64_t>(64)})));
  const int k_per_split = static_cast<int>(ceil_div(ceil_div(M, splits), 64) * 64);
  splits = static_cast<int>(ceil_div(M, k_per_split));
  const int64_t n_dw = w_blocks * splits;
  if (n_dw + x_blocks > 0x7fffffffLL) return MG_OK;
  const int64_t numel = N * K;
  Scratch partial, db_part;
  if (splits > 1) {
    MG_TRY(partial.take(splits * numel * static_cast<int64_t>(sizeof(float))));
    if (db) MG_TRY(db_part.take(splits * N * static_cast<int64_t>(sizeof(float))));
  }
  const float* dyf = static_cast<const float*>(dy);
  Gemm32Problem pw{dyf, static_cast<const float*>(x), nullptr, static_cast<float*>(dw), partial.as<float>(),
                   static_cast<int>(N), static_cast<int>(K), static_cast<int>(M), N, K, K, 0, 0, numel,
                   static_cast<int>(tiles_n), static_cast<int>(tiles_k), 1, k_per_split, splits,
                   GemmEpilogue<float>{nullptr, nullptr, 0}};
  pw.colsum = !db ? nullptr : splits > 1 ? db_part.as<float>() : static_cast<float*>(db);
  const Gemm32Problem px{dyf, static_cast<const float*>(w), nullptr, static_cast<float*>(dx), nullptr,
                         static_cast<int>(M), static_cast<int>(K), static_cast<int>(N), N, K, K, 0, 0, M * K,
                         static_cast<int>(tiles_m), static_cast<int>(tiles_k), 1, static_cast<int>(N), 1,
                         GemmEpilogue<float>{dx_accumulate ? static_cast<const float*>(dx) : nullptr,
                                             static_cast<const float*>(relu_mask), 0}};
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(n_dw + x_blocks)), dim3(256), 0, stream, pw, px,
                       static_cast<int>(n_dw));
  };
  if (splits > 1) launch(linear_bwd_f32_kernel<kTile, true>);
  else launch(linear_bwd_f32_kernel<kTile, false>);
  MG_LAUNCH_CHECK();
  *done = true;
  *db_done = db != nullptr;
  if (splits == 1) return MG_OK;
  const int dw_blocks = static_cast<int>(ceil_div(numel, 1024));
  const int db_blocks = db ? static_cast<int>(ceil_div(N, 64)) : 0;
  if (DeferredList* dl = deferred_current()) {
    dl->push(kDeferSplitRows, partial.as<float>(), dw, numel, static_cast<int>(N), static_cast<int>(K), splits,
             ceil_div(ceil_div(numel, 4), 1024));
    dl->hold(partial);
    if (db) {
      dl->push(kDeferBiasRows, db_part.as<float>(), db, 0, 0, static_cast<int>(N), splits, ceil_div(db_blocks, 4));
      dl->hold(db_part);
    }
    return MG_OK;
  }
  hipLaunchKernelGGL((linear_bwd_finish_kernel<float, false>), dim3(static_cast<unsigned>(dw_blocks + db_blocks)), dim3(256),
                     0, stream, partial.as<float>(), static_cast<float*>(dw), static_cast<int>(N), numel, splits,
                     static_cast<int>(K), dw_blocks, db_part.as<float>(), static_cast<float*>(db), splits,
                     static_cast<int>(N));
  MG_LAUNCH_CHECK();
  return MG_OK;
}

// Whether the `_deferred` entry point that runs on this thread wants fp32 gradients of 16-bit tensors.
static bool gradients_in_f32(int dtype) {
  const DeferredList* dl = deferred_current();
  return dl && dl->out_dtype == MG_F32 && dtype != MG_F32;
}

// db (N) = the column sums of dY (M, N): in the tensors' type, or as the running `_deferred` entry point wants them.
static int linear_bwd_bias(const void* dy, void* db, int64_t M, int64_t N, int dtype, hipStream_t stream) {
  return colsum_dispatch(dy, db, 1, M, N, dtype, stream, gradients_in_f32(dtype));
}

// dx may be null: the gradients of the weights alone.
// *done: dX and dW are on their way; *db_done: so is db (else the caller sums dY's columns).
int linear_bwd_products(const void* dy, const void* x, const void* w, void* dx, void* dw, void* db, int64_t M, int64_t N,
                        int64_t K, const void* relu_mask, bool dx_accumulate, int dtype, hipStream_t stream, bool* done,
                        bool* db_done, const LinearBwdLayerNorm* ln = nullptr) {
  *done = false;
  *db_done = false;
  if (dtype == MG_BF16)
    return linear_bwd_one_launch<bf16_t>(dy, x, w, dx, dw, db, M, N, K, relu_mask, dx_accumulate, stream, done, db_done, ln);
  if (dtype == MG_F16)
    return linear_bwd_one_launch<f16_t>(dy, x, w, dx, dw, db, M, N, K, relu_mask, dx_accumulate, stream, done, db_done, ln);
  if (dtype == MG_F32 && !ln)
    return linear_bwd_f32_one_launch(dy, x, w, dx, dw, db, M, N, K, relu_mask, dx_accumulate, stream, done, db_done);
  return MG_OK;
}

}  // namespace mg

extern "C" {

int mg_matmul(const void* a, const void* b, void* dst, int64_t batch, int64_t M, int64_t N, int64_t K, int64_t lda0,
              int64_t lda1, int64_t ldb0, int64_t ldb1, int64_t batch_stride_a, int64_t batch_stride_b, int dtype,
              mg_stream stream) {
  mg::GemmArgs g{a, b, nullptr, dst, batch, M, N, K, lda0, lda1, ldb0, ldb1, batch_stride_a, batch_stride_b, dtype};
  return mg::gemm_dispatch("matmul", g, mg::to_stream(stream));
}

int mg_matmul_bt(const void* a, const void* b, void* dst, int64_t batch, int64_t M, int64_t N, int64_t K, int64_t lda0,
                 int64_t lda1, int64_t ldb0, int64_t ldb1, int64_t batch_stride_a, int64_t batch_stride_b, int dtype,
                 mg_stream stream) {
  // B arrives as (N, K): element (k, n) of the product's right operand is b[n * ldb0 + k * ldb1].
  mg::GemmArgs g{a, b, nullptr, dst, batch, M, N, K, lda0, lda1, ldb1, ldb0, batch_stride_a, batch_stride_b, dtype};
  return mg::gemm_dispatch("matmul", g, mg::to_stream(stream));
}

int mg_matmul_bias_bt(const void* a, const void* b, const void* bias, void* dst, int64_t batch, int64_t M, int64_t N,
                      int64_t K, int64_t lda0, int64_t lda1, int64_t ldb0, int64_t ldb1, int64_t batch_stride_a,
                      int64_t batch_stride_b, int dtype, mg_stream stream) {
  if (!bias) return mg::fail(MG_ERR_INVALID, "matmul_bias: null bias pointer");
  mg::GemmArgs g{a, b, bias, dst, batch, M, N, K, lda0, lda1, ldb1, ldb0, batch_stride_a, batch_stride_b, dtype};
  return mg::gemm_dispatch("matmul_bias", g, mg::to_stream(stream));
}

int mg_matmul_bt_add(const void* a, const void* b, const void* residual, void* dst, int64_t batch, int64_t M, int64_t N,
                     int64_t K, int64_t lda0, int64_t lda1, int64_t ldb0, int64_t ldb1, int64_t batch_stride_a,
                     int64_t batch_stride_b, int dtype, mg_stream stream) {
  if (!residual) return mg::fail(MG_ERR_INVALID, "matmul_add: null residual pointer");
  mg::GemmArgs g{a, b, nullptr, dst, batch, M, N, K, lda0, lda1, ldb1, ldb0, batch_stride_a, batch_stride_b, dtype};
  g.residual = residual;
  return mg::gemm_dispatch("matmul_add", g, mg::to_stream(stream));
}

int mg_matmul_bias_relu_bt(const void* a, const void* b, const void* bias, void* dst, int64_t batch, int64_t M, int64_t N,
                           int64_t K, int64_t lda0, int64_t lda1, int64_t ldb0, int64_t ldb1, int64_t batch_stride_a,
                           int64_t batch_stride_b, int dtype, mg_stream stream) {
  if (!bias) return mg::fail(MG_ERR_INVALID, "matmul_bias_relu: null bias pointer");
  mg::GemmArgs g{a, b, bias, dst, batch, M, N, K, lda0, lda1, ldb1, ldb0, batch_stride_a, batch_stride_b, dtype};
  g.relu = 1;
  return mg::gemm_dispatch("matmul_bias_relu", g, mg::to_stream(stream));
}

static int linear_bwd_impl(const void* dy, const void* x, const void* w, void* dx, void* dw, void* db, int64_t M,
                           int64_t N, int64_t K, bool dx_accumulate, bool x_is_relu_output, int dtype, mg_stream stream) {
  hipStream_t s = mg::to_stream(stream);
  if (x_is_relu_output && dx && !x) return mg::fail(MG_ERR_INVALID, "linear_bwd: x is needed as the relu mask");
  if (dw && dy && x && (w || !dx)) {
    bool done = false, db_done = false;
    MG_TRY(mg::linear_bwd_products(dy, x, w, dx, dw, db, M, N, K, x_is_relu_output ? x : nullptr, dx_accumulate, dtype,
                                   s, &done, &db_done));
    if (done) {
      if (db && !db_done) MG_TRY(mg::linear_bwd_bias(dy, db, M, N, dtype, s));
      return MG_OK;
    }
  }
  if (dx) {  // dX (M,K) = dY (M,N) x W (N,K): reduction over N, W read as an n-contiguous right operand
    mg::GemmArgs g{dy, w, nullptr, dx, 1, M, K, N, N, 1, K, 1, 0, 0, dtype};
    if (x_is_relu_output) {
      if (!x) return mg::fail(MG_ERR_INVALID, "linear_bwd: x is needed as the relu mask");
      g.relu_mask = x;  // (M, K), laid out like dX
    }
    if (dx_accumulate) g.residual = dx;
    MG_TRY(mg::gemm_dispatch("linear_bwd(dx)", g, s));
  }
  if (dw) {  // dW (N,K) = dY^T (N,M) x X (M,K): reduction over M, dY read as an m-contiguous left operand
    mg::GemmArgs g{dy, x, nullptr, dw, 1, N, K, M, 1, N, K, 1, 0, 0, dtype};
    g.deferred = mg::deferred_current() != nullptr;
    g.c_f32 = mg::gradients_in_f32(dtype);
    MG_TRY(mg::gemm_dispatch("linear_bwd(dw)", g, s));
  }
  if (db) MG_TRY(mg::linear_bwd_bias(dy, db, M, N, dtype, s));
  return MG_OK;
}

int mg_linear_bwd(const void* dy, const void* x, const void* w, void* dx, void* dw, void* db, int64_t M, int64_t N,
                  int64_t K, int dtype, mg_stream stream) {
  return linear_bwd_impl(dy, x, w, dx, dw, db, M, N, K, false, false, dtype, stream);
}

int mg_linear_bwd_fused(const void* dy, const void* x, const void* w, void* dx, void* dw, void* db, int64_t M, int64_t N,
                        int64_t K, int dx_accumulate, int x_is_relu_output, int dtype, mg_stream stream) {
  return linear_bwd_impl(dy, x, w, dx, dw, db, M, N, K, dx_accumulate != 0, x_is_relu_output != 0, dtype, stream);
}

int mg_linear_bwd_deferred(const void* dy, const void* x, const void* w, void* dx, void* dw, void* db, int64_t M,
                           int64_t N, int64_t K, int dx_accumulate, int x_is_relu_output, int dtype, int grad_dtype,
                           mg_deferred list, mg_stream stream) {
  if (!mg::is_float_dtype(dtype))
    return mg::fail(MG_ERR_INVALID, "linear_bwd_deferred: unsupported dtype %s", mg::dtype_name(dtype));
  MG_TRY(mg::deferred_check("linear_bwd_deferred", list, dtype, grad_dtype));
  if (M < 0 || N < 0 || K < 0) return mg::fail(MG_ERR_INVALID, "linear_bwd_deferred: negative size");
  // (every kernel of a Linear backward writes dW and db in the type that they are wanted in: no substitutes)
  mg::DeferredScope scope(static_cast<mg::DeferredList*>(list), dtype, grad_dtype);
  return linear_bwd_impl(dy, x, w, dx, dw, db, M, N, K, dx_accumulate != 0, x_is_relu_output != 0, dtype, stream);
}

int mg_linear_bwd_layer_norm_bwd(const void* dy, const void* x, const void* w, const void* ln_x, const void* gamma,
                                 const float* mean, const float* rstd, void* dx, void* dw, void* db, void* dgamma,
                                 void* dbeta, int64_t M, int64_t N, int64_t K, int dx_accumulate, int dtype,
                                 int grad_dtype, mg_deferred list, mg_stream stream) {
  const char* who = "linear_bwd_layer_norm_bwd";
  if (!mg::is_float_dtype(dtype)) return mg::fail(MG_ERR_INVALID, "%s: unsupported dtype %s", who, mg::dtype_name(dtype));
  if (M < 0 || N < 0 || K <= 0) return mg::fail(MG_ERR_INVALID, "%s: bad size", who);
  if (!dy || !x || !w || !ln_x || !gamma || !mean || !rstd || !dx || !dw || !dgamma || !dbeta)
    return mg::fail(MG_ERR_INVALID, "%s: null pointer argument", who);
  if (list) MG_TRY(mg::deferred_check(who, list, dtype, grad_dtype));
  else if (grad_dtype != dtype) return mg::fail(MG_ERR_INVALID, "%s: without a deferred list the gradients have the tensors' dtype", who);
  hipStream_t s = mg::to_stream(stream);
  auto run = [&](void* dg_use, void* dbt_use) -> int {
    bool done = false, db_done = false;
    const mg::LinearBwdLayerNorm ln{ln_x, gamma, mean, rstd, dg_use, dbt_use};
    MG_TRY(mg::linear_bwd_products(dy, x, w, dx, dw, db, M, N, K, nullptr, dx_accumulate != 0, dtype, s, &done,
                                   &db_done, &ln));
    if (done) {
      if (db && !db_done) MG_TRY(mg::linear_bwd_bias(dy, db, M, N, dtype, s));
      return MG_OK;
    }
    // Other shapes: dY W into a scratch tensor with the separate entry's kernels, then the LayerNorm backward.
    mg::Scratch dy_ln;
    MG_TRY(dy_ln.take(M * K * static_cast<int64_t>(mg::dtype_size(dtype))));
    MG_TRY(linear_bwd_impl(dy, x, w, dy_ln.as<char>(), dw, db, M, N, K, false, false, dtype, stream));
    return mg::ln_bwd(dy_ln.as<char>(), ln_x, gamma, mean, rstd, dx_accumulate ? dx : nullptr, dx, dg_use, dbt_use, M, K,
                      0.f, dtype, stream);
  };
  if (!list) return run(dgamma, dbeta);
  mg::DeferredScope scope(static_cast<mg::DeferredList*>(list), dtype, grad_dtype);
  void *dg_use, *dbt_use;
  MG_TRY(scope.substitute(dgamma, K, &dg_use));
  MG_TRY(scope.substitute(dbeta, K, &dbt_use));
  MG_TRY(run(dg_use, dbt_use));
  return scope.finish(s);
}

}  // extern "C"
