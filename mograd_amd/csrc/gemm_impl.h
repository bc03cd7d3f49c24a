// Matrix products C = A x B (+ bias) for the Linear forward and its gradients.
//
// An operand is described by which of its two dimensions is contiguous in memory:
//   A (M x K): "k-contiguous"  A[m * lda + k]   (a row-major (M,K) array), or
//              "m-contiguous"  A[k * lda + m]   (the transposed view of a (K,M) array)
//   B (K x N): "k-contiguous"  B[n * ldb + k]   (a row-major (N,K) array, i.e. B^T given), or
//              "n-contiguous"  B[k * ldb + n]   (a row-major (K,N) array)
// so Y = X W^T is (k,k), dX = dY W is (k,n) and dW = dY^T X is (m,n), all without
// materialising a transpose.  C is row-major (M,N) with leading dimension ldc.
#pragma once

#include <type_traits>

#include "mg_device.h"
#include "mg_internal.h"

namespace mg {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kGemmBM = 128;
constexpr int kGemmBN = 128;
constexpr int kGemmBK = 32;
constexpr int kGemmThreads = 256;

// Workgroup -> output tile.  Consecutive workgroup ids go to different XCDs (id % 8), each
// with its own L2; ids are regrouped so that one XCD works on a compact block of tiles
// that share operand rows and columns.
constexpr int kXcd = 8;
__device__ __forceinline__ void gemm_tile_of_block(int bid, int tiles_m, int tiles_n, int& tm, int& tn,
                                                   bool regroup = true) {
  const int total = tiles_m * tiles_n;
  int id = bid;
  if (regroup && total % kXcd == 0) id = (bid % kXcd) * (total / kXcd) + bid / kXcd;
  // Raster in bands of 4 tile-rows so that a band's A rows stay in L2.
  constexpr int kBand = 4;
  const int band_tiles = kBand * tiles_n;
  const int band = id / band_tiles;
  const int in_band = id % band_tiles;
  const int rows_here = min(kBand, tiles_m - band * kBand);
  tm = band * kBand + in_band % rows_here;
  tn = in_band / rows_here;
}

// Split-K launches use one grid axis.  The work items, one per (batch, K range, output tile),
// are numbered with the tile varying fastest, and XCD x (the workgroups whose id is x mod kXcd)
// takes the contiguous block [x n / kXcd, (x + 1) n / kXcd) of the n items: every XCD gets the
// same number of items to within one (dealing out whole K ranges left two XCDs with twice the
// work of the others whenever the ranges were no multiple of eight), and an XCD's items are
// mostly whole K ranges, whose tiles read the same rows of both operands, so a range is fetched
// into one or two L2s instead of all eight (the dW of a 384 -> 1536 layer over 16384 rows
// fetched 240 MB for 63 MB of operands with tiles dealt out round robin).  Returns false for
// the few padding workgroups at the end of the shorter blocks.
__device__ __forceinline__ bool gemm_split_work(int bid, int tiles, int splits, int batches, int& tile, int& split,
                                                int& batch) {
  const int64_t n = static_cast<int64_t>(tiles) * splits * batches;
  const int x = bid % kXcd;
  const int64_t item = x * n / kXcd + bid / kXcd;
  if (item >= (x + 1) * n / kXcd) return false;
  const int group = static_cast<int>(item / tiles);
  tile = static_cast<int>(item % tiles);
  split = group % splits;
  batch = group / splits;
  return true;
}
inline int64_t gemm_split_grid(int64_t tiles, int64_t splits, int64_t batches) {
  return kXcd * ((tiles * splits * batches + kXcd - 1) / kXcd);
}

// What happens to a product element after the bias: v = acc + bias; relu: v = max(v, 0);
// relu_mask (laid out like C): v = 0 where mask <= 0; v is rounded to T; residual (laid out
// like C, may be C itself): v = round(v + residual).  For 16-bit types the residual is added
// to the rounded product, which is bit for bit what a separate add kernel computes.
template <typename T>
struct GemmEpilogue {
  const T* residual;
  const T* relu_mask;
  int relu;
};

// A x B with A element (m, k) at a[m * sam + k * sak] and B element (k, n) at
// b[k * sbk + n * sbn]; C row-major (M, N).
struct GemmArgs {
  const void* a;
  const void* b;
  const void* bias;
  void* c;
  int64_t batch, M, N, K;
  int64_t sam, sak, sbk, sbn;
  int64_t bsa, bsb;
  int dtype;
  // Epilogue (see GemmEpilogue): all optional.
  const void* residual = nullptr;
  const void* relu_mask = nullptr;
  int relu = 0;
  // A weight gradient (no epilogue, one batch) of a `_deferred` entry point: the sum of its K ranges may be left on the
  // current list; c_f32: C is fp32 where A and B are 16-bit, written from the accumulators.
  bool deferred = false;
  bool c_f32 = false;
};

template <typename T>
inline GemmEpilogue<T> epilogue_of(const GemmArgs& g) {
  return GemmEpilogue<T>{static_cast<const T*>(g.residual), static_cast<const T*>(g.relu_mask), g.relu};
}

template <typename T>
__device__ __forceinline__ T gemm_finish(float v, const GemmEpilogue<T>& ep, int64_t index) {
  if (ep.relu) v = v > 0.f ? v : 0.f;
  if (ep.relu_mask) v = to_float(ep.relu_mask[index]) > 0.f ? v : 0.f;
  T out = from_float<T>(v);
  if (ep.residual) out = from_float<T>(to_float(out) + to_float(ep.residual[index]));
  return out;
}

// ------------------------------------------------------------------------------------
// Any strides, any of the three float types: 64x64 tile, 256 threads, 4x4 outputs per
// thread, fp32 FMA.  The path for operands the MFMA kernels cannot take (unaligned
// leading dimensions, both strides non-unit, skinny edge shapes).
//   A element (m, k) at A[m * sam + k * sak];  B element (k, n) at B[k * sbk + n * sbn].
// ------------------------------------------------------------------------------------

constexpr int kGenericBK = 16;  // k per step

template <typename T, bool HAS_BIAS, typename OutT = T>
__global__ __launch_bounds__(256) void gemm_generic_kernel(const T* __restrict__ A, const T* __restrict__ B,
                                                           const T* __restrict__ bias, OutT* __restrict__ C, int M, int N,
                                                           int K, int64_t sam, int64_t sak, int64_t sbk, int64_t sbn,
                                                           int64_t ldc, int64_t bsa, int64_t bsb, int64_t bsc,
                                                           GemmEpilogue<T> ep) {
  constexpr int TM = 64, TN = 64, TK = kGenericBK;
  __shared__ float as[TK][TM + 1];
  __shared__ float bs[TK][TN + 1];
  const int batch = blockIdx.z;
  A += batch * bsa;
  B += batch * bsb;
  C += batch * bsc;
  if (ep.residual) ep.residual += batch * bsc;
  if (ep.relu_mask) ep.relu_mask += batch * bsc;
  const int m0 = blockIdx.y * TM;
  const int n0 = blockIdx.x * TN;
  const int tx = threadIdx.x % 16;
  const int ty = threadIdx.x / 16;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += TK) {
    for (int idx = threadIdx.x; idx < TM * TK; idx += 256) {
      // Walk the contiguous dimension fastest for whichever stride is 1.
      int m, k;
      if (sak == 1) { k = idx % TK; m = idx / TK; } else { m = idx % TM; k = idx / TM; }
      const int gm = m0 + m, gk = k0 + k;
      as[k][m] = (gm < M && gk < K) ? to_float(A[gm * sam + gk * sak]) : 0.f;
    }
    for (int idx = threadIdx.x; idx < TN * TK; idx += 256) {
      int n, k;
      if (sbk == 1) { k = idx % TK; n = idx / TK; } else { n = idx % TN; k = idx / TN; }
      const int gn = n0 + n, gk = k0 + k;
      bs[k][n] = (gn < N && gk < K) ? to_float(B[gk * sbk + gn * sbn]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TK; ++k) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = as[k][ty + i * 16];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = bs[k][tx + j * 16];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gm = m0 + ty + i * 16, gn = n0 + tx + j * 16;
      if (gm < M && gn < N) {
        const float bv = HAS_BIAS ? to_float(bias[gn]) : 0.f;
        const int64_t at = static_cast<int64_t>(gm) * ldc + gn;
        if constexpr (std::is_same_v<OutT, T>) C[at] = gemm_finish<T>(acc[i][j] + bv, ep, at);
        else C[at] = acc[i][j];  // (an fp32 weight gradient has neither bias nor epilogue)
      }
    }
}

}  // namespace mg

// ------------------------------------------------------------------------------------
// 16-bit storage (bf16, fp16) on v_mfma_f32_32x32x16: 128x128 output tile, K-chunks of 64,
// four waves in a 2x2 grid, each a 64x64 tile (2x2 accumulators), fp32 accumulation.
// Both operand tiles live in LDS as [row][k] with k contiguous, which is what the MFMA
// wants (8 consecutive k per lane).  A k-contiguous operand is copied as is; an
// m/n-contiguous operand is transposed on the way in: a thread loads 8 columns of two
// consecutive k rows and stores 8 dwords, each packing (k, k+1) for one column.
// SPLIT_K: a workgroup takes one K range (gemm_split_work) and fp32 partial tiles go to scratch
// (splits, M, N); gemm_splitk_reduce_kernel sums them in a fixed order.
// ------------------------------------------------------------------------------------

namespace mg {

typedef __bf16 gemm_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 gemm_f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 gemm_bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 gemm_f16x2 __attribute__((ext_vector_type(2)));
typedef float gemm_f32x2 __attribute__((ext_vector_type(2)));

// Two fp32 values rounded to T (nearest even), the first in the low half.
template <typename T>
__device__ __forceinline__ uint32_t gemm16_pack2(float lo, float hi);
template <>
__device__ __forceinline__ uint32_t gemm16_pack2<bf16_t>(float lo, float hi) {
  return bf16_pack2_rne(lo, hi);
}
template <>
__device__ __forceinline__ uint32_t gemm16_pack2<f16_t>(float lo, float hi) {
  const gemm_f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, gemm_f16x2));
}

template <typename T>
struct GemmMma16;
template <>
struct GemmMma16<bf16_t> {
  static __device__ __forceinline__ floatx16 run(uint4 a, uint4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(gemm_bf16x8, a), __builtin_bit_cast(gemm_bf16x8, b),
                                                   c, 0, 0, 0);
  }
};
template <>
struct GemmMma16<f16_t> {
  static __device__ __forceinline__ floatx16 run(uint4 a, uint4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(gemm_f16x8, a), __builtin_bit_cast(gemm_f16x8, b), c,
                                                  0, 0, 0);
  }
};

constexpr int kG16BK = 64;
constexpr int kG16Stride = kG16BK + 8;  // elements per LDS row: 144 bytes, 16-byte aligned, bank-spreading
// fp32 partial tiles of a product split along K: [K range][batch][tile_m][tile_n] tiles of
// 128 x 128 values, each stored as its four waves' accumulators,
//   [wave][ti][tj][g][lane][j]  =  row (wave / 2) * 64 + ti * 32 + g * 8 + (lane / 32) * 4 + j,
//                                  column (wave % 2) * 64 + tj * 32 + lane % 32
// of the tile.  Tiles are stored whole; rows and columns past the matrix hold whatever the
// clamped operand rows produced and are dropped by the reduction.
constexpr int kG16PartialTile = kGemmBM * kGemmBN;
inline int64_t gemm16_partial_floats(int64_t M, int64_t N, int64_t batches, int64_t splits) {
  return splits * batches * ((M + kGemmBM - 1) / kGemmBM) * ((N + kGemmBN - 1) / kGemmBN) * kG16PartialTile;
}

struct Gemm16Stage {
  uint4 v[4];
};

// KC: element (o, k) at base[o * ld + k].  4 chunks of 8 k-values per thread.
// else: element (o, k) at base[k * ld + o].  2 tasks per thread, each two k rows x 8 o.
// Leading dimension, extents and base address may be anything.  A whole
// chunk is one 16-byte load, at whatever even address it lies (the memory pipeline takes
// global accesses of any alignment); only the chunk over the edge is assembled from 2-byte
// loads with per-element bounds.  (All chunks by 2-byte loads: (1999, 768) = dY (1999, 1001) W
// took 105 us, against 24 us.)
typedef uint32_t gemm_u4_any __attribute__((ext_vector_type(4), aligned(2)));
template <typename T>
__device__ __forceinline__ uint4 gemm16_gather8(const T* __restrict__ p, int valid) {
  if (valid >= 8) {
    const gemm_u4_any v = *reinterpret_cast<const gemm_u4_any*>(p);
    return make_uint4(v[0], v[1], v[2], v[3]);
  }
  const uint16_t* q = reinterpret_cast<const uint16_t*>(p);
  uint32_t w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo = 2 * e < valid ? q[2 * e] : 0u;
    const uint32_t hi = 2 * e + 1 < valid ? q[2 * e + 1] : 0u;
    w[e] = lo | (hi << 16);
  }
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// The 16-byte chunk at any address, `valid` elements of it and zeros behind.
template <typename T>
__device__ __forceinline__ uint4 gemm_gather_chunk(const T* __restrict__ p, int valid) {
  if constexpr (sizeof(T) == 2) {
    return gemm16_gather8(p, valid);
  } else {
    const uint32_t* q = reinterpret_cast<const uint32_t*>(p);
    return make_uint4(q[0], valid > 1 ? q[1] : 0u, valid > 2 ? q[2] : 0u, valid > 3 ? q[3] : 0u);
  }
}

template <typename T, bool KC>
__device__ __forceinline__ void gemm16_load(const T* __restrict__ base, int64_t ld, int o0, int k0, int O, int k_end,
                                            Gemm16Stage& st) {
  const int t = threadIdx.x;
  if constexpr (KC) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = t + i * kGemmThreads;
      const int o = min(o0 + idx / 8, O - 1);
      const int k = k0 + (idx % 8) * 8;
      st.v[i] = gemm16_gather8(base + static_cast<int64_t>(o) * ld + k, k_end - k);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = t + i * kGemmThreads;
      const int oc = idx % 16, kp = idx / 16;
      const int k = k0 + 2 * kp;
      const int o = o0 + oc * 8;
      st.v[2 * i] = gemm16_gather8(base + static_cast<int64_t>(k) * ld + o, k < k_end ? O - o : 0);
      st.v[2 * i + 1] = gemm16_gather8(base + static_cast<int64_t>(k + 1) * ld + o, k + 1 < k_end ? O - o : 0);
    }
  }
}

template <bool KC>
__device__ __forceinline__ void gemm16_store(uint16_t* __restrict__ lds, const Gemm16Stage& st) {
  const int t = threadIdx.x;
  if constexpr (KC) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = t + i * kGemmThreads;
      *reinterpret_cast<uint4*>(lds + (idx / 8) * kG16Stride + (idx % 8) * 8) = st.v[i];
    }
  } else {
    uint32_t* lds32 = reinterpret_cast<uint32_t*>(lds);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = t + i * kGemmThreads;
      const int oc = idx % 16, kp = idx / 16;
      const uint32_t a[4] = {st.v[2 * i].x, st.v[2 * i].y, st.v[2 * i].z, st.v[2 * i].w};
      const uint32_t b[4] = {st.v[2 * i + 1].x, st.v[2 * i + 1].y, st.v[2 * i + 1].z, st.v[2 * i + 1].w};
      // The 16-byte k group of a row is stored at group index (g ^ (row / 8) % 8): the 16
      // lanes that hold different 8-row blocks of the same k pair then hit different banks
      // (row stride 36 dwords is 4 mod 32, so 8-row blocks alone would all collide).
      uint32_t* dst = lds32 + (oc * 8) * (kG16Stride / 2) + (((kp / 4) ^ (oc & 7)) * 4 + kp % 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        dst[(2 * e) * (kG16Stride / 2)] = __builtin_amdgcn_perm(b[e], a[e], 0x05040100);
        dst[(2 * e + 1) * (kG16Stride / 2)] = __builtin_amdgcn_perm(b[e], a[e], 0x07060302);
      }
    }
  }
}

template <bool SWIZZLED>
__device__ __forceinline__ uint4 gemm16_frag(const uint16_t* __restrict__ lds, int o_base, int ks, int lane) {
  const int row = o_base + lane % 32;
  int g = ks * 2 + lane / 32;  // 16-byte k group
  if constexpr (SWIZZLED) g ^= (row >> 3) & 7;
  return *reinterpret_cast<const uint4*>(lds + row * kG16Stride + g * 8);
}

// Eight consecutive elements from and to any even address.
template <typename T>
__device__ __forceinline__ void gemm16_load8(const T* p, float (&v)[8]) {
  const gemm_u4_any r = *reinterpret_cast<const gemm_u4_any*>(p);
  const uint32_t w[4] = {r[0], r[1], r[2], r[3]};
  VecIO<T, 8>::unpack(w, v);
}
template <typename T>
__device__ __forceinline__ void gemm16_store8(T* p, const float (&v)[8]) {
  gemm_u4_any r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = gemm16_pack2<T>(v[2 * e], v[2 * e + 1]);
  *reinterpret_cast<gemm_u4_any*>(p) = r;
}

// A 32 x 32 accumulator block at (row0, col0) into an fp32 C, as it lies in the registers: every store is two runs of 128 bytes.
__device__ __forceinline__ void gemm16_write_f32(const floatx16& acc, float* __restrict__ C, int M, int N, int64_t ldc, int row0,
                                                 int col0, int lane) {
  const int col = col0 + lane % 32;
  if (col >= N) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = row0 + (r / 4) * 8 + (lane / 32) * 4 + r % 4;
    if (row < M) C[static_cast<int64_t>(row) * ldc + col] = acc[r];
  }
}

// Output of one 128x128 tile from the four waves' accumulators (wave tile 64x64 at (wm, wn)).
// The accumulators have lanes along n and registers along m, so a direct store writes
// 2-byte elements.  Each wave instead transposes its tile through `mine`, 64 rows of kG16Stride
// elements of LDS that no wave reads any more, and stores eight elements per lane, at whatever
// address the row starts (only the chunk over the right edge goes out in 2-byte elements).  SPLIT_K: fp32 partial tiles go to
// partial[(split * batches + batch), M, N].
template <typename T, bool HAS_BIAS, bool SPLIT_K>
__device__ __forceinline__ void gemm16_write_tile(const floatx16 (&acc)[2][2], uint16_t* __restrict__ mine,
                                                  const float (&bias_v)[2], T* __restrict__ C,
                                                  float* __restrict__ partial, int M, int N, int64_t ldc, int64_t bsc,
                                                  int batch, int split, int batches, int m0, int n0, int wm, int wn,
                                                  int lane, const GemmEpilogue<T>& ep) {
  if constexpr (SPLIT_K) {
    // A K range's partial tile goes out as the accumulators lie in the registers: sixteen
    // unguarded 16-byte stores per thread, each a contiguous kilobyte of the wave
    // (see gemm16_partial_floats for the layout; gemm_splitk_reduce_block undoes it).
    const int tiles_n = (N + kGemmBN - 1) / kGemmBN, tiles_m = (M + kGemmBM - 1) / kGemmBM;
    const int col0 = n0 + wn;  // a multiple of 64; the workgroup's tile may span several partial tiles
    const int64_t tile_at = (static_cast<int64_t>(split) * batches + batch) * tiles_m * tiles_n +
                            static_cast<int64_t>(m0 / kGemmBM) * tiles_n + col0 / kGemmBN;
    float4* dst = reinterpret_cast<float4*>(partial) + tile_at * (kG16PartialTile / 4) +
                  ((wm / 64) * 2 + (col0 / 64) % 2) * 1024 + lane;
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
#pragma unroll
      for (int tj = 0; tj < 2; ++tj)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          dst[((ti * 2 + tj) * 4 + g) * 64] = make_float4(acc[ti][tj][4 * g], acc[ti][tj][4 * g + 1],
                                                          acc[ti][tj][4 * g + 2], acc[ti][tj][4 * g + 3]);
    return;
  } else {
    {
      // An accumulator holds one column and, per group of four registers, four consecutive
      // rows.  Two lanes with neighbouring columns swap packed pairs of rows, so that the even
      // lane holds (own, neighbour) of the first row of a pair and the odd lane (neighbour,
      // own) of the second: 32 four-byte LDS writes per thread instead of 64 two-byte ones,
      // and three VALU instructions per pair (convert, swap, byte select).
      const int odd = lane & 1;
      const uint32_t select = odd ? 0x03020706u : 0x05040100u;
      uint32_t* const base32 =
          reinterpret_cast<uint32_t*>(mine + ((lane / 32) * 4 + odd) * kG16Stride + (lane % 32 - odd));
      // (One copy of the loop per setting of the relu flag: inside the loop the flag would
      // cost two more instructions per value.)
      auto stage = [&](auto relu) {
#pragma unroll
        for (int ti = 0; ti < 2; ++ti)
#pragma unroll
          for (int tj = 0; tj < 2; ++tj) {
#pragma unroll
            for (int rp = 0; rp < 8; ++rp) {  // rows 2 rp and 2 rp + 1 of the sixteen
              float f0 = acc[ti][tj][2 * rp], f1 = acc[ti][tj][2 * rp + 1];
              if constexpr (HAS_BIAS) f0 += bias_v[tj], f1 += bias_v[tj];
              if constexpr (decltype(relu)::value) {
                f0 = f0 > 0.f ? f0 : 0.f;
                f1 = f1 > 0.f ? f1 : 0.f;
              }
              const uint32_t w = gemm16_pack2<T>(f0, f1);
              const uint32_t y = __builtin_amdgcn_update_dpp(w, w, kDppQuadXor1, 0xf, 0xf, false);
              const int rl = ti * 32 + (rp / 2) * 8 + (rp % 2) * 2;  // without the lane's own (lane / 32) * 4 + odd
              base32[(rl * kG16Stride + tj * 32) / 2] = __builtin_amdgcn_perm(y, w, select);
            }
          }
      };
      if (ep.relu) stage(std::true_type{});
      else stage(std::false_type{});
      __syncthreads();
      // Rows of the wave's 64 x 64 tile go out 16 bytes per lane, eight lanes to a row, eight
      // rows per store: one address per thread, stepped by eight rows.
      const int rl0 = lane / 8, ch = lane % 8;
      const int row0 = m0 + wm + rl0;
      const int col = n0 + wn + ch * 8;
      if (col >= N) return;
      const int64_t at0 = batch * bsc + static_cast<int64_t>(row0) * ldc + col;
      const int64_t step = 8 * ldc;
      const uint16_t* src = mine + rl0 * kG16Stride + ch * 8;
      const T* rbase = ep.residual;
      const T* mbase = ep.relu_mask;
      if (col + 8 > N) {  // the chunk over the right edge, element by element
        for (int i = 0; i < 8 && row0 + 8 * i < M; ++i)
          for (int e = 0; col + e < N; ++e) {
            const int64_t at = at0 + i * step + e;
            float v = to_float(reinterpret_cast<const T*>(src + i * 8 * kG16Stride)[e]);
            if (mbase) v = to_float(mbase[at]) > 0.f ? v : 0.f;
            if (rbase) v += to_float(rbase[at]);
            C[at] = from_float<T>(v);
          }
        return;
      }
      if (!rbase && !mbase) {
        T* dst = C + at0;
        uint4 v[8];  // all eight LDS reads first: their latencies overlap
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const uint4*>(src + i * 8 * kG16Stride);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (row0 + 8 * i < M) {
            const gemm_u4_any out = {v[i].x, v[i].y, v[i].z, v[i].w};
            *reinterpret_cast<gemm_u4_any*>(dst + i * step) = out;
          }
        return;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (row0 + 8 * i >= M) break;
        const int64_t at = at0 + i * step;
        float v[8];
        VecIO<T, 8>::load(reinterpret_cast<const T*>(src + i * 8 * kG16Stride), v);
        if (mbase) {
          float mk[8];
          gemm16_load8(mbase + at, mk);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = mk[e] > 0.f ? v[e] : 0.f;
        }
        if (rbase) {
          float rs[8];
          gemm16_load8(rbase + at, rs);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += rs[e];
        }
        gemm16_store8(C + at, v);
      }
    }
  }
}

// What a product's output tile needs to continue as a LayerNorm backward (see gemm16_deep_ln_bwd).
template <typename T>
struct Gemm16LayerNormBwd {
  const T* x = nullptr;         // the LayerNorm's input, laid out like the product's output
  const T* gamma = nullptr;     // (cols)
  const float* mean = nullptr;  // (rows) saved by the forward
  const float* rstd = nullptr;
  float* part_g = nullptr;      // (row tiles, cols) partial column sums of dy * xhat and of dy
  float* part_b = nullptr;
};

template <typename T, bool A_KC, bool B_KC, bool HAS_BIAS, bool SPLIT_K, typename OutT = T>
__global__ __launch_bounds__(kGemmThreads, 2) void gemm_16bit_mfma_kernel(
    const T* __restrict__ A, const T* __restrict__ B, const T* __restrict__ bias, OutT* __restrict__ C,
    float* __restrict__ partial, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int64_t bsa, int64_t bsb,
    int64_t bsc, int tiles_m, int tiles_n, int k_per_split, int splits, int batches, GemmEpilogue<T> ep) {
  __shared__ __attribute__((aligned(16))) uint16_t lds_a[kGemmBM * kG16Stride];
  __shared__ __attribute__((aligned(16))) uint16_t lds_b[kGemmBN * kG16Stride];

  const int tiles = tiles_m * tiles_n;
  // Split along K: see gemm_split_work.  Otherwise the batch index is folded into the tile id.
  int batch = blockIdx.x / tiles, tile = blockIdx.x % tiles, split = 0;
  if constexpr (SPLIT_K) {
    if (!gemm_split_work(blockIdx.x, tiles, splits, batches, tile, split, batch)) return;
  }
  int tm, tn;
  gemm_tile_of_block(tile, tiles_m, tiles_n, tm, tn, !SPLIT_K);
  const int m0 = tm * kGemmBM;
  const int n0 = tn * kGemmBN;
  A += batch * bsa;
  B += batch * bsb;
  const int k_begin = SPLIT_K ? split * k_per_split : 0;
  const int k_end = SPLIT_K ? min(K, k_begin + k_per_split) : K;

  const int wave = threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  const int wm = (wave / 2) * 64;
  const int wn = (wave % 2) * 64;

  floatx16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // The lane's two bias values, requested ahead of the first tiles (a load in the epilogue
  // would be waited for by every tile with nothing to overlap it).
  float bias_v[2] = {0.f, 0.f};
  if constexpr (HAS_BIAS && !SPLIT_K) {
#pragma unroll
    for (int tj = 0; tj < 2; ++tj) {
      const int col = n0 + wn + tj * 32 + lane % 32;
      bias_v[tj] = col < N ? to_float(bias[col]) : 0.f;
    }
  }
  Gemm16Stage sa, sb;
  gemm16_load<T, A_KC>(A, lda, m0, k_begin, M, k_end, sa);
  gemm16_load<T, B_KC>(B, ldb, n0, k_begin, N, k_end, sb);

  for (int k0 = k_begin; k0 < k_end; k0 += kG16BK) {
    gemm16_store<A_KC>(lds_a, sa);
    gemm16_store<B_KC>(lds_b, sb);
    __syncthreads();
    if (k0 + kG16BK < k_end) {
      gemm16_load<T, A_KC>(A, lda, m0, k0 + kG16BK, M, k_end, sa);
      gemm16_load<T, B_KC>(B, ldb, n0, k0 + kG16BK, N, k_end, sb);
    }
#pragma unroll
    for (int ks = 0; ks < kG16BK / 16; ++ks) {
      const uint4 fa0 = gemm16_frag<!A_KC>(lds_a, wm, ks, lane);
      const uint4 fa1 = gemm16_frag<!A_KC>(lds_a, wm + 32, ks, lane);
      const uint4 fb0 = gemm16_frag<!B_KC>(lds_b, wn, ks, lane);
      const uint4 fb1 = gemm16_frag<!B_KC>(lds_b, wn + 32, ks, lane);
      acc[0][0] = GemmMma16<T>::run(fa0, fb0, acc[0][0]);
      acc[0][1] = GemmMma16<T>::run(fa0, fb1, acc[0][1]);
      acc[1][0] = GemmMma16<T>::run(fa1, fb0, acc[1][0]);
      acc[1][1] = GemmMma16<T>::run(fa1, fb1, acc[1][1]);
    }
    __syncthreads();
  }

  if constexpr (!std::is_same_v<OutT, T>) {
    static_assert(!SPLIT_K && !HAS_BIAS, "a whole weight gradient");
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) gemm16_write_f32(acc[i][j], C, M, N, ldc, m0 + wm + 32 * i, n0 + wn + 32 * j, lane);
  } else {
    uint16_t* mine = (wave < 2 ? lds_a : lds_b) + (wave % 2) * 64 * kG16Stride;  // staging memory, idle now
    gemm16_write_tile<T, HAS_BIAS, SPLIT_K>(acc, mine, bias_v, C, partial, M, N, ldc, bsc, batch, split, SPLIT_K ? batches : 1,
                                            m0, n0, wm, wn, lane, ep);
  }
}

// ------------------------------------------------------------------------------------
// Tiles copied global memory -> LDS by the memory pipeline itself (`global_load_lds_dwordx4`: every
// lane names a 16-byte source, the wave's 64 chunks land back to back at an LDS address common to the
// wave), several k-steps ahead: what the kernels of gemm_16bit_deep.h (output tiles of 128 x 128 to 256 x 256)
// and gemm_16bit_small.h (64 x 64) share.  No registers hold data in flight.  Operands as above, all
// extents and strides multiples of 8 elements, every K split a multiple of 64.
//
// LDS image of one operand's step of 64 k, chosen per 16-byte chunk by which source chunk each lane
// names (64 banks of four bytes; a 128-bit read is served 16 lanes per clock):
//   k-contiguous: [rows][8 chunks], chunk c of row r at position c ^ (r/2 % 8): the sixteen
//     consecutive rows of a fragment read then hit sixteen different 16-byte bank groups
//     (timed on the device: 18.5-18.7 clocks per read with four waves reading, as for
//     consecutive addresses; 32 with c ^ (r % 8));
//   otherwise: [k][rows / 8 chunks], chunk c of k-row kk at position
//     c ^ gemm16_tr_swizzle(kk), read with `ds_read_b64_tr_b16` (within 16 lanes, lane i supplies
//     the four elements 4*i .. 4*i+3 of a 4 x 16 block and receives column i), which turns
//     four k-rows of 16 consecutive rows into each lane's four consecutive k.
// ------------------------------------------------------------------------------------

typedef short gemm_i16x4 __attribute__((ext_vector_type(4)));

// Where 16-byte chunk c of k-row kk of an m/n-contiguous operand sits in its LDS row:
// c ^ swizzle(kk).  A k-row is 256 or 512 bytes, a whole number of trips round the 64 banks,
// so without it every k-row would start on bank 0.  A transposing read takes 32 bytes of each
// of four k-rows (kk % 4 = 0..3) per sixteen lanes: 4 * (kk % 4) puts those on four different
// 32-byte bank groups that leave the neighbouring sixteen lanes' groups (chunk + 2) free, and
// 2 * (kk / 8 % 2) moves the upper half-wave (k-rows + 8) onto the remaining groups, so that
// whichever 32 lanes the LDS serves together touch every bank once.  (With c ^ 2 * (kk % 4),
// two sixteen-lane groups shared their bank groups: 43 % of the LDS cycles of the Linear
// backward kernel were conflict cycles.)
// With 64 rows a k-row is half a trip round the banks: the k-rows of one parity share a half, and
// 4 * (kk / 2 % 2) keeps those of a group apart.
template <int ROWS>
__device__ __forceinline__ constexpr int gemm16_tr_swizzle(int kk) {
  return (ROWS == 64 ? 4 * ((kk / 2) % 2) : 4 * (kk % 4)) ^ 2 * ((kk / 8) % 2);
}

// Copying one k-step of an operand of ROWS rows in a workgroup of NW waves: the waves that
// take part (all of them, unless the step has fewer kilobytes than the workgroup has waves)
// and the 16-byte requests of each of their threads.
constexpr int gemm16_pipe_waves(int rows, int bk, int nw) {
  const int kb = rows * bk * 2 / 1024;
  int w = kb < nw ? kb : nw;
  while (kb % w) --w;  // every taking wave the same number of kilobytes
  return w;
}
constexpr int gemm16_pipe_requests(int rows, int bk, int nw) {
  return rows * bk * 2 / 16 / (gemm16_pipe_waves(rows, bk, nw) * 64);
}

// The 16-byte source chunks this thread names for every k-step of one operand of ROWS rows,
// as element offsets from the operand's (batch, k_begin) origin; they advance by BK
// (k-contiguous) or BK * ld per step.
template <bool KC, int BK, int ROWS, int NW>  // NW: the waves that take part in this operand's copy
__device__ __forceinline__ void gemm16_pipe_sources(int64_t ld, int o0, int O,
                                                    int64_t (&src)[gemm16_pipe_requests(ROWS, BK, NW)]) {
  constexpr int CPR = BK / 8;     // chunks per k-contiguous row
  constexpr int CPK = ROWS / 8;   // chunks per k-row of the other image
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
#pragma unroll
  for (int i = 0; i < gemm16_pipe_requests(ROWS, BK, NW); ++i) {
    const int slot = (i * NW + wave) * kWave + lane;  // 16-byte position in the LDS image
    if constexpr (KC) {
      const int r = slot / CPR, c = (slot % CPR) ^ ((r / (16 / CPR)) % CPR);
      src[i] = static_cast<int64_t>(min(o0 + r, O - 1)) * ld + c * 8;  // rows past the edge are never stored
    } else {
      const int kk = slot / CPK, c = (slot % CPK) ^ gemm16_tr_swizzle<ROWS>(kk);
      const int o = o0 + c * 8;
      src[i] = static_cast<int64_t>(kk) * ld + (o < O ? o : o0);
    }
  }
}

// Written as assembly on purpose.  Through the compiler's builtin for this instruction every
// later LDS read of a kind whose aliasing it cannot judge (the transposing reads here) gets a
// wait for *all* outstanding copies, the younger steps' included, which would undo the
// pipeline; the waits are placed by hand in the kernel instead (MG_WAIT_VMCNT).  m0 (the
// wave's LDS destination) is written here and used by nothing else in these kernels.
template <int NI, int NW>
__device__ __forceinline__ void gemm16_pipe_issue(const uint16_t* base, const int64_t* src, char* lds_step) {
  using lds_ptr = __attribute__((address_space(3))) char*;
  const int wave = threadIdx.x / kWave;
  const unsigned dst = static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_ptr)lds_step)) + wave * 1024;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const unsigned dst_i = __builtin_amdgcn_readfirstlane(dst + i * NW * 1024);
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst_i), "v"(base + src[i]) : "memory");
  }
}

// The last, short step of a reduction that is no multiple of BK (`rem` k left, whole chunks of 8 for a
// k-contiguous operand): chunks past the end are copied from sixteen bytes of zeros, so nothing beyond the operand
// is read, the step multiplies like any other, and a wave's requests number the same in every step.  (Through
// registers the tail waited for every older copy as well: (39, 625 <- 920), forward + backward, 16.7 us against
// 15.6.)
__device__ const uint32_t kGemmZeros[4] __attribute__((aligned(16))) = {0, 0, 0, 0};
template <bool KC, int BK, int ROWS, int NW>
__device__ __forceinline__ void gemm16_pipe_issue_short(const uint16_t* base, const int64_t* src, int rem, char* lds_step) {
  using lds_ptr = __attribute__((address_space(3))) char*;
  constexpr int CPR = BK / 8, CPK = ROWS / 8;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const unsigned dst = static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_ptr)lds_step)) + wave * 1024;
#pragma unroll
  for (int i = 0; i < gemm16_pipe_requests(ROWS, BK, NW); ++i) {
    const int slot = (i * NW + wave) * kWave + lane;
    const int k = KC ? ((slot % CPR) ^ ((slot / CPR / (16 / CPR)) % CPR)) * 8 : slot / CPK;
    const uint16_t* p = k < rem ? base + src[i] : reinterpret_cast<const uint16_t*>(kGemmZeros);
    const unsigned dst_i = __builtin_amdgcn_readfirstlane(dst + i * NW * 1024);
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst_i), "v"(p) : "memory");
  }
}

// MFMA operand fragment: row o_base + lane % 32, k = ks * 16 + (lane / 32) * 8 .. + 7.
template <bool KC, int BK, int ROWS>
__device__ __forceinline__ uint4 gemm16_pipe_frag(const char* __restrict__ lds_step, int o_base, int ks, int lane) {
  if constexpr (KC) {
    constexpr int CPR = BK / 8;
    const int r = o_base + lane % 32;
    const int g = ks * 2 + lane / 32;
    return *reinterpret_cast<const uint4*>(lds_step + r * (BK * 2) + ((g ^ ((r / (16 / CPR)) % CPR)) * 16));
  } else {
    const int o = o_base + ((lane / 16) % 2) * 16 + 4 * (lane % 4);  // first of the 4 rows this lane supplies
    const int kq = (lane % 16) / 4;                                 // its k-row within a group of 4
    const int kk = ks * 16 + (lane / 32) * 8 + kq;
    const char* at = lds_step + kk * (ROWS * 2) + (((o / 8) ^ gemm16_tr_swizzle<ROWS>(kk)) * 16) + (o % 8) * 2;
    using lds_i16x4 = __attribute__((address_space(3))) gemm_i16x4;
    const gemm_i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        reinterpret_cast<lds_i16x4*>(reinterpret_cast<uintptr_t>(at)));
    const gemm_i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        reinterpret_cast<lds_i16x4*>(reinterpret_cast<uintptr_t>(at + 4 * (ROWS * 2))));
    uint2 l = __builtin_bit_cast(uint2, lo), h = __builtin_bit_cast(uint2, hi);
    return make_uint4(l.x, l.y, h.x, h.y);
  }
}

// s_waitcnt with only the vector-memory counter set (gfx9 encoding: vmcnt in bits 3:0 and
// 15:14, expcnt 6:4 and lgkmcnt 11:8 left at "no wait").
#define MG_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | 0x0f70)

// One product's arguments, as the kernels below take them.
template <typename T>
struct Gemm16Problem {
  const T* A;
  const T* B;
  const T* bias;
  T* C;
  float* partial;
  int M, N, K;
  int64_t lda, ldb, ldc, bsa, bsb, bsc;
  int tiles_m, tiles_n, k_per_split, splits, batches;
  GemmEpilogue<T> ep;
  // Split along K with an m-contiguous A only (dW = dY^T X): when set, the workgroups of the
  // first tile column also sum their A tiles over k, i.e. dY over its rows, and leave one
  // partial row of the bias gradient per K range at colsum_part[split * M + m].
  float* colsum_part = nullptr;
  // Not split (64 x 64 tiles only): the sums themselves, or in fp32.
  T* colsum = nullptr;
  float* colsum32 = nullptr;
  // An fp32 C (not split), see GemmArgs::c_f32.
  float* c32 = nullptr;
  // The partial tiles are read back much later (their sum is deferred to the end of a training
  // step): store them past the caches.
  bool partial_stream = false;
  // The output continues as a LayerNorm backward inside the launch (gemm16_deep_ln_bwd).
  Gemm16LayerNormBwd<T> ln;
};

// How a product's weight gradient is to be left (GemmArgs::deferred, c_f32).
// Partial tiles whose sum is deferred are read back at the end of the training step: stored past
// the caches they do not evict the activations the next kernels read (GPT step 2.48 -> 2.43 ms
// on one box; MOGRAD_HIP_DEFER_NT_STORE=0 keeps ordinary stores).
template <typename T>
inline void gemm16_gradient(const GemmArgs& g, Gemm16Problem<T>& pr) {
  pr.partial_stream = g.deferred && env_int("MOGRAD_HIP_DEFER_NT_STORE", 1) != 0;
  if (g.c_f32) pr.c32 = static_cast<float*>(g.c);
}

// The output tiles of gemm_16bit_deep.h.
enum Gemm16Tile { kTile128 = 0, kTile192 = 1, kTile256 = 2, kTileWide = 3 };  // 128 x 128, 128 x 192, 256 x 256, 128 x 384
constexpr int kGemm16TileM[4] = {128, 128, 256, 128};
constexpr int kGemm16TileN[4] = {128, 192, 256, 384};
constexpr int64_t kGemmDeepMaxLd = 1 << 22;  // offsets within a tile are kept in 32 bits
// One product of them (not kTileWide); partial: `splits` K ranges of k_per_split each, partial tiles (splits == 1: null).
template <typename T>
int launch_16bit_deep(const GemmArgs& g, Gemm16Tile tile, int splits, int k_per_split, float* partial, hipStream_t stream);
// dX and dW of a Linear layer (not kTile256), see linear_bwd_16bit_kernel; kTileWide: dX continues as px.ln says.
template <typename T>
int launch_linear_bwd_deep(const Gemm16Problem<T>& pw, const Gemm16Problem<T>& px, Gemm16Tile tile, int64_t n_dw,
                           int64_t n_dx, hipStream_t stream);

// ------------------------------------------------------------------------------------
// fp32 product with the tiles copied global memory -> LDS by `global_load_lds_dwordx4`, two
// copies of each TS x 32 tile: the copy of k-step i + 1 runs under the MFMAs of step i with
// one barrier per step and no registers or VALU work spent on staging.  TS is 128 (wave tiles of
// 64 x 64: 85-88 % of the matrix pipe at 2048 x 4096 x 4096) or, for outputs with too few such
// tiles for the device, 64 (wave tiles of 32 x 32).  A product of K steps and a remainder ends on a short step whose tiles come
// through registers, zeros behind (gemm32_pipe_tail).
//
// MFMA j of k-group g multiplies k in {g*8 + j, g*8 + 4 + j}: lane (o = l % 32, h = l / 32) takes
// k = g*8 + h*4 + j for j = 0..3, so a k-contiguous operand is read with one 128-bit LDS load.
//
// LDS image of one operand's step:
//   k-contiguous: [TS rows][8 chunks of 4 k], chunk c of row r at position c ^ (r/2 % 8)
//     (sixteen consecutive rows of a 128-bit fragment read hit sixteen bank groups);
//   otherwise: [32 k][TS / 4 chunks of 4 rows], chunk c of k-row kk at position
//     c ^ (8 * (kk/4 % 2)): the two halves of a wave read k and k + 4 of the same rows, 128
//     bytes apart in the banks.
// ------------------------------------------------------------------------------------

template <bool KC, int TS>
__device__ __forceinline__ void gemm32_pipe_sources(int64_t ld, int o0, int O, int64_t (&src)[TS / 32]) {
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
#pragma unroll
  for (int i = 0; i < TS / 32; ++i) {
    const int slot = (i * 4 + wave) * kWave + lane;  // 16-byte position in the LDS image
    if constexpr (KC) {
      const int r = slot / 8, c = (slot % 8) ^ ((r / 2) % 8);
      src[i] = static_cast<int64_t>(min(o0 + r, O - 1)) * ld + c * 4;  // rows past the edge are never stored
    } else {
      const int kk = slot / (TS / 4), c = (slot % (TS / 4)) ^ (8 * ((kk / 4) % 2));
      const int o = o0 + c * 4;
      src[i] = static_cast<int64_t>(kk) * ld + (o < O ? o : o0);
    }
  }
}

// See gemm16_pipe_issue for why this is assembly.
template <int NI>
__device__ __forceinline__ void gemm32_pipe_issue(const float* base, const int64_t* src, char* lds_step) {
  using lds_ptr = __attribute__((address_space(3))) char*;
  const int wave = threadIdx.x / kWave;
  const unsigned dst = static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_ptr)lds_step)) + wave * 1024;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const unsigned dst_i = __builtin_amdgcn_readfirstlane(dst + i * 4096);
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst_i), "v"(base + src[i]) : "memory");
  }
}

// The short last step (`rem` k left) comes through registers, zeros past the end.
template <bool KC, int TS>
__device__ __forceinline__ void gemm32_pipe_tail(const float* base, const int64_t* src, int rem, char* lds_step) {
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
#pragma unroll
  for (int i = 0; i < TS / 32; ++i) {
    const int slot = (i * 4 + wave) * kWave + lane;
    const int k = KC ? ((slot % 8) ^ ((slot / 16) % 8)) * 4 : slot / (TS / 4);
    const float4 v = k < rem ? *reinterpret_cast<const float4*>(base + src[i]) : make_float4(0.f, 0.f, 0.f, 0.f);
    *reinterpret_cast<float4*>(lds_step + slot * 16) = v;
  }
}

// MFMA operand values of one 32-wide tile for k-group g.
template <bool KC, int TS>
__device__ __forceinline__ void gemm32_pipe_frag(const char* __restrict__ lds_step, int o_base, int g, int lane,
                                                 float (&f)[4]) {
  const int o = o_base + lane % 32;
  if constexpr (KC) {
    const int c = g * 2 + lane / 32;
    const float4 r = *reinterpret_cast<const float4*>(lds_step + o * 128 + ((c ^ ((o / 2) % 8)) * 16));
    f[0] = r.x; f[1] = r.y; f[2] = r.z; f[3] = r.w;
  } else {
    const int kk = g * 8 + (lane / 32) * 4;  // (kk / 4) % 2 == lane / 32 for all four k of this lane
    const char* at = lds_step + kk * (TS * 4) + ((((o / 4) ^ (8 * (lane / 32))) * 16) + (o % 4) * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] = *reinterpret_cast<const float*>(at + j * (TS * 4));
  }
}

// SPLIT_K: a work item is (K range, batch, tile); the fp32 partial tiles go to
// partial[(split * batches + batch), M, N] and gemm_splitk_reduce_kernel adds them up in a
// fixed order (for outputs with too few tiles to fill the device, e.g. a 10-class head).
template <bool A_KC, bool B_KC, bool HAS_BIAS, bool SPLIT_K, int TS>
__global__ __launch_bounds__(kGemmThreads, TS == 128 ? 2 : 4) void gemm_f32_pipe_kernel(
    const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias, float* __restrict__ C,
    float* __restrict__ partial, int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, int64_t bsa, int64_t bsb,
    int64_t bsc, int tiles_m, int tiles_n, int batches, int k_per_split, int total_work, GemmEpilogue<float> ep_in) {
  constexpr int OP = TS * kGemmBK * 4;  // bytes of one operand's step
  constexpr int NT = TS / 64;           // 32 x 32 tiles of a wave along either axis
  constexpr int NI = TS / 32;           // copy requests per thread, operand and step
  __shared__ __attribute__((aligned(1024))) char lds[2][2][OP];

  const int tiles = tiles_m * tiles_n;
  const int wave = threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  const int wm = (wave / 2) * (TS / 2);
  const int wn = (wave % 2) * (TS / 2);
  const int64_t a_step = A_KC ? kGemmBK : kGemmBK * lda;
  const int64_t b_step = B_KC ? kGemmBK : kGemmBK * ldb;
  // The grid holds at most the workgroups that are resident at once; each takes output tiles
  // work, work + gridDim.x, ...  Workgroups that share operand slabs then start every tile
  // together, which keeps their fetches of the shared rows close in time.
  for (int work = blockIdx.x; work < total_work; work += gridDim.x) {
    const int split = SPLIT_K ? work / (tiles * batches) : 0;
    const int in_split = SPLIT_K ? work % (tiles * batches) : work;
    const int batch = in_split / tiles;
    int tm, tn;
    gemm_tile_of_block(in_split % tiles, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * TS;
    const int n0 = tn * TS;
    const int k_begin = SPLIT_K ? split * k_per_split : 0;
    const int k_here = SPLIT_K ? min(K - k_begin, k_per_split) : K;
    const int full_steps = k_here / kGemmBK, rem = k_here % kGemmBK;
    const int steps = full_steps + (rem > 0 ? 1 : 0);
    const float* a = A + batch * bsa + (A_KC ? static_cast<int64_t>(k_begin) : k_begin * lda);
    const float* b = B + batch * bsb + (B_KC ? static_cast<int64_t>(k_begin) : k_begin * ldb);
    float* c = C + batch * bsc;
    GemmEpilogue<float> ep = ep_in;
    if (ep.residual) ep.residual += batch * bsc;
    if (ep.relu_mask) ep.relu_mask += batch * bsc;

    floatx16 acc[NT][NT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    int64_t src_a[NI], src_b[NI];
    gemm32_pipe_sources<A_KC, TS>(lda, m0, M, src_a);
    gemm32_pipe_sources<B_KC, TS>(ldb, n0, N, src_b);
    auto request = [&](int step, int copy) {
      if (step == full_steps) {
        gemm32_pipe_tail<A_KC, TS>(a + step * a_step, src_a, rem, lds[copy][0]);
        gemm32_pipe_tail<B_KC, TS>(b + step * b_step, src_b, rem, lds[copy][1]);
        return;
      }
      gemm32_pipe_issue<NI>(a + step * a_step, src_a, lds[copy][0]);
      gemm32_pipe_issue<NI>(b + step * b_step, src_b, lds[copy][1]);
    };
    request(0, 0);
    for (int it = 0; it < steps; ++it) {
      const int cur = it & 1;
      // This wave's copies of step `it` have landed; the barrier covers the other waves' and
      // tells that everyone is done reading the other copy.  (A plain barrier: __syncthreads()
      // would be the same here, every copy being waited for, but costs a fence.)
      MG_WAIT_VMCNT(0);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (it + 1 < steps) request(it + 1, cur ^ 1);
      const char* la = lds[cur][0];
      const char* lb = lds[cur][1];
      // The fragments of k-group g + 1 are requested before the products of group g.
      float fa[2][NT][4], fb[2][NT][4];
      auto frags = [&](int buf, int g) {
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          gemm32_pipe_frag<A_KC, TS>(la, wm + 32 * i, g, lane, fa[buf][i]);
          gemm32_pipe_frag<B_KC, TS>(lb, wn + 32 * i, g, lane, fb[buf][i]);
        }
      };
      frags(0, 0);
#pragma unroll
      for (int g = 0; g < kGemmBK / 8; ++g) {
        const int p = g % 2;
        if (g + 1 < kGemmBK / 8) frags(p ^ 1, g + 1);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int ti = 0; ti < NT; ++ti)
#pragma unroll
            for (int tj = 0; tj < NT; ++tj)
              acc[ti][tj] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[p][ti][j], fb[p][tj][j], acc[ti][tj], 0, 0, 0);
      }
    }
    // The next tile's first copy goes into lds[0]: every wave must be done reading it.
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // Accumulator element r of a lane is row (r/4)*8 + (lane/32)*4 + r%4, column lane%32.
#pragma unroll
    for (int ti = 0; ti < NT; ++ti)
#pragma unroll
      for (int tj = 0; tj < NT; ++tj) {
        const int col = n0 + wn + tj * 32 + lane % 32;
        if (col >= N) continue;
        const float bv = (HAS_BIAS && !SPLIT_K) ? bias[col] : 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = m0 + wm + ti * 32 + (r / 4) * 8 + (lane / 32) * 4 + (r % 4);
          if (row < M) {
            if constexpr (SPLIT_K) {
              partial[((static_cast<int64_t>(split) * batches + batch) * M + row) * N + col] = acc[ti][tj][r];
            } else {
              const int64_t at = static_cast<int64_t>(row) * ldc + col;
              c[at] = gemm_finish<float>(acc[ti][tj][r] + bv, ep, at);
            }
          }
        }
      }
  }  // tiles of this workgroup
}

// out[i] = sum_s partial[s * slice + i] (+ bias[i % N]) for i < numel <= slice, converted to T.  One thread
// sums group g, four consecutive outputs, over all K ranges: range s goes to one of eight
// running sums, number (s / 4 % 2, s % 4), in increasing s, and the eight meet as
// ((a00 + a10) + (a01 + a11)) + ((a02 + a12) + (a03 + a13)).  The order is fixed, so the result is
// deterministic; it is the order of an earlier form of this reduction (four waves summing
// every fourth range each and meeting in LDS), kept so that results did not change, with
// eight independent 16-byte loads in flight per thread and no barrier.
// TILED: the partials are whole 128 x 128 tiles in accumulator order (kG16PartialTile), numel
// = slice = their count per K range, and a group of four is four consecutive rows of one
// column of `out` (rows x N per batch; tiles_n tile columns; rows and columns past the matrix
// are dropped).
template <typename T, bool HAS_BIAS, bool TILED = false, bool STREAM = false>
__device__ __forceinline__ void gemm_splitk_reduce_group(int64_t g, const float* __restrict__ partial,
                                                         const T* __restrict__ bias, T* __restrict__ out, int64_t numel,
                                                         int64_t slice, int splits, int N, const GemmEpilogue<T>& ep,
                                                         int rows = 0, int tiles_n = 0) {
  const int64_t i = g * 4;
  if (i >= numel) return;
  float r[4];
  if (TILED || i + 3 < numel) {
    float4 acc[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[h][j] = make_float4(0.f, 0.f, 0.f, 0.f);
    const float* p = partial + i;
    constexpr int NB = 8;  // K ranges in flight per thread (2 or 1 measured 2-7 % slower on a step's sums)
    for (int s0 = 0; s0 < splits; s0 += 8) {
#pragma unroll
      for (int h = 0; h < 8; h += NB) {
        float4 v[NB];
#pragma unroll
        for (int e = 0; e < NB; ++e)
          if (s0 + h + e >= splits) {
            v[e] = make_float4(0.f, 0.f, 0.f, 0.f);
          } else if constexpr (STREAM) {
            // read once, long after it was written: a streaming load that leaves the caches to
            // the tensors of the next step (a step's deferred sums: 137 -> 103 us)
            const floatx4 nt =
                __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(p + static_cast<int64_t>(s0 + h + e) * slice));
            v[e] = make_float4(nt[0], nt[1], nt[2], nt[3]);
          } else {
            v[e] = *reinterpret_cast<const float4*>(p + static_cast<int64_t>(s0 + h + e) * slice);
          }
#pragma unroll
        for (int e = 0; e < NB; ++e) {
          if (s0 + h + e < splits) {  // (adding the zero would turn a -0 sum into +0)
            float4& a = acc[(h + e) / 4][(h + e) % 4];
            a.x += v[e].x; a.y += v[e].y; a.z += v[e].z; a.w += v[e].w;
          }
        }
      }
    }
    float4 t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      t[j] = make_float4(acc[0][j].x + acc[1][j].x, acc[0][j].y + acc[1][j].y, acc[0][j].z + acc[1][j].z,
                         acc[0][j].w + acc[1][j].w);
    r[0] = (t[0].x + t[1].x) + (t[2].x + t[3].x);
    r[1] = (t[0].y + t[1].y) + (t[2].y + t[3].y);
    r[2] = (t[0].z + t[1].z) + (t[2].z + t[3].z);
    r[3] = (t[0].w + t[1].w) + (t[2].w + t[3].w);
  } else {
    // the last, partial group of an untiled slice: element by element, four running sums
    float a[4][3];
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j][0] = a[j][1] = a[j][2] = 0.f;
    for (int s = 0; s < splits; ++s) {
      const float* p = partial + static_cast<int64_t>(s) * slice + i;
      a[s % 4][0] += p[0];
      if (i + 1 < numel) a[s % 4][1] += p[1];
      if (i + 2 < numel) a[s % 4][2] += p[2];
    }
#pragma unroll
    for (int e = 0; e < 3; ++e) r[e] = ((a[0][e] + 0.f) + (a[1][e] + 0.f)) + ((a[2][e] + 0.f) + (a[3][e] + 0.f));
    r[3] = 0.f;
  }
  if constexpr (TILED) {
    // g = ((((t * 4 + wave) * 2 + ti) * 2 + tj) * 4 + q) * 64 + lane
    const int lane = static_cast<int>(g % 64), q = static_cast<int>(g / 64 % 4), tj = static_cast<int>(g / 256 % 2),
              ti = static_cast<int>(g / 512 % 2), wave = static_cast<int>(g / 1024 % 4);
    const int64_t t = g / 4096;  // tile over (batch, tile row, tile column)
    const int tiles_m = (rows + kGemmBM - 1) / kGemmBM;
    const int tn = static_cast<int>(t % tiles_n), tm = static_cast<int>(t / tiles_n % tiles_m);
    const int64_t batch = t / tiles_n / tiles_m;
    const int row = tm * kGemmBM + (wave / 2) * 64 + ti * 32 + q * 8 + (lane / 32) * 4;
    const int col = tn * kGemmBN + (wave % 2) * 64 + tj * 32 + lane % 32;
    if (col >= N) return;
    const float bv = HAS_BIAS ? to_float(bias[col]) : 0.f;
    for (int e = 0; e < 4 && row + e < rows; ++e) {
      const int64_t at = (batch * rows + row + e) * N + col;
      out[at] = gemm_finish<T>(r[e] + bv, ep, at);
    }
  } else {
    for (int e = 0; e < 4 && i + e < numel; ++e) {
      const float bv = HAS_BIAS ? to_float(bias[(i + e) % N]) : 0.f;
      out[i + e] = gemm_finish<T>(r[e] + bv, ep, i + e);
    }
  }
}

template <typename T, bool HAS_BIAS, bool TILED = false>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ partial,
                                                                 const T* __restrict__ bias, T* __restrict__ out,
                                                                 int64_t numel, int64_t slice, int splits, int N,
                                                                 GemmEpilogue<T> ep, int rows = 0, int tiles_n = 0) {
  gemm_splitk_reduce_group<T, HAS_BIAS, TILED>(static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x, partial, bias, out,
                                               numel, slice, splits, N, ep, rows, tiles_n);
}

// db[c] = sum over the `groups` partial rows db_part[g][c], 64 columns per 256 threads (`tid`
// of them, column block `bx`): every fourth row per 64 threads, then (t0 + t1) + (t2 + t3).
// `sums_` is 256 floats of LDS; every one of the 256 threads must make the call.
template <typename T>
__device__ __forceinline__ void linear_bwd_db_block(float* __restrict__ sums_, int tid, int bx,
                                                    const float* __restrict__ db_part, T* __restrict__ db, int groups,
                                                    int N) {
  float(&sums)[4][64] = *reinterpret_cast<float(*)[4][64]>(sums_);
  const int cx = tid % 64, sl = tid / 64;
  const int c = bx * 64 + cx;
  float a0 = 0.f, a1 = 0.f;
  if (c < N) {
    int g = sl;
    for (; g + 4 < groups; g += 8) {
      a0 += db_part[static_cast<int64_t>(g) * N + c];
      a1 += db_part[static_cast<int64_t>(g + 4) * N + c];
    }
    for (; g < groups; g += 4) a0 += db_part[static_cast<int64_t>(g) * N + c];
  }
  sums[sl][cx] = a0 + a1;
  __syncthreads();
  if (sl == 0 && c < N) db[c] = from_float<T>((sums[0][cx] + sums[1][cx]) + (sums[2][cx] + sums[3][cx]));
}

// What follows the common launch of a Linear layer's backward: workgroups [0, dw_blocks) sum
// the K ranges of dW (gemm_splitk_reduce_block), the rest sum the `groups` partial rows of
// the bias gradient that the launch left (one per K range), 64 columns per workgroup,
// every fourth row per 64 threads, then (t0 + t1) + (t2 + t3).  Fixed order, no atomics.
// dw_blocks = ceil(slice / 1024): a thread sums four consecutive values of a partial tile (TILED) or
// of a partial (dw_rows, K) matrix.
template <typename T, bool TILED = true>
__global__ __launch_bounds__(256) void linear_bwd_finish_kernel(const float* __restrict__ partial, T* __restrict__ dw,
                                                                int dw_rows, int64_t slice, int splits, int K,
                                                                int dw_blocks, const float* __restrict__ db_part,
                                                                T* __restrict__ db, int groups, int N) {
  __shared__ float sums[256];
  const int bid = blockIdx.x;
  if (bid < dw_blocks) {
    // dW is (dw_rows, K); the partial tiles cover the (N, K) product of the launch
    gemm_splitk_reduce_group<T, false, TILED>(static_cast<int64_t>(bid) * 256 + threadIdx.x, partial,
                                             static_cast<const T*>(nullptr), dw, slice, slice, splits, K,
                                             GemmEpilogue<T>{nullptr, nullptr, 0}, dw_rows, (K + kGemmBN - 1) / kGemmBN);
    return;
  }
  linear_bwd_db_block<T>(sums, threadIdx.x, bid - dw_blocks, db_part, db, groups, N);
}

}  // namespace mg
