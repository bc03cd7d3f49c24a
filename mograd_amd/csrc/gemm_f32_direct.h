// fp32 products of any alignment, and those too small to fill the device with 128 x 128 tiles.
//
// The MFMA fragments come straight from memory into registers: a lane of v_mfma_f32_32x32x2 (or
// 16x16x4) holds one value per instruction, so a k-contiguous operand is one 16-byte load per four
// instructions and any other a 128-byte (64-byte) row of the wave per instruction, and 64 (32)
// cycles of arithmetic stand against each.  Nothing is staged, nothing waits at a barrier inside
// the k loop, and a load needs no more than 4-byte alignment.  A workgroup is four
// waves that share the reduction of one WT x WT tile: superblock s of the k range goes to wave
// s mod 4, and the four partial tiles meet in LDS in wave order.  With tiles of 16 or 32,
// a 64 x 256 output is 64 (16) workgroups of four short loops, where a single
// 128 x 128 tile walks its whole k range in one workgroup: what bounds such a product is the
// latency of that walk.  Three sizes of it on one MI355X, 128 x 128 tiles -> this kernel:
//   (64, 256) <- 784            68 -> 6.2 us      (317, 568) <- 2400          33 -> 17 us
//   (128, 64) <- 64             18 -> 4.1 us
// Not for large outputs with a short reduction, which are bound by their stores ((2048, 4096) <- 16: 36 us
// here, 13 with the plain kernel): dispatch_f32 sends none.
#pragma once

#include "gemm_impl.h"

namespace mg {

typedef float gemm_f4_any __attribute__((ext_vector_type(4), aligned(4)));

struct Gemm32Problem {
  const float* A;
  const float* B;
  const float* bias;
  float* C;
  float* partial;  // split along K: (splits, batches, M, N) partial sums instead of C
  int M, N, K;
  int64_t lda, ldb, ldc, bsa, bsb, bsc;
  int tiles_m, tiles_n, batches, k_per_split, splits;
  GemmEpilogue<float> ep;
  // m-contiguous A only (dW = dY^T X): the workgroups of the first tile column also sum A over k,
  // into colsum[m], or colsum[split * M + m] when split.
  float* colsum = nullptr;
};

// Four consecutive k of row (or column) `o` of an operand, from k0 on; past k_end zeros.
template <bool KC, bool TAIL>
__device__ __forceinline__ void gemm32_direct_load(const float* __restrict__ base, int64_t ld, int o, int k0, int k_end,
                                                   float (&f)[4]) {
  if constexpr (KC) {
    const float* p = base + static_cast<int64_t>(o) * ld + k0;
    if (!TAIL || k0 + 4 <= k_end) {
      const gemm_f4_any v = *reinterpret_cast<const gemm_f4_any*>(p);
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = v[j];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = k0 + j < k_end ? p[j] : 0.f;
    }
  } else {
    const float* p = base + static_cast<int64_t>(k0) * ld + o;
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] = !TAIL || k0 + j < k_end ? p[j * ld] : 0.f;
  }
}

template <int WT>
struct Gemm32Tile;  // the wave's accumulator: WT x WT values, 4 k-quads of KG k per four MFMAs
template <>
struct Gemm32Tile<32> {
  static constexpr int ACC = 16, KG = 8;
  floatx16 v;
  __device__ __forceinline__ void mma(float a, float b) { v = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, v, 0, 0, 0); }
  static __device__ __forceinline__ int row(int r, int lane) { return (r / 4) * 8 + (lane / 32) * 4 + r % 4; }
};
template <>
struct Gemm32Tile<16> {
  static constexpr int ACC = 4, KG = 16;
  floatx4 v;
  __device__ __forceinline__ void mma(float a, float b) { v = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, v, 0, 0, 0); }
  static __device__ __forceinline__ int row(int r, int lane) { return (lane / 16) * 4 + r; }
};

constexpr int kDirectWK = 4;  // waves along k
template <int WT>
constexpr int gemm32_direct_lds_floats() {
  // partial tiles of the waves, and behind them their column sums of A
  return kDirectWK * Gemm32Tile<WT>::ACC * 64 + kDirectWK * WT;
}

// The work of workgroup `bid` of a launch for one product.
template <bool A_KC, bool B_KC, int WT, bool SPLIT>
__device__ __forceinline__ void gemm32_direct_block(float* lds, int bid, const Gemm32Problem& pr) {
  using Tile = Gemm32Tile<WT>;
  constexpr int ACC = Tile::ACC, KG = Tile::KG, WK = kDirectWK;
  constexpr int U = 32 / KG < 4 ? 4 : 32 / KG;  // k groups in flight per operand
  constexpr int SB = U * KG;                    // k of a superblock
  const int tiles = pr.tiles_m * pr.tiles_n;
  int batch, split = 0, tile;
  if constexpr (SPLIT) {
    split = bid / (tiles * pr.batches);
    bid -= split * tiles * pr.batches;
  }
  batch = bid / tiles;
  tile = bid % tiles;
  int tm, tn;
  gemm_tile_of_block(tile, pr.tiles_m, pr.tiles_n, tm, tn, !SPLIT);
  const int wk = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int row0 = tm * WT, col0 = tn * WT;
  const int k_begin = SPLIT ? split * pr.k_per_split : 0;
  const int k_end = SPLIT ? min(pr.K, k_begin + pr.k_per_split) : pr.K;
  const float* A = pr.A + batch * pr.bsa;
  const float* B = pr.B + batch * pr.bsb;
  const int oa = min(row0 + lane % WT, pr.M - 1), ob = min(col0 + lane % WT, pr.N - 1);  // past the edge: never stored
  const int kl = (lane / WT) * 4;  // the lane's four k within a group

  constexpr bool CAN_COLSUM = !A_KC;
  const bool colsum = CAN_COLSUM && pr.colsum != nullptr && tn == 0;
  float cs = 0.f;

  Tile acc;
#pragma unroll
  for (int r = 0; r < ACC; ++r) acc.v[r] = 0.f;

  float fa[2][U][4], fb[2][U][4];
  auto load = [&](int buf, int k, auto tail) {
    constexpr bool TAIL = decltype(tail)::value;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      gemm32_direct_load<A_KC, TAIL>(A, pr.lda, oa, k + u * KG + kl, k_end, fa[buf][u]);
      gemm32_direct_load<B_KC, TAIL>(B, pr.ldb, ob, k + u * KG + kl, k_end, fb[buf][u]);
    }
  };
  auto multiply = [&](int buf) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc.mma(fa[buf][u][j], fb[buf][u][j]);
    if constexpr (CAN_COLSUM) {
      if (colsum) {
#pragma unroll
        for (int u = 0; u < U; ++u) cs += (fa[buf][u][0] + fa[buf][u][1]) + (fa[buf][u][2] + fa[buf][u][3]);
      }
    }
  };
  const int full = (k_end - k_begin) / SB;  // whole superblocks
  int s = wk;
  if (s < full) {
    load(0, k_begin + s * SB, std::false_type{});
    // two superblocks per turn, so that the register buffers have fixed names
    for (; s + WK < full; s += 2 * WK) {
      load(1, k_begin + (s + WK) * SB, std::false_type{});
      multiply(0);
      if (s + 2 * WK < full) load(0, k_begin + (s + 2 * WK) * SB, std::false_type{});
      multiply(1);
    }
    if (s < full) multiply(0);
  }
  if (k_begin + full * SB < k_end && full % WK == wk) {
    load(0, k_begin + full * SB, std::true_type{});
    multiply(0);
  }

  if constexpr (CAN_COLSUM) {
    if (colsum) {  // uniform over the workgroup
      float* cs_lds = lds + WK * ACC * 64;
      // the lane groups hold different k of the same row
#pragma unroll
      for (int w = WT; w < kWave; w *= 2) cs += __shfl_xor(cs, w);
      if (lane < WT) cs_lds[wk * WT + lane] = cs;
      __syncthreads();
      if (threadIdx.x < WT && row0 + static_cast<int>(threadIdx.x) < pr.M) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < WK; ++w) sum += cs_lds[w * WT + threadIdx.x];
        pr.colsum[(SPLIT ? static_cast<int64_t>(split) * pr.M : 0) + row0 + threadIdx.x] = sum;
      }
    }
  }

  const int col = col0 + lane % WT;
  const float bv = pr.bias && col < pr.N ? pr.bias[col] : 0.f;
  auto store = [&](int r, float v) {
    const int row = row0 + Tile::row(r, lane);
    if (row >= pr.M || col >= pr.N) return;
    if constexpr (SPLIT) {
      pr.partial[((static_cast<int64_t>(split) * pr.batches + batch) * pr.M + row) * pr.N + col] = v;
    } else {
      const int64_t at = batch * pr.bsc + static_cast<int64_t>(row) * pr.ldc + col;
      pr.C[at] = gemm_finish<float>(v + bv, pr.ep, at);
    }
  };
  static_assert(ACC % WK == 0, "each wave finishes its share of the accumulator rows");
#pragma unroll
  for (int r = 0; r < ACC; ++r) lds[(wk * ACC + r) * 64 + lane] = acc.v[r];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ACC / WK; ++i) {
    const int r = wk * (ACC / WK) + i;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < WK; ++w) v += lds[(w * ACC + r) * 64 + lane];
    store(r, v);
  }
}

template <bool A_KC, bool B_KC, int WT, bool SPLIT>
__global__ __launch_bounds__(64 * kDirectWK) void gemm_f32_direct_kernel(Gemm32Problem pr) {
  __shared__ float lds[gemm32_direct_lds_floats<WT>()];
  gemm32_direct_block<A_KC, B_KC, WT, SPLIT>(lds, blockIdx.x, pr);
}

// dX = dY W and dW = dY^T X (with db, the column sums of dY) of an fp32 layer in one launch:
// workgroups [0, n_dw) take dW, the rest dX.
template <int WT, bool SPLIT>
__global__ __launch_bounds__(64 * kDirectWK) void linear_bwd_f32_kernel(Gemm32Problem dw, Gemm32Problem dx, int n_dw) {
  __shared__ float lds[gemm32_direct_lds_floats<WT>()];
  const int bid = blockIdx.x;
  if (bid < n_dw) gemm32_direct_block<false, false, WT, SPLIT>(lds, bid, dw);
  else gemm32_direct_block<true, false, WT, false>(lds, bid - n_dw, dx);
}

}  // namespace mg
