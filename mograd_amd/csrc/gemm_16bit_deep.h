// 16-bit products (bf16, fp16) on v_mfma_f32_32x32x16 with the tiles copied global memory -> LDS more than
// a k-step ahead.
#pragma once

#include "gemm_impl.h"

namespace mg {

// ------------------------------------------------------------------------------------
// A workgroup of 2 x WN waves has an output tile of 128 AI rows x 32 (BJ0 + BJ1) WN columns, a wave 64 AI x
// 32 (BJ0 + BJ1) of it; 64 k per step, two copies of a step's tiles in LDS.
//
// The wave tile is cut into two row halves A0, A1 and two column parts B0, B1, and a step into
// four phases, one per (half, part).  All four k-slices of a phase's products run before the next
// phase, and meanwhile the fragments that the next phase needs and this one does not hold are read:
//   A0 B0 (reads B1) | A0 B1 (A1) | A1 B1 (A0 of the next step) | A1 B0 (B0 of the next step)
// so each fragment is read from LDS once per step and held in one place.  The LDS rows of a half or
// part (an image of its own) are free again as soon as all waves have its fragments in registers, and
// the copy of the step after next into them is requested from there on, one request per thread
// between every few MFMAs.  So a copy has more than a whole step to arrive in, no
// requests are made in a burst (a wave whose request does not fit the queue cannot issue its MFMAs
// either), and the matrix pipe does not drain at a step's end.  Two synchronisations a step, S1 in
// the first phase and S2 in the third, behind a first k-slice of MFMAs: the data that is read until the next one
// has arrived (younger requests stay outstanding), and no wave still reads what is requested until then.
// ------------------------------------------------------------------------------------
template <int AI_, int BJ0_, int BJ1_, int WN_ = 2>
struct Gemm16Deep {
  static constexpr int AI = AI_, BJ0 = BJ0_, BJ1 = BJ1_, BJ = BJ0_ + BJ1_, WN = WN_;
  static constexpr int kThreads = 2 * WN * 64;
  static constexpr int kWaveM = 64 * AI, kWaveN = 32 * BJ;
  static constexpr int kTM = 2 * kWaveM, kTN = WN * kWaveN;
  static constexpr int kBK = 64;
  // Images of a step: A0, A1, B0, B1; rows (of both wave rows, of all wave columns) and bytes.
  static constexpr int kRowsA = 64 * AI, kRowsB0 = 32 * BJ0 * WN, kRowsB1 = 32 * BJ1 * WN;
  static constexpr int rows(int image) { return image < 2 ? kRowsA : image == 2 ? kRowsB0 : image == 3 ? kRowsB1 : 0; }
  static constexpr int at(int image) {
    return 2 * kBK * (image == 0 ? 0 : image == 1 ? kRowsA : image == 2 ? 2 * kRowsA : 2 * kRowsA + kRowsB0);
  }
  static constexpr int kStep = 2 * kBK * (2 * kRowsA + kRowsB0 + kRowsB1);  // bytes of a step's tiles
  static constexpr int requests(int image) { return rows(image) * 8 / kThreads; }  // of 16 bytes, per thread and step
  static constexpr int kStripStride = kWaveN + 8;  // elements of a row of a wave's output strip (64 rows)
  static constexpr int kStrips = 2 * WN * 64 * kStripStride * 2;
  static constexpr int kLds = 2 * kStep > kStrips ? 2 * kStep : kStrips;
  // Workgroups per CU: by LDS (160 KB) and by the register file (512 per lane and SIMD; fragments and
  // addresses next to the accumulators).
  static constexpr int kWavesPerSimd = AI * BJ <= 3 ? 2 : 1;
  static constexpr int kOccupancy = kWavesPerSimd * 2 / WN < 1 ? 1
                                    : 160 * 1024 / kLds < kWavesPerSimd * 2 / WN ? 160 * 1024 / kLds : kWavesPerSimd * 2 / WN;
  static_assert(kRowsA * 8 % kThreads == 0 && kRowsB0 * 8 % kThreads == 0 && kRowsB1 * 8 % kThreads == 0, "whole requests");
};
// Byte offsets, from the tile's first row and the step's first k, of the 16-byte chunks that this thread
// requests for one image.  Image row r is row (r / PER_WAVE) * WAVE_ROWS + first + r % PER_WAVE of the
// tile.  LDS images as in gemm16_pipe_sources.
template <bool KC, int ROWS, int NT, int PER_WAVE, int WAVE_ROWS>
__device__ __forceinline__ void gemm16_deep_sources(int64_t ld, int o0, int O, int first, uint32_t (&off)[ROWS * 8 / NT]) {
  constexpr int CPK = ROWS / 8;
#pragma unroll
  for (int i = 0; i < ROWS * 8 / NT; ++i) {
    const int slot = i * NT + threadIdx.x;
    if constexpr (KC) {
      const int r = slot / 8, c = (slot % 8) ^ ((r / 2) % 8);
      const int row = (r / PER_WAVE) * WAVE_ROWS + first + r % PER_WAVE;
      off[i] = static_cast<uint32_t>((min(row, O - 1 - o0) * ld + c * 8) * 2);  // rows past the edge are never stored
    } else {
      const int kk = slot / CPK, r = ((slot % CPK) ^ gemm16_tr_swizzle<ROWS>(kk)) * 8;
      const int row = (r / PER_WAVE) * WAVE_ROWS + first + r % PER_WAVE;
      off[i] = static_cast<uint32_t>((kk * ld + (o0 + row < O ? row : 0)) * 2);
    }
  }
}

// See gemm16_pipe_issue; `base` is the same for the wave, `dst` its LDS destination.
__device__ __forceinline__ void gemm16_deep_issue(const uint16_t* base, uint32_t off, uint32_t dst) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory");
}

// The same for request i of an image of the last, short step (`rem` k left), zeros past the end (see
// gemm16_pipe_issue_short).
template <bool KC, int ROWS, int NT>
__device__ __forceinline__ void gemm16_deep_issue_short(const uint16_t* base, uint32_t off, int i, int rem, uint32_t dst) {
  const int slot = i * NT + threadIdx.x;
  const int k = KC ? ((slot % 8) ^ ((slot / 8 / 2) % 8)) * 8 : slot / (ROWS / 8);
  const char* p = k < rem ? reinterpret_cast<const char*>(base) + off : reinterpret_cast<const char*>(kGemmZeros);
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(p) : "memory");
}

// A wave's 64 x (32 BJ) values into its strip of LDS, rounded.  The accumulators have lanes along n and
// registers along m; two lanes with neighbouring columns swap packed pairs of rows (see gemm16_write_tile).
template <typename T, bool HAS_BIAS, bool RELU, int BJ>
__device__ __forceinline__ void gemm16_deep_stage(const floatx16 (*acc)[BJ], const float (&bias_v)[BJ],
                                                  uint16_t* __restrict__ mine, int lane) {
  constexpr int STRIDE = 32 * BJ + 8;
  const int odd = lane & 1;
  const uint32_t select = odd ? 0x03020706u : 0x05040100u;
  uint32_t* const base32 = reinterpret_cast<uint32_t*>(mine + ((lane / 32) * 4 + odd) * STRIDE + (lane % 32 - odd));
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int tj = 0; tj < BJ; ++tj)
#pragma unroll
      for (int rp = 0; rp < 8; ++rp) {  // rows 2 rp and 2 rp + 1 of the sixteen
        float f0 = acc[ti][tj][2 * rp], f1 = acc[ti][tj][2 * rp + 1];
        if constexpr (HAS_BIAS) f0 += bias_v[tj], f1 += bias_v[tj];
        if constexpr (RELU) {
          f0 = f0 > 0.f ? f0 : 0.f;
          f1 = f1 > 0.f ? f1 : 0.f;
        }
        const uint32_t w = gemm16_pack2<T>(f0, f1);
        const uint32_t y = __builtin_amdgcn_update_dpp(w, w, kDppQuadXor1, 0xf, 0xf, false);
        const int rl = ti * 32 + (rp / 2) * 8 + (rp % 2) * 2;
        base32[(rl * STRIDE + tj * 32) / 2] = __builtin_amdgcn_perm(y, w, select);
      }
}

// Output of a wave's 64 x (32 BJ) values (two rows of accumulator blocks): through the wave's own strip of LDS
// and out as 16 bytes per lane, whole rows of the strip one after the other.  EARLY (where
// registers are free): what the epilogue reads is requested before the strip is written.
template <typename T, bool HAS_BIAS, int BJ, bool EARLY>
__device__ __forceinline__ void gemm16_deep_write(const floatx16 (*acc)[BJ], const float (&bias_v)[BJ],
                                                 uint16_t* __restrict__ mine, T* __restrict__ C, int M, int N, int64_t ldc,
                                                 int row0, int col0, int lane, const T* residual, const T* relu_mask,
                                                 int relu) {
  constexpr int STRIDE = 32 * BJ + 8;
  constexpr int CPR = 4 * BJ;                                    // 16-byte chunks of a row
  constexpr int PERIOD = CPR % 3 == 0 ? 3 : 1;                   // stores after which the rows of a lane repeat
  constexpr int ROWS = 64 * PERIOD / CPR;                        // rows of a period
  int row[PERIOD], ch[PERIOD];
#pragma unroll
  for (int p = 0; p < PERIOD; ++p) row[p] = (p * 64 + lane) / CPR, ch[p] = (p * 64 + lane) % CPR;
  const bool plain = !residual && !relu_mask;
  gemm_u4_any rs[CPR], mk[CPR];
  auto fetch = [&](int i) {  // (past the edge: the last place that exists, and dropped)
    const int r = min(row0 + row[i % PERIOD] + i / PERIOD * ROWS, M - 1), c = min(col0 + ch[i % PERIOD] * 8, N - 8);
    const int64_t at = r * ldc + c;
    if (residual) rs[i] = *reinterpret_cast<const gemm_u4_any*>(residual + at);
    if (relu_mask) mk[i] = *reinterpret_cast<const gemm_u4_any*>(relu_mask + at);
  };
  if (EARLY && !plain && N >= 8) {
#pragma unroll
    for (int i = 0; i < CPR; ++i) fetch(i);
  }
  if (relu) gemm16_deep_stage<T, HAS_BIAS, true, BJ>(acc, bias_v, mine, lane);
  else gemm16_deep_stage<T, HAS_BIAS, false, BJ>(acc, bias_v, mine, lane);
  __builtin_amdgcn_wave_barrier();  // the strip is the wave's own: its LDS accesses are in order
#pragma unroll
  for (int i = 0; i < CPR; ++i) {
    const int rl = row[i % PERIOD] + i / PERIOD * ROWS, r = row0 + rl, c = col0 + ch[i % PERIOD] * 8;
    const uint16_t* src = mine + rl * STRIDE + ch[i % PERIOD] * 8;
    if (r >= M || c >= N) continue;
    const int64_t at = r * ldc + c;
    const uint4 v = *reinterpret_cast<const uint4*>(src);
    const uint32_t vw[4] = {v.x, v.y, v.z, v.w};
    if (c + 8 > N) {  // the chunk over the right edge, element by element
#pragma unroll
      for (int e = 0; e < 7; ++e)
        if (c + e < N) {
          T one = __builtin_bit_cast(T, static_cast<uint16_t>(vw[e / 2] >> (e % 2 * 16)));
          if (relu_mask) one = to_float(relu_mask[at + e]) > 0.f ? one : from_float<T>(0.f);
          if (residual) one = from_float<T>(to_float(one) + to_float(residual[at + e]));
          C[at + e] = one;
        }
      continue;
    }
    if (plain) {
      const gemm_u4_any out = {v.x, v.y, v.z, v.w};
      *reinterpret_cast<gemm_u4_any*>(C + at) = out;
      continue;
    }
    if (!EARLY) fetch(i);
    float f[8], g[8];
    VecIO<T, 8>::unpack(vw, f);
    if (relu_mask) {
      const uint32_t mw[4] = {mk[i][0], mk[i][1], mk[i][2], mk[i][3]};
      VecIO<T, 8>::unpack(mw, g);
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = g[e] > 0.f ? f[e] : 0.f;
    }
    if (residual) {
      const uint32_t rw[4] = {rs[i][0], rs[i][1], rs[i][2], rs[i][3]};
      VecIO<T, 8>::unpack(rw, g);
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] += g[e];
    }
    gemm16_store8(C + at, f);
  }
}

// Output of a workgroup's 128 rows of a result with S::kTN columns, when the result dY is only wanted as the
// upstream of a LayerNorm backward: the tile is staged in LDS as the rounded 16-bit values a store would
// have written, and the workgroup then computes, from LDS and the matching rows of the LayerNorm's input x,
//   dx = rstd (dY gamma - mean_n(dY gamma) - xhat mean_n(dY gamma xhat)),  xhat = (x - mean) rstd,
// written to C as round(dx) (+ the residual, as the separate kernels give it), and the tile's
// column sums of dY xhat and dY as one row of part_g / part_b.  dY itself never reaches memory.
// Four lanes share a row of the wave's 64 x 96 (three chunks of 8 columns each), sixteen rows at a time: a row's
// sums go over its four lanes by DPP and over the waves that share it through LDS, the column sums
// over the sixteen lanes of a chunk by DPP (rows of sixteen lanes) and LDS; every order is fixed.
template <typename T, class S>
__device__ __forceinline__ void gemm16_deep_ln_bwd(const floatx16 (&acc)[2][S::BJ], char* lds, int wave, int lane, T* C, int M,
                                                   int64_t ldc, int tile_m, int m0, const T* residual,
                                                   const Gemm16LayerNormBwd<T>& ln) {  // residual may be C itself
  static_assert(S::AI == 1 && S::BJ == 3, "a wave has 64 x 96");
  constexpr int COLS = S::kTN, WN = S::WN, NG = 4, NT = 3;  // groups of sixteen rows, chunks per lane
  static_assert(S::kLds >= S::kStrips + 128 * WN * 8 && S::kStrips >= 8 * 2 * COLS * 4, "LDS for the sums");
  uint16_t* const mine = reinterpret_cast<uint16_t*>(lds) + wave * 64 * S::kStripStride;
  float2* const row_sums = reinterpret_cast<float2*>(lds + S::kStrips);  // [128][WN]
  const int wr = wave / WN, wc = wave % WN, q = lane % 4, r0 = lane / 4;
  const float no_bias[S::BJ] = {};
  uint4 xraw[NG][NT], rraw[NG][NT];
  float mu[NG], rs[NG], gam[NT][8];
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    const int row = min(m0 + wr * 64 + r0 + 16 * i, M - 1);  // rows past the end: computed, never stored or summed
    mu[i] = ln.mean[row];
    rs[i] = ln.rstd[row];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int64_t at = row * ldc + wc * S::kWaveN + (q + 4 * t) * 8;
      xraw[i][t] = *reinterpret_cast<const uint4*>(ln.x + at);
      rraw[i][t] = residual ? *reinterpret_cast<const uint4*>(residual + at) : make_uint4(0, 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) VecIO<T, 8>::load(ln.gamma + wc * S::kWaveN + (q + 4 * t) * 8, gam[t]);
  gemm16_deep_stage<T, false, false, S::BJ>(acc, no_bias, mine, lane);
  __builtin_amdgcn_wave_barrier();
  auto value = [&](int i, int t, float (&dy)[8], float (&xhat)[8]) {
    VecIO<T, 8>::load(reinterpret_cast<const T*>(mine + (r0 + 16 * i) * S::kStripStride + (q + 4 * t) * 8), dy);
    VecIO<T, 8>::load(reinterpret_cast<const T*>(&xraw[i][t]), xhat);
#pragma unroll
    for (int e = 0; e < 8; ++e) xhat[e] = (xhat[e] - mu[i]) * rs[i];
  };
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float dy[8], xhat[8];
      value(i, t, dy, xhat);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float dyg = dy[e] * gam[t][e];
        s0 += dyg;
        s1 += dyg * xhat[e];
      }
    }
    s0 += dpp_move<kDppQuadXor1>(s0);
    s1 += dpp_move<kDppQuadXor1>(s1);
    s0 += dpp_move<kDppQuadXor2>(s0);
    s1 += dpp_move<kDppQuadXor2>(s1);
    if (q == 0) row_sums[(wr * 64 + r0 + 16 * i) * WN + wc] = make_float2(s0, s1);
  }
  __syncthreads();
  const float inv_n = 1.0f / static_cast<float>(COLS);
  float acc_g[NT][8], acc_b[NT][8];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc_g[t][e] = acc_b[t][e] = 0.f;
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    const int rl = wr * 64 + r0 + 16 * i, row = m0 + rl;
    const bool ok = row < M;
    float c1 = 0.f, c2 = 0.f;
#pragma unroll
    for (int w = 0; w < WN; ++w) {
      const float2 p = row_sums[rl * WN + w];
      c1 += p.x;
      c2 += p.y;
    }
    c1 *= inv_n;
    c2 *= inv_n;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float dy[8], xhat[8], rv[8], out[8];
      value(i, t, dy, xhat);
      VecIO<T, 8>::load(reinterpret_cast<const T*>(&rraw[i][t]), rv);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = ok ? dy[e] : 0.f;
        out[e] = rs[i] * (d * gam[t][e] - c1 - xhat[e] * c2);
        acc_g[t][e] += d * xhat[e];
        acc_b[t][e] += d;
      }
      if (residual) {
        // round(gradient) + residual: a plain addition, as the separate add performs it
#pragma clang fp contract(off)
#pragma unroll
        for (int e = 0; e < 8; ++e) out[e] = to_float(from_float<T>(out[e])) + rv[e];
      }
      if (ok) VecIO<T, 8>::store(C + row * ldc + wc * S::kWaveN + (q + 4 * t) * 8, out);
    }
  }
  __syncthreads();  // the strips are read out: their memory takes the column sums of four rows of sixteen lanes and two waves
  float* const part = reinterpret_cast<float*>(lds) + (wr * 4 + lane / 16) * 2 * COLS + wc * S::kWaveN + q * 8;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      acc_g[t][e] += dpp_move<kDppRowRor8>(acc_g[t][e]);
      acc_b[t][e] += dpp_move<kDppRowRor8>(acc_b[t][e]);
      acc_g[t][e] += dpp_move<kDppRowRor4>(acc_g[t][e]);
      acc_b[t][e] += dpp_move<kDppRowRor4>(acc_b[t][e]);
      if (lane % 16 < 4) part[t * 32 + e] = acc_g[t][e], part[COLS + t * 32 + e] = acc_b[t][e];
    }
  __syncthreads();
  for (int c = threadIdx.x; c < 2 * COLS; c += S::kThreads) {
    float sum = 0.f;
#pragma unroll
    for (int p = 0; p < 8; ++p) sum += reinterpret_cast<const float*>(lds)[p * 2 * COLS + c];
    if (c < COLS) ln.part_g[static_cast<int64_t>(tile_m) * COLS + c] = sum;
    else ln.part_b[static_cast<int64_t>(tile_m) * COLS + c - COLS] = sum;
  }
}

// The work of workgroup `bid` of a launch for one product; `lds` is S::kLds bytes, aligned to 1024.
// pr.tiles_m, pr.tiles_n count tiles of S::kTM x S::kTN.  COLSUM: the sums of A over k as well (see Gemm16Problem).  LN_BWD: see gemm16_deep_ln_bwd.
// OUT_F32: the result goes to pr.c32.
template <typename T, class S, bool A_KC, bool B_KC, bool HAS_BIAS, bool SPLIT_K, bool COLSUM = false, bool LN_BWD = false,
          bool OUT_F32 = false>
__device__ __forceinline__ void gemm16_deep_block(char* lds, int bid, const Gemm16Problem<T>& pr) {
  constexpr int AI = S::AI, BJ0 = S::BJ0, BJ1 = S::BJ1, BJ = S::BJ, WN = S::WN, NT = S::kThreads;
  const int M = pr.M, N = pr.N;
  const int64_t lda = pr.lda, ldb = pr.ldb;
  const int tiles = pr.tiles_m * pr.tiles_n;
  int batch = bid / tiles, tile = bid % tiles, split = 0;
  if constexpr (SPLIT_K) {
    if (!gemm_split_work(bid, tiles, pr.splits, pr.batches, tile, split, batch)) return;
  }
  int tm, tn;
  gemm_tile_of_block(tile, pr.tiles_m, pr.tiles_n, tm, tn, !SPLIT_K);
  // (the divisions ran on the vector unit: back into scalars, which the requests' base addresses are made of)
  tm = __builtin_amdgcn_readfirstlane(tm), tn = __builtin_amdgcn_readfirstlane(tn);
  split = __builtin_amdgcn_readfirstlane(split), batch = __builtin_amdgcn_readfirstlane(batch);
  const int m0 = tm * S::kTM, n0 = tn * S::kTN;
  const int k_begin = SPLIT_K ? split * pr.k_per_split : 0;
  const int k_end = SPLIT_K ? min(pr.K, k_begin + pr.k_per_split) : pr.K;
  // A reduction of fewer steps than there are copies ends on steps of zeros.
  const int full_steps = (k_end - k_begin) / S::kBK, rem = (k_end - k_begin) % S::kBK;
  const int steps = max(2, full_steps + (rem > 0 ? 1 : 0));
  const int64_t a_step = A_KC ? S::kBK : S::kBK * lda;
  const int64_t b_step = B_KC ? S::kBK : S::kBK * ldb;
  const uint16_t* a16 = reinterpret_cast<const uint16_t*>(pr.A) + batch * pr.bsa + (A_KC ? m0 * lda + k_begin : m0 + k_begin * lda);
  const uint16_t* b16 = reinterpret_cast<const uint16_t*>(pr.B) + batch * pr.bsb + (B_KC ? n0 * ldb + k_begin : n0 + k_begin * ldb);

  const int wave = threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  const int wr = wave / WN, wc = wave % WN;  // the wave's row and column of wave tiles

  floatx16 acc[2 * AI][BJ];
#pragma unroll
  for (int i = 0; i < 2 * AI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  float col_sum[2 * AI];
#pragma unroll
  for (int i = 0; i < 2 * AI; ++i) col_sum[i] = 0.f;

  constexpr int RA = S::requests(0), RB0 = S::requests(2), RB1 = S::requests(3), R = 2 * RA + RB0 + RB1;
  uint32_t src_a0[RA], src_a1[RA], src_b0[RB0], src_b1[RB1];
  gemm16_deep_sources<A_KC, S::kRowsA, NT, 32 * AI, S::kWaveM>(lda, m0, M, 0, src_a0);
  gemm16_deep_sources<A_KC, S::kRowsA, NT, 32 * AI, S::kWaveM>(lda, m0, M, 32 * AI, src_a1);
  gemm16_deep_sources<B_KC, S::kRowsB0, NT, 32 * BJ0, S::kWaveN>(ldb, n0, N, 0, src_b0);
  gemm16_deep_sources<B_KC, S::kRowsB1, NT, 32 * BJ1, S::kWaveN>(ldb, n0, N, 32 * BJ0, src_b1);
  using lds_ptr = __attribute__((address_space(3))) char*;
  const uint32_t lds_wave = __builtin_amdgcn_readfirstlane(
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr)lds)) + wave * 1024);

  // Request i of an image of `step`, into copy `copy`.
  auto request = [&](auto image, int i, int step, int copy) {
    constexpr int IM = decltype(image)::value;
    const uint32_t dst = lds_wave + copy * S::kStep + S::at(IM) + i * (NT * 16);
    if constexpr (IM == 0) gemm16_deep_issue(a16 + step * a_step, src_a0[i], dst);
    if constexpr (IM == 1) gemm16_deep_issue(a16 + step * a_step, src_a1[i], dst);
    if constexpr (IM == 2) gemm16_deep_issue(b16 + step * b_step, src_b0[i], dst);
    if constexpr (IM == 3) gemm16_deep_issue(b16 + step * b_step, src_b1[i], dst);
  };
  auto request_short = [&](auto image, int i, int step, int copy, int left) {
    constexpr int IM = decltype(image)::value;
    const uint32_t dst = lds_wave + copy * S::kStep + S::at(IM) + i * (NT * 16);
    if constexpr (IM == 0) gemm16_deep_issue_short<A_KC, S::kRowsA, NT>(a16 + step * a_step, src_a0[i], i, left, dst);
    if constexpr (IM == 1) gemm16_deep_issue_short<A_KC, S::kRowsA, NT>(a16 + step * a_step, src_a1[i], i, left, dst);
    if constexpr (IM == 2) gemm16_deep_issue_short<B_KC, S::kRowsB0, NT>(b16 + step * b_step, src_b0[i], i, left, dst);
    if constexpr (IM == 3) gemm16_deep_issue_short<B_KC, S::kRowsB1, NT>(b16 + step * b_step, src_b1[i], i, left, dst);
  };

  uint4 fa[2][AI][4], fb0[BJ0][4], fb1[BJ1][4];  // fragments [block of 32 rows][k-slice of 16]
  // Fragment n (all of a k-slice first) of an image of copy `copy`.
  auto read = [&](auto image, int n, int copy) {
    constexpr int IM = decltype(image)::value;
    const char* at = lds + copy * S::kStep + S::at(IM);
    if constexpr (IM < 2)
      fa[IM][n % AI][n / AI] = gemm16_pipe_frag<A_KC, 64, S::kRowsA>(at, wr * 32 * AI + 32 * (n % AI), n / AI, lane);
    else if constexpr (IM == 2)
      fb0[n % BJ0][n / BJ0] = gemm16_pipe_frag<B_KC, 64, S::kRowsB0>(at, wc * 32 * BJ0 + 32 * (n % BJ0), n / BJ0, lane);
    else
      fb1[n % BJ1][n / BJ1] = gemm16_pipe_frag<B_KC, 64, S::kRowsB1>(at, wc * 32 * BJ1 + 32 * (n % BJ1), n / BJ1, lane);
  };
  float bias_v[BJ];
#pragma unroll
  for (int j = 0; j < BJ; ++j) bias_v[j] = 0.f;
  using A0 = std::integral_constant<int, 0>;
  using A1 = std::integral_constant<int, 1>;
  using B0 = std::integral_constant<int, 2>;
  using B1 = std::integral_constant<int, 3>;
  using None = std::integral_constant<int, 4>;
  constexpr auto blocks = [](int im) constexpr { return im < 2 ? AI : im == 2 ? BJ0 : im == 3 ? BJ1 : 0; };
  // One phase: half `ah` x part `bh`.  Meanwhile the fragments of `rd` are read from copy `rd_copy` (those of a
  // part that is being multiplied: each k-slice when it has been), and image `rq` of step `rq_step` is
  // requested (`is_short`: the last, short one).  `sync` runs after the first k-slice.
  auto phase = [&](auto ah, auto bh, auto rd, int rd_copy, auto rq, int rq_step, int rq_copy, auto is_short, auto sync) {
    constexpr int AH = decltype(ah)::value, BH = decltype(bh)::value - 2;
    constexpr int RD = decltype(rd)::value, RQ = decltype(rq)::value;
    constexpr int NB = BH ? BJ1 : BJ0, KS = AI * NB, NM = 4 * KS;
    constexpr int NR = 4 * blocks(RD), NQ = S::requests(RQ);
    constexpr bool OVER = RD == BH + 2;  // reads the next step's fragments over the present ones
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const int ks = m / KS, i = m / NB % AI, j = m % NB;
      floatx16& c = acc[AH * AI + i][BH * BJ0 + j];
      if constexpr (BH == 0) c = GemmMma16<T>::run(fa[AH][i][ks], fb0[j][ks], c);
      else c = GemmMma16<T>::run(fa[AH][i][ks], fb1[j][ks], c);
      if constexpr (COLSUM && BH == 0) {
        if (j == 0) {
          const uint32_t w[4] = {fa[AH][i][ks].x, fa[AH][i][ks].y, fa[AH][i][ks].z, fa[AH][i][ks].w};
          float v[8];
          VecIO<T, 8>::unpack(w, v);
          col_sum[AH * AI + i] += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        }
      }
      if (m == KS - 1) {
        __builtin_amdgcn_sched_barrier(0);
        sync();
      }
      if constexpr (NR > 0) {
#pragma unroll
        for (int n = 0; n < NR; ++n) {
          const int when = OVER ? (n / blocks(RD) + 1) * KS - 1 : KS - 1 + n * (NM - 2 * KS) / NR;
          if (when == m) read(rd, n, rd_copy);
        }
      }
      if constexpr (NQ > 0) {
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          if (KS + (2 * q + 1) * (NM - KS) / (2 * NQ) == m) {
            if constexpr (decltype(is_short)::value) request_short(rq, q, rq_step, rq_copy, rem);
            else request(rq, q, rq_step, rq_copy);
          }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Step `it`, with LEFT more steps behind it.  LEFT == 2: so many at least, and step it + 2 is requested (SHORT:
  // it is the short one).
  auto do_step = [&](int it, auto left, auto is_short) {
    constexpr int LEFT = decltype(left)::value;
    constexpr bool STEADY = LEFT == 2;
    constexpr int YOUNGER = LEFT < 1 ? LEFT : 1;  // whole steps requested after this one
    const int copy = it % 2, next = (it + 1) % 2;
    auto s1 = [] {
      MG_WAIT_VMCNT(YOUNGER * R);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    auto s2 = [] {
      if constexpr (LEFT > 0) {
        MG_WAIT_VMCNT(RA + RB1 + (STEADY ? RA + RB0 : 0));
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      }
    };
    auto no_sync = [] {};
    using QA0 = std::conditional_t<STEADY, A0, None>;
    using QA1 = std::conditional_t<STEADY, A1, None>;
    using QB0 = std::conditional_t<STEADY, B0, None>;
    using QB1 = std::conditional_t<STEADY, B1, None>;
    using NA = std::conditional_t<(LEFT > 0), A0, None>;
    using NB = std::conditional_t<(LEFT > 0), B0, None>;
    phase(A0{}, B0{}, B1{}, copy, QA0{}, it + 2, copy, is_short, s1);
    if constexpr (HAS_BIAS && !SPLIT_K && LEFT == 0) {  // arrives under the last three phases
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        const int col = n0 + wc * S::kWaveN + j * 32 + lane % 32;
        bias_v[j] = col < N ? to_float(pr.bias[col]) : 0.f;
      }
    }
    phase(A0{}, B1{}, A1{}, copy, QB0{}, it + 2, copy, is_short, no_sync);
    phase(A1{}, B1{}, NA{}, next, QB1{}, it + 2, copy, is_short, s2);
    phase(A1{}, B0{}, NB{}, next, QA1{}, it + 2, copy, is_short, no_sync);
  };
  // Requested in the order in which the steps before would have done it.
  auto request_all = [&](auto image, int step) {
    constexpr int IM = decltype(image)::value;
    if (step >= full_steps) {
#pragma unroll
      for (int i = 0; i < S::requests(IM); ++i) request_short(image, i, step, step, step == full_steps ? rem : 0);
      return;
    }
#pragma unroll
    for (int i = 0; i < S::requests(IM); ++i) request(image, i, step, step);
  };
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    request_all(A0{}, s);
    request_all(B0{}, s);
    request_all(B1{}, s);
    request_all(A1{}, s);
  }
  MG_WAIT_VMCNT(RB1 + RA + R);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int n = 0; n < 4 * AI; ++n) read(A0{}, n, 0);
#pragma unroll
  for (int n = 0; n < 4 * BJ0; ++n) read(B0{}, n, 0);
  __builtin_amdgcn_sched_barrier(0);
  int it = 0;
  for (; it + 2 < full_steps; ++it) do_step(it, std::integral_constant<int, 2>{}, std::false_type{});
  if (it < steps - 2) do_step(it, std::integral_constant<int, 2>{}, std::true_type{});
  do_step(steps - 2, std::integral_constant<int, 1>{}, std::false_type{});
  do_step(steps - 1, std::integral_constant<int, 0>{}, std::false_type{});

  const int row0 = m0 + wr * S::kWaveM, col0 = n0 + wc * S::kWaveN;
  if constexpr (COLSUM) {  // a row's two lanes hold the sums over the two halves of every eight-wide slice
#pragma unroll
    for (int i = 0; i < 2 * AI; ++i) {
      const float sum = col_sum[i] + __shfl_xor(col_sum[i], 32);
      const int m = row0 + 32 * i + lane;
      if (wc == 0 && lane < 32 && m < M) pr.colsum_part[static_cast<int64_t>(split) * M + m] = sum;
    }
  }
  if constexpr (SPLIT_K) {
    // Partial tiles in accumulator order (gemm16_partial_floats): sixteen-byte stores, each a contiguous kilobyte.
    const int tiles_m = (M + kGemmBM - 1) / kGemmBM, tiles_n = (N + kGemmBN - 1) / kGemmBN;
    floatx4* const partial = reinterpret_cast<floatx4*>(pr.partial) +
                             (static_cast<int64_t>(split) * pr.batches + batch) * tiles_m * tiles_n * (kG16PartialTile / 4) + lane;
#pragma unroll
    for (int i = 0; i < 2 * AI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        const int r = row0 + 32 * i, c = col0 + 32 * j;
        if (r / kGemmBM >= tiles_m || c / kGemmBN >= tiles_n) continue;
        floatx4* dst = partial + static_cast<int64_t>(r / kGemmBM * tiles_n + c / kGemmBN) * (kG16PartialTile / 4) +
                       ((r / 64 % 2) * 2 + c / 64 % 2) * 1024 + ((r / 32 % 2) * 2 + c / 32 % 2) * 256;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const floatx4 v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
          if (pr.partial_stream) __builtin_nontemporal_store(v, dst + g * 64);
          else dst[g * 64] = v;
        }
      }
  } else {
    if constexpr (OUT_F32) {
      static_assert(!HAS_BIAS && !LN_BWD, "a weight gradient");
#pragma unroll
      for (int i = 0; i < 2 * AI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) gemm16_write_f32(acc[i][j], pr.c32, M, N, pr.ldc, row0 + 32 * i, col0 + 32 * j, lane);
      return;
    }
    __syncthreads();  // every wave is done with the staged tiles: their memory serves the output
    const int64_t at = batch * pr.bsc;
    if constexpr (LN_BWD) {
      gemm16_deep_ln_bwd<T, S>(acc, lds, wave, lane, pr.C + at, M, pr.ldc, tm, m0, pr.ep.residual, pr.ln);
      return;
    }
    uint16_t* mine = reinterpret_cast<uint16_t*>(lds) + wave * 64 * S::kStripStride;
#pragma unroll
    for (int h = 0; h < AI; ++h) {
      gemm16_deep_write<T, HAS_BIAS, BJ, AI == 1>(&acc[2 * h], bias_v, mine, pr.C + at, M, N, pr.ldc, row0 + 64 * h, col0, lane,
                                                 pr.ep.residual ? pr.ep.residual + at : nullptr,
                                                 pr.ep.relu_mask ? pr.ep.relu_mask + at : nullptr, pr.ep.relu);
      __builtin_amdgcn_wave_barrier();
    }
  }
}

template <typename T, class S, bool A_KC, bool B_KC, bool HAS_BIAS, bool SPLIT_K, bool OUT_F32 = false>
__global__ __launch_bounds__(S::kThreads, S::kOccupancy * S::WN / 2) void gemm_16bit_deep_kernel(Gemm16Problem<T> pr) {
  __shared__ __attribute__((aligned(1024))) char lds[S::kLds];
  gemm16_deep_block<T, S, A_KC, B_KC, HAS_BIAS, SPLIT_K, false, false, OUT_F32>(lds, blockIdx.x, pr);
}

// Both products of a Linear layer's backward in one launch: workgroups [0, n_dw) take the K ranges of
// dW = dY^T X (their partial tiles are summed by linear_bwd_finish_kernel afterwards), the rest the
// tiles of dX = dY W.  The longer-running dW ranges start first and the dX tiles fill the CUs as those
// drain, where two launches each end in a tail of half-empty CUs and pay a launch apiece.  With
// dw.colsum_part set, the dW workgroups of the first tile column also produce the bias gradient's
// partial rows from the fragments of dY that they multiply.
template <typename T, class S, bool LN_BWD>
__global__ __launch_bounds__(S::kThreads, S::kOccupancy * S::WN / 2) void linear_bwd_16bit_kernel(Gemm16Problem<T> dw,
                                                                                                 Gemm16Problem<T> dx, int n_dw) {
  __shared__ __attribute__((aligned(1024))) char lds[S::kLds];
  const int bid = blockIdx.x;
  if (bid >= n_dw) {
    gemm16_deep_block<T, S, true, false, false, false, false, LN_BWD>(lds, bid - n_dw, dx);
    return;
  }
  int tile = 0, split, batch, tm, tn = 1;
  if (dw.colsum_part && gemm_split_work(bid, dw.tiles_m * dw.tiles_n, dw.splits, 1, tile, split, batch))
    gemm_tile_of_block(tile, dw.tiles_m, dw.tiles_n, tm, tn, false);
  if (tn == 0) gemm16_deep_block<T, S, false, false, false, true, true>(lds, bid, dw);
  else gemm16_deep_block<T, S, false, false, false, true>(lds, bid, dw);
}

template <typename T>
int launch_16bit_deep(const GemmArgs& g, Gemm16Tile tile, int splits, int k_per_split, float* partial, hipStream_t stream) {
  const bool a_kc = g.sak == 1, b_kc = g.sbk == 1;
  const int64_t tiles_m = ceil_div(g.M, kGemm16TileM[tile]), tiles_n = ceil_div(g.N, kGemm16TileN[tile]);
  const int64_t grid = splits > 1 ? gemm_split_grid(tiles_m * tiles_n, splits, g.batch) : tiles_m * tiles_n * g.batch;
  if (grid > 0x7fffffffLL) return fail(MG_ERR_INVALID, "matmul: too many output tiles");
  Gemm16Problem<T> pr{static_cast<const T*>(g.a), static_cast<const T*>(g.b), static_cast<const T*>(g.bias),
                      static_cast<T*>(g.c), partial, static_cast<int>(g.M), static_cast<int>(g.N), static_cast<int>(g.K),
                      a_kc ? g.sam : g.sak, b_kc ? g.sbn : g.sbk, g.N, g.bsa, g.bsb, g.M * g.N,
                      static_cast<int>(tiles_m), static_cast<int>(tiles_n), k_per_split, splits,
                      static_cast<int>(g.batch), epilogue_of<T>(g)};
  gemm16_gradient(g, pr);
  auto with = [&](auto shape, auto a_layout, auto b_layout) {
    using S = decltype(shape);
    constexpr bool AK = decltype(a_layout)::value, BK = decltype(b_layout)::value;
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(S::kThreads), 0, stream, pr);
    };
    if constexpr (S::AI == 1) {
      if (splits > 1) return launch(gemm_16bit_deep_kernel<T, S, AK, BK, false, true>);
    }
    if constexpr (!AK && !BK) {
      if (g.c_f32) return launch(gemm_16bit_deep_kernel<T, S, AK, BK, false, false, true>);
    }
    if (g.bias) launch(gemm_16bit_deep_kernel<T, S, AK, BK, true, false>);
    else launch(gemm_16bit_deep_kernel<T, S, AK, BK, false, false>);
  };
  auto layouts = [&](auto shape) {
    if (a_kc && b_kc) with(shape, std::true_type{}, std::true_type{});
    else if (a_kc) with(shape, std::true_type{}, std::false_type{});
    else if (b_kc) with(shape, std::false_type{}, std::true_type{});
    else with(shape, std::false_type{}, std::false_type{});
  };
  if (tile == kTile256 && splits <= 1) layouts(Gemm16Deep<2, 2, 2>{});
  else if (tile == kTile192) layouts(Gemm16Deep<1, 2, 1>{});
  else if (tile == kTile128) layouts(Gemm16Deep<1, 1, 1>{});
  else return fail(MG_ERR_INVALID, "matmul: no such tile");
  MG_LAUNCH_CHECK();
  return MG_OK;
}

template <typename T>
int launch_linear_bwd_deep(const Gemm16Problem<T>& pw, const Gemm16Problem<T>& px, Gemm16Tile tile, int64_t n_dw, int64_t n_dx,
                           hipStream_t stream) {
  auto launch = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(n_dw + n_dx)), dim3(threads), 0, stream, pw, px, static_cast<int>(n_dw));
  };
  if (tile == kTileWide) launch(linear_bwd_16bit_kernel<T, Gemm16Deep<1, 2, 1, 4>, true>, 512);
  else if (tile == kTile192) launch(linear_bwd_16bit_kernel<T, Gemm16Deep<1, 2, 1>, false>, 256);
  else if (tile == kTile128) launch(linear_bwd_16bit_kernel<T, Gemm16Deep<1, 1, 1>, false>, 256);
  else return fail(MG_ERR_INVALID, "linear_bwd: no such tile");
  MG_LAUNCH_CHECK();
  return MG_OK;
}

}  // namespace mg
