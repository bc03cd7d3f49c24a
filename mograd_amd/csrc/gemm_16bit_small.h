// 16-bit products with too few 128 x 128 tiles to keep the device busy: 64 x 64 output tiles, four
// waves of 32 x 32, 64 k per step, four copies of the tiles (64 KB of LDS, two workgroups per CU).
//
// What bounds such a product is not a rate but the walk of one workgroup along K: with two copies
// of the tiles a k-step lasts one trip to memory, about 1 us when the CU has no other workgroup to
// turn to ((262, 768) <- 768: 12 steps, 14.8 us in 18 workgroups).  Three k-steps in flight
// and four times the workgroups take both down.  The price is LDS traffic: a 32 x 32 wave tile reads
// two fragments per MFMA where a 64 x 64 one reads one, so half the matrix rate is the most this
// kernel can reach, and products that fill the device with 128 x 128 tiles keep those.
// Copies, LDS images, partial tiles and the order of every sum are those of gemm16_deep_block.
#pragma once

#include "gemm_impl.h"

namespace mg {

constexpr int kSmallT = 64;
constexpr int kSmallBK = 64;
constexpr int kSmallStages = 4;
constexpr int kSmallLdsBytes = kSmallStages * 2 * kSmallT * kSmallBK * 2;

// Output of the 64 x 64 tile: see gemm16_write_tile.  Each wave stages its quadrant, then all 256
// threads store 16 bytes of two rows each.
template <typename T, bool HAS_BIAS, bool SPLIT_K, bool MAY_F32>
__device__ __forceinline__ void gemm16_small_write(const floatx16& acc, uint16_t* __restrict__ strip,
                                                   const Gemm16Problem<T>& pr, int batch, int split, int m0, int n0,
                                                   int wm, int wn, int lane, float bias_v) {
  const int M = pr.M, N = pr.N;
  if constexpr (SPLIT_K) {
    const int tiles_n = (N + kGemmBN - 1) / kGemmBN, tiles_m = (M + kGemmBM - 1) / kGemmBM;
    const int64_t tile_at = (static_cast<int64_t>(split) * pr.batches + batch) * tiles_m * tiles_n +
                            static_cast<int64_t>(m0 / kGemmBM) * tiles_n + n0 / kGemmBN;
    float4* dst = reinterpret_cast<float4*>(pr.partial) + tile_at * (kG16PartialTile / 4) +
                  ((m0 / 64) % 2 * 2 + (n0 / 64) % 2) * 1024 + ((wm / 32) * 2 + wn / 32) * 256 + lane;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const floatx4 v = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
      if (pr.partial_stream) __builtin_nontemporal_store(v, reinterpret_cast<floatx4*>(dst + g * 64));
      else *reinterpret_cast<floatx4*>(dst + g * 64) = v;
    }
    return;
  } else {
    if constexpr (MAY_F32) {
      if (pr.c32) {
        gemm16_write_f32(acc, pr.c32, M, N, pr.ldc, m0 + wm, n0 + wn, lane);
        return;
      }
    }
    const GemmEpilogue<T>& ep = pr.ep;
    const int odd = lane & 1;
    const uint32_t select = odd ? 0x03020706u : 0x05040100u;
    uint32_t* const base32 = reinterpret_cast<uint32_t*>(
        strip + (wm + (lane / 32) * 4 + odd) * kG16Stride + wn + (lane % 32 - odd));
#pragma unroll
    for (int rp = 0; rp < 8; ++rp) {
      float f0 = acc[2 * rp], f1 = acc[2 * rp + 1];
      if constexpr (HAS_BIAS) f0 += bias_v, f1 += bias_v;
      if (ep.relu) {
        f0 = f0 > 0.f ? f0 : 0.f;
        f1 = f1 > 0.f ? f1 : 0.f;
      }
      const uint32_t w = gemm16_pack2<T>(f0, f1);
      const uint32_t y = __builtin_amdgcn_update_dpp(w, w, kDppQuadXor1, 0xf, 0xf, false);
      const int rl = (rp / 2) * 8 + (rp % 2) * 2;
      base32[(rl * kG16Stride) / 2] = __builtin_amdgcn_perm(y, w, select);
    }
    __syncthreads();
    const int rl0 = threadIdx.x / 8, ch = threadIdx.x % 8;
    const int col = n0 + ch * 8;
    if (col >= N) return;
    T* C = pr.C + batch * pr.bsc;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = m0 + rl0 + 32 * i;
      if (row >= M) break;
      const uint16_t* src = strip + (rl0 + 32 * i) * kG16Stride + ch * 8;
      const int64_t at = static_cast<int64_t>(row) * pr.ldc + col;
      const int64_t eat = batch * pr.bsc + at;  // the epilogue's arrays are laid out like the whole of C
      if (col + 8 > N) {  // the chunk over the right edge, element by element
        for (int e = 0; col + e < N; ++e) {
          float v = to_float(reinterpret_cast<const T*>(src)[e]);
          if (ep.relu_mask) v = to_float(ep.relu_mask[eat + e]) > 0.f ? v : 0.f;
          if (ep.residual) v += to_float(ep.residual[eat + e]);
          C[at + e] = from_float<T>(v);
        }
        continue;
      }
      if (!ep.residual && !ep.relu_mask) {
        const uint4 r = *reinterpret_cast<const uint4*>(src);
        const gemm_u4_any out = {r.x, r.y, r.z, r.w};
        *reinterpret_cast<gemm_u4_any*>(C + at) = out;
        continue;
      }
      float v[8];
      VecIO<T, 8>::load(reinterpret_cast<const T*>(src), v);
      if (ep.relu_mask) {
        float mk[8];
        gemm16_load8(ep.relu_mask + eat, mk);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = mk[e] > 0.f ? v[e] : 0.f;
      }
      if (ep.residual) {
        float rs[8];
        gemm16_load8(ep.residual + eat, rs);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += rs[e];
      }
      gemm16_store8(C + at, v);
    }
  }
}

// What a thread carries of an operand that does not lie on 16-byte chunks: its chunks of a step, read from any address
// (extents along the contiguous axis: at least 8).  A chunk that reaches past the end of its row is read as the sixteen
// bytes that end it and moved down when it is put into LDS, so that no load stands under a condition and none is waited
// for before its step (moved when they arrive, the tiles on an edge paid a memory latency per step: backward of
// (1999, 1001 <- 768) 40 us).
template <bool KC>
struct SmallAnySource {
  static constexpr int NW = 4, NI = gemm16_pipe_requests(kSmallT, kSmallBK, NW);
  const uint16_t* base;
  int64_t ld;
  int o0, O, k_begin, K;
  const uint16_t* row[NI];  // the chunks of the first step
  __device__ __forceinline__ static void place(int i, int& line, int& chunk) {  // as gemm16_pipe_sources has them
    const int slot = (i * NW + threadIdx.x / kWave) * kWave + threadIdx.x % kWave;
    line = slot / 8;
    chunk = (slot % 8) ^ (KC ? (line / 2) % 8 : gemm16_tr_swizzle<kSmallT>(line));
  }
  __device__ __forceinline__ void init(const uint16_t* base_, int64_t ld_, int o0_, int O_, int k_begin_, int K_) {
    base = base_, ld = ld_, o0 = o0_, O = O_, k_begin = k_begin_, K = K_;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      int line, chunk;
      place(i, line, chunk);
      row[i] = KC ? base + static_cast<int64_t>(min(o0 + line, O - 1)) * ld + k_begin + chunk * 8
                  : base + static_cast<int64_t>(k_begin + line) * ld + min(o0 + chunk * 8, O - 8);
    }
  }
  __device__ __forceinline__ void fetch(int step, uint4 (&v)[NI]) const {
    const int k0 = k_begin + step * kSmallBK;
    int64_t back[NI] = {};  // in the last step: what a chunk past the end is moved back by
    if (k0 + kSmallBK > K) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        int line, chunk;
        place(i, line, chunk);
        back[i] = KC ? max(k0 + chunk * 8 + 8 - K, 0) : max(k0 + line + 1 - K, 0) * ld;
      }
    }
    const int64_t by = step * (KC ? static_cast<int64_t>(kSmallBK) : kSmallBK * ld);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const gemm_u4_any r = *reinterpret_cast<const gemm_u4_any*>(row[i] + by - back[i]);
      v[i] = make_uint4(r[0], r[1], r[2], r[3]);
    }
  }
  __device__ __forceinline__ void put(int step, uint4 (&v)[NI], char* lds_step) const {
    const int k0 = k_begin + step * kSmallBK;
    if (k0 + kSmallBK > K || (!KC && o0 + kSmallT > O)) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        int line, chunk;
        place(i, line, chunk);
        const int past = max((KC ? k0 : o0) + chunk * 8 + 8 - (KC ? K : O), 0);
        const bool odd = past & 1, one = past & 2, two = past & 4, none = past >= 8 || (!KC && k0 + line >= K);
        uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = odd ? w[j] >> 16 | (j < 3 ? w[j + 1] << 16 : 0u) : w[j];
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = one ? (j < 3 ? w[j + 1] : 0u) : w[j];
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = none ? 0u : two ? (j < 2 ? w[j + 2] : 0u) : w[j];
        v[i] = make_uint4(w[0], w[1], w[2], w[3]);
      }
    }
#pragma unroll
    for (int i = 0; i < NI; ++i)
      *reinterpret_cast<uint4*>(lds_step + ((i * NW + threadIdx.x / kWave) * kWave + threadIdx.x % kWave) * 16) = v[i];
  }
};

// The work of workgroup `bid` of a launch for one product (see gemm16_deep_block); pr.tiles_m and
// pr.tiles_n count tiles of 64.  MAY_F32: pr.c32 is looked at.  ANY: operands that do not lie on 16-byte chunks, which the
// copies into LDS cannot take, come through registers, two steps of them under way and two in LDS.  Copied to rows that do
// they cost a launch and a pass of 5 us, and the 128 x 128 kernel that stages them leaves CUs idle: (700, 701 <- 703) bf16
// forward + backward 38.7 -> 20.6 us, (2048, 1000 <- 1001) forward 20.7 -> 15.1.  A step takes a third longer than a copied one,
// misaligned chunks being two of the memory path's; more steps under way (four) measured the same.
template <typename T, bool A_KC, bool B_KC, bool HAS_BIAS, bool SPLIT_K, bool COLSUM, bool MAY_F32 = COLSUM, bool ANY = false>
__device__ __forceinline__ void gemm16_small_block(char* lds, int bid, const Gemm16Problem<T>& pr) {
  constexpr int TT = kSmallT, BK = kSmallBK, NSTAGE = kSmallStages, NW = 4;
  constexpr int NI = gemm16_pipe_requests(TT, BK, NW);  // copy requests per thread, operand and step
  static_assert(gemm16_pipe_waves(TT, BK, NW) == NW, "every wave copies its share of either operand");
  constexpr int OP = TT * BK * 2;  // bytes of an operand's step
  const int M = pr.M, N = pr.N, K = pr.K;

  const int tiles = pr.tiles_m * pr.tiles_n;
  int batch = bid / tiles, tile = bid % tiles, split = 0;
  if constexpr (SPLIT_K) {
    if (!gemm_split_work(bid, tiles, pr.splits, pr.batches, tile, split, batch)) return;
  }
  int tm, tn;
  gemm_tile_of_block(tile, pr.tiles_m, pr.tiles_n, tm, tn, !SPLIT_K);
  const int m0 = tm * TT, n0 = tn * TT;
  const int k_begin = SPLIT_K ? split * pr.k_per_split : 0;
  const int k_end = SPLIT_K ? min(K, k_begin + pr.k_per_split) : K;
  const int full_steps = (k_end - k_begin) / BK, rem = (k_end - k_begin) % BK;
  const int steps = full_steps + (rem > 0 ? 1 : 0);
  const T* A = pr.A + batch * pr.bsa + (A_KC ? static_cast<int64_t>(k_begin) : k_begin * pr.lda);
  const T* B = pr.B + batch * pr.bsb + (B_KC ? static_cast<int64_t>(k_begin) : k_begin * pr.ldb);
  const int64_t a_step = A_KC ? BK : BK * pr.lda;
  const int64_t b_step = B_KC ? BK : BK * pr.ldb;

  const int wave = threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  const int wm = (wave / 2) * 32;
  const int wn = (wave % 2) * 32;

  floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;

  // Column sums of the A tiles (see Gemm16Problem::colsum_part): the tiles times a column of ones, one
  // more MFMA per slice for the waves of the tile's first half.  (Read back from LDS and added by
  // the vector units they cost half a step again: dW (256, 256) <- 2587 with db 18.4 us against 13.5.)
  static_assert(!COLSUM || !A_KC, "the columns of dY are summed from an m-contiguous operand");
  const bool colsum = COLSUM && tn == 0 && wn == 0 &&
                      (SPLIT_K ? pr.colsum_part != nullptr : pr.colsum != nullptr || pr.colsum32 != nullptr);
  floatx16 cs;
#pragma unroll
  for (int r = 0; r < 16; ++r) cs[r] = 0.f;
  const uint32_t one = gemm16_pack2<T>(1.f, 1.f);
  const uint4 ones = make_uint4(one, one, one, one);

  const uint16_t* a16 = reinterpret_cast<const uint16_t*>(A);
  const uint16_t* b16 = reinterpret_cast<const uint16_t*>(B);
  int64_t src_a[NI], src_b[NI];
  SmallAnySource<A_KC> any_a;
  SmallAnySource<B_KC> any_b;
  uint4 va[2][NI], vb[2][NI];  // ANY: the steps under way
  if constexpr (ANY) {
    any_a.init(reinterpret_cast<const uint16_t*>(pr.A + batch * pr.bsa), pr.lda, m0, M, k_begin, K);
    any_b.init(reinterpret_cast<const uint16_t*>(pr.B + batch * pr.bsb), pr.ldb, n0, N, k_begin, K);
  } else {
    gemm16_pipe_sources<A_KC, BK, TT, NW>(pr.lda, m0, M, src_a);
    gemm16_pipe_sources<B_KC, BK, TT, NW>(pr.ldb, n0, N, src_b);
  }
  auto fetch = [&](int set, int step) {
    any_a.fetch(step, va[set]);
    any_b.fetch(step, vb[set]);
  };
  auto put = [&](int set, int step) {
    char* at = lds + step % NSTAGE * 2 * OP;
    any_a.put(step, va[set], at);
    any_b.put(step, vb[set], at + OP);
  };
  auto request = [&](int step, int copy) {
    char* at = lds + copy * 2 * OP;
    if (step == full_steps) {
      gemm16_pipe_issue_short<A_KC, BK, TT, NW>(a16 + step * a_step, src_a, rem, at);
      gemm16_pipe_issue_short<B_KC, BK, TT, NW>(b16 + step * b_step, src_b, rem, at + OP);
      return;
    }
    gemm16_pipe_issue<NI, NW>(a16 + step * a_step, src_a, at);
    gemm16_pipe_issue<NI, NW>(b16 + step * b_step, src_b, at + OP);
  };

  if constexpr (!ANY) {
#pragma unroll
    for (int s = 0; s < NSTAGE; ++s)
      if (s < steps) request(s, s);
  } else {
#pragma unroll
    for (int s = 0; s < 2; ++s)
      if (s < steps) fetch(s, s);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (s < steps) put(s, s);
      if (s + 2 < steps) fetch(s, s + 2);
    }
  }
  // The fragments of step `it` + 1 are read while those of step `it` are multiplied, so a step's one
  // synchronisation says two things: step it + 1 has arrived, and every wave holds its fragments of
  // step it, whose copy then takes step it + NSTAGE.
  uint4 fa[2][BK / 16], fb[2][BK / 16];
  // (The waits are builtins here: the compiler then knows that step it's fragments are in their
  // registers and does not wait for step it + 1's as well before it multiplies.)
  auto meet = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto arrive = [&](int younger) {  // all but the `younger` steps' requests are there
    static_assert(NSTAGE == 4, "cases below");
    switch (younger) {
      case 3: MG_WAIT_VMCNT(2 * NI * 3); break;
      case 2: MG_WAIT_VMCNT(2 * NI * 2); break;
      case 1: MG_WAIT_VMCNT(2 * NI * 1); break;
      default: MG_WAIT_VMCNT(0);
    }
    meet();
  };
  auto read = [&](int buf, int step) {
    const char* la = lds + (step % NSTAGE) * 2 * OP;
    const char* lb = la + OP;
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      fa[buf][ks] = gemm16_pipe_frag<A_KC, BK, TT>(la, wm, ks, lane);
      fb[buf][ks] = gemm16_pipe_frag<B_KC, BK, TT>(lb, wn, ks, lane);
    }
  };
  auto multiply = [&](int buf) {
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) acc = GemmMma16<T>::run(fa[buf][ks], fb[buf][ks], acc);
    if constexpr (COLSUM) {
      if (colsum) {
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) cs = GemmMma16<T>::run(fa[buf][ks], ones, cs);
      }
    }
  };
  auto turn = [&](int buf, int it, auto steady) {
    if constexpr (ANY) {
      meet();
      if (it + 2 < steps) put(buf, it + 2);  // (its place was last read two steps ago)
      if (it + 4 < steps) fetch(buf, it + 4);
    } else if constexpr (decltype(steady)::value) {
      MG_WAIT_VMCNT(2 * NI * (NSTAGE - 2));
      meet();
    } else {
      arrive(min(steps - 2 - it, NSTAGE - 2));
    }
    if (!ANY && it + NSTAGE < steps) request(it + NSTAGE, it % NSTAGE);
    read(buf ^ 1, it + 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(buf);
  };
  if constexpr (ANY) meet();
  else arrive(min(steps - 1, NSTAGE - 1));
  read(0, 0);
  // two turns at a time, so that the fragment buffers have fixed names
  int it = 0;
  for (; !ANY && it + NSTAGE < full_steps; it += 2) {
    turn(0, it, std::true_type{});
    turn(1, it + 1, std::true_type{});
  }
  for (; it + 2 < steps; it += 2) {
    turn(0, it, std::false_type{});
    turn(1, it + 1, std::false_type{});
  }
  float bias_v = 0.f;  // under the last products: ahead of the tiles, the wait for it took in all their copies
  if constexpr (HAS_BIAS && !SPLIT_K) {
    const int col = n0 + wn + lane % 32;
    bias_v = col < N ? to_float(pr.bias[col]) : 0.f;
  }
  if (it + 1 < steps) {
    turn(0, it, std::false_type{});
    multiply(1);
  } else {
    multiply(0);
  }
  __syncthreads();  // every wave is done with the staged tiles: their memory serves the output

  if constexpr (COLSUM) {
    if (colsum && lane % 32 == 0) {  // every column holds the sums
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + wm + (r / 4) * 8 + (lane / 32) * 4 + r % 4;
        if (m >= M) continue;
        if constexpr (SPLIT_K) pr.colsum_part[static_cast<int64_t>(split) * M + m] = cs[r];
        else if (pr.colsum32) pr.colsum32[m] = cs[r];
        else pr.colsum[m] = from_float<T>(cs[r]);
      }
    }
  }
  gemm16_small_write<T, HAS_BIAS, SPLIT_K, MAY_F32>(acc, reinterpret_cast<uint16_t*>(lds), pr, batch, split, m0, n0, wm, wn, lane,
                                           bias_v);
}

template <typename T, bool A_KC, bool B_KC, bool HAS_BIAS, bool SPLIT_K, bool ANY>
__global__ __launch_bounds__(256, 2) void gemm_16bit_small_kernel(Gemm16Problem<T> pr) {
  __shared__ __attribute__((aligned(1024))) char lds[kSmallLdsBytes];
  // (dW = dY^T X is the layout that fp32 weight gradients come in)
  gemm16_small_block<T, A_KC, B_KC, HAS_BIAS, SPLIT_K, false, !A_KC && !B_KC && !HAS_BIAS, ANY>(lds, blockIdx.x, pr);
}

// dX and dW (with db, the column sums of dY) of a Linear layer in one launch, see
// linear_bwd_16bit_kernel: workgroups [0, n_dw) take dW, the rest dX.
template <typename T, bool SPLIT, bool ANY>
__global__ __launch_bounds__(256, 2) void linear_bwd_small_16bit_kernel(Gemm16Problem<T> dw, Gemm16Problem<T> dx,
                                                                        int n_dw) {
  __shared__ __attribute__((aligned(1024))) char lds[kSmallLdsBytes];
  const int bid = blockIdx.x;
  if (bid < n_dw) gemm16_small_block<T, false, false, false, SPLIT, true, true, ANY>(lds, bid, dw);
  else gemm16_small_block<T, true, false, false, false, false, false, ANY>(lds, bid - n_dw, dx);
}

}  // namespace mg
