// Flash attention of fp32 tensors on the matrix cores (v_mfma_f32_32x32x2_f32) with waves that walk on
// their own: what fp32 tensors of up to 256 head columns take when their rows lie on 16-byte chunks.
//
// A workgroup owns 32 rows of one head (queries in the forward and dQ, keys in dK/dV), and its
// four waves share the walk over the streamed rows.  Up to 128 head columns wave w takes the tiles
// w, w + 4, ... of 32 streamed rows, and the four partial results meet in LDS at the end; with
// more columns every wave takes every tile but only a quarter of the columns, and the partial
// scores of a step meet in LDS.  A wave's tiles are its own: they are copied straight into its part
// of LDS (`global_load_lds`), waited for with its own counter, and no barrier stands in the loop of
// the first form.  The other fp32 kernels give a workgroup 128 rows, all waves the same tiles and
// two barriers a step: three heads of 777 rows are then 21 workgroups where 75 of these fill a
// third of the device, and a sequence of 32 is one wave's work.  80 and 96 columns have kernels of
// their own instead of the 128-column one.
//   fp32 forward + backward, one MI355X, before these kernels -> with a launch for each walk -> with one for both:
//     (3, 777, 8 heads, 80), bias        645 -> 381 -> 336 us      (1, 1236, 6, 256), causal  3930 -> 520 -> 406 us
//     (1, 500, 2 heads, 64), bias               66 ->  46 us       (2, 8 heads of 1500, 128)   816 -> 782 -> 777 us
//     (4, 32, 2, 32), causal              65 ->  18 ->  12 us      (21, 79, 8, 32), causal      35 ->  28 ->  27 us
// Where the walks have little to gain from each other's company, each has a launch (f32_wave_together has the choice): two
// walks of 600 workgroups end in two rounds of which a third is empty, five rounds of both together in one, and a short sequence
// waits for one kernel instead of two, but walks of whole rounds lose dQ's second workgroup per CU.  The arithmetic is the matrix pipe's: 64 cycles per 32 x 32 x 2 product, two
// products per column and step forward, seven over the two backward kernels.  What stands beside it on the one
// wave of a SIMD is vector arithmetic, 1300 instructions a step at 80 columns until the copies took a scalar base
// and a byte offset per lane, the bias' places were computed once, and exp2f became the one instruction:
// 414 -> 389 us at 777 rows with bias, 260 -> 228 us at (2, 8 heads of 1024, 64) with bias; 1.5 and 2 % of that went
// back to weights below 2^-126, see f32_wave_exp2.
//
// Layouts as in attention_f32_mfma.h: a score tile comes out with the workgroup's rows along the
// lanes and the streamed rows along the registers, which is the operand of the products that
// contract over the streamed rows; lane half h takes every second chunk of four
// head columns, from chunk h on, of a score.
// A single copy of each tile suffices because the two tensors of a step are used in turn: the next
// step's tile of one is copied while the other is multiplied.
//
// LDS image of a tile: [32 rows][DP / 4 chunks of 16 bytes], the chunks of a group of X permuted by
// c ^ (r / (16 / X)) in row r, which puts the sixteen rows of a 128-bit read on sixteen different bank
// groups and leaves few distinct addresses per lane (a rotation instead took 150 registers of them).  Rows past the sequence are copies of the last one, columns past D repeat the last
// chunk; the mask, zeros in the resident operand and the bounds of the stores drop what they give.
#pragma once

#include "attention_f32_mfma.h"

namespace mg {

constexpr int kF32WaveMaxD = 256;

// 2^x of a lane's sixteen weights, as exp2f gives them.  exp2f scales its argument around v_exp_f32 so that results below
// 2^-126 come out as denormals, which show where a key's weights are all such (its dK, dV) or its V is all there is, and costs
// six instructions a weight; here that is done only where a lane of the wave has such a weight (x in [-150, -126): what a
// mask hides is far below), and v_exp_f32 alone gives the same bits elsewhere.  (3, 777, 8 heads, 80), bias, with a launch for
// each walk: forward 99.5 us against 103 with exp2f; the dK/dV walk, whose accumulators then move about, is faster with
// exp2f: whole backward 285 us against 290, (2, 8 heads of 1024, 64), bias, 162 against 165.
__device__ __forceinline__ void f32_wave_exp2(f32x16& x) {
  float least = x[0];
#pragma unroll
  for (int r = 1; r < 16; ++r) least = fminf(least, x[r]);
  if (__builtin_expect(__any(least < -126.0f), 0)) {
    float off = INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) off = fminf(off, fabsf(x[r] + 138.0f));
    if (__any(off <= 12.0f)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) x[r] = exp2f(x[r]);
      return;
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) x[r] = __builtin_amdgcn_exp2f(x[r]);
}

// The same in two parts: v_exp_f32 of all sixteen, which no branch keeps from standing among other work, and exp2f in its
// place where a lane has such a weight.
__device__ __forceinline__ void f32_wave_exp2_amend(const f32x16& x, f32x16& p) {
  float least = x[0];
#pragma unroll
  for (int r = 1; r < 16; ++r) least = fminf(least, x[r]);
  if (__builtin_expect(!__any(least < -126.0f), 1)) return;
  float off = INFINITY;
#pragma unroll
  for (int r = 0; r < 16; ++r) off = fminf(off, fabsf(x[r] + 138.0f));
  if (!__any(off <= 12.0f)) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) p[r] = exp2f(x[r]);
}

// What the four waves of a workgroup share: the streamed rows of one tile of 32, nothing (each has a
// tile of its own), or the head columns of one tile.
enum F32WaveMode { kF32SplitRows, kF32OwnTiles, kF32SplitColumns };

template <int DP>
struct F32Wave {
  static constexpr int CH = DP / 4;  // chunks of a row
  static constexpr int X = CH % 16 == 0 ? 16 : CH % 8 == 0 ? 8 : 4;  // chunks that are permuted among themselves
  static constexpr int NI = DP / 8;          // copies of a wave per tile
  static constexpr int NB = (DP + 31) / 32;  // 32-column blocks of a result
  static constexpr int TILE = 32 * DP * 4;   // bytes
  static_assert(CH % 4 == 0 && DP % 16 == 0, "whole groups of chunks");
  static __device__ __forceinline__ int swizzle(int row) { return row / (16 / X) % X; }
  // Place, in floats, of chunk X * group + c (c < X) of a row.
  static __device__ __forceinline__ int place(int row, int c, int group) {
    return row * DP + (c ^ swizzle(row)) * 4 + group * (X * 4);
  }
};
constexpr int kF32BiasTile = 32 * 32 * 4;

// Bytes of a wave's tiles, and of a workgroup's LDS: the tiles and, when the columns are divided among
// the waves, two copies of the exchange of `scores` score tiles.
template <int DP, bool HAS_BIAS>
constexpr int f32_wave_bytes() { return 2 * F32Wave<DP>::TILE + (HAS_BIAS ? kF32BiasTile : 0); }
template <int DP, F32WaveMode MODE, bool HAS_BIAS>
constexpr int f32_wave_lds(int scores) {
  return 4 * f32_wave_bytes<DP, HAS_BIAS>() + (MODE == kF32SplitColumns ? 2 * 4 * scores * 4096 : 0);
}
// Whether the dK/dV walk is handed delta or forms it itself: 64 registers of O's row beside the resident rows and accumulators
// of 128 columns are spilled.
template <int DP>
constexpr bool f32_wave_delta_given() { return DP == 128; }
// Workgroups per CU that the registers are budgeted for.  80 columns without a bias are 80 KB of LDS, two to a CU,
// one's softmax beside the other's products: (3, 777, 8 heads, 80) 92 + 265 us -> 78 + 242, causal 50 + 154 ->
// 40 + 139.  With a bias it is 96 KB; loading that straight to registers instead, to get under, is slower than
// its copies (32 rows to a load: 96 columns 70 -> 77 us, 128 columns 76 -> 86), and dQ then spills.
template <int DP, F32WaveMode MODE, bool HAS_BIAS>
constexpr int f32_wave_occupancy(int results) {
  if (MODE == kF32SplitColumns) return 1;
  return DP <= 32 || (DP <= 64 && results == 1) || (DP <= 80 && !HAS_BIAS && results == 1) ? 2 : 1;
}

// See gemm16_deep_issue for why these are assembly.  `base` is the same for the wave; with a byte offset per lane
// a copy costs no vector arithmetic (a 64-bit address per lane and copy was 3 instructions).
__device__ __forceinline__ void f32_wave_copy16(const float* base, unsigned bytes, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(bytes), "s"(base) : "memory");
}
__device__ __forceinline__ void f32_wave_copy4(const float* base, unsigned bytes, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2" ::"s"(dst), "v"(bytes), "s"(base) : "memory");
}
__device__ __forceinline__ void f32_wave_copy4_at(const float* src, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off" ::"s"(dst), "v"(src) : "memory");
}
__device__ __forceinline__ unsigned f32_wave_lds_at(const char* p) {
  using lds_ptr = __attribute__((address_space(3))) const char*;
  return __builtin_amdgcn_readfirstlane(static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_ptr)p)));
}
// At most N of the wave's copies are outstanding, and none of its LDS reads.
#define MG_F32_WAVE_WAIT(N)                                                        \
  do {                                                                             \
    asm volatile("" ::: "memory");                                                 \
    __builtin_amdgcn_s_waitcnt(((N) & 15) | (((N) >> 4) << 14) | 0x0070);          \
    asm volatile("" ::: "memory");                                                 \
  } while (0)

// A tensor whose tiles a wave copies: rows of `ld` elements, S of them, the wave's columns first.
template <int DP>
struct F32WaveTiles {
  const float* base;
  int64_t ld;
  int S, last_chunk;
  unsigned off[F32Wave<DP>::NI];  // the lane's place in a whole tile, in bytes
  __device__ __forceinline__ void source(int i, int lane, int& row, int& c) const {
    using W = F32Wave<DP>;
    const int slot = i * 64 + lane;
    row = slot / W::CH;
    c = slot % W::CH;
    c = min((c % W::X ^ W::swizzle(row)) + c / W::X * W::X, last_chunk);
  }
  __device__ __forceinline__ void init(const float* base_, int64_t ld_, int S_, int columns, int lane) {
    base = base_;
    ld = ld_;
    S = S_;
    last_chunk = columns / 4 - 1;
#pragma unroll
    for (int i = 0; i < F32Wave<DP>::NI; ++i) {
      int row, c;
      source(i, lane, row, c);
      off[i] = static_cast<unsigned>(row * ld + c * 4) * 4;
    }
  }
  __device__ __forceinline__ void copy(int row0, const char* tile, int lane) const {
    const unsigned dst = f32_wave_lds_at(tile);
    const float* p = base + row0 * ld;
    if (row0 + 32 <= S) {
#pragma unroll
      for (int i = 0; i < F32Wave<DP>::NI; ++i) f32_wave_copy16(p, off[i], dst + i * 1024);
      return;
    }
    asm volatile("" : "+v"(lane));  // computed here, once per walk, and not kept in registers throughout
#pragma unroll
    for (int i = 0; i < F32Wave<DP>::NI; ++i) {
      int row, c;
      source(i, lane, row, c);
      f32_wave_copy16(p, static_cast<unsigned>(min(row, S - 1 - row0) * ld + c * 4) * 4, dst + i * 1024);
    }
  }
};

// The bias of queries i0 .. + 31 and keys j0 .. + 31, as a tile of 32 columns, in 4-byte copies (its rows
// start anywhere).  Copy i takes rows 2 i and 2 i + 1, whose chunks are permuted by i % 8: the lane's byte in a row
// is (4 (lane % 32)) ^ 16 (i % 8).  A tile that reaches past the sequence has its places computed one by one.
struct F32WaveBias {
  unsigned off[8];
  __device__ __forceinline__ void init(int S, int lane) {
    static_assert(F32Wave<32>::X == 8, "rows 2 i and 2 i + 1 are permuted alike, eight ways");
#pragma unroll
    for (int i = 0; i < 8; ++i) off[i] = static_cast<unsigned>(lane / 32 * S) * 4 + ((lane % 32 * 4) ^ (i * 16));
  }
  __device__ __forceinline__ void copy(const float* mask, int i0, int j0, int S, const char* tile, int lane) const {
    const unsigned dst = f32_wave_lds_at(tile);
    if (i0 + 32 <= S && j0 + 32 <= S) {
      const float* p = mask + static_cast<int64_t>(i0) * S + j0;
#pragma unroll
      for (int i = 0; i < 16; ++i) f32_wave_copy4(p + 2 * i * static_cast<int64_t>(S), off[i % 8], dst + i * 256);
      return;
    }
    asm volatile("" : "+v"(lane));  // (not kept in registers)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 2 * i + lane / 32, col = (lane % 32) ^ (i % 8 * 4);
      f32_wave_copy4_at(mask + static_cast<int64_t>(min(i0 + row, S - 1)) * S + min(j0 + col, S - 1), dst + i * 256);
    }
  }
};

// The fragments of a group of products are read while the group before it is multiplied: left to itself the compiler
// reads each a few cycles ahead of its product, and with one wave to a SIMD the matrix pipe waits for LDS every time
// (vector arithmetic may pass these fences).
#define MG_F32_WAVE_GROUP() __builtin_amdgcn_sched_barrier(0x6)

// tile * resident^T over the wave's columns (see f32_attn_scores).  DOT: and the lane's share of the dot product of the
// tile's row with `other`, whose chunks past `columns` columns hold anything.
template <int DP, bool DOT>
__device__ __forceinline__ f32x16 f32_wave_scores_dot(const char* tile, const float (&resident)[DP / 2],
                                                      const float4 (&other)[DP / 8], int columns, int lane, float& dot) {
  using W = F32Wave<DP>;
  constexpr int N = 2, GROUPS = DP / 8 / N;  // chunks to a group
  static_assert(DP / 8 % N == 0, "whole groups");
  const float* t = reinterpret_cast<const float*>(tile);
  const int row = lane % 32, half = lane / 32;
  f32x16 acc[2] = {f32x16_zero(), f32x16_zero()};  // two chains: a product does not wait for the one before it
  if constexpr (DOT) dot = 0.f;
  float4 w[2][N];
  auto read = [&](int g) {
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const int c = g * N + e;
      w[g % 2][e] = *reinterpret_cast<const float4*>(t + W::place(row, 2 * (c % (W::X / 2)) + half, c / (W::X / 2)));
    }
  };
  read(0);
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    if (g + 1 < GROUPS) read(g + 1);
    MG_F32_WAVE_GROUP();
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const int c = g * N + e;
      const float4 x = w[g % 2][e];
      acc[0] = f32_mfma(x.x, resident[c * 4], acc[0]);
      acc[1] = f32_mfma(x.y, resident[c * 4 + 1], acc[1]);
      acc[0] = f32_mfma(x.z, resident[c * 4 + 2], acc[0]);
      acc[1] = f32_mfma(x.w, resident[c * 4 + 3], acc[1]);
      if constexpr (DOT) {
        float d = dot;
        d = fmaf(x.x, other[c].x, d);
        d = fmaf(x.y, other[c].y, d);
        d = fmaf(x.z, other[c].z, d);
        d = fmaf(x.w, other[c].w, d);
        dot = (2 * c + half) * 4 < columns ? d : dot;
      }
    }
    MG_F32_WAVE_GROUP();
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[0][r] += acc[1][r];
  return acc[0];
}
template <int DP>
__device__ __forceinline__ f32x16 f32_wave_scores(const char* tile, const float (&resident)[DP / 2], int lane) {
  float4 none[DP / 8];
  float dot;
  return f32_wave_scores_dot<DP, false>(tile, resident, none, 0, lane, dot);
}

// out[db] += tile^T * w over the tile's 32 rows (see f32_attn_weighted).
template <int DP>
__device__ __forceinline__ void f32_wave_weighted(const char* tile, const f32x16& w, int lane,
                                                  f32x16 (&out)[F32Wave<DP>::NB]) {
  using W = F32Wave<DP>;
  constexpr int N = W::NB > 2 ? 4 : 8;  // rows to a group
  const float* t = reinterpret_cast<const float*>(tile);
  const int half = lane / 32, col = lane % 32;
  float x[2][N][W::NB];
  auto read = [&](int g) {
#pragma unroll
    for (int e = 0; e < N; ++e) {
      const int j = g * N + e;
      // row 8 (j / 4) + 4 half + j % 4, with what the lane adds to it apart
      const int fixed = j / 4 * 8 + j % 4, row = fixed + half * 4;
#pragma unroll
      for (int db = 0; db < W::NB; ++db) {
        // Chunks db * 8 .. + 7; of a last block of sixteen columns its four chunks twice over (dropped).
        const int left = W::CH - db * 8 < 8 ? W::CH - db * 8 : 8;
        const int c = col / 4 % left;
        if constexpr (W::X == 16) x[g % 2][e][db] = t[W::place(row, db % 2 * 8 + c, db / 2) + col % 4];
        else if constexpr (W::X == 8) x[g % 2][e][db] = t[W::place(row, c, db) + col % 4];
        else x[g % 2][e][db] = t[W::place(row, c % 4, 2 * db) + c / 4 * 16 + col % 4];
      }
    }
  };
  read(0);
#pragma unroll
  for (int g = 0; g < 16 / N; ++g) {
    if (g + 1 < 16 / N) read(g + 1);
    MG_F32_WAVE_GROUP();
#pragma unroll
    for (int e = 0; e < N; ++e)
#pragma unroll
      for (int db = 0; db < W::NB; ++db) out[db] = f32_mfma(x[g % 2][e][db], w[g * N + e], out[db]);
    MG_F32_WAVE_GROUP();
  }
}

// Sums the four waves' score tiles of a step; `area` is the step's half of the exchange.  Every wave adds
// in the same order, so all hold the same scores.
template <int N>
__device__ __forceinline__ void f32_wave_exchange(char* area, int wave, int lane, f32x16 (&s)[N]) {
  float4* x = reinterpret_cast<float4*>(area);  // [wave][tile][register / 4][lane]
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      x[((wave * N + n) * 4 + g) * 64 + lane] = make_float4(s[n][4 * g], s[n][4 * g + 1], s[n][4 * g + 2], s[n][4 * g + 3]);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (not __syncthreads(): the copies go on)
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float4 v = x[((w * N + n) * 4 + g) * 64 + lane];
        t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w;
      }
      s[n][4 * g] = t.x; s[n][4 * g + 1] = t.y; s[n][4 * g + 2] = t.z; s[n][4 * g + 3] = t.w;
    }
}

// Block id -> (head, 32-row tile).  Tiles of a head are consecutive work items and an XCD (id mod 8) takes a
// contiguous range of items, so that a head's rows stay in one L2.
template <F32WaveMode MODE>
__device__ __forceinline__ bool f32_wave_item(int block, int heads, int tiles, int wave, int& bh, int& tile) {
  const int64_t n = static_cast<int64_t>(heads) * tiles;
  const int x = block % 8;
  const int64_t item = x * n / 8 + (MODE == kF32OwnTiles ? block / 8 * 4 + wave : block / 8);
  if (item >= (x + 1) * n / 8) return false;
  bh = static_cast<int>(item / tiles);
  tile = static_cast<int>(item % tiles);
  return true;
}
inline int64_t f32_wave_grid(int64_t heads, int64_t tiles, bool own_tiles) {
  const int64_t per_xcd = (heads * tiles + 7) / 8;
  return 8 * (own_tiles ? (per_xcd + 3) / 4 : per_xcd);
}

// Adds up the waves' partial results, wave w's scaled by f[w] of the lane's row, and stores them times
// `scale`: wave w takes register group w of every block.  `lds` may hold anything; 4 * NB * 4096 bytes.
template <int DP>
__device__ __forceinline__ void f32_wave_merge(char* lds, const f32x16 (&acc)[F32Wave<DP>::NB], const float (&f)[4],
                                               float* row, bool row_ok, float scale, int D, int wave, int lane) {
  constexpr int NB = F32Wave<DP>::NB;
  float4* x = reinterpret_cast<float4*>(lds);  // [wave][block][group][lane]
  __syncthreads();
#pragma unroll
  for (int db = 0; db < NB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      x[((wave * NB + db) * 4 + g) * 64 + lane] =
          make_float4(acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]);
  __syncthreads();
#pragma unroll
  for (int db = 0; db < NB; ++db) {
    float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float4 v = x[((w * NB + db) * 4 + wave) * 64 + lane];
      t.x = fmaf(v.x, f[w], t.x); t.y = fmaf(v.y, f[w], t.y); t.z = fmaf(v.z, f[w], t.z); t.w = fmaf(v.w, f[w], t.w);
    }
    const int d = db * 32 + wave * 8 + (lane / 32) * 4;
    if (row_ok && d < D)  // D is a multiple of 4
      *reinterpret_cast<float4*>(row + d) = make_float4(t.x * scale, t.y * scale, t.z * scale, t.w * scale);
  }
}

// The lane's row gets its share of a result, times f (see f32_attn_store).
template <int DP>
__device__ __forceinline__ void f32_wave_store(float* row, const f32x16 (&acc)[F32Wave<DP>::NB], float f, int half, int D) {
#pragma unroll
  for (int db = 0; db < F32Wave<DP>::NB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d = db * 32 + g * 8 + half * 4;
      if (d < D && d < DP)
        *reinterpret_cast<float4*>(row + d) =
            make_float4(acc[db][g * 4] * f, acc[db][g * 4 + 1] * f, acc[db][g * 4 + 2] * f, acc[db][g * 4 + 3] * f);
    }
}

// A resident row's values of the wave, every second chunk, times f; zeros past D and past the sequence.
template <int DP>
__device__ __forceinline__ void f32_wave_resident(const float* row, bool row_ok, int col0, int half, int D, float f,
                                                  float (&v)[DP / 2]) {
#pragma unroll
  for (int c = 0; c < DP / 8; ++c) {
    const int d = col0 + (2 * c + half) * 4;
    const float4 w = row_ok && d < D ? *reinterpret_cast<const float4*>(row + d) : make_float4(0.f, 0.f, 0.f, 0.f);
    v[c * 4] = w.x * f;
    v[c * 4 + 1] = w.y * f;
    v[c * 4 + 2] = w.z * f;
    v[c * 4 + 3] = w.w * f;
  }
}

// Forward.  The scores of the next step's keys are multiplied while this step's weights are formed: only one wave is on a
// SIMD, so what stands between two products without one of its own is time in which the matrix pipe is idle.
template <int DP, F32WaveMode MODE, bool CAUSAL, bool HAS_BIAS>
__global__ __launch_bounds__(256, (f32_wave_occupancy<DP, MODE, HAS_BIAS>(1))) void attn_fwd_f32_wave_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ mask,
    float* __restrict__ o, float* __restrict__ lse, AttnDims a, float scale, int tiles) {
  using W = F32Wave<DP>;
  constexpr int NI = W::NI, NM = HAS_BIAS ? 16 : 0;
  __shared__ __attribute__((aligned(1024))) char lds[f32_wave_lds<DP, MODE, HAS_BIAS>(1)];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // (known to be one value per wave)
  const int lane = threadIdx.x % kWave, half = lane / 32;
  int bh, tile;
  if (!f32_wave_item<MODE>(blockIdx.x, a.B * a.H, tiles, wave, bh, tile)) return;  // (waves with tiles of their own never meet)
  const int b = bh / a.H, h = bh % a.H;
  const int r0 = (CAUSAL ? tiles - 1 - tile : tile) * 32;  // longest walks first
  constexpr bool DSPLIT = MODE == kF32SplitColumns;
  const int col0 = DSPLIT ? wave * DP : 0;
  const bool columns = !DSPLIT || col0 < a.D;
  const int i = r0 + lane % 32, ic = min(i, a.S - 1);
  const bool row_ok = i < a.S;
  char* k_s = lds + wave * f32_wave_bytes<DP, HAS_BIAS>();
  char* v_s = k_s + W::TILE;
  char* m_s = v_s + W::TILE;
  char* xch = lds + 4 * f32_wave_bytes<DP, HAS_BIAS>();

  const int steps = (CAUSAL ? min(a.S, r0 + 32) + 31 : a.S + 31) / 32;
  const int stride = MODE == kF32SplitRows ? 4 : 1, first = MODE == kF32SplitRows ? wave : 0;
  F32WaveTiles<DP> kt;
  const int width = columns ? a.D - col0 : 4;  // (a wave without columns copies some and multiplies zeros)
  const int64_t head = qkv_at(a, b, 0, h) + (columns ? col0 : 0);
  kt.init(k + head, a.ld, a.S, min(width, DP), lane);
  const int64_t to_v = (v + head) - kt.base;
  auto copy_k = [&](int t) { kt.copy(min(t, steps - 1) * 32, k_s, lane); };
  auto copy_v = [&](int t) {
    F32WaveTiles<DP> vt = kt;
    vt.base += to_v;
    vt.copy(min(t, steps - 1) * 32, v_s, lane);
  };
  const float* mhead = HAS_BIAS ? mask + static_cast<int64_t>(bh) * a.S * a.S : nullptr;
  F32WaveBias mt_copies;
  if constexpr (HAS_BIAS) mt_copies.init(a.S, lane);
  auto copy_m = [&](int t) {
    if constexpr (HAS_BIAS) mt_copies.copy(mhead, r0, min(t, steps - 1) * 32, a.S, m_s, lane);
  };
  float qr[DP / 2];
  f32_wave_resident<DP>(q + qkv_at(a, b, ic, h), row_ok && columns, col0, half, a.D, scale * kAttnLog2e, qr);
  copy_k(first);
  copy_m(first);
  copy_v(first);
#pragma unroll
  for (int c = 0; c < DP / 2; ++c) asm volatile("" : "+v"(qr[c]));  // their wait stands here

  f32x16 acc[W::NB];
#pragma unroll
  for (int db = 0; db < W::NB; ++db) acc[db] = f32x16_zero();
  float m = -INFINITY, l = 0.f;  // l: this lane's half of the row's sum
  // Copies are requested in the order bias, K of the next step, V (past the end the last tile again, so that
  // the counts below hold), except ahead of the first step, where V is there before K.
  f32x16 s[1];
  auto scores = [&](int t) {
    s[0] = f32_wave_scores<DP>(k_s, qr, lane);
    if constexpr (DSPLIT) f32_wave_exchange<1>(xch + (t & 1) * 4 * 4096, wave, lane, s);
  };
  auto step = [&](int t, auto more) {
    float bias[16];
    if constexpr (HAS_BIAS) {
      MG_F32_WAVE_WAIT(2 * NI);
      const float* mt = reinterpret_cast<const float*>(m_s);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 w = *reinterpret_cast<const float4*>(mt + F32Wave<32>::place(lane % 32, 2 * g + half, 0));
        bias[4 * g] = w.x; bias[4 * g + 1] = w.y; bias[4 * g + 2] = w.z; bias[4 * g + 3] = w.w;
      }
      MG_F32_WAVE_WAIT(2 * NI);  // (the tile is read)
      copy_m(t + stride);
    }
    const int j0 = t * 32;
    f32x16 x, p;
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = HAS_BIAS ? fmaf(bias[r], kAttnLog2e, s[0][r]) : s[0][r];
    if (j0 + 32 > a.S || (CAUSAL && j0 + 31 > r0)) {  // the end of the sequence, the diagonal
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int j = j0 + f32_acc_row(r, half);
        x[r] = j < a.S && (!CAUSAL || j <= i) ? x[r] : -INFINITY;
      }
    }
    float m_tile = x[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) m_tile = fmaxf(m_tile, x[r]);
    m_tile = fmaxf(m_tile, __shfl_xor(m_tile, 32));
    // The reference point moves only when a score passes it by more than 2^8 (the weights stay exact:
    // the sum and the result are relative to the same point).
    if (__any(m_tile > m + 8.0f)) {
      const float m_new = fmaxf(m, m_tile);
      const float corr = m_new == -INFINITY ? 0.f : exp2f(m - m_new);
      l *= corr;
#pragma unroll
      for (int db = 0; db < W::NB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] *= corr;
      m = m_new;
    }
    const float base = m == -INFINITY ? 0.f : m;  // (nothing visible to this row yet: its weights are zero)
    if constexpr (decltype(more)::value) {
      if (t == first) MG_F32_WAVE_WAIT(NM);
      else MG_F32_WAVE_WAIT(NI + NM);
      scores(t + stride);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      x[r] -= base;
      p[r] = __builtin_amdgcn_exp2f(x[r]);
    }
    f32_wave_exp2_amend(x, p);
#pragma unroll
    for (int r = 0; r < 16; ++r) l += p[r];
    if constexpr (decltype(more)::value) {
      MG_F32_WAVE_WAIT(NI + NM);
      copy_k(t + 2 * stride);
      MG_F32_WAVE_WAIT(NI + NM);
    } else {
      MG_F32_WAVE_WAIT(NM);
    }
    f32_wave_weighted<DP>(v_s, p, lane, acc);
    MG_F32_WAVE_WAIT(NI + NM);
    if constexpr (decltype(more)::value) copy_v(t + stride);
  };
  if (first < steps) {
    MG_F32_WAVE_WAIT(NI + NM);
    scores(first);
    MG_F32_WAVE_WAIT(NI + NM);
    copy_k(first + stride);
    int t = first;
    for (; t + stride < steps; t += stride) step(t, std::true_type{});
    if (t == first) MG_F32_WAVE_WAIT(0);
    step(t, std::false_type{});
  }
  MG_F32_WAVE_WAIT(0);
  float l_row = l + __shfl_xor(l, 32);
  float* orow = o + o_at(a, b, h, ic);
  float* lrow = lse + static_cast<int64_t>(bh) * a.S + i;
  if constexpr (MODE != kF32SplitRows) {
    if (!row_ok || !columns) return;
    f32_wave_store<DP>(orow + col0, acc, 1.0f / l_row, half, a.D - col0);
    if (col0 == 0 && half == 0) *lrow = m * kAttnLn2 + logf(l_row);
  } else {
    float(*ml)[4][32] = reinterpret_cast<float(*)[4][32]>(lds);  // [max, sum][wave][row]
    __syncthreads();  // every wave is done with its tiles
    if (half == 0) {
      ml[0][wave][lane] = m;
      ml[1][wave][lane] = l_row;
    }
    __syncthreads();
    float f[4];
    m = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) m = fmaxf(m, ml[0][w][lane % 32]);
    l_row = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = ml[0][w][lane % 32];
      f[w] = mw == -INFINITY ? 0.f : exp2f(mw - m);
      l_row += f[w] * ml[1][w][lane % 32];
    }
    f32_wave_merge<DP>(lds, acc, f, orow, row_ok, 1.0f / l_row, a.D, wave, lane);
    if (row_ok && wave == 0 && half == 0) *lrow = m * kAttnLn2 + logf(l_row);
  }
}

// dQ, and where `delta` is not null the rows' delta.  `lds` holds f32_wave_lds<DP, MODE, HAS_BIAS>(2) bytes.
template <int DP, F32WaveMode MODE, bool CAUSAL, bool HAS_BIAS>
__device__ __forceinline__ void attn_dq_f32_wave_block(
    int block, char* lds, const float* __restrict__ d_o, const float* __restrict__ o, const float* __restrict__ q,
    const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ mask, const float* __restrict__ lse,
    float* __restrict__ delta, float* __restrict__ dq, const AttnDims& a, float scale, int tiles) {
  using W = F32Wave<DP>;
  constexpr int NI = W::NI, NM = HAS_BIAS ? 16 : 0;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // (known to be one value per wave)
  const int lane = threadIdx.x % kWave, half = lane / 32;
  int bh, tile;
  if (!f32_wave_item<MODE>(block, a.B * a.H, tiles, wave, bh, tile)) return;  // (waves with tiles of their own never meet)
  const int b = bh / a.H, h = bh % a.H;
  const int r0 = (CAUSAL ? tiles - 1 - tile : tile) * 32;
  constexpr bool DSPLIT = MODE == kF32SplitColumns;
  const int col0 = DSPLIT ? wave * DP : 0;
  const bool columns = !DSPLIT || col0 < a.D;
  const int i = r0 + lane % 32, ic = min(i, a.S - 1);
  const bool row_ok = i < a.S;
  char* k_s = lds + wave * f32_wave_bytes<DP, HAS_BIAS>();
  char* v_s = k_s + W::TILE;
  char* m_s = v_s + W::TILE;
  char* xch = lds + 4 * f32_wave_bytes<DP, HAS_BIAS>();

  const int steps = (CAUSAL ? min(a.S, r0 + 32) + 31 : a.S + 31) / 32;
  const int stride = MODE == kF32SplitRows ? 4 : 1, first = MODE == kF32SplitRows ? wave : 0;
  F32WaveTiles<DP> kt;
  const int width = columns ? a.D - col0 : 4;
  const int64_t head = qkv_at(a, b, 0, h) + (columns ? col0 : 0);
  kt.init(k + head, a.ld, a.S, min(width, DP), lane);
  const int64_t to_v = (v + head) - kt.base;
  auto copy_k = [&](int t) { kt.copy(min(t, steps - 1) * 32, k_s, lane); };
  auto copy_v = [&](int t) {
    F32WaveTiles<DP> vt = kt;
    vt.base += to_v;
    vt.copy(min(t, steps - 1) * 32, v_s, lane);
  };
  const float* mhead = HAS_BIAS ? mask + static_cast<int64_t>(bh) * a.S * a.S : nullptr;
  F32WaveBias mt_copies;
  if constexpr (HAS_BIAS) mt_copies.init(a.S, lane);
  auto copy_m = [&](int t) {
    if constexpr (HAS_BIAS) mt_copies.copy(mhead, r0, min(t, steps - 1) * 32, a.S, m_s, lane);
  };
  float qr[DP / 2], dor[DP / 2], orow[DP / 2];
  f32_wave_resident<DP>(d_o + o_at(a, b, h, ic), row_ok && columns, col0, half, a.D, 1.0f, dor);
  f32_wave_resident<DP>(o + o_at(a, b, h, ic), row_ok && columns, col0, half, a.D, 1.0f, orow);
  f32_wave_resident<DP>(q + qkv_at(a, b, ic, h), row_ok && columns, col0, half, a.D, scale * kAttnLog2e, qr);
  float lse2 = row_ok ? lse[static_cast<int64_t>(bh) * a.S + i] * kAttnLog2e : INFINITY;
  copy_v(first);
  copy_m(first);
  copy_k(first);
  float dl = 0.f;
#pragma unroll
  for (int c = 0; c < DP / 2; ++c) dl = fmaf(dor[c], orow[c], dl);
  dl += __shfl_xor(dl, 32);
  if constexpr (DSPLIT) {
    float* part = reinterpret_cast<float*>(xch);
    if (half == 0) part[wave * 32 + lane] = dl;
    __syncthreads();
    dl = (part[lane % 32] + part[32 + lane % 32]) + (part[64 + lane % 32] + part[96 + lane % 32]);
    __syncthreads();
  }
  if (delta != nullptr && row_ok && (MODE == kF32OwnTiles || wave == 0) && half == 0) delta[static_cast<int64_t>(bh) * a.S + i] = dl;
#pragma unroll
  for (int c = 0; c < DP / 2; ++c) asm volatile("" : "+v"(qr[c]), "+v"(dor[c]));  // their wait stands here
  asm volatile("" : "+v"(lse2));

  f32x16 acc[W::NB];
#pragma unroll
  for (int db = 0; db < W::NB; ++db) acc[db] = f32x16_zero();
  auto read_bias = [&](float (&bias)[16]) {
    if constexpr (HAS_BIAS) {
      const float* mt = reinterpret_cast<const float*>(m_s);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 w = *reinterpret_cast<const float4*>(mt + F32Wave<32>::place(lane % 32, 2 * g + half, 0));
        bias[4 * g] = w.x; bias[4 * g + 1] = w.y; bias[4 * g + 2] = w.z; bias[4 * g + 3] = w.w;
      }
    }
  };
  auto exponents = [&](int t, const f32x16& s, const float (&bias)[16]) {
    f32x16 x;
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = (HAS_BIAS ? fmaf(bias[r], kAttnLog2e, s[r]) : s[r]) - lse2;
    if (t * 32 + 32 > a.S || (CAUSAL && t * 32 + 31 > r0)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int j = t * 32 + f32_acc_row(r, half);
        x[r] = j < a.S && (!CAUSAL || j <= i) ? x[r] : -INFINITY;
      }
    }
    return x;
  };
  for (int t = first; t < steps; t += stride) {
    f32x16 s[2], p;
    float bias[16];
    // dP first: the K tile, in use to the end of a step, is copied meanwhile.
    MG_F32_WAVE_WAIT(NI + NM);
    s[1] = f32_wave_scores<DP>(v_s, dor, lane);
    MG_F32_WAVE_WAIT(NI + NM);
    copy_v(t + stride);
    MG_F32_WAVE_WAIT(NI);
    s[0] = f32_wave_scores<DP>(k_s, qr, lane);
    if constexpr (DSPLIT) f32_wave_exchange<2>(xch + (t & 1) * 8 * 4096, wave, lane, s);
    read_bias(bias);
    if constexpr (HAS_BIAS) {
      MG_F32_WAVE_WAIT(NI);
      copy_m(t + stride);
    }
    p = exponents(t, s[0], bias);
    f32_wave_exp2(p);
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] *= s[1][r] - dl;
    f32_wave_weighted<DP>(k_s, p, lane, acc);
    MG_F32_WAVE_WAIT(NI + NM);
    copy_k(t + stride);
  }
  MG_F32_WAVE_WAIT(0);
  float* row = dq + qkv_at(a, b, ic, h);
  if constexpr (MODE != kF32SplitRows) {
    if (row_ok && columns) f32_wave_store<DP>(row + col0, acc, scale, half, a.D - col0);
  } else {
    const float f[4] = {1.f, 1.f, 1.f, 1.f};
    f32_wave_merge<DP>(lds, acc, f, row, row_ok, scale, a.D, wave, lane);
  }
}

// dK, dV: the workgroup's keys along the lanes, the streamed queries along the registers.  delta = rowsum(dO * O) of the
// streamed rows is formed here as in dQ, from the dO tile that the products with V read anyway and O's rows in registers, so
// that neither walk waits for the other (at 128 columns those registers are taken: `delta` has it, from a launch of its own).
template <int DP, F32WaveMode MODE, bool CAUSAL, bool HAS_BIAS, bool GIVEN>
__device__ __forceinline__ void attn_dkdv_f32_wave_block(
    int block, char* lds, float (*stats)[4][64], const float* __restrict__ d_o, const float* __restrict__ o,
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ mask,
    const float* __restrict__ lse, const float* __restrict__ delta, float* __restrict__ dk, float* __restrict__ dv,
    const AttnDims& a, float scale, int tiles) {
  using W = F32Wave<DP>;
  constexpr int NI = W::NI, NM = HAS_BIAS ? 16 : 0;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // (known to be one value per wave)
  const int lane = threadIdx.x % kWave, half = lane / 32;
  int bh, tile;
  if (!f32_wave_item<MODE>(block, a.B * a.H, tiles, wave, bh, tile)) return;  // (waves with tiles of their own never meet)
  const int b = bh / a.H, h = bh % a.H;
  const int r0 = tile * 32;  // causal: the first keys have the longest walks
  constexpr bool DSPLIT = MODE == kF32SplitColumns;
  const int col0 = DSPLIT ? wave * DP : 0;
  const bool columns = !DSPLIT || col0 < a.D;
  const int j = r0 + lane % 32, jc = min(j, a.S - 1);
  const bool row_ok = j < a.S;
  char* q_s = lds + wave * f32_wave_bytes<DP, HAS_BIAS>();
  char* do_s = q_s + W::TILE;
  char* m_s = do_s + W::TILE;
  char* xch = lds + 4 * f32_wave_bytes<DP, HAS_BIAS>();

  const int steps = (a.S + 31) / 32;
  const int stride = MODE == kF32SplitRows ? 4 : 1, first = (CAUSAL ? tile : 0) + (MODE == kF32SplitRows ? wave : 0);
  F32WaveTiles<DP> qt, dt;
  const int width = min(columns ? a.D - col0 : 4, DP);
  qt.init(q + qkv_at(a, b, 0, h) + (columns ? col0 : 0), a.ld, a.S, width, lane);
  dt.init(d_o + o_at(a, b, h, 0) + (columns ? col0 : 0), o_ld(a), a.S, width, lane);
  const float* lse_h = lse + static_cast<int64_t>(bh) * a.S;
  const float* o_h = o + o_at(a, b, h, 0) + (columns ? col0 : 0);
  auto copy_q = [&](int t) { qt.copy(min(t, steps - 1) * 32, q_s, lane); };
  auto copy_d = [&](int t) { dt.copy(min(t, steps - 1) * 32, do_s, lane); };
  const float* mhead = HAS_BIAS ? mask + static_cast<int64_t>(bh) * a.S * a.S : nullptr;
  F32WaveBias mt_copies;
  if constexpr (HAS_BIAS) mt_copies.init(a.S, lane);
  auto copy_m = [&](int t) {
    if constexpr (HAS_BIAS) mt_copies.copy(mhead, min(t, steps - 1) * 32, r0, a.S, m_s, lane);
  };
  // O's row (or its delta) and the LSE of streamed row lane % 32, requested a step ahead.
  const float* delta_h = delta + static_cast<int64_t>(bh) * a.S;
  float4 orow[DP / 8];
  float lse_i, dl_i;
  auto load_o = [&](int t) {
    const int i = min(min(t, steps - 1) * 32 + lane % 32, a.S - 1);
    if constexpr (GIVEN) {
      dl_i = delta_h[i];
    } else {
      const float* row = o_h + i * o_ld(a);
#pragma unroll
      for (int c = 0; c < DP / 8; ++c) orow[c] = *reinterpret_cast<const float4*>(row + min((2 * c + half) * 4, width - 4));
    }
    lse_i = lse_h[i];
  };
  float kr[DP / 2], vr[DP / 2];
  f32_wave_resident<DP>(k + qkv_at(a, b, jc, h), row_ok && columns, col0, half, a.D, scale * kAttnLog2e, kr);
  f32_wave_resident<DP>(v + qkv_at(a, b, jc, h), row_ok && columns, col0, half, a.D, 1.0f, vr);
  load_o(first);
  copy_q(first);
  copy_d(first);
  copy_m(first);
#pragma unroll
  for (int c = 0; c < DP / 2; ++c) asm volatile("" : "+v"(kr[c]), "+v"(vr[c]));  // their wait stands here

  f32x16 acck[W::NB], accv[W::NB];
#pragma unroll
  for (int db = 0; db < W::NB; ++db) acck[db] = accv[db] = f32x16_zero();
  // The Q tile is read first and let go of first, so that the weights are formed beside the products of dO with V and
  // either tile's next copy has other products to arrive under.
  for (int t = first; t < steps; t += stride) {
    MG_F32_WAVE_WAIT(NI + NM);
    f32x16 s[2];
    s[0] = f32_wave_scores<DP>(q_s, kr, lane);
    MG_F32_WAVE_WAIT(0);
    float* const st = stats[DSPLIT ? t & 1 : 0][wave];  // [LSE][delta] of the tile's rows (both halves of the wave write)
    const int i0 = t * 32;
    float dl;
    auto weights = [&]() {
      st[lane % 32] = lse_i;
      float lv[16], bias[16];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float4 l4 = *reinterpret_cast<const float4*>(st + g * 8 + half * 4);
        lv[4 * g] = l4.x; lv[4 * g + 1] = l4.y; lv[4 * g + 2] = l4.z; lv[4 * g + 3] = l4.w;
      }
      if constexpr (HAS_BIAS) {
        const float* mt = reinterpret_cast<const float*>(m_s);
#pragma unroll
        for (int r = 0; r < 16; ++r) bias[r] = mt[F32Wave<32>::place(f32_acc_row(r, half), (lane % 32) / 4, 0) + lane % 4];
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float sv = fmaf(-lv[r], kAttnLog2e, s[0][r]);
        if (HAS_BIAS) sv = fmaf(bias[r], kAttnLog2e, sv);
        const int i = i0 + f32_acc_row(r, half);
        s[0][r] = i < a.S && (!CAUSAL || j <= i) ? exp2f(sv) : 0.f;
      }
    };
    if constexpr (!DSPLIT) weights();
    s[1] = f32_wave_scores_dot<DP, !GIVEN>(do_s, vr, orow, width, lane, dl);
    if constexpr (GIVEN) {
      dl = dl_i;
    } else {
      if constexpr (DSPLIT) dl = columns ? dl : 0.f;
      dl += __shfl_xor(dl, 32);
    }
    st[32 + lane % 32] = dl;
    if constexpr (DSPLIT) {
      f32_wave_exchange<2>(xch + (t & 1) * 8 * 4096, wave, lane, s);
      weights();
    }
    load_o(t + stride);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int rr = g * 8 + half * 4;
      float4 d4 = *reinterpret_cast<const float4*>(st + 32 + rr);
      if constexpr (DSPLIT && !GIVEN) {  // each wave has its columns' share
        float4 w4[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) w4[w] = *reinterpret_cast<const float4*>(stats[t & 1][w] + 32 + rr);
        d4 = make_float4((w4[0].x + w4[1].x) + (w4[2].x + w4[3].x), (w4[0].y + w4[1].y) + (w4[2].y + w4[3].y),
                         (w4[0].z + w4[1].z) + (w4[2].z + w4[3].z), (w4[0].w + w4[1].w) + (w4[2].w + w4[3].w));
      }
      const float dv4[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) s[1][g * 4 + e] = s[0][g * 4 + e] * (s[1][g * 4 + e] - dv4[e]);
    }
    f32_wave_weighted<DP>(q_s, s[1], lane, acck);
    MG_F32_WAVE_WAIT(0);
    copy_q(t + stride);
    f32_wave_weighted<DP>(do_s, s[0], lane, accv);
    MG_F32_WAVE_WAIT(NI);
    copy_d(t + stride);
    copy_m(t + stride);
  }
  MG_F32_WAVE_WAIT(0);
  float* krow = dk + qkv_at(a, b, jc, h);
  float* vrow = dv + qkv_at(a, b, jc, h);
  if constexpr (MODE != kF32SplitRows) {
    if (!row_ok || !columns) return;
    f32_wave_store<DP>(krow + col0, acck, scale, half, a.D - col0);
    f32_wave_store<DP>(vrow + col0, accv, 1.0f, half, a.D - col0);
  } else {
    const float f[4] = {1.f, 1.f, 1.f, 1.f};
    f32_wave_merge<DP>(lds, acck, f, krow, row_ok, scale, a.D, wave, lane);
    f32_wave_merge<DP>(lds, accv, f, vrow, row_ok, 1.0f, a.D, wave, lane);
  }
}

// Both walks in one launch: workgroups [0, blocks) take dK and dV, whose steps are the longer ones, the rest dQ.
template <int DP, F32WaveMode MODE, bool CAUSAL, bool HAS_BIAS>
__global__ __launch_bounds__(256, (f32_wave_occupancy<DP, MODE, HAS_BIAS>(2))) void attn_bwd_f32_wave_kernel(
    const float* __restrict__ d_o, const float* __restrict__ o, const float* __restrict__ q, const float* __restrict__ k,
    const float* __restrict__ v, const float* __restrict__ mask, const float* __restrict__ lse, const float* __restrict__ delta,
    float* __restrict__ dq, float* __restrict__ dk, float* __restrict__ dv, AttnDims a, float scale, int tiles, int blocks) {
  __shared__ __attribute__((aligned(1024))) char lds[f32_wave_lds<DP, MODE, HAS_BIAS>(2)];
  __shared__ __attribute__((aligned(256))) float stats[MODE == kF32SplitColumns ? 2 : 1][4][64];
  if (static_cast<int>(blockIdx.x) < blocks)
    attn_dkdv_f32_wave_block<DP, MODE, CAUSAL, HAS_BIAS, f32_wave_delta_given<DP>()>(blockIdx.x, lds, stats, d_o, o, q, k, v, mask, lse, delta, dk, dv, a, scale, tiles);
  else
    attn_dq_f32_wave_block<DP, MODE, CAUSAL, HAS_BIAS>(blockIdx.x - blocks, lds, d_o, o, q, k, v, mask, lse, nullptr, dq, a, scale, tiles);
}

// A launch for each walk: dQ, which leaves delta behind, and then dK and dV.
template <int DP, F32WaveMode MODE, bool CAUSAL, bool HAS_BIAS>
__global__ __launch_bounds__(256, (f32_wave_occupancy<DP, MODE, HAS_BIAS>(1))) void attn_dq_f32_wave_kernel(
    const float* __restrict__ d_o, const float* __restrict__ o, const float* __restrict__ q, const float* __restrict__ k,
    const float* __restrict__ v, const float* __restrict__ mask, const float* __restrict__ lse, float* __restrict__ delta,
    float* __restrict__ dq, AttnDims a, float scale, int tiles) {
  __shared__ __attribute__((aligned(1024))) char lds[f32_wave_lds<DP, MODE, HAS_BIAS>(2)];
  attn_dq_f32_wave_block<DP, MODE, CAUSAL, HAS_BIAS>(blockIdx.x, lds, d_o, o, q, k, v, mask, lse, delta, dq, a, scale, tiles);
}
template <int DP, F32WaveMode MODE, bool CAUSAL, bool HAS_BIAS>
__global__ __launch_bounds__(256, (f32_wave_occupancy<DP, MODE, HAS_BIAS>(2))) void attn_dkdv_f32_wave_kernel(
    const float* __restrict__ d_o, const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ mask, const float* __restrict__ lse, const float* __restrict__ delta, float* __restrict__ dk,
    float* __restrict__ dv, AttnDims a, float scale, int tiles) {
  __shared__ __attribute__((aligned(1024))) char lds[f32_wave_lds<DP, MODE, HAS_BIAS>(2)];
  __shared__ __attribute__((aligned(256))) float stats[MODE == kF32SplitColumns ? 2 : 1][4][64];
  attn_dkdv_f32_wave_block<DP, MODE, CAUSAL, HAS_BIAS, true>(blockIdx.x, lds, stats, d_o, nullptr, q, k, v, mask, lse, delta, dk, dv, a,
                                                             scale, tiles);
}

}  // namespace mg
