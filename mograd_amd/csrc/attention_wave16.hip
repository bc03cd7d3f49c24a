// Flash attention of 16-bit tensors whose 128-row workgroups would leave most of the device idle (head dim <= 128): a workgroup
// owns 32 rows of one head (queries in the forward and dQ, keys in dK/dV) and its four waves share the walk over the
// streamed rows, tile w, w + 4, ... of 32 to wave w; the four partial results meet in LDS at the end.
//
// What bounds few heads is not a rate but the walk of one workgroup: at (3, 1755, 2 heads, 64), causal, 84 workgroups of 128
// queries walk up to 28 blocks of 64 keys one after the other, and the backward walks behind a launch of its own
// that forms delta.  Here four times the workgroups walk a quarter as far each, no barrier stands in the walk (a wave's tiles are
// copied into LDS of its own and waited for with its own counter), and both backward walks are one launch: dK/dV forms delta =
// rowsum(dO * O) of its streamed rows from the dO fragments it multiplies anyway.  The price is that no wave's copy serves
// another, four times the bytes from L2, so larger grids keep the kernels of attention_mfma.hip.
//
// Products, operands and rounding are theirs (S^T = K Q^T, the score tile of a product is the operand of the next), except that
// the scale is applied to the fp32 scores and not to a rounded operand.
#include "attention_16bit_tiles.h"
#include "mg_internal.h"

namespace mg {

constexpr int kAttnWaveSlots = 2;  // tiles of a streamed tensor: the one in use and the next

template <int DP>
constexpr int attn_wave_tile() { return 32 * tile_row_bytes<DP>(); }
template <int DP>
constexpr int attn_wave_lds() { return 4 * kAttnWaveSlots * 2 * attn_wave_tile<DP>(); }

__device__ __forceinline__ void attn_wave_copy16(const char* base, unsigned bytes, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(bytes), "s"(base) : "memory");
}
// The same for the lanes of `mask` alone (a lane's bytes go to its own place, whichever lanes copy).  Every lane is here.
__device__ __forceinline__ void attn_wave_copy16_of(uint64_t mask, const char* base, unsigned bytes, unsigned dst) {
  asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1" ::"s"(dst), "v"(bytes),
               "s"(base), "s"(mask)
               : "memory");
}
// All of the wave's copies, loads and LDS reads are done.
__device__ __forceinline__ void attn_wave_settle() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070);
  asm volatile("" ::: "memory");
}

// A tensor whose 32-row tiles a wave copies: the image of TileLane16, chunks past D copies of the row's first one (what they
// give meets zeros or is not stored), rows past S zeros (their weights are zero, but a last row's copies with an
// infinity, an overflowed gradient's, would make NaN of it).  KEPT: chunks past D are left as they are in LDS, zeros (clear_tiles).
// K's are, in the forward and in dQ: a key whose first chunk is -inf has no weight, but products of the query's zeros with that
// chunk would be NaN.  The wave's next attn_wave_settle waits for all of these.
template <int DP, bool KEPT = false>
struct WaveTiles16 {
  static constexpr int CH = DP / 8, ROWS = 64 / CH, NI = 32 / ROWS;  // chunks of a row, rows and copies per tile
  const char* base;
  unsigned pitch;
  int S, D;
  unsigned off[NI];
  uint64_t own[NI];  // the lanes whose chunk is one of the row's
  __device__ __forceinline__ void init(const void* base_, int64_t ld, int S_, int D_, int lane) {
    base = static_cast<const char*>(base_);
    pitch = static_cast<unsigned>(ld) * 2;
    S = S_;
    D = D_;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int row = i * ROWS + lane / CH, c = (lane % CH) ^ tile_swz16<DP>(row);
      own[i] = __ballot(c * 8 < D);
      off[i] = row * pitch + (c * 8 < D ? c * 16 : 0);
    }
  }
  __device__ __forceinline__ void copy(int row0, char* tile, int lane) const {
    const unsigned dst = __builtin_amdgcn_readfirstlane(lds_address(tile));
    const char* p = base + static_cast<int64_t>(row0) * pitch;
    if (row0 + 32 <= S) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if constexpr (KEPT) attn_wave_copy16_of(own[i], p, off[i], dst + i * 1024);
        else attn_wave_copy16(p, off[i], dst + i * 1024);
      }
      return;
    }
    // a copy is ROWS rows, CH lanes to a row
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int lanes = (S - row0 - i * ROWS) * CH;
      if (lanes > 0) {
        const uint64_t rows = lanes >= 64 ? ~uint64_t{0} : (uint64_t{1} << lanes) - 1;
        attn_wave_copy16_of(KEPT ? rows & own[i] : rows, p, off[i], dst + i * 1024);
      }
      if (lane >= lanes) *reinterpret_cast<uint4*>(tile + i * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
    }
  }
  // Zeros for chunks D / 8 .. DC / 8 - 1 of the tile at `tile` and of the other slot's.  (Clearing whole tiles was 7 % of a backward
  // of 13 us.)
  template <int DC>
  __device__ __forceinline__ void clear_tiles(char* tile, int lane) const {
    for (int c = D / 8; c < DC / 8; ++c)
      *reinterpret_cast<uint4*>(tile + lane / 32 * 2 * attn_wave_tile<DP>() + tile16_chunk_at<DP>(lane % 32, c)) = make_uint4(0, 0, 0, 0);
  }
};

// Block id -> (head, 32-row tile): an XCD (id mod 8) takes a contiguous range of items, so that a head's rows stay in one L2.
__device__ __forceinline__ bool attn_wave_item(int block, int heads, int tiles, int& bh, int& tile) {
  const int64_t n = static_cast<int64_t>(heads) * tiles;
  const int x = block % 8;
  const int64_t item = x * n / 8 + block / 8;
  if (item >= (x + 1) * n / 8) return false;
  bh = static_cast<int>(item / tiles);
  tile = static_cast<int>(item % tiles);
  return true;
}
static int attn_wave_blocks(int64_t heads, int64_t tiles) { return static_cast<int>(8 * ((heads * tiles + 7) / 8)); }

// Adds up the waves' partial results, wave w's times f[w], and stores them times `scale`: a lane takes eight columns of its
// row, 16 bytes, and its other half the next eight.  `lds` may hold anything; DT * 16 KB.
template <typename T, int DT>
__device__ __forceinline__ void attn_wave_merge(char* lds, const floatx16 (&acc)[DT], const float (&f)[4], T* row, bool row_ok,
                                                float scale, int D, int wave, int lane) {
  float4* x = reinterpret_cast<float4*>(lds);  // [wave][block][group][lane]
  __syncthreads();
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      x[((wave * DT + dt) * 4 + g) * 64 + lane] = make_float4(acc[dt][4 * g], acc[dt][4 * g + 1], acc[dt][4 * g + 2], acc[dt][4 * g + 3]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < (DT + 1) / 2; ++i) {
    const int g = 8 * i + 2 * wave + lane / 32;
    if (DT % 2 == 1 && i == DT / 2 && wave >= 2) break;  // past the last tile
    uint32_t out[4];
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float4 v = x[(w * DT * 4 + g) * 64 + part * 32 + lane % 32];
        t.x = fmaf(v.x, f[w], t.x); t.y = fmaf(v.y, f[w], t.y); t.z = fmaf(v.z, f[w], t.z); t.w = fmaf(v.w, f[w], t.w);
      }
      out[2 * part] = Mma<T>::pack2(t.x * scale, t.y * scale);
      out[2 * part + 1] = Mma<T>::pack2(t.z * scale, t.w * scale);
    }
    if (row_ok && g * 8 < D) *reinterpret_cast<uint4*>(row + g * 8) = make_uint4(out[0], out[1], out[2], out[3]);
  }
}

// sum of a[e] * b[e] over eight packed elements, added to `dot`.
template <typename T>
__device__ __forceinline__ float attn_wave_dot8(const uint4& a, const uint4& b, float dot) {
  const uint32_t x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float2_t u = Mma<T>::unpack2(x[i]), v = Mma<T>::unpack2(y[i]);
    dot = fmaf(u[0], v[0], dot);
    dot = fmaf(u[1], v[1], dot);
  }
  return dot;
}

// CUT: D is less than the DC columns that are multiplied.  The masked copies and the cleared chunks cost such heads up to 3 % of the
// forward ((1, 8, 500, 80) 9.2 us | 9.3; (1, 8, 1000, 40), bias, 12.7 | 13.0) and nothing of the backward; in one form for all they
// cost those that fill DC as much ((1, 6, 1200, 96), bias, 19.2 | 19.8).
template <typename T, int DP, int DC, bool CAUSAL, bool HAS_BIAS, bool CUT>
__global__ __launch_bounds__(kAttnThreads, DP <= 64 ? 2 : 1) void attn_fwd_wave_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, const T* __restrict__ mask, T* __restrict__ o,
    float* __restrict__ lse, AttnDims a, float scale, int tiles) {
  constexpr int KS = DC / 16, DT = DC / 32, TILE = attn_wave_tile<DP>();
  __shared__ __attribute__((aligned(1024))) char lds[attn_wave_lds<DP>()];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x % kWave, half = lane / 32;
  int bh, tile;
  if (!attn_wave_item(blockIdx.x, a.B * a.H, tiles, bh, tile)) return;
  const int b = bh / a.H, h = bh % a.H;
  const int r0 = (CAUSAL ? tiles - 1 - tile : tile) * 32;  // longest walks first
  const int m = r0 + lane % 32, mc = min(m, a.S - 1);
  const bool row_ok = m < a.S;
  char* const own = lds + wave * kAttnWaveSlots * 2 * TILE;  // [slot][K, V]
  const int steps = (CAUSAL ? min(a.S, r0 + 32) + 31 : a.S + 31) / 32;

  uint4 qf[KS];
  request_row(q + qkv_at(a, b, mc, h), half, a.D, qf);
  WaveTiles16<DP, CUT> kt;
  WaveTiles16<DP> vt;
  kt.init(k + qkv_at(a, b, 0, h), a.ld, a.S, a.D, lane);
  if constexpr (CUT) kt.template clear_tiles<DC>(own, lane);
  vt.init(v + qkv_at(a, b, 0, h), a.ld, a.S, a.D, lane);
  const T* mrow = HAS_BIAS ? mask + (static_cast<int64_t>(bh) * a.S + mc) * a.S : nullptr;
  uint2 bias_next[4];
  auto request = [&](int t, int slot) {
    if constexpr (HAS_BIAS) {
      const bool packed = t * 32 + 32 <= a.S;
#pragma unroll
      for (int g = 0; g < 4; ++g) bias_next[g] = bias_group<T>(mrow, t * 32 + g * 8 + half * 4, a.S, packed);
    }
    kt.copy(t * 32, own + slot * 2 * TILE, lane);
    vt.copy(t * 32, own + slot * 2 * TILE + TILE, lane);
  };
  if (wave < steps) request(wave, 0);
  clear_row(row_ok, half, a.D, qf);
  const TileLane16<DP> at(lane);
  const float c = scale * kAttnLog2e;
  floatx16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16();
  float m_run = -INFINITY, l_run = 0.f;  // l_run: this lane's half of the row's sum
  int slot = 0;
  for (int t = wave; t < steps; t += 4, slot ^= 1) {
    attn_wave_settle();
    uint2 bias_w[4];
    if constexpr (HAS_BIAS) {
#pragma unroll
      for (int g = 0; g < 4; ++g) bias_w[g] = bias_next[g];
    }
    if (t + 4 < steps) request(t + 4, slot ^ 1);
    const char* k_s = own + slot * 2 * TILE;
    const char* v_s = k_s + TILE;
    floatx16 s = zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s = Mma<T>::run(frag_rows<DP>(k_s, at, 0, ks), qf[ks], s);
    uint4 tv[2][DT];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) tv[hf][dt] = frag_transposed<DP>(v_s, at, dt, hf);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] *= c;
      if constexpr (HAS_BIAS) s[r] = fmaf(bias_at<T>(bias_w[r / 4], r % 4), kAttnLog2e, s[r]);
    }
    if (t * 32 + 32 > a.S || (CAUSAL && t * 32 + 31 > r0)) {  // the end of the sequence, the diagonal
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = t * 32 + acc_row(r, lane);
        s[r] = n < a.S && (!CAUSAL || n <= m) ? s[r] : -INFINITY;
      }
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = max_halves(mx);
    // (Each wave's largest weight is exactly one, before its rounding as after it: a reference point that moves only now and
    // then, as in the fp32 kernels, costs O 6 % in error.)
    if (__any(mx > m_run)) {
      const float m_new = fmaxf(m_run, mx);
      const float corr = m_new == -INFINITY ? 0.f : fexp2(m_run - m_new);
      l_run *= corr;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] *= corr;
      m_run = m_new;
    }
    const float base = m_run == -INFINITY ? 0.f : m_run;  // (nothing visible to this row yet: its weights are zero)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fexp2(s[r] - base);
      l_run += s[r];
    }
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const uint4 pf = frag_from_acc<T>(s, hf);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) acc[dt] = Mma<T>::run(tv[hf][dt], pf, acc[dt]);
    }
  }
  float l_row = sum_halves(l_run);
  T* orow = o + o_at(a, b, h, mc);
  float* lrow = lse + static_cast<int64_t>(bh) * a.S + m;
  if (steps == 1) {
    if (wave != 0) return;
    store_tile<T>(o + o_at(a, b, h, r0), o_ld(a), a.S - r0, acc, 1.0f / l_row, a.D);
    if (row_ok && half == 0) *lrow = m_run * kAttnLn2 + logf(l_row);
    return;
  }
  float(*ml)[4][32] = reinterpret_cast<float(*)[4][32]>(lds);  // [max, sum][wave][row]
  __syncthreads();  // every wave is done with its tiles
  if (half == 0) {
    ml[0][wave][lane] = m_run;
    ml[1][wave][lane] = l_row;
  }
  __syncthreads();
  float f[4];
  float m_row = -INFINITY;
#pragma unroll
  for (int w = 0; w < 4; ++w) m_row = fmaxf(m_row, ml[0][w][lane % 32]);
  l_row = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float mw = ml[0][w][lane % 32];
    f[w] = mw == -INFINITY ? 0.f : fexp2(mw - m_row);
    l_row += f[w] * ml[1][w][lane % 32];
  }
  attn_wave_merge<T, DT>(lds, acc, f, orow, row_ok, 1.0f / l_row, a.D, wave, lane);
  if (row_ok && wave == 0 && half == 0) *lrow = m_row * kAttnLn2 + logf(l_row);
}

// dQ of block `block`; `lds` holds attn_wave_lds<DP>() bytes.
template <typename T, int DP, int DC, bool CAUSAL, bool HAS_BIAS, bool CUT>
__device__ __forceinline__ void attn_dq_wave_block(int block, char* lds, const T* __restrict__ d_o, const T* __restrict__ o,
                                                   const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
                                                   const T* __restrict__ mask, const float* __restrict__ lse,
                                                   T* __restrict__ dq, const AttnDims& a, float scale, int tiles) {
  constexpr int KS = DC / 16, DT = DC / 32, TILE = attn_wave_tile<DP>();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x % kWave, half = lane / 32;
  int bh, tile;
  if (!attn_wave_item(block, a.B * a.H, tiles, bh, tile)) return;
  const int b = bh / a.H, h = bh % a.H;
  const int r0 = (CAUSAL ? tiles - 1 - tile : tile) * 32;
  const int m = r0 + lane % 32, mc = min(m, a.S - 1);
  const bool row_ok = m < a.S;
  char* const own = lds + wave * kAttnWaveSlots * 2 * TILE;  // [slot][K, V]
  const int steps = (CAUSAL ? min(a.S, r0 + 32) + 31 : a.S + 31) / 32;

  uint4 qf[KS], dof[KS], of[KS];
  request_row(d_o + o_at(a, b, h, mc), half, a.D, dof);
  request_row(o + o_at(a, b, h, mc), half, a.D, of);
  request_row(q + qkv_at(a, b, mc, h), half, a.D, qf);
  float lse2 = lse[static_cast<int64_t>(bh) * a.S + mc] * kAttnLog2e;
  WaveTiles16<DP, CUT> kt;
  WaveTiles16<DP> vt;
  kt.init(k + qkv_at(a, b, 0, h), a.ld, a.S, a.D, lane);
  vt.init(v + qkv_at(a, b, 0, h), a.ld, a.S, a.D, lane);
  if constexpr (CUT) kt.template clear_tiles<DC>(own, lane);
  const T* mrow = HAS_BIAS ? mask + (static_cast<int64_t>(bh) * a.S + mc) * a.S : nullptr;
  uint2 bias_next[4];
  auto request = [&](int t, int slot) {
    if constexpr (HAS_BIAS) {
      const bool packed = t * 32 + 32 <= a.S;
#pragma unroll
      for (int g = 0; g < 4; ++g) bias_next[g] = bias_group<T>(mrow, t * 32 + g * 8 + half * 4, a.S, packed);
    }
    kt.copy(t * 32, own + slot * 2 * TILE, lane);
    vt.copy(t * 32, own + slot * 2 * TILE + TILE, lane);
  };
  if (wave < steps) request(wave, 0);
  clear_row(row_ok, half, a.D, qf);
  clear_row(row_ok, half, a.D, dof);
  clear_row(row_ok, half, a.D, of);
  float dl = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) dl = attn_wave_dot8<T>(dof[ks], of[ks], dl);
  dl = sum_halves(dl);
  const TileLane16<DP> at(lane);
  const float c = scale * kAttnLog2e;
  floatx16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16();
  int slot = 0;
  for (int t = wave; t < steps; t += 4, slot ^= 1) {
    attn_wave_settle();
    uint2 bias_w[4];
    if constexpr (HAS_BIAS) {
#pragma unroll
      for (int g = 0; g < 4; ++g) bias_w[g] = bias_next[g];
    }
    if (t + 4 < steps) request(t + 4, slot ^ 1);
    const char* k_s = own + slot * 2 * TILE;
    const char* v_s = k_s + TILE;
    floatx16 s = zero16(), dp = zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s = Mma<T>::run(frag_rows<DP>(k_s, at, 0, ks), qf[ks], s);
      dp = Mma<T>::run(frag_rows<DP>(v_s, at, 0, ks), dof[ks], dp);
    }
    uint4 tk[2][DT];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) tk[hf][dt] = frag_transposed<DP>(k_s, at, dt, hf);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if constexpr (HAS_BIAS) s[r] = fmaf(s[r], c, fmaf(bias_at<T>(bias_w[r / 4], r % 4), kAttnLog2e, -lse2));
      else s[r] = fmaf(s[r], c, -lse2);
    }
    if (t * 32 + 32 > a.S || (CAUSAL && t * 32 + 31 > r0)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = t * 32 + acc_row(r, lane);
        s[r] = n < a.S && (!CAUSAL || n <= m) ? s[r] : -INFINITY;
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fexp2(s[r]) * (dp[r] - dl);
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const uint4 dsf = frag_from_acc<T>(s, hf);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) acc[dt] = Mma<T>::run(tk[hf][dt], dsf, acc[dt]);
    }
  }
  T* row = dq + qkv_at(a, b, mc, h);
  if (steps == 1) {
    if (wave == 0) store_tile<T>(dq + qkv_at(a, b, r0, h), a.ld, a.S - r0, acc, scale, a.D);
    return;
  }
  const float f[4] = {1.f, 1.f, 1.f, 1.f};
  attn_wave_merge<T, DT>(lds, acc, f, row, row_ok, scale, a.D, wave, lane);
}

// dK, dV: the workgroup's keys along the lanes, the streamed queries along the registers.
template <typename T, int DP, int DC, bool CAUSAL, bool HAS_BIAS>
__device__ __forceinline__ void attn_dkdv_wave_block(int block, char* lds, float (*stats)[64], const T* __restrict__ d_o,
                                                     const T* __restrict__ o, const T* __restrict__ q, const T* __restrict__ k,
                                                     const T* __restrict__ v, const T* __restrict__ mask,
                                                     const float* __restrict__ lse, T* __restrict__ dk, T* __restrict__ dv,
                                                     const AttnDims& a, float scale, int tiles) {
  constexpr int KS = DC / 16, DT = DC / 32, TILE = attn_wave_tile<DP>();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lane = threadIdx.x % kWave, half = lane / 32;
  int bh, tile;
  if (!attn_wave_item(block, a.B * a.H, tiles, bh, tile)) return;
  const int b = bh / a.H, h = bh % a.H;
  const int r0 = tile * 32;  // causal: the first keys have the longest walks
  const int n = r0 + lane % 32, nc = min(n, a.S - 1);
  const bool row_ok = n < a.S;
  char* const own = lds + wave * kAttnWaveSlots * 2 * TILE;  // [slot][Q, dO]
  const int steps = (a.S + 31) / 32, first = (CAUSAL ? tile : 0) + wave;

  uint4 kf[KS], vf[KS];
  request_row(k + qkv_at(a, b, nc, h), half, a.D, kf);
  request_row(v + qkv_at(a, b, nc, h), half, a.D, vf);
  WaveTiles16<DP> qt, dt_;
  qt.init(q + qkv_at(a, b, 0, h), a.ld, a.S, a.D, lane);
  dt_.init(d_o + o_at(a, b, h, 0), o_ld(a), a.S, a.D, lane);
  const T* o_h = o + o_at(a, b, h, 0);
  const float* lse_h = lse + static_cast<int64_t>(bh) * a.S;
  const T* mcol = HAS_BIAS ? mask + static_cast<int64_t>(bh) * a.S * a.S + nc : nullptr;
  uint4 o_next[KS];  // O's row and the LSE of streamed row lane % 32, and the bias of the lane's key
  float lse_next;
  T bias_next[16];
  auto request = [&](int t, int slot) {
    const int i = min(t * 32 + lane % 32, a.S - 1);
    request_row(o_h + i * o_ld(a), half, a.D, o_next);
    lse_next = lse_h[i];
    if constexpr (HAS_BIAS) {
#pragma unroll
      for (int r = 0; r < 16; ++r) bias_next[r] = mcol[static_cast<int64_t>(min(t * 32 + acc_row(r, lane), a.S - 1)) * a.S];
    }
    qt.copy(t * 32, own + slot * 2 * TILE, lane);
    dt_.copy(t * 32, own + slot * 2 * TILE + TILE, lane);
  };
  if (first < steps) request(first, 0);
  clear_row(row_ok, half, a.D, kf);
  clear_row(row_ok, half, a.D, vf);
  const TileLane16<DP> at(lane);
  const float c = scale * kAttnLog2e;
  floatx16 acc_k[DT], acc_v[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc_k[dt] = acc_v[dt] = zero16();
  float* const st = stats[wave];  // [-LSE in log2 units][delta] of the tile's rows
  int slot = 0;
  for (int t = first; t < steps; t += 4, slot ^= 1) {
    attn_wave_settle();
    const char* q_s = own + slot * 2 * TILE;
    const char* do_s = q_s + TILE;
    uint4 dor[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) dor[ks] = frag_rows<DP>(do_s, at, 0, ks);
    float dl = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float d = attn_wave_dot8<T>(dor[ks], o_next[ks], dl);
      dl = ks * 16 + half * 8 < a.D ? d : dl;
    }
    st[lane % 32] = -lse_next * kAttnLog2e;  // (both halves of the wave write the same)
    dl = sum_halves(dl);
    st[32 + lane % 32] = t * 32 + lane % 32 < a.S ? dl : 0.f;
    T bias_v[16];
    if constexpr (HAS_BIAS) {
#pragma unroll
      for (int r = 0; r < 16; ++r) bias_v[r] = bias_next[r];
    }
    if (t + 4 < steps) request(t + 4, slot ^ 1);
    floatx16 s = zero16(), dp = zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s = Mma<T>::run(frag_rows<DP>(q_s, at, 0, ks), kf[ks], s);
      dp = Mma<T>::run(dor[ks], vf[ks], dp);
    }
    uint4 tq[2][DT], tdo[2][DT];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        tdo[hf][dt] = frag_transposed<DP>(do_s, at, dt, hf);
        tq[hf][dt] = frag_transposed<DP>(q_s, at, dt, hf);
      }
    float nl[16], dr[16];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 l4 = *reinterpret_cast<const float4*>(st + g * 8 + half * 4);
      const float4 d4 = *reinterpret_cast<const float4*>(st + 32 + g * 8 + half * 4);
      nl[4 * g] = l4.x; nl[4 * g + 1] = l4.y; nl[4 * g + 2] = l4.z; nl[4 * g + 3] = l4.w;
      dr[4 * g] = d4.x; dr[4 * g + 1] = d4.y; dr[4 * g + 2] = d4.z; dr[4 * g + 3] = d4.w;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if constexpr (HAS_BIAS) s[r] = fmaf(s[r], c, fmaf(to_float(bias_v[r]), kAttnLog2e, nl[r]));
      else s[r] = fmaf(s[r], c, nl[r]);
    }
    if (t * 32 + 32 > a.S || r0 + 32 > a.S || (CAUSAL && t * 32 < r0 + 31)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = t * 32 + acc_row(r, lane);
        s[r] = i < a.S && row_ok && (!CAUSAL || n <= i) ? s[r] : -INFINITY;
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fexp2(s[r]);
      dp[r] = s[r] * (dp[r] - dr[r]);
    }
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      const uint4 pf = frag_from_acc<T>(s, hf);
      const uint4 dsf = frag_from_acc<T>(dp, hf);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        acc_v[dt] = Mma<T>::run(tdo[hf][dt], pf, acc_v[dt]);
        acc_k[dt] = Mma<T>::run(tq[hf][dt], dsf, acc_k[dt]);
      }
    }
  }
  T* krow = dk + qkv_at(a, b, nc, h);
  T* vrow = dv + qkv_at(a, b, nc, h);
  if (steps - (CAUSAL ? tile : 0) == 1) {
    if (wave != 0) return;
    const int64_t out = qkv_at(a, b, r0, h);
    store_tile<T>(dk + out, a.ld, a.S - r0, acc_k, scale, a.D);
    store_tile<T>(dv + out, a.ld, a.S - r0, acc_v, 1.0f, a.D);
    return;
  }
  const float f[4] = {1.f, 1.f, 1.f, 1.f};
  attn_wave_merge<T, DT>(lds, acc_k, f, krow, row_ok, scale, a.D, wave, lane);
  attn_wave_merge<T, DT>(lds, acc_v, f, vrow, row_ok, 1.0f, a.D, wave, lane);
}

// Both walks in one launch: workgroups [0, blocks) take dK and dV, whose steps are the longer ones, the rest dQ.
template <typename T, int DP, int DC, bool CAUSAL, bool HAS_BIAS, bool CUT>
__global__ __launch_bounds__(kAttnThreads, DP <= 64 && !(HAS_BIAS && DC > 32) ? 2 : 1) void attn_bwd_wave_kernel(
    const T* __restrict__ d_o, const T* __restrict__ o, const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
    const T* __restrict__ mask, const float* __restrict__ lse, T* __restrict__ dq, T* __restrict__ dk, T* __restrict__ dv,
    AttnDims a, float scale, int tiles, int blocks) {
  __shared__ __attribute__((aligned(1024))) char lds[attn_wave_lds<DP>()];
  __shared__ __attribute__((aligned(256))) float stats[4][64];
  if (static_cast<int>(blockIdx.x) < blocks)
    attn_dkdv_wave_block<T, DP, DC, CAUSAL, HAS_BIAS>(blockIdx.x, lds, stats, d_o, o, q, k, v, mask, lse, dk, dv, a, scale, tiles);
  else
    attn_dq_wave_block<T, DP, DC, CAUSAL, HAS_BIAS, CUT>(blockIdx.x - blocks, lds, d_o, o, q, k, v, mask, lse, dq, a, scale, tiles);
}

// f(T, DP, DC, CAUSAL, HAS_BIAS) with the constants that the call asks for.
template <typename F>
static void attn_wave_pick(int dtype, int D, bool causal, bool has_bias, F f) {
  auto modes = [&](auto t, auto dp, auto dc) {
    if (causal) f(t, dp, dc, std::true_type{}, std::false_type{});
    else if (has_bias) f(t, dp, dc, std::false_type{}, std::true_type{});
    else f(t, dp, dc, std::false_type{}, std::false_type{});
  };
  auto widths = [&](auto t) {
    const std::integral_constant<int, 64> narrow;
    const std::integral_constant<int, 128> wide;
    if (D <= 32) modes(t, narrow, std::integral_constant<int, 32>{});
    else if (D <= 64) modes(t, narrow, narrow);
    else if (D <= 96) modes(t, wide, std::integral_constant<int, 96>{});
    else modes(t, wide, wide);
  };
  if (dtype == MG_BF16) widths(bf16_t{});
  else widths(f16_t{});
}

int attn_fwd_wave16(const void* q, const void* k, const void* v, const void* mask, void* o, float* lse, const AttnDims& a,
                    float scale, bool causal, bool has_bias, int dtype, hipStream_t stream) {
  const int tiles = static_cast<int>(ceil_div(a.S, 32));
  const dim3 grid(static_cast<unsigned>(attn_wave_blocks(static_cast<int64_t>(a.B) * a.H, tiles)));
  attn_wave_pick(dtype, a.D, causal, has_bias, [&](auto t, auto dp, auto dc, auto cz, auto hb) {
    using T = decltype(t);
    auto launch = [&](auto cut) {
      hipLaunchKernelGGL((attn_fwd_wave_kernel<T, decltype(dp)::value, decltype(dc)::value, decltype(cz)::value, decltype(hb)::value, decltype(cut)::value>),
                         grid, dim3(kAttnThreads), 0, stream, static_cast<const T*>(q), static_cast<const T*>(k), static_cast<const T*>(v),
                         static_cast<const T*>(mask), static_cast<T*>(o), lse, a, scale, tiles);
    };
    if (a.D < decltype(dc)::value) launch(std::true_type{});
    else launch(std::false_type{});
  });
  MG_LAUNCH_CHECK();
  return MG_OK;
}

int attn_bwd_wave16(const void* d_o, const void* o, const void* q, const void* k, const void* v, const void* mask, const float* lse,
                    void* dq, void* dk, void* dv, const AttnDims& a, float scale, bool causal, bool has_bias, int dtype,
                    hipStream_t stream) {
  const int tiles = static_cast<int>(ceil_div(a.S, 32));
  const int blocks = attn_wave_blocks(static_cast<int64_t>(a.B) * a.H, tiles);
  attn_wave_pick(dtype, a.D, causal, has_bias, [&](auto t, auto dp, auto dc, auto cz, auto hb) {
    using T = decltype(t);
    auto launch = [&](auto cut) {
      hipLaunchKernelGGL((attn_bwd_wave_kernel<T, decltype(dp)::value, decltype(dc)::value, decltype(cz)::value, decltype(hb)::value, decltype(cut)::value>),
                         dim3(2 * static_cast<unsigned>(blocks)), dim3(kAttnThreads), 0, stream, static_cast<const T*>(d_o),
                         static_cast<const T*>(o), static_cast<const T*>(q), static_cast<const T*>(k), static_cast<const T*>(v),
                         static_cast<const T*>(mask), lse, static_cast<T*>(dq), static_cast<T*>(dk), static_cast<T*>(dv), a, scale,
                         tiles, blocks);
    };
    if (a.D < decltype(dc)::value) launch(std::true_type{});
    else launch(std::false_type{});
  });
  MG_LAUNCH_CHECK();
  return MG_OK;
}

}  // namespace mg
