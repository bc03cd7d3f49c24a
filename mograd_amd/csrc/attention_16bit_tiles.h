// What the 16-bit attention kernels share: the matrix instruction and its operands, resident rows, the LDS images of
// streamed tiles and their fragments, bias reads.
#pragma once

#include "attention_generic.h"

namespace mg {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

template <typename T>
struct Mma;
template <>
struct Mma<bf16_t> {
  static __device__ __forceinline__ floatx16 run(uint4 a, uint4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                   0, 0);
  }
  // Two fp32 -> packed pair, round to nearest even (one v_cvt_pk_bf16_f32).
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    const float2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
  }
  static __device__ __forceinline__ float2_t unpack2(uint32_t w) {
    return __builtin_convertvector(__builtin_bit_cast(bf16x2_t, w), float2_t);
  }
};
template <>
struct Mma<f16_t> {
  static __device__ __forceinline__ floatx16 run(uint4 a, uint4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0,
                                                  0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    const float2_t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
  }
  static __device__ __forceinline__ float2_t unpack2(uint32_t w) {
    return __builtin_convertvector(__builtin_bit_cast(f16x2_t, w), float2_t);
  }
};

// Eight packed elements times `f`, rounded back to T.  Used once per workgroup to fold the
// softmax scale (times log2 e) into the resident operand of the score product, so that the
// product comes out of the matrix core already in the exponent's units.
template <typename T>
__device__ __forceinline__ uint4 scale_frag(uint4 v, float f) {
  const uint32_t in[4] = {v.x, v.y, v.z, v.w};
  uint32_t out[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float2_t x = Mma<T>::unpack2(in[i]);
    out[i] = Mma<T>::pack2(x[0] * f, x[1] * f);
  }
  return make_uint4(out[0], out[1], out[2], out[3]);
}

// Makes a fragment loaded from global memory before a loop count as "arrived" at this
// point.  Without it the compiler's wait-count bookkeeping treats the load as possibly
// still in flight at the loop header and waits for *all* outstanding global loads at the
// fragment's first use inside the loop, which also drains the tile prefetch issued a few
// instructions earlier.
__device__ __forceinline__ void settle(uint4& v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)); }

// The fragments of a lane's resident row (`row`: one inside the sequence): requested without a condition, chunks past
// D as the row's first one, and cleared where they do not count.  A load under a condition is waited for at the
// end of its branch: rows of 64 columns of two operands were eight memory latencies one behind the other ahead
// of the walk, and the walk's own copies a ninth.  (8, 12 heads of 1024, 64), causal: backward 76.5 -> 71.5 us,
// forward 27.3 -> 26.9; (2, 12, 4096, 64): forward 126.5 -> 124.4; (17, 11, 52, 80), causal: forward + backward
// 25.6 -> 23.8.
template <typename T, int KS>
__device__ __forceinline__ void request_row(const T* row, int half, int D, uint4 (&f)[KS]) {
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d = ks * 16 + half * 8;
    f[ks] = *reinterpret_cast<const uint4*>(row + (d < D ? d : 0));
  }
}
__device__ __forceinline__ void keep_if(bool ok, uint4& v) {
  v.x = ok ? v.x : 0;
  v.y = ok ? v.y : 0;
  v.z = ok ? v.z : 0;
  v.w = ok ? v.w : 0;
}
template <int KS>
__device__ __forceinline__ void clear_row(bool row_ok, int half, int D, uint4 (&f)[KS]) {
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    settle(f[ks]);
    keep_if(row_ok && ks * 16 + half * 8 < D, f[ks]);
  }
}

__device__ __forceinline__ floatx16 splat16(float v) {
  floatx16 z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = v;
  return z;
}

constexpr int kAttnThreads = 256;
typedef short short4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float fexp2(float v) { return __builtin_amdgcn_exp2f(v); }

// ---- LDS tiles -------------------------------------------------------------------------
// A staged tile is R rows x DP columns of T, row-major, rows of DP * 2 bytes without padding.
// The 16-byte chunk c of row r is stored at chunk position c ^ swz(r) (low three bits), with
// swz(r) = 2 * (r % 4) + (r / 4) % 2.  The transposing 64-bit reads (16 lanes: four rows x 32
// bytes) and the staging stores are free of bank conflicts with it; the 128-bit row reads
// are served two rows per bank group (LDS has 64 banks and serves 16 lanes of a 128-bit
// read per clock; timed with four waves reading back to back: 32 clocks per read against
// 19 for consecutive addresses).  A swizzle over r % 16 that removes that too, 4 * (r/2 % 2)
// + (r/4 % 4), was measured in these kernels: 25 % fewer LDS-busy cycles, but the two
// transposing reads of a fragment then need separate address registers and adds, and the
// forward, which is bound by its VALU work, ran 3-5 % slower (backward within 1 %).  Storing
// tile row r in LDS row (r & ~15) | r3 | r0 << 1 | r1 << 2 | r2 << 3 instead keeps this swizzle,
// spreads the row reads over all banks and leaves the second transposing read at a constant
// distance; it measured the same as this layout to within 2 % either way (forward at
// S = 4096 4 % slower, D = 128 backward 2 % faster).  LDS conflicts are not what limits
// these kernels, so the plain row order stays.  One image serves the products that contract over the tile's columns and
// those that contract over its rows.
template <int DP>
constexpr int tile_row_bytes() { return DP * 2; }
__device__ __forceinline__ int tile_swz(int r) { return 2 * (r % 4) + (r / 4) % 2; }
template <int DP>
__device__ __forceinline__ int tile_chunk_at(int r, int c) { return r * tile_row_bytes<DP>() + ((c ^ tile_swz(r)) * 16); }

// Where a lane reads its fragments inside a staged tile, as byte offsets that depend on the
// lane only; everything else (which 32-row block, which 16 rows, which tile copy) is a
// compile-time or wave-uniform addend, so the fragment reads of a whole step share these few
// address registers.  That works because a row's swizzle depends only on r % 8, and the rows
// a lane reads differ from its first one by multiples of 8.
template <int DP>
struct TileLane {
  int rows[DP / 16];  // per 16-column slice ks: row lane%32, columns ks*16 + (lane/32)*8 .. +7
  int tr[DP / 32];    // per 32-column block dt: row 4*(lane/32) + (lane%16)/4, columns dt*32 + ((lane/16)%2)*16 + 4*(lane%4) .. +3
  __device__ __forceinline__ explicit TileLane(int lane) {
#pragma unroll
    for (int ks = 0; ks < DP / 16; ++ks) rows[ks] = tile_chunk_at<DP>(lane % 32, ks * 2 + lane / 32);
    const int col = ((lane / 16) % 2) * 16 + 4 * (lane % 4);
#pragma unroll
    for (int dt = 0; dt < DP / 32; ++dt)
      tr[dt] = tile_chunk_at<DP>(4 * (lane / 32) + (lane % 16) / 4, (dt * 32 + col) / 8) + (col % 8) * 2;
  }
};

// A operand for a product that contracts over the tile's columns: rows rt*32 + lane%32,
// columns ks*16 + (lane/32)*8 .. +7.
template <int DP>
__device__ __forceinline__ uint4 frag_rows(const char* __restrict__ lds, const TileLane<DP>& at, int rt, int ks) {
  return *reinterpret_cast<const uint4*>(lds + at.rows[ks] + rt * 32 * tile_row_bytes<DP>());
}

// A operand for a product that contracts over the tile's rows: MFMA row = tile column
// dt*32 + lane%32; k-slot e of lane half h stands for tile row t*16 + (e/4)*8 + 4h + e%4, the
// same assignment the score tile's registers have (see frag_from_acc).  Read with
// ds_read_b64_tr_b16: within 16 lanes, lane i supplies the address of four consecutive
// columns 4*(i%4).. of row i/4 of a 4 x 16 block and receives the four rows of column i.
template <int DP>
__device__ __forceinline__ uint4 frag_transposed(const char* __restrict__ lds, const TileLane<DP>& at, int dt, int t) {
  using lds_i16x4 = __attribute__((address_space(3))) short4_t;
  const char* p = lds + at.tr[dt] + t * 16 * tile_row_bytes<DP>();
  const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lds_i16x4*>(reinterpret_cast<uintptr_t>(p)));
  const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      reinterpret_cast<lds_i16x4*>(reinterpret_cast<uintptr_t>(p + 8 * tile_row_bytes<DP>())));
  const uint2 l = __builtin_bit_cast(uint2, lo), h = __builtin_bit_cast(uint2, hi);
  return make_uint4(l.x, l.y, h.x, h.y);
}

// B operand from a 32x32 accumulator tile: registers 8*half .. 8*half+7, i.e. rows
// half*16 + (e/4)*8 + 4*(lane/32) + e%4 of column lane%32.
template <typename T>
__device__ __forceinline__ uint4 frag_from_acc(const floatx16& acc, int half) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = Mma<T>::pack2(acc[half * 8 + 2 * i], acc[half * 8 + 2 * i + 1]);
  return make_uint4(w[0], w[1], w[2], w[3]);
}

// Row index inside a 32-row tile of accumulator register r.
__device__ __forceinline__ int acc_row(int r, int lane) { return (r / 4) * 8 + (lane / 32) * 4 + (r % 4); }

__device__ __forceinline__ floatx16 zero16() {
  floatx16 z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = 0.f;
  return z;
}

// The two lanes that share a query (lane and lane ^ 32) exchange a value with one
// v_permlane32_swap instead of a round trip through LDS (ds_bpermute): afterwards `lo` holds
// lanes 0..31 of v in both halves of the wave and `hi` lanes 32..63.  The no-ops cover the
// wait states between a VALU write of the operands, the swap, and a VALU read of the
// results, which the compiler cannot see inside the asm.
__device__ __forceinline__ void split_halves(float v, float& lo, float& hi) {
  lo = v;
  hi = v;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(lo), "+v"(hi));
}
__device__ __forceinline__ float max_halves(float v) {
  float lo, hi;
  split_halves(v, lo, hi);
  return fmaxf(lo, hi);
}
__device__ __forceinline__ float sum_halves(float v) {
  float lo, hi;
  split_halves(v, lo, hi);
  return lo + hi;
}

// Packed store of four consecutive accumulator registers (four consecutive d) times `f`.
template <typename T>
__device__ __forceinline__ void store4(T* dst, const floatx16& acc, int g, float f) {
  uint2 w;
  w.x = Mma<T>::pack2(acc[g * 4] * f, acc[g * 4 + 1] * f);
  w.y = Mma<T>::pack2(acc[g * 4 + 2] * f, acc[g * 4 + 3] * f);
  *reinterpret_cast<uint2*>(dst) = w;
}

// Stores accumulator tiles, 32 rows of DT x 32 columns, times `f`.  A lane holds a row's columns four by four: of every eight
// the lower or the upper four.  Stored as they lie, an instruction writes 16 bytes at a place, and the L2 takes
// that many requests; so the halves of the wave swap first, and a lane stores eight columns, an instruction 32 bytes of every row.
// B8 H16 S1024, causal: 64 columns, backward 97 -> 91 us; 128 columns, 258 -> 236, forward 54.7 -> 50.1; full backward 128 -> 125 and
// 326 -> 319; B64 H6 S256 D64, backward 37.4 -> 35.8, forward 15.1 -> 14.4.  (Quarters as well, 64 bytes of 16 rows: another 1.5 %
// at 64 columns of S1024, but B64 H6 S256 36.4, and 128 columns 236 -> 244 and 319 -> 355 for want of registers.)
// `tile`: its first row's first column; `rows` are left from there (any number), and `cols` columns, a multiple of 8.
// The whole wave comes here.
template <typename T, int DT>
__device__ __forceinline__ void store_tile(T* __restrict__ tile, int64_t ld, int rows, const floatx16 (&acc)[DT], float f, int cols) {
  int lane = __builtin_amdgcn_mbcnt_hi(-1, __builtin_amdgcn_mbcnt_lo(-1, 0));
  asm volatile("" : "+v"(lane));  // formed here: no address is held over the caller's walk
  const int row = lane % 32, half = lane / 32;
  T* const at = tile + row * ld;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = Mma<T>::pack2(acc[dt][g * 8 + 2 * i] * f, acc[dt][g * 8 + 2 * i + 1] * f);
      const auto x = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
      const int d = dt * 32 + g * 16 + half * 8;
      if (row < rows && d < cols) *reinterpret_cast<uint4*>(at + d) = make_uint4(x[0], y[0], x[1], y[1]);
    }
}

// Additive bias (B, H, S, S): in the forward and the dQ walk a lane keeps one query row and its
// accumulator registers run over keys in groups of four consecutive ones, so the bias of a
// group inside the row is one 8-byte load, at whatever even address it lies; the two lanes of a row then
// read whole 16-byte pieces and, over a step's eight groups, exactly the row's 128 bytes.
// (Element by element, 32 two-byte loads per lane and step, the forward ran at 0.7 TB/s of bias:
// 1.10 ms at B2 H12 S4096 against 0.17 ms without a bias; and with rows of 1061, which start on no
// 8-byte boundary, forward and backward took 279 us at B19 H2 D64 against 180.)
template <typename T>
__device__ __forceinline__ float bias_at(const uint2& w, int j) {
  T h[4];
  __builtin_memcpy(h, &w, 8);
  return to_float(h[j]);
}
typedef uint32_t bias_u2_any __attribute__((ext_vector_type(2), aligned(2)));
// row[n .. n + 3] as four packed 16-bit values; `packed`: one 8-byte load, else element by element
// with the index clamped to the row (the values past its end are never used).
template <typename T>
__device__ __forceinline__ uint2 bias_group(const T* __restrict__ row, int n, int S, bool packed) {
  static_assert(sizeof(T) == 2, "16-bit tensors");
  if (packed) {
    const bias_u2_any v = *reinterpret_cast<const bias_u2_any*>(row + n);
    return make_uint2(v[0], v[1]);
  }
  const uint16_t* raw = reinterpret_cast<const uint16_t*>(row);
  uint2 w;
  w.x = raw[min(n, S - 1)] | static_cast<uint32_t>(raw[min(n + 1, S - 1)]) << 16;
  w.y = raw[min(n + 2, S - 1)] | static_cast<uint32_t>(raw[min(n + 3, S - 1)]) << 16;
  return w;
}

// The LDS image of the pipelined walks: as above, but chunk c of row r sits at position
// c ^ swz16(r) with swz16(r) = 4 * (r/2 % 2) + (r/4 % 2) + 2 * (r/8 % 2).  The 128-bit row reads
// of sixteen consecutive rows then fall on sixteen different bank groups (the plain swizzle
// serves them two rows per group, which doubles the cycles of half of all fragment reads),
// and the transposing reads stay conflict-free.  The price is that rows r and r + 8 no longer
// swizzle alike, so the second transposing read of a fragment has an address register of its
// own.  The tiles are written by global_load_lds, a kilobyte (eight rows) per wave
// instruction, so the image costs nothing on the way in.
// Rows of 128 columns are a whole trip round the banks each: 4 * (r % 4) + (r/4 % 4) there, sixteen chunk positions
// for sixteen rows, and four groups of four chunks for the four rows of a transposing read.
template <int DP>
__device__ __forceinline__ int tile_swz16(int r) {
  return DP == 128 ? 4 * (r % 4) + (r / 4) % 4 : 4 * ((r / 2) % 2) + (r / 4) % 2 + 2 * ((r / 8) % 2);
}
template <int DP>
__device__ __forceinline__ int tile16_chunk_at(int r, int c) { return r * tile_row_bytes<DP>() + ((c ^ tile_swz16<DP>(r)) * 16); }
template <int DP>
struct TileLane16 {
  int rows[DP / 16];
  int tr_lo[DP / 32], tr_hi[DP / 32];
  __device__ __forceinline__ explicit TileLane16(int lane) {
#pragma unroll
    for (int ks = 0; ks < DP / 16; ++ks) rows[ks] = tile16_chunk_at<DP>(lane % 32, ks * 2 + lane / 32);
    const int col = ((lane / 16) % 2) * 16 + 4 * (lane % 4);
    const int r = 4 * (lane / 32) + (lane % 16) / 4;
#pragma unroll
    for (int dt = 0; dt < DP / 32; ++dt) {
      tr_lo[dt] = tile16_chunk_at<DP>(r, (dt * 32 + col) / 8) + (col % 8) * 2;
      tr_hi[dt] = tile16_chunk_at<DP>(r + 8, (dt * 32 + col) / 8) + (col % 8) * 2;
    }
  }
};
template <int DP>
__device__ __forceinline__ uint4 frag_rows(const char* __restrict__ lds, const TileLane16<DP>& at, int rt, int ks) {
  return *reinterpret_cast<const uint4*>(lds + at.rows[ks] + rt * 32 * tile_row_bytes<DP>());
}
template <int DP>
__device__ __forceinline__ uint4 frag_transposed(const char* __restrict__ lds, const TileLane16<DP>& at, int dt, int t) {
  using lds_i16x4 = __attribute__((address_space(3))) short4_t;
  const char* base = lds + t * 16 * tile_row_bytes<DP>();
  const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      reinterpret_cast<lds_i16x4*>(reinterpret_cast<uintptr_t>(base + at.tr_lo[dt])));
  const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      reinterpret_cast<lds_i16x4*>(reinterpret_cast<uintptr_t>(base + at.tr_hi[dt])));
  const uint2 l = __builtin_bit_cast(uint2, lo), h = __builtin_bit_cast(uint2, hi);
  return make_uint4(l.x, l.y, h.x, h.y);
}

// s_waitcnt with only the vector-memory counter set (vmcnt in bits 3:0 and 15:14, the
// other counters left at "no wait").
#define MG_ATTN_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | 0x0f70)

__device__ __forceinline__ unsigned lds_address(const void* p) {
  using lds_ptr = __attribute__((address_space(3))) const char*;
  return static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_ptr)p));
}
}  // namespace mg
