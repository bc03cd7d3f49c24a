// Softmax cross-entropy forward / gradient / fused for one storage type T.  Included by
// one translation unit per dtype, which instantiates `CrossEntropyOps<T>`.
//
// Layout in HBM: logits, dense labels and dlogits are row-major (N, C); integer labels
// are (N) int32 or int64; per-row losses are (N) fp32 scratch; loss is one element of T.
//
// Gradient and fused kernels hold a row of logits in registers (chunks of VEC elements dealt
// round-robin to the TPR threads that share the row), so the logits are read from HBM once
// and dlogits written once; rows of more than kMostChunks chunks are streamed twice, the first time
// with an online softmax.  The loss-only kernel streams the row once that way and keeps nothing.
#pragma once

#include <cfloat>
#include <cstdlib>

#include "mg_device.h"
#include "mg_internal.h"
#include "mg_rows.h"

namespace mg {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

__device__ __forceinline__ float fast_exp2(float v) { return __builtin_amdgcn_exp2f(v); }

// What is taken off a row's logits before anything else: its largest one where that overflows in log2 units (a row of classes
// that are all masked with the type's lowest value), or zero.  Such logits are the largest one or at least 2^103 below it.
__device__ __forceinline__ float row_base(float m) { return fabsf(m) <= FLT_MAX && fabsf(m) > FLT_MAX / kLog2e ? m : 0.f; }

// Rows that do not lie on 16-byte chunks (ANY below) are read and written in misaligned ones, with -inf past a row's end: it
// is no maximum and adds nothing to a sum of exponentials.
template <typename T>
constexpr uint32_t kMinusInfWord = sizeof(T) == 4 ? 0xff800000u : std::is_same<T, f16_t>::value ? 0xfc00fc00u : 0xff80ff80u;

template <int TPR, int WG, int K>
__device__ __forceinline__ void row_allreduce_max(float (&v)[K], float* slots, int& phase) {
  if constexpr (TPR == 16) {
    // four rows side by side in a wave, each on one row of 16 lanes
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = row16_allreduce<MaxOp>(v[k]);
  } else if constexpr (TPR == kWave) {
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = wave_max(v[k]);
  } else {
    static_assert(TPR == WG, "a row is shared by sixteen lanes, one wave or the whole workgroup");
    block_allreduce<MaxOp, WG / kWave, K>(v, slots, phase);
    phase ^= 1;
  }
}

__device__ __forceinline__ int64_t load_id(const void* ids, int64_t row, bool id64) {
  return id64 ? static_cast<const int64_t*>(ids)[row] : static_cast<int64_t>(static_cast<const int32_t*>(ids)[row]);
}

// ------------------------------------------------------------------------------------
// Gradient (and optionally loss) with the row resident in registers.
//   labels: dense rows of T when DENSE, else N integer ids (int64 when id64).
//   rowloss: per-row loss term -sum(label * log_softmax) / N, or nullptr to skip.
//   upstream: one element of T, or nullptr for 1.
// ------------------------------------------------------------------------------------

template <typename T, int VEC, int TPR, int VPT, int WG, bool DENSE, bool ANY>
__global__ __launch_bounds__(WG, (TPR == 256 && VPT * VEC > 128) ? 2 : 1) void ce_rows_kernel(
    const T* __restrict__ logits, const void* __restrict__ labels, const T* __restrict__ upstream,
    float* __restrict__ rowloss, T* __restrict__ dlogits, int64_t N, int C, int id64) {
  constexpr int RPW = WG / TPR;
  using Tile = RowTile<T, VEC, TPR, VPT, ANY>;
  __shared__ float slots[2 * (WG / kWave)];
  int t, sub;
  row_thread<TPR, WG>(t, sub);
  int phase = 0;
  const float inv_rows = 1.0f / static_cast<float>(N);
  const float scale = (upstream != nullptr ? to_float(upstream[0]) : 1.0f) * inv_rows;

  // One row per TPR threads and no row loop: a loop would let the compiler start the next
  // row's loads before this row's stores and double the register footprint.
  {
    const int64_t row = static_cast<int64_t>(blockIdx.x) * RPW + sub;
    if (row >= N) return;  // per 16-lane row, per wave or per workgroup (RPW == 1); no barrier follows for TPR <= 64
    const T* xr = logits + row * C;
    Tile x;
    x.load(xr, t, C, kMinusInfWord<T>);

    // Absent chunks hold zeros: mask them to -inf for the max and skip them in the sums.
    const int nfull = Tile::full_chunks(C);
    float m[1] = {-INFINITY};
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      if (i < nfull) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) m[0] = fmaxf(m[0], x.v[i][e]);
      } else if (i == nfull) {
        const bool valid = Tile::col(i, t) < C;
#pragma unroll
        for (int e = 0; e < VEC; ++e) m[0] = fmaxf(m[0], valid ? x.v[i][e] : -INFINITY);
      }
    }
    row_allreduce_max<TPR, WG, 1>(m, slots, phase);
    const float base = row_base(m[0]);
    if (__builtin_expect(base != 0.f, 0)) {
#pragma unroll
      for (int i = 0; i < VPT; ++i)
#pragma unroll
        for (int e = 0; e < VEC; ++e) x.v[i][e] -= base;
      m[0] = 0.f;
    }
    const float m2 = m[0] * kLog2e;
    T* out_row = dlogits + row * C;

    if constexpr (DENSE) {
      float s[1] = {0.f};
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        if (i < nfull) {
#pragma unroll
          for (int e = 0; e < VEC; ++e) s[0] += fast_exp2(fmaf(x.v[i][e], kLog2e, -m2));
        } else if (i == nfull) {
          const bool valid = Tile::col(i, t) < C;
#pragma unroll
          for (int e = 0; e < VEC; ++e) s[0] += valid ? fast_exp2(fmaf(x.v[i][e], kLog2e, -m2)) : 0.f;
        }
      }
      row_allreduce_sum<TPR, WG, 1>(s, slots, phase);
      // softmax = exp(x - lse), formed directly from the log-sum-exp so that the
      // exponentials of the previous pass need not stay live next to the logits.
      const float shift = m[0] + logf(s[0]);
      const float shift2 = shift * kLog2e;
      const T* yr = static_cast<const T*>(labels) + row * C;
      float acc[1] = {0.f};
      const unsigned lane_off = static_cast<unsigned>(t) * VEC;
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        if (i < nfull || (i == nfull && Tile::col(i, t) < C)) {
          float y[VEC], out[VEC];
          const int c = Tile::col(i, t);
          if (i < nfull) Tile::load_chunk(yr + i * (TPR * VEC) + lane_off, y);
          else Tile::load_end(yr + i * (TPR * VEC) + lane_off, c, C, y);
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            const float term = (x.v[i][e] - shift) * y[e];
            acc[0] += !ANY || i < nfull || Tile::in_row(c, e, C) ? term : 0.f;
            out[e] = (fast_exp2(fmaf(x.v[i][e], kLog2e, -shift2)) - y[e]) * scale;
          }
          if (i < nfull) Tile::store_chunk(out_row + i * (TPR * VEC) + lane_off, out);
          else Tile::store_end(out_row + i * (TPR * VEC) + lane_off, c, C, out);
        }
      }
      if (rowloss != nullptr) {
        row_allreduce_sum<TPR, WG, 1>(acc, slots, phase);
        if (t == 0) rowloss[row] = -acc[0] * inv_rows;
      }
    } else {
      // Integer labels: the exponentials replace the logits in registers, the gradient is
      // one multiply per element, and the single "- 1" at the label column is patched by
      // its owner thread with a scalar store issued after its vector stores (same thread,
      // same address: program order holds).
      float s[1] = {0.f};
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        if (i < nfull) {
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            x.v[i][e] = fast_exp2(fmaf(x.v[i][e], kLog2e, -m2));
            s[0] += x.v[i][e];
          }
        } else if (i == nfull) {
          const bool valid = Tile::col(i, t) < C;
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            x.v[i][e] = fast_exp2(fmaf(x.v[i][e], kLog2e, -m2));
            s[0] += valid ? x.v[i][e] : 0.f;
          }
        }
      }
      row_allreduce_sum<TPR, WG, 1>(s, slots, phase);
      const float k = scale / s[0];
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        if (i <= nfull) {
#pragma unroll
          for (int e = 0; e < VEC; ++e) x.v[i][e] *= k;
        }
      }
      x.store(out_row, t, C);
      const int64_t id = load_id(labels, row, id64 != 0);
      const bool id_ok = id >= 0 && id < C;
      const bool owner = id_ok && (static_cast<int>(id) / VEC) % TPR == t;
      if (owner) {
        const float xl = to_float(xr[id]) - base;
        const float lp = xl - m[0] - logf(s[0]);  // log softmax at the label
        out_row[id] = from_float<T>((fast_exp2(fmaf(xl, kLog2e, -m2)) / s[0] - 1.0f) * scale);
        if (rowloss != nullptr) rowloss[row] = -lp * inv_rows;
      }
      // An id outside [0, C) selects no column: the row's loss term is flagged NaN.
      if (rowloss != nullptr && !id_ok && t == 0) rowloss[row] = NAN;
    }
  }
}

// exp(x - m), as 2^(x log2(e) - m log2(e)), or where that overflows as 2^(x - m), the same for such logits (see row_base).
struct ExpReference {
  float by, top;
  __device__ __forceinline__ explicit ExpReference(float m) {
    const float m2 = m * kLog2e;
    const bool plain = fabsf(m2) <= FLT_MAX;
    by = plain ? kLog2e : 1.f;
    top = plain ? m2 : m;
  }
  __device__ __forceinline__ float weight(float x) const { return fast_exp2(fmaf(x, by, -top)); }
};

// Eight 16-bit values out of four registers, word by word: seen as an array of eight, fp16 values were held one to a
// register, and spilled ((8192, 50304) 610 us against 341).
template <typename T>
__device__ __forceinline__ void unpack_words(const uint4& r, float (&x)[8]) {
  const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (std::is_same<T, f16_t>::value) {
      typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
      const half2_t h = __builtin_bit_cast(half2_t, w[i]);
      x[2 * i] = static_cast<float>(h[0]);
      x[2 * i + 1] = static_cast<float>(h[1]);
    } else {
      x[2 * i] = __uint_as_float(w[i] << 16);
      x[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
}

// Integer labels, 16-bit logits, rows of thousands of columns: the row stays in
// registers as loaded (eight 16-bit values per 128-bit register quad) and is unpacked in each of
// its three passes (maximum, sum of exponentials, gradient), so a thread holds VPT * 4 registers
// for VPT * 8 columns instead of VPT * 8: 200 fp32 values per thread next to the 100 registers
// they were loaded into spill (656 bytes per lane at 50304 columns: 1.36 TB/s).  The second
// exponential per element is free in a kernel that waits for memory.  The arithmetic per element
// is that of ce_rows_kernel, so are the bits.  One row per workgroup.
template <typename T, int TPR, int VPT, bool ANY>
__global__ __launch_bounds__(TPR, TPR <= 256 ? (VPT > 16 ? 3 : 4) : (TPR <= 512 ? 2 : 1)) void ce_rows_packed_kernel(
    const T* __restrict__ logits, const void* __restrict__ labels, const T* __restrict__ upstream,
    float* __restrict__ rowloss, T* __restrict__ dlogits, int64_t N, int C, int id64) {
  static_assert(sizeof(T) == 2, "16-bit element types");
  constexpr int VEC = 8;
  __shared__ float slots[2 * (TPR / kWave)];
  const int t = threadIdx.x;
  int phase = 0;
  const float inv_rows = 1.0f / static_cast<float>(N);
  const float scale = (upstream != nullptr ? to_float(upstream[0]) : 1.0f) * inv_rows;
  const int64_t row = blockIdx.x;
  const T* xr = logits + row * C;
  T* out_row = dlogits + row * C;
  const int nfull = (C / VEC) / TPR;  // chunk indices below it exist for every thread
  const int last = (nfull * TPR + t) * VEC;  // the column of this thread's chunk `nfull`,
  const bool tail = last < C;                // if it exists
  // On 16-byte chunks it is one like the others; else it may end with the row, and has registers and code of its own, which
  // as a case of every one of VPT chunks took 25 more registers ((8192, 50257) bf16 391 us; in the aligned form the own
  // registers cost 1.5 %).
  auto here = [&](int i) { return i < nfull || (!ANY && i == nfull && tail); };

  using Tile = RowTile<T, VEC, TPR, VPT, ANY>;
  uint4 raw[VPT], end = make_uint4(0, 0, 0, 0);
  if (ANY && tail) {
    uint32_t w[4];
    VecAny<T, VEC>::words_end(xr + last, max(last + VEC - C, 0), kMinusInfWord<T>, w);
    end = make_uint4(w[0], w[1], w[2], w[3]);
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    raw[i] = make_uint4(0, 0, 0, 0);
    if (here(i)) {
      using Chunk = typename std::conditional<ANY, mg_u4_any, mg_u4>::type;
      const Chunk w = *reinterpret_cast<const Chunk*>(xr + (i * TPR + t) * VEC);
      raw[i] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  float m[1] = {-INFINITY};
  auto top = [&](const uint4& r) {
    float x[VEC];
    unpack_words<T>(r, x);
#pragma unroll
    for (int e = 0; e < VEC; ++e) m[0] = fmaxf(m[0], x[e]);
  };
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    if (here(i)) top(raw[i]);
  if (ANY && tail) top(end);
  row_allreduce_max<TPR, TPR, 1>(m, slots, phase);
  const ExpReference ref(m[0]);
  // Between the passes the packed registers are made opaque to the compiler, which would
  // otherwise keep the unpacked values of one pass for the next.
  auto forget = [&]() {
#pragma unroll
    for (int i = 0; i < VPT; ++i) asm volatile("" : "+v"(raw[i].x), "+v"(raw[i].y), "+v"(raw[i].z), "+v"(raw[i].w));
    if constexpr (ANY) asm volatile("" : "+v"(end.x), "+v"(end.y), "+v"(end.z), "+v"(end.w));
  };
  forget();
  float s[1] = {0.f};
  auto add = [&](const uint4& r) {
    float x[VEC];
    unpack_words<T>(r, x);
#pragma unroll
    for (int e = 0; e < VEC; ++e) s[0] += ref.weight(x[e]);
  };
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    if (here(i)) add(raw[i]);
  if (ANY && tail) add(end);
  row_allreduce_sum<TPR, TPR, 1>(s, slots, phase);
  const float k = scale / s[0];
  forget();
  auto gradient = [&](const uint4& r, float (&x)[VEC]) {
    unpack_words<T>(r, x);
#pragma unroll
    for (int e = 0; e < VEC; ++e) x[e] = ref.weight(x[e]) * k;
  };
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    if (here(i)) {
      float x[VEC];
      gradient(raw[i], x);
      Tile::store_chunk(out_row + (i * TPR + t) * VEC, x);
    }
  }
  if (ANY && tail) {
    float x[VEC];
    gradient(end, x);
    Tile::store_end(out_row + last, last, C, x);
  }
  // the "- 1" at the label column: a scalar store by the thread that owns the column, after its
  // vector stores (same thread, same address: program order holds)
  const int64_t id = load_id(labels, row, id64 != 0);
  const bool id_ok = id >= 0 && id < C;
  if (id_ok && (static_cast<int>(id) / VEC) % TPR == t) {
    const float xl = to_float(xr[id]);
    const float lp = xl - m[0] - logf(s[0]);  // log softmax at the label
    out_row[id] = from_float<T>((ref.weight(xl) / s[0] - 1.0f) * scale);
    if (rowloss != nullptr) rowloss[row] = -lp * inv_rows;
  }
  // An id outside [0, C) selects no column: the row's loss term is flagged NaN.
  if (rowloss != nullptr && !id_ok && t == 0) rowloss[row] = NAN;
}

// ------------------------------------------------------------------------------------
// Streaming kernels: any C.  One workgroup per row.  ANY: at any address, C >= VEC.
// ------------------------------------------------------------------------------------

// The chunk at column c < C of a row at any address, `fill` past the row's end.
template <typename T, int VEC>
__device__ __forceinline__ void stream_load(const T* row, int64_t c, int64_t C, uint32_t fill, float (&v)[VEC]) {
  uint32_t w[4];
  VecAny<T, VEC>::words_end(row + c, static_cast<int>(max(c + VEC - C, int64_t{0})), fill, w);
  VecAny<T, VEC>::unpack(w, v);
}

// What an online sum of exponentials subtracts, in log2 units: the maximum so far, but no less than the least float, so that
// classes masked with -inf or with the type's lowest value, where a thread has seen nothing else yet, add zeros (from minus
// infinity they would be NaN, which no later maximum takes out of the sum).
__device__ __forceinline__ float online_reference(float m) { return fmaxf(m * kLog2e, -FLT_MAX); }

// A thread's share of the sum of exponentials (and of label * x) of a row from its base (see row_base), once more and an element at
// a time.
template <typename T, int WG, bool DENSE>
__device__ __forceinline__ void rebased_sums(const T* xr, const T* yr, int64_t C, float base, float& sum, float& dot) {
  sum = dot = 0.f;
  for (int64_t c = threadIdx.x; c < C; c += WG) {
    const float x = to_float(xr[c]) - base;
    sum += fast_exp2(x * kLog2e);
    if constexpr (DENSE) dot += x * to_float(yr[c]);
  }
}

// Online (max, sum-exp) over the elements a thread visits, merged across the workgroup, the maximum less the row's base.  ONCE: the
// row is not read again by this kernel, so its loads go past the caches.
template <typename T, int VEC, int WG, bool ONCE = false, bool ANY = false>
__device__ __forceinline__ void stream_max_sum(const T* __restrict__ xr, int64_t C, float* slots, int& phase, float& m_out,
                                               float& s_out, float& base_out) {
  auto fetch = [](const T* p, float (&v)[VEC]) {
    if constexpr (ANY) VecAny<T, VEC>::load(p, v);
    else if constexpr (ONCE) VecIO<T, VEC>::load_stream(p, v);
    else VecIO<T, VEC>::load(p, v);
  };
  float m = -INFINITY, s = 0.f;
  constexpr int U = 4;  // chunks in flight per thread: the loop is bound by memory-level parallelism
  const int64_t step = static_cast<int64_t>(WG) * VEC;
  const int64_t whole = ANY ? C - C % VEC : C;  // where the last whole chunk ends
  int64_t c = static_cast<int64_t>(threadIdx.x) * VEC;
  for (; c + (U - 1) * step < whole; c += U * step) {
    float v[U][VEC];
#pragma unroll
    for (int u = 0; u < U; ++u) fetch(xr + c + u * step, v[u]);
    float cm = v[0][0];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < VEC; ++e) cm = fmaxf(cm, v[u][e]);
    if (cm > m) {
      s *= fast_exp2((m - cm) * kLog2e);  // exp2(-inf) == 0 on the first chunk
      m = cm;
    }
    const float m2 = online_reference(m);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < VEC; ++e) s += fast_exp2(fmaf(v[u][e], kLog2e, -m2));
  }
  for (; c < C; c += step) {
    float v[VEC];
    if constexpr (ANY) stream_load<T, VEC>(xr, c, C, kMinusInfWord<T>, v);
    else fetch(xr + c, v);
    float cm = v[0];
#pragma unroll
    for (int e = 1; e < VEC; ++e) cm = fmaxf(cm, v[e]);
    if (cm > m) {
      s *= fast_exp2((m - cm) * kLog2e);
      m = cm;
    }
    const float m2 = online_reference(m);
#pragma unroll
    for (int e = 0; e < VEC; ++e) s += fast_exp2(fmaf(v[e], kLog2e, -m2));
  }
  float mm[1] = {m};
  block_allreduce<MaxOp, WG / kWave, 1>(mm, slots, phase);
  phase ^= 1;
  // Threads that saw nothing have m == -inf and s == 0; (m - mm) would be nan only if the
  // whole row were empty, which C > 0 excludes.
  float ss[1] = {m == -INFINITY ? 0.f : s * fast_exp2((m - mm[0]) * kLog2e)};
  base_out = row_base(mm[0]);
  float no_dot;
  if (__builtin_expect(base_out != 0.f, 0)) rebased_sums<T, WG, false>(xr, nullptr, C, base_out, ss[0], no_dot);
  block_allreduce<SumOp, WG / kWave, 1>(ss, slots, phase);
  phase ^= 1;
  m_out = mm[0] - base_out;
  s_out = ss[0];
}

// Loss only.  Dense: sum(label * (x - lse)) = sum(label * x) - lse * sum(label), so one
// pass over logits and labels suffices.
// ONCE: the logits (and dense labels) are larger than the memory-side cache can hold, so they are
// read past the caches (1.65 GB of logits: 266 -> 238 us, 6.9 TB/s; smaller tensors may still be
// cached from the kernel that wrote them and keep the plain loads).
template <typename T, int VEC, int WG, bool DENSE, bool ONCE = false, bool ANY = false>
__global__ __launch_bounds__(WG) void ce_fwd_stream_kernel(const T* __restrict__ logits, const void* __restrict__ labels,
                                                           float* __restrict__ rowloss, int64_t N, int64_t C, int id64) {
  __shared__ float slots[2 * 2 * (WG / kWave)];
  int phase = 0;
  const int64_t row = blockIdx.x;
  if (row >= N) return;
  const T* xr = logits + row * C;
  float m, s, base;
  const float inv_rows = 1.0f / static_cast<float>(N);
  if constexpr (DENSE) {
    const T* yr = static_cast<const T*>(labels) + row * C;
    float dot[2] = {0.f, 0.f};  // sum(label * x), sum(label)
    float tm = -INFINITY, ts = 0.f;
    for (int64_t c = static_cast<int64_t>(threadIdx.x) * VEC; c < C; c += static_cast<int64_t>(WG) * VEC) {
      float v[VEC], y[VEC];
      if constexpr (ANY) {
        stream_load<T, VEC>(xr, c, C, kMinusInfWord<T>, v);
        stream_load<T, VEC>(yr, c, C, 0, y);
      } else if constexpr (ONCE) {
        VecIO<T, VEC>::load_stream(xr + c, v);
        VecIO<T, VEC>::load_stream(yr + c, y);
      } else {
        VecIO<T, VEC>::load(xr + c, v);
        VecIO<T, VEC>::load(yr + c, y);
      }
      float cm = v[0];
#pragma unroll
      for (int e = 1; e < VEC; ++e) cm = fmaxf(cm, v[e]);
      if (cm > tm) {
        ts *= fast_exp2((tm - cm) * kLog2e);
        tm = cm;
      }
      const float m2 = online_reference(tm);
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        ts += fast_exp2(fmaf(v[e], kLog2e, -m2));
        dot[0] += !ANY || c + e < C ? v[e] * y[e] : 0.f;
        dot[1] += y[e];
      }
    }
    float mm[1] = {tm};
    block_allreduce<MaxOp, WG / kWave, 1>(mm, slots, phase);
    phase ^= 1;
    float red[3] = {tm == -INFINITY ? 0.f : ts * fast_exp2((tm - mm[0]) * kLog2e), dot[0], dot[1]};
    base = row_base(mm[0]);
    if (__builtin_expect(base != 0.f, 0)) rebased_sums<T, WG, true>(xr, yr, C, base, red[0], red[1]);
    __shared__ float slots3[2 * 3 * (WG / kWave)];
    block_allreduce<SumOp, WG / kWave, 3>(red, slots3, 0);
    m = mm[0] - base;
    s = red[0];
    if (threadIdx.x == 0) rowloss[row] = -(red[1] - (m + logf(s)) * red[2]) * inv_rows;
  } else {
    stream_max_sum<T, VEC, WG, ONCE, ANY>(xr, C, slots, phase, m, s, base);
    if (threadIdx.x == 0) {
      const int64_t id = load_id(labels, row, id64 != 0);
      rowloss[row] = (id < 0 || id >= C) ? NAN : -((to_float(xr[id]) - base) - (m + logf(s))) * inv_rows;
    }
  }
}

// Gradient (and optionally loss) for rows too wide for registers: two passes.
template <typename T, int VEC, int WG, bool DENSE, bool ANY = false>
__global__ __launch_bounds__(WG) void ce_grad_stream_kernel(const T* __restrict__ logits, const void* __restrict__ labels,
                                                            const T* __restrict__ upstream, float* __restrict__ rowloss,
                                                            T* __restrict__ dlogits, int64_t N, int64_t C, int id64) {
  __shared__ float slots[2 * 2 * (WG / kWave)];
  int phase = 0;
  const int64_t row = blockIdx.x;
  if (row >= N) return;
  const T* xr = logits + row * C;
  T* out_row = dlogits + row * C;
  const float inv_rows = 1.0f / static_cast<float>(N);
  const float scale = (upstream != nullptr ? to_float(upstream[0]) : 1.0f) * inv_rows;
  float m, s, base;
  stream_max_sum<T, VEC, WG, false, ANY>(xr, C, slots, phase, m, s, base);
  const float m2 = m * kLog2e;
  const float inv_sum = 1.0f / s;
  const float shift = m + logf(s);
  const int64_t id = DENSE ? 0 : load_id(labels, row, id64 != 0);
  float acc[1] = {0.f};
  constexpr int U = DENSE ? 1 : 4;  // integer labels: four chunks in flight per thread
  const int64_t step = static_cast<int64_t>(WG) * VEC;
  const int64_t whole = ANY ? C - C % VEC : C;  // where the last whole chunk ends
  int64_t c0 = static_cast<int64_t>(threadIdx.x) * VEC;
  if (__builtin_expect(base != 0.f, 0)) {
    for (int64_t c = threadIdx.x; c < C; c += WG) {
      const float x = to_float(xr[c]) - base;
      const float y = DENSE ? to_float((static_cast<const T*>(labels) + row * C)[c]) : c == id ? 1.f : 0.f;
      if (y != 0.f) acc[0] += (x - shift) * y;
      out_row[c] = from_float<T>((fast_exp2(x * kLog2e) * inv_sum - y) * scale);
    }
    c0 = C;
  }
  auto put = [&](int64_t c, const float (&out)[VEC]) {
    if constexpr (!ANY) VecIO<T, VEC>::store(out_row + c, out);
    else if (c < whole) VecAny<T, VEC>::store(out_row + c, out);
    else VecAny<T, VEC>::store_first(out_row + c, static_cast<int>(C - c), out);
  };
  if constexpr (!DENSE) {
    for (; c0 + (U - 1) * step < whole; c0 += U * step) {
      float v[U][VEC];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if constexpr (ANY) VecAny<T, VEC>::load(xr + c0 + u * step, v[u]);
        else VecIO<T, VEC>::load(xr + c0 + u * step, v[u]);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t c = c0 + u * step;
        float out[VEC];
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
          float p = fast_exp2(fmaf(v[u][e], kLog2e, -m2)) * inv_sum;
          if (c + e == id) {
            p -= 1.0f;
            acc[0] += v[u][e] - shift;
          }
          out[e] = p * scale;
        }
        put(c, out);
      }
    }
  }
  for (int64_t c = c0; c < C; c += step) {
    float v[VEC], out[VEC];
    if constexpr (ANY) stream_load<T, VEC>(xr, c, C, kMinusInfWord<T>, v);
    else VecIO<T, VEC>::load(xr + c, v);
    if constexpr (DENSE) {
      const T* yr = static_cast<const T*>(labels) + row * C;
      float y[VEC];
      if constexpr (ANY) stream_load<T, VEC>(yr, c, C, 0, y);
      else VecIO<T, VEC>::load(yr + c, y);
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const float term = (v[e] - shift) * y[e];
        acc[0] += !ANY || c + e < C ? term : 0.f;
        out[e] = (fast_exp2(fmaf(v[e], kLog2e, -m2)) * inv_sum - y[e]) * scale;
      }
    } else {
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        float p = fast_exp2(fmaf(v[e], kLog2e, -m2)) * inv_sum;
        if (c + e == id) {
          p -= 1.0f;
          acc[0] += v[e] - shift;
        }
        out[e] = p * scale;
      }
    }
    put(c, out);
  }
  if (rowloss != nullptr) {
    block_allreduce<SumOp, WG / kWave, 1>(acc, slots, phase);
    if (threadIdx.x == 0) rowloss[row] = (!DENSE && (id < 0 || id >= C)) ? NAN : -acc[0] * inv_rows;
  }
}

// ------------------------------------------------------------------------------------
// Strided views (rank <= 8): element offset from a flat index by div/mod over the shape,
// as the reference's strided kernels do (kernels/cross_entropy.mojo:80-152,244-307).
// ------------------------------------------------------------------------------------

__device__ __forceinline__ int64_t strided_offset(int64_t flat, const StridedView& v) {
  int64_t off = 0;
  for (int d = v.rank - 1; d >= 0; --d) {
    off += (flat % v.shape[d]) * v.stride[d];
    flat /= v.shape[d];
  }
  return off;
}

template <typename T, int WG, bool WANT_GRAD>
__global__ __launch_bounds__(WG) void ce_strided_kernel(const T* __restrict__ logits, const T* __restrict__ labels,
                                                        const T* __restrict__ upstream, float* __restrict__ rowloss,
                                                        T* __restrict__ dlogits, int64_t N, int64_t C, StridedView la,
                                                        StridedView lb) {
  __shared__ float slots[2 * (WG / kWave)];
  int phase = 0;
  const int64_t row = blockIdx.x;
  if (row >= N) return;
  const int64_t base = row * C;
  float m[1] = {-INFINITY};
  for (int64_t c = threadIdx.x; c < C; c += WG) m[0] = fmaxf(m[0], to_float(logits[strided_offset(base + c, la)]));
  block_allreduce<MaxOp, WG / kWave, 1>(m, slots, phase);
  phase ^= 1;
  const float m2 = m[0] * kLog2e;
  float s[1] = {0.f};
  for (int64_t c = threadIdx.x; c < C; c += WG)
    s[0] += fast_exp2(fmaf(to_float(logits[strided_offset(base + c, la)]), kLog2e, -m2));
  block_allreduce<SumOp, WG / kWave, 1>(s, slots, phase);
  phase ^= 1;
  const float inv_rows = 1.0f / static_cast<float>(N);
  if constexpr (WANT_GRAD) {
    const float inv_sum = 1.0f / s[0];
    const float scale = (upstream != nullptr ? to_float(upstream[0]) : 1.0f) * inv_rows;
    for (int64_t c = threadIdx.x; c < C; c += WG) {
      const float x = to_float(logits[strided_offset(base + c, la)]);
      const float y = to_float(labels[strided_offset(base + c, lb)]);
      dlogits[base + c] = from_float<T>((fast_exp2(fmaf(x, kLog2e, -m2)) * inv_sum - y) * scale);
    }
  } else {
    const float shift = m[0] + logf(s[0]);
    float acc[1] = {0.f};
    for (int64_t c = threadIdx.x; c < C; c += WG) {
      const float x = to_float(logits[strided_offset(base + c, la)]);
      const float y = to_float(labels[strided_offset(base + c, lb)]);
      acc[0] += (x - shift) * y;
    }
    block_allreduce<SumOp, WG / kWave, 1>(acc, slots, phase);
    if (threadIdx.x == 0) rowloss[row] = -acc[0] * inv_rows;
  }
}

// loss[0] = sum of the N per-row terms, one workgroup, fixed order (no atomics).  It waits for memory, so U terms are in flight to
// a thread: one after the other, 16384 rows took 5.7 us, with sixteen 4.7, of which a launch of one workgroup is half.  Up to 2048
// rows the shorter code with one is faster, by 0.7 us at 300 and at 760.
template <typename T, int U>
__global__ __launch_bounds__(1024) void sum_rows_kernel(const float* __restrict__ rowloss, T* __restrict__ loss, int64_t N) {
  __shared__ float slots[2 * 16];
  float acc[1] = {0.f};
  for (int64_t first = 0; first < N; first += U * 1024) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t i = first + u * 1024 + threadIdx.x;
      v[u] = 0.f;
      if (first + u * 1024 < N && i < N) v[u] = rowloss[i];  // the first condition is the workgroup's: few rows branch past the rest
    }
#pragma unroll
    for (int u = 0; u < U; ++u) acc[0] += v[u];
  }
  block_allreduce<SumOp, 16, 1>(acc, slots, 0);
  if (threadIdx.x == 0) loss[0] = from_float<T>(acc[0]);
}

// ------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------

template <typename T>
struct CrossEntropyOps {
  static constexpr int WIDE = WideVec<T>::value;
  struct Shape {
    int tpr, vpt;
  };

  // Rows of more chunks than these are streamed twice.  With dense labels, 32 chunks of two tensors a thread are more than
  // registers hold well: (8192, 50304) bf16 683 us held | 475 streamed, fp32 1300 | 1000, (4096, 40000) bf16 288 | 195.
  template <bool DENSE>
  static constexpr int64_t kMostChunks = !DENSE ? 16384 : 4096;

  // Thread layout for a row of `chunks` chunks held in registers; false if too wide.  Up to 16 chunks, and up to 32 where there are
  // rows enough: sixteen lanes per row, four rows per wave, as one wave per row left most lanes idle ((16384, 65) bf16 12.9 us | 9.4,
  // (16384, 128) 12.5 | 9.5, (16384, 129) 13.5 | 10.3; but (1905, 127) fp32, dense, 3.3 | 3.8).  Few rows of up to 256 chunks have a
  // workgroup each, whose threads have one chunk, instead of a wave, whose lanes have four ((228, 924) fp32, dense, 3.8 us | 3.0;
  // from 1100 rows of 128 chunks on, and 3600 of 256, waves are faster).
  static bool pick_shape(int64_t chunks, int64_t rows, Shape* s) {
    const bool narrow = env_int("MOGRAD_HIP_CE_NARROW", chunks <= 16 || rows >= 4096) != 0;
    const bool few = env_int("MOGRAD_HIP_CE_FEW", chunks > 64 && rows < (chunks <= 128 ? 768 : 2048)) != 0;
    if (narrow && chunks <= 16) *s = {16, 1};
    else if (narrow && chunks <= 32) *s = {16, 2};
    else if (chunks <= 64) *s = {64, 1};
    else if (few && chunks <= 256) *s = {256, 1};
    else if (chunks <= 128) *s = {64, 2};
    else if (chunks <= 256) *s = {64, 4};
    else if (chunks <= 1024) *s = {256, 4};
    else if (chunks <= 2048) *s = {512, 4};
    else if (chunks <= 4096) *s = {512, 8};
    else if (WIDE == 8 && chunks <= 6400) *s = {256, 25};  // 16-bit rows up to 51200 columns: see below
    else if (chunks <= 8192) *s = {512, 16};
    else if (WIDE == 4 && chunks <= 12800) *s = {256, 50};
    else if (chunks <= 16384) *s = {1024, 16};
    else return false;
    // Rows of about 50k columns (8193..12800 fp32 chunks, 4097..6400 16-bit chunks: 200
    // values per thread either way): 256 threads x 50 (fp32) or x 25 (16-bit) chunks by
    // default, which leaves room for two workgroups per CU so that one row's arithmetic
    // overlaps the other's memory traffic.  MOGRAD_HIP_CE_WIDE_ROW=512|1024 selects the
    // 512 x 25 or 1024 x 13 layout instead (tuning aid).
    if (WIDE == 4 && chunks > 8192 && chunks <= 12800) {
      const int pick = env_int("MOGRAD_HIP_CE_WIDE_ROW", 256);
      if (pick == 512) *s = {512, 25};
      if (pick == 1024) *s = {1024, 13};
    }
    return true;
  }

  static bool can_vectorise(int64_t C, std::initializer_list<const void*> ptrs) {
    if (WIDE == 1 || C % WIDE != 0) return false;
    for (const void* p : ptrs)
      if (p != nullptr && !aligned16(p)) return false;
    return true;
  }

  static unsigned row_grid(int64_t N, int rpw) {
    return static_cast<unsigned>(ceil_div(N, rpw));
  }

  template <int VEC, int TPR, int VPT, bool DENSE, bool ANY>
  static int launch_rows(const T* logits, const void* labels, const T* upstream, float* rowloss, T* dlogits, int64_t N,
                         int64_t C, int id64, hipStream_t stream) {
    constexpr int WG = TPR <= 64 ? 256 : TPR;
    hipLaunchKernelGGL((ce_rows_kernel<T, VEC, TPR, VPT, WG, DENSE, ANY>), dim3(row_grid(N, WG / TPR)), dim3(WG), 0, stream,
                       logits, labels, upstream, rowloss, dlogits, N, static_cast<int>(C), id64);
    MG_LAUNCH_CHECK();
    return MG_OK;
  }

  template <bool DENSE, bool ANY>
  static int dispatch_rows(Shape s, const T* logits, const void* labels, const T* upstream, float* rowloss, T* dlogits,
                           int64_t N, int64_t C, int id64, hipStream_t stream) {
#define MG_CE_CASE(TPR_, VPT_)        \
  if (s.tpr == TPR_ && s.vpt == VPT_) \
  return launch_rows<WIDE, TPR_, VPT_, DENSE, ANY>(logits, labels, upstream, rowloss, dlogits, N, C, id64, stream)
    MG_CE_CASE(16, 1);
    MG_CE_CASE(16, 2);
    MG_CE_CASE(64, 1);
    MG_CE_CASE(64, 2);
    MG_CE_CASE(64, 4);
    MG_CE_CASE(256, 1);
    MG_CE_CASE(256, 4);
    MG_CE_CASE(512, 4);
    MG_CE_CASE(512, 8);
    if constexpr (kMostChunks<DENSE> > 4096) MG_CE_CASE(512, 16);
    if constexpr (!DENSE) MG_CE_CASE(1024, 16);
    if constexpr (!DENSE && WIDE == 8) MG_CE_CASE(256, 25);
    if constexpr (!DENSE && WIDE == 4) {
      MG_CE_CASE(256, 50);
      MG_CE_CASE(512, 25);
      MG_CE_CASE(1024, 13);
    }
#undef MG_CE_CASE
    return fail(MG_ERR_UNSUPPORTED, "cross_entropy: no kernel for row shape (%d, %d)", s.tpr, s.vpt);
  }

  // 16-bit rows of more than 512 chunks with integer labels.
  template <bool ANY>
  static void launch_packed(int64_t chunks, const T* logits, const void* labels, const T* upstream, float* rowloss, T* dlogits,
                            int64_t N, int64_t C, int id64, hipStream_t stream) {
    auto launch = [&](auto kernel, int tpr) {
      hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(N)), dim3(tpr), 0, stream, logits, labels, upstream, rowloss, dlogits,
                         N, static_cast<int>(C), id64);
    };
    if constexpr (sizeof(T) == 2) {
      if (chunks <= 1024) launch(ce_rows_packed_kernel<T, 256, 4, ANY>, 256);
      else if (chunks <= 2048) launch(ce_rows_packed_kernel<T, 256, 8, ANY>, 256);
      else if (chunks <= 4096) launch(ce_rows_packed_kernel<T, 256, 16, ANY>, 256);
      else if (chunks <= 6400) launch(ce_rows_packed_kernel<T, 256, 25, ANY>, 256);
      else if (chunks <= 12800) launch(ce_rows_packed_kernel<T, 512, 25, ANY>, 512);
      else launch(ce_rows_packed_kernel<T, 1024, 16, ANY>, 1024);
    }
  }

  static int finish_loss(const float* rowloss, T* loss, int64_t N, hipStream_t stream) {
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(1), dim3(1024), 0, stream, rowloss, loss, N); };
    if (env_int("MOGRAD_HIP_CE_SUM_DEEP", N > 2048) != 0) launch(sum_rows_kernel<T, 16>);
    else launch(sum_rows_kernel<T, 1>);
    MG_LAUNCH_CHECK();
    return MG_OK;
  }

  // Gradient and/or loss.  `loss` and `dlogits` may each be null (not both).
  // `rowloss_ext`, when not null, is a buffer of at least N floats that takes the per-row
  // loss terms instead of a block from the pool (the entry point that allocates nothing).
  template <bool DENSE>
  static int run(const void* logits_, const void* labels, const void* upstream_, void* loss_, void* dlogits_, int64_t N,
                 int64_t C, int id64, hipStream_t stream, float* rowloss_ext = nullptr) {
    const T* logits = static_cast<const T*>(logits_);
    const T* upstream = static_cast<const T*>(upstream_);
    T* loss = static_cast<T*>(loss_);
    T* dlogits = static_cast<T*>(dlogits_);
    Scratch rowloss_buf;
    float* rowloss = nullptr;
    if (loss != nullptr && rowloss_ext != nullptr) {
      rowloss = rowloss_ext;
    } else if (loss != nullptr) {
      MG_TRY(rowloss_buf.take(N * static_cast<int64_t>(sizeof(float))));
      rowloss = rowloss_buf.as<float>();
    }
    const bool wide = can_vectorise(C, {logits, DENSE ? labels : nullptr, dlogits});
    // Rows off the 16-byte chunks, of one chunk and more: misaligned chunks instead of an element at a time ((8192, 50257) bf16
    // 480 us | 361, fp32 779 | 620; (16384, 8191) bf16 288 | 114, 4099 148 | 53, 2001 62 | 30, 333 27 | 14; fp32 257 26 | 15).
    const bool any = !wide && C >= WIDE;
    constexpr int SWG = 1024;
    if (dlogits == nullptr) {
      // larger than the 256 MB memory-side cache: read once, past the caches
      const bool once = N * C * static_cast<int64_t>(sizeof(T)) >= (int64_t{256} << 20);
      if (wide && once)
        hipLaunchKernelGGL((ce_fwd_stream_kernel<T, WIDE, SWG, DENSE, true>), dim3(static_cast<unsigned>(N)), dim3(SWG), 0,
                           stream, logits, labels, rowloss, N, C, id64);
      else if (wide)
        hipLaunchKernelGGL((ce_fwd_stream_kernel<T, WIDE, SWG, DENSE>), dim3(static_cast<unsigned>(N)), dim3(SWG), 0,
                           stream, logits, labels, rowloss, N, C, id64);
      // (rows of fewer elements than the workgroup has threads: one each; chunks were up to 23 % slower, (16239, 65) bf16 dense 12.8 us | 15.7)
      else if (any && env_int("MOGRAD_HIP_CE_LOSS_CHUNKS", C >= 256) != 0)
        hipLaunchKernelGGL((ce_fwd_stream_kernel<T, WIDE, 256, DENSE, false, true>), dim3(static_cast<unsigned>(N)), dim3(256),
                           0, stream, logits, labels, rowloss, N, C, id64);
      else
        hipLaunchKernelGGL((ce_fwd_stream_kernel<T, 1, 256, DENSE>), dim3(static_cast<unsigned>(N)), dim3(256), 0,
                           stream, logits, labels, rowloss, N, C, id64);
      MG_LAUNCH_CHECK();
      return finish_loss(rowloss, loss, N, stream);
    }
    Shape s;
    const int64_t chunks = ceil_div(C, WIDE);
    if constexpr (sizeof(T) == 2 && !DENSE) {
      // 16-bit rows of more than 512 chunks (4096 columns) with integer labels: the packed row
      // kernel ((8192, 50304) bf16 1220 -> 344 us, (16384, 16392) 415 -> 209 us, (65536, 4104)
      // 275 -> 205 us, (32768, 8192) 197 us either way).  MOGRAD_HIP_CE_PACKED=0: the fp32 tiles.
      if ((wide || any) && chunks > 512 && chunks <= 16384 && env_int("MOGRAD_HIP_CE_PACKED", 1) != 0) {
        if (wide) launch_packed<false>(chunks, logits, labels, upstream, rowloss, dlogits, N, C, id64, stream);
        else launch_packed<true>(chunks, logits, labels, upstream, rowloss, dlogits, N, C, id64, stream);
        MG_LAUNCH_CHECK();
        if (loss != nullptr) return finish_loss(rowloss, loss, N, stream);
        return MG_OK;
      }
    }
    // (Up to 16 elements off the chunks: one to a lane; bf16, dense, (801, 13) 3.6 us in chunks | 3.0, (9159, 10) 3.8 | 3.4.)
    if (C < WIDE || (any && C <= 16)) {
      MG_TRY((launch_rows<1, 16, 1, DENSE, false>(logits, labels, upstream, rowloss, dlogits, N, C, id64, stream)));
    } else if (chunks <= kMostChunks<DENSE> && pick_shape(chunks, N, &s)) {
      if (wide) MG_TRY((dispatch_rows<DENSE, false>(s, logits, labels, upstream, rowloss, dlogits, N, C, id64, stream)));
      else MG_TRY((dispatch_rows<DENSE, true>(s, logits, labels, upstream, rowloss, dlogits, N, C, id64, stream)));
    } else {
      auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(N)), dim3(SWG), 0, stream, logits, labels, upstream, rowloss,
                           dlogits, N, C, id64);
      };
      if (wide) launch(ce_grad_stream_kernel<T, WIDE, SWG, DENSE>);
      else launch(ce_grad_stream_kernel<T, WIDE, SWG, DENSE, true>);
      MG_LAUNCH_CHECK();
    }
    if (loss != nullptr) return finish_loss(rowloss, loss, N, stream);
    return MG_OK;
  }

  static int run_strided(const void* logits_, const void* labels_, const void* upstream_, void* loss_, void* dlogits_,
                         int64_t N, int64_t C, const StridedView& la, const StridedView& lb, hipStream_t stream) {
    const T* logits = static_cast<const T*>(logits_);
    const T* labels = static_cast<const T*>(labels_);
    const T* upstream = static_cast<const T*>(upstream_);
    T* loss = static_cast<T*>(loss_);
    T* dlogits = static_cast<T*>(dlogits_);
    if (dlogits != nullptr) {
      hipLaunchKernelGGL((ce_strided_kernel<T, 256, true>), dim3(static_cast<unsigned>(N)), dim3(256), 0, stream, logits,
                         labels, upstream, nullptr, dlogits, N, C, la, lb);
      MG_LAUNCH_CHECK();
      return MG_OK;
    }
    Scratch rowloss;
    MG_TRY(rowloss.take(N * static_cast<int64_t>(sizeof(float))));
    hipLaunchKernelGGL((ce_strided_kernel<T, 256, false>), dim3(static_cast<unsigned>(N)), dim3(256), 0, stream, logits,
                       labels, upstream, rowloss.as<float>(), dlogits, N, C, la, lb);
    MG_LAUNCH_CHECK();
    return finish_loss(rowloss.as<float>(), loss, N, stream);
  }
};

}  // namespace mg

// Defines the per-dtype entry points that cross_entropy.hip dispatches to.
#define MG_DEFINE_CROSS_ENTROPY(T, SUFFIX)                                                                          \
  namespace mg {                                                                                                    \
  int ce_run_##SUFFIX(bool dense, const void* logits, const void* labels, const void* upstream, void* loss,         \
                      void* dlogits, int64_t N, int64_t C, int id64, hipStream_t stream, float* rowloss_ext) {      \
    if (dense)                                                                                                      \
      return CrossEntropyOps<T>::template run<true>(logits, labels, upstream, loss, dlogits, N, C, id64, stream,    \
                                                    rowloss_ext);                                                   \
    return CrossEntropyOps<T>::template run<false>(logits, labels, upstream, loss, dlogits, N, C, id64, stream,     \
                                                   rowloss_ext);                                                    \
  }                                                                                                                 \
  int ce_run_strided_##SUFFIX(const void* logits, const void* labels, const void* upstream, void* loss,             \
                              void* dlogits, int64_t N, int64_t C, const StridedView& la, const StridedView& lb,    \
                              hipStream_t stream) {                                                                 \
    return CrossEntropyOps<T>::run_strided(logits, labels, upstream, loss, dlogits, N, C, la, lb, stream);          \
  }                                                                                                                 \
  }
