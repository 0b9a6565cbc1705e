// Device-side building blocks shared by every switchyard kernel (gfx950 only).
//
// Data moves in 16-byte chunks: 8 bf16/fp16 values or 4 fp32 values, one
// buffer_load_dwordx4 per lane. Each lane owns fixed chunks of a row; 64 lanes
// of a wave read 1 KiB of contiguous row memory per instruction.
//
// All arithmetic is fp32. Sums of squares and query dot products of 16-bit
// data use v_dot2_f32_{bf16,f16} (two exact products, fp32 accumulate), which
// halves the VALU count of the reductions; fp32 data uses plain FMAs.
//
// Timings in the comments of these sources are MI355X measurements, bf16
// unless stated. Named shapes: "config 2" is N=9 sources, B=1, T=4096,
// D=2048 (the operator's forward and backward); "config 3" the same sources
// with 8 queries (the batched forward); "config 4" the N / T / D sweeps around
// config 2; "config 5" the 1.3B decoder training step.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sy {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));

// dtype tags. `code` matches sy_dtype in include/switchyard.h.
struct BF16 { using storage = uint16_t; static constexpr int code = 2; static constexpr int ce = 8; };
struct F16  { using storage = uint16_t; static constexpr int code = 1; static constexpr int ce = 8; };
struct F32  { using storage = float;    static constexpr int code = 0; static constexpr int ce = 4; };

// Where the N source rows of a token start (and, for dv, the N gradient rows).
// Row n of token t is at row_of(table, n) + t*D. Rows n < kTableRows come from
// p[n]; rows beyond are p[0] + n*stride_bytes, the stacked [N][n_tok][D]
// layout. A stacked caller fills p[n] = base + n*stride; a caller with one
// tensor per source fills p[0..N) directly and needs N <= kTableRows. The table
// travels in the kernel arguments, so the resident kernels (compile-time n)
// read each row pointer with one scalar load.
constexpr int kTableRows = 16;
struct RowTable {
  void* p[kTableRows];
  int64_t stride_bytes;
};

template <class S>
__host__ __device__ __forceinline__ S* row_of(const RowTable& t, int n) {
  return n < kTableRows ? static_cast<S*>(t.p[n])
                        : reinterpret_cast<S*>(static_cast<char*>(t.p[0]) + (int64_t)n * t.stride_bytes);
}

// Row n with the addressing mode fixed at compile time: LISTED reads p[n]
// (n < kTableRows), otherwise p[0] + n*stride_bytes. Kernels that are short of
// SGPRs use this: the stacked form keeps one pointer and a stride live, where
// per-row pointers would take two SGPRs per row.
template <bool LISTED, class S>
__device__ __forceinline__ S* row_at(const RowTable& t, int n) {
  if constexpr (LISTED) {
    return static_cast<S*>(t.p[n]);
  } else {
    return reinterpret_cast<S*>(static_cast<char*>(t.p[0]) + (int64_t)n * t.stride_bytes);
  }
}

// Threads per backward workgroup (token slots x waves per token), at least one
// token's waves. Two- and one-chunk tiles use SY_BWD_BLOCK (512 measured best on
// MI355X: 128 +9%, 256 equal), i.e. two waves per SIMD at <= 256 VGPRs. Four-chunk
// tiles use 256 threads: one wave per SIMD, so a wave may hold 512 registers
// (256 VGPRs + 256 AGPRs) -- the 144-register tile plus everything else, with
// no spills. The 32-row kernel (k_bwd_tall) runs 512 threads with one chunk a
// lane (two waves per SIMD: a 128-VGPR tile) and 256 with two; its 64-row
// tiles (one chunk a lane, 256 tile VGPRs) run 256. Build-time
// constants so that kernels and the host plan agree.
#ifndef SY_BWD_BLOCK
#define SY_BWD_BLOCK 512
#endif
constexpr int bwd_block_base(int vpl, int nr) {
  return nr > 16 ? (vpl == 1 && nr <= 32 ? 512 : 256) : vpl >= 4 ? 256 : SY_BWD_BLOCK;
}
constexpr int bwd_block(int w, int vpl, int nr = 0) {
  return bwd_block_base(vpl, nr) > 64 * w ? bwd_block_base(vpl, nr) : 64 * w;
}

// Buffer resource word 3 for gfx9-family raw buffers (32-bit dword format).
constexpr int kRsrcFlags = 0x00020000;

// A raw buffer over [p, p + bytes). Loads past `bytes` return 0 and stores
// past it are dropped, which gives free masking of partial rows.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, kRsrcFlags);
}

// Cache policy of streamed traffic (v, grad_out in; out, dv out): every byte
// is touched once, so the loads carry the `nt` (non-temporal) hint by default.
// Operands every wave re-reads (w, queries) use the default policy.
#ifndef SY_STREAM_LOAD_AUX
#define SY_STREAM_LOAD_AUX 2
#endif
#ifndef SY_STREAM_STORE_AUX
#define SY_STREAM_STORE_AUX 2
#endif

__device__ __forceinline__ i32x4_t ld16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
}
__device__ __forceinline__ i32x4_t ld16_stream(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, SY_STREAM_LOAD_AUX);
}
__device__ __forceinline__ void st16(__amdgpu_buffer_rsrc_t r, uint32_t off, i32x4_t x) {
  __builtin_amdgcn_raw_buffer_store_b128(x, r, off, 0, 0);
}
__device__ __forceinline__ void st16_stream(__amdgpu_buffer_rsrc_t r, uint32_t off, i32x4_t x) {
  __builtin_amdgcn_raw_buffer_store_b128(x, r, off, 0, SY_STREAM_STORE_AUX);
}
// Policy of the dv stores that measured faster with the device-scope bit (sc1 = 16)
// next to nt: the operator backward's 16-bit 9-row tiles whose wave slice spans four
// chunks, and its 32- and 64-row tiles (k_bwd, k_bwd_tall); the other tiles and
// kernels measured slower with it and keep SY_STREAM_STORE_AUX.
#ifndef SY_DV_STORE_AUX
#define SY_DV_STORE_AUX 18
#endif
template <int AUX>
__device__ __forceinline__ void st16_aux(__amdgpu_buffer_rsrc_t r, uint32_t off, i32x4_t x) {
  __builtin_amdgcn_raw_buffer_store_b128(x, r, off, 0, AUX);
}

// ---------------------------------------------------------------- conversion

__device__ __forceinline__ float bf_lo(uint32_t x) { return __uint_as_float(x << 16); }
__device__ __forceinline__ float bf_hi(uint32_t x) { return __uint_as_float(x & 0xffff0000u); }

// Element e of a 16-byte chunk as fp32.
template <class T> __device__ __forceinline__ float elem(const i32x4_t& c, int e);
template <> __device__ __forceinline__ float elem<BF16>(const i32x4_t& c, int e) {
  const uint32_t x = (uint32_t)c[e >> 1];
  return (e & 1) ? bf_hi(x) : bf_lo(x);
}
template <> __device__ __forceinline__ float elem<F16>(const i32x4_t& c, int e) {
  const int word = c[e >> 1];  // copy first: bit_cast of a vector element reads lane 0
  const f16x2_t h = __builtin_bit_cast(f16x2_t, word);
  return (e & 1) ? (float)h.y : (float)h.x;
}
template <> __device__ __forceinline__ float elem<F32>(const i32x4_t& c, int e) {
  return __int_as_float(c[e]);
}

// Round fp32 values to the storage type (round-to-nearest-even) and pack.
template <class T> __device__ __forceinline__ i32x4_t pack(const float* f);
template <> __device__ __forceinline__ i32x4_t pack<BF16>(const float* f) {
  i32x4_t r;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const f32x2_t p = {f[2 * k], f[2 * k + 1]};
    r[k] = __builtin_bit_cast(int, __builtin_convertvector(p, bf16x2_t));
  }
  return r;
}
template <> __device__ __forceinline__ i32x4_t pack<F16>(const float* f) {
  i32x4_t r;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const f32x2_t p = {f[2 * k], f[2 * k + 1]};
    r[k] = __builtin_bit_cast(int, __builtin_convertvector(p, f16x2_t));
  }
  return r;
}
template <> __device__ __forceinline__ i32x4_t pack<F32>(const float* f) {
  i32x4_t r;
#pragma unroll
  for (int k = 0; k < 4; ++k) r[k] = __float_as_int(f[k]);
  return r;
}

// acc + sum_e a[e] * b[e] over one chunk.
template <class T> __device__ __forceinline__ float dot(const i32x4_t& a, const i32x4_t& b, float acc);
template <> __device__ __forceinline__ float dot<BF16>(const i32x4_t& a, const i32x4_t& b, float acc) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    // Copy the dwords out first: __builtin_bit_cast applied directly to an
    // ext_vector element reads element 0 whatever the index.
    const int ak = a[k], bk = b[k];
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, ak),
                                          __builtin_bit_cast(bf16x2_t, bk), acc, false);
  }
  return acc;
}
template <> __device__ __forceinline__ float dot<F16>(const i32x4_t& a, const i32x4_t& b, float acc) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int ak = a[k], bk = b[k];
    acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, ak), __builtin_bit_cast(f16x2_t, bk),
                                 acc, false);
  }
  return acc;
}
template <> __device__ __forceinline__ float dot<F32>(const i32x4_t& a, const i32x4_t& b, float acc) {
#pragma unroll
  for (int k = 0; k < 4; ++k) acc = fmaf(__int_as_float(a[k]), __int_as_float(b[k]), acc);
  return acc;
}

// The same with the chunk summed from zero before it joins acc, fp32 in two halves: a
// lane's chunks would else be one long chain. Rows of any start and queries of another
// dtype use it; their error against float64 is then that of a block a row, whose threads
// sum a few elements each (gradients: fp32 N=5 T=300 D=777 8.9e-7 -> 6.0e-7, the block
// 6.4e-7; bf16 rows, fp32 query with a gain, N=9 T=300 D=2048 2.2e-6 -> 1.7e-6, 1.6e-6).
template <class T> __device__ __forceinline__ float dot_short(const i32x4_t& a, const i32x4_t& b, float acc) {
  if constexpr (T::code == F32::code) {
    const float lo = fmaf(__int_as_float(a[1]), __int_as_float(b[1]), __int_as_float(a[0]) * __int_as_float(b[0]));
    const float hi = fmaf(__int_as_float(a[3]), __int_as_float(b[3]), __int_as_float(a[2]) * __int_as_float(b[2]));
    return acc + (lo + hi);
  } else {
    return acc + dot<T>(a, b, 0.0f);
  }
}

template <class T, bool SHORT>
__device__ __forceinline__ float row_dot(const i32x4_t& a, const i32x4_t& b, float acc) {
  if constexpr (SHORT) return dot_short<T>(a, b, acc);
  else return dot<T>(a, b, acc);
}

// The elements of a lane's VPL chunks (CE elements each, `step` bytes of the sources'
// row apart) of a query row of dtype wt (0 fp32, 1 fp16, 2 bf16, uniform over the
// launch) as fp32, times the same of gain where the query is given as its two factors
// (gain may be nullptr). Elements past the row read 0. A query may have another dtype
// than the sources (fp32 parameters with 16-bit activations); the widening is exact,
// and the product is formed in fp32 and never rounded. Every load is issued before the
// first is used: chunk by chunk, with the branches on dtype and gain inside, a launch
// began with VPL (with a gain 2 VPL) memory latencies in a row. Forward + backward, us:
// bf16 N=9 D=4096 B=4 T=4096 687 -> 676, D=2048 T=4096 88.3 -> 87.0, with fp32 query and
// gain 92.5 -> 91.5. Dtypes are told apart outside the loads, not per element.
template <int CE>
struct RawQuery {  // a chunk as it lies in memory, at most CE fp32 elements
  int x[CE];
};
template <int CE, int VPL>
__device__ __forceinline__ void ld_raw(const void* row, bool f32, uint32_t d, uint32_t lane_off,
                                       uint32_t step, RawQuery<CE> (&r)[VPL]) {
  const auto rs = make_rsrc(row, d * (f32 ? 4u : 2u));
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const uint32_t c = (lane_off + j * step) / 16u;
    if (f32 || CE == 8) {
#pragma unroll
      for (int q = 0; q < (f32 ? CE / 4 : 1); ++q) {
        const i32x4_t t = ld16(rs, f32 ? (c * CE + 4 * q) * 4u : c * 16u);
#pragma unroll
        for (int e = 0; e < 4; ++e) r[j].x[4 * q + e] = t[e];
      }
    } else {
      const auto t = __builtin_amdgcn_raw_buffer_load_b64(rs, c * 8u, 0, 0);
      r[j].x[0] = (int)t[0];
      r[j].x[1] = (int)t[1];
    }
  }
}
// Element e of a raw chunk.
template <int CE>
__device__ __forceinline__ float raw_elem(const RawQuery<CE>& r, bool f32, bool bf, int e) {
  if (f32) return __int_as_float(r.x[e]);
  const int p = r.x[e / 2];
  const f16x2_t h = __builtin_bit_cast(f16x2_t, p);
  if (e % 2 == 0) return bf ? bf_lo((uint32_t)p) : (float)h.x;
  return bf ? bf_hi((uint32_t)p) : (float)h.y;
}
template <int CE, int VPL>
__device__ __forceinline__ void ld_query_of(const void* w, const void* gain, bool f32, bool bf, uint32_t d,
                                            uint32_t lane_off, uint32_t step, float (&f)[VPL][CE]) {
  RawQuery<CE> x[VPL];
  if (gain == nullptr) {
    ld_raw(w, f32, d, lane_off, step, x);
#pragma unroll
    for (int j = 0; j < VPL; ++j)
#pragma unroll
      for (int e = 0; e < CE; ++e) f[j][e] = raw_elem(x[j], f32, bf, e);
  } else {
    RawQuery<CE> y[VPL];
    ld_raw(w, f32, d, lane_off, step, x);
    ld_raw(gain, f32, d, lane_off, step, y);
#pragma unroll
    for (int j = 0; j < VPL; ++j)
#pragma unroll
      for (int e = 0; e < CE; ++e) f[j][e] = raw_elem(x[j], f32, bf, e) * raw_elem(y[j], f32, bf, e);
  }
}
template <int CE, int VPL>
__device__ __forceinline__ void ld_query_row(const void* w, const void* gain, int wt, uint32_t d,
                                             uint32_t lane_off, uint32_t step, float (&f)[VPL][CE]) {
  if (wt == F32::code)
    ld_query_of(w, gain, true, false, d, lane_off, step, f);
  else if (wt == BF16::code)
    ld_query_of(w, gain, false, true, d, lane_off, step, f);
  else
    ld_query_of(w, gain, false, false, d, lane_off, step, f);
}

// The same where the query mostly has the sources' dtype and no gain: that one is loaded
// first, as packed words, and all others out of line. Behind their branches its loads were
// waited for before the first rows were asked for, and the launch's code was longer to
// fetch (fp32 N=6 T=1430 D=512 forward 6.0 -> 6.6 us, backward 8.9 -> 9.4; forward +
// backward 22.5 so, 21.3 now and without any of them. Loads without branches, finished
// after the first rows are asked for, took 22.8).
// An fp32 query stays in the words it was loaded to (no copies, which would wait for it).
template <class T, int VPL>
__device__ __forceinline__ void ld_query(const void* w, const void* gain, int wt, uint32_t d,
                                         uint32_t lane_off, uint32_t step, float (&f)[VPL][T::ce]) {
  constexpr bool kF32 = T::code == F32::code;
  i32x4_t q[VPL];
  if (__builtin_expect(gain == nullptr && wt == T::code, 1)) {
    const auto r = make_rsrc(w, d * (uint32_t)sizeof(typename T::storage));
#pragma unroll
    for (int j = 0; j < VPL; ++j) q[j] = ld16(r, lane_off + j * step);
#pragma unroll
    for (int j = 0; j < VPL; ++j)
#pragma unroll
      for (int e = 0; e < (kF32 ? 0 : T::ce); ++e) f[j][e] = elem<T>(q[j], e);
  } else {
    ld_query_row(w, gain, wt, d, lane_off, step, f);
#pragma unroll
    for (int j = 0; j < VPL; ++j)
#pragma unroll
      for (int e = 0; e < (kF32 ? 4 : 0); ++e) q[j][e] = __float_as_int(f[j][e]);
  }
  if constexpr (kF32) {
#pragma unroll
    for (int j = 0; j < VPL; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) f[j][e] = __int_as_float(q[j][e]);
  }
}

// acc + sum_e x[e] * f[e] with an fp32 query chunk.
template <class T>
__device__ __forceinline__ float dot_wide(const i32x4_t& x, const float* f, float acc) {
#pragma unroll
  for (int e = 0; e < T::ce; e += 4) {
    const float lo = fmaf(elem<T>(x, e + 1), f[e + 1], elem<T>(x, e) * f[e]);
    const float hi = fmaf(elem<T>(x, e + 3), f[e + 3], elem<T>(x, e + 2) * f[e + 2]);
    acc += lo + hi;
  }
  return acc;
}

// A lane's query chunks: packed in the sources' dtype, or as fp32 values when the query
// has another dtype or a gain (kWideQuery), or for two 16-bit factors of the sources' dtype
// as the two packed parts of their product
// (kSplitQuery). fp32 sources hold any query as fp32 chunks.
enum QueryForm { kPacked = 0, kWideQuery = 1, kSplitQuery = 2 };
template <class T, int FORM, int VPL>
struct Query {
  i32x4_t q[VPL];
  __device__ __forceinline__ void load(const void* w, const void* gain, int wt, uint32_t d,
                                       uint32_t lane_off, uint32_t step) {
    if constexpr (T::code == F32::code) {
      float f[VPL][4];
      ld_query<T>(w, gain, wt, d, lane_off, step, f);
#pragma unroll
      for (int j = 0; j < VPL; ++j) q[j] = pack<T>(f[j]);
    } else {
      const auto r = make_rsrc(w, d * 2u);
#pragma unroll
      for (int j = 0; j < VPL; ++j) q[j] = ld16(r, lane_off + j * step);
    }
  }
  __device__ __forceinline__ float dot(const i32x4_t& x, int j, float acc) const {
    return sy::dot<T>(x, q[j], acc);
  }
  __device__ __forceinline__ float dot_short(const i32x4_t& x, int j, float acc) const {
    return sy::dot_short<T>(x, q[j], acc);
  }
};
template <class T, int VPL>
struct Query<T, kWideQuery, VPL> {
  float f[VPL][T::ce];
  __device__ __forceinline__ void load(const void* w, const void* gain, int wt, uint32_t d,
                                       uint32_t lane_off, uint32_t step) {
    ld_query_row(w, gain, wt, d, lane_off, step, f);
  }
  __device__ __forceinline__ float dot(const i32x4_t& x, int j, float acc) const {
    return dot_wide<T>(x, f[j], acc);
  }
  __device__ __forceinline__ float dot_short(const i32x4_t& x, int j, float acc) const {
    return dot_wide<T>(x, f[j], acc);
  }
};

// The product of two bf16 (fp16) factors has at most 16 (22) significant bits: its
// rounding to that type and what that leaves are both exact, and two packed dots cost half
// the operations of one on widened elements. fp16 has not the exponents for that, so a
// lane scales its products by the power of two that brings the largest below 2^15, and
// their remainders by 2^11: what then lies below fp16's range is under 2^-29 of the
// largest. The second part is in LDS, as the registers are full (each thread reads only
// what it wrote; the opaque index keeps the compiler from holding it).
template <class T, int VPL, int THREADS>
struct QuerySplit {
  static constexpr bool kF16 = T::code == F16::code;
  typedef i32x4_t Lds[VPL][THREADS];
  i32x4_t hi[VPL];
  float scale;
  __device__ __forceinline__ void load(Lds& lo, const void* w, const void* gain, int wt, uint32_t d,
                                       uint32_t lane_off, uint32_t step) {
    float f[VPL][T::ce];
    ld_query_row(w, gain, wt, d, lane_off, step, f);
    int shift = 0;
    if constexpr (kF16) {
      float top = 0.0f;
#pragma unroll
      for (int j = 0; j < VPL; ++j)
#pragma unroll
        for (int e = 0; e < T::ce; ++e) top = fmaxf(top, fabsf(f[j][e]));
      shift = 15 - __builtin_amdgcn_frexp_expf(top);
      scale = ldexpf(1.0f, -shift);
    }
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      if constexpr (kF16) {
#pragma unroll
        for (int e = 0; e < T::ce; ++e) f[j][e] = ldexpf(f[j][e], shift);
      }
      hi[j] = pack<T>(f[j]);
#pragma unroll
      for (int e = 0; e < T::ce; ++e) f[j][e] = (f[j][e] - elem<T>(hi[j], e)) * (kF16 ? 2048.0f : 1.0f);
      lo[j][threadIdx.x] = pack<T>(f[j]);
    }
  }
  // A row's chunks are added from zero; done() is then its dot.
  __device__ __forceinline__ float dot(const Lds& lo, const i32x4_t& x, int j, float acc) const {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    if constexpr (kF16) {
      const float rest = sy::dot<T>(x, lo[j][t], 0.0f);
      return sy::dot<T>(x, hi[j], fmaf(rest, 1.0f / 2048.0f, acc));
    } else {
      return sy::dot<T>(x, lo[j][t], sy::dot<T>(x, hi[j], acc));
    }
  }
  __device__ __forceinline__ float done(float acc) const { return kF16 ? acc * scale : acc; }
};

// A wide query in LDS, for 16-bit tiles whose registers are full: four elements a piece, a
// lane's pieces `THREADS` apart (a wave's reads are contiguous). Each thread reads only
// what it wrote, so no barrier is needed.
template <class T, int VPL, int THREADS>
struct QueryLds {
  static constexpr int kPer = T::ce / 4;  // pieces of a chunk
  i32x4_t s[VPL * kPer][THREADS];
  __device__ __forceinline__ void load(const void* w, const void* gain, int wt, uint32_t d,
                                       uint32_t lane_off, uint32_t step) {
    float f[VPL][T::ce];
    ld_query_row(w, gain, wt, d, lane_off, step, f);
#pragma unroll
    for (int i = 0; i < VPL * kPer; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[i][threadIdx.x][e] = __float_as_int(f[i / kPer][4 * (i % kPer) + e]);
  }
  // Chunk j. The opaque index keeps the compiler from reading a chunk once and holding
  // it, which would take the registers again.
  __device__ __forceinline__ void chunk(int j, float* f) const {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
#pragma unroll
    for (int h = 0; h < kPer; ++h) {
      const i32x4_t x = s[j * kPer + h][t];
#pragma unroll
      for (int e = 0; e < 4; ++e) f[4 * h + e] = __int_as_float(x[e]);
    }
  }
};

// Scalar element load/store for the generic (unaligned) path.
__device__ __forceinline__ float load_elem(const void* p, int64_t i, int dtype) {
  if (dtype == 2) return __uint_as_float((uint32_t)((const uint16_t*)p)[i] << 16);
  if (dtype == 1) return (float)((const _Float16*)p)[i];
  return ((const float*)p)[i];
}
__device__ __forceinline__ void store_elem(void* p, int64_t i, float x, int dtype) {
  if (dtype == 2) {
    ((__bf16*)p)[i] = (__bf16)x;
  } else if (dtype == 1) {
    ((_Float16*)p)[i] = (_Float16)x;
  } else {
    ((float*)p)[i] = x;
  }
}

// ------------------------------------------------------------ row access
//
// A lane's 16-byte chunk of a row. UNAL = false: the row starts at a 16-byte
// boundary and holds whole chunks; the buffer resource masks what lies past it.
// UNAL = true: a row of at least 16 bytes that starts at any element. The chunk is
// read and written with unaligned 16-byte global accesses, the last one moved back to
// end with the row: it overlaps the chunk before it and repeats its last elements.
// Lanes past the row read that chunk too and store nothing. Everything element-wise
// (out, dv, dw) then holds the same value in both lanes; only sums over the row have
// to leave the repeated elements out (TailMask).
typedef int i32x4_any_t __attribute__((ext_vector_type(4), aligned(2)));
typedef int i32x4_f32_t __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ uint32_t tail_off(uint32_t off, uint32_t row_bytes) {
  return min(off, row_bytes - 16u);
}
template <bool UNAL, class S>
__device__ __forceinline__ i32x4_t ld_row(const S* row, uint32_t row_bytes, uint32_t off) {
  if constexpr (UNAL) {
    const char* p = reinterpret_cast<const char*>(row) + tail_off(off, row_bytes);
    if constexpr (sizeof(S) == 4) return __builtin_nontemporal_load(reinterpret_cast<const i32x4_f32_t*>(p));
    else return __builtin_nontemporal_load(reinterpret_cast<const i32x4_any_t*>(p));
  } else {
    return ld16_stream(make_rsrc(row, row_bytes), off);
  }
}
template <bool UNAL, int AUX, class S>
__device__ __forceinline__ void st_row(S* row, uint32_t row_bytes, uint32_t off, bool live, i32x4_t x) {
  if constexpr (UNAL) {
    if (live && off < row_bytes) {
      char* p = reinterpret_cast<char*>(row) + tail_off(off, row_bytes);
      if constexpr (sizeof(S) == 4) __builtin_nontemporal_store(x, reinterpret_cast<i32x4_f32_t*>(p));
      else __builtin_nontemporal_store(x, reinterpret_cast<i32x4_any_t*>(p));
    }
  } else {
    st16_aux<AUX>(make_rsrc(row, live ? row_bytes : 0u), off, x);
  }
}
// The bits of the chunk at `off` that are not repeats: all of them, or for the row's
// last chunk its last (row_bytes - off) bytes, or none past the row.
__device__ __forceinline__ i32x4_t tail_mask(uint32_t off, uint32_t row_bytes) {
  const int dup = off >= row_bytes ? 16 : max(0, (int)(off + 16u - row_bytes));  // bytes
  i32x4_t m;
#pragma unroll
  for (int k = 0; k < 4; ++k) m[k] = dup <= 4 * k ? -1 : dup >= 4 * k + 4 ? 0 : (int)0xffff0000;
  return m;
}
template <bool UNAL, int VPL>
__device__ __forceinline__ i32x4_t own_part(const i32x4_t& x, int j, const i32x4_t& mask) {
  if constexpr (UNAL) return j == VPL - 1 ? (x & mask) : x;
  else return x;
}

// The query elements from element c on (no alignment assumed).
template <int CE>
__device__ __forceinline__ void ld_query_at(const void* w, int64_t c, int wt, float* f) {
  if (wt == F32::code) {
#pragma unroll
    for (int q = 0; q < CE / 4; ++q) {
      const i32x4_t x = *reinterpret_cast<const i32x4_f32_t*>(static_cast<const float*>(w) + c + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) f[4 * q + e] = __int_as_float(x[e]);
    }
    return;
  }
  const uint16_t* h = static_cast<const uint16_t*>(w) + c;
  uint32_t x[CE];
  if constexpr (CE == 8) {
    const i32x4_t t = *reinterpret_cast<const i32x4_any_t*>(h);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (uint32_t)t[e / 2] >> (16 * (e & 1)) & 0xffffu;
  } else {
#pragma unroll
    for (int e = 0; e < CE; ++e) x[e] = h[e];
  }
#pragma unroll
  for (int e = 0; e < CE; ++e)
    f[e] = wt == BF16::code ? __uint_as_float(x[e] << 16)
                            : (float)__builtin_bit_cast(_Float16, (uint16_t)x[e]);
}

// Those of the chunk at `off` of an unaligned row, times the gain's.
template <int CE>
__device__ __forceinline__ void ld_query_any(const void* w, const void* gain, uint32_t off,
                                             uint32_t row_bytes, int wt, float* f) {
  const int64_t c = tail_off(off, row_bytes) / (16 / CE);
  ld_query_at<CE>(w, c, wt, f);
  if (gain != nullptr) {
    float g[CE];
    ld_query_at<CE>(gain, c, wt, g);
#pragma unroll
    for (int e = 0; e < CE; ++e) f[e] *= g[e];
  }
}

// ---------------------------------------------------------------- reductions

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, ROW_MASK, 0xf, false));
}

// Sum over the 64 lanes of a wave, returned as a wave-uniform value. Six DPP
// adds leave the total in lane 63 (quad swaps, half-row and row mirrors, then
// the two row broadcasts), and one readlane makes it uniform. The order of the
// adds is fixed, so every wave of a kernel rounds identically.
__device__ __forceinline__ float wave_sum(float x) {
  x += dpp<0xB1>(x);          // quad_perm [1,0,3,2]
  x += dpp<0x4E>(x);          // quad_perm [2,3,0,1]
  x += dpp<0x141>(x);         // row_half_mirror
  x += dpp<0x140>(x);         // row_mirror: every lane holds its row's sum
  x += dpp<0x142, 0xa>(x);    // row_bcast:15 into rows 1 and 3
  x += dpp<0x143, 0xc>(x);    // row_bcast:31 into rows 2 and 3
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

// Sums of P per-lane values over the 64 lanes, transposed (P = 2, 4, ..., 32):
// lane l ends up with the total of v[tsum_row<P>(l)]. Each step halves the
// values a lane carries: gfx950's permlane32/permlane16 swaps pair the halves
// across lane bits 5 and 4, then DPP row rotation by 8, the half-row mirror and
// a quad permutation pair lanes across bits 3, 2 and 0, each taking the next
// lower bit of the value index; the lane bits left over are summed out by the
// same DPP steps without a split. So v[n] lands in the lanes l with
// n = b5..b2 of l for P = 16 (l >> 2), l >> 3 for P = 8, and for P = 32 in
// n = b0 + 2*b2 + 4*b3 + 8*b4 + 16*b5 -- 70 VALU instructions for 32 values
// where 32 separate six-step reductions take ~380, 36 for 16. tsum_lane<P>(n)
// is one lane that holds v[n]'s total. The order of the adds is fixed, so the
// result is deterministic; lanes that hold the same total hold the same bits
// within a quad, but may differ by rounding between quads for P <= 8.
template <int P>
__device__ __forceinline__ constexpr int tsum_lane(int n) {
  static_assert(P >= 2 && P <= 32 && (P & (P - 1)) == 0, "P is a power of two in [2, 32]");
  if constexpr (P == 32) return (n & 1) | ((n >> 1) << 2);
  return n << (P == 16 ? 2 : P == 8 ? 3 : P == 4 ? 4 : 5);
}
template <int P>
__device__ __forceinline__ int tsum_row(int lane) {
  if constexpr (P == 32) return (lane & 1) | ((lane >> 1) & ~1);
  return lane >> (P == 16 ? 2 : P == 8 ? 3 : P == 4 ? 4 : 5);
}
template <int P>
__device__ __forceinline__ float tsum(const float (&v)[P], int lane) {
  static_assert(P >= 2 && P <= 32 && (P & (P - 1)) == 0, "P is a power of two in [2, 32]");
  const bool b3 = (lane & 8) != 0, b2 = (lane & 4) != 0, b0 = (lane & 1) != 0;
  float a[P / 2];
#pragma unroll
  for (int i = 0; i < P / 2; ++i) {  // value i + (P/2)*b5
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[i]), __float_as_uint(v[i + P / 2]),
                                                    false, false);
    a[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  if constexpr (P == 2) {
    // one value: halve across bit 4 with the swap on itself, then sum bits 3..0
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a[0]), __float_as_uint(a[0]),
                                                    false, false);
    float f = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    f += dpp<0x128>(f);  // row_ror:8
    f += dpp<0x141>(f);  // row_half_mirror
    f += dpp<0xB1>(f);
    return f + dpp<0x4E>(f);
  } else {
    float b[P / 4];
#pragma unroll
    for (int i = 0; i < P / 4; ++i) {  // value i + (P/4)*b4 + (P/2)*b5
      const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a[i]), __float_as_uint(a[i + P / 4]),
                                                      false, false);
      b[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    if constexpr (P == 4) {
      float f = b[0] + dpp<0x128>(b[0]);
      f += dpp<0x141>(f);
      f += dpp<0xB1>(f);
      return f + dpp<0x4E>(f);
    } else {
      float c[P / 8];
#pragma unroll
      for (int i = 0; i < P / 8; ++i)  // row_ror:8 pairs l with l ^ 8
        c[i] = (b3 ? b[i + P / 8] : b[i]) + dpp<0x128>(b3 ? b[i] : b[i + P / 8]);
      if constexpr (P == 8) {
        float f = c[0] + dpp<0x141>(c[0]);
        f += dpp<0xB1>(f);
        return f + dpp<0x4E>(f);
      } else {
        float e[P / 16];
#pragma unroll
        for (int i = 0; i < P / 16; ++i)  // row_half_mirror pairs l with 7 - l in each 8 lanes
          e[i] = (b2 ? c[i + P / 16] : c[i]) + dpp<0x141>(b2 ? c[i] : c[i + P / 16]);
        if constexpr (P == 16) {
          const float f = e[0] + dpp<0xB1>(e[0]);
          return f + dpp<0x4E>(f);
        } else {
          const float f = (b0 ? e[1] : e[0]) + dpp<0xB1>(b0 ? e[0] : e[1]);  // quad_perm [1,0,3,2]
          return f + dpp<0x4E>(f);                                          // quad_perm [2,3,0,1]
        }
      }
    }
  }
}
__device__ __forceinline__ int tsum32_row(int lane) { return tsum_row<32>(lane); }
__device__ __forceinline__ float tsum32(const float (&v)[32], int lane) { return tsum<32>(v, lane); }

// Smallest power of two >= x (x >= 1), for sizing a tsum.
__host__ __device__ constexpr int pow2_at_least(int x) { return x <= 1 ? 1 : 2 * pow2_at_least((x + 1) / 2); }

// Max over the 64 lanes, wave-uniform. Rows that a broadcast skips see -inf
// from the DPP `old` operand, which leaves the max unchanged.
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ float dpp_or_ninf(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp((int)0xff800000, __float_as_int(x), CTRL,
                                                    ROW_MASK, 0xf, false));
}
__device__ __forceinline__ float wave_max(float x) {
  x = fmaxf(x, dpp_or_ninf<0xB1>(x));
  x = fmaxf(x, dpp_or_ninf<0x4E>(x));
  x = fmaxf(x, dpp_or_ninf<0x141>(x));
  x = fmaxf(x, dpp_or_ninf<0x140>(x));
  x = fmaxf(x, dpp_or_ninf<0x142, 0xa>(x));
  x = fmaxf(x, dpp_or_ninf<0x143, 0xc>(x));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

__device__ __forceinline__ int wave_id() {
  return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

}  // namespace sy
