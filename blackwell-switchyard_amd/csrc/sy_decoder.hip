// The decoder's element-wise sublayer work around its GEMMs and attention, one kernel
// each way: RMSNorm, rotary position embedding together with the split of a fused QKV
// projection into attention's layout, and SwiGLU. Evaluated operation by operation
// these are 8, 24 and 2 launches a call, each reading and writing whole activations,
// and the small decoder's forward (8 layers, 2048 tokens of 512) is bound by launching
// them. All are HBM- or launch-bound; arithmetic is fp32 with one rounding of each
// output.
//
// Reference: src/switchyard/model.py:238-319 (RMSNorm, rotary, attention, SwiGLU of
// the reference's decoder, eager there).
#include <algorithm>

#include "sy_launch.hpp"

namespace sy {

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;

// ------------------------------------------------------------------ RMSNorm
//
// out = x r w, r = 1 / sqrt(mean(x^2) + eps). One wave per token, the row in registers
// (VPL chunks a lane; chunks past the row read 0 and are not stored). rinv[tok]
// receives r for the backward when given.
template <class T, int VPL>
__global__ void __launch_bounds__(kBlock)
k_rms_norm(const typename T::storage* __restrict__ x, const typename T::storage* __restrict__ w,
           typename T::storage* __restrict__ out, float* __restrict__ rinv, int64_t n_tok, int d,
           float eps, float inv_d) {
  using S = typename T::storage;
  const int lane = threadIdx.x & 63;
  const uint32_t row_bytes = (uint32_t)d * sizeof(S);
  const auto wr = make_rsrc(w, row_bytes);
  for (int64_t tok = (int64_t)blockIdx.x * kWaves + wave_id(); tok < n_tok; tok += (int64_t)gridDim.x * kWaves) {
    const auto xr = make_rsrc(x + tok * d, row_bytes);
    i32x4_t v[VPL], g[VPL];
#pragma unroll
    for (int j = 0; j < VPL; ++j) v[j] = ld16_stream(xr, (lane + 64 * j) * 16u);
#pragma unroll
    for (int j = 0; j < VPL; ++j) g[j] = ld16(wr, (lane + 64 * j) * 16u);
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < VPL; ++j) ss = dot<T>(v[j], v[j], ss);
    const float r = rsqrtf(fmaf(wave_sum(ss), inv_d, eps));
    if (rinv != nullptr && lane == 0) rinv[tok] = r;
    const auto orr = make_rsrc(out + tok * d, row_bytes);
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      float f[T::ce];
#pragma unroll
      for (int e = 0; e < T::ce; ++e) f[e] = elem<T>(v[j], e) * r * elem<T>(g[j], e);
      st16(orr, (lane + 64 * j) * 16u, pack<T>(f));
    }
  }
}

// dx = r (g w) - x r^3 / D <g w, x>; dw += g x r. Persistent over tokens; each wave's
// dw stays in registers, the four are folded through LDS in wave order and the
// workgroup writes one fp32 partial row (summed by k_dw_reduce).
template <class T, int VPL>
__global__ void __launch_bounds__(kBlock)
k_rms_norm_bwd(const typename T::storage* __restrict__ x, const typename T::storage* __restrict__ w,
               const typename T::storage* __restrict__ go, const float* __restrict__ rinv,
               typename T::storage* __restrict__ dx, float* __restrict__ partial, int64_t n_tok, int d,
               float inv_d) {
  using S = typename T::storage;
  constexpr int CE = T::ce;
  __shared__ float fold[64][VPL * CE + 1];
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const uint32_t row_bytes = (uint32_t)d * sizeof(S);
  const auto wr = make_rsrc(w, row_bytes);
  i32x4_t wq[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) wq[j] = ld16(wr, (lane + 64 * j) * 16u);
  float dw[VPL][CE];
#pragma unroll
  for (int j = 0; j < VPL; ++j)
#pragma unroll
    for (int e = 0; e < CE; ++e) dw[j][e] = 0.0f;
  for (int64_t tok = (int64_t)blockIdx.x * kWaves + wave; tok < n_tok; tok += (int64_t)gridDim.x * kWaves) {
    const auto xr = make_rsrc(x + tok * d, row_bytes);
    const auto gr = make_rsrc(go + tok * d, row_bytes);
    i32x4_t v[VPL], g[VPL];
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      v[j] = ld16_stream(xr, (lane + 64 * j) * 16u);
      g[j] = ld16_stream(gr, (lane + 64 * j) * 16u);
    }
    const float r = rinv[tok];
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < VPL; ++j)
#pragma unroll
      for (int e = 0; e < CE; ++e) s = fmaf(elem<T>(g[j], e) * elem<T>(wq[j], e), elem<T>(v[j], e), s);
    const float c = wave_sum(s) * r * r * r * inv_d;
    const auto dr = make_rsrc(dx + tok * d, row_bytes);
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      float f[CE];
#pragma unroll
      for (int e = 0; e < CE; ++e) {
        const float xv = elem<T>(v[j], e), gv = elem<T>(g[j], e);
        f[e] = fmaf(r, gv * elem<T>(wq[j], e), -c * xv);
        dw[j][e] = fmaf(gv * r, xv, dw[j][e]);
      }
      st16(dr, (lane + 64 * j) * 16u, pack<T>(f));
    }
  }
#pragma unroll 1
  for (int k = 1; k < kWaves; ++k) {
    __syncthreads();
    if (wave == k) {
#pragma unroll
      for (int j = 0; j < VPL; ++j)
#pragma unroll
        for (int e = 0; e < CE; ++e) fold[lane][j * CE + e] = dw[j][e];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int j = 0; j < VPL; ++j)
#pragma unroll
        for (int e = 0; e < CE; ++e) dw[j][e] += fold[lane][j * CE + e];
    }
  }
  if (wave != 0) return;
  const auto pr = make_rsrc(partial + (int64_t)blockIdx.x * d, (uint32_t)d * 4u);
#pragma unroll
  for (int j = 0; j < VPL; ++j)
#pragma unroll
    for (int q = 0; q < CE / 4; ++q) {
      i32x4_t t;
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] = __float_as_int(dw[j][4 * q + e]);
      st16(pr, (uint32_t)(lane + 64 * j) * CE * 4u + q * 16u, t);
    }
}

// ------------------------------------------------------- rotary and QKV split
//
// qkv [B*T][3][H][hd] <-> q, k, v each [B][H][T][hd], with channel i of a head's first
// half turned with channel i of its second half by the angle of position t (q and k;
// v is moved only). BWD is the transpose: the gradients of q, k, v back into qkv's
// layout, turned the other way. A thread owns the two 16-byte chunks that turn
// together.
template <class T, bool BWD>
__global__ void __launch_bounds__(kBlock)
k_rope_qkv(typename T::storage* __restrict__ qkv, typename T::storage* __restrict__ q,
           typename T::storage* __restrict__ k, typename T::storage* __restrict__ v,
           const float* __restrict__ cosv, const float* __restrict__ sinv, int64_t n_tok, int seq,
           int heads, int hd) {
  using S = typename T::storage;
  constexpr int CE = T::ce;
  const int half = hd / 2;
  const int cpr = half / CE;  // chunk pairs of a head row
  const int64_t items = n_tok * 3 * heads * cpr;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < items; i += (int64_t)gridDim.x * kBlock) {
    const int c = (int)(i % cpr);
    const int64_t row = i / cpr;  // (token, which, head)
    const int h = (int)(row % heads);
    const int64_t tw = row / heads;
    const int which = (int)(tw % 3);
    const int64_t tok = tw / 3;
    const int64_t b = tok / seq;
    const int t = (int)(tok % seq);
    S* const packed = qkv + row * hd + c * CE;
    S* const split = (which == 0 ? q : which == 1 ? k : v) + ((b * heads + h) * seq + t) * hd + c * CE;
    S* const src = BWD ? split : packed;
    S* const dst = BWD ? packed : split;
    i32x4_t lo = *reinterpret_cast<const i32x4_t*>(src);
    i32x4_t hi = *reinterpret_cast<const i32x4_t*>(src + half);
    if (which < 2) {
      const float* const cp = cosv + (int64_t)t * half + c * CE;
      const float* const sp = sinv + (int64_t)t * half + c * CE;
      float a[CE], e2[CE];
#pragma unroll
      for (int e = 0; e < CE; ++e) {
        const float x = elem<T>(lo, e), y = elem<T>(hi, e);
        const float co = cp[e], si = BWD ? -sp[e] : sp[e];
        a[e] = x * co - y * si;
        e2[e] = x * si + y * co;
      }
      lo = pack<T>(a);
      hi = pack<T>(e2);
    }
    *reinterpret_cast<i32x4_t*>(dst) = lo;
    *reinterpret_cast<i32x4_t*>(dst + half) = hi;
  }
}

// ------------------------------------------------------------------- SwiGLU
//
// out = silu(gate) up over gate_up [n_tok][2 F] (gate first), and its gradient.
template <class T, bool BWD>
__global__ void __launch_bounds__(kBlock)
k_swiglu(const typename T::storage* __restrict__ gu, const typename T::storage* __restrict__ go,
         typename T::storage* __restrict__ out, int64_t n_tok, int f) {
  constexpr int CE = T::ce;
  const int cpr = f / CE;
  const int64_t items = n_tok * cpr;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < items; i += (int64_t)gridDim.x * kBlock) {
    const int64_t tok = i / cpr;
    const int64_t off = (int64_t)(i % cpr) * CE;
    const i32x4_t g = *reinterpret_cast<const i32x4_t*>(gu + tok * 2 * f + off);
    const i32x4_t u = *reinterpret_cast<const i32x4_t*>(gu + tok * 2 * f + f + off);
    float a[CE], b[CE];
    [[maybe_unused]] i32x4_t y;
    if constexpr (BWD) y = *reinterpret_cast<const i32x4_t*>(go + tok * f + off);
#pragma unroll
    for (int e = 0; e < CE; ++e) {
      const float gv = elem<T>(g, e), uv = elem<T>(u, e);
      const float sg = 1.0f / (1.0f + expf(-gv));
      if constexpr (BWD) {
        const float yv = elem<T>(y, e);
        a[e] = yv * uv * sg * (1.0f + gv * (1.0f - sg));
        b[e] = yv * gv * sg;
      } else {
        a[e] = gv * sg * uv;
      }
    }
    if constexpr (BWD) {
      *reinterpret_cast<i32x4_t*>(out + tok * 2 * f + off) = pack<T>(a);
      *reinterpret_cast<i32x4_t*>(out + tok * 2 * f + f + off) = pack<T>(b);
    } else {
      *reinterpret_cast<i32x4_t*>(out + tok * f + off) = pack<T>(a);
    }
  }
}

unsigned item_grid(int64_t items) {
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>((items + kBlock - 1) / kBlock, 65536));
}

int norm_slots(int64_t d, int ce) {
  const int64_t c = (d / ce + 63) / 64;
  return c <= 1 ? 1 : c <= 2 ? 2 : c <= 4 ? 4 : c <= 8 ? 8 : 0;
}

template <class T, int VPL>
hipError_t norm_t(const NormArgs& a, hipStream_t s) {
  using St = typename T::storage;
  const float inv_d = 1.0f / (float)a.d;
  if (a.go == nullptr) {
    // A workgroup for every four tokens, up to a grid that is a launch at any token count
    // (2^32 threads are none).
    const unsigned grid = (unsigned)std::min<int64_t>((a.n_tok + kWaves - 1) / kWaves, 1 << 20);
    hipLaunchKernelGGL((k_rms_norm<T, VPL>), dim3(grid), dim3(kBlock), 0, s, (const St*)a.x, (const St*)a.w,
                       (St*)a.out, a.rinv, a.n_tok, a.d, a.eps, inv_d);
  } else {
    hipLaunchKernelGGL((k_rms_norm_bwd<T, VPL>), dim3((unsigned)a.rows), dim3(kBlock), 0, s, (const St*)a.x,
                       (const St*)a.w, (const St*)a.go, a.rinv, (St*)a.out, a.partial, a.n_tok, a.d, inv_d);
  }
  return hipGetLastError();
}

template <class T>
hipError_t norm_slots_t(const NormArgs& a, hipStream_t s) {
  switch (norm_slots(a.d, T::ce)) {
    case 1: return norm_t<T, 1>(a, s);
    case 2: return norm_t<T, 2>(a, s);
    case 4: return norm_t<T, 4>(a, s);
    case 8: return norm_t<T, 8>(a, s);
    default: return hipErrorInvalidConfiguration;
  }
}

template <class T>
hipError_t rope_t(const RopeArgs& a, hipStream_t s) {
  using St = typename T::storage;
  const unsigned grid = item_grid(a.n_tok * 3 * a.heads * (a.hd / 2 / T::ce));
  if (a.backward)
    hipLaunchKernelGGL((k_rope_qkv<T, true>), dim3(grid), dim3(kBlock), 0, s, (St*)a.qkv, (St*)a.q, (St*)a.k,
                       (St*)a.v, a.cosv, a.sinv, a.n_tok, a.seq, a.heads, a.hd);
  else
    hipLaunchKernelGGL((k_rope_qkv<T, false>), dim3(grid), dim3(kBlock), 0, s, (St*)a.qkv, (St*)a.q, (St*)a.k,
                       (St*)a.v, a.cosv, a.sinv, a.n_tok, a.seq, a.heads, a.hd);
  return hipGetLastError();
}

template <class T>
hipError_t swiglu_t(const void* gu, const void* go, void* out, int64_t n_tok, int f, hipStream_t s) {
  using St = typename T::storage;
  const unsigned grid = item_grid(n_tok * (f / T::ce));
  if (go != nullptr)
    hipLaunchKernelGGL((k_swiglu<T, true>), dim3(grid), dim3(kBlock), 0, s, (const St*)gu, (const St*)go,
                       (St*)out, n_tok, f);
  else
    hipLaunchKernelGGL((k_swiglu<T, false>), dim3(grid), dim3(kBlock), 0, s, (const St*)gu, (const St*)go,
                       (St*)out, n_tok, f);
  return hipGetLastError();
}

}  // namespace

bool norm_fits(int64_t d, int dtype) {
  const int ce = dtype == SY_F32 ? 4 : 8;
  return d % ce == 0 && norm_slots(d, ce) != 0;
}

int norm_bwd_rows(int64_t n_tok) {
  int cus = 0;
  if (cu_count(&cus) != hipSuccess || cus < 1) cus = 1;
  return (int)std::max<int64_t>(1, std::min<int64_t>(cus, (n_tok + kWaves - 1) / kWaves));
}

hipError_t launch_rms_norm(const NormArgs& a, int dtype, hipStream_t s) {
  if (dtype == SY_BF16) return norm_slots_t<BF16>(a, s);
  if (dtype == SY_F16) return norm_slots_t<F16>(a, s);
  return norm_slots_t<F32>(a, s);
}

hipError_t launch_rope_qkv(const RopeArgs& a, int dtype, hipStream_t s) {
  if (dtype == SY_BF16) return rope_t<BF16>(a, s);
  if (dtype == SY_F16) return rope_t<F16>(a, s);
  return rope_t<F32>(a, s);
}

hipError_t launch_swiglu(const void* gu, const void* go, void* out, int64_t n_tok, int f, int dtype,
                         hipStream_t s) {
  if (dtype == SY_BF16) return swiglu_t<BF16>(gu, go, out, n_tok, f, s);
  if (dtype == SY_F16) return swiglu_t<F16>(gu, go, out, n_tok, f, s);
  return swiglu_t<F32>(gu, go, out, n_tok, f, s);
}

}  // namespace sy
