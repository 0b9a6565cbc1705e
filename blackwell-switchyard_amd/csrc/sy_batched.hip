// The batched operator for rows and counts that the matrix-core kernels of
// sy_matrix.hip do not take.
//
// Backward in two passes: any row of 16-byte chunks, 16-bit or fp32, up to
// 16 sources and 16 queries (the gradient's algebra is at k_bwd_batched_mx in
// sy_matrix.hip, whose single pass needs g, the queries and the sources of a token
// in one CU's LDS and serves 16-bit D <= 2048 with S <= 8).
//
//   k_bb_coef   per token: all dots <g_s, v_n> and <q_s, v_n> and the softmax
//               backward -> its coefficients alpha_sn, da_sn, c_n (1.2 KB at
//               N=9, S=8) in the workspace;
//   k_bb_apply  per token and column: dv_n = sum_s alpha_sn g_s + da_sn q_s + c_n v_n
//               and dq_s += sum_n da_sn v_n.
//
// v and g are read twice (43 slabs of [tokens, D] where one pass needs 26 at N=9,
// S=8), against the register tile's single pass with 18 wave reductions and a barrier
// a query and three VALU operations for every (query, source, element). N=9 S=8
// T=4096 D=4096 bf16: 574 us in one pass, 295 in two -- coefficients 130-145 (570 MB,
// 3.9-4.4 TB/s: 64-byte row pieces), apply 160-170 (885 MB, 5.2-5.5 TB/s), reduction 5.
//
// Reference: the batched forward is src/switchyard/triton_op.py:378-501; it has no
// backward (the single-query derivation is at :205-214).
#include <algorithm>
#include <type_traits>
#include <utility>

#include "sy_launch.hpp"

namespace sy {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kCoefWaves = 4;     // waves of a k_bb_coef workgroup
constexpr int kApplyBlock = 256;  // four waves

// Calls f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>): unrolled
// steps whose index is a constant expression (MFMA modifiers are immediates).
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// The coefficients of one token for NG groups of four sources and SG groups of four
// queries (floats): alpha[s][n], da[s][n], then da transposed [n][s], then c[n], each
// n running to 4 NG and s to 4 SG. Four consecutive values of a table are one A
// operand of k_bb_apply's products; entries past N or S are zero.
template <int NG, int SG>
struct Coef {
  static constexpr int kN = 4 * NG, kS = 4 * SG;
  static constexpr int kTable = kN * kS;
  static constexpr int kDa = kTable, kDaT = 2 * kTable, kC = 3 * kTable;
  static constexpr int kVgprs = (kC + kN + 63) / 64;
  static constexpr int kStride = 64 * kVgprs;  // floats per token
};

// acc + A B over one 16-byte chunk of each lane's row: rows lane % 16 of A (sources)
// and B (g / queries), the chunk of lane / 16. Any order of the columns serves, as
// both operands use the same one.
template <class T>
__device__ __forceinline__ f32x4_t mma(const i32x4_t& a, const i32x4_t& b, f32x4_t c) {
  if constexpr (T::code == BF16::code) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  } else if constexpr (T::code == F16::code) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  } else {
    // Four products of four from zero, added pairwise (add_batch says why).
    f32x4_t p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      p[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__int_as_float(a[j]), __int_as_float(b[j]),
                                                  f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
    return c + ((p[0] + p[1]) + (p[2] + p[3]));
  }
}

// U steps of products (and of the A rows' sums of squares) into two running sums each.
// 16-bit rows add step by step. fp32 rows, whose results are held to fp32 error, form
// every step from zero and add the steps pairwise: one running sum over a row rounds at
// every product of its chain (fp32 gradients, error against float64, N=11 S=4 T=1262
// D=1024: 2.2e-6 running, 1.1e-6 so and 1.1e-6 with a reduction over 64 lanes).
template <int U, class V>
__device__ __forceinline__ V tree_sum(V (&c)[U]) {
#pragma unroll
  for (int h = U / 2; h >= 1; h /= 2)
#pragma unroll
    for (int u = 0; u < h; ++u) c[u] = c[u] + c[u + h];
  return c[0];
}
template <class T, int U, bool TWO>
__device__ __forceinline__ void add_batch(const i32x4_t (&a)[U], const i32x4_t (&b)[U],
                                          const i32x4_t (&bq)[TWO ? U : 1], f32x4_t (&acc)[2],
                                          f32x4_t (&accq)[2], float (&ss)[2]) {
  if constexpr (T::code == F32::code) {
    f32x4_t c[U];
    float sq[U];
#pragma unroll
    for (int u = 0; u < U; ++u) sq[u] = dot<T>(a[u], a[u], 0.0f);
    ss[0] += tree_sum<U>(sq);
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] = mma<T>(a[u], b[u], f32x4_t{0.0f, 0.0f, 0.0f, 0.0f});
    acc[0] = acc[0] + tree_sum<U>(c);
    if constexpr (TWO) {
#pragma unroll
      for (int u = 0; u < U; ++u) c[u] = mma<T>(a[u], bq[u], f32x4_t{0.0f, 0.0f, 0.0f, 0.0f});
      accq[0] = accq[0] + tree_sum<U>(c);
    }
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      ss[u & 1] = dot<T>(a[u], a[u], ss[u & 1]);
      acc[u & 1] = mma<T>(a[u], b[u], acc[u & 1]);
      if constexpr (TWO) accq[u & 1] = mma<T>(a[u], bq[u], accq[u & 1]);
    }
  }
}

__device__ __forceinline__ float sum_groups(float x) {  // over the four 16-lane groups
  const uint32_t u = __float_as_uint(x);
  const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const uint32_t y = __float_as_uint(__uint_as_float(p[0]) + __uint_as_float(p[1]));
  const auto r = __builtin_amdgcn_permlane32_swap(y, y, false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float max_groups(float x) {
  const uint32_t u = __float_as_uint(x);
  const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const uint32_t y = __float_as_uint(fmaxf(__uint_as_float(p[0]), __uint_as_float(p[1])));
  const auto r = __builtin_amdgcn_permlane32_swap(y, y, false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// ------------------------------------------------------------- coefficients
//
// One token per workgroup of four waves, each a quarter of the columns. With at
// most 8 queries (SG <= 2) g and q share the 16 columns of one product, as in
// k_bwd_batched_mx; with up to 16 they are two products. Operands go from global
// memory straight into the MFMA registers: 16 rows x 64 bytes a load, no LDS. Rows
// past N or S repeat the last one (the same cache lines) and are masked in the
// softmax. Bound by HBM: v and g are read once, the queries come from L2. A batch of
// 256 columns (17 rows x 512 bytes at N=9, S=8) is in flight a wave.
template <class T, int NG, int SG, int W>
__global__ void __launch_bounds__(64 * kCoefWaves)
k_bb_coef(const RowTable v, const typename T::storage* __restrict__ q,
          const typename T::storage* __restrict__ g, float* __restrict__ coef, int n_src, int n_q,
          int64_t n_tok, int d, float eps, float inv_d) {
  using C = Coef<NG, SG>;
  constexpr bool TWO = SG > 2;
  constexpr int CE = T::ce;
  constexpr int kCols = 4 * CE;  // columns of a step
  constexpr int kU = TWO ? 4 : 8;  // steps of a batch
  constexpr int kTpb = kCoefWaves / W;  // tokens a workgroup takes at once
  static_assert(W == 1 || W == kCoefWaves, "a token is a wave's or a workgroup's");
  __shared__ __align__(16) float xl[TWO ? 2 : 1][W > 1 ? W : 1][64][4];
  __shared__ __align__(16) float xs[kTpb][W][16];
  const int lane = threadIdx.x & 63;
  const int slot = wave_id() / W;
  const int w = wave_id() % W;
  const int qi = lane & 15, grp = lane >> 4;
  using S = typename T::storage;
  const int64_t hop = (int64_t)gridDim.x * kTpb;
  for (int64_t tok = (int64_t)blockIdx.x * kTpb + slot; tok < n_tok; tok += hop) {
    const int rn = min(qi, n_src - 1);
    const S* pa = row_at<false, const S>(v, rn) + tok * d + grp * CE;
    // Column qi: g of query qi, or (SG <= 2) g of query qi < 8, then query qi - 8.
    const int sc = min(TWO ? qi : (qi & 7), n_q - 1);
    const S* pg = g + ((int64_t)sc * n_tok + tok) * d + grp * CE;
    const S* pq = q + (int64_t)sc * d + grp * CE;
    const S* pb = TWO || qi < 8 ? pg : pq;

    const int full = d / kCols;  // steps wholly inside the row
    const int beg = (int)((int64_t)full * w / W);
    const int end = (int)((int64_t)full * (w + 1) / W);
    f32x4_t acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    [[maybe_unused]] f32x4_t accq[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    float ss[2] = {0.0f, 0.0f};
    auto ld = [](const S* p) { return *reinterpret_cast<const i32x4_t*>(p); };
    int k = beg;
    for (; k + kU <= end; k += kU) {
      i32x4_t a[kU], b[kU];
      [[maybe_unused]] i32x4_t bq[TWO ? kU : 1];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        a[u] = ld(pa + (k + u) * kCols);
        b[u] = ld(pb + (k + u) * kCols);
        if constexpr (TWO) bq[u] = ld(pq + (k + u) * kCols);
      }
      add_batch<T, kU, TWO>(a, b, bq, acc, accq, ss);
    }
    // The rest of this wave's steps, and (last wave) the row's partial step.
    constexpr int kR = 4;
    const int stop = w == W - 1 ? (d + kCols - 1) / kCols : end;
    for (; k < stop; k += kR) {
      i32x4_t a[kR], b[kR];
      [[maybe_unused]] i32x4_t bq[TWO ? kR : 1];
#pragma unroll
      for (int u = 0; u < kR; ++u) {
        const bool in = k + u < stop && (k + u) * kCols + grp * CE < d;
        a[u] = b[u] = i32x4_t{0, 0, 0, 0};
        if constexpr (TWO) bq[u] = i32x4_t{0, 0, 0, 0};
        if (in) {
          a[u] = ld(pa + (k + u) * kCols);
          b[u] = ld(pb + (k + u) * kCols);
          if constexpr (TWO) bq[u] = ld(pq + (k + u) * kCols);
        }
      }
      add_batch<T, kR, TWO>(a, b, bq, acc, accq, ss);
    }
    f32x4_t lt = acc[0] + acc[1];
    [[maybe_unused]] f32x4_t lq = accq[0] + accq[1];
    const float sw = sum_groups(ss[0] + ss[1]);
    if (lane < 16) xs[slot][w][lane] = sw;
    if constexpr (W > 1) {
      *(f32x4_t*)&xl[0][w][lane][0] = lt;
      if constexpr (TWO) *(f32x4_t*)&xl[1][w][lane][0] = lq;
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    if (w == 0) {
      // Lane (grp, qi): rows n = 4 grp + j of column qi.
      f32x4_t sq = *(const f32x4_t*)&xs[slot][0][4 * grp];
#pragma unroll
      for (int ww = 1; ww < W; ++ww) {
        lt += *(const f32x4_t*)&xl[0][ww][lane][0];
        sq += *(const f32x4_t*)&xs[slot][ww][4 * grp];
        if constexpr (TWO) lq += *(const f32x4_t*)&xl[1][ww][lane][0];
      }
      const bool gl = TWO || qi < 8;           // this lane's column is G
      const int s = TWO ? qi : (qi & 7);       // its query
      const bool real_q = s < n_q;
      float G[4], lg[4], r[4];
      float mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float dotq;
        if constexpr (TWO) {
          G[j] = lt[j];
          dotq = lq[j];
        } else {
          const float o = dpp<0x128>(lt[j]);  // row_ror:8: the lane qi ^ 8 value
          G[j] = gl ? lt[j] : o;
          dotq = gl ? o : lt[j];
        }
        r[j] = rsqrtf(fmaf(sq[j], inv_d, eps));
        lg[j] = dotq * r[j];
        if (4 * grp + j < n_src) mx = fmaxf(mx, lg[j]);
      }
      mx = max_groups(mx);
      float p[4];
      int top = 64;  // first row at the maximum
#pragma unroll
      for (int j = 3; j >= 0; --j) {
        const bool real = 4 * grp + j < n_src;
        p[j] = real ? expf(lg[j] - mx) : 0.0f;
        if (real && lg[j] == mx) top = 4 * grp + j;
      }
      const float inv_l = 1.0f / sum_groups((p[0] + p[1]) + (p[2] + p[3]));
      top = (int)-max_groups(-(float)top);
      // The dots are taken relative to the top row's, as in the single-query backward.
      const int tj = top & 3;
      const float gsel = tj == 0 ? G[0] : tj == 1 ? G[1] : tj == 2 ? G[2] : G[3];
      const float gref = sum_groups(grp == ((top >> 2) & 3) ? gsel : 0.0f);
      float al[4], dg[4], sdev = 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        al[j] = p[j] * inv_l;
        dg[j] = 4 * grp + j < n_src ? G[j] - gref : 0.0f;
        sdev = fmaf(al[j], dg[j], sdev);
      }
      sdev = sum_groups(sdev);
      f32x4_t alv, dav, cv;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool real = real_q && 4 * grp + j < n_src;
        const float dl = al[j] * (dg[j] - sdev);
        alv[j] = real ? al[j] : 0.0f;
        dav[j] = real ? dl * r[j] : 0.0f;
        // c_n: sum over the queries (8 lanes: both halves of a row agree; or 16).
        float c = real ? -dl * lg[j] * (r[j] * r[j] * inv_d) : 0.0f;
        c += dpp<0xB1>(c);   // quad_perm [1,0,3,2]
        c += dpp<0x4E>(c);   // quad_perm [2,3,0,1]
        c += dpp<0x141>(c);  // row_half_mirror
        if constexpr (TWO) c += dpp<0x140>(c);  // row_mirror
        cv[j] = c;
      }
      float* const o = coef + tok * C::kStride;
      if (grp < NG && s < C::kS) {
        if (gl) *(f32x4_t*)(o + s * C::kN + 4 * grp) = alv;
        if (TWO || !gl) *(f32x4_t*)(o + C::kDa + s * C::kN + 4 * grp) = dav;
        if (gl) {
#pragma unroll
          for (int j = 0; j < 4; ++j) o[C::kDaT + (4 * grp + j) * C::kS + s] = dav[j];
        }
        if (qi == 0) *(f32x4_t*)(o + C::kC + 4 * grp) = cv;
      }
    }
    if constexpr (W > 1) {
      if (tok + hop < n_tok) __syncthreads();  // the exchange is rewritten
    } else {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// -------------------------------------------------------------------- apply
//
// The four waves of a workgroup own the same 64 chunks (one a lane) of every row
// and take the workgroup's tokens in turn, independently. The coefficients of a
// token are a few VGPRs, one value a lane, and the sums over queries and sources run
// on v_mfma_f32_4x4x1: 16 blocks of 4 lanes, where a lane's column is its own
// element of a g, q or v row, and the A operand -- four coefficients, broadcast to
// all blocks from block ABID of one of those VGPRs (CBSZ = 4) -- covers four
// outputs. So four multiply-adds a lane in two passes, with exact fp32
// coefficients and widened elements, and no lane ever needs another lane's data:
// rows enter and leave as whole 16-byte chunks. (As VALU FMAs the same sums take
// twice the cycles and 153 live coefficients.) dv overwrites the source's chunk
// dword by dword and is stored row by row. dq stays in registers for the kernel;
// the four waves' sums are folded through LDS in wave order, one partial row per
// query and workgroup, reduced afterwards in a fixed order.
// NR >= n_src compile-time rows, SG = ceil(n_q / 4) (1, 2 or 4) query groups.
template <class T, int NR, int SG>
__global__ void __launch_bounds__(kApplyBlock, NR <= 9 && SG <= 2 ? 2 : 1)
k_bb_apply(const RowTable v, const typename T::storage* __restrict__ q,
           const typename T::storage* __restrict__ g, const float* __restrict__ coef,
           const RowTable dv, float* __restrict__ partial, int n_src, int n_q, int64_t n_tok, int d,
           int slices, int groups) {
  constexpr int NG = (NR + 3) / 4;
  using C = Coef<NG, SG>;
  using S = typename T::storage;
  constexpr int CE = T::ce;
  constexpr int SQ = 4 * SG;
  constexpr int kEpd = CE / 4;  // elements of a dword
  constexpr int kWaves = kApplyBlock / 64;
  __shared__ float fold[64][CE * SQ + 1];
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int slice = (int)blockIdx.x % slices, group = (int)blockIdx.x / slices;
  const uint32_t row_bytes = (uint32_t)d * sizeof(S);
  const uint32_t off = (uint32_t)(slice * 64 + lane) * 16u;

  i32x4_t qq[SQ];
#pragma unroll
  for (int s = 0; s < SQ; ++s)
    qq[s] = ld16(make_rsrc(q + (int64_t)(s < n_q ? s : 0) * d, s < n_q ? row_bytes : 0u), off);
  f32x4_t dq[CE][SG];
#pragma unroll
  for (int e = 0; e < CE; ++e)
#pragma unroll
    for (int k = 0; k < SG; ++k) dq[e][k] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  for (int64_t tok = (int64_t)group * kWaves + wave; tok < n_tok; tok += (int64_t)groups * kWaves) {
    // Opaque each token: the queries' widened values (twice the registers) would
    // otherwise be held across the loop.
#pragma unroll
    for (int s = 0; s < SQ; ++s) asm volatile("" : "+v"(qq[s]));
    float cf[C::kVgprs];
#pragma unroll
    for (int k = 0; k < C::kVgprs; ++k) cf[k] = coef[tok * C::kStride + 64 * k + lane];
    i32x4_t x[NR], gg[SQ];
#pragma unroll
    for (int n = 0; n < NR; ++n)
      x[n] = ld16_stream(make_rsrc(row_at<false, const S>(v, n < n_src ? n : 0) + tok * d,
                                   n < n_src ? row_bytes : 0u), off);
#pragma unroll
    for (int s = 0; s < SQ; ++s)
      gg[s] = ld16_stream(make_rsrc(g + ((int64_t)(s < n_q ? s : 0) * n_tok + tok) * d,
                                    s < n_q ? row_bytes : 0u), off);
    float cn[NR];
    static_for<NR>([&](auto I) {
      constexpr int i = C::kC + I.value;
      cn[I.value] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cf[i / 64]), i % 64));
    });
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float res[NR][2];
#pragma unroll
      for (int h = 0; h < kEpd; ++h) {
        const int e = k * kEpd + h;
        f32x4_t acc[NG];
#pragma unroll
        for (int a = 0; a < NG; ++a) acc[a] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        float xe[NR];
#pragma unroll
        for (int n = 0; n < NR; ++n) {
          xe[n] = elem<T>(x[n], e);
          acc[n / 4][n % 4] = cn[n] * xe[n];
        }
        static_for<SQ>([&](auto SI) {
          const float ge = elem<T>(gg[SI.value], e), qe = elem<T>(qq[SI.value], e);
          static_for<NG>([&](auto AI) {
            constexpr int ia = SI.value * NG + AI.value;  // operand of alpha[s][4a..]
            constexpr int id = C::kDa / 4 + ia;
            acc[AI.value] = __builtin_amdgcn_mfma_f32_4x4x1f32(cf[ia / 16], ge, acc[AI.value], 4, ia % 16, 0);
            acc[AI.value] = __builtin_amdgcn_mfma_f32_4x4x1f32(cf[id / 16], qe, acc[AI.value], 4, id % 16, 0);
          });
        });
        // fp32: a token's share from zero, so that the running sum rounds once a token.
        f32x4_t part[SG];
#pragma unroll
        for (int a = 0; a < SG; ++a)
          part[a] = T::code == F32::code ? f32x4_t{0.0f, 0.0f, 0.0f, 0.0f} : dq[e][a];
        static_for<NR>([&](auto NI) {
          static_for<SG>([&](auto KI) {
            constexpr int it = C::kDaT / 4 + NI.value * SG + KI.value;  // da[4k..][n]
            part[KI.value] =
                __builtin_amdgcn_mfma_f32_4x4x1f32(cf[it / 16], xe[NI.value], part[KI.value], 4, it % 16, 0);
          });
        });
#pragma unroll
        for (int a = 0; a < SG; ++a) dq[e][a] = T::code == F32::code ? dq[e][a] + part[a] : part[a];
#pragma unroll
        for (int n = 0; n < NR; ++n) res[n][h] = acc[n / 4][n % 4];
      }
#pragma unroll
      for (int n = 0; n < NR; ++n) {
        if constexpr (T::code == F32::code) {
          x[n][k] = __float_as_int(res[n][0]);
        } else {
          const f32x2_t two = {res[n][0], res[n][1]};
          if constexpr (T::code == BF16::code)
            x[n][k] = __builtin_bit_cast(int, __builtin_convertvector(two, bf16x2_t));
          else
            x[n][k] = __builtin_bit_cast(int, __builtin_convertvector(two, f16x2_t));
        }
      }
    }
#pragma unroll
    for (int n = 0; n < NR; ++n)
      st16_stream(make_rsrc(row_at<false, S>(dv, n < n_src ? n : 0) + tok * d,
                            n < n_src ? row_bytes : 0u), off, x[n]);
  }

  // The waves' dq in wave order, then one partial row a query.
#pragma unroll 1
  for (int k = 1; k < kWaves; ++k) {
    __syncthreads();
    if (wave == k) {
#pragma unroll
      for (int e = 0; e < CE; ++e)
#pragma unroll
        for (int s = 0; s < SQ; ++s) fold[lane][e * SQ + s] = dq[e][s / 4][s % 4];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int e = 0; e < CE; ++e)
#pragma unroll
        for (int s = 0; s < SQ; ++s) dq[e][s / 4][s % 4] += fold[lane][e * SQ + s];
    }
  }
  if (wave != 0) return;
#pragma unroll
  for (int s = 0; s < SQ; ++s) {
    const auto pr = make_rsrc(partial + ((int64_t)group * n_q + (s < n_q ? s : 0)) * d,
                              s < n_q ? (uint32_t)d * 4u : 0u);
#pragma unroll
    for (int c = 0; c < CE / 4; ++c) {
      i32x4_t t;
#pragma unroll
      for (int j = 0; j < 4; ++j) t[j] = __float_as_int(dq[4 * c + j][s / 4][s % 4]);
      st16(pr, off / 16u * (CE * 4u) + c * 16u, t);
    }
  }
}

// ------------------------------------------------------------------ forward
//
// S <= 16 queries, N <= NR sources, rows of any start and of at least one chunk. A
// token is a workgroup's (W = 4: each wave a quarter of the columns) or a wave's
// (W = 1). First the logits, straight from memory on MFMA as in k_bb_coef (queries as
// B), summed over the waves through LDS; every wave then forms the softmax and keeps
// the token's weights [n][s] as A operands, one value a lane, and in a second walk over
// the token's rows out_s = sum_n P_sn v_n on v_mfma_f32_4x4x1 as in k_bb_apply: whole
// chunks in and out, exact fp32 weights. Memory-bound: the second walk finds part of the
// rows in L2 and the rest in the last-level cache (N=12 S=8 T=4096 D=1280: 1.6 times the
// rows' bytes pass the L2); the register tile computes S dots and S sums a row on the VALU.
// bf16 T=4096: N=9 S=8 D=1280 74 -> 62 us, D=2560 144 -> 108; N=12 S=8 D=1280 159 (a
// launch a query) -> 64; N=9 S=8 T=1023 D=777 195 -> 17.5. Its two walks do not
// overlap within a wave, which leaves it at 1.5-1.8x the bytes' time.
template <class T, int NR, int SG, int W>
__global__ void __launch_bounds__(64 * kCoefWaves)
k_batched_any(const RowTable v, const typename T::storage* __restrict__ q,
              typename T::storage* __restrict__ out, float* __restrict__ m_out,
              float* __restrict__ l_out, int normalize, int n_src, int n_q, int64_t n_tok, int d,
              float eps, float inv_d) {
  using S = typename T::storage;
  constexpr int CE = T::ce;
  constexpr int NG = (NR + 3) / 4, kS = 4 * SG;
  constexpr int kCols = 4 * CE;  // columns of a logit step
  constexpr int kU = 4;
  constexpr int kTpb = kCoefWaves / W;
  constexpr int kVgprs = (4 * NG * kS + 63) / 64;
  constexpr int kEpd = CE / 4;
  __shared__ __align__(16) float xl[W > 1 ? W : 1][64][4];
  __shared__ __align__(16) float xs[kTpb][W][16];
  __shared__ __align__(16) float tab[kCoefWaves][64 * kVgprs];
  const int lane = threadIdx.x & 63;
  const int wave = wave_id();
  const int slot = wave / W, w = wave % W;
  const int qi = lane & 15, grp = lane >> 4;
  const uint32_t row_bytes = (uint32_t)d * sizeof(S);
  using any_t = std::conditional_t<sizeof(S) == 4, i32x4_f32_t, i32x4_any_t>;
  const int64_t hop = (int64_t)gridDim.x * kTpb;
  for (int64_t tok = (int64_t)blockIdx.x * kTpb + slot; tok < n_tok; tok += hop) {
    // 1. Logit and sum-of-squares partials over this wave's columns.
    const S* pa = row_of<const S>(v, min(qi, n_src - 1)) + tok * d + grp * CE;
    const S* pb = q + (int64_t)min(qi, n_q - 1) * d + grp * CE;
    const int full = d / kCols;
    const int beg = (int)((int64_t)full * w / W), end = (int)((int64_t)full * (w + 1) / W);
    f32x4_t acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
    f32x4_t accn[2];     // one group of queries: no second product
    const i32x4_t none[1] = {};
    float ss[2] = {0.0f, 0.0f};
    auto ld = [](const S* p) { return (i32x4_t)*reinterpret_cast<const any_t*>(p); };
    int k = beg;
    for (; k < end; k += kU) {
      i32x4_t a[kU], b[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        a[u] = b[u] = i32x4_t{0, 0, 0, 0};
        if (k + u < end) {
          a[u] = ld(pa + (k + u) * kCols);
          b[u] = ld(pb + (k + u) * kCols);
        }
      }
      add_batch<T, kU, false>(a, b, none, acc, accn, ss);
    }
    if (w == W - 1 && full * kCols < d) {
      // The row's partial step: a partial chunk is read back to end with the row, less
      // the elements the chunk before it holds.
      const int c0 = full * kCols + grp * CE;  // this lane's first column
      i32x4_t a = {0, 0, 0, 0}, b = {0, 0, 0, 0};
      if (c0 < d) {
        const int back = max(0, c0 + CE - d);
        a = ld(pa + full * kCols - back) & tail_mask((uint32_t)c0 * sizeof(S), row_bytes);
        b = ld(pb + full * kCols - back);
        if (back > 0) b = b & tail_mask((uint32_t)c0 * sizeof(S), row_bytes);
      }
      ss[0] = dot<T>(a, a, ss[0]);
      acc[0] = mma<T>(a, b, acc[0]);
    }
    f32x4_t lt = acc[0] + acc[1];
    const float sw = sum_groups(ss[0] + ss[1]);
    if (lane < 16) xs[slot][w][lane] = sw;
    if constexpr (W > 1) {
      *(f32x4_t*)&xl[w][lane][0] = lt;
      __syncthreads();
      lt = *(const f32x4_t*)&xl[0][lane][0];
    } else {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    f32x4_t sq = *(const f32x4_t*)&xs[slot][0][4 * grp];
#pragma unroll
    for (int ww = 1; ww < W; ++ww) {
      lt += *(const f32x4_t*)&xl[ww][lane][0];
      sq += *(const f32x4_t*)&xs[slot][ww][4 * grp];
    }

    // 2. Softmax of query qi over rows n = 4 grp + j; the weights as a table [n][s].
    float lg[4], p[4], mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      lg[j] = lt[j] * rsqrtf(fmaf(sq[j], inv_d, eps));
      if (4 * grp + j < n_src) mx = fmaxf(mx, lg[j]);
    }
    mx = max_groups(mx);
#pragma unroll
    for (int j = 0; j < 4; ++j) p[j] = 4 * grp + j < n_src ? expf(lg[j] - mx) : 0.0f;
    const float l = sum_groups((p[0] + p[1]) + (p[2] + p[3]));
    if (m_out != nullptr && w == 0 && grp == 0 && qi < n_q) {
      m_out[(int64_t)qi * n_tok + tok] = mx;
      l_out[(int64_t)qi * n_tok + tok] = l;
    }
    const float inv_l = normalize ? 1.0f / l : 1.0f;
    if (grp < NG && qi < kS) {
#pragma unroll
      for (int j = 0; j < 4; ++j) tab[wave][(4 * grp + j) * kS + qi] = p[j] * inv_l;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float cf[kVgprs];
#pragma unroll
    for (int i = 0; i < kVgprs; ++i) cf[i] = tab[wave][64 * i + lane];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();

    // 3. The outputs, 64 chunks a wave at a time.
    for (uint32_t base = (uint32_t)w * 1024u; base < row_bytes; base += 1024u * W) {
      const uint32_t off = base + lane * 16u;
      i32x4_t x[NR];
#pragma unroll
      for (int n = 0; n < NR; ++n) {
        x[n] = i32x4_t{0, 0, 0, 0};
        if (n < n_src) x[n] = ld_row<true>(row_of<const S>(v, n) + tok * d, row_bytes, off);
      }
      i32x4_t o[kS];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        float res[kS][2];
#pragma unroll
        for (int h = 0; h < kEpd; ++h) {
          f32x4_t y[SG];
#pragma unroll
          for (int g = 0; g < SG; ++g) y[g] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
          static_for<NR>([&](auto NI) {
            const float xe = elem<T>(x[NI.value], kk * kEpd + h);
            static_for<SG>([&](auto GI) {
              constexpr int op = NI.value * SG + GI.value;
              y[GI.value] = __builtin_amdgcn_mfma_f32_4x4x1f32(cf[op / 16], xe, y[GI.value], 4, op % 16, 0);
            });
          });
#pragma unroll
          for (int s = 0; s < kS; ++s) res[s][h] = y[s / 4][s % 4];
        }
#pragma unroll
        for (int s = 0; s < kS; ++s) {
          if constexpr (T::code == F32::code) {
            o[s][kk] = __float_as_int(res[s][0]);
          } else {
            const f32x2_t two = {res[s][0], res[s][1]};
            if constexpr (T::code == BF16::code)
              o[s][kk] = __builtin_bit_cast(int, __builtin_convertvector(two, bf16x2_t));
            else
              o[s][kk] = __builtin_bit_cast(int, __builtin_convertvector(two, f16x2_t));
          }
        }
      }
#pragma unroll
      for (int s = 0; s < kS; ++s)
        if (s < n_q)
          st_row<true, 0>(out + ((int64_t)s * n_tok + tok) * d, row_bytes, off, true, o[s]);
    }
    if constexpr (W > 1) {
      if (tok + hop < n_tok) __syncthreads();  // the exchange is rewritten
    }
  }
}

// ------------------------------------------------------------------- launch

template <class T, int NR, int SG>
hipError_t two_pass(const BwdBatchedArgs* a, const TwoPass& want, hipStream_t s, TwoPass* info) {
  constexpr int NG = (NR + 3) / 4;
  using C = Coef<NG, SG>;
  using St = typename T::storage;
  if (info != nullptr) {
    static hipFuncAttributes fa;
    static const hipError_t err =
        hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(k_bb_apply<T, NR, SG>));
    if (err != hipSuccess) return err;
    const int alloc = std::max(8, (fa.numRegs + 7) / 8 * 8);
    info->waves_per_simd = std::max(1, std::min(8, 512 / alloc));
    info->coef_stride = C::kStride;
    return hipSuccess;
  }
  // A wave per token (no exchange, four tokens a workgroup) once the device is full
  // of them and a token's chain of products is short; else four waves. N=9, backward,
  // us, four waves -> one: bf16 T=8192 D=256 S=8 67.6 -> 64.3, D=1280 205.9 -> 200.5;
  // T=64 D=1280 19.2 -> 23.5; T=4096 D=4096 (this kernel) 130 -> 147; fp32 T=1024
  // D=1024 S=8 47.0 -> 57.7.
  int cus = 0;
  if (cu_count(&cus) != hipSuccess || cus < 1) cus = 1;
  const int products = a->d / (a->dtype == SY_F32 ? 4 : 32);
  const bool wave_token = a->n_tok >= 4 * (int64_t)cus && products <= 64;
  const int tpb = wave_token ? kCoefWaves : 1;
  const dim3 grid((unsigned)std::min<int64_t>((a->n_tok + tpb - 1) / tpb, 1 << 20));
  if (wave_token)
    hipLaunchKernelGGL((k_bb_coef<T, NG, SG, 1>), grid, dim3(64 * kCoefWaves), 0, s, a->v,
                       (const St*)a->q, (const St*)a->g, want.coef, a->n_src, a->n_q, a->n_tok, a->d,
                       a->eps, 1.0f / (float)a->d);
  else
    hipLaunchKernelGGL((k_bb_coef<T, NG, SG, kCoefWaves>), grid, dim3(64 * kCoefWaves), 0, s, a->v,
                       (const St*)a->q, (const St*)a->g, want.coef, a->n_src, a->n_q, a->n_tok, a->d,
                       a->eps, 1.0f / (float)a->d);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_bb_apply<T, NR, SG>), dim3((unsigned)(want.slices * want.groups)), dim3(kApplyBlock), 0, s,
                     a->v, (const St*)a->q, (const St*)a->g, want.coef, a->dv, a->partial, a->n_src,
                     a->n_q, a->n_tok, a->d, want.slices, want.groups);
  return hipGetLastError();
}

template <class T, int NR>
hipError_t two_pass_q(int n_q, const BwdBatchedArgs* a, const TwoPass& t, hipStream_t s, TwoPass* info) {
  if (n_q <= 4) return two_pass<T, NR, 1>(a, t, s, info);
  if (n_q <= 8) return two_pass<T, NR, 2>(a, t, s, info);
  return two_pass<T, NR, 4>(a, t, s, info);
}

template <class T>
hipError_t two_pass_n(int n_src, int n_q, const BwdBatchedArgs* a, const TwoPass& t, hipStream_t s,
                      TwoPass* info) {
  if (n_src <= 4) return two_pass_q<T, 4>(n_q, a, t, s, info);
  if (n_src <= 9) return two_pass_q<T, 9>(n_q, a, t, s, info);
  return two_pass_q<T, 16>(n_q, a, t, s, info);
}

hipError_t two_pass_t(int dtype, int n_src, int n_q, const BwdBatchedArgs* a, const TwoPass& t,
                      hipStream_t s, TwoPass* info) {
  if (dtype == SY_BF16) return two_pass_n<BF16>(n_src, n_q, a, t, s, info);
  if (dtype == SY_F16) return two_pass_n<F16>(n_src, n_q, a, t, s, info);
  return two_pass_n<F32>(n_src, n_q, a, t, s, info);
}

template <class T, int NR, int SG>
hipError_t any_w(const BatchedArgs& a, hipStream_t s) {
  using St = typename T::storage;
  // A wave per token once the device is full of them and a row is at most four
  // 64-chunk walks; else four waves share it. bf16, us, four waves -> one: N=9 S=8
  // T=8192 D=256 52.1 -> 25.9, T=4096 D=768 44.3 -> 35.9, N=12 D=1280 87.0 -> 63.6;
  // N=9 D=2560 108 -> 117, T=64 D=1280 7.2 -> 13.9.
  int cus = 0;
  if (cu_count(&cus) != hipSuccess || cus < 1) cus = 1;
  const bool wave_token = a.n_tok >= 4 * (int64_t)cus && a.d <= 256 * T::ce;
  const int tpb = wave_token ? kCoefWaves : 1;
  const dim3 grid((unsigned)std::min<int64_t>((a.n_tok + tpb - 1) / tpb, 1 << 20));
  const float inv_d = 1.0f / (float)a.d;
  if (wave_token)
    hipLaunchKernelGGL((k_batched_any<T, NR, SG, 1>), grid, dim3(64 * kCoefWaves), 0, s, a.v, (const St*)a.q,
                       (St*)a.out, a.m_out, a.l_out, a.normalize, a.n_src, a.n_q, a.n_tok, a.d, a.eps, inv_d);
  else
    hipLaunchKernelGGL((k_batched_any<T, NR, SG, kCoefWaves>), grid, dim3(64 * kCoefWaves), 0, s, a.v,
                       (const St*)a.q, (St*)a.out, a.m_out, a.l_out, a.normalize, a.n_src, a.n_q, a.n_tok,
                       a.d, a.eps, inv_d);
  return hipGetLastError();
}

template <class T, int NR>
hipError_t any_q(const BatchedArgs& a, hipStream_t s) {
  if (a.n_q <= 4) return any_w<T, NR, 1>(a, s);
  if (a.n_q <= 8) return any_w<T, NR, 2>(a, s);
  return any_w<T, NR, 4>(a, s);
}

template <class T>
hipError_t any_n(const BatchedArgs& a, hipStream_t s) {
  if (a.n_src <= 4) return any_q<T, 4>(a, s);
  if (a.n_src <= 9) return any_q<T, 9>(a, s);
  return any_q<T, 16>(a, s);
}

}  // namespace

hipError_t launch_batched_any(const BatchedArgs& a, hipStream_t s) {
  if (!batched_any_fits(a.n_src, a.n_q, a.d, a.dtype)) return hipErrorInvalidConfiguration;
  if (a.n_tok == 0) return hipSuccess;
  if (a.dtype == SY_BF16) return any_n<BF16>(a, s);
  if (a.dtype == SY_F16) return any_n<F16>(a, s);
  return any_n<F32>(a, s);
}

hipError_t two_pass_shape(int64_t n_src, int64_t n_q, int64_t n_tok, int64_t d, int dtype, TwoPass* out) {
  hipError_t e = two_pass_t(dtype, (int)n_src, (int)n_q, nullptr, *out, nullptr, out);
  if (e != hipSuccess) return e;
  int cus = 0;
  e = cu_count(&cus);
  if (e != hipSuccess) return e;
  const int64_t chunks = d / (dtype == SY_F32 ? 4 : 8);
  out->slices = (int)((chunks + 63) / 64);
  // A workgroup for every four wave slots of the device, while each wave has a token.
  const int64_t groups = std::min<int64_t>((int64_t)cus * out->waves_per_simd / out->slices, (n_tok + 3) / 4);
  out->groups = (int)std::max<int64_t>(1, groups);
  return hipSuccess;
}

hipError_t launch_bwd_two_pass(const BwdBatchedArgs& a, const TwoPass& t, hipStream_t s) {
  if (!two_pass_fits(a.n_src, a.n_q, a.d, a.dtype) || t.coef == nullptr || t.groups < 1)
    return hipErrorInvalidConfiguration;
  if (a.n_tok == 0) return hipSuccess;
  return two_pass_t(a.dtype, a.n_src, a.n_q, &a, t, s, nullptr);
}

}  // namespace sy
