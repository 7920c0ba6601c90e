// Router projection: logits [m, e] fp32 = x [m, h] . W [e, h]^T, the
// F.linear(x.float(), W.float()) at the head of Router.forward
// (model/layers.py:128) and Gate.forward (.mosaicvm/source/inference_model.py:570).
//
// Each logit is defined as the exact dot product rounded once to fp32: the
// products of fp32 (or bf16) inputs are exact in fp64, and the kernel sums
// them in fp64 (in a fixed order, so the result is reproducible) before one
// rounding to fp32.  The fp64 sum is within n * 2^-53 * sum|terms| of the
// exact one, so the fp32 result is the correctly rounded exact dot unless the
// exact value lies that close to a rounding boundary.  Routing keys therefore
// do not depend on a summation order.
//
// Two kernels: a thread-per-element one for few tokens or ragged rows
// (router_logits_kernel), and one on the fp64 matrix unit for the rest
// (router_mfma_kernel).
#include <hip/hip_runtime.h>

#include "../../include/mosaic_amd.h"
#include "common.h"

namespace mosaic {
namespace {

template <typename T>
__device__ __forceinline__ double load_f64(const T* p, int64_t i);
template <>
__device__ __forceinline__ double load_f64<uint16_t>(const uint16_t* p, int64_t i) {
  return (double)bf16_f32(p[i]);
}
template <>
__device__ __forceinline__ double load_f64<float>(const float* p, int64_t i) {
  return (double)p[i];
}

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Few tokens: a workgroup of 256 threads owns ET experts x MT tokens; every
// thread strides over h and keeps MT x ET fp64 partial sums, which a
// wave-level then cross-wave reduction folds.  The weight is the HBM stream
// (e x h, read once per token tile); x rows are re-read from L2 by the
// workgroups of other experts.
template <typename TX, typename TW, int MT, int ET>
__global__ void __launch_bounds__(256) router_logits_kernel(const TX* __restrict__ x, const TW* __restrict__ w,
                                                            float* __restrict__ logits, int M, int E, int H) {
  __shared__ double s_part[4][MT * ET];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int e0 = blockIdx.x * ET, m0 = blockIdx.y * MT;
  double acc[MT][ET];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < ET; ++j) acc[i][j] = 0.0;
  for (int h = tid; h < H; h += 256) {
    double wv[ET];
#pragma unroll
    for (int j = 0; j < ET; ++j) wv[j] = (e0 + j < E) ? load_f64(w, (int64_t)(e0 + j) * H + h) : 0.0;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const double xv = (m0 + i < M) ? load_f64(x, (int64_t)(m0 + i) * H + h) : 0.0;
#pragma unroll
      for (int j = 0; j < ET; ++j) acc[i][j] = fma(xv, wv[j], acc[i][j]);  // the product is exact
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < ET; ++j) {
      const double s = wave_sum_f64(acc[i][j]);
      if (lane == 0) s_part[wave][i * ET + j] = s;
    }
  __syncthreads();
  if (tid < MT * ET) {
    const int i = tid / ET, j = tid % ET;
    const double s = ((s_part[0][tid] + s_part[1][tid]) + s_part[2][tid]) + s_part[3][tid];
    if (m0 + i < M && e0 + j < E) logits[(int64_t)(m0 + i) * E + e0 + j] = (float)s;
  }
}

typedef double f64x4_t __attribute__((ext_vector_type(4)));

// 8 consecutive elements of a row, converted to fp64 one at a time
template <typename T>
struct Row8;
template <>
struct Row8<uint16_t> {
  u32x4_t v;
  __device__ __forceinline__ void load(const uint16_t* p) { v = *reinterpret_cast<const u32x4_t*>(p); }
  __device__ __forceinline__ double get(int i) const {
    return (double)__uint_as_float((i & 1) ? v[i >> 1] & 0xFFFF0000u : v[i >> 1] << 16);
  }
};
template <>
struct Row8<float> {
  f32x4_t v[2];
  __device__ __forceinline__ void load(const float* p) {
    v[0] = *reinterpret_cast<const f32x4_t*>(p);
    v[1] = *reinterpret_cast<const f32x4_t*>(p + 4);
  }
  __device__ __forceinline__ double get(int i) const { return (double)v[i >> 2][i & 3]; }
};

// Many tokens: v_mfma_f64_16x16x4.  A wave owns 16 MT tokens x 16 ET experts
// over the 32-element chunks ks, ks + KS, ... of h; the KS waves of a workgroup
// meet in LDS and are added in wave order.  Lane (g = lane / 16, c = lane % 16)
// holds elements 8 g .. 8 g + 7 of a chunk of token row and expert row c (one
// 64- or 128-byte run per row), and product step i of the chunk multiplies
// element 8 g + i of both, so every element pairs once.  D: token row
// g + 4 r, expert c.  The next chunk's rows are loaded while this one is
// multiplied.  Rows past M or E repeat the last row and are not stored.
template <typename TX, typename TW, int MT, int ET, int KS>
__global__ void __launch_bounds__(64 * KS) router_mfma_kernel(const TX* __restrict__ x, const TW* __restrict__ w,
                                                              float* __restrict__ logits, int M, int E, int H) {
  __shared__ double part[KS][MT * ET][64];
  const int lane = threadIdx.x & 63, ks = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
  const int e0 = blockIdx.x * 16 * ET, m0 = blockIdx.y * 16 * MT;
  const TX* xr[MT];
  const TW* wr[ET];
#pragma unroll
  for (int i = 0; i < MT; ++i) xr[i] = x + (int64_t)min(m0 + 16 * i + c, M - 1) * H + 8 * g;
#pragma unroll
  for (int j = 0; j < ET; ++j) wr[j] = w + (int64_t)min(e0 + 16 * j + c, E - 1) * H + 8 * g;
  f64x4_t acc[MT][ET];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < ET; ++j) acc[i][j] = f64x4_t{0.0, 0.0, 0.0, 0.0};
  const int nch = H / 32;
  Row8<TX> xv[2][MT];
  Row8<TW> wv[2][ET];
  auto load = [&](int s, int ch) {
    const int o = 32 * min(ch, nch - 1);
#pragma unroll
    for (int i = 0; i < MT; ++i) xv[s][i].load(xr[i] + o);
#pragma unroll
    for (int j = 0; j < ET; ++j) wv[s][j].load(wr[j] + o);
  };
  auto compute = [&](int s) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      double b[ET];
#pragma unroll
      for (int j = 0; j < ET; ++j) b[j] = wv[s][j].get(k);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const double a = xv[s][i].get(k);
#pragma unroll
        for (int j = 0; j < ET; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b[j], acc[i][j], 0, 0, 0);
      }
    }
  };
  if (ks < nch) {
    load(0, ks);
    for (int ch = ks; ch < nch; ch += 2 * KS) {
      load(1, ch + KS);
      compute(0);
      if (ch + KS >= nch) break;
      load(0, ch + 2 * KS);
      compute(1);
    }
  }
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < ET; ++j) part[ks][i * ET + j][lane] = acc[i][j][r];
    __syncthreads();
    for (int o = threadIdx.x; o < MT * ET * 64; o += 64 * KS) {
      const int t = o >> 6, ln = o & 63;
      double s = part[0][t][ln];
#pragma unroll
      for (int k = 1; k < KS; ++k) s += part[k][t][ln];
      const int m = m0 + 16 * (t / ET) + (ln >> 4) + 4 * r, e = e0 + 16 * (t % ET) + (ln & 15);
      if (m < M && e < E) logits[(int64_t)m * E + e] = (float)s;
    }
    __syncthreads();
  }
}

template <int MT, int ET, int KS, typename TX, typename TW>
void launch_router_mfma(const TX* x, const TW* w, float* logits, int64_t m, int64_t e, int64_t h, hipStream_t st) {
  MOSAIC_LAUNCH((router_mfma_kernel<TX, TW, MT, ET, KS>),
                dim3((unsigned)((e + 16 * ET - 1) / (16 * ET)), (unsigned)((m + 16 * MT - 1) / (16 * MT))),
                dim3(64 * KS), 0, st, x, w, logits, (int)m, (int)e, (int)h);
}

template <typename TX, typename TW>
void launch_router(const void* x, const void* w, float* logits, int64_t m, int64_t e, int64_t h, hipStream_t st) {
  // The matrix kernel takes whole 32-element chunks of 16-byte aligned rows, from
  // 5 tokens (256 experts x 7168, bf16 x, fp32 w: 4 tokens 17.5 us on the kernel
  // below against 20.8; 5 tokens 28.9 against 20.9, 64 tokens 45.3 against 22.2,
  // 4096 tokens 2472 against 252 us = 60 TFLOP/s, a library fp64 GEMM's rate).
  // Up to 256 tiles of 16 x 16 a workgroup splits h over 16 waves, up to 512 over
  // 8 (512 tokens: 43 us either way, 73 us with the wider tile); past that 32 x 32
  // tiles halve the operand reads and conversions per product (1024 tokens: 75 us).
  if (m > 4 && h % 32 == 0 && ((uintptr_t)x | (uintptr_t)w) % 16 == 0) {
    const int64_t tiles = ((m + 15) / 16) * ((e + 15) / 16);
    if (tiles <= 256) return launch_router_mfma<1, 1, 16>((const TX*)x, (const TW*)w, logits, m, e, h, st);
    if (tiles <= 512) return launch_router_mfma<1, 1, 8>((const TX*)x, (const TW*)w, logits, m, e, h, st);
    return launch_router_mfma<2, 2, 8>((const TX*)x, (const TW*)w, logits, m, e, h, st);
  }
  if (m <= 4) {
    MOSAIC_LAUNCH((router_logits_kernel<TX, TW, 4, 1>), dim3((unsigned)e, (unsigned)((m + 3) / 4)), dim3(256), 0,
                       st, (const TX*)x, (const TW*)w, logits, (int)m, (int)e, (int)h);
  } else {
    MOSAIC_LAUNCH((router_logits_kernel<TX, TW, 8, 2>), dim3((unsigned)((e + 1) / 2), (unsigned)((m + 7) / 8)),
                       dim3(256), 0, st, (const TX*)x, (const TW*)w, logits, (int)m, (int)e, (int)h);
  }
}

}  // namespace
}  // namespace mosaic

extern "C" int mosaic_router_logits(const void* x, int x_dtype, const void* w, int w_dtype, float* logits, int64_t m,
                                    int64_t e, int64_t h, void* stream) {
  using namespace mosaic;
  MOSAIC_CHECK_ARG(x && w && logits, "router_logits: null pointer");
  MOSAIC_CHECK_ARG(m >= 0 && e >= 1 && h >= 1 && m < (1ll << 31) && e <= 65535 && h < (1ll << 31),
                   "router_logits: bad shape m=%lld e=%lld h=%lld", (long long)m, (long long)e, (long long)h);
  MOSAIC_CHECK_ARG((x_dtype == MOSAIC_DTYPE_F32 || x_dtype == MOSAIC_DTYPE_BF16) &&
                       (w_dtype == MOSAIC_DTYPE_F32 || w_dtype == MOSAIC_DTYPE_BF16),
                   "router_logits: dtypes must be f32 or bf16");
  if (m == 0) return kOk;
  hipStream_t st = (hipStream_t)stream;
  const bool xb = x_dtype == MOSAIC_DTYPE_BF16, wb = w_dtype == MOSAIC_DTYPE_BF16;
  if (xb && wb)
    launch_router<uint16_t, uint16_t>(x, w, logits, m, e, h, st);
  else if (xb)
    launch_router<uint16_t, float>(x, w, logits, m, e, h, st);
  else if (wb)
    launch_router<float, uint16_t>(x, w, logits, m, e, h, st);
  else
    launch_router<float, float>(x, w, logits, m, e, h, st);
  MOSAIC_RETURN_LAUNCH("router_logits");
}
