// DSA decode on gfx950: the FP8 lightning indexer with an exact top-k, and
// MLA decode over the selected KV entries.
//
// Indexer (Indexer.forward, .mosaicvm/source/inference_model.py:408-439):
//   score[t] = sum_h w_h * ReLU(q_h . k_t * q_scale[h] * k_scale[t]),  top-k over t.
// The canonical score (the one the indices are defined on) is fixed step by step:
//   d = exact dot of the decoded e4m3 values rounded once to fp32;
//   a = fp32(fp32(d * q_scale[h]) * k_scale[t]); r = a > 0 ? a : +0;
//   s = sequential fp32 sum over h ascending, from +0, of fp32(r * w_h);
// top-k lists descending s, ties to the lower index, NaN lowest.
//
// The exact dot is cheap per token but not for every token, so selection is
// certified in two stages:
//   1. dsa_index_bound_kernel streams k once, converts the codes to bf16
//      (exact) and takes the dots on the bf16 MFMA, whose sums behave like fp32
//      additions; it writes per token an interval [lo, hi] that contains the
//      canonical score.  The half-width is
//        2^-14 * 448 * |k_scale[t]| * sum_h |w_h| |q_scale[h]| ||q_h||_1 * (1 + 2^-9),
//      where 448 ||q_h||_1 bounds sum_d |q_hd k_td| (|k| <= 448): at least 8x the
//      error of any fp32 summation order of the 128 products (< 2^-17 of their
//      absolute sum) and 4x that error plus the rounding of the remaining steps.
//      (The fp8 MFMA does not allow such a bound: it adds each run of 8 products
//      aligned to the largest one and keeps only about 14 bits below it, so a
//      small product next to a large one is dropped.)
//   2. tau = the lower edge of the histogram digit (top kHistBits bits of the
//      order key) that holds the k-th largest lo.  Any token with hi < tau is
//      beaten by k tokens whose lo >= tau, so the true top-k lies inside
//      {t : hi >= tau}.  Those candidates (typically k + a few tens of percent)
//      get the exact score, then the k best are ranked (dsa_finish_kernel).
// Exact dots on the integer MFMA: every e4m3 value times 512 is an integer X
// with |X| <= 229376, written X = L2*2^14 + L1*2^7 + L0 with L0, L1 in [0, 127]
// and L2 in [-14, 14] (three int8 limbs).  The nine limb products accumulate in
// int32 (v_mfma_i32_16x16x64_i8, exact), grouped by weight into five sums, and
// their weighted fp64 sum (< 2^43, integer) is 2^18 times the exact dot.  (The
// fp8 MFMA is not used here: its fp32 accumulation drops low-order bits once the
// operands span more than about four binades.)
//
// MLA decode (sparse_attn_kernel, .mosaicvm/source/inference_kernel.py:276-352;
// sparse_attn_ref, mosaicvm/model/dsa.py:214-242): per (row, head)
//   o = sum_t bf16(p_t) * v_t / (sum_t p_t + exp(sink - m)),  p_t = exp(s_t - m),
//   s_t = q . kv_t * scale over the selected t (index -1 masked), kv_t = [latent
//   e4m3 * scale -> bf16, rope bf16], v_t = latent.  Online softmax over 32-token
//   blocks in each of several token splits, then a combine over splits.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "../../include/mosaic_amd.h"

namespace mosaic {

// ===================================================================== indexer
constexpr int kIdxD = 128;
constexpr int kHistBits = 13;       // lower-bound key digits: sign, exponent, 4 mantissa bits
constexpr int kHistBins = 1 << kHistBits;
constexpr int kHistShift = 32 - kHistBits;
constexpr int kSortCap = 4096;      // candidates ranked in LDS
constexpr int kMaxTopk = 4096;
constexpr float kBoundFactor = 448.0f / 16384.0f * (1.0f + 1.0f / 512.0f);

// order-preserving keys of fp32 values: NaN lowest (exact scores, lower bounds)
// or highest (upper bounds)
__device__ __forceinline__ uint32_t f32_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ uint32_t key_low_nan(float f) { return (f != f) ? 0u : f32_key(f); }
__device__ __forceinline__ uint32_t key_high_nan(float f) { return (f != f) ? 0xFFFFFFFFu : f32_key(f); }

__device__ __forceinline__ int64_t row_length(const int32_t* lengths, int b, int64_t L) {
  if (!lengths) return L;
  const int64_t n = lengths[b];
  return n < 0 ? 0 : (n > L ? L : n);
}

// Sum over the 64 lanes (all lanes active) on DPP moves (the wave_max_u32
// steps), broadcast from lane 63
__device__ __forceinline__ float wave_sum_f32(float v) {
  v += __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0xB1, 0xF));
  v += __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x4E, 0xF));
  v += __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x141, 0xF));
  v += __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x140, 0xF));
  v += __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x142, 0xA));
  v += __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x143, 0xC));
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), 63));
}

// Sum of |decoded e4m3| over the 32 code bytes of one MFMA operand lane.
__device__ __forceinline__ float abs_sum_fp8(const i32x8_t v) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const f32x2_t a = __builtin_amdgcn_cvt_pk_f32_fp8(v[i], false);
    const f32x2_t b = __builtin_amdgcn_cvt_pk_f32_fp8(v[i], true);
    s += fabsf(a[0]) + fabsf(a[1]) + fabsf(b[0]) + fabsf(b[1]);
  }
  return s;
}

// Sum over the four lanes c, c + 16, c + 32, c + 48 of a 16-column MFMA result
// (v_permlane16/32_swap: no LDS round trip), the same value in all four.
__device__ __forceinline__ float sum_lane_quad(float x) {
  const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float y = __uint_as_float(r16[0]) + __uint_as_float(r16[1]);
  const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(y), __float_as_uint(y), false, false);
  return __uint_as_float(r32[0]) + __uint_as_float(r32[1]);
}

// The 32 e4m3 codes of one fp8 MFMA operand lane -> 4 x 8 bf16 (exact), chunk
// kc = code bytes [8 kc, 8 kc + 8); `neg` flips every sign.
__device__ __forceinline__ void fp8x32_to_bf16(const i32x8_t v, bf16x8_t (&out)[4], bool neg) {
  const uint32_t flip = neg ? 0x80008000u : 0u;
#pragma unroll
  for (int kc = 0; kc < 4; ++kc) {
    uint32_t p[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bf16x2_t lo = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v[2 * kc + h], 1.0f, false);
      const bf16x2_t hi = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v[2 * kc + h], 1.0f, true);
      p[2 * h] = __builtin_bit_cast(uint32_t, lo) ^ flip;
      p[2 * h + 1] = __builtin_bit_cast(uint32_t, hi) ^ flip;
    }
    const u32x4_t pv = {p[0], p[1], p[2], p[3]};
    out[kc] = __builtin_bit_cast(bf16x8_t, pv);
  }
}

// lanes with `active` add 1 to lh[bin]; lanes that share a bin are merged
// first, so a wave issues one LDS atomic per distinct bin
__device__ __forceinline__ void lds_hist_add(uint32_t* lh, uint32_t bin, bool active) {
  const int lane = threadIdx.x & 63;
  uint64_t pending = __ballot(active);
  while (pending) {
    const int leader = __builtin_ctzll(pending);
    const uint32_t lb = (uint32_t)__builtin_amdgcn_readlane((int)bin, leader);
    const uint64_t same = __ballot(bin == lb) & pending;
    if (lane == leader) atomicAdd(&lh[lb], (uint32_t)__builtin_popcountll(same));
    pending &= ~same;
  }
}

// Buffer resource over `records` bytes from `base` (raw addressing): loads past
// the range read zero and stores past it are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, int records) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, records, 0x00020000);
}

// Stage 1: fp8 MFMA scores with a rigorous interval; optional histogram of the
// top kHistBits bits of the lower-bound keys (per row, merged with global atomics per
// workgroup).  grid (gx, B): wave wid of row b takes the groups g = wid, wid +
// nw, ... of U 16-token tiles and streams them through a register ring of D
// groups.  Each group's loads and stores go through buffer resources that end
// at the row's length, so tokens past it read as zero and are not written: the
// ring issues every load unconditionally and its waits stay exact.  `lo` may
// be null (the top-k path reads only the upper bounds and the histogram).
template <int HT, int U, int D>
__global__ void __launch_bounds__(256) dsa_index_bound_kernel(
    const uint8_t* __restrict__ q, const float* __restrict__ qs, const uint8_t* __restrict__ k,
    const float* __restrict__ ks, const float* __restrict__ w, const int32_t* __restrict__ lengths,
    float* __restrict__ lo, float* __restrict__ hi, uint32_t* __restrict__ hist1, int64_t L, int kdiv,
    int64_t kstride) {
  constexpr int H = HT * 16;
  constexpr int GT = 16 * U;  // tokens per group
  constexpr int kQv = H * kIdxD / 16;  // 16-byte pieces of the q row
  __shared__ uint32_t lh[kHistBins];
  __shared__ u32x4_t qsh[kQv];
  __shared__ float qssh[H], wsh[H];
  const int b = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int c = lane & 15, qq = lane >> 4;
  const int64_t n = row_length(lengths, b, L);
  // the q row, its scales and weights are loaded once per workgroup (first,
  // so that staging them waits for nothing else) and read from LDS below
  u32x4_t qv[(kQv + 255) / 256];
  {
    const u32x4_t* q4 = reinterpret_cast<const u32x4_t*>(q + (int64_t)b * H * kIdxD);
#pragma unroll
    for (int i = 0; i < (kQv + 255) / 256; ++i)
      if (kQv % 256 == 0 || threadIdx.x + 256 * i < kQv) qv[i] = q4[threadIdx.x + 256 * i];
  }
  const float qsl = threadIdx.x < H ? qs[(int64_t)b * H + threadIdx.x] : 0.f;
  const float wl = threadIdx.x < H ? w[(int64_t)b * H + threadIdx.x] : 0.f;
  const int64_t n_groups = (n + GT - 1) / GT;
  const int64_t nw = (int64_t)gridDim.x * 4, wid = (int64_t)blockIdx.x * 4 + wv;
  const int64_t iters = wid < n_groups ? (n_groups - 1 - wid) / nw + 1 : 0;
  // kdiv query rows share one key cache; caches start kstride tokens apart
  const uint8_t* kb = k + (int64_t)(b / kdiv) * kstride * kIdxD;
  const float* ksb = ks + (int64_t)(b / kdiv) * kstride;
  float* hib = hi + (int64_t)b * L;
  float* lob = lo ? lo + (int64_t)b * L : hib;  // without lo: a zero-length range, the stores drop
  i32x8_t kr[D][U];
  float sr[D][U];
  // tokens of group g inside the row (wave-uniform)
  auto group_tokens = [&](int64_t g) { return (int)min((int64_t)GT, n - g * GT); };
  auto load = [&](int s, int64_t i) {
    const int64_t g = wid + (i < iters ? i : iters - 1) * nw;  // past the end: reload the last group
    const int nt = group_tokens(g);
    const __amdgpu_buffer_rsrc_t rk = buf_rsrc(kb + g * GT * kIdxD, nt * kIdxD);
    const __amdgpu_buffer_rsrc_t rs = buf_rsrc(ksb + g * GT, nt * 4);
    // the scales first: the wait for a group's codes then covers them too
#pragma unroll
    for (int u = 0; u < U; ++u) sr[s][u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (16 * u + c) * 4, 0, 0));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int off = (16 * u + c) * kIdxD + 16 * qq;
      const u32x4_t a0 = __builtin_amdgcn_raw_buffer_load_b128(rk, off, 0, 0);
      const u32x4_t a1 = __builtin_amdgcn_raw_buffer_load_b128(rk, off + 64, 0, 0);
      kr[s][u] = i32x8_t{(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
    }
  };
  // the ring's first groups go out before the q setup below, so their latency
  // overlaps it (the k stream does not depend on q)
  if (iters > 0) {
#pragma unroll
    for (int s = 0; s < D; ++s) load(s, s);
  }
  if (hist1)
    for (int i = threadIdx.x; i < kHistBins; i += 256) lh[i] = 0u;
#pragma unroll
  for (int i = 0; i < (kQv + 255) / 256; ++i)
    if (kQv % 256 == 0 || threadIdx.x + 256 * i < kQv) qsh[threadIdx.x + 256 * i] = qv[i];
  if (threadIdx.x < H) {
    qssh[threadIdx.x] = qsl;
    wsh[threadIdx.x] = wl;
  }
  __syncthreads();
  // A operands: head rows 16 j + c as bf16, in 4 chunks of 8 of this lane's 32
  // code bytes (the same byte order as the k operand, so every K pairs once),
  // negated where q_scale < 0; per-lane weights c = w |q_scale| of the D rows
  // (heads 16 j + 4 qq + r)
  bf16x8_t qa[HT][4];
  float cw[HT][4];
  i32x8_t raw[HT];
  float qsr[HT], wr[HT], cq[HT][4], cwr[HT][4];
#pragma unroll
  for (int j = 0; j < HT; ++j) {
    const u32x4_t a0 = qsh[(16 * j + c) * (kIdxD / 16) + qq], a1 = qsh[(16 * j + c) * (kIdxD / 16) + 4 + qq];
    raw[j] = i32x8_t{(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
    qsr[j] = qssh[16 * j + c];
    wr[j] = wsh[16 * j + c];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      cq[j][r] = qssh[16 * j + 4 * qq + r];
      cwr[j][r] = wsh[16 * j + 4 * qq + r];
    }
  }
  float bound = 0.f;
#pragma unroll
  for (int j = 0; j < HT; ++j) {
    const float l1 = sum_lane_quad(abs_sum_fp8(raw[j]));  // |q| sum of head row 16 j + c over the 4 lanes
    bound += qq == 0 ? fabsf(wr[j]) * fabsf(qsr[j]) * l1 : 0.f;
    fp8x32_to_bf16(raw[j], qa[j], qsr[j] < 0.f);
#pragma unroll
    for (int r = 0; r < 4; ++r) cw[j][r] = cwr[j][r] * fabsf(cq[j][r]);
  }
  const float qbound = wave_sum_f32(bound) * kBoundFactor;  // any fp32 summation order is within the slack
  auto compute = [&](int s, int64_t i) {
    const int64_t g = wid + i * nw;
    const int nt = group_tokens(g);
    const __amdgpu_buffer_rsrc_t rl = buf_rsrc(lob + g * GT, lo ? nt * 4 : 0);
    const __amdgpu_buffer_rsrc_t rh = buf_rsrc(hib + g * GT, nt * 4);
    f32x4_t d[U][HT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      bf16x8_t kv[4];
      fp8x32_to_bf16(kr[s][u], kv, false);
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[j][kc], kv[kc], acc, 0, 0, 0);
        d[u][j] = acc;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // with d' = d sign(q_scale): max(d q_scale k_scale, 0) w
      //   = |q_scale k_scale| w (|d'| + sign(k_scale) d') / 2
      // partial sums per head row r (independent chains), then across r and lanes
      float pa[4], pb[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pa[r] = cw[0][r] * fabsf(d[u][0][r]);
        pb[r] = cw[0][r] * d[u][0][r];
      }
#pragma unroll
      for (int j = 1; j < HT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          pa[r] = fmaf(cw[j][r], fabsf(d[u][j][r]), pa[r]);
          pb[r] = fmaf(cw[j][r], d[u][j][r], pb[r]);
        }
      const float sa = sum_lane_quad((pa[0] + pa[1]) + (pa[2] + pa[3]));
      const float sb = sum_lane_quad((pb[0] + pb[1]) + (pb[2] + pb[3]));
      const float ksu = sr[s][u];
      const float part = 0.5f * fabsf(ksu) * (ksu < 0.f ? sa - sb : sa + sb);
      const float e = fabsf(sr[s][u]) * qbound;
      const float l = part - e, h = part + e;
      // lanes qq > 0 hold the same token: their stores fall outside the range
      const int off = qq == 0 ? (16 * u + c) * 4 : 0x40000000;
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(l), rl, off, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(h), rh, off, 0, 0);
      if (hist1 && qq == 0 && 16 * u + c < nt) atomicAdd(&lh[key_low_nan(l) >> kHistShift], 1u);
    }
  };
  if (iters > 0) {
    int64_t i0 = 0;
    for (; i0 + D < iters; i0 += D) {
#pragma unroll
      for (int s = 0; s < D; ++s) {
        compute(s, i0 + s);
        load(s, i0 + s + D);
      }
    }
#pragma unroll
    for (int s = 0; s < D; ++s)
      if (i0 + s < iters) compute(s, i0 + s);
  }
  if (hist1) {
    __syncthreads();
    // adjacent digits share one 64-bit add (each count < 2^32: no carry between them)
    unsigned long long* h2 = reinterpret_cast<unsigned long long*>(hist1 + (int64_t)b * kHistBins);
    for (int i = threadIdx.x; i < kHistBins / 2; i += 256) {
      const unsigned long long v = (unsigned long long)lh[2 * i] | ((unsigned long long)lh[2 * i + 1] << 32);
      if (v) atomicAdd(&h2[i], v);
    }
  }
}

typedef __attribute__((ext_vector_type(4))) int i32x4_v;

// 4 e4m3 codes -> three int8 limb words: 512 v = L2 2^14 + L1 2^7 + L0
__device__ __forceinline__ void e4m3_limbs_word(uint32_t x, int (&o)[3]) {
  const f32x2_t a = __builtin_amdgcn_cvt_pk_f32_fp8((int)x, false);
  const f32x2_t c = __builtin_amdgcn_cvt_pk_f32_fp8((int)x, true);
  const int v0 = (int)(a[0] * 512.f), v1 = (int)(a[1] * 512.f);
  const int v2 = (int)(c[0] * 512.f), v3 = (int)(c[1] * 512.f);
  o[0] = (v0 & 127) | ((v1 & 127) << 8) | ((v2 & 127) << 16) | ((v3 & 127) << 24);
  o[1] = ((v0 >> 7) & 127) | (((v1 >> 7) & 127) << 8) | (((v2 >> 7) & 127) << 16) | (((v3 >> 7) & 127) << 24);
  o[2] = ((v0 >> 14) & 255) | (((v1 >> 14) & 255) << 8) | (((v2 >> 14) & 255) << 16) | ((v3 >> 14) << 24);
}
// 16 e4m3 codes -> three int8 limb vectors
__device__ __forceinline__ void e4m3_limbs(const u32x4_t x, i32x4_v (&o)[3]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int t[3];
    e4m3_limbs_word(x[i], t);
    o[0][i] = t[0];
    o[1][i] = t[1];
    o[2][i] = t[2];
  }
}

// First kernel of a top-k call: clears the row histograms and writes q's int8
// limbs in the rescoring kernel's operand order, so that its workgroups load
// them (one coalesced 6 KB block per 16 heads) instead of converting q each:
// row r, heads 16 j + c, dims 64 ch + 16 qd + 4 i .. +3, limb la is word
// ((((r * HT + j) * 2 + ch) * 3 + la) * 64 + c + 16 qd) * 4 + i, HT = heads / 16.
__global__ void dsa_prep_kernel(uint32_t* __restrict__ hist, int64_t n_hist, const uint32_t* __restrict__ q,
                                uint32_t* __restrict__ qlimbs, int64_t n_qwords, int heads) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_hist) hist[i] = 0u;
  if (i < n_qwords) {
    constexpr int W = kIdxD / 4;  // code words per head row
    const int64_t hrow = i / W;    // row * heads + head
    const int wd = (int)(i - hrow * W), head = (int)(hrow % heads);
    const int64_t r = hrow / heads;
    const int j = head >> 4, c = head & 15, ch = wd >> 4, qd = (wd >> 2) & 3, e = wd & 3;
    const int64_t base = (r * (heads >> 4) + j) * 2 + ch;
    int t[3];
    e4m3_limbs_word(q[i], t);
#pragma unroll
    for (int la = 0; la < 3; ++la) qlimbs[((base * 3 + la) * 64 + c + 16 * qd) * 4 + e] = (uint32_t)t[la];
  }
}

__device__ __forceinline__ i32x4_v mfma_i8(const i32x4_v a, const i32x4_v b, const i32x4_v c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// Stage 2: exact scores.  A workgroup owns `range` consecutive tokens of one
// row.  With `hi` set it keeps the tokens whose upper bound reaches tau, the
// lower edge of the histogram digit that holds the topk-th largest lower bound
// (at least topk tokens have lo >= tau, so a token with hi < tau is beaten by
// topk others), scores them 16 at a time on the MFMA (lanes = 16 candidates x
// 4 head groups) and appends 64-bit keys (score key << 32 | ~index) to the
// row's key list; without `hi` it scores every token into `scores`.  The
// histogram, the range's upper bounds and q are loaded together up front, and
// a range of at most kRsPfRange tokens loads its k rows and scales with them
// into LDS (PF), so the candidates' rows are there once tau is known.  The
// histogram is scanned from registers.
constexpr int kRsMaxRange = 4096;
constexpr int kRsPer = kRsMaxRange / 256;
constexpr int kRsMaxWgs = 4096;  // rescoring workgroups per row (rows up to 2^24 tokens)
constexpr int kRsPfRange = 256;  // ranges up to this many tokens stage their k rows in LDS up front
static_assert(kHistBins == 8 * 4 * 256, "the threshold scan gives each of 256 threads 8 vectors of 4 digits");
template <int HT, bool PF, bool QL>
__global__ void __launch_bounds__(256) dsa_rescore_kernel(
    const uint8_t* __restrict__ q, const float* __restrict__ qs, const uint8_t* __restrict__ k,
    const float* __restrict__ ks, const float* __restrict__ w, const int32_t* __restrict__ lengths,
    const float* __restrict__ hi, const uint32_t* __restrict__ hist1, const uint32_t* __restrict__ qlimbs,
    uint64_t* __restrict__ keys, uint32_t* __restrict__ wg_counts, float* __restrict__ scores, int64_t L, int topk,
    int range, int kdiv, int64_t kstride) {
  constexpr int H = HT * 16;
  constexpr int kCand = PF ? kRsPfRange : kRsMaxRange;
  constexpr int kPfVec = PF ? kRsPfRange * kIdxD / 16 : 1;  // 16-byte pieces of the staged k rows
  constexpr int kPfPer = PF ? kPfVec / 256 : 1;
  __shared__ uint32_t sh[1];
  __shared__ uint32_t hsum[8][4];
  __shared__ uint32_t wsum[4];
  __shared__ int cand[kCand];
  __shared__ float terms[4][16][H + 1];
  __shared__ u32x4_t kpf[kPfVec];
  __shared__ float kspf[PF ? kRsPfRange : 1];
  constexpr int kQlVec = HT * 2 * 3 * 64;  // 16-byte vectors of this row's q limbs
  constexpr int kQlPer = (kQlVec + 255) / 256;
  __shared__ i32x4_v qls[QL ? kQlVec : 1];
  const int b = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const int c = lane & 15, qd = lane >> 4;
  const int64_t n = row_length(lengths, b, L);
  const int64_t t_begin = (int64_t)blockIdx.x * range;
  if (t_begin >= n) return;
  const int nr = (int)min((int64_t)range, n - t_begin);  // tokens of this workgroup
  const bool select = hi != nullptr && n > topk;
  const uint8_t* kb = k + (int64_t)(b / kdiv) * kstride * kIdxD;
  const float* ksb = ks + (int64_t)(b / kdiv) * kstride;
  // in flight together: the row's histogram (thread tid holds digit vectors
  // v = tid + 256 i, digits 4 v .. 4 v + 3, coalesced), this range's upper
  // bounds, q, and the range's k rows and scales when they are staged
  u32x4_t hbuf[8];
  if (select) {
    const u32x4_t* src = reinterpret_cast<const u32x4_t*>(hist1 + (int64_t)b * kHistBins);
#pragma unroll
    for (int i = 0; i < 8; ++i) hbuf[i] = src[tid + 256 * i];
  }
  constexpr int kPer = PF ? kRsPfRange / 256 : kRsPer;  // tokens per thread
  float hv[kPer];
  if (hi) {
    const __amdgpu_buffer_rsrc_t rh = buf_rsrc(hi + (int64_t)b * L + t_begin, nr * 4);
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      hv[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rh, (tid + 256 * i) * 4, 0, 0));
  }
  // A operands (rows = heads 16 j + c) as int8 limbs of dims 64 ch + 16 qd ..+16:
  // with QL the row's limbs (written by the prep kernel) are staged in LDS once
  // per workgroup and read after the compaction, otherwise converted here;
  // per-lane constants of the D layout (heads 16 j + 4 qd + r)
  i32x4_v ql[HT][2][3];
  i32x4_v qlb[kQlPer];
  if constexpr (QL) {
    const i32x4_v* src = reinterpret_cast<const i32x4_v*>(qlimbs) + (int64_t)b * kQlVec;
#pragma unroll
    for (int i = 0; i < kQlPer; ++i)
      if (kQlVec % 256 == 0 || tid + 256 * i < kQlVec) qlb[i] = src[tid + 256 * i];
  }
  float qsv[HT][4], wvv[HT][4];
#pragma unroll
  for (int j = 0; j < HT; ++j) {
    if constexpr (!QL) {
      const uint8_t* qrow = q + ((int64_t)b * H + 16 * j + c) * kIdxD + 16 * qd;
#pragma unroll
      for (int ch = 0; ch < 2; ++ch) e4m3_limbs(*reinterpret_cast<const u32x4_t*>(qrow + 64 * ch), ql[j][ch]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      qsv[j][r] = qs[(int64_t)b * H + 16 * j + 4 * qd + r];
      wvv[j][r] = w[(int64_t)b * H + 16 * j + 4 * qd + r];
    }
  }
  // the staged k rows go out last: tau and the compaction wait only for the
  // loads issued before them
  u32x4_t kbuf[kPfPer];
  float ksv = 0.f;
  if constexpr (PF) {
    const __amdgpu_buffer_rsrc_t rk = buf_rsrc(kb + t_begin * kIdxD, nr * kIdxD);
    const __amdgpu_buffer_rsrc_t rs = buf_rsrc(ksb + t_begin, nr * 4);
#pragma unroll
    for (int i = 0; i < kPfPer; ++i) kbuf[i] = __builtin_amdgcn_raw_buffer_load_b128(rk, (tid + 256 * i) * 16, 0, 0);
    ksv = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, tid * 4, 0, 0));
  }
  // tau: the digit holding the topk-th largest lower bound.  Chunk i (digits
  // 1024 i .. 1024 i + 1023) is one vector per thread: a block scan per chunk
  // gives each vector the count of digits above it (the chunks above, plus the
  // higher vectors of its chunk), and the thread whose digits cross topk names it.
  uint32_t tau = 0u;
  if (select) {
    uint32_t vs[8], incl[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      vs[i] = (hbuf[i][0] + hbuf[i][1]) + (hbuf[i][2] + hbuf[i][3]);
      incl[i] = wave_incl_scan_u32(vs[i]);
    }
    if (lane == 63)
#pragma unroll
      for (int i = 0; i < 8; ++i) hsum[i][wv] = incl[i];
    __syncthreads();
    const uint32_t rem = (uint32_t)topk;
    uint32_t above = 0;  // digits in the chunks above chunk i
#pragma unroll
    for (int i = 7; i >= 0; --i) {
      uint32_t tot = 0, before = 0;
#pragma unroll
      for (int w2 = 0; w2 < 4; ++w2) {
        tot += hsum[i][w2];
        before += w2 < wv ? hsum[i][w2] : 0u;
      }
      uint32_t acc = above + (tot - (before + incl[i]));  // digits above this thread's top digit
#pragma unroll
      for (int r = 3; r >= 0; --r) {
        const uint32_t cnt = hbuf[i][r];
        if (acc < rem && rem <= acc + cnt) sh[0] = (uint32_t)(4 * (tid + 256 * i) + r);
        acc += cnt;
      }
      above += tot;
    }
    __syncthreads();
    tau = sh[0] << kHistShift;
  }
  if constexpr (QL) {  // visible after the compaction's barriers
#pragma unroll
    for (int i = 0; i < kQlPer; ++i)
      if (kQlVec % 256 == 0 || tid + 256 * i < kQlVec) qls[tid + 256 * i] = qlb[i];
  }
  if constexpr (PF) {
#pragma unroll
    for (int i = 0; i < kPfPer; ++i) kpf[tid + 256 * i] = kbuf[i];
    kspf[tid] = ksv;
  }
  // compaction: thread tid's tokens are tid + 256 i; a block scan of the
  // per-thread counts places them
  uint32_t keep = 0u, nk = 0u;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const bool ok = tid + 256 * i < nr && (!hi || key_high_nan(hv[i]) >= tau);
    keep |= ok ? 1u << i : 0u;
    nk += ok ? 1u : 0u;
  }
  const uint32_t incl = wave_incl_scan_u32(nk);
  if (lane == 63) wsum[wv] = incl;
  __syncthreads();
  uint32_t pos = incl - nk;
#pragma unroll
  for (int i = 0; i < 4; ++i) pos += i < wv ? wsum[i] : 0u;
  const int C = (int)(wsum[0] + wsum[1] + wsum[2] + wsum[3]);
#pragma unroll
  for (int i = 0; i < kPer; ++i)
    if (keep & (1u << i)) cand[pos++] = (int)(t_begin + tid + 256 * i);
  __syncthreads();
  // the keys go to this workgroup's own token range, keys[b][t_begin + i] for
  // candidate i, and the count to wg_counts[b][blockIdx.x] (no atomics)
  if (hi && tid == 0) wg_counts[(int64_t)b * kRsMaxWgs + blockIdx.x] = (uint32_t)C;
  const int nb = __builtin_amdgcn_readfirstlane((C + 15) / 16);  // batches of 16 candidates (block-uniform)
  if (nb == 0) return;
  if constexpr (QL) {
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
      for (int ch = 0; ch < 2; ++ch)
#pragma unroll
        for (int la = 0; la < 3; ++la) ql[j][ch][la] = qls[((j * 2 + ch) * 3 + la) * 64 + lane];
  }
  struct Batch {
    u32x4_t x[2];
    float ks;
    int t;
  };
  auto load_batch = [&](int bt, Batch& o) {
    const int i = bt * 16 + c;
    const bool ok = i < C;
    o.t = ok ? cand[i] : -1;
    const int64_t tt = ok ? o.t : cand[0];
    if constexpr (PF) {
      const int r = (int)(tt - t_begin);
      o.ks = kspf[r];
#pragma unroll
      for (int ch = 0; ch < 2; ++ch) o.x[ch] = kpf[r * (kIdxD / 16) + 4 * ch + qd];
    } else {
      o.ks = ksb[tt];
#pragma unroll
      for (int ch = 0; ch < 2; ++ch)
        o.x[ch] = *reinterpret_cast<const u32x4_t*>(kb + tt * kIdxD + 64 * ch + 16 * qd);
    }
  };
  // head tile j of a batch (18 MFMAs): the terms of heads 16 j .. 16 j + 15 into tm[candidate][head]
  auto head_tile = [&](int j, const i32x4_v (&kl)[2][3], float kscale, float (*tm)[H + 1]) {
    i32x4_v g[5];
#pragma unroll
    for (int mm = 0; mm < 5; ++mm) g[mm] = i32x4_v{0, 0, 0, 0};
#pragma unroll
    for (int ch = 0; ch < 2; ++ch)
#pragma unroll
      for (int la = 0; la < 3; ++la)
#pragma unroll
        for (int lb = 0; lb < 3; ++lb) g[la + lb] = mfma_i8(ql[j][ch][la], kl[ch][lb], g[la + lb]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double x = (double)g[4][r];
      x = fma(x, 128.0, (double)g[3][r]);
      x = fma(x, 128.0, (double)g[2][r]);
      x = fma(x, 128.0, (double)g[1][r]);
      x = fma(x, 128.0, (double)g[0][r]);
      const float d = (float)(x * 0x1p-18);
      const float a = (d * qsv[j][r]) * kscale;
      const float rr = a > 0.f ? a : 0.f;
      tm[c][16 * j + 4 * qd + r] = rr * wvv[j][r];
    }
  };
  // candidate i (token t): its terms summed in head order, then its key (or score)
  auto emit = [&](int i, int t, const float* row) {
    float tv[H];
#pragma unroll
    for (int h = 0; h < H; ++h) tv[h] = row[h];
    float sc = 0.f;
#pragma unroll
    for (int h = 0; h < H; ++h) sc = sc + tv[h];
    if (hi)
      keys[(int64_t)b * L + t_begin + i] = ((uint64_t)key_low_nan(sc) << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)t);
    else
      scores[(int64_t)b * L + t] = sc;
  };
  if (HT == 4 && nb <= 4) {
    // At most 64 candidates: the four waves share the batches' head tiles,
    // each wave one batch (4 / nbw waves per batch, nbw tiles each), and the
    // terms meet in LDS.
    const int nbw = nb == 3 ? 4 : nb;
    const int bt = wv * nbw / 4, j0 = (wv % (4 / nbw)) * nbw;
    Batch in;
    load_batch(bt, in);  // a batch past the candidates reads candidate 0's row and writes unused terms
    i32x4_v kl[2][3];
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) e4m3_limbs(in.x[ch], kl[ch]);
#pragma unroll
    for (int j = 0; j < HT; ++j)
      if (j >= j0 && j < j0 + nbw) head_tile(j, kl, in.ks, terms[bt]);
    __syncthreads();
    if (tid < C) emit(tid, cand[tid], terms[tid >> 4][tid & 15]);
    return;
  }
  // More candidates: wave wv scores batches bt = wv, wv + 4, ... whole.
  const int my_batches = nb > wv ? (nb - 1 - wv) / 4 + 1 : 0;
  if (my_batches == 0) return;
  auto score_batch = [&](int m, const Batch& in) {
    i32x4_v kl[2][3];
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) e4m3_limbs(in.x[ch], kl[ch]);
#pragma unroll
    for (int j = 0; j < HT; ++j) head_tile(j, kl, in.ks, terms[wv]);
    wave_lds_fence();  // the terms are in LDS
    if (qd == 0 && in.t >= 0) emit(16 * (wv + 4 * m) + c, in.t, terms[wv][c]);
    __builtin_amdgcn_wave_barrier();
  };
  // ping-pong over this wave's batches (bt = wv + 4 m).  The loads are
  // unconditional (a batch past the candidates reads candidate 0's row and
  // scores nothing): a branch around them would make the compiler wait for
  // them at its join, before the current batch is scored.
  Batch ba, bb;
  load_batch(wv, ba);
  for (int m = 0; m < my_batches; m += 2) {
    const bool more = m + 1 < my_batches;
    load_batch(wv + 4 * (m + 1), bb);
    score_batch(m, ba);
    if (!more) break;
    load_batch(wv + 4 * (m + 2), ba);
    score_batch(m + 1, bb);
  }
}

// 64-bit min / max over the 64 lanes (all lanes active) on DPP moves of both
// halves (the wave_max_u32 steps; lanes without a source get the identity),
// broadcast from lane 63
#define MOSAIC_DPP64(ident, v, ctrl, rmask)                                                       \
  (((uint64_t)MOSAIC_DPP((uint32_t)((ident) >> 32), (uint32_t)((v) >> 32), ctrl, rmask) << 32) | \
   (uint64_t)MOSAIC_DPP((uint32_t)(ident), (uint32_t)(v), ctrl, rmask))
__device__ __forceinline__ uint64_t wave_bcast63_u64(uint64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), 63);
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v) {
  constexpr uint64_t I = ~0ull;
  uint64_t o;
  o = MOSAIC_DPP64(I, v, 0xB1, 0xF);
  v = o < v ? o : v;
  o = MOSAIC_DPP64(I, v, 0x4E, 0xF);
  v = o < v ? o : v;
  o = MOSAIC_DPP64(I, v, 0x141, 0xF);
  v = o < v ? o : v;
  o = MOSAIC_DPP64(I, v, 0x140, 0xF);
  v = o < v ? o : v;
  o = MOSAIC_DPP64(I, v, 0x142, 0xA);
  v = o < v ? o : v;
  o = MOSAIC_DPP64(I, v, 0x143, 0xC);
  v = o < v ? o : v;
  return wave_bcast63_u64(v);
}
__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) {
  constexpr uint64_t I = 0ull;
  uint64_t o;
  o = MOSAIC_DPP64(I, v, 0xB1, 0xF);
  v = o > v ? o : v;
  o = MOSAIC_DPP64(I, v, 0x4E, 0xF);
  v = o > v ? o : v;
  o = MOSAIC_DPP64(I, v, 0x141, 0xF);
  v = o > v ? o : v;
  o = MOSAIC_DPP64(I, v, 0x140, 0xF);
  v = o > v ? o : v;
  o = MOSAIC_DPP64(I, v, 0x142, 0xA);
  v = o > v ? o : v;
  o = MOSAIC_DPP64(I, v, 0x143, 0xC);
  v = o > v ? o : v;
  return wave_bcast63_u64(v);
}

// Stage 3: the kk best of the row's candidate keys (unique: exact score key <<
// 32 | ~index), in descending order, to idx_out.  One workgroup of 1024
// threads per row.  Rescoring workgroup w left wg_counts[b][w] keys at
// keys[b][w * range ..].
//  - At most kSortCap candidates: every key goes to registers (4 per thread),
//    placed through the prefix of the per-workgroup counts (the first key
//    slots of every workgroup are read together with the counts).  Otherwise a radix
//    select over the keys in global memory finds the kk-th largest key and
//    only the kk keys at or above it are kept.
//  - Keys are bucketed by (key - smallest key) >> shift into kBuckets buckets,
//    the buckets are laid out largest first by a scan of their counts, and a
//    key's rank is its bucket's start plus the number of larger keys in it.
constexpr int kBuckets = 4096;
static_assert(kBuckets == kRsMaxWgs, "the bucket edges hold the workgroup prefix first");
__global__ void __launch_bounds__(1024) dsa_finish_kernel(const uint64_t* __restrict__ keys,
                                                          const uint32_t* __restrict__ wg_counts,
                                                          const int32_t* __restrict__ lengths, int64_t L, int range,
                                                          int topk, int offset, int32_t* __restrict__ idx_out) {
  __shared__ uint64_t bk[kSortCap];
  __shared__ uint32_t edge[kBuckets + 1];  // workgroup prefix
  __shared__ uint32_t bcnt[kBuckets];      // bucket counts, then bucket edges
  __shared__ uint32_t lh[256];
  __shared__ uint32_t sh[4];
  __shared__ uint64_t red[2][16];
  __shared__ uint32_t wtot[16];
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  for (int i = tid; i < kBuckets; i += 1024) bcnt[i] = 0u;  // visible after the prefix's barriers
  const int64_t n = row_length(lengths, b, L);
  const int nwg = (int)((n + range - 1) / range);
  const uint64_t* kb = keys + (int64_t)b * L;
  // In flight with the counts: the first 4 S key slots of every rescoring
  // workgroup (S = 1024 / nwg threads each), read before their counts are
  // known and kept where the count covers them.
  const int S = nwg <= 1024 ? 1024 / nwg : 0;
  const bool spec = S > 0 && tid < S * nwg;
  const int sw = spec ? tid / S : 0, ss = spec ? tid - sw * S : 0;
  uint32_t sc = 0u;
  uint64_t sk[4];
  if (spec) {
    sc = wg_counts[(int64_t)b * kRsMaxWgs + sw];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t slot = (int64_t)sw * range + ss + S * r;
      sk[r] = slot < L ? kb[slot] : 0ull;
    }
  }
  // edge[w] = first slot of rescoring workgroup w (exclusive prefix)
  {
    uint32_t cw[4], local = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int w = 4 * tid + r;
      cw[r] = w < nwg ? wg_counts[(int64_t)b * kRsMaxWgs + w] : 0u;
      local += cw[r];
    }
    const uint32_t incl = wave_incl_scan_u32(local);
    if (lane == 63) wtot[wv] = incl;
    __syncthreads();
    uint32_t acc = incl - local;
    for (int i = 0; i < wv; ++i) acc += wtot[i];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      edge[4 * tid + r] = acc;
      acc += cw[r];
    }
    __syncthreads();
  }
  uint32_t total = 0;
  for (int i = 0; i < 16; ++i) total += wtot[i];
  const int64_t cnt = min((int64_t)total, n);
  const int kk = (int)min((int64_t)topk, cnt);
  int32_t* dst = idx_out + (int64_t)b * topk;
  for (int i = kk + tid; i < topk; i += 1024) dst[i] = -1;
  if (kk == 0) return;
  // slot i -> its key: the last workgroup w with edge[w] <= i owns it
  auto key_at = [&](int i) -> uint64_t {
    int lo = 0, hi = nwg - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (edge[mid] <= (uint32_t)i) lo = mid; else hi = mid - 1;
    }
    return kb[(int64_t)lo * range + (i - (int)edge[lo])];
  };
  int m;
  uint64_t x[4];
  if (cnt <= kSortCap && S > 0) {
    // the keys into LDS at their workgroup's edge (the slots past 4 S one at a time), then 4 per thread
    m = (int)cnt;
    if (spec) {
      const uint32_t e0 = edge[sw];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if ((uint32_t)(ss + S * r) < sc) bk[e0 + ss + S * r] = sk[r];
      for (uint32_t j = (uint32_t)(ss + 4 * S); j < sc; j += (uint32_t)S) bk[e0 + j] = kb[(int64_t)sw * range + j];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = tid + 1024 * r < m ? bk[tid + 1024 * r] : 0ull;
  } else if (cnt <= kSortCap) {
    m = (int)cnt;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = tid + 1024 * r < m ? key_at(tid + 1024 * r) : 0ull;
  } else {
    // radix select of the kk-th largest key, 8 bits at a time
    uint64_t prefix = 0, pmask = 0;
    uint32_t rem = (uint32_t)kk;
    for (int shift = 56; shift >= 0; shift -= 8) {
      if (tid < 256) lh[tid] = 0u;
      __syncthreads();
      for (int i = tid; i < (int)cnt; i += 1024) {
        const uint64_t key = key_at(i);
        if ((key & pmask) == prefix) atomicAdd(&lh[(key >> shift) & 255u], 1u);
      }
      __syncthreads();
      if (tid < 64) {  // one wave finds the digit: 4 bins per lane, scanned from the top
        uint32_t cnt4[4], local = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          cnt4[i] = lh[255 - (4 * lane + i)];
          local += cnt4[i];
        }
        uint32_t acc = wave_incl_scan_u32(local) - local;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (acc < rem && rem <= acc + cnt4[i]) {
            sh[0] = 255u - (uint32_t)(4 * lane + i);
            sh[1] = acc;
          }
          acc += cnt4[i];
        }
      }
      __syncthreads();
      prefix |= (uint64_t)sh[0] << shift;
      pmask |= 255ull << shift;
      rem -= sh[1];
      const bool whole = lh[sh[0]] == rem;  // every key with this prefix is selected
      __syncthreads();
      if (whole) break;
    }
    if (tid == 0) sh[2] = 0u;
    __syncthreads();
    for (int i = tid; i < (int)cnt; i += 1024) {
      const uint64_t key = key_at(i);
      if (key >= prefix) bk[atomicAdd(&sh[2], 1u)] = key;
    }
    __syncthreads();
    m = kk;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = tid + 1024 * r < m ? bk[tid + 1024 * r] : 0ull;
  }
  // smallest and largest key
  uint64_t mn = ~0ull, mx = 0ull;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (tid + 1024 * r < m) {
      mn = x[r] < mn ? x[r] : mn;
      mx = x[r] > mx ? x[r] : mx;
    }
  mn = wave_min_u64(mn);
  mx = wave_max_u64(mx);
  if (lane == 0) {
    red[0][wv] = mn;
    red[1][wv] = mx;
  }
  __syncthreads();
  mn = red[0][0];
  mx = red[1][0];
#pragma unroll
  for (int i = 1; i < 16; ++i) {
    mn = red[0][i] < mn ? red[0][i] : mn;
    mx = red[1][i] > mx ? red[1][i] : mx;
  }
  const uint64_t span = mx - mn;
  const int bits = span == 0 ? 0 : 64 - __clzll((long long)span);
  const int shift = bits > 12 ? bits - 12 : 0;
  uint32_t bx[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    bx[r] = (uint32_t)((x[r] - mn) >> shift);
    if (tid + 1024 * r < m) atomicAdd(&bcnt[bx[r]], 1u);
  }
  __syncthreads();
  // descending exclusive scan: bcnt[d] = number of keys in buckets above d
  // (thread tid owns buckets kBuckets-1-4 tid .. kBuckets-4-4 tid)
  uint32_t cb[4], local = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    cb[i] = bcnt[kBuckets - 1 - (4 * tid + i)];
    local += cb[i];
  }
  const uint32_t incl = wave_incl_scan_u32(local);
  if (lane == 63) wtot[wv] = incl;
  __syncthreads();
  uint32_t acc = incl - local;
  for (int i = 0; i < wv; ++i) acc += wtot[i];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    bcnt[kBuckets - 1 - (4 * tid + i)] = acc;
    acc += cb[i];
  }
  __syncthreads();
  // scatter into bucket order; afterwards bcnt[d] = the end of bucket d
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (tid + 1024 * r < m) bk[atomicAdd(&bcnt[bx[r]], 1u)] = x[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (tid + 1024 * r >= m) continue;
    const uint32_t s = bx[r] + 1 < kBuckets ? bcnt[bx[r] + 1] : 0u, e = bcnt[bx[r]];
    uint32_t rank = s;
    for (uint32_t j = s; j < e; ++j) rank += bk[j] > x[r] ? 1u : 0u;
    if (rank < (uint32_t)kk) dst[rank] = (int32_t)(0xFFFFFFFFu - (uint32_t)x[r]) + offset;
  }
}

// ---------------------------------------------- many rows over short caches
// Indexer + exact top-k of many query rows that share short key caches (a
// prompt: row t sees the first (t + 1) / ratio entries).  Picks are most of a
// row's entries there, so bounding first would save little: every entry gets
// its exact score, and the row's keys are sorted, in one kernel that needs no
// workspace (its callers give the certified path's, which it leaves alone).
//
// A workgroup takes kDrRows consecutive rows of one cache, one wave each (q's
// int8 limbs in registers).  The cache goes through LDS in chunks of 128 tokens,
// already as int8 limbs in MFMA operand order (wave w converts tokens 16 w ..
// + 15 of a chunk for all the rows), the next chunk's codes loaded during the
// products.  Row i of the A operand holds head (i / 4) * H / 4 + 4 j + i % 4 in
// head tile j, so lane quarter qd holds the terms of heads qd H / 4 .. + H / 4 - 1
// of token c, and the canonical head order is four runs of in-lane additions
// with the sum handed from quarter to quarter.  The five limb sums go through
// two int32 before one fp64 multiply-add (|g0 + 2^7 g1| and |g2 + 2^7 g3 + 2^14
// g4| < 2^30).  Then each wave sorts its row: a bitonic network over E keys a lane.
//
// Bound by the matrix unit and the term arithmetic about equally (1152 MFMA
// cycles and ~1400 VALU cycles a wave per 16 tokens and row).
constexpr int kDrRows = 8;
constexpr int kDrMaxL = 2048;
constexpr int kDrChunk = 128;

// Sort keys as positive doubles in [1, 2): the mantissa holds the 32-bit score
// key, then kDrIdxBits of the inverted token.  Their order is the keys', and a
// compare-exchange is one v_max_f64 and one v_min_f64 (no NaN, infinity or
// subnormal among them).
constexpr int kDrIdxBits = 11;
static_assert(kDrMaxL <= 1 << kDrIdxBits, "a token must fit its bits of the key");
__device__ __forceinline__ double key_max(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double key_min(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double key_flip(double a, uint32_t sign) {
  const uint64_t u = __builtin_bit_cast(uint64_t, a);
  return __builtin_bit_cast(double, u ^ ((uint64_t)sign << 32));
}

// Descending bitonic sort over the wave, position lane * E + e.  The lanes whose
// runs a phase sorts upwards hold their keys negated during it, so every
// exchange keeps the larger key at the lower position.
template <int E>
__device__ __forceinline__ void wave_sort_desc(double (&x)[E]) {
  const int lane = threadIdx.x & 63;
  auto order = [&](double& a, double& b) {
    const double t = key_max(a, b);
    b = key_min(a, b);
    a = t;
  };
  // runs of E in each lane, descending in even lanes
#pragma unroll
  for (int sz = 2; sz < E; sz *= 2)
#pragma unroll
    for (int st = sz / 2; st > 0; st /= 2)
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (!(e & st)) {
          if ((e & sz) == 0)
            order(x[e], x[e | st]);
          else
            order(x[e | st], x[e]);
        }
  uint32_t up = 0u;  // sign of this lane's keys in the current phase
  auto phase = [&](bool desc) {
    const uint32_t want = desc ? 0u : 0x80000000u;
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = key_flip(x[e], want ^ up);
    up = want;
  };
  auto merge = [&]() {
#pragma unroll
    for (int st = E / 2; st > 0; st /= 2)
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (!(e & st)) order(x[e], x[e | st]);
  };
  phase((lane & 1) == 0);
  merge();
  for (int sz = 2; sz <= 64; sz *= 2) {
    phase((lane & sz) == 0);  // (the last size: all descending)
    for (int st = sz / 2; st > 0; st /= 2) {
      double y[E];
#pragma unroll
      for (int e = 0; e < E; ++e) y[e] = __shfl_xor(x[e], st);
      if (lane & st) {
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = key_min(x[e], y[e]);
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = key_max(x[e], y[e]);
      }
    }
    merge();
  }
}

// sort the n <= 64 E scores of a row and write its topk picks; `buf` is the
// row's LDS (its scores, then its sorted indices)
template <int E>
__device__ __forceinline__ void dsa_row_picks(float* buf, int n, int topk, int offset, int32_t* dst) {
  const int lane = threadIdx.x & 63;
  constexpr uint32_t kMask = (1u << kDrIdxBits) - 1;
  double x[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int t = 64 * e + lane;
    // (a token's inverted bits are never 0 past the last one, so no key equals the padding's)
    const uint64_t key = ((uint64_t)key_low_nan(buf[t]) << kDrIdxBits) | (uint64_t)(kMask - (uint32_t)t);
    x[e] = __builtin_bit_cast(double, 0x3FF0000000000000ull | (t < n ? key + 1 : 0ull));
  }
  wave_sort_desc<E>(x);
  wave_lds_fence();
  int* sorted = reinterpret_cast<int*>(buf);
#pragma unroll
  for (int e = 0; e < E; ++e)
    sorted[lane * E + e] = (int)(kMask - ((uint32_t)(__builtin_bit_cast(uint64_t, x[e]) - 1) & kMask));
  wave_lds_fence();
  const int kk = min(topk, n);
  for (int i = lane; i < topk; i += 64) dst[i] = i < kk ? sorted[i] + offset : -1;
}

template <int HT>
__global__ void __launch_bounds__(64 * kDrRows) dsa_rows_topk_kernel(
    const uint8_t* __restrict__ q, const float* __restrict__ qs, const uint8_t* __restrict__ k,
    const float* __restrict__ ks, const float* __restrict__ w, const int32_t* __restrict__ lengths,
    int32_t* __restrict__ idx_out, int64_t L, int groups, int kdiv, int64_t kstride, int topk, int offset) {
  constexpr int H = HT * 16, HB = H / 4;
  __shared__ i32x4_v kls[kDrChunk / 16][2][3][64];
  __shared__ float kss[kDrChunk];
  __shared__ float scs[kDrRows][kDrMaxL];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int c = lane & 15, qd = lane >> 4;
  // a cache's last rows first: in a prompt they see the most entries
  const int g = (int)blockIdx.x % groups, r0 = ((kdiv + kDrRows - 1) / kDrRows - 1 - (int)blockIdx.x / groups) * kDrRows;
  const bool active = r0 + wv < kdiv;
  const int64_t row = (int64_t)g * kdiv + (active ? r0 + wv : r0);
  const int n = active ? (int)row_length(lengths, (int)row, L) : 0;
  int nmax = 0;
  for (int r = r0; r < min(r0 + kDrRows, kdiv); ++r)
    nmax = max(nmax, (int)row_length(lengths, g * kdiv + r, L));
  nmax = __builtin_amdgcn_readfirstlane(nmax);
  const uint8_t* kb = k + (int64_t)g * kstride * kIdxD;
  const float* ksb = ks + (int64_t)g * kstride;
  u32x4_t kx[2];
  float kscale = 0.f;
  auto load_chunk = [&](int t0) {
    const int t = t0 + 16 * wv + c;
    const bool ok = t < L;
#pragma unroll
    for (int ch = 0; ch < 2; ++ch)
      kx[ch] = ok ? *reinterpret_cast<const u32x4_t*>(kb + (int64_t)t * kIdxD + 64 * ch + 16 * qd) : u32x4_t{0u, 0u, 0u, 0u};
    kscale = ok ? ksb[t] : 0.f;
  };
  if (nmax > 0) load_chunk(0);
  i32x4_v ql[HT][2][3];
  float qsv[HT][4], wvv[HT][4];
#pragma unroll
  for (int j = 0; j < HT; ++j) {
    const uint8_t* qrow = q + (row * H + (c >> 2) * HB + 4 * j + (c & 3)) * kIdxD + 16 * qd;
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) e4m3_limbs(*reinterpret_cast<const u32x4_t*>(qrow + 64 * ch), ql[j][ch]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      qsv[j][r] = qs[row * H + qd * HB + 4 * j + r];
      wvv[j][r] = w[row * H + qd * HB + 4 * j + r];
    }
  }
  for (int t0 = 0; t0 < nmax; t0 += kDrChunk) {
    __syncthreads();  // the previous chunk is no longer read
    {
      i32x4_v o[2][3];
#pragma unroll
      for (int ch = 0; ch < 2; ++ch) {
        e4m3_limbs(kx[ch], o[ch]);
#pragma unroll
        for (int la = 0; la < 3; ++la) kls[wv][ch][la][lane] = o[ch][la];
      }
      if (qd == 0) kss[16 * wv + c] = kscale;
    }
    __syncthreads();
    if (t0 + kDrChunk < nmax) load_chunk(t0 + kDrChunk);
    const int nb = min(kDrChunk / 16, (n - t0 + 15) / 16);  // batches of this row in the chunk (<= 0: none)
    for (int bt = 0; bt < nb; ++bt) {
      i32x4_v kl[2][3];
#pragma unroll
      for (int ch = 0; ch < 2; ++ch)
#pragma unroll
        for (int la = 0; la < 3; ++la) kl[ch][la] = kls[bt][ch][la][lane];
      const float ksc = kss[16 * bt + c];
      float tv[HB];
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        i32x4_v gs[5];
#pragma unroll
        for (int mm = 0; mm < 5; ++mm) gs[mm] = i32x4_v{0, 0, 0, 0};
#pragma unroll
        for (int ch = 0; ch < 2; ++ch)
#pragma unroll
          for (int la = 0; la < 3; ++la)
#pragma unroll
            for (int lb = 0; lb < 3; ++lb) gs[la + lb] = mfma_i8(ql[j][ch][la], kl[ch][lb], gs[la + lb]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int x0 = (gs[1][r] << 7) + gs[0][r];
          const int x1 = (gs[4][r] << 14) + ((gs[3][r] << 7) + gs[2][r]);
          // x1 2^14 + x0 is 2^18 times the exact dot, and exact in fp64
          const float d = (float)fma((double)x1, 16384.0, (double)x0) * 0x1p-18f;
          const float a = (d * qsv[j][r]) * ksc;
          const float rr = a > 0.f ? a : 0.f;
          tv[4 * j + r] = rr * wvv[j][r];
        }
      }
      // heads in order: quarter 0's, then 1's, ... (each quarter's lanes go on from the previous one's sum)
      float sum = 0.f;
#pragma unroll
      for (int h = 0; h < HB; ++h) sum = sum + tv[h];
      sum = __uint_as_float(__builtin_amdgcn_permlane16_swap(__float_as_uint(sum), __float_as_uint(sum), false, false)[0]);
#pragma unroll
      for (int h = 0; h < HB; ++h) sum = sum + tv[h];
      {
        const uint32_t odd = __builtin_amdgcn_permlane16_swap(__float_as_uint(sum), __float_as_uint(sum), false, false)[1];
        sum = __uint_as_float(__builtin_amdgcn_permlane32_swap(odd, odd, false, false)[0]);
      }
#pragma unroll
      for (int h = 0; h < HB; ++h) sum = sum + tv[h];
      sum = __uint_as_float(__builtin_amdgcn_permlane16_swap(__float_as_uint(sum), __float_as_uint(sum), false, false)[0]);
#pragma unroll
      for (int h = 0; h < HB; ++h) sum = sum + tv[h];
      if (qd == 3) scs[wv][t0 + 16 * bt + c] = sum;
    }
  }
  wave_lds_fence();
  if (!active) return;
  int32_t* dst = idx_out + row * topk;
  if (n <= 64)
    dsa_row_picks<1>(scs[wv], n, topk, offset, dst);
  else if (n <= 128)
    dsa_row_picks<2>(scs[wv], n, topk, offset, dst);
  else if (n <= 256)
    dsa_row_picks<4>(scs[wv], n, topk, offset, dst);
  else if (n <= 512)
    dsa_row_picks<8>(scs[wv], n, topk, offset, dst);
  else if (n <= 1024)
    dsa_row_picks<16>(scs[wv], n, topk, offset, dst);
  else
    dsa_row_picks<32>(scs[wv], n, topk, offset, dst);
}

// ===================================================================== MLA
constexpr int kMlaBT = 32;        // tokens per online-softmax block
constexpr int kMlaDl = 512;       // latent (value) width
constexpr int kMlaDt = kMlaDl / 16;  // 16-wide latent column tiles
constexpr int kPsStride = 40;     // bf16 per row of the P exchange (32 tokens + 8)
constexpr int kMlaMaxSplits = 64;
// A head's running maximum moves only when a block's maximum exceeds it by
// more than this (natural log units): probabilities stay below e^8, which
// bf16 P and the fp32 sums hold with their usual relative precision, and the
// O rescale is skipped for almost every block after the first.
constexpr float kMlaLazyMax = 8.f;

constexpr int kMlaMaxChunk = 1024;  // token ids of one split (staged in LDS)
// FP8 gather stages: raw latent rows, scale rows (up to 32 floats), rope rows
constexpr int kMlaStages = 3;
constexpr int kMlaStgLat = kMlaBT * kMlaDl;
constexpr int kMlaStgSc = kMlaBT * 32 * 4;
constexpr int kMlaStgRope = kMlaBT * 64 * 2;
constexpr int kMlaStage = kMlaStgLat + kMlaStgSc + kMlaStgRope;
constexpr int kMlaCopies = 9;  // copies per wave per block: 4 latent, 4 scale, 1 rope

typedef short mla_v4s __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t mla_lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
// one 16-byte (resp. 4-byte) global -> LDS copy per lane; the LDS address of
// lane i is base + 16 i (resp. 4 i).  Issued from inline asm so the compiler
// neither waits for them before LDS reads nor stages them in registers; the
// kernel waits with explicit vmcnt counts.
__device__ __forceinline__ void mla_copy16(const void* g, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(__builtin_amdgcn_readfirstlane(lds)),
               "v"(g) : "memory", "m0");
}
// the same from a wave-uniform base plus this lane's byte offset
__device__ __forceinline__ void mla_copy16_s(const void* base, int off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds)),
               "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void mla_copy4(const void* g, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off" ::"s"(__builtin_amdgcn_readfirstlane(lds)),
               "v"(g) : "memory", "m0");
}

__device__ __forceinline__ f32x4_t mfma_bf16(const bf16x8_t a, const bf16x8_t b, const f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Token order inside a block: MFMA K index / P slot p = 8 g + 4 r + i holds
// block token 8 g + 2 i + r.  With it the four 4-token LDS transpose reads of
// two 16-lane groups touch 8 rows whose bank offsets (36 dwords apart) are
// 8 dwords apart, and a QK A-operand read still takes 16 rows distinct mod 16.
__device__ __forceinline__ int mla_slot_token(int p) { return (p & ~7) | ((p & 3) << 1) | ((p >> 2) & 1); }

// 4 bf16 of V column c' (of a 16-column tile) for 4 tokens, from row-major
// K rows in LDS: with lane 4 i + j of a 16-lane group pointing at row token_i,
// columns 4 j .. 4 j + 3, lane c' receives row token_i, column c' as element i.
__device__ __forceinline__ mla_v4s lds_read_tr16(const uint16_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) mla_v4s*)(p));
}

// max / sum over the 16 lanes of each row (pair, quad, half-row and row
// mirrors); every lane of the row gets the result
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0xB1, 0xF)));
  v = fmaxf(v, __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x4E, 0xF)));
  v = fmaxf(v, __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x141, 0xF)));
  return fmaxf(v, __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x140, 0xF)));
}
__device__ __forceinline__ float row16_sum(float v) {
  v += __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0xB1, 0xF));
  v += __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x4E, 0xF));
  v += __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x141, 0xF));
  return v + __uint_as_float(MOSAIC_DPP(0u, __float_as_uint(v), 0x140, 0xF));
}

// Where the KV of a row lives.  FP8: latent e4m3 [rows, 512] + f32 scales
// [rows, 512 >> sb_shift] + rope bf16 [rows, DR].  BF16: one bf16 tensor
// [rows, 512 + DR] (latent first).  Row r of the queries reads KV batch
// r / rows_per_kv.
struct MlaKv {
  const void* lat;
  const float* lat_s;
  const uint16_t* rope;
  int64_t n;
  int rows_per_kv;
  int sb_shift;
};

// One split (a contiguous slice of the selected tokens) of one query row and
// one group of 16*HT heads (HT head tiles): partial (m, l, O) per head.  The
// split's token ids are staged in LDS first (masked or out-of-range ids as -1).
// Blocks of kMlaBT tokens then go through two LDS buffers of bf16 K rows
// (latent then rope).  FP8 caches: raw rows, their scales and rope rows are
// copied global -> LDS directly (global_load_lds) into a ring of kMlaStages
// stages, issued three blocks ahead of their conversion to bf16, so the gather
// latency hides behind three blocks of math; every wave issues kMlaCopies
// copies per block, so `s_waitcnt vmcnt` + a barrier hands a stage over.  BF16
// caches: each thread gathers its item of block i + 1 into registers while
// block i is multiplied out, and stores it after.
//
// Four waves.  Wave w < HT scores and soft-maxes head tile w (S = Q K^T:
// its heads' q kept in registers as the A operand, K rows from LDS as B), then
// the workgroup swaps roles for O += P V: P (bf16) and the per-head rescale
// factors go through LDS, and each wave multiplies every head of the group
// into its own quarter of the 512 latent columns, reading V straight out of
// the K rows with LDS transpose reads.  So V is read once per workgroup rather
// than once per 16 heads, and no transposed copy of it is written.  A
// workgroup runs one wave per SIMD, which leaves room for the O tiles (16 HT
// heads x 128 columns per wave) in accumulation registers.
template <int HT, bool FP8, int DR>
__global__ void __launch_bounds__(256) mla_decode_split_kernel(
    const uint16_t* __restrict__ q, const MlaKv kv, const int32_t* __restrict__ idx, uint16_t* __restrict__ part_o,
    float* __restrict__ part_ml, int topk, float scale, int chunk) {
  constexpr int DQK = kMlaDl + DR;
  constexpr int KS = DQK + 8;  // bf16 per K row in LDS: 16-byte reads of 16 rows hit distinct banks
  constexpr int NW = 4, NT = NW * 64;
  constexpr int RAWV = FP8 ? 4 : 8;               // 16-byte vectors per (token, 64-wide segment) item
  constexpr int DTW = kMlaDt / NW;                // latent column tiles per wave in O += P V
  static_assert(kMlaBT * 8 == NT && (DR == 0 || kMlaBT * (DR / 8) == NT), "one item and one rope chunk a thread");
  static_assert(!FP8 || DR == 64, "FP8 caches carry a 64-wide bf16 rope");
  __shared__ __attribute__((aligned(16))) uint16_t Kt[2][kMlaBT * KS];
  __shared__ __attribute__((aligned(16))) uint8_t Stg[FP8 ? kMlaStages * kMlaStage : 16];
  __shared__ __attribute__((aligned(16))) uint16_t Ps[16 * HT * kPsStride];
  __shared__ __attribute__((aligned(16))) float As[16 * HT];
  __shared__ int Fl[HT];
  __shared__ int Ids[kMlaMaxChunk];
  const int H = HT * 16 * gridDim.z;
  const int split = blockIdx.x, b = blockIdx.y, S = gridDim.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool scorer = wv < HT;             // this wave scores head tile wv
  const int hw = (int)blockIdx.z * HT + (scorer ? wv : 0);  // its 16-head group in the row
  const int c = lane & 15, qd = lane >> 4;
  const int head = 16 * hw + c;
  const int dt0 = wv * DTW;  // this wave's first latent column tile
  const int64_t n = kv.n;
  const int64_t kvb = b / kv.rows_per_kv;
  const int t_begin = split * chunk;
  const int t_end = min(topk, t_begin + chunk);
  // (an empty cache masks every token: nothing is read)
  const int nblk = t_end > t_begin && n > 0 ? (t_end - t_begin + kMlaBT - 1) / kMlaBT : 0;
  const int nsc = kMlaDl >> kv.sb_shift;  // scales per FP8 row
  // the split's ids (loaded first, so that they fly together with q)
  constexpr int IDS_PT = kMlaMaxChunk / NT;
  int idv[IDS_PT];
#pragma unroll
  for (int k = 0; k < IDS_PT; ++k) {
    const int s = tid + NT * k, ti = t_begin + s;
    idv[k] = s < nblk * kMlaBT && ti < t_end ? idx[(int64_t)b * topk + ti] : -1;
  }
  // q as the A operand of S = Q K^T: lane (c, qd) holds q[head][32 s + 8 qd .. +8]
  // (kept in registers: the empty asm stops the compiler from re-loading q in
  // every block, where those loads would queue behind the gather)
  bf16x8_t qb[DQK / 32];
  {
    const uint16_t* qrow = q + ((int64_t)b * H + head) * DQK;
#pragma unroll
    for (int s = 0; s < DQK / 32; ++s) qb[s] = *reinterpret_cast<const bf16x8_t*>(qrow + 32 * s + 8 * qd);
#pragma unroll
    for (int s = 0; s < DQK / 32; ++s) asm volatile("" : "+v"(qb[s]));
  }
#pragma unroll
  for (int k = 0; k < IDS_PT; ++k) {
    const int s = tid + NT * k;
    if (s < nblk * kMlaBT) Ids[s] = idv[k] >= 0 && (int64_t)idv[k] < n ? idv[k] : -1;
  }
  __syncthreads();
  // row of the cache that token t of block j reads (masked tokens read row 0
  // of their batch and are zeroed when converted)
  auto row_of = [&](int j, int t) -> int64_t {
    const int id = Ids[j * kMlaBT + t];
    return kvb * n + (id >= 0 ? id : 0);
  };
  // ---- FP8: global -> LDS copies of block j into stage j % kMlaStages.  Latent
  // rows keep their 16-byte chunks XOR-swizzled by (token & 15) and scale rows
  // their floats by (token & 31), so the conversion's reads of 16 tokens hit
  // distinct banks.
  auto issue_fp8 = [&](int j) {
    uint8_t* st = &Stg[(j % kMlaStages) * kMlaStage];
#pragma unroll
    for (int k = 0; k < 4; ++k) {  // latent: tokens 8 wv + 2 k (lanes 0-31) and + 1 (lanes 32-63)
      const int t = 8 * wv + 2 * k + (lane >> 5), p = lane & 31;
      const uint8_t* src = reinterpret_cast<const uint8_t*>(kv.lat) + row_of(j, t) * kMlaDl + 16 * (p ^ (t & 15));
      mla_copy16(src, mla_lds_addr(st + (8 * wv + 2 * k) * kMlaDl));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {  // scales: floats 64 (wv + 4 k) + lane = (token f / 32, slot f % 32)
      const int f = 64 * (wv + 4 * k) + lane, t = f >> 5, p = f & 31;
      const int e = min(p ^ (t & 31), nsc - 1);
      mla_copy4(kv.lat_s + row_of(j, t) * nsc + e, mla_lds_addr(st + kMlaStgLat + 256 * (wv + 4 * k)));
    }
    {  // rope: tokens 8 wv .. 8 wv + 7
      const int t = 8 * wv + (lane >> 3), pc = lane & 7;
      mla_copy16(kv.rope + row_of(j, t) * DR + 8 * pc, mla_lds_addr(st + kMlaStgLat + kMlaStgSc + 1024 * wv));
    }
  };
  // wait until at most `after` blocks' copies of this wave are in flight, then barrier
  auto wait_stage = [&](int after) {
    if (after >= 2)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * kMlaCopies) : "memory");
    else if (after == 1)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kMlaCopies) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  };
  // item of thread tid: token tid % 32, latent segment tid / 32 (64 values);
  // rope chunk: token tid / 8, 8 values at 8 (tid % 8)
  const int tk = tid % kMlaBT, seg = tid / kMlaBT;
  const int rtk = tid / 8, rpc = tid % 8;
  // stage of block j -> bf16 K rows of buffer j & 1
  auto convert_fp8 = [&](int j) {
    const uint8_t* st = &Stg[(j % kMlaStages) * kMlaStage];
    const bool ok = Ids[j * kMlaBT + tk] >= 0;
    const float* srow = reinterpret_cast<const float*>(st + kMlaStgLat) + tk * 32;
    uint32_t outw[32];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const u32x4_t w = *reinterpret_cast<const u32x4_t*>(st + tk * kMlaDl + 16 * ((4 * seg + v) ^ (tk & 15)));
      const float sc = srow[((seg * 64 + 16 * v) >> kv.sb_shift) ^ (tk & 31)];
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        // exact e4m3 -> fp32, fp32 product with the scale, one RNE rounding to bf16
        f32x2_t a2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[e2], false);
        f32x2_t b2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[e2], true);
        a2[0] *= sc;
        a2[1] *= sc;
        b2[0] *= sc;
        b2[1] *= sc;
        outw[8 * v + 2 * e2] = __builtin_bit_cast(uint32_t, __builtin_convertvector(a2, bf16x2_t));
        outw[8 * v + 2 * e2 + 1] = __builtin_bit_cast(uint32_t, __builtin_convertvector(b2, bf16x2_t));
      }
    }
    u32x4_t* kdst = reinterpret_cast<u32x4_t*>(&Kt[j & 1][tk * KS + seg * 64]);
#pragma unroll
    for (int v = 0; v < 8; ++v)
      kdst[v] = ok ? u32x4_t{outw[4 * v], outw[4 * v + 1], outw[4 * v + 2], outw[4 * v + 3]} : u32x4_t{0u, 0u, 0u, 0u};
    const u32x4_t r = *reinterpret_cast<const u32x4_t*>(st + kMlaStgLat + kMlaStgSc + rtk * 128 + 16 * rpc);
    *reinterpret_cast<u32x4_t*>(&Kt[j & 1][rtk * KS + kMlaDl + 8 * rpc]) =
        Ids[j * kMlaBT + rtk] >= 0 ? r : u32x4_t{0u, 0u, 0u, 0u};
  };
  // ---- BF16: register-staged gather of block j, stored by fill_bf16
  u32x4_t raw[RAWV];
  u32x4_t rrope;
  auto issue_bf16 = [&](int j) {
    const uint16_t* src = reinterpret_cast<const uint16_t*>(kv.lat) + row_of(j, tk) * DQK + seg * 64;
#pragma unroll
    for (int v = 0; v < RAWV; ++v) raw[v] = *reinterpret_cast<const u32x4_t*>(src + 8 * v);
    if constexpr (DR > 0)
      rrope = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint16_t*>(kv.lat) + row_of(j, rtk) * DQK +
                                                 kMlaDl + 8 * rpc);
  };
  auto fill_bf16 = [&](int j) {
    const bool ok = Ids[j * kMlaBT + tk] >= 0;
    u32x4_t* kdst = reinterpret_cast<u32x4_t*>(&Kt[j & 1][tk * KS + seg * 64]);
#pragma unroll
    for (int v = 0; v < 8; ++v) kdst[v] = ok ? raw[v] : u32x4_t{0u, 0u, 0u, 0u};
    if constexpr (DR > 0)
      *reinterpret_cast<u32x4_t*>(&Kt[j & 1][rtk * KS + kMlaDl + 8 * rpc]) =
          Ids[j * kMlaBT + rtk] >= 0 ? rrope : u32x4_t{0u, 0u, 0u, 0u};
  };
  // O tiles: rows = heads 16 ht + 4 qd + r of the group, columns 16 (dt0 + dl) + c
  f32x4_t o[HT][DTW];
#pragma unroll
  for (int ht = 0; ht < HT; ++ht)
#pragma unroll
    for (int dl = 0; dl < DTW; ++dl) o[ht][dl] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // running maximum and sum of heads 16 hw + 4 qd + r (all 16 lanes of a row agree)
  float m_run[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY}, l_run[4] = {0.f, 0.f, 0.f, 0.f};
  if (nblk > 0) {
    if constexpr (FP8) {
      issue_fp8(0);
      if (nblk > 1) issue_fp8(1);
      wait_stage(nblk > 1 ? 1 : 0);
      convert_fp8(0);
      if (nblk > 2) issue_fp8(2);
    } else {
      issue_bf16(0);
      fill_bf16(0);
    }
  }
  // V transpose reads: lane 4 vi + vj of group qd points at block token
  // 8 qd + 2 vi (+ 1 for the second read), columns 4 vj .. 4 vj + 3 of a tile
  const int vi = c >> 2, vj = c & 3;
  for (int blk = 0; blk < nblk; ++blk) {
    const int bf = blk & 1;
    const int* bid = &Ids[blk * kMlaBT];
    __syncthreads();  // buffer bf is filled; buffer bf ^ 1, its stage, P and the rescale flags are no longer read
    const bool more = blk + 1 < nblk;
    if constexpr (FP8) {
      if (blk + 3 < nblk) issue_fp8(blk + 3);  // into the stage block blk came from
    } else {
      if (more) issue_bf16(blk + 1);  // block blk + 1 flies while block blk is multiplied out
    }
    if (scorer) {  // QK and the online softmax of head tile wv
      // S tiles (rows = heads 4 qd + r of the tile, column = slot 16 j + c): A = q
      // (registers), B = K rows; two accumulators per tile (even and odd K steps)
      // halve the dependent MFMA chain.  The ids of this lane's two tokens are
      // read first so that their LDS latency hides behind the products.
      bool live[kMlaBT / 16];
#pragma unroll
      for (int j = 0; j < kMlaBT / 16; ++j) live[j] = bid[mla_slot_token(16 * j + c)] >= 0;
      f32x4_t st[kMlaBT / 16], st2[kMlaBT / 16];
#pragma unroll
      for (int j = 0; j < kMlaBT / 16; ++j) st[j] = st2[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      // K fragments in batches of KB steps, double-buffered: batch i + 1's LDS
      // reads are issued before batch i's products (the scheduling barriers keep
      // the compiler from interleaving them into a read-wait-multiply chain)
      constexpr int KB = 3, NSQ = DQK / 32, NKB = (NSQ + KB - 1) / KB;
      bf16x8_t kop[2][KB][kMlaBT / 16];
      int krow[kMlaBT / 16];
#pragma unroll
      for (int j = 0; j < kMlaBT / 16; ++j) krow[j] = mla_slot_token(16 * j + c) * KS + 8 * qd;
      auto read_k = [&](int kb2, bf16x8_t (&dst)[KB][kMlaBT / 16]) {
#pragma unroll
        for (int ss = 0; ss < KB; ++ss)
#pragma unroll
          for (int j = 0; j < kMlaBT / 16; ++j)
            if (kb2 * KB + ss < NSQ)
              dst[ss][j] = *reinterpret_cast<const bf16x8_t*>(&Kt[bf][krow[j] + 32 * (kb2 * KB + ss)]);
      };
      read_k(0, kop[0]);
#pragma unroll
      for (int kb2 = 0; kb2 < NKB; ++kb2) {
        if (kb2 + 1 < NKB) read_k(kb2 + 1, kop[(kb2 + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ss = 0; ss < KB; ++ss)
#pragma unroll
          for (int j = 0; j < kMlaBT / 16; ++j) {
            const int s = kb2 * KB + ss;
            if (s >= NSQ) continue;
            if (s & 1)
              st2[j] = mfma_bf16(qb[s], kop[kb2 & 1][ss][j], st2[j]);
            else
              st[j] = mfma_bf16(qb[s], kop[kb2 & 1][ss][j], st[j]);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < kMlaBT / 16; ++j) st[j] += st2[j];
      // online softmax of heads 4 qd + r: reductions over the 16 lanes of a row
      float sc[kMlaBT / 16][4], p[kMlaBT / 16][4], alpha[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float bm = -INFINITY;
#pragma unroll
        for (int j = 0; j < kMlaBT / 16; ++j) {
          sc[j][r] = live[j] ? st[j][r] * scale : -INFINITY;
          bm = fmaxf(bm, sc[j][r]);
        }
        bm = row16_max(bm);
        // the running maximum moves only past the lazy margin (or from -inf)
        const bool move = bm > m_run[r] + kMlaLazyMax;
        const float m_new = move ? bm : m_run[r];
        alpha[r] = (move && m_run[r] != -INFINITY) ? __expf(m_run[r] - m_new) : 1.f;
        float psum = 0.f;
#pragma unroll
        for (int j = 0; j < kMlaBT / 16; ++j) {
          p[j][r] = m_new == -INFINITY ? 0.f : __expf(sc[j][r] - m_new);
          psum += p[j][r];
        }
        l_run[r] = l_run[r] * alpha[r] + row16_sum(psum);
        m_run[r] = m_new;
      }
      // P (bf16, rows = the tile's heads, columns = slots) and the heads' O
      // rescale factors into LDS; a flag per wave says whether any is not 1
#pragma unroll
      for (int j = 0; j < kMlaBT / 16; ++j)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          const uint32_t pw =
              __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{p[j][r], p[j][r + 1]}, bf16x2_t));
          Ps[(16 * wv + 4 * qd + r) * kPsStride + 16 * j + c] = (uint16_t)(pw & 0xFFFFu);
          Ps[(16 * wv + 4 * qd + r + 1) * kPsStride + 16 * j + c] = (uint16_t)(pw >> 16);
        }
      if (c == 0) *reinterpret_cast<f32x4_t*>(&As[16 * wv + 4 * qd]) = f32x4_t{alpha[0], alpha[1], alpha[2], alpha[3]};
      const bool rescale = __ballot(alpha[0] != 1.f || alpha[1] != 1.f || alpha[2] != 1.f || alpha[3] != 1.f) != 0;
      if (lane == 0) Fl[wv] = rescale ? 1 : 0;
    }
    __syncthreads();  // P, the factors and the flags of every wave are in
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      if (__builtin_amdgcn_readfirstlane(Fl[ht])) {  // the same word for every lane
        const f32x4_t al = *reinterpret_cast<const f32x4_t*>(&As[16 * ht + 4 * qd]);
#pragma unroll
        for (int dl = 0; dl < DTW; ++dl) o[ht][dl] *= al;
      }
    }
    // O += P V over this wave's column tiles: A = P rows of every head tile
    // (k = slots 8 qd .. 8 qd + 7), B = V by two transpose reads per tile
    bf16x8_t pa[HT];
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) pa[ht] = *reinterpret_cast<const bf16x8_t*>(&Ps[(16 * ht + c) * kPsStride + 8 * qd]);
    const uint16_t* vbase = &Kt[bf][(8 * qd + 2 * vi) * KS + 4 * vj];
    constexpr int VB = 4, NVB = DTW / VB;
    bf16x8_t vv[2][VB];
    auto read_v = [&](int vb2, bf16x8_t (&dst)[VB]) {
#pragma unroll
      for (int dd = 0; dd < VB; ++dd) {
        const uint16_t* vp = vbase + 16 * (dt0 + vb2 * VB + dd);
        const mla_v4s a = lds_read_tr16(vp), e = lds_read_tr16(vp + KS);
        dst[dd] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a, e, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    read_v(0, vv[0]);
#pragma unroll
    for (int vb2 = 0; vb2 < NVB; ++vb2) {
      if (vb2 + 1 < NVB) read_v(vb2 + 1, vv[(vb2 + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int dd = 0; dd < VB; ++dd)
#pragma unroll
        for (int ht = 0; ht < HT; ++ht)
          o[ht][vb2 * VB + dd] = mfma_bf16(pa[ht], vv[vb2 & 1][dd], o[ht][vb2 * VB + dd]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (more) {
      if constexpr (FP8) {
        wait_stage(min(2, nblk - blk - 2));  // block blk + 1's copies (of every wave) have landed
        convert_fp8(blk + 1);
      } else {
        fill_bf16(blk + 1);
      }
    }
  }
  // partial O (bf16, un-normalized) in MFMA tile order:
  // part_o[b][split][head tile][column tile][lane][4] (rows = heads 16 tile + 4 qd + r,
  // column 16 tile + c); bf16 halves the partials' store and the combine's read
  uint16_t* po = part_o + ((int64_t)b * S + split) * (H / 16) * (kMlaDt * 256);
#pragma unroll
  for (int ht = 0; ht < HT; ++ht)
#pragma unroll
    for (int dl = 0; dl < DTW; ++dl) {
      const f32x4_t v = o[ht][dl];
      *reinterpret_cast<uint2*>(po + (((int64_t)(blockIdx.z * HT + ht) * kMlaDt + dt0 + dl) * 64 + lane) * 4) =
          uint2{(uint32_t)f32_bf16(v[0]) | ((uint32_t)f32_bf16(v[1]) << 16),
                (uint32_t)f32_bf16(v[2]) | ((uint32_t)f32_bf16(v[3]) << 16)};
    }
  if (scorer && c == 0) {
    float* pml = part_ml + (((int64_t)b * S + split) * H + 16 * hw + 4 * qd) * 2;
    *reinterpret_cast<f32x4_t*>(pml) = f32x4_t{m_run[0], l_run[0], m_run[1], l_run[1]};
    *reinterpret_cast<f32x4_t*>(pml + 4) = f32x4_t{m_run[2], l_run[2], m_run[3], l_run[3]};
  }
}

// Four partial values of a lane, bf16 or fp32
__device__ __forceinline__ void store_part(uint16_t* p, f32x4_t v) {
  *reinterpret_cast<uint2*>(p) = uint2{__builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{v[0], v[1]}, bf16x2_t)),
                                       __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{v[2], v[3]}, bf16x2_t))};
}
__device__ __forceinline__ void store_part(float* p, f32x4_t v) { *reinterpret_cast<f32x4_t*>(p) = v; }
__device__ __forceinline__ f32x4_t part_value(uint2 raw) {
  return f32x4_t{__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xFFFF0000u), __uint_as_float(raw.y << 16),
                 __uint_as_float(raw.y & 0xFFFF0000u)};
}
__device__ __forceinline__ f32x4_t part_value(f32x4_t raw) { return raw; }
template <typename TP>
struct MlaPart;  // a lane's load of four partial values
template <>
struct MlaPart<uint16_t> {
  typedef uint2 vec;
};
template <>
struct MlaPart<float> {
  typedef f32x4_t vec;
};

// A split of at most 128 selected tokens of one row and 64 heads over an FP8
// cache, all tokens at once: decode calls of a few rows are bound by the chain
// of latencies of a split (ids, gather, conversion, scores, softmax, values),
// which the block loop above pays once per 32 tokens.  Here each step runs once
// over the whole split, on eight waves (two a SIMD, so that one's LDS reads
// overlap the other's products).
//
//   * every thread loads its tokens' ids, then 8 16-byte pieces of latent rows
//     with their scales and 2 of rope rows, straight to registers, and writes
//     them to LDS as bf16 (rounded as act_quant_sim stores them; zeros for masked
//     tokens);
//   * wave w scores tokens 32 (w / 2) .. + 31 against heads 32 (w % 2) .. + 31
//     (S^T = K Q^T: q in registers, each K fragment used for two head tiles); the
//     heads' maxima over the four token quarters meet in LDS, then the
//     probabilities go to LDS over the rope rows, which are no longer needed;
//   * wave w multiplies all heads into columns 64 w .. + 63, V read out of the
//     latent rows with transposing reads.
// Partials are laid out as the block kernel's, in fp32 up to kMdF32Chunks splits:
// a row of few large splits averages their bf16 roundings less than the block
// kernel's many small ones (512 picks, relative error against 64 bits: 2.4e-3 on
// the block kernel, 2.5e-3 with bf16 partials here).  q goes through LDS first (its
// fragments straight from memory cost 36 scattered loads a wave, 8 us of the
// chain).  Measured, 8 rows x 128 heads x 2048 picks: the whole call 32.1 -> 22.4
// us, of which this kernel takes 17.1 in a kernel trace and the combine 7.1; what is
// left is the chain itself (about 24,000 cycles by timestamps in a scratch build:
// ids and q 9,000, conversion 4,000, scores 3,400, softmax 2,300, values 2,700,
// stores 1,800).
constexpr int kMdTokens = 128;
constexpr int kMdF32Chunks = 8;      // up to this many splits store fp32 partials
constexpr int kMdRow = kMlaDl + 8;   // bf16 per latent row in LDS
constexpr int kMdRope = 64 + 8;      // bf16 per rope row
constexpr int kMdPs = kMdTokens + 8; // bf16 per row of P
static_assert(64 * kMdPs <= kMdTokens * kMdRope, "P overlays the rope rows");
constexpr int kMdQCopies = 64 * (kMlaDl + 64) * 2 / 1024 / 8;  // 1 KB copies of q a wave
constexpr int kMdLat = kMdTokens * kMlaDl / (512 * 16);        // latent pieces (16 bytes) a thread, each with its scale
constexpr int kMdRopes = kMdTokens * 64 * 2 / (512 * 16);      // rope pieces (16 bytes) a thread
// Vector loads a wave issues between q's copies and the wait for them.  Loads
// complete in order, so at most this many in flight means that q has landed;
// tests/test_codegen.py counts them in the built kernel (fewer, merged or moved
// past the wait, would let waves read q's LDS early).
constexpr int kMdGather = 2 * kMdLat + kMdRopes;
static_assert(64 * (kMlaDl + 64) <= kMdTokens * kMdRow, "q is staged where the latent rows go");

template <typename TP>
__global__ void __launch_bounds__(512) mla_decode_chunk_kernel(const uint16_t* __restrict__ q, const MlaKv kv,
                                                               const int32_t* __restrict__ idx,
                                                               TP* __restrict__ part_o, float* __restrict__ part_ml,
                                                               int topk, float scale) {
  constexpr int DQK = kMlaDl + 64, NS = DQK / 32, NSL = kMlaDl / 32;
  __shared__ __attribute__((aligned(16))) uint16_t Kt[kMdTokens * kMdRow];
  __shared__ __attribute__((aligned(16))) uint16_t Rp[kMdTokens * kMdRope];
  __shared__ float Mx[4][64], Lx[4][64];
  __shared__ int Live[kMdTokens];
  const int H = 64 * gridDim.z;
  const int split = blockIdx.x, b = blockIdx.y, S = gridDim.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, qd = lane >> 4;
  const int64_t n = kv.n, kvb = (int64_t)(b / kv.rows_per_kv) * n;
  const int t0 = split * kMdTokens, nt = min(kMdTokens, topk - t0);  // tokens of this split (> 0)
  const int nblk = (nt + 31) / 32;
  const int nsc = kMlaDl >> kv.sb_shift;
  // the group's q rows (73,728 contiguous bytes) into LDS, each row's 16-byte
  // chunks XOR-swizzled by (row / 2) % 8 within eights, so that the 16 rows of a
  // fragment read fall in distinct banks
  const int hh = wv & 1, tb = wv >> 1;
  {
    const uint16_t* qg = q + ((int64_t)b * H + 64 * blockIdx.z) * DQK;
#pragma unroll
    for (int i = 0; i < kMdQCopies; ++i) {
      const int u = 64 * (kMdQCopies * wv + i) + lane, r = u / (DQK / 8), p = u - r * (DQK / 8);
      mla_copy16(qg + r * DQK + 8 * (p ^ ((r >> 1) & 7)), mla_lds_addr(&Kt[512 * (kMdQCopies * wv + i)]));
    }
  }
  // Wave wv gathers tokens 16 i + 2 wv + {0, 1}: latent piece i is token 2 wv +
  // lane / 32 of the i-th 16, bytes 16 (lane % 32); rope piece j covers eight of
  // the tokens, 8 values at 8 (lane % 8).  The ids are wave-uniform and come by
  // scalar loads.  (The choice between a half-wave's two ids compiles to private
  // memory, 80 bytes a lane, whose loads come back behind q's copies: the gather's
  // addresses wait for q, a part of the 9,000 cycles above.)
  const int32_t* ids = idx + (int64_t)b * topk + t0;
  const int lp = lane & 31, rp = lane & 7, lt = 2 * wv + (lane >> 5);
  int id2[kMdLat][2];
#pragma unroll
  for (int i = 0; i < kMdLat; ++i)
#pragma unroll
    for (int u = 0; u < 2; ++u) id2[i][u] = ids[min(16 * i + 2 * wv + u, nt - 1)];
  __builtin_amdgcn_sched_barrier(0);  // the loads first: a wait for eight of them at a time
#pragma unroll
  for (int i = 0; i < kMdLat; ++i)
#pragma unroll
    for (int u = 0; u < 2; ++u)  // (a negative id stays negative)
      id2[i][u] = 16 * i + 2 * wv + u < nt && (int64_t)id2[i][u] < n ? id2[i][u] : -1;
  int lid[kMdLat], rid[kMdRopes], rt[kMdRopes];
#pragma unroll
  for (int i = 0; i < kMdLat; ++i) lid[i] = lane < 32 ? id2[i][0] : id2[i][1];
#pragma unroll
  for (int j = 0; j < kMdRopes; ++j) {
    rid[j] = id2[4 * j][0];
#pragma unroll
    for (int g = 1; g < 8; ++g) rid[j] = (lane >> 3) == g ? id2[4 * j + (g >> 1)][g & 1] : rid[j];
    rt[j] = 16 * (4 * j + (lane >> 4)) + 2 * wv + ((lane >> 3) & 1);
  }
  // masked tokens read row 0 and are zeroed below (loads under a branch would be
  // waited for at its end)
  u32x4_t raw[kMdLat], rope[kMdRopes];
  float sc[kMdLat];
#pragma unroll
  for (int i = 0; i < kMdLat; ++i) {
    const int64_t r = kvb + max(lid[i], 0);
    raw[i] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint8_t*>(kv.lat) + r * kMlaDl + 16 * lp);
    sc[i] = kv.lat_s[r * nsc + ((16 * lp) >> kv.sb_shift)];
  }
#pragma unroll
  for (int i = 0; i < kMdRopes; ++i) {
    rope[i] = *reinterpret_cast<const u32x4_t*>(kv.rope + (kvb + max(rid[i], 0)) * 64 + 8 * rp);
  }
  // q has landed (the gather may still fly); it becomes the B operand of S^T:
  // heads 32 hh + 16 t + c of the group
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(kMdGather) : "memory");
  bf16x8_t qf[2][NS];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int r = 32 * hh + 16 * t + c;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      qf[t][s] = *reinterpret_cast<const bf16x8_t*>(&Kt[r * DQK + 8 * ((4 * s + qd) ^ ((r >> 1) & 7))]);
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // q's LDS may be overwritten
  if (lp == 0) {
#pragma unroll
    for (int i = 0; i < kMdLat; ++i) Live[16 * i + lt] = lid[i] >= 0 ? 1 : 0;
  }
#pragma unroll
  for (int i = 0; i < kMdLat; ++i) {
    uint32_t o[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      // exact e4m3 -> fp32, fp32 product with the scale, one RNE rounding to bf16
      f32x2_t a2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)raw[i][e], false);
      f32x2_t b2 = __builtin_amdgcn_cvt_pk_f32_fp8((int)raw[i][e], true);
      a2[0] *= sc[i];
      a2[1] *= sc[i];
      b2[0] *= sc[i];
      b2[1] *= sc[i];
      o[2 * e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(a2, bf16x2_t));
      o[2 * e + 1] = __builtin_bit_cast(uint32_t, __builtin_convertvector(b2, bf16x2_t));
    }
    u32x4_t* dst = reinterpret_cast<u32x4_t*>(&Kt[(16 * i + lt) * kMdRow + 16 * lp]);
    const bool ok = lid[i] >= 0;
    dst[0] = ok ? u32x4_t{o[0], o[1], o[2], o[3]} : u32x4_t{0u, 0u, 0u, 0u};
    dst[1] = ok ? u32x4_t{o[4], o[5], o[6], o[7]} : u32x4_t{0u, 0u, 0u, 0u};
  }
#pragma unroll
  for (int i = 0; i < kMdRopes; ++i) {
    *reinterpret_cast<u32x4_t*>(&Rp[rt[i] * kMdRope + 8 * rp]) = rid[i] >= 0 ? rope[i] : u32x4_t{0u, 0u, 0u, 0u};
  }
  __syncthreads();
  // scores of this wave's 32 tokens (slot order, see mla_slot_token) x 32 heads
  f32x4_t st[2][2];  // [head tile][slot tile]
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) st[t][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  bool live[2][4];
  const bool scorer = tb < nblk;
  if (scorer) {
    int krow[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      krow[j] = 32 * tb + mla_slot_token(16 * j + c);
#pragma unroll
      for (int r = 0; r < 4; ++r) live[j][r] = Live[32 * tb + mla_slot_token(16 * j + 4 * qd + r)] != 0;
    }
    // K fragments in batches of KB steps, one batch ahead of the products
    constexpr int KB = 3, NKB = NS / KB;
    bf16x8_t kf[2][KB][2];
    auto read_k = [&](int kb2, bf16x8_t (&dst)[KB][2]) {
#pragma unroll
      for (int ss = 0; ss < KB; ++ss)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int s = kb2 * KB + ss;
          dst[ss][j] = *reinterpret_cast<const bf16x8_t*>(s < NSL ? &Kt[krow[j] * kMdRow + 32 * s + 8 * qd]
                                                                  : &Rp[krow[j] * kMdRope + 32 * (s - NSL) + 8 * qd]);
        }
    };
    read_k(0, kf[0]);
#pragma unroll
    for (int kb2 = 0; kb2 < NKB; ++kb2) {
      if (kb2 + 1 < NKB) read_k(kb2 + 1, kf[(kb2 + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ss = 0; ss < KB; ++ss)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int j = 0; j < 2; ++j) st[t][j] = mfma_bf16(kf[kb2 & 1][ss][j], qf[t][kb2 * KB + ss], st[t][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    float bm = -INFINITY;
    if (scorer) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          st[t][j][r] = live[j][r] ? st[t][j][r] * scale : -INFINITY;
          bm = fmaxf(bm, st[t][j][r]);
        }
      bm = fmaxf(bm, __shfl_xor(bm, 16));
      bm = fmaxf(bm, __shfl_xor(bm, 32));
    }
    if (qd == 0) Mx[tb][32 * hh + 16 * t + c] = bm;
  }
  __syncthreads();  // the maxima are in, and no wave reads the rope rows any more
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int hd = 32 * hh + 16 * t + c;
    const float m = fmaxf(fmaxf(Mx[0][hd], Mx[1][hd]), fmaxf(Mx[2][hd], Mx[3][hd]));
    float l = 0.f;
    if (scorer) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[r] = m == -INFINITY ? 0.f : __expf(st[t][j][r] - m);
          l += p[r];
        }
        *reinterpret_cast<uint2*>(&Rp[hd * kMdPs + 32 * tb + 16 * j + 4 * qd]) =
            uint2{__builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{p[0], p[1]}, bf16x2_t)),
                  __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{p[2], p[3]}, bf16x2_t))};
      }
      l += __shfl_xor(l, 16);
      l += __shfl_xor(l, 32);
    }
    if (qd == 0) Lx[tb][hd] = l;
  }
  __syncthreads();
  // O = P V over this wave's 64 columns
  f32x4_t o[4][4];
#pragma unroll
  for (int ht = 0; ht < 4; ++ht)
#pragma unroll
    for (int dl = 0; dl < 4; ++dl) o[ht][dl] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int vi = c >> 2, vj = c & 3;
  for (int bk = 0; bk < nblk; ++bk) {
    bf16x8_t pa[4], vv[4];
#pragma unroll
    for (int ht = 0; ht < 4; ++ht)
      pa[ht] = *reinterpret_cast<const bf16x8_t*>(&Rp[(16 * ht + c) * kMdPs + 32 * bk + 8 * qd]);
#pragma unroll
    for (int dl = 0; dl < 4; ++dl) {
      const uint16_t* vp = &Kt[(32 * bk + 8 * qd + 2 * vi) * kMdRow + 4 * vj + 64 * wv + 16 * dl];
      const mla_v4s a = lds_read_tr16(vp), e = lds_read_tr16(vp + kMdRow);
      vv[dl] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a, e, 0, 1, 2, 3, 4, 5, 6, 7));
    }
#pragma unroll
    for (int dl = 0; dl < 4; ++dl)
#pragma unroll
      for (int ht = 0; ht < 4; ++ht) o[ht][dl] = mfma_bf16(pa[ht], vv[dl], o[ht][dl]);
  }
  TP* po = part_o + ((int64_t)b * S + split) * (H / 16) * (kMlaDt * 256);
#pragma unroll
  for (int ht = 0; ht < 4; ++ht)
#pragma unroll
    for (int dl = 0; dl < 4; ++dl)
      store_part(po + (((int64_t)(4 * blockIdx.z + ht) * kMlaDt + 4 * wv + dl) * 64 + lane) * 4, o[ht][dl]);
  if (tid < 64) {
    const float m = fmaxf(fmaxf(Mx[0][tid], Mx[1][tid]), fmaxf(Mx[2][tid], Mx[3][tid]));
    const float l = (Lx[0][tid] + Lx[1][tid]) + (Lx[2][tid] + Lx[3][tid]);
    float* pml = part_ml + (((int64_t)b * S + split) * H + 64 * blockIdx.z + tid) * 2;
    *reinterpret_cast<f32x2_t*>(pml) = f32x2_t{m, l};
  }
}

// Merge the splits of one (row, 16-head tile, 16-column tile) with the sink
// term and normalize.  Each wave turns the split maxima/sums of four heads
// into weights (lane = split); then wave w blends splits w, w + 4, ... of the
// tile's 64 x 4 partial values, and wave 0 sums the four and writes bf16.
template <typename TP>
__global__ void __launch_bounds__(256) mla_combine_kernel(const TP* __restrict__ part_o,
                                                          const float* __restrict__ part_ml,
                                                          const float* __restrict__ sink, uint16_t* __restrict__ out,
                                                          int H, int S) {
  __shared__ float wgt[kMlaMaxSplits][16];
  __shared__ f32x4_t red[4][64];
  const int dt = blockIdx.x, ht = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int hh = 4 * wv + k, h = 16 * ht + hh;
    const bool ok = lane < S;
    const float m = ok ? part_ml[(((int64_t)b * S + lane) * H + h) * 2] : -INFINITY;
    const float l = ok ? part_ml[(((int64_t)b * S + lane) * H + h) * 2 + 1] : 0.f;
    // DPP max (exact in any order); a NaN lane is left out, as fmaxf would
    const float M = wave_max_f32(m == m ? m : -INFINITY);
    const float e = (m == -INFINITY) ? 0.f : __expf(m - M);
    const float lsum = wave_sum_f32(l * e) + ((sink && M != -INFINITY) ? __expf(sink[h] - M) : 0.f);
    if (ok) wgt[lane][hh] = (M == -INFINITY) ? 0.f : e / lsum;
  }
  __syncthreads();
  const int hq = lane >> 4;  // rows 4 hq + r of the tile
  const int64_t sstride = (int64_t)(H / 16) * kMlaDt * 256;
  const TP* po = part_o + (int64_t)b * S * sstride + ((int64_t)ht * kMlaDt + dt) * 256 + lane * 4;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = wv; s < S; s += 4) {
    const f32x4_t v = part_value(*reinterpret_cast<const typename MlaPart<TP>::vec*>(po + s * sstride));
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] += wgt[s][4 * hq + r] * v[r];
  }
  red[wv][lane] = acc;
  __syncthreads();
  if (wv == 0) {
    const f32x4_t v = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      out[((int64_t)b * H + 16 * ht + 4 * hq + r) * kMlaDl + 16 * dt + (lane & 15)] = f32_bf16(v[r]);
  }
}

// The same merge for grids of many rows: a workgroup takes four 16-column
// tiles, and wave w blends every split of column tile 4 x + w (x = blockIdx.x)
// in split order and writes bf16 (no cross-wave sum).  A wave's first 32
// splits are loaded before the weights are formed.  Four times fewer
// workgroups, each reading its splits' tiles once: used from 4 rows of 128
// heads up (B = 8: 35.7 -> 33.7 us a call; at B = 1 the 64 workgroups were
// slower, 19.5 against 17.5 us).
constexpr int kMlaCombineTiles = 4;  // 16-column tiles a workgroup

template <typename TP>
__global__ void __launch_bounds__(256) mla_combine_tiles_kernel(const TP* __restrict__ part_o,
                                                          const float* __restrict__ part_ml,
                                                          const float* __restrict__ sink, uint16_t* __restrict__ out,
                                                          int H, int S) {
  __shared__ float wgt[kMlaMaxSplits][16];
  const int ht = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int dt = blockIdx.x * kMlaCombineTiles + wv;
  const int hq = lane >> 4;  // rows 4 hq + r of the tile
  const int64_t sstride = (int64_t)(H / 16) * kMlaDt * 256;
  const TP* po = part_o + (int64_t)b * S * sstride + ((int64_t)ht * kMlaDt + dt) * 256 + lane * 4;
  typedef typename MlaPart<TP>::vec vec_t;
  constexpr int CH = sizeof(TP) == 2 ? 32 : kMdF32Chunks;
  vec_t raw[CH];
  auto load_chunk = [&](int s0) {
#pragma unroll
    for (int i = 0; i < CH; ++i)
      raw[i] = s0 + i < S ? *reinterpret_cast<const vec_t*>(po + (s0 + i) * sstride) : vec_t{};
  };
  load_chunk(0);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int hh = 4 * wv + k, h = 16 * ht + hh;
    const bool ok = lane < S;
    const float m = ok ? part_ml[(((int64_t)b * S + lane) * H + h) * 2] : -INFINITY;
    const float l = ok ? part_ml[(((int64_t)b * S + lane) * H + h) * 2 + 1] : 0.f;
    // DPP max (exact in any order); a NaN lane is left out, as fmaxf would
    const float M = wave_max_f32(m == m ? m : -INFINITY);
    const float e = (m == -INFINITY) ? 0.f : __expf(m - M);
    const float lsum = wave_sum_f32(l * e) + ((sink && M != -INFINITY) ? __expf(sink[h] - M) : 0.f);
    if (ok) wgt[lane][hh] = (M == -INFINITY) ? 0.f : e / lsum;
  }
  __syncthreads();
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < S; s0 += CH) {
    if (s0) load_chunk(s0);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if (s0 + i < S) {
        const f32x4_t v = part_value(raw[i]);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] += wgt[s0 + i][4 * hq + r] * v[r];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    out[((int64_t)b * H + 16 * ht + 4 * hq + r) * kMlaDl + 16 * dt + (lane & 15)] = f32_bf16(acc[r]);
}

// Sparse attention of many query rows (a prompt) over a bf16 cache of 512-wide
// rows (V = K).  An item is one (row, group of 16 HT heads); its whole pick
// list goes through one workgroup and the normalized output is written
// directly, so there are no partials and no combine.  At most one workgroup of
// eight waves a CU walks the items w, w + grid, ...
//
// An item's valid picks are compacted first (order kept), so masked picks cost
// nothing and only the last block's tail is masked.  Blocks of 32 picks move
// through a ring of four LDS stages by global -> LDS copies (one 1 KB row an
// instruction), issued three blocks ahead by the value waves.  Waves 0..3 score
// block p (wave w: head tile w, q in registers; K rows from LDS) and soft-max it
// into P, while waves 4..7 multiply block p - 1 (wave 4 + w: columns 128 w ..
// + 127 of every head tile, V read out of the K rows with transposing reads), so
// each SIMD holds one wave of either kind and the two contractions, the
// softmax chain and the LDS reads overlap.  The first K fragments of a block
// and all its V fragments are read in the period before their products.  One
// barrier a period hands over the stage, P and the rescale factors.  Both
// products have the picks' or columns' side as their MFMA rows, so a lane's
// entries share a head.
//
// The items' blocks form one sequence: the next item's picks are loaded at the
// start of an item and compacted during it, its first blocks are copied during
// the last three periods, its q is prefetched, and the value waves normalize and
// store an item while the scoring waves are in the next one.  An item takes at
// least kMrMinPeriods periods (the compaction's hand-overs).
//
// Bound by the chains of a period (scoring: 32 MFMAs on LDS operands, then the
// softmax; value: copies, then 32 MFMAs) and by the gather, 32 KB a block and
// CU: a call of 2048 rows x 64 heads x 512 with 128 + up to 512 picks 666 -> 178 us
// (570 TFLOP/s on the valid picks), of which copies alone take ~100.  All 256
// registers are taken and 9 spill: the scoring waves reload them between the pick
// loads at an item's start.
constexpr int kMrStages = 4;
constexpr int kMrRow = kMlaDl * 2 + 16;  // bytes per staged row
constexpr int kMrStage = kMlaBT * kMrRow;
constexpr int kMrMaxPicks = 2048;
constexpr int kMrMinRows = 64;
constexpr int kMrCopies = kMlaBT / 4;  // copies a value wave a block
constexpr int kMrMinPeriods = 8;
constexpr int kMrPer = kMrMaxPicks / 512;  // picks a thread
constexpr float kLog2e = 1.4426950408889634f;

template <int HT>
__global__ void __launch_bounds__(512) mla_rows_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ kv,
                                                       const int32_t* __restrict__ idx, const float* __restrict__ sink,
                                                       uint16_t* __restrict__ out, int64_t n, int rows,
                                                       int rows_per_kv, int n_groups, int topk, float scale) {
  constexpr int NSQ = kMlaDl / 32, DTW = kMlaDt / 4;
  constexpr int KS = kMrRow / 2;
  __shared__ __attribute__((aligned(16))) uint8_t Kt[kMrStages * kMrStage];
  __shared__ __attribute__((aligned(16))) uint16_t Ps[2][16 * HT * kPsStride];
  __shared__ float As[2][16 * HT], Ml[2][16 * HT];
  __shared__ int Fl[2][HT];
  __shared__ int Ids[2][kMrMaxPicks];
  __shared__ int cnt[kMrPer][8];
  __shared__ float Sink[256];  // heads <= 256
  const int H = HT * 16 * n_groups;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, qd = lane >> 4;
  const int n_items = rows * n_groups;
  // item -> row (a prompt's last rows have the most picks: first) and head group
  auto row_of = [&](int it) { return rows - 1 - it / n_groups; };
  int idv[kMrPer], before[kMrPer];
  auto load_picks = [&](int it) {
    const int64_t r0 = (int64_t)row_of(it) * topk;
#pragma unroll
    for (int k = 0; k < kMrPer; ++k) {
      const int t = 512 * k + tid;
      idv[k] = t < topk ? idx[r0 + t] : -1;
    }
  };
  // compaction, first half: each wave's valid picks counted
  auto count_picks = [&]() {
#pragma unroll
    for (int k = 0; k < kMrPer; ++k) {
      const bool ok = idv[k] >= 0 && (int64_t)idv[k] < n;
      if (!ok) idv[k] = -1;
      const uint64_t mask = __ballot(ok);
      before[k] = __popcll(mask & ((1ull << lane) - 1));
      if (lane == 0) cnt[k][wv] = __popcll(mask);
    }
  };
  // second half, a barrier later: the picks into `dst` in order; returns their number
  auto place_picks = [&](int* dst) {
    int nv = 0;
#pragma unroll
    for (int k = 0; k < kMrPer; ++k)
#pragma unroll
      for (int w = 0; w < 8; ++w) {
        if (w == wv && idv[k] >= 0) dst[nv + before[k]] = idv[k];
        nv += cnt[k][w];
      }
    return __builtin_amdgcn_readfirstlane(nv);
  };
  auto blocks_of = [&](int nv) { return (nv + kMlaBT - 1) / kMlaBT; };
  int it = blockIdx.x;  // grid <= n_items
  load_picks(it);
  if (sink && tid < H) Sink[tid] = sink[tid];
  count_picks();
  __syncthreads();
  int nv = place_picks(Ids[0]), nv_next = 0;
  __syncthreads();
  int par = 0;     // picks buffer of the current item
  int stage = 0;   // ring stage of the item's next block (the period's block p)
  int period = 0;  // parity of P, the factors and the flags
  // copies of block j of an item into a stage: rows 4 wv + i; slots past the
  // last pick repeat its row (masked in the softmax).  The wave's picks are read
  // ahead (lane i: row i), so an issue waits for no LDS round trip.
  auto read_ids = [&](const int* ids, int nvj, int j) {
    return ids[max(0, min(j * kMlaBT + kMrCopies * (wv & 3) + (lane & (kMrCopies - 1)), nvj - 1))];
  };
  auto issue = [&](int ids4, const uint16_t* base, int stg, int i) {
    mla_copy16_s(base + (int64_t)__builtin_amdgcn_readlane(ids4, i) * kMlaDl, 16 * lane,
                 mla_lds_addr(&Kt[(stg % kMrStages) * kMrStage + (kMrCopies * (wv - 4) + i) * kMrRow]));
  };
  auto cache_of = [&](int i) { return kv + (int64_t)(row_of(i) / rows_per_kv) * n * kMlaDl; };
  // every copy of this wave but those of this period has landed, then the
  // barrier (a value wave's stores of an item are its period's last, and may fly)
  constexpr int kStores = HT * DTW / 2;
  auto hand_over = [&](bool flying, bool stored) {
    if (wv < 4)
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else if (flying && stored)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kMrCopies + kStores) : "memory");
    else if (stored)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kStores) : "memory");
    else if (flying)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kMrCopies) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  const uint16_t* kvb = cache_of(it);  // the item's cache, and the next one's (set once an item: divisions)
  const uint16_t* kvn = kvb;
  for (int j = 0; j < (wv < 4 ? 0 : min(3, blocks_of(nv))); ++j) {
    const int ids4 = read_ids(Ids[0], nv, j);
#pragma unroll
    for (int i = 0; i < kMrCopies; ++i) issue(ids4, kvb, j, i);
  }
  int id4 = read_ids(Ids[0], nv, 3);  // the picks of the next block to copy
  // One period's shared work at period p of the item: the next item's picks, and
  // the copies three blocks ahead (of this item, or the next one's first three),
  // set up here and issued by copy().
  bool cp_on = false;
  const uint16_t* cp_base = nullptr;
  int cp_ids = 0, cp_stage = 0;
  auto advance = [&](int p, int nblk, int nper, int next) {
    if (next < n_items) {
      if (p == 2) count_picks();
      if (p == 3) nv_next = place_picks(Ids[par ^ 1]);
    }
    if (wv < 4) return;
    const int j = p + 3 - nper;  // block of the next item (nper >= 8: its picks were placed a barrier ago)
    const bool own = p + 3 < nblk;
    cp_on = own || (j >= 0 && next < n_items && j < blocks_of(nv_next));
    cp_ids = id4;
    cp_base = own ? kvb : kvn;
    // (the stages the current item has left count from its end)
    cp_stage = own ? stage + 3 : stage + (nblk > p ? nblk - p : 0) + j;
    // next period: block p + 4 of this item, or block j + 1 of the next
    id4 = j + 1 >= 0 ? read_ids(Ids[par ^ 1], nv_next, j + 1) : read_ids(Ids[par], nv, p + 4);
  };
  auto copy = [&]() {
    if (!cp_on) return;
#pragma unroll
    for (int i = 0; i < kMrCopies; ++i) issue(cp_ids, cp_base, cp_stage, i);
  };
  if (wv < 4) {
    const bool scorer = wv < HT;
    bf16x8_t qn[NSQ];
    auto load_q = [&](int i) {
      const uint16_t* qrow =
          q + ((int64_t)row_of(i) * H + 16 * ((i % n_groups) * HT + (scorer ? wv : 0)) + c) * kMlaDl;
#pragma unroll
      for (int s = 0; s < NSQ; ++s) qn[s] = *reinterpret_cast<const bf16x8_t*>(qrow + 32 * s + 8 * qd);
    };
    load_q(it);
    // S^T tiles: rows = slots 16 j + 4 qd + r, column = head c, so a lane's scores
    // share a head: its running maximum, and this lane's part of the sum
    const float sl2 = scale * kLog2e;  // probabilities as exp2(s * scale * log2(e) - m)
    int krow[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) krow[j] = mla_slot_token(16 * j + c) * KS + 8 * qd;
    // K fragments in batches of KB steps, read two batches ahead of the products;
    // the first two of a block are read at the end of the period before
    constexpr int KB = 2, NKB = NSQ / KB;
    bf16x8_t kop[3][KB][2];
    auto read_k = [&](int stg, int kb2, bf16x8_t (&dst)[KB][2]) {
      const uint16_t* kst = reinterpret_cast<const uint16_t*>(&Kt[(stg % kMrStages) * kMrStage]);
#pragma unroll
      for (int ss = 0; ss < KB; ++ss)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          dst[ss][j] = *reinterpret_cast<const bf16x8_t*>(&kst[krow[j] + 32 * (kb2 * KB + ss)]);
    };
    hand_over(false, false);
    if (scorer && nv > 0) {
      read_k(0, 0, kop[0]);
      read_k(0, 1, kop[1]);
    }
    for (; it < n_items;) {
      const int next = it + gridDim.x;
      const int nblk = blocks_of(nv), nper = max(nblk, kMrMinPeriods);
      bf16x8_t qb[NSQ];
#pragma unroll
      for (int s = 0; s < NSQ; ++s) {
        qb[s] = qn[s];
        asm volatile("" : "+v"(qb[s]));
      }
      kvn = cache_of(min(next, n_items - 1));
      load_picks(min(next, n_items - 1));
      load_q(min(next, n_items - 1));
      float m_run = -INFINITY, l_run = 0.f;
      for (int p = 0; p < nper; ++p) {
        advance(p, nblk, nper, next);
        const bool score = scorer && p < nblk;
        f32x4_t st[2], st2[2];
        if (score) {
#pragma unroll
          for (int j = 0; j < 2; ++j) st[j] = st2[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kb2 = 0; kb2 < NKB; ++kb2) {
            if (kb2 + 2 < NKB) read_k(stage, kb2 + 2, kop[(kb2 + 2) % 3]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ss = 0; ss < KB; ++ss)
#pragma unroll
              for (int j = 0; j < 2; ++j) {
                const int s = kb2 * KB + ss;
                if (s & 1)
                  st2[j] = mfma_bf16(kop[kb2 % 3][ss][j], qb[s], st2[j]);
                else
                  st[j] = mfma_bf16(kop[kb2 % 3][ss][j], qb[s], st[j]);
              }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        // next period's block (this item's, or the next one's first) has landed
        if (scorer && (p + 1 < nblk || (p + 1 == nper && next < n_items && nv_next > 0))) {
          read_k(stage + (p < nblk ? 1 : 0), 0, kop[0]);
          read_k(stage + (p < nblk ? 1 : 0), 1, kop[1]);
        }
        if (score) {
          float sv[2][4];
          bool over = false;  // the running maximum moves only past the lazy margin (or from -inf)
          const float lim = m_run + kMlaLazyMax * kLog2e;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            st[j] += st2[j];
#pragma unroll
            for (int r = 0; r < 4; ++r) sv[j][r] = st[j][r] * sl2;
          }
          if ((p + 1) * kMlaBT > nv) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                sv[j][r] = p * kMlaBT + mla_slot_token(16 * j + 4 * qd + r) < nv ? sv[j][r] : -INFINITY;
          }
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) over |= sv[j][r] > lim;
          const bool move = __ballot(over) != 0;
          if (move) {  // rare past the first block
            float bm = -INFINITY;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int r = 0; r < 4; ++r) bm = fmaxf(bm, sv[j][r]);
            bm = fmaxf(bm, __shfl_xor(bm, 16));
            bm = fmaxf(bm, __shfl_xor(bm, 32));
            const float m_new = bm > lim ? bm : m_run;
            const float alpha = (bm > lim && m_run != -INFINITY) ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.f;
            l_run *= alpha;
            m_run = m_new;
            if (qd == 0) As[period & 1][16 * wv + c] = alpha;
          }
          if (lane == 0) Fl[period & 1][wv] = move ? 1 : 0;
          uint16_t* ps = Ps[period & 1];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            float pr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              pr[r] = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sv[j][r] - m_run);
              l_run += pr[r];
            }
            const uint2 pw = {__builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{pr[0], pr[1]}, bf16x2_t)),
                              __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{pr[2], pr[3]}, bf16x2_t))};
            *reinterpret_cast<uint2*>(&ps[(16 * wv + c) * kPsStride + 16 * j + 4 * qd]) = pw;
          }
        }
        if (scorer && p == nper - 1) {  // the item's maxima and sums, read by the value waves next period
          float l = l_run;
          l += __shfl_xor(l, 16);
          l += __shfl_xor(l, 32);
          if (qd == 0) {
            Ml[0][16 * wv + c] = m_run;
            Ml[1][16 * wv + c] = l;
          }
        }
        hand_over(false, false);
        stage += p < nblk ? 1 : 0;
        ++period;
      }
      it = next;
      par ^= 1;
      nv = nv_next;
      kvb = kvn;
    }
    return;
  }
  // value waves: O^T tiles, rows = columns 16 (dt0 + dl) + 4 qd + r, column = head 16 ht + c
  const int dt0 = (wv - 4) * DTW;
  f32x4_t o[HT][DTW];
#pragma unroll
  for (int ht = 0; ht < HT; ++ht)
#pragma unroll
    for (int dl = 0; dl < DTW; ++dl) o[ht][dl] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int vi = c >> 2, vj = c & 3;
  // multiply the block scored last period (parity pb), whose V fragments were
  // read during that period, and read those of the block scored in this one
  bf16x8_t vv[DTW];
  auto read_v = [&](int stg, int dd) {
    const uint16_t* vp = reinterpret_cast<const uint16_t*>(&Kt[(stg % kMrStages) * kMrStage]) +
                         (8 * qd + 2 * vi) * KS + 4 * vj + 16 * (dt0 + dd);
    const mla_v4s a = lds_read_tr16(vp), e = lds_read_tr16(vp + KS);
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a, e, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  auto value = [&](int stg, int pb) {
    int fl[HT];
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) fl[ht] = Fl[pb][ht];
    bf16x8_t pa[HT];
#pragma unroll
    for (int ht = 0; ht < HT; ++ht)
      pa[ht] = *reinterpret_cast<const bf16x8_t*>(&Ps[pb][(16 * ht + c) * kPsStride + 8 * qd]);
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      if (__builtin_amdgcn_readfirstlane(fl[ht])) {  // the same word for every lane
        const float al = As[pb][16 * ht + c];
#pragma unroll
        for (int dl = 0; dl < DTW; ++dl) o[ht][dl] *= al;
      }
    }
#pragma unroll
    for (int dd = 0; dd < DTW; ++dd) {
#pragma unroll
      for (int ht = 0; ht < HT; ++ht) o[ht][dd] = mfma_bf16(vv[dd], pa[ht], o[ht][dd]);
      __builtin_amdgcn_sched_barrier(0);
      vv[dd] = read_v(stg, dd);  // (unused if no block is scored in this period)
    }
  };
  // normalize and store an item, and clear the tiles for the next
  auto store = [&](int i) {
    const int64_t b = row_of(i);
#pragma unroll
    for (int ht = 0; ht < HT; ++ht) {
      const int head = 16 * ((i % n_groups) * HT + ht) + c;
      const float m = Ml[0][16 * ht + c];
      const float l =
          Ml[1][16 * ht + c] + ((sink && m != -INFINITY) ? __builtin_amdgcn_exp2f(Sink[head] * kLog2e - m) : 0.f);
      const float inv = m == -INFINITY ? 0.f : 1.0f / l;
      // two column tiles at a time: lane rows 4 qd .. + 3 of both are exchanged
      // (row 1 of the first with row 0 of the second, 3 with 2), so that a lane
      // stores 8 consecutive columns: tile dl + (qd & 1), columns 8 (qd >> 1) ..
      uint16_t* orow = out + (b * H + head) * kMlaDl + 16 * (dt0 + (qd & 1)) + 8 * (qd >> 1);
#pragma unroll
      for (int dl = 0; dl < DTW; dl += 2) {
        uint32_t w[2][2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const f32x4_t v = o[ht][dl + t] * inv;
          o[ht][dl + t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          w[t][0] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{v[0], v[1]}, bf16x2_t));
          w[t][1] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{v[2], v[3]}, bf16x2_t));
        }
        const auto x0 = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
        const auto x1 = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
        *reinterpret_cast<u32x4_t*>(orow + 16 * dl) = u32x4_t{x0[0], x1[0], x0[1], x1[1]};
      }
    }
  };
  hand_over(false, false);
  bool scored = false;  // a block was scored last period
  int prev = -1;        // the item to store
  for (; it < n_items;) {
    const int next = it + gridDim.x;
    const int nblk = blocks_of(nv), nper = max(nblk, kMrMinPeriods);
    kvn = cache_of(min(next, n_items - 1));
    load_picks(min(next, n_items - 1));
    for (int p = 0; p < nper; ++p) {
      advance(p, nblk, nper, next);
      if (scored) {
        value(stage, (period - 1) & 1);
      } else if (p < nblk) {
#pragma unroll
        for (int dd = 0; dd < DTW; ++dd) vv[dd] = read_v(stage, dd);
      }
      copy();
      const bool stored = p == 0 && prev >= 0;
      if (stored) store(prev);
      hand_over(cp_on, stored);
      scored = p < nblk;
      stage += scored ? 1 : 0;
      ++period;
    }
    prev = it;
    it = next;
    par ^= 1;
    nv = nv_next;
    kvb = kvn;
  }
  if (scored) value(stage, (period - 1) & 1);
  store(prev);
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct IndexerWs {
  float* hi;
  uint64_t* keys;
  uint32_t *wg_counts, *hist1;
  size_t zero_words;  // hist1
  uint32_t* qlimbs;   // q's int8 limbs, written by the prep kernel
};

static size_t indexer_ws(int64_t b, int64_t l, char* base, IndexerWs* w) {
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char* p = base ? base + off : nullptr;
    off += align256(bytes);
    return p;
  };
  float* hi = (float*)take((size_t)b * l * 4);
  uint64_t* keys = (uint64_t*)take((size_t)b * l * 8);
  uint32_t* wgc = (uint32_t*)take((size_t)b * kRsMaxWgs * 4);
  const size_t zbytes = (size_t)b * kHistBins * 4;
  uint32_t* z = (uint32_t*)take(zbytes);
  uint32_t* qlimbs = (uint32_t*)take((size_t)b * 64 * 3 * kIdxD);  // q's int8 limbs, up to 64 heads
  if (w) {
    w->hi = hi;
    w->keys = keys;
    w->wg_counts = wgc;
    w->hist1 = z;
    w->zero_words = zbytes / 4;
    w->qlimbs = qlimbs;
  }
  return off;
}

// Bound kernel shape: one 16-token tile per group, a ring of up to 4 groups
// (its registers then leave three waves per SIMD: about 3072 resident waves on
// 256 CUs) spread over the rows, and at least one full ring per wave where the
// rows are short (each workgroup merges its whole histogram once).
constexpr int kBoundU = 1;
static void bound_shape(int64_t b, int64_t l, int& gx, int& depth) {
  const int64_t groups = (l + 16 * kBoundU - 1) / (16 * kBoundU);
  int64_t g = (768 + b - 1) / b;
  g = std::min<int64_t>(g, (groups + 15) / 16);
  gx = (int)std::max<int64_t>(g, 1);
  const int64_t iters = (groups + 4 * gx - 1) / (4 * gx);
  depth = iters >= 4 ? 4 : (iters >= 2 ? 2 : 1);
}

template <int HT, int D>
static void launch_bound_d(const uint8_t* q, const float* qs, const uint8_t* k, const float* ks, const float* w,
                           const int32_t* lengths, float* lo, float* hi, uint32_t* hist1, int64_t b, int64_t l,
                           int gx, int kdiv, int64_t kstride, hipStream_t st) {
  MOSAIC_LAUNCH((dsa_index_bound_kernel<HT, kBoundU, D>), dim3((unsigned)gx, (unsigned)b), dim3(256), 0, st, q,
                     qs, k, ks, w, lengths, lo, hi, hist1, l, kdiv, kstride);
}

template <int HT>
static void launch_bound(const uint8_t* q, const float* qs, const uint8_t* k, const float* ks, const float* w,
                         const int32_t* lengths, float* lo, float* hi, uint32_t* hist1, int64_t b, int64_t l,
                         int kdiv, int64_t kstride, hipStream_t st) {
  int gx, depth;
  bound_shape(b, l, gx, depth);
  if (depth == 4)
    launch_bound_d<HT, 4>(q, qs, k, ks, w, lengths, lo, hi, hist1, b, l, gx, kdiv, kstride, st);
  else if (depth == 2)
    launch_bound_d<HT, 2>(q, qs, k, ks, w, lengths, lo, hi, hist1, b, l, gx, kdiv, kstride, st);
  else
    launch_bound_d<HT, 1>(q, qs, k, ks, w, lengths, lo, hi, hist1, b, l, gx, kdiv, kstride, st);
}

static int check_indexer(const void* q, const void* qs, const void* k, const void* ks, const void* w, int64_t b,
                         int64_t h, int64_t d, int64_t l) {
  MOSAIC_CHECK_ARG(q && qs && k && ks && w, "dsa_indexer: null pointer");
  MOSAIC_CHECK_ARG(d == kIdxD, "dsa_indexer: head dim %lld (128 supported)", (long long)d);
  MOSAIC_CHECK_ARG(h >= 16 && h <= 64 && h % 16 == 0, "dsa_indexer: heads %lld (16, 32, 48 or 64)", (long long)h);
  MOSAIC_CHECK_ARG(b >= 0 && b <= 65535 && l >= 0 && l < (1ll << 31), "dsa_indexer: shape out of range");
  return kOk;
}

static void dispatch_bound(const uint8_t* q, const float* qs, const uint8_t* k, const float* ks, const float* w,
                           const int32_t* lengths, float* lo, float* hi, uint32_t* hist1, int64_t b, int64_t h,
                           int64_t l, int kdiv, int64_t kstride, hipStream_t st) {
  switch (h / 16) {
    case 1: launch_bound<1>(q, qs, k, ks, w, lengths, lo, hi, hist1, b, l, kdiv, kstride, st); break;
    case 2: launch_bound<2>(q, qs, k, ks, w, lengths, lo, hi, hist1, b, l, kdiv, kstride, st); break;
    case 3: launch_bound<3>(q, qs, k, ks, w, lengths, lo, hi, hist1, b, l, kdiv, kstride, st); break;
    default: launch_bound<4>(q, qs, k, ks, w, lengths, lo, hi, hist1, b, l, kdiv, kstride, st); break;
  }
}

// tokens per rescoring workgroup: about one workgroup per CU over the batch
// (its registers leave one wave per SIMD), a multiple of 64, at most the LDS
// candidate list, and few enough workgroups per row for the finish kernel
static int rescore_range(int64_t b, int64_t l) {
  const int64_t target = std::max<int64_t>(1, 256 / std::max<int64_t>(b, 1));
  int64_t r = (l + target - 1) / target;
  r = std::max<int64_t>(r, (l + kRsMaxWgs - 1) / kRsMaxWgs);
  r = (r + 63) / 64 * 64;
  return (int)std::min<int64_t>(std::max<int64_t>(r, 64), kRsMaxRange);
}

static void launch_rescore(const uint8_t* q, const float* qs, const uint8_t* k, const float* ks, const float* w,
                           const int32_t* lengths, const float* hi, const uint32_t* hist1, const uint32_t* qlimbs,
                           uint64_t* keys, uint32_t* wg_counts, float* scores, int64_t b, int64_t h, int64_t l,
                           int topk, int kdiv, int64_t kstride, hipStream_t st) {
  const int range = rescore_range(b, l);
  const dim3 grid((unsigned)((l + range - 1) / range), (unsigned)b);
#define MOSAIC_RESCORE(HT)                                                                                          \
  if (!qlimbs)                                                                                                      \
    MOSAIC_LAUNCH((dsa_rescore_kernel<HT, false, false>), grid, dim3(256), 0, st, q, qs, k, ks, w, lengths,   \
                       hi, hist1, qlimbs, keys, wg_counts, scores, l, topk, range, kdiv, kstride);                           \
  else if (range <= kRsPfRange)                                                                                     \
    MOSAIC_LAUNCH((dsa_rescore_kernel<HT, true, true>), grid, dim3(256), 0, st, q, qs, k, ks, w, lengths, hi, \
                       hist1, qlimbs, keys, wg_counts, scores, l, topk, range, kdiv, kstride);                             \
  else                                                                                                              \
    MOSAIC_LAUNCH((dsa_rescore_kernel<HT, false, true>), grid, dim3(256), 0, st, q, qs, k, ks, w, lengths,    \
                       hi, hist1, qlimbs, keys, wg_counts, scores, l, topk, range, kdiv, kstride);
  switch (h / 16) {
    case 1: MOSAIC_RESCORE(1) break;
    case 2: MOSAIC_RESCORE(2) break;
    case 3: MOSAIC_RESCORE(3) break;
    default: MOSAIC_RESCORE(4) break;
  }
#undef MOSAIC_RESCORE
}

// Where the row kernel runs: on the shortest caches (us, certified path against
// row kernel, 64 heads, 64 entries: 1 row 18.2 / 12.4, 4096 rows of a cache each
// 211 / 185, 16384 rows 917 / 746), and where many rows share a short one.  It
// takes about 0.13 us an entry for each round of 256 workgroups, whatever topk;
// the certified path's time goes with the rows and grows with topk.  The line is
// where the row kernel is ahead both with every row at full length and with a
// prompt's triangular lengths, which the host does not see: entries times rounds
// up to 13/16 of the rows from 512 picks (all of them where it runs several
// rounds), 5/8 from 256, 1/2 below (512 picks, full / triangular: 1280 rows over 1024
// entries 185 -> 135 and 160 -> 133, 512 over 448 62 -> 64 triangular, 1100 over 1100
// 185 -> 161 but 152 -> 160, 4096 over 2048 639 -> 534 and 546 -> 303, 2560 over 2048
// 387 -> 528; 64 picks: 1024 over 512 89 -> 70 and 86 -> 69, 1024 over 1024 98 -> 134;
// 1 pick: 2048 over 1024 154 -> 136 and 142 -> 135, 4096 over 2048 387 -> 530).
static bool dsa_rows_kernel(int64_t b, int64_t kdiv, int64_t l, int64_t topk) {
  if (l <= 0 || l > kDrMaxL) return false;
  if (l <= 64) return true;
  if (kdiv < kDrRows || b < (l <= 128 ? 256 : 512)) return false;
  const int64_t rounds = (b / kdiv * ((kdiv + kDrRows - 1) / kDrRows) + 255) / 256;
  const int64_t sixteenths = topk >= 512 ? (rounds > 1 ? 16 : 13) : topk >= 256 ? 10 : 8;
  return 16 * l * rounds <= sixteenths * b;
}

struct MlaWs {
  uint16_t* part_o;
  float* part_ml;
};

// splits per row: about 256 workgroups over the batch (two head groups per
// row), at most one per block and at most 32
static int mla_splits(int64_t b, int64_t topk) {
  const int64_t blocks = (topk + kMlaBT - 1) / kMlaBT;
  int64_t s = (128 + b - 1) / b;
  s = std::min<int64_t>(s, blocks);
  s = std::min<int64_t>(s, 32);
  // a split's ids must fit the LDS id buffer
  s = std::max<int64_t>(s, (blocks + kMlaMaxChunk / kMlaBT - 1) / (kMlaMaxChunk / kMlaBT));
  static_assert(32 <= kMlaMaxSplits, "the combine kernel weighs at most kMlaMaxSplits splits");
  return (int)std::max<int64_t>(s, 1);
}
// head tiles per workgroup: as many as divide the heads (at most 4), fewer
// while the grid has fewer workgroups than CUs (B = 1, 128 heads: 32 splits x
// 8 groups of 16 heads, 18.3 against 19.6 us for 4 groups of 32 heads)
static int mla_head_tiles(int64_t b, int64_t h, int S) {
  int ht = 4;
  while (ht > 1 && (h / 16) % ht != 0) --ht;
  while (ht > 1 && (h / 16) % (ht / 2) == 0 && (int64_t)S * b * (h / (16 * ht)) < 256) ht /= 2;
  return ht;
}
// Splits of the whole-split kernel (kMdTokens selected tokens each), 0 where the
// block kernel runs: it takes groups of 64 heads, and from 24 to 1024 workgroups
// (us, block kernel against whole splits, 128 heads unless said: 8 rows of 2048
// picks 34.1 / 23.6, 3 rows 31.5 / 18.8, 12 rows 60.9 / 35.6, 3 rows of 512 22.3 /
// 16.1; below, the block kernel spreads 16-head groups wider: 2 rows of 512 14.7 /
// 15.4, 64 heads x 4 rows of 512 14.6 / 15.4; above, its fewer partials win: 32
// rows of 4096 128 / 139).
//
// fp32 partials past 320 workgroups (42 MB) cost more than the shorter chain gives
// where the block kernel's grid is one whole round: 32 rows of 128 heads, 896 picks
// 45.5 / 47.5, 1000 48.6 / 52.3, but 640 picks 39.2 / 38.9; 24 rows, whose blocks
// need a second round, 1000 picks 67.3 / 42.5.
static int mla_chunks(int64_t b, int64_t h, int64_t topk) {
  const int64_t chunks = (topk + kMdTokens - 1) / kMdTokens;
  const int64_t wgs = b * (h / 64) * chunks;
  if (chunks <= kMdF32Chunks && wgs > 320 && (int64_t)mla_splits(b, topk) * wgs <= 256 * chunks) return 0;
  return h % 64 == 0 && chunks <= 32 && b <= 32 && wgs >= 24 && wgs <= 1024 ? (int)chunks : 0;
}
// `chunks`: splits of the whole-split kernel, 0 for the block kernel.  Queries
// ask for the larger of both; a call with room for the block kernel's partials
// only (a workspace sized for the bf16 cache, or for another batch) runs that.
static size_t mla_ws(int64_t b, int64_t h, int64_t topk, int64_t chunks, char* base, MlaWs* w) {
  const int64_t S = std::max<int64_t>(mla_splits(b, topk), chunks <= kMdF32Chunks ? 2 * chunks : chunks);
  const size_t ob = align256((size_t)b * S * h * kMlaDl * 2);
  const size_t mb = align256((size_t)b * S * h * 2 * 4);
  if (w) {
    w->part_o = (uint16_t*)base;
    w->part_ml = (float*)(base + ob);
  }
  return ob + mb;
}

}  // namespace mosaic

using namespace mosaic;

extern "C" size_t mosaic_dsa_indexer_workspace_bytes(int64_t b, int64_t l) {
  if (b < 0 || l < 0) return 0;
  return indexer_ws(b, l, nullptr, nullptr);
}

namespace mosaic {
static int indexer_topk_impl(const uint8_t* q, const float* q_s, const uint8_t* k, const float* k_s, const float* w,
                             const int32_t* lengths, int32_t* idx_out, int64_t b, int64_t h, int64_t d, int64_t l,
                             int64_t topk, int32_t offset, int64_t kdiv, int64_t kstride, void* workspace,
                             size_t workspace_bytes, void* stream) {
  int rc = check_indexer(q, q_s, k, k_s, w, b, h, d, l);
  if (rc) return rc;
  MOSAIC_CHECK_ARG(idx_out, "dsa_indexer_topk: null output");
  MOSAIC_CHECK_ARG(topk >= 1 && topk <= kMaxTopk, "dsa_indexer_topk: topk %lld (1..%d)", (long long)topk, kMaxTopk);
  MOSAIC_CHECK_ARG(l <= (int64_t)kRsMaxWgs * kRsMaxRange, "dsa_indexer_topk: l %lld (at most %lld)", (long long)l,
                   (long long)kRsMaxWgs * kRsMaxRange);
  MOSAIC_CHECK_ARG(kdiv >= 1 && b % kdiv == 0, "dsa_indexer_topk: %lld query rows do not split into groups of %lld",
                   (long long)b, (long long)kdiv);
  MOSAIC_CHECK_ARG(kstride >= l && kstride < (1ll << 40), "dsa_indexer_topk: cache length %lld < l %lld",
                   (long long)kstride, (long long)l);
  const size_t need = indexer_ws(b, l, nullptr, nullptr);
  MOSAIC_CHECK_ARG(workspace && workspace_bytes >= need, "dsa_indexer_topk: workspace %zu bytes < %zu",
                   workspace_bytes, need);
  if (b == 0) return kOk;
  hipStream_t st = (hipStream_t)stream;
  if (dsa_rows_kernel(b, kdiv, l, topk)) {
    const int groups = (int)(b / kdiv);
    const dim3 grid((unsigned)(groups * ((kdiv + kDrRows - 1) / kDrRows)));
#define MOSAIC_ROWS_TOPK(HT)                                                                                        \
  MOSAIC_LAUNCH((dsa_rows_topk_kernel<HT>), grid, dim3(64 * kDrRows), 0, st, q, q_s, k, k_s, w, lengths, idx_out, l, \
                groups, (int)kdiv, kstride, (int)topk, (int)offset)
    switch (h / 16) {
      case 1: MOSAIC_ROWS_TOPK(1); break;
      case 2: MOSAIC_ROWS_TOPK(2); break;
      case 3: MOSAIC_ROWS_TOPK(3); break;
      default: MOSAIC_ROWS_TOPK(4); break;
    }
#undef MOSAIC_ROWS_TOPK
    MOSAIC_RETURN_LAUNCH("dsa_indexer_topk_rows");
  }
  IndexerWs ws;
  indexer_ws(b, l, (char*)workspace, &ws);
  const int64_t qwords = b * h * (kIdxD / 4);
  const int64_t prep_n = std::max<int64_t>((int64_t)ws.zero_words, qwords);
  MOSAIC_LAUNCH(dsa_prep_kernel, dim3((unsigned)((prep_n + 255) / 256)), dim3(256), 0, st, ws.hist1,
                     (int64_t)ws.zero_words, reinterpret_cast<const uint32_t*>(q), ws.qlimbs, qwords, (int)h);
  if (l > 0) {
    dispatch_bound(q, q_s, k, k_s, w, lengths, nullptr, ws.hi, ws.hist1, b, h, l, (int)kdiv, kstride, st);
    launch_rescore(q, q_s, k, k_s, w, lengths, ws.hi, ws.hist1, ws.qlimbs, ws.keys, ws.wg_counts, nullptr, b, h, l,
                   (int)topk, (int)kdiv, kstride, st);
  }
  MOSAIC_LAUNCH(dsa_finish_kernel, dim3((unsigned)b), dim3(1024), 0, st, ws.keys, ws.wg_counts, lengths, l,
                     rescore_range(b, l), (int)topk, (int)offset, idx_out);
  MOSAIC_RETURN_LAUNCH("dsa_indexer_topk");
}
}  // namespace mosaic

extern "C" int mosaic_dsa_indexer_topk(const uint8_t* q, const float* q_s, const uint8_t* k, const float* k_s,
                                       const float* w, const int32_t* lengths, int32_t* idx_out, int64_t b, int64_t h,
                                       int64_t d, int64_t l, int64_t topk, int32_t offset, void* workspace,
                                       size_t workspace_bytes, void* stream) {
  return indexer_topk_impl(q, q_s, k, k_s, w, lengths, idx_out, b, h, d, l, topk, offset, 1, l, workspace,
                           workspace_bytes, stream);
}

extern "C" int mosaic_dsa_indexer_topk_shared(const uint8_t* q, const float* q_s, const uint8_t* k, const float* k_s,
                                              const float* w, const int32_t* lengths, int32_t* idx_out, int64_t rows,
                                              int64_t h, int64_t d, int64_t l, int64_t cache_len, int64_t rows_per_k,
                                              int64_t topk, int32_t offset, void* workspace, size_t workspace_bytes,
                                              void* stream) {
  return indexer_topk_impl(q, q_s, k, k_s, w, lengths, idx_out, rows, h, d, l, topk, offset, rows_per_k, cache_len,
                           workspace, workspace_bytes, stream);
}

extern "C" int mosaic_dsa_indexer_scores(const uint8_t* q, const float* q_s, const uint8_t* k, const float* k_s,
                                         const float* w, float* scores, int64_t b, int64_t h, int64_t d, int64_t l,
                                         void* stream) {
  int rc = check_indexer(q, q_s, k, k_s, w, b, h, d, l);
  if (rc) return rc;
  MOSAIC_CHECK_ARG(scores, "dsa_indexer_scores: null output");
  if (b == 0 || l == 0) return kOk;
  launch_rescore(q, q_s, k, k_s, w, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, scores, b, h, l, 0, 1, l,
                 (hipStream_t)stream);
  MOSAIC_RETURN_LAUNCH("dsa_indexer_scores");
}

extern "C" int mosaic_dsa_indexer_bounds(const uint8_t* q, const float* q_s, const uint8_t* k, const float* k_s,
                                         const float* w, float* lo, float* hi, int64_t b, int64_t h, int64_t d,
                                         int64_t l, void* stream) {
  int rc = check_indexer(q, q_s, k, k_s, w, b, h, d, l);
  if (rc) return rc;
  MOSAIC_CHECK_ARG(lo && hi, "dsa_indexer_bounds: null output");
  if (b == 0 || l == 0) return kOk;
  dispatch_bound(q, q_s, k, k_s, w, nullptr, lo, hi, nullptr, b, h, l, 1, l, (hipStream_t)stream);
  MOSAIC_RETURN_LAUNCH("dsa_indexer_bounds");
}

extern "C" size_t mosaic_mla_decode_workspace_bytes(int64_t b, int64_t h, int64_t topk) {
  if (b < 0 || h < 0 || topk < 0) return 0;
  return mla_ws(b, h, topk, mla_chunks(b, h, topk), nullptr, nullptr);
}

namespace mosaic {

template <bool FP8, int DR>
static int launch_mla(const uint16_t* q, const MlaKv& kv, const float* sink, const int32_t* idx, uint16_t* out,
                      int64_t rows, int64_t h, int64_t topk, float softmax_scale, void* workspace, size_t workspace_bytes,
                      hipStream_t st) {
  MlaWs ws;
  int S = mla_splits(rows, topk);
  // (q goes straight into LDS there, 16 bytes a lane: other alignments keep the block kernel's register loads)
  int chunks = FP8 && kv.n > 0 && (uintptr_t)q % 16 == 0 ? mla_chunks(rows, h, topk) : 0;
  if (mla_ws(rows, h, topk, chunks, nullptr, nullptr) > workspace_bytes) chunks = 0;
  mla_ws(rows, h, topk, chunks, (char*)workspace, &ws);
  const bool f32 = chunks > 0 && chunks <= kMdF32Chunks;
  if (chunks > 0) {
    S = chunks;
    const dim3 grid((unsigned)S, (unsigned)rows, (unsigned)(h / 64));
    if (f32)
      MOSAIC_LAUNCH(mla_decode_chunk_kernel<float>, grid, dim3(512), 0, st, q, kv, idx,
                    reinterpret_cast<float*>(ws.part_o), ws.part_ml, (int)topk, softmax_scale);
    else
      MOSAIC_LAUNCH(mla_decode_chunk_kernel<uint16_t>, grid, dim3(512), 0, st, q, kv, idx, ws.part_o, ws.part_ml,
                    (int)topk, softmax_scale);
    MOSAIC_LAUNCH_CHECK("mla_decode_chunk");
  } else {
    const int blocks = (int)((topk + kMlaBT - 1) / kMlaBT);
    const int chunk = ((blocks + S - 1) / S) * kMlaBT;
    const int ht = mla_head_tiles(rows, h, S);
    dim3 grid((unsigned)S, (unsigned)rows, (unsigned)(h / (16 * ht)));
    switch (ht) {
#define MLA_CASE(HTV)                                                                                                  \
  case HTV:                                                                                                            \
    MOSAIC_LAUNCH((mla_decode_split_kernel<HTV, FP8, DR>), grid, dim3(256), 0, st, q, kv, idx, ws.part_o,       \
                       ws.part_ml, (int)topk, softmax_scale, chunk);                                                   \
    break;
      MLA_CASE(1) MLA_CASE(2) MLA_CASE(3) MLA_CASE(4)
#undef MLA_CASE
    }
    MOSAIC_LAUNCH_CHECK("mla_decode_split");
  }
  auto combine = [&](auto* part) {
    using TP = std::remove_pointer_t<decltype(part)>;
    if (rows * (h / 16) * (kMlaDt / kMlaCombineTiles) >= 256)
      MOSAIC_LAUNCH(mla_combine_tiles_kernel<TP>,
                    dim3((unsigned)(kMlaDt / kMlaCombineTiles), (unsigned)(h / 16), (unsigned)rows), dim3(256), 0, st,
                    part, ws.part_ml, sink, out, (int)h, S);
    else
      MOSAIC_LAUNCH(mla_combine_kernel<TP>, dim3((unsigned)kMlaDt, (unsigned)(h / 16), (unsigned)rows), dim3(256), 0,
                    st, part, ws.part_ml, sink, out, (int)h, S);
  };
  if (f32)
    combine(reinterpret_cast<float*>(ws.part_o));
  else
    combine(ws.part_o);
  MOSAIC_RETURN_LAUNCH("mla_sparse_decode");
}

static int check_mla_common(int64_t rows, int64_t h, int64_t n, int64_t topk, int64_t rows_per_kv, void* workspace,
                            size_t workspace_bytes) {
  MOSAIC_CHECK_ARG(h >= 16 && h <= 256 && h % 16 == 0 && (h <= 64 || h % 64 == 0),
                   "mla_sparse_decode: heads %lld (16, 32, 48, 64 or a multiple of 64 up to 256)", (long long)h);
  MOSAIC_CHECK_ARG(rows >= 0 && rows <= 65535 && n >= 0 && n < (1ll << 31) && topk >= 0 &&
                       topk <= (int64_t)kMlaMaxSplits * kMlaMaxChunk,
                   "mla_sparse_decode: shape out of range (topk at most %d)", kMlaMaxSplits * kMlaMaxChunk);
  MOSAIC_CHECK_ARG(rows_per_kv >= 1 && rows % rows_per_kv == 0, "mla_sparse_decode: rows %lld, rows_per_kv %lld",
                   (long long)rows, (long long)rows_per_kv);
  const size_t need = mla_ws(rows, h, topk, 0, nullptr, nullptr);
  MOSAIC_CHECK_ARG(workspace && workspace_bytes >= need, "mla_sparse_decode: workspace %zu bytes < %zu",
                   workspace_bytes, need);
  return kOk;
}

}  // namespace mosaic

extern "C" int mosaic_mla_sparse_decode(const uint16_t* q, const uint8_t* kv_latent, const float* kv_scale,
                                        const uint16_t* kv_rope, const float* sink, const int32_t* idx, uint16_t* out,
                                        int64_t b, int64_t h, int64_t n, int64_t topk, int64_t d_latent,
                                        int64_t d_rope, int64_t scale_block, float softmax_scale, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  MOSAIC_CHECK_ARG(q && kv_latent && kv_scale && kv_rope && idx && out, "mla_sparse_decode: null pointer");
  MOSAIC_CHECK_ARG(d_latent == kMlaDl && d_rope == 64, "mla_sparse_decode: dims %lld+%lld (512+64 supported)",
                   (long long)d_latent, (long long)d_rope);
  int sb_shift = -1;
  for (int s = 4; s <= 9; ++s)
    if (scale_block == (1ll << s)) sb_shift = s;
  MOSAIC_CHECK_ARG(sb_shift >= 0, "mla_sparse_decode: scale_block %lld (16..512, power of two)",
                   (long long)scale_block);
  int rc = check_mla_common(b, h, n, topk, 1, workspace, workspace_bytes);
  if (rc) return rc;
  if (b == 0) return kOk;
  const MlaKv kv{kv_latent, kv_scale, kv_rope, n, 1, sb_shift};
  return launch_mla<true, 64>(q, kv, sink, idx, out, b, h, topk, softmax_scale, workspace, workspace_bytes,
                              (hipStream_t)stream);
}

extern "C" int mosaic_mla_sparse_decode_bf16(const uint16_t* q, const uint16_t* kv, const float* sink,
                                             const int32_t* idx, uint16_t* out, int64_t rows, int64_t h, int64_t n,
                                             int64_t topk, int64_t d, int64_t rows_per_kv, float softmax_scale,
                                             void* workspace, size_t workspace_bytes, void* stream) {
  MOSAIC_CHECK_ARG(q && kv && idx && out, "mla_sparse_decode_bf16: null pointer");
  MOSAIC_CHECK_ARG(d == 512 || d == 576, "mla_sparse_decode_bf16: head dim %lld (512 or 576)", (long long)d);
  int rc = check_mla_common(rows, h, n, topk, rows_per_kv, workspace, workspace_bytes);
  if (rc) return rc;
  if (rows == 0) return kOk;
  // From 64 rows the row kernel: splitting a row over workgroups no longer pays
  // for its partials and combine (64 heads, us, split path against rows: 32 rows
  // of 640 picks 27.1 / 32.3, 64 rows 40.1 / 33.6, 64 rows of 2048 picks 86.1 /
  // 82.5, 128 rows 112.7 / 83.7; 16 heads, 64 rows of 640 30.6 / 24.6).  It copies
  // the cache's rows straight into LDS, 16 bytes a lane, and stores 16 bytes: rows
  // that are not aligned for that keep the split kernel's register loads.
  const bool aligned = ((uintptr_t)q | (uintptr_t)kv | (uintptr_t)out) % 16 == 0;
  if (d == 512 && topk <= kMrMaxPicks && rows >= kMrMinRows && aligned) {
    int ht = 4;
    while (ht > 1 && (h / 16) % ht != 0) --ht;
    const int groups = (int)(h / (16 * ht));
    const dim3 grid((unsigned)std::min<int64_t>(rows * groups, 256));
    hipStream_t st = (hipStream_t)stream;
    switch (ht) {
#define MLA_CASE(HTV)                                                                                                  \
  case HTV:                                                                                                            \
    MOSAIC_LAUNCH((mla_rows_kernel<HTV>), grid, dim3(512), 0, st, q, kv, idx, sink, out, n, (int)rows,                 \
                  (int)rows_per_kv, groups, (int)topk, softmax_scale);                                                 \
    break;
      MLA_CASE(1) MLA_CASE(2) MLA_CASE(3) MLA_CASE(4)
#undef MLA_CASE
    }
    MOSAIC_RETURN_LAUNCH("mla_rows");
  }
  const MlaKv kvd{kv, nullptr, nullptr, n, (int)rows_per_kv, 0};
  if (d == 576)
    return launch_mla<false, 64>(q, kvd, sink, idx, out, rows, h, topk, softmax_scale, workspace, workspace_bytes,
                                 (hipStream_t)stream);
  return launch_mla<false, 0>(q, kvd, sink, idx, out, rows, h, topk, softmax_scale, workspace, workspace_bytes,
                              (hipStream_t)stream);
}
