// mq_quant.hip — f32 [n, k] on the device -> GGUF blocks (candle
// QTensor::quantize / quantize_onto, called by mold at
// crates/mold-inference/src/flux/pipeline.rs:219-229 (FP8 -> Q8_0 cache) and
// crates/mold-inference/src/flux/lora.rs:849 (LoRA re-quantize)).
//
// The block contents follow ggml's reference quantizers (quantize_row_*_ref,
// make_qx_quants, make_q3_quants, make_qkx2_quants; ggml, MIT License,
// Copyright (c) 2023-2024 The ggml authors).  To produce byte-identical
// blocks the arithmetic is performed in the same order with IEEE
// single-precision operations: FMA contraction is disabled in this file,
// divisions and square roots are the correctly rounded ones, and
// nearest_int() uses the same 1.5*2^23 magic add.  Byte identity is held
// against that ggml restatement only.  Whether candle's k_quants port makes
// the same bytes is unpinned: its source is not available here, and its
// Q2_K/Q4_K/Q5_K from_float may use make_qkx1_quants instead of
// make_qkx2_quants.  Q4_0/Q4_1/Q5_0/Q5_1/Q8_0 have a single formula.
// A thread quantizes one 32-element block, or one sub-block of a super-block,
// and stores its fields straight into the tiled device layout.
#include <utility>

#include "mq_kernels.h"

#pragma clang fp contract(off)

namespace mq {
namespace {

constexpr float kGroupMaxEps = 1e-15f;

__device__ __forceinline__ int nearest_int(float f) {
  const float v = f + 12582912.f;
  int i;
  __builtin_memcpy(&i, &v, 4);
  return (i & 0x007fffff) - 0x00400000;
}

// f32 -> f16, round to nearest even.  The empty asm pins `f` in a register:
// without it the backend folds a preceding multiply into the conversion as
// v_fma_mix(a, b, +0), which turns a -0 product (e.g. 0 * -1/8 for an all-zero
// Q4_0 block) into +0 and changes the stored scale bits.
__device__ __forceinline__ uint16_t f2h(float f) {
  asm volatile("" : "+v"(f));
  _Float16 h = (_Float16)f;
  uint16_t u;
  __builtin_memcpy(&u, &h, 2);
  return u;
}

__device__ __forceinline__ void put16(uint8_t *p, uint16_t v) {
  p[0] = (uint8_t)(v & 0xFF);
  p[1] = (uint8_t)(v >> 8);
}

template <typename T>
__device__ __forceinline__ T mn(T a, T b) { return a < b ? a : b; }
template <typename T>
__device__ __forceinline__ T mx(T a, T b) { return a > b ? a : b; }

// ------------------------------------------------------------ 32-element types

__device__ void q_q4_0(const float *x, uint8_t *o) {
  float amax = 0.f, vmax = 0.f;
  for (int j = 0; j < 32; ++j)
    if (amax < fabsf(x[j])) { amax = fabsf(x[j]); vmax = x[j]; }
  const float d = vmax / -8;
  const float id = d ? 1.0f / d : 0.0f;
  put16(o, f2h(d));
  for (int j = 0; j < 16; ++j) {
    const float x0 = x[j] * id, x1 = x[16 + j] * id;
    const uint8_t a = (uint8_t)mn<int>(15, (int8_t)(x0 + 8.5f));
    const uint8_t b = (uint8_t)mn<int>(15, (int8_t)(x1 + 8.5f));
    o[2 + j] = (uint8_t)(a | (b << 4));
  }
}

__device__ void q_q4_1(const float *x, uint8_t *o) {
  float vmin = 3.402823466e+38f, vmax = -3.402823466e+38f;
  for (int j = 0; j < 32; ++j) {
    if (x[j] < vmin) vmin = x[j];
    if (x[j] > vmax) vmax = x[j];
  }
  const float d = (vmax - vmin) / 15;
  const float id = d ? 1.0f / d : 0.0f;
  put16(o, f2h(d));
  put16(o + 2, f2h(vmin));
  for (int j = 0; j < 16; ++j) {
    const float x0 = (x[j] - vmin) * id, x1 = (x[16 + j] - vmin) * id;
    const uint8_t a = (uint8_t)mn<int>(15, (int8_t)(x0 + 0.5f));
    const uint8_t b = (uint8_t)mn<int>(15, (int8_t)(x1 + 0.5f));
    o[4 + j] = (uint8_t)(a | (b << 4));
  }
}

__device__ void q_q5_0(const float *x, uint8_t *o) {
  float amax = 0.f, vmax = 0.f;
  for (int j = 0; j < 32; ++j)
    if (amax < fabsf(x[j])) { amax = fabsf(x[j]); vmax = x[j]; }
  const float d = vmax / -16;
  const float id = d ? 1.0f / d : 0.0f;
  put16(o, f2h(d));
  uint32_t qh = 0;
  for (int j = 0; j < 16; ++j) {
    const float x0 = x[j] * id, x1 = x[16 + j] * id;
    const uint8_t a = (uint8_t)mn<int>(31, (int8_t)(x0 + 16.5f));
    const uint8_t b = (uint8_t)mn<int>(31, (int8_t)(x1 + 16.5f));
    o[6 + j] = (uint8_t)((a & 0xF) | ((b & 0xF) << 4));
    qh |= ((uint32_t)(a & 0x10) >> 4) << j;
    qh |= ((uint32_t)(b & 0x10) >> 4) << (j + 16);
  }
  for (int i = 0; i < 4; ++i) o[2 + i] = (uint8_t)(qh >> (8 * i));
}

__device__ void q_q5_1(const float *x, uint8_t *o) {
  float vmin = x[0], vmax = x[0];
  for (int j = 1; j < 32; ++j) {
    if (x[j] < vmin) vmin = x[j];
    if (x[j] > vmax) vmax = x[j];
  }
  const float d = (vmax - vmin) / 31;
  const float id = d ? 1.0f / d : 0.0f;
  put16(o, f2h(d));
  put16(o + 2, f2h(vmin));
  uint32_t qh = 0;
  for (int j = 0; j < 16; ++j) {
    const float x0 = (x[j] - vmin) * id, x1 = (x[16 + j] - vmin) * id;
    const uint8_t a = (uint8_t)(x0 + 0.5f);
    const uint8_t b = (uint8_t)(x1 + 0.5f);
    o[8 + j] = (uint8_t)((a & 0xF) | ((b & 0xF) << 4));
    qh |= ((uint32_t)(a & 0x10) >> 4) << j;
    qh |= ((uint32_t)(b & 0x10) >> 4) << (j + 16);
  }
  for (int i = 0; i < 4; ++i) o[4 + i] = (uint8_t)(qh >> (8 * i));
}

__device__ void q_q8_0(const float *x, uint8_t *o) {
  float amax = 0.f;
  for (int j = 0; j < 32; ++j) amax = mx(amax, fabsf(x[j]));
  const float d = amax / 127;
  const float id = d ? 1.0f / d : 0.0f;
  put16(o, f2h(d));
  for (int j = 0; j < 32; ++j) o[2 + j] = (uint8_t)(int8_t)roundf(x[j] * id);
}

// ------------------------------------------------------------- k-quant searches
// One thread searches one sub-block (N = 32 or 16 values, all in registers);
// the 8 or 16 threads of a super-block are neighbouring lanes.

// nearest_int clamped to [0, nmax] as a float.  Exact: ggml's integer steps.
// Otherwise for |f| < 2^22, where the magic sum's ulp is 1 and nearest_int
// rounds to the nearest even integer: two operations for the integer form's
// six.  (A -0 in place of 0 changes no sum: they start at +0, and a product's
// sign of zero is lost in the square or magnitude it ends in.)
template <bool EXACT>
__device__ __forceinline__ float nearest_clamped(float f, int nmax) {
  if constexpr (EXACT) {
    return (float)mx(0, mn(nmax, nearest_int(f)));
  } else {
    return __builtin_amdgcn_fmed3f(__builtin_rintf(f), 0.f, (float)nmax);
  }
}

// Scale and min search over a group of N values (ggml make_qkx2_quants); the
// quants of the best step are nearest_clamped(best_iscale * (x - best_min)).
// VALU-bound: 16 operations per value and step (one rounded multiply and add
// at a time, in ggml's order).
struct Qkx2 {
  float scale, the_min, best_iscale, best_min;
};
template <int N, bool MAD>
__device__ __forceinline__ Qkx2 qkx2(int nmax, const float (&x)[N], const float (&w)[N], float rmin, float rdelta, int nstep) {
  float vmin = x[0], vmax = x[0];
  float sum_w = w[0];
  float sum_x = sum_w * x[0];
#pragma unroll
  for (int i = 1; i < N; ++i) {
    if (x[i] < vmin) vmin = x[i];
    if (x[i] > vmax) vmax = x[i];
    sum_w += w[i];
    sum_x += w[i] * x[i];
  }
  const float xmin = vmin;
  if (vmin > 0) vmin = 0;
  Qkx2 r{0.f, -vmin, 0.f, 0.f};
  if (vmax == vmin) return r;
  float iscale = nmax / (vmax - vmin);
  float scale = 1 / iscale;
  float best = 0;
  r.best_iscale = iscale;
  r.best_min = vmin;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float diff = scale * nearest_clamped<true>(iscale * (x[i] - vmin), nmax) + vmin - x[i];
    diff = MAD ? fabsf(diff) : diff * diff;
    best += w[i] * diff;
  }
  auto step = [&]<bool EXACT>() {
    float q[N];
    float sum_l = 0, sum_l2 = 0, sum_xl = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      q[i] = nearest_clamped<EXACT>(iscale * (x[i] - vmin), nmax);
      const float wl = w[i] * q[i];
      sum_l += wl;
      sum_l2 += wl * q[i];
      sum_xl += wl * x[i];
    }
    const float D = sum_w * sum_l2 - sum_l * sum_l;
    if (D > 0) {
      float this_scale = (sum_w * sum_xl - sum_x * sum_l) / D;
      float this_min = (sum_l2 * sum_x - sum_l * sum_xl) / D;
      if (this_min > 0) {
        this_min = 0;
        this_scale = sum_xl / sum_l2;
      }
      float mad = 0;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        float diff = this_scale * q[i] + this_min - x[i];
        diff = MAD ? fabsf(diff) : diff * diff;
        mad += w[i] * diff;
      }
      if (mad < best) {
        r.best_iscale = iscale;
        r.best_min = vmin;
        best = mad;
        scale = this_scale;
        vmin = this_min;
      }
    }
  };
  for (int is = 0; is <= nstep; ++is) {
    iscale = (rmin + rdelta * is + nmax) / (vmax - vmin);
    // iscale * (x - vmin) is monotone in x, so its ends bound it (NaN takes the exact form)
    const bool tame = fabsf(iscale * (vmax - vmin)) < 4194304.f && fabsf(iscale * (xmin - vmin)) < 4194304.f;
    if (__all(tame)) step.template operator()<false>();
    else step.template operator()<true>();
  }
  r.the_min = -vmin;
  r.scale = scale;
  return r;
}

// Symmetric scale search with weights x^2 (ggml make_qx_quants, rmse_type 1);
// the best step's quants are nmax + clamp(nearest_int(best_iscale * x)), or
// all 0 for a group of zeros (zero set).
template <int N>
__device__ __forceinline__ float qx_rmse1(int nmax, const float (&x)[N], float &best_iscale, bool &zero) {
  float vmax = 0, amax = 0;
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (fabsf(x[i]) > amax) { amax = fabsf(x[i]); vmax = x[i]; }
  zero = amax < kGroupMaxEps;
  best_iscale = 0.f;
  if (zero) return 0.f;
  float sumlx = 0, suml2 = 0;
  auto sums = [&](float iscale) {
    sumlx = suml2 = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      int l = nearest_int(iscale * x[i]);
      l = mx(-nmax, mn(nmax - 1, l));
      const float wl = x[i] * x[i];
      sumlx += wl * x[i] * l;
      suml2 += wl * l * l;
    }
  };
  best_iscale = -nmax / vmax;
  sums(best_iscale);
  float scale = suml2 ? sumlx / suml2 : 0.0f;
  float best = scale * sumlx;
  for (int is = -9; is <= 9; ++is) {
    if (is == 0) continue;
    const float iscale = -(nmax + 0.1f * is) / vmax;
    sums(iscale);
    if (suml2 > 0 && sumlx * sumlx > best * suml2) {
      best_iscale = iscale;
      scale = sumlx / suml2;
      best = scale * sumlx;
    }
  }
  return scale;
}

// Q3_K group search (ggml make_q3_quants with do_rmse).
template <int N>
__device__ __forceinline__ float q3_group(int nmax, const float (&x)[N], int (&L)[N]) {
  float vmax = 0, amax = 0;
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (fabsf(x[i]) > amax) { amax = fabsf(x[i]); vmax = x[i]; }
  if (amax < kGroupMaxEps) {
#pragma unroll
    for (int i = 0; i < N; ++i) L[i] = 0;
    return 0.f;
  }
  const float iscale = -nmax / vmax;
  float sumlx = 0, suml2 = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    int l = nearest_int(iscale * x[i]);
    l = mx(-nmax, mn(nmax - 1, l));
    L[i] = l;
    const float w = x[i] * x[i];
    sumlx += w * x[i] * l;
    suml2 += w * l * l;
  }
  for (int itry = 0; itry < 5; ++itry) {
    int changed = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float w = x[i] * x[i];
      float slx = sumlx - w * x[i] * L[i];
      if (slx > 0) {
        float sl2 = suml2 - w * L[i] * L[i];
        int nl = nearest_int(x[i] * sl2 / slx);
        nl = mx(-nmax, mn(nmax - 1, nl));
        if (nl != L[i]) {
          slx += w * x[i] * nl;
          sl2 += w * nl * nl;
          if (sl2 > 0 && slx * slx * suml2 > sumlx * sumlx * sl2) {
            L[i] = nl;
            sumlx = slx;
            suml2 = sl2;
            ++changed;
          }
        }
      }
    }
    if (!changed) break;
  }
#pragma unroll
  for (int i = 0; i < N; ++i) L[i] += nmax;
  return sumlx / suml2;
}

template <typename F, int... I>
__device__ __forceinline__ void static_for_q_impl(F &&f, std::integer_sequence<int, I...>) {
  (f.template operator()<I>(), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for_q(F &&f) {
  static_for_q_impl(f, std::make_integer_sequence<int, N>{});
}

// FP8 E4M3 ("fn": bias 7, no infinities, S.1111.111 is NaN) to f32, exact.
__device__ __forceinline__ float e4m3_to_f32(uint8_t b) {
  const uint32_t sign = (uint32_t)(b & 0x80) << 24;
  const uint32_t e = (b >> 3) & 0xF, m = b & 7;
  if (e == 0xF && m == 7) return __uint_as_float(sign | 0x7FC00000u);
  if (e == 0) {
    const float v = (float)m * 0.001953125f;  // m / 8 * 2^-6
    return sign ? -v : v;
  }
  return __uint_as_float(sign | ((e + 120u) << 23) | (m << 20));
}

// A block image's bytes [OFF, OFF + 4) as a little-endian word (constant
// offsets, so the image stays in registers).
template <int OFF>
__device__ __forceinline__ uint32_t image_word(const uint8_t *o) {
  return (uint32_t)o[OFF] | ((uint32_t)o[OFF + 1] << 8) | ((uint32_t)o[OFF + 2] << 16) | ((uint32_t)o[OFF + 3] << 24);
}

// Field F of a block image into the tiled planes at (tile-block tb, row r):
// a 16-byte column per chunk of a chunked field, one run for a record (the
// same places the repack writes).
template <int TYPE, int F>
__device__ __forceinline__ void store_field(uint8_t *tiled, const Geo &g, int64_t tb, int r, const uint8_t *o) {
  constexpr TypeInfo ti = type_info(TYPE);
  constexpr int size = ti.f[F].size, off = ti.f[F].off;
  if constexpr (size % 16 == 0) {
    static_for_q<size / 16>([&]<int C>() {
      const uint4 v = make_uint4(image_word<off + 16 * C>(o), image_word<off + 16 * C + 4>(o),
                                 image_word<off + 16 * C + 8>(o), image_word<off + 16 * C + 12>(o));
      *reinterpret_cast<uint4 *>(tiled + g.plane[F] + ((tb * (size / 16) + C) * kRowTile + r) * 16) = v;
    });
  } else if constexpr (size == 4) {
    *reinterpret_cast<uint32_t *>(tiled + g.plane[F] + (tb * kRowTile + r) * 4) = image_word<off>(o);
  } else {
    static_assert(size == 2, "record fields of the 32-element types are 2 or 4 bytes");
    *reinterpret_cast<uint16_t *>(tiled + g.plane[F] + (tb * kRowTile + r) * 2) =
        (uint16_t)((uint32_t)o[off] | ((uint32_t)o[off + 1] << 8));
  }
}

// The 32-element types straight into the device layout: one 64-thread
// workgroup per (4 consecutive blocks, 64-row tile t); thread r quantizes row
// t * 64 + r's blocks (a 128-byte run of FP8 or 512 bytes of f32: whole cache
// lines; rows past n: zeros, as the repack writes them) and stores each
// block's fields where the repack would put them, so there is no raw staging
// and no repack pass (the repack reads these 18-34-byte blocks 2 bytes at a
// time).
constexpr int kQtBlocks = 4;

template <int TYPE>
__device__ __forceinline__ void quant_block(const float *x, uint8_t *o) {
  if constexpr (TYPE == Q4_0) q_q4_0(x, o);
  else if constexpr (TYPE == Q4_1) q_q4_1(x, o);
  else if constexpr (TYPE == Q5_0) q_q5_0(x, o);
  else if constexpr (TYPE == Q5_1) q_q5_1(x, o);
  else q_q8_0(x, o);
}

template <int TYPE, bool FP8, bool VEC>
__global__ __launch_bounds__(64) void quantize_tiled_kernel(const void *__restrict__ src, int64_t ld, Geo g,
                                                            float scale, uint8_t *__restrict__ tiled) {
  constexpr TypeInfo ti = type_info(TYPE);
  static_assert(ti.bs == 32, "32-element block types only");
  const int64_t t = blockIdx.y;
  const int r = threadIdx.x;
  const int64_t row = t * kRowTile + r;
#pragma unroll
  for (int j = 0; j < kQtBlocks; ++j) {
    const int64_t b = (int64_t)blockIdx.x * kQtBlocks + j;
    if (b >= g.nb) break;  // uniform across the workgroup
    uint8_t o[ti.ts];
    if (row < g.n) {
      float x[32];
      if constexpr (FP8) {
        const uint8_t *p = static_cast<const uint8_t *>(src) + row * ld + b * 32;
        if constexpr (VEC) {
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const uint4 v = reinterpret_cast<const uint4 *>(p)[c];
            const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 16; ++i) x[16 * c + i] = e4m3_to_f32((uint8_t)(wd[i >> 2] >> (8 * (i & 3)))) * scale;
          }
        } else {
#pragma unroll
          for (int i = 0; i < 32; ++i) x[i] = e4m3_to_f32(p[i]) * scale;
        }
      } else {
        const float *p = static_cast<const float *>(src) + row * ld + b * 32;
        if constexpr (VEC) {
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            const float4 v = reinterpret_cast<const float4 *>(p)[c];
            x[4 * c] = v.x;
            x[4 * c + 1] = v.y;
            x[4 * c + 2] = v.z;
            x[4 * c + 3] = v.w;
          }
        } else {
#pragma unroll
          for (int i = 0; i < 32; ++i) x[i] = p[i];
        }
      }
      quant_block<TYPE>(x, o);
    } else {
#pragma unroll
      for (int i = 0; i < ti.ts; ++i) o[i] = 0;
    }
    const int64_t tb = t * g.nb + b;
    static_for_q<ti.nf>([&]<int F>() { store_field<TYPE, F>(tiled, g, tb, r, o); });
  }
}

// ------------------------------------------------------------- k-quant blocks
// Each thread quantizes one sub-block and the super-block's 8 (Q4_K, Q5_K) or
// 16 lanes share the rest: the largest scale by lane exchanges, packed words
// or-ed across the lanes that hold their other bits, and every 16-byte chunk
// stored by one lane straight into the device layout (rows past n as zeros).
// With one thread a super-block (the values, quants and search candidates in
// private memory, raw blocks to a staging buffer, then a repack pass) Q4_K
// [21504, 3072] took 1022 + 39 us, now 640 (VALU-bound: 438 instructions a value,
// a wave instruction every 3.1 cycles per SIMD at 2.1 GHz); [8192, 3072] whole calls, before -> now: Q2_K 496 ->
// 242 us, Q3_K 428 -> 133, Q4_K 567 -> 298, Q5_K 538 -> 247, Q6_K 383 -> 182.

// v combined over the W lanes of a super-block by or / by maximum (values never NaN there).
template <int W>
__device__ __forceinline__ uint32_t group_or(uint32_t v) {
#pragma unroll
  for (int m = 1; m < W; m *= 2) v |= (uint32_t)__shfl_xor((int)v, m);
  return v;
}
template <int W>
__device__ __forceinline__ float group_max0(float v) {
  v = v > 0.f ? v : 0.f;  // ggml: max = 0; if (v > max) max = v
#pragma unroll
  for (int m = 1; m < W; m *= 2) {
    const float u = __shfl_xor(v, m);
    v = u > v ? u : v;
  }
  return v;
}
// The value of largest magnitude over the group's 16 lanes, the lowest lane's
// on a tie (0 if every magnitude is 0 or NaN).
__device__ __forceinline__ float group_absmax(float v, float &amax) {
  float a = fabsf(v);
  if (!(a > 0.f)) { a = 0.f; v = 0.f; }
  int at = threadIdx.x & 15;
#pragma unroll
  for (int m = 1; m < 16; m *= 2) {
    const float ua = __shfl_xor(a, m), uv = __shfl_xor(v, m);
    const int ut = __shfl_xor(at, m);
    if (ua > a || (ua == a && ut < at)) { a = ua; v = uv; at = ut; }
  }
  amax = a;
  return v;
}

// Words of 4 quants, one per byte.
template <int N>
__device__ __forceinline__ void pack_bytes(const int (&L)[N], uint32_t (&p)[N / 4]) {
#pragma unroll
  for (int i = 0; i < N / 4; ++i)
    p[i] = (uint32_t)L[4 * i] | ((uint32_t)L[4 * i + 1] << 8) | ((uint32_t)L[4 * i + 2] << 16) |
           ((uint32_t)L[4 * i + 3] << 24);
}
// p |= the lanes' at distance m, each lane's already shifted to its bits.
template <int N>
__device__ __forceinline__ void or_lanes(uint32_t (&p)[N], int m) {
#pragma unroll
  for (int i = 0; i < N; ++i) p[i] |= (uint32_t)__shfl_xor((int)p[i], m);
}
__device__ __forceinline__ void put_chunk(uint8_t *tiled, int64_t plane, int nchunks, int64_t tb, int c, int r,
                                          const uint32_t *w) {
  *reinterpret_cast<uint4 *>(tiled + plane + ((tb * nchunks + c) * kRowTile + r) * 16) =
      make_uint4(w[0], w[1], w[2], w[3]);
}
// The low or high four of eight words (by value: a run-time pointer into w
// would put it in private memory).
__device__ __forceinline__ void put_half(uint8_t *tiled, int64_t plane, int nchunks, int64_t tb, int c, int r,
                                         const uint32_t (&w)[8], bool high) {
  const uint32_t v[4] = {high ? w[4] : w[0], high ? w[5] : w[1], high ? w[6] : w[2], high ? w[7] : w[3]};
  put_chunk(tiled, plane, nchunks, tb, c, r, v);
}
template <typename V>
__device__ __forceinline__ void put_record(uint8_t *tiled, int64_t plane, int size, int64_t tb, int r, int off, V v) {
  *reinterpret_cast<V *>(tiled + plane + (tb * kRowTile + r) * size + off) = v;
}

template <int TYPE>
constexpr int kq_lanes() {
  return TYPE == Q4_K || TYPE == Q5_K ? 8 : 16;
}

// Sub-block j of block tb, tile row r, from its values x (`real`: a row of the
// tensor; padding rows are zero bytes).  Every lane of the wave joins.
template <int TYPE, int N>
__device__ __forceinline__ void quantize_sub(const float (&x)[N], bool real, int j, uint8_t *t, const Geo &g, int64_t tb,
                                             int r) {
  int L[N];
  uint32_t p[N / 4];
  if constexpr (TYPE == Q4_K || TYPE == Q5_K) {
    constexpr bool FIVE = TYPE == Q5_K;
    constexpr int nmax = FIVE ? 31 : 15;
    float w[N], sum_x2 = 0;
#pragma unroll
    for (int l = 0; l < N; ++l) sum_x2 += x[l] * x[l];
    const float av_x = sqrtf(sum_x2 / 32);
#pragma unroll
    for (int l = 0; l < N; ++l) w[l] = av_x + fabsf(x[l]);
    const Qkx2 s = qkx2<N, false>(nmax, x, w, FIVE ? -0.5f : -1.f, 0.1f, FIVE ? 15 : 20);
    const float max_scale = group_max0<8>(s.scale), max_min = group_max0<8>(s.the_min);
    const float inv_scale = max_scale > 0 ? 63.f / max_scale : 0.f;
    const float inv_min = max_min > 0 ? 63.f / max_min : 0.f;
    const uint32_t ls = mn<uint8_t>(63, (uint8_t)nearest_int(inv_scale * s.scale));
    const uint32_t lm = mn<uint8_t>(63, (uint8_t)nearest_int(inv_min * s.the_min));
    // byte j of words 0 / 1: the low 6 bits for j < 4; nibbles in word 2 and the
    // top 2 bits above words 0 / 1's for j >= 4
    const int sh = 8 * (j & 3);
    const uint32_t s0 = group_or<8>((j < 4 ? ls : (ls >> 4) << 6) << sh);
    const uint32_t s1 = group_or<8>((j < 4 ? lm : (lm >> 4) << 6) << sh);
    const uint32_t s2 = group_or<8>(j < 4 ? 0u : ((ls & 0xF) | ((lm & 0xF) << 4)) << sh);
    const uint16_t dh = f2h(max_scale / 63.f), mh = f2h(max_min / 63.f);
    const float d = h2f(dh) * (float)ls, dm = h2f(mh) * (float)lm;
    if (d) {
#pragma unroll
      for (int i = 0; i < N; ++i) L[i] = mx(0, mn(nmax, nearest_int((x[i] + dm) / d)));
    } else {  // the search's quants stay
#pragma unroll
      for (int i = 0; i < N; ++i) L[i] = mx(0, mn(nmax, nearest_int(s.best_iscale * (x[i] - s.best_min))));
    }
    pack_bytes(L, p);
    if constexpr (FIVE) {
      uint32_t hb[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        hb[i] = ((p[i] >> 4) & 0x01010101u) << j;
        p[i] &= 0x0F0F0F0Fu;
      }
      or_lanes(hb, 1);
      or_lanes(hb, 2);
      or_lanes(hb, 4);
#pragma unroll
      for (int i = 0; i < 8; ++i) hb[i] = real ? hb[i] : 0u;
      if (j < 2) put_half(t, g.plane[2], 2, tb, j, r, hb, j != 0);
    }
    // sub-blocks 2g and 2g + 1 are the low and high nibbles of bytes 32 g ..
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] <<= 4 * (j & 1);
    or_lanes(p, 1);
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = real ? p[i] : 0u;
    put_half(t, g.plane[FIVE ? 3 : 2], 8, tb, j, r, p, (j & 1) != 0);
    if (j == 0) {
      put_record<uint32_t>(t, g.plane[0], 4, tb, r, 0, real ? (uint32_t)dh | ((uint32_t)mh << 16) : 0u);
      put_record<uint32_t>(t, g.plane[1], 12, tb, r, 0, real ? s0 : 0u);
      put_record<uint32_t>(t, g.plane[1], 12, tb, r, 4, real ? s1 : 0u);
      put_record<uint32_t>(t, g.plane[1], 12, tb, r, 8, real ? s2 : 0u);
    }
  } else {
    // sub-block j = 8 H + 2 p + half: elements 128 H + 32 p + 16 half ..
    const int H = j >> 3, pp = (j >> 1) & 3, half = j & 1;
    if constexpr (TYPE == Q2_K) {
      float w[N];
#pragma unroll
      for (int l = 0; l < N; ++l) w[l] = fabsf(x[l]);
      const Qkx2 s = qkx2<N, true>(3, x, w, -0.5f, 0.1f, 15);
      const float max_scale = group_max0<16>(s.scale), max_min = group_max0<16>(s.the_min);
      uint32_t sc = 0;
      uint16_t dh = f2h(0.f), mh = f2h(0.f);
      if (max_scale > 0) {
        const float iscale = 15.f / max_scale;
        sc = (uint8_t)nearest_int(iscale * s.scale);
        dh = f2h(max_scale / 15.f);
      }
      if (max_min > 0) {
        const float iscale = 15.f / max_min;
        sc |= (uint8_t)(nearest_int(iscale * s.the_min) << 4);
        mh = f2h(max_min / 15.f);
      }
      const float d = h2f(dh) * (float)(sc & 0xF), dm = h2f(mh) * (float)(sc >> 4);
      if (d) {
#pragma unroll
        for (int i = 0; i < N; ++i) L[i] = mx(0, mn(3, nearest_int((x[i] + dm) / d)));
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i) L[i] = mx(0, mn(3, nearest_int(s.best_iscale * (x[i] - s.best_min))));
      }
      pack_bytes(L, p);
      put_record<uint8_t>(t, g.plane[0], 16, tb, r, j, real ? (uint8_t)sc : 0);
      if (j == 0) put_record<uint32_t>(t, g.plane[2], 4, tb, r, 0, real ? (uint32_t)dh | ((uint32_t)mh << 16) : 0u);
    } else if constexpr (TYPE == Q3_K) {
      float amax;
      const float scale = q3_group<N>(4, x, L);
      const float max_scale = group_absmax(scale, amax);
      uint32_t l6 = 0;
      uint16_t dh = f2h(0.f);
      if (max_scale) {
        const float iscale = -32.f / max_scale;
        const int8_t l = (int8_t)nearest_int(iscale * scale);
        l6 = (uint32_t)(mx(-32, mn(31, (int)l)) + 32);
        dh = f2h(1 / iscale);
      }
      const uint32_t low = (l6 & 0xF) << (8 * (j & 3) + 4 * (j >> 3));
      const uint32_t s0 = group_or<16>((j & 4) ? 0u : low), s1 = group_or<16>((j & 4) ? low : 0u);
      const uint32_t s2 = group_or<16>((l6 >> 4) << (8 * (j & 3) + 2 * (j >> 2)));
      // without a scale the 12 bytes are zero, which reads back as -32
      const float d = h2f(dh) * (float)((int)l6 - 32);
      if (d) {
#pragma unroll
        for (int i = 0; i < N; ++i) L[i] = mx(-4, mn(3, nearest_int(x[i] / d))) + 4;
      }
      uint32_t hm[4];
      pack_bytes(L, p);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        hm[i] = ((p[i] >> 2) & 0x01010101u) << (j >> 1);  // bit 4 H + p: the value is above 3
        p[i] &= 0x03030303u;
      }
      or_lanes(hm, 2);
      or_lanes(hm, 4);
      or_lanes(hm, 8);
#pragma unroll
      for (int i = 0; i < 4; ++i) hm[i] = real ? hm[i] : 0u;
      if (j < 2) put_chunk(t, g.plane[0], 2, tb, j, r, hm);
      if (j == 0) {
        put_record<uint32_t>(t, g.plane[2], 12, tb, r, 0, real ? s0 : 0u);
        put_record<uint32_t>(t, g.plane[2], 12, tb, r, 4, real ? s1 : 0u);
        put_record<uint32_t>(t, g.plane[2], 12, tb, r, 8, real ? s2 : 0u);
        put_record<uint16_t>(t, g.plane[3], 2, tb, r, 0, real ? dh : 0);
      }
    } else {
      static_assert(TYPE == Q6_K);
      float best_iscale, amax;
      bool zero;
      const float scale = qx_rmse1<N>(32, x, best_iscale, zero);
      const float max_scale = group_absmax(scale, amax);
      const bool none = amax < kGroupMaxEps;  // a super-block of zeros is zero bytes
      const float iscale = -128.f / max_scale;
      const uint16_t dh = none ? f2h(0.f) : f2h(1 / iscale);
      const int sc = none ? 0 : (int)(int8_t)mn(127, nearest_int(iscale * scale));
      const float d = h2f(dh) * (float)sc;
      if (d) {
#pragma unroll
        for (int i = 0; i < N; ++i) L[i] = mx(-32, mn(31, nearest_int(x[i] / d))) + 32;
      } else {
#pragma unroll
        for (int i = 0; i < N; ++i) L[i] = zero || none ? 0 : 32 + mx(-32, mn(31, nearest_int(best_iscale * x[i])));
      }
      uint32_t ph[4];
      pack_bytes(L, p);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ph[i] = ((p[i] >> 4) & 0x03030303u) << (2 * pp);
        p[i] = (p[i] & 0x0F0F0F0Fu) << (4 * (pp >> 1));
      }
      or_lanes(ph, 2);
      or_lanes(ph, 4);
      or_lanes(p, 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[i] = real ? p[i] : 0u;
        ph[i] = real ? ph[i] : 0u;
      }
      if (pp < 2) put_chunk(t, g.plane[0], 8, tb, 4 * H + 2 * pp + half, r, p);
      if (pp == 0) put_chunk(t, g.plane[1], 4, tb, 2 * H + half, r, ph);
      put_record<uint8_t>(t, g.plane[2], 16, tb, r, j, real ? (uint8_t)sc : 0);
      if (j == 0) put_record<uint16_t>(t, g.plane[3], 2, tb, r, 0, real ? dh : 0);
    }
    if constexpr (TYPE == Q2_K || TYPE == Q3_K) {
      // the 2-bit planes: byte 32 H + 16 half + i holds the four p's at bits 2 p
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] <<= 2 * pp;
      or_lanes(p, 2);
      or_lanes(p, 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] = real ? p[i] : 0u;
      if (pp == 0) put_chunk(t, g.plane[1], 4, tb, 2 * H + half, r, p);
    }
  }
}

// Workgroup: 256 / lanes rows of one super-block column (columns fastest);
// lane -> (row, sub-block), sub-block fastest.
template <int TYPE, bool FP8, bool VEC>
__global__ __launch_bounds__(256) void quantize_k_kernel(const void *__restrict__ src, int64_t ld, Geo g, float scale,
                                                         uint8_t *__restrict__ tiled) {
  constexpr int kL = kq_lanes<TYPE>(), N = 256 / kL;
  const int j = threadIdx.x % kL;
  const int64_t rg = blockIdx.x / (uint32_t)g.nb, b = blockIdx.x - rg * g.nb;
  const int64_t row = rg * (256 / kL) + threadIdx.x / kL;  // < 64 ntiles
  const bool real = row < g.n;
  float x[N];
  const int64_t at = (real ? row : 0) * ld + b * 256 + j * N;
  if constexpr (FP8) {
    const uint8_t *p = static_cast<const uint8_t *>(src) + at;
    if constexpr (VEC) {
#pragma unroll
      for (int c = 0; c < N / 16; ++c) {
        const uint4 v = reinterpret_cast<const uint4 *>(p)[c];
        const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 16; ++i) x[16 * c + i] = e4m3_to_f32((uint8_t)(wd[i >> 2] >> (8 * (i & 3)))) * scale;
      }
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) x[i] = e4m3_to_f32(p[i]) * scale;
    }
  } else {
    const float *p = static_cast<const float *>(src) + at;
    if constexpr (VEC) {
#pragma unroll
      for (int c = 0; c < N / 4; ++c) {
        const float4 v = reinterpret_cast<const float4 *>(p)[c];
        x[4 * c] = v.x;
        x[4 * c + 1] = v.y;
        x[4 * c + 2] = v.z;
        x[4 * c + 3] = v.w;
      }
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) x[i] = p[i];
    }
  }
  quantize_sub<TYPE, N>(x, real, j, tiled, g, (row / kRowTile) * g.nb + b, (int)(row % kRowTile));
}

// A LoRA merge in one pass: the weight's own values (decoded as dequantize
// does), plus each patch's (b . a) * scale on its rows, quantized again; the
// steps and their order are those of dequantize, lora_apply per patch and
// quantize, so the blocks are the same.  Bound by the search's VALU work as
// quantize_k_kernel is: decode and rank-32 patches add 52 instructions a value to
// 438, where the separate passes moved 17 bytes a value through HBM (written 4,
// read and written 4 + 4 by the patches, read 4, the blocks 0.6 each way; Q4_K
// [21504, 3072], four rank-32 patches: 55 + 234 + 640 us, in one pass 685; the
// merge call 1003 -> 721).  A patch's a (kLoraR ranks of the workgroup's 256
// columns) and b are staged in LDS, a with the lanes' 16-byte pieces side by side
// (piece c of sub-block j at c * lanes + j: the lanes of a row read 128 or 256
// consecutive bytes).
constexpr int kLoraR = 32;

template <int TYPE>
__global__ __launch_bounds__(256, 2) void lora_merge_kernel(WView w, Geo g, LoraPatches patches, uint8_t *__restrict__ tiled) {
  constexpr int kL = kq_lanes<TYPE>(), N = 256 / kL, kRows = 256 / kL;
  __shared__ __align__(16) float as[kLoraR][256];
  __shared__ float bs[kLoraR][kRows];
  const int tid = threadIdx.x, j = tid % kL, rl = tid / kL;
  const int64_t rg = blockIdx.x / (uint32_t)g.nb, blk = blockIdx.x - rg * g.nb;
  const int64_t row0 = rg * kRows, row = row0 + rl;
  const bool real = row < g.n;
  const int64_t tile = row / kRowTile;
  const int r64 = (int)(row % kRowTile);
  float x[N];
#pragma unroll
  for (int c = 0; c < N / 8; ++c) {
    float v[8];
    decode8<TYPE>(w, tile, r64, blk, j * N + 8 * c, v);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      // the f32 weight itself: without this the decoder's last multiply-add may
      // move past the patch's add
      asm volatile("" : "+v"(v[i]));
      x[8 * c + i] = v[i];
    }
  }
  for (int p = 0; p < patches.count; ++p) {
    const LoraPatch &q = patches.p[p];
    if (row0 + kRows <= q.row0 || row0 >= q.row0 + q.rows) continue;  // none of the workgroup's rows
    const bool mine = row >= q.row0 && row < q.row0 + q.rows;
    float d[N];
#pragma unroll
    for (int i = 0; i < N; ++i) d[i] = 0.f;
    for (int r0 = 0; r0 < q.rank; r0 += kLoraR) {
      const int rn = q.rank - r0 < kLoraR ? q.rank - r0 : kLoraR;
      __syncthreads();  // the chunk before is read
      for (int e = tid; e < rn * 256; e += 256) {
        const int rr = e >> 8, col = e & 255, sub = col / N, in = col % N;
        as[rr][((in >> 2) * kL + sub) * 4 + (in & 3)] = q.a[(int64_t)(r0 + rr) * q.lda + blk * 256 + col];
      }
      for (int e = tid; e < rn * kRows; e += 256) {
        const int rr = e / kRows, ii = e % kRows;
        const int64_t pr = row0 + ii - q.row0;
        bs[rr][ii] = pr >= 0 && pr < q.rows ? q.b[pr * q.ldb + r0 + rr] : 0.f;
      }
      __syncthreads();
      for (int rr = 0; rr < rn; ++rr) {
        const float bv = bs[rr][rl];
#pragma unroll
        for (int c = 0; c < N / 4; ++c) {
          const float4 av = *reinterpret_cast<const float4 *>(&as[rr][(c * kL + j) * 4]);
          d[4 * c] = __builtin_fmaf(bv, av.x, d[4 * c]);
          d[4 * c + 1] = __builtin_fmaf(bv, av.y, d[4 * c + 1]);
          d[4 * c + 2] = __builtin_fmaf(bv, av.z, d[4 * c + 2]);
          d[4 * c + 3] = __builtin_fmaf(bv, av.w, d[4 * c + 3]);
        }
      }
    }
    if (mine) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const float t = d[i] * q.scale;
        x[i] = x[i] + t;
      }
    }
  }
  quantize_sub<TYPE, N>(x, real, j, tiled, g, tile * g.nb + blk, r64);
}

template <bool FP8>
hipError_t launch_quantize_src(int type, const void *src, int64_t ld, float scale, void *tiled, const Geo &g,
                                     hipStream_t stream) {
  if (g.n == 0 || g.nb == 0) return hipSuccess;
  const int64_t es = FP8 ? 1 : 4;
  const bool vec = (reinterpret_cast<uintptr_t>(src) & 15) == 0 && (ld * es) % 16 == 0;
  bool ok = dispatch_type(type, [&]<int T>() {
    if constexpr (type_info(T).bs == 32) {
      const dim3 grid((unsigned)((g.nb + kQtBlocks - 1) / kQtBlocks), (unsigned)g.ntiles);
      if (vec)
        hipLaunchKernelGGL((quantize_tiled_kernel<T, FP8, true>), grid, dim3(64), 0, stream, src, ld, g, scale,
                           static_cast<uint8_t *>(tiled));
      else
        hipLaunchKernelGGL((quantize_tiled_kernel<T, FP8, false>), grid, dim3(64), 0, stream, src, ld, g, scale,
                           static_cast<uint8_t *>(tiled));
    } else {
      const dim3 grid((unsigned)(g.nb * (g.ntiles * kRowTile * kq_lanes<T>() / 256)));
      if (vec)
        hipLaunchKernelGGL((quantize_k_kernel<T, FP8, true>), grid, dim3(256), 0, stream, src, ld, g, scale,
                           static_cast<uint8_t *>(tiled));
      else
        hipLaunchKernelGGL((quantize_k_kernel<T, FP8, false>), grid, dim3(256), 0, stream, src, ld, g, scale,
                           static_cast<uint8_t *>(tiled));
    }
  });
  if (!ok) return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace

hipError_t launch_lora_merge(int type, const WView &w, const Geo &g, const LoraPatches &patches, void *tiled,
                             hipStream_t stream) {
  if (g.n == 0 || g.nb == 0) return hipSuccess;
  bool ok = false;
  dispatch_type(type, [&]<int T>() {
    if constexpr (type_info(T).bs == 256) {
      const dim3 grid((unsigned)(g.nb * (g.ntiles * kRowTile * kq_lanes<T>() / 256)));
      hipLaunchKernelGGL((lora_merge_kernel<T>), grid, dim3(256), 0, stream, w, g, patches, static_cast<uint8_t *>(tiled));
      ok = true;
    }
  });
  if (!ok) return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_quantize(int type, const void *src, bool fp8, int64_t ld, float scale, void *tiled, const Geo &g,
                           hipStream_t stream) {
  return fp8 ? launch_quantize_src<true>(type, src, ld, scale, tiled, g, stream)
             : launch_quantize_src<false>(type, src, ld, 1.0f, tiled, g, stream);
}

}  // namespace mq
