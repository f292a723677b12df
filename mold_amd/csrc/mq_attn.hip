// mq_attn.hip — the DiT blocks' joint attention: softmax(q k^T / sqrt(128)) v
// over bf16 heads of 128, f32 scores, softmax and sums, written in the
// [rows, heads * 128] layout the out-projection reads (FLUX
// crates/mold-inference/src/flux/offload.rs:39-73, Qwen-Image qwen_image/
// quantized_transformer.rs:753-823).
//
// What bounds it: two contractions of 2 rows * keys * 128 FLOP per head on the
// matrix cores, with one exponential per score to hide behind them: 226 vector
// instructions per 32 MFMAs.  Counted at 24 x 7145 and 1.85 GHz: matrix pipes busy
// 0.46 of the cycles, vector ALU 0.41 (4 cycles an instruction), no LDS conflict.
// Shape of the work for gfx950:
//   * a workgroup of W waves takes 32 W query rows of one head, a wave 32 of
//     them; keys come in blocks of 64, K and V global -> LDS by LDS DMA one
//     block ahead (K in a ring of two blocks, V of three: 80 KiB);
//   * the scores are computed transposed, S^T = K Q^T (v_mfma_f32_32x32x16):
//     a lane then holds 16 keys of one query, so the row maximum and sum are
//     in-lane but for one exchange between the wave's halves, and the
//     probabilities are, rounded to bf16, the B operand of O^T = V^T P^T as
//     they stand (no shuffle, no LDS round trip);
//   * V^T, that product's A operand, is read from row-major V by
//     ds_read_b64_tr_b16 (4 keys x 16 columns per 16 lanes, transposed on the
//     way); both tiles are swizzled in 16-byte chunks so that neither read
//     conflicts: K's chunk c of key r in slot c ^ (r & 15), V's in
//     c ^ 4 (r & 3);
//   * the scores run one 32-key half block ahead of the softmax, so a wave's
//     own MFMAs and exponentials overlap (7 % faster than the same kernel in
//     program order at 24 x 4608, 4 % at 24 x 7145);
//   * the running maximum is exact after every half block (the probabilities
//     round to bf16, and those near the row's maximum then sit just under 1,
//     where bf16's step is relatively smallest; letting it lag until it was
//     2^8 off was 8-12 % faster and put the result 2-20 % further from
//     float64, more the sharper the scores), and O is rescaled only when it
//     rose for some row of the wave.
// Keys past the last one and a masked range [drop_lo, drop_hi) never enter:
// the kept keys are numbered in order and only the last block is masked.
//
// Measured against the fused attention PyTorch ships for this device (same
// process, scores N(0, 1)): 24 x 4608 tokens 529 -> 280 us (931 TFLOP/s),
// 24 x 7145 of 7168 with its correction pass 960 -> 604 us (1038 TFLOP/s), 24 x
// 300 of 512 30 -> 9 us; distance to float64 the same without padding
// (2.25e-3, 1.93e-3 and 1.71e-3 at scores of 1, 2 and 6) and smaller with it,
// where the separate correction rounded to bf16 a second time (2.8e-3 ->
// 2.3e-3).
#include "../../include/moldq.h"
#include "mq_kernels.h"

namespace mq {
int set_error(int code, const char *msg);
}

namespace mq {
namespace {

typedef __attribute__((address_space(3))) char lds_char;
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kHd = 128;       // head dim
constexpr int kKeys = 64;      // keys per block
constexpr int kMaxBatch = 8;   // elements per launch (their masks are kernel arguments)
constexpr int kCus = 256;      // MI355X
constexpr int kMaxParts = 8;   // key shares of a split tile
constexpr int64_t kPart = 256 * (kHd + 2);  // floats of one share's sums

// Per batch element: kept keys, the masked range's start and length, and the
// zero keys that the caller's guard counts.
struct AttnKeys {
  int nk[kMaxBatch], lo[kMaxBatch], gap[kMaxBatch];
  float npad[kMaxBatch];
};

// 16 bytes per lane from base + off straight into LDS (lane i at lds + 16 i);
// base and lds are wave-uniform.  Read only after block_barrier.
__device__ __forceinline__ void dma16(const char *base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds)
               : "memory", "m0");
}

// This wave's DMA has landed and its LDS reads are complete; then every wave arrives.
__device__ __forceinline__ void block_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) expcnt(7) lgkmcnt(0)
  asm volatile("s_barrier" ::: "memory");
}

// The value combined with lane ^ 32's.
__device__ __forceinline__ float half_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __builtin_fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_add(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ uint32_t pack2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 p = __builtin_convertvector((f32x2){a, b}, bf16x2);
  uint32_t u;
  __builtin_memcpy(&u, &p, 4);
  return u;
}

// The log-sum-exp and guard of a row with sum l relative to 2^ms, which all
// lanes of a half wave (or both halves) share or hold one each; `one`: the
// lane that stores it.  Z + npad, the sum of exp over the kept keys and npad
// zero scores, is taken relative to 2^max(ms, 0).  Every lane of the wave joins.
__device__ __forceinline__ void row_sums(float ms, float l, float npad, bool stored, bool one, float *lse,
                                         unsigned int *guard) {
  const float top = __builtin_fmaxf(ms, 0.f);
  const float zero = npad * __builtin_amdgcn_exp2f(-top);
  const float z = l * __builtin_amdgcn_exp2f(ms - top) + zero;
  if (lse && stored && one) *lse = 0.69314718055994531f * (top + __builtin_amdgcn_logf(z));
  if (guard) {
    float share = stored ? zero / z : 0.f;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const float u = __shfl_xor(share, off);
      share = (u > share || u != u) ? u : share;
    }
    const unsigned int bits = __float_as_uint(share);
    if ((threadIdx.x & 63) == 0 && bits > __hip_atomic_load(guard, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(guard, bits);
  }
}

template <int S>
struct Slot {
  static constexpr int v = S;
};

template <int W, bool kSplit>
__global__ __launch_bounds__(64 * W, 2) void attention_kernel(
    const __bf16 *__restrict__ q, const __bf16 *__restrict__ k, const __bf16 *__restrict__ v, int heads,
    int64_t l_total, int rows, int qtiles, AttnKeys keys, float scale, __bf16 *__restrict__ out, int64_t sb_out,
    int64_t ldo, float *__restrict__ lse, unsigned int *__restrict__ guard, int full_tiles, int kparts,
    float *__restrict__ partial) {
  __shared__ uint4 lds_k[2][kKeys * kHd / 8];
  __shared__ uint4 lds_v[3][kKeys * kHd / 8];

  // Workgroup i runs on XCD i % 8: each XCD takes a contiguous run of (head,
  // query tile), so one head's K and V stay in its L2.  Tiles from full_tiles
  // (then a multiple of kCus) on run as kparts workgroups, each over a share of
  // the keys, whose sums combine_kernel adds.
  const bool split = kSplit && (int)blockIdx.x >= full_tiles;
  const int i0 = split ? blockIdx.x - full_tiles : blockIdx.x;
  const int total = !kSplit ? gridDim.x : split ? gridDim.x - full_tiles : full_tiles;
  const int xcd = i0 & 7, base = total >> 3, extra = total & 7;
  const int unit = xcd * base + (xcd < extra ? xcd : extra) + (i0 >> 3);
  const int tile = split ? full_tiles + unit / kparts : unit, part = split ? unit % kparts : 0;
  const int bh = tile / qtiles, qt = tile - bh * qtiles;
  const int b = bh / heads, head = bh - b * heads;
  const int nk = keys.nk[b], lo = keys.lo[b], gap = keys.gap[b];
  const int all = (nk + kKeys - 1) / kKeys;
  const int b0 = split ? part * all / kparts : 0;  // first block of keys
  const int nblk = (split ? (part + 1) * all / kparts : all) - b0;

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = 32 * (W * qt + wave) + l32;  // this lane's query
  const int64_t hoff = (int64_t)bh * l_total * kHd;

  bf16x8 qf[8];  // the B operand of the scores; rows past the last repeat it and are not stored
  {
    const __bf16 *p = q + hoff + (int64_t)(row < rows ? row : rows - 1) * kHd + 8 * h;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *reinterpret_cast<const bf16x8 *>(p + 16 * s);
  }

  // DMA of a block: load j of a wave fills LDS rows 4 (wave + W j) .. + 3,
  // lane -> row lane / 16, slot lane % 16, fetching the chunk the swizzle puts
  // there.  Rows past the last key repeat it (its score is masked).
  const char *kbase = reinterpret_cast<const char *>(k + hoff), *vbase = reinterpret_cast<const char *>(v + hoff);
  const int drow = 4 * wave + (lane >> 4);
  const uint32_t kch = (uint32_t)(((lane & 15) ^ (drow & 15)) << 4);
  const uint32_t vch = (uint32_t)(((lane & 15) ^ ((lane >> 4) << 2)) << 4);
  const uint32_t lkw = (uint32_t)(uintptr_t)(&lds_k[0][0]) + 1024 * wave;
  const uint32_t lvw = (uint32_t)(uintptr_t)(&lds_v[0][0]) + 1024 * wave;
  auto dma = [&](int blk, int kslot, int vslot) {
#pragma unroll
    for (int j = 0; j < 16 / W; ++j) {
      int r = (b0 + blk) * kKeys + drow + 4 * W * j;
      r = r < nk ? r : nk - 1;
      const uint32_t off = (uint32_t)(r + (r >= lo ? gap : 0)) * (2 * kHd);
      dma16(kbase, off + kch, __builtin_amdgcn_readfirstlane(lkw + kslot * 16384 + 1024 * W * j));
      dma16(vbase, off + vch, __builtin_amdgcn_readfirstlane(lvw + vslot * 16384 + 1024 * W * j));
    }
  };

  f32x16 o[4];  // O^T: this lane's query, columns 32 d + 8 (e / 4) + 4 h + e % 4
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[d][e] = 0.f;
  // running maximum (both halves), finite so that scores of -inf before the first
  // finite one give 0 and not NaN, and this half's sum
  float m = -__FLT_MAX__, l = 0.f;

  const int i16 = lane & 15;
  lds_char *ka[8], *va[4];
#pragma unroll
  for (int s = 0; s < 8; ++s)
    ka[s] = (lds_char *)&lds_k[0][0] + (uint32_t)(l32 * 256 + (((2 * s + h) ^ (l32 & 15)) << 4));
#pragma unroll
  for (int d = 0; d < 4; ++d)
    va[d] = (lds_char *)&lds_v[0][0] + (uint32_t)((4 * h + (i16 >> 2)) * 256 + ((d ^ (i16 >> 2)) << 6) +
                                                  32 * ((lane >> 4) & 1) + 8 * (i16 & 3));

  // scores of keys 32 kb .. + 31 of the block in K slot `slot`: lane l32's
  // query, keys 8 (e / 4) + 4 h + e % 4
  auto scores = [&](int slot, int kb, f32x16 &s) {
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bf16x8 a = *(__attribute__((address_space(3))) bf16x8 *)(ka[i] + slot * 16384 + kb * 8192);
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qf[i], s, 0, 0, 0);
    }
  };
  auto mask = [&](f32x16 &s, int key0) {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (key0 + 8 * (e >> 2) + 4 * h + (e & 3) >= nk) s[e] = -__builtin_inff();
  };
  auto max16 = [&](const f32x16 &s) {
    float r = s[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) r = __builtin_fmaxf(r, s[e]);
    return r;
  };
  auto raise_max = [&](float mx) {
    mx = half_max(mx);
    if (__any(mx > m)) {
      const float mn = __builtin_fmaxf(m, mx);
      const float f = __builtin_amdgcn_exp2f((m - mn) * scale);
      m = mn;
      l *= f;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[d][e] *= f;
    }
  };
  // probabilities 2^(scale (s - m)): summed in f32, rounded once to bf16 in
  // the B operand's order
  auto probs = [&](const f32x16 &s, bf16x8 *p) {
    const float ms = m * scale;
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      uint32_t u[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * t + 2 * i], scale, -ms));
        const float c = __builtin_amdgcn_exp2f(__builtin_fmaf(s[8 * t + 2 * i + 1], scale, -ms));
        sum[t] += a + c;
        u[i] = pack2(a, c);
      }
      __builtin_memcpy(&p[t], u, 16);
    }
    l += sum[0] + sum[1];
  };
  // O^T += V^T P^T over keys 32 kb .. + 31 of the block in V slot `slot`: the
  // A operand's key order is the probabilities' (4 h + 0..3 and 8 + 4 h + 0..3
  // of each 16)
  auto accumulate = [&](int slot, int kb, const bf16x8 *p) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        s16x4 x[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
          x[j] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) s16x4 *)(va[d] + slot * 16384 + (2 * kb + t) * 4096 + j * 2048));
        bf16x8 a;
        __builtin_memcpy(&a, x, 16);
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, p[t], o[d], 0, 0, 0);
      }
  };

  // a share without keys (masked ranges leave an element fewer blocks than the
  // plan counted): the whole workgroup returns before its first barrier
  float *po = nullptr;
  if constexpr (kSplit)
    if (split) {
      po = partial + (int64_t)unit * kPart + (32 * wave + l32) * (int64_t)kHd;
      if (nblk == 0) {
        for (int d = 0; d < 16; ++d) *reinterpret_cast<float4 *>(po + 64 * h + 4 * d) = make_float4(0.f, 0.f, 0.f, 0.f);
        if (h == 0)
          *reinterpret_cast<float2 *>(partial + (int64_t)unit * kPart + 256 * kHd + 2 * (32 * wave + l32)) =
              make_float2(-__builtin_inff(), 0.f);
        return;
      }
    }

  dma(0, 0, 0);
  block_barrier();
  if (nblk > 1) dma(1, 1, 1);
  f32x16 s0, s1;
  scores(0, 0, s0);
  int vs = 0;  // V slot of block i
  // Block i: its first half's scores are in s0.  The barrier in the middle
  // says that block i + 1 has landed and that every wave has read all of K(i)
  // and V(i - 1), whose slots block i + 2 then takes.
  auto block = [&](int i, auto kslot, bool last, bool more) {
    constexpr int ks = decltype(kslot)::v;
    bf16x8 p[2];
    if (last) mask(s0, (b0 + i) * kKeys);
    raise_max(max16(s0));
    scores(ks, 1, s1);
    probs(s0, p);
    accumulate(vs, 0, p);
    if (last) mask(s1, (b0 + i) * kKeys + 32);
    const float mx = max16(s1);
    if (!last) {
      block_barrier();
      if (more) dma(i + 2, ks, vs == 0 ? 2 : vs - 1);
    }
    raise_max(mx);
    if (!last) scores(ks ^ 1, 0, s0);
    probs(s1, p);
    accumulate(vs, 1, p);
    vs = vs == 2 ? 0 : vs + 1;
  };
  int i = 0;
  for (; i + 3 < nblk; i += 2) {
    block(i, Slot<0>{}, false, true);
    block(i + 1, Slot<1>{}, false, true);
  }
  if (i + 2 < nblk) {
    block(i, Slot<0>{}, false, true);
    block(i + 1, Slot<1>{}, false, false);
    block(i + 2, Slot<0>{}, true, false);
  } else if (i + 1 < nblk) {
    block(i, Slot<0>{}, false, false);
    block(i + 1, Slot<1>{}, true, false);
  } else {
    block(i, Slot<0>{}, true, false);
  }

  l = half_add(l);
  const bool stored = row < rows;
  if constexpr (kSplit)
    if (split) {
      // this share's unscaled O (row-major [256][128]), then (scale m, l) of its rows
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<float4 *>(po + 32 * d + 8 * g + 4 * h) =
              make_float4(o[d][4 * g], o[d][4 * g + 1], o[d][4 * g + 2], o[d][4 * g + 3]);
      if (h == 0)
        *reinterpret_cast<float2 *>(partial + (int64_t)unit * kPart + 256 * kHd + 2 * (32 * wave + l32)) =
            make_float2(m * scale, l);
      return;
    }
  const float inv = 1.f / l;
  __bf16 *orow = out + (int64_t)b * sb_out + (int64_t)row * ldo + (int64_t)head * kHd;
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      // columns 32 d + 16 g + 0..15 of this query sit in lanes l32 and l32 + 32
      // by fours; exchanged so that lane half h stores columns 8 h .. 8 h + 7
      const f32x16 &t = o[d];
      const uint32_t a0 = pack2(t[8 * g] * inv, t[8 * g + 1] * inv), a1 = pack2(t[8 * g + 2] * inv, t[8 * g + 3] * inv);
      const uint32_t c0 = pack2(t[8 * g + 4] * inv, t[8 * g + 5] * inv),
                     c1 = pack2(t[8 * g + 6] * inv, t[8 * g + 7] * inv);
      const auto x = __builtin_amdgcn_permlane32_swap(a0, c0, false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(a1, c1, false, false);
      if (stored) *reinterpret_cast<uint4 *>(orow + 32 * d + 16 * g + 8 * h) = make_uint4(x[0], y[0], x[1], y[1]);
    }
  if (lse || guard)
    row_sums(m * scale, l, keys.npad[b], stored, h == 0, lse ? lse + (int64_t)bh * rows + row : nullptr, guard);
}

// The split tiles: a row's parts, each relative to its own maximum, added in
// part order.  Half a wave per row, 4 columns a lane, every part's load in
// flight at once: bound by reading the sums (133 KB a share).
__global__ __launch_bounds__(256) void combine_kernel(const float *__restrict__ partial, int kparts, int full_tiles,
                                                      int heads, int rows, int qtiles, AttnKeys keys,
                                                      __bf16 *__restrict__ out, int64_t sb_out, int64_t ldo,
                                                      float *__restrict__ lse, unsigned int *__restrict__ guard) {
  const int t = blockIdx.y, tile = full_tiles + t;
  const int bh = tile / qtiles, qt = tile - bh * qtiles;
  const int b = bh / heads, head = bh - b * heads;
  const int rl = blockIdx.x * 8 + (threadIdx.x >> 5), l32 = threadIdx.x & 31;
  const int row = 256 * qt + rl;
  const float *p0 = partial + (int64_t)t * kparts * kPart;
  float ms[kMaxParts], ls[kMaxParts];
  float4 v[kMaxParts];
  float top = -__builtin_inff();
#pragma unroll
  for (int p = 0; p < kMaxParts; ++p)
    if (p < kparts) {
      const float2 ml = *reinterpret_cast<const float2 *>(p0 + p * kPart + 256 * kHd + 2 * rl);
      v[p] = *reinterpret_cast<const float4 *>(p0 + p * kPart + rl * kHd + 4 * l32);
      ms[p] = ml.x;
      ls[p] = ml.y;
      top = __builtin_fmaxf(top, ml.x);
    }
  float z = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int p = 0; p < kMaxParts; ++p)
    if (p < kparts) {
      const float f = ms[p] == -__builtin_inff() ? 0.f : __builtin_amdgcn_exp2f(ms[p] - top);
      z = __builtin_fmaf(f, ls[p], z);
      o.x = __builtin_fmaf(f, v[p].x, o.x);
      o.y = __builtin_fmaf(f, v[p].y, o.y);
      o.z = __builtin_fmaf(f, v[p].z, o.z);
      o.w = __builtin_fmaf(f, v[p].w, o.w);
    }
  const float inv = 1.f / z;
  const bool stored = row < rows;
  if (stored)
    *reinterpret_cast<uint2 *>(out + (int64_t)b * sb_out + (int64_t)row * ldo + (int64_t)head * kHd + 4 * l32) =
        make_uint2(pack2(o.x * inv, o.y * inv), pack2(o.z * inv, o.w * inv));
  if (lse || guard)
    row_sums(top, z, keys.npad[b], stored, l32 == 0, lse ? lse + (int64_t)bh * rows + row : nullptr, guard);
}

// How a launch of `heads` heads x `rows` rows over `keys` keys runs: waves per
// workgroup, the tiles run whole, and the key shares of the rest.  8 waves: 256
// query rows, one workgroup per CU.  4 waves: 128 rows, two per CU, each with
// its own K and V tiles.  The last, partial round of 8-wave tiles may be split
// over the keys so that it fills the CUs, at the price of the shares' f32 sums
// (written and read once) and a launch.  The estimates are in us: an 8-wave tile
// takes 1.85 per block of 64 keys, a round of 4-wave tiles 1.10 of that with
// two per CU and 0.70 with one (24 heads x 1100 tokens, 216 of them: 24.8 us
// against 32.5 with 8 waves; 32 x 1100, 288: 36.2 against 32.6; 8 x 3500, 224:
// 66), sums move at 5 TB/s.  A split has to look 10 % better, since a round that
// leaves CUs idle clocks higher: measured, whole -> split, heads x tokens: 2 x
// 4608 82 -> 41 us, 24 x 2816 140 -> 117, 40 x 1664 88 -> 80, 48 x 7145 1279 ->
// 1181, 24 x 16896 3411 -> 3145; below the line 24 x 7145 620 -> 619, 8 x 3500
// 66 -> 70, 48 x 4608 558 -> 531.
struct AttnPlan {
  int waves, full, kparts;
};
AttnPlan attn_plan(int64_t heads, int64_t rows, int64_t keys, bool may_split) {
  const int64_t t8 = heads * ((rows + 255) / 256), t4 = heads * ((rows + 127) / 128), blocks = (keys + kKeys - 1) / kKeys;
  const double tile = 1.85 * blocks;
  const int64_t full4 = t4 / (2 * kCus), rest4 = t4 % (2 * kCus);
  AttnPlan best{4, (int)t4, 1};
  double us = tile * (1.10 * full4 + (rest4 == 0 ? 0.0 : rest4 <= kCus ? 0.70 : 1.10));
  const int64_t rest8 = t8 % kCus, rounds = t8 / kCus;
  const double eight = tile * ((t8 + kCus - 1) / kCus);
  if (eight <= us) {
    us = eight;
    best = AttnPlan{8, (int)t8, 1};
  }
  us *= 0.90;
  for (int64_t kp = 2; may_split && rest8 && kp <= kMaxParts && 4 * kp <= blocks; ++kp) {
    const double t = tile * rounds + 1.85 * ((blocks + kp - 1) / kp) * ((rest8 * kp + kCus - 1) / kCus) + 5.0 +
                     2.0 * rest8 * kp * kPart * 4 / 5e6;
    if (t < us) {
      us = t;
      best = AttnPlan{8, (int)(t8 - rest8), (int)kp};
    }
  }
  return best;
}

size_t attn_scratch_bytes(const AttnPlan &p, int64_t heads, int64_t rows) {
  if (p.kparts < 2) return 0;
  const int64_t tiles = heads * ((rows + 255) / 256) - p.full;
  return (size_t)(tiles * p.kparts * kPart) * sizeof(float);
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace mq

extern "C" size_t mq_attention_scratch_size(int64_t batch, int heads, int64_t valid) {
  using namespace mq;
  if (batch <= 0 || heads <= 0 || valid <= 0) return 0;
  const int64_t nb = batch < kMaxBatch ? batch : kMaxBatch, last = batch % kMaxBatch;
  size_t n = attn_scratch_bytes(attn_plan(nb * heads, valid, valid, true), nb * heads, valid);
  if (batch > kMaxBatch && last) {
    const size_t m = attn_scratch_bytes(attn_plan(last * heads, valid, valid, true), last * heads, valid);
    n = m > n ? m : n;
  }
  return n;
}

extern "C" int mq_attention_bf16(const void *q, const void *k, const void *v, int64_t batch, int heads,
                                 int64_t l_total, int head_dim, int64_t valid, const int64_t *drop, void *out,
                                 int64_t out_batch_stride, int64_t ldo, float *lse, float *guard, void *scratch,
                                 size_t scratch_bytes, void *stream) {
  using namespace mq;
  auto invalid = [](const char *msg) { return set_error(MQ_E_INVALID, msg); };
  if (head_dim != kHd) return invalid("mq_attention_bf16: head_dim must be 128");
  if (batch < 0 || heads <= 0 || valid < 0 || valid > l_total)
    return invalid("mq_attention_bf16: negative batch, heads < 1, or valid outside 0 .. l_total");
  if (l_total > (int64_t(1) << 23) || batch > (int64_t(1) << 20) / heads)
    return invalid("mq_attention_bf16: l_total above 2^23 or more than 2^20 heads");
  if (!q || !k || !v || !out) return invalid("mq_attention_bf16: NULL pointer");
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out) || !aligned16(scratch) || ldo % 8 ||
      out_batch_stride % 8)
    return invalid("mq_attention_bf16: buffers must be 16-byte aligned, out's strides multiples of 8 elements");
  if (ldo < (int64_t)heads * kHd || out_batch_stride < 0) return invalid("mq_attention_bf16: bad out strides");
  for (int64_t b = 0; drop && b < batch; ++b)
    if (drop[2 * b] < 0 || drop[2 * b + 1] < drop[2 * b] || drop[2 * b + 1] > valid ||
        drop[2 * b + 1] - drop[2 * b] >= (valid > 0 ? valid : 1))
      return invalid("mq_attention_bf16: a masked range must lie in 0 .. valid and leave a key");
  if (batch == 0 || valid == 0) return MQ_OK;
  // a tile's rows are stored while other workgroups still read q, k and v
  const uintptr_t in_bytes = (uintptr_t)(batch * heads * l_total * kHd) * 2, o0 = reinterpret_cast<uintptr_t>(out);
  const uintptr_t o1 = o0 + (uintptr_t)((batch - 1) * out_batch_stride + (valid - 1) * ldo + heads * (int64_t)kHd) * 2;
  for (const void *in : {q, k, v}) {
    const uintptr_t i0 = reinterpret_cast<uintptr_t>(in);
    if (o0 < i0 + in_bytes && i0 < o1) return invalid("mq_attention_bf16: out lies over q, k or v");
  }
  const int64_t hsize = heads * l_total * kHd;
  const float scale = 0.12751743f;  // log2(e) / sqrt(128)
  for (int64_t b0 = 0; b0 < batch; b0 += kMaxBatch) {
    const int nb = (int)(batch - b0 < kMaxBatch ? batch - b0 : kMaxBatch);
    AttnKeys keys{};
    for (int i = 0; i < nb; ++i) {
      const int64_t lo = drop ? drop[2 * (b0 + i)] : 0, gap = drop ? drop[2 * (b0 + i) + 1] - lo : 0;
      keys.nk[i] = (int)(valid - gap);
      keys.lo[i] = (int)lo;
      keys.gap[i] = (int)gap;
      keys.npad[i] = (float)(l_total - valid + gap);
    }
    AttnPlan plan = attn_plan(nb * heads, valid, valid, scratch != nullptr);
    if (attn_scratch_bytes(plan, nb * heads, valid) > scratch_bytes) plan = attn_plan(nb * heads, valid, valid, false);
    auto launch = [&]<int W, bool kSplit>() {
      const int qtiles = (int)((valid + 32 * W - 1) / (32 * W)), tiles = nb * heads * qtiles;
      hipStream_t s = static_cast<hipStream_t>(stream);
      __bf16 *o = static_cast<__bf16 *>(out) + b0 * out_batch_stride;
      float *le = lse ? lse + b0 * heads * valid : nullptr, *part = static_cast<float *>(scratch);
      unsigned int *gu = reinterpret_cast<unsigned int *>(guard);
      hipLaunchKernelGGL((attention_kernel<W, kSplit>), dim3((unsigned)(plan.full + (tiles - plan.full) * plan.kparts)),
                         dim3(64 * W), 0, s, static_cast<const __bf16 *>(q) + b0 * hsize,
                         static_cast<const __bf16 *>(k) + b0 * hsize, static_cast<const __bf16 *>(v) + b0 * hsize, heads,
                         l_total, (int)valid, qtiles, keys, scale, o, out_batch_stride, ldo, le, gu, plan.full,
                         plan.kparts, part);
      if constexpr (kSplit)
        hipLaunchKernelGGL(combine_kernel, dim3(32, (unsigned)(tiles - plan.full)), dim3(256), 0, s, part,
                           plan.kparts, plan.full, heads, (int)valid, qtiles, keys, o, out_batch_stride, ldo, le, gu);
    };
    if (plan.kparts > 1) launch.template operator()<8, true>();
    else if (plan.waves == 8) launch.template operator()<8, false>();
    else launch.template operator()<4, false>();
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(MQ_E_HIP, hipGetErrorString(e));
  }
  return MQ_OK;
}
