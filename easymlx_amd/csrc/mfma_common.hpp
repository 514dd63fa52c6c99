// Shared pieces of the MFMA attention kernels over any cache (decode_mfma.hpp,
// prefill_mfma.hpp): operand types, the probability split, and the exact fallback for
// non-finite rows.
#pragma once

#include "common.hpp"
#include "decode_affine.hpp"
#include "decode_split.hpp"

namespace emx {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef h16 h16x2 __attribute__((ext_vector_type(2)));

// Cache kinds: the element type of the pages, and of the queries and outputs.
struct KvF16 {
  typedef h16 QT;       // queries, outputs
  typedef h16x8 Op;     // one lane's MFMA operand
  typedef h16 ET;       // cache element
  static constexpr int kParts = 2;  // 16-bit parts of a probability
  static constexpr bool kFp8 = false, kAffine = false;
};
struct KvBF16 {
  typedef uint16_t QT;
  typedef bf16x8 Op;
  typedef uint16_t ET;
  static constexpr int kParts = 3;
  static constexpr bool kFp8 = false, kAffine = false;
};
struct KvFp8 {
  typedef h16 QT;
  typedef h16x8 Op;
  typedef uint8_t ET;
  static constexpr int kParts = 2;
  static constexpr bool kFp8 = true, kAffine = false;
};
// Affine pages: codes enter the MFMA as exact fp16 sub-normals, at 4 bits as code * 2^-18
// and at 8 bits as code * 2^-24.  The matrix unit aligns a sub-normal's products as if it
// had the smallest normal exponent, so what the code leaves of the 10 mantissa bits is lost
// from the sum's precision: 4-bit codes at 2^-24 put scores off by up to 3e-5 where the fp32
// bias and scale terms leave 3e-6.
template <int BITS, int GS>
struct KvAffine {
  typedef h16 QT;
  typedef h16x8 Op;
  typedef uint8_t ET;
  static constexpr int kParts = 2;
  static constexpr bool kFp8 = false, kAffine = true;
  static constexpr int kBits = BITS, kGS = GS;
  static constexpr int kCodeExp = BITS == 4 ? 18 : 24;
};

// One word of 4-bit codes -> code * 2^-18, in unpack4's element order.
__device__ __forceinline__ h16x8 unpack4_high(const uint32_t w) {
  return as_h8((w << 6) & 0x03C003C0u, (w << 2) & 0x03C003C0u, (w >> 2) & 0x03C003C0u, (w >> 6) & 0x03C003C0u);
}

// The element loader of a call's cache (paged_generic.hpp).
template <class C>
__device__ __forceinline__ auto kv_loader(const DecodeArgs& a, const int D) {
  if constexpr (C::kAffine)
    return AffineKV<C::kBits>{a.kc, a.ks, a.kb, a.vc, a.vs, a.vb, a.Hkv, D, a.bs, C::kGS};
  else if constexpr (C::kFp8)
    return Fp8KV{reinterpret_cast<const uint8_t*>(a.kc), reinterpret_cast<const uint8_t*>(a.vc), a.kps, a.vps, a.Hkv,
                 D, a.bs};
  else if constexpr (__is_same(typename C::QT, h16))
    return DenseKV<F16>{reinterpret_cast<const h16*>(a.kc), reinterpret_cast<const h16*>(a.vc), a.Hkv, D, a.bs};
  else
    return DenseKV<BF16>{reinterpret_cast<const uint16_t*>(a.kc), reinterpret_cast<const uint16_t*>(a.vc), a.Hkv, D,
                         a.bs};
}

__device__ __forceinline__ f32x4 mfma_op(const h16x8 a, const h16x8 b, const f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_op(const bf16x8 a, const bf16x8 b, const f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Probabilities enter the matrix unit as a sum of 16-bit parts, so that the
// products with V keep the fp32 probability: fp16 in two parts (11 + 11 bits of
// the 24; the exponent offset kPBias lifts p out of fp16's sub-normals), bf16
// in three (8 + 8 + 8, exact).
constexpr float kPBias = 8.f;  // p = 2^(x - m + kPBias)
constexpr float kPScale = 256.f;  // 2^kPBias

__device__ __forceinline__ void split_p(const float (&x)[8], h16x8 (&p)[2]) {
  typedef float f32x2v __attribute__((ext_vector_type(2)));
  uint32_t hi[4], lo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const h16x2 h = __builtin_convertvector(f32x2v{x[2 * i], x[2 * i + 1]}, h16x2);
    // (as fused multiply-adds: one mixed-precision instruction each)
    const h16x2 l = __builtin_convertvector(
        f32x2v{__builtin_fmaf((float)h[0], -1.f, x[2 * i]), __builtin_fmaf((float)h[1], -1.f, x[2 * i + 1])}, h16x2);
    hi[i] = __builtin_bit_cast(uint32_t, h);
    lo[i] = __builtin_bit_cast(uint32_t, l);
  }
  p[0] = as_h8(hi[0], hi[1], hi[2], hi[3]);
  p[1] = as_h8(lo[0], lo[1], lo[2], lo[3]);
}
__device__ __forceinline__ void split_p(const float (&x)[8], bf16x8 (&p)[3]) {
  uint32_t w[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t a = __float_as_uint(x[2 * i]), b = __float_as_uint(x[2 * i + 1]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      w[k][i] = __builtin_amdgcn_perm(b, a, 0x07060302u);  // the top halves
      if (k < 2) {
        a = __float_as_uint(__uint_as_float(a) - __uint_as_float(a & 0xFFFF0000u));
        b = __float_as_uint(__uint_as_float(b) - __uint_as_float(b & 0xFFFF0000u));
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) p[k] = __builtin_bit_cast(bf16x8, u32x4{w[k][0], w[k][1], w[k][2], w[k][3]});
}

// page of position p for pages of bs tokens, inv = ceil(2^32 / bs) (bs >= 2):
// exact while p * bs < 2^32, which the host checks for the whole table.
__device__ __forceinline__ int page_of(const int p, const uint32_t inv) { return (int)__umulhi((uint32_t)p, inv); }

// One query row against keys [k0, k1) in fp32 on one wave: the rows whose MFMA result is not
// finite are computed again here.  On the matrix unit a masked key still enters its tile's
// product with p = 0, and 0 * inf (an infinity or NaN in a masked or stale value, or in the low
// part of a visible one) would make NaN of what these arithmetic rules leave finite or infinite.
// 64 keys at a time, a key to a lane for the scores, then lane L holds dims L + 64 i and every
// key's page is read in groups of 8 (one page each).  m, l: maximum (base 2) and sum of the
// probabilities.  With an infinite value in one page: a context of 1024 tokens, fp16, D 64, 26 us (a
// key at a time, over the merged row: 812), batch 32 of 512 .. 4096 tokens, bf16, 289 (2000), four
// 512-token chunks beside 28 rows 7500 (34700; 18500 on paged_generic, finite or not).
template <class C, int D>
__device__ void attend_row(const DecodeArgs& a, const int s, const int kvh, const typename C::QT* q, const int k0,
                           const int k1, float& m, float& l, float (&acc)[D / 64], const int lane) {
  constexpr int N = D / 64;
  const auto kv = kv_loader<C>(a, D);
  float qv[N];
  m = -INFINITY;
  l = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    qv[i] = to_f32(q[lane + 64 * i]);
    acc[i] = 0.f;
  }
#pragma unroll 1
  for (int base = k0 & ~63; base < k1; base += 64) {
    const int k = base + lane;
    const int blk = k >= k0 && k < k1 ? a.block_tables[(size_t)s * a.max_blocks + k / a.bs] : -1;
    const bool ok = (unsigned)blk < (unsigned)a.nb;
    const uint64_t okm = __ballot(ok);
    float x = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll 1
      for (int d = 0; d < 64; d += 32) {
        float kd[32] = {};
        if (ok) key32(kv, blk, k % a.bs, kvh, 64 * i + d, kd);
#pragma unroll
        for (int j = 0; j < 32; ++j)
          x = fmaf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(qv[i]), d + j)), kd[j], x);
      }
    x = ok ? x * a.scale_log2 : -INFINITY;
    const float mn = fmaxf(m, wave_max(x));
    const float p = ok && (mn != -INFINITY || x != x) ? exp2f(x - mn) : 0.f;
    const float al = m == mn ? 1.f : exp2f(m - mn);
    l = l * al + wave_sum(p);
    m = mn;
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] *= al;
#pragma unroll 1
    for (int t = 0; t < 64; t += 8) {
      const uint32_t live = (uint32_t)(okm >> t) & 0xFFu;
      if (!live) continue;
      const int b = __builtin_amdgcn_readlane(blk, t + __builtin_ctz(live));
#pragma unroll
      for (int i = 0; i < N; ++i) {
        float v[8];
        val8(kv, b, (base + t) % a.bs, kvh, lane + 64 * i, v);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float pj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), t + j));
          acc[i] = (live >> j) & 1u ? fmaf(pj, v[j], acc[i]) : acc[i];
        }
      }
    }
  }
}

__device__ __forceinline__ bool not_finite(const float x) {
  return (__float_as_uint(x) & 0x7F800000u) == 0x7F800000u;
}

}  // namespace emx
