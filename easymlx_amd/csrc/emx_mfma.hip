// MFMA attention kernels over any cache (token-major and affine pages) and their launchers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "decode_mfma.hpp"
#include "mfma_launch.hpp"
#include "prefill_mfma.hpp"

namespace emx {
namespace {

constexpr int kDecodeMfmaWGs = 512;  // persistent grid: two workgroups per compute unit ..
int decode_wgs(int D) { return D == 256 ? kDecodeMfmaWGs / 2 : kDecodeMfmaWGs; }  // .. or the one that fits

bool head_ok(int D) { return D == 64 || D == 128 || D == 256; }
int head_chunk(int Hq, int Hkv) { return std::min(Hq / Hkv, 16); }
int head_chunks(int Hq, int Hkv) { return (Hq / Hkv + head_chunk(Hq, Hkv) - 1) / head_chunk(Hq, Hkv); }
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

typedef void (*DecodeMfmaFn)(DecodeMfmaArgs);

template <class C>
DecodeMfmaFn pick_decode(int D) {
  return D == 64 ? decode_mfma<C, 64> : D == 128 ? decode_mfma<C, 128> : decode_mfma<C, 256>;
}
template <int BITS>
DecodeMfmaFn pick_decode_affine(int D, int gs) {
  if (gs == 64) return pick_decode<KvAffine<BITS, 64>>(D);
  return D == 128 ? decode_mfma<KvAffine<BITS, 128>, 128> : decode_mfma<KvAffine<BITS, 128>, 256>;
}
DecodeMfmaFn decode_fn(const MfmaCall& c) {
  switch (c.kind) {
    case KvKind::f16: return pick_decode<KvF16>(c.D);
    case KvKind::bf16: return pick_decode<KvBF16>(c.D);
    case KvKind::fp8: return pick_decode<KvFp8>(c.D);
    case KvKind::affine: break;
  }
  return c.bits == 4 ? pick_decode_affine<4>(c.D, c.gs) : pick_decode_affine<8>(c.D, c.gs);
}

}  // namespace

bool mfma_ok(const MfmaCall& c) {
  // page_of() is exact for power-of-two pages, and for the others while position * bs < 2^32
  const bool pages = c.bs % 8 == 0 && ((c.bs & (c.bs - 1)) == 0 || (long long)c.max_blocks * c.bs * c.bs < (1LL << 32));
  if (c.kind == KvKind::affine) {
    const int tile = 256 / c.bits;
    if ((c.gs != 64 && c.gs != 128) || c.D % c.gs || c.bs % (tile / 4) || (c.bs % tile && (c.bs & (c.bs - 1))) ||
        !aligned16(c.ks) || !aligned16(c.kb) || !aligned16(c.vs) || !aligned16(c.vb))
      return false;
  }
  const long long units = (long long)c.S * c.Hkv * head_chunks(c.Hq, c.Hkv);
  return head_ok(c.D) && pages && (long long)c.max_blocks * c.bs < (1LL << 31) && c.S <= kMaxSeqs &&
         units <= kMaxUnits && units * ((long long)c.max_blocks * c.bs / 128 + 2) < (1LL << 31) && aligned16(c.q) && aligned16(c.out) &&
         aligned16(c.k) && aligned16(c.v);
}

size_t decode_mfma_partial_bytes(int S, int Hq, int Hkv, int D) {
  if (!head_ok(D)) return 0;
  const size_t slots = kDecodeMfmaWGs + (size_t)S * Hkv * head_chunks(Hq, Hkv);
  return slots * head_chunk(Hq, Hkv) * (D + 2) * sizeof(float);
}

static DecodeMfmaArgs decode_args(const MfmaCall& c, int* ws_cnt, float* partials) {
  DecodeMfmaArgs A{};
  DecodeArgs& a = A.d;
  a.q = static_cast<const h16*>(c.q);
  a.kc = static_cast<const uint32_t*>(c.k);
  a.vc = static_cast<const uint32_t*>(c.v);
  a.kps = c.kps;
  a.vps = c.vps;
  a.block_tables = c.block_tables;
  a.kv_lens = c.kv_lens;
  a.qsl = c.qsl;
  a.out = static_cast<h16*>(c.out);
  a.S = c.S;
  a.Hq = c.Hq;
  a.Hkv = c.Hkv;
  a.bs = c.bs;
  a.nb = c.nb;
  a.max_blocks = c.max_blocks;
  a.scale_log2 = c.scale_log2;
  a.window = c.window;
  a.ks = static_cast<const h16*>(c.ks);
  a.kb = static_cast<const h16*>(c.kb);
  a.vs = static_cast<const h16*>(c.vs);
  a.vb = static_cast<const h16*>(c.vb);
  a.nt = c.kind == KvKind::affine ? 4 * (256 / c.bits) : 128;  // DecodeMfmaCfg::NT
  A.hc = head_chunk(c.Hq, c.Hkv);
  A.nhc = head_chunks(c.Hq, c.Hkv);
  A.inv_bs = (uint32_t)(((1ULL << 32) + c.bs - 1) / c.bs);
  A.T = c.T;
  a.ws_cnt = ws_cnt;
  a.ws_o = partials;
  a.ws_ml = partials + (kDecodeMfmaWGs + (size_t)c.S * c.Hkv * A.nhc) * A.hc * c.D;
  return A;
}

void launch_decode_mfma(const MfmaCall& c, int* ws_cnt, float* partials, hipStream_t st) {
  hipLaunchKernelGGL(decode_fn(c), dim3(decode_wgs(c.D)), dim3(256), 0, st, decode_args(c, ws_cnt, partials));
}

namespace {

// Query columns per wave: 16 CT.  More columns read each K and V operand from LDS fewer
// times; at D = 256 the accumulator of 32 columns leaves one wave per SIMD.
constexpr int ct_of(int D) { return D > 128 ? 1 : 2; }
// Most query tiles per kv head: a sequence of q >= min_q query tokens has at most q / tokb + 1.
long tile_items(int T, int S, int tokb, int min_q) { return (long)(T + tokb - 1) / tokb + std::min(S, T / min_q); }
// Fewest: all but one token of a sequence at most are in tiles.
long tile_items_least(int T, int S, int tokb) { return (std::max(T - S, 0) + tokb - 1) / tokb; }

typedef void (*MixedFn)(PrefillMfmaArgs, DecodeMfmaArgs, int);

template <class C>
MixedFn pick_mixed(int D) {
  return D == 64 ? mixed_mfma<C, 64, ct_of(64)> : D == 128 ? mixed_mfma<C, 128, ct_of(128)>
                                                            : mixed_mfma<C, 256, ct_of(256)>;
}
template <int BITS>
MixedFn pick_mixed_affine(int D, int gs) {
  if (gs == 64) return pick_mixed<KvAffine<BITS, 64>>(D);
  return D == 128 ? mixed_mfma<KvAffine<BITS, 128>, 128, ct_of(128)>
                  : mixed_mfma<KvAffine<BITS, 128>, 256, ct_of(256)>;
}
MixedFn mixed_fn(const MfmaCall& c) {
  switch (c.kind) {
    case KvKind::f16: return pick_mixed<KvF16>(c.D);
    case KvKind::bf16: return pick_mixed<KvBF16>(c.D);
    case KvKind::fp8: return pick_mixed<KvFp8>(c.D);
    case KvKind::affine: break;
  }
  return c.bits == 4 ? pick_mixed_affine<4>(c.D, c.gs) : pick_mixed_affine<8>(c.D, c.gs);
}

}  // namespace

bool mixed_mfma_ok(const MfmaCall& c) {
  return mfma_ok(c) && c.qsl && c.Hq / c.Hkv <= 64 * ct_of(c.D) && (long long)c.nb * c.bs * (c.kind == KvKind::affine ? c.Hkv : 1) < (1LL << 31);
}

size_t mixed_mfma_part_bytes(int T, int S, int Hq, int Hkv, int D) {
  const int hg = Hq / Hkv;
  if (!head_ok(D) || hg > 64 * ct_of(D)) return 0;
  const int tokb = 64 * ct_of(D) / hg;
  const long least = tile_items_least(T, S, tokb) * Hkv, most = tile_items(T, S, tokb, 2) * Hkv;
  const int parts = MfmaRule::most_parts(least, INFINITY);
  if (parts == 1) return 0;
  // (tile, part) pairs: the kernel counts the tiles, anything between the two bounds
  const long slots = std::min<long>(most * parts, 2 * kPrefillCutTiles);
  return (size_t)slots * (4 * (ct_of(D) * (D / 16) + 1) * 1024);
}

void launch_mixed_mfma(const MfmaCall& c, int* ws_cnt, float* partials, int* ws_part_cnt, float* part,
                       hipStream_t st) {
  const DecodeMfmaArgs d = decode_args(c, ws_cnt, partials);
  PrefillMfmaArgs p{};
  p.d = d.d;
  p.inv_bs = d.inv_bs;
  p.min_q = ws_cnt ? 2 : 1;
  p.tokb = 64 * ct_of(c.D) / (c.Hq / c.Hkv);
  const long items = tile_items(c.T, c.S, p.tokb, p.min_q);
  p.T = c.T;
  p.items = (int)items;
  p.places = part ? prefill_places(tile_items_least(c.T, c.S, p.tokb) * c.Hkv) : 1;
  p.ws_cnt = ws_part_cnt;
  p.ws_part = part;
  // Decode workgroups by the decode rows' share of the step (at most S of the T rows), so that
  // their streams end with the matrix work.  512-token chunks beside 28 rows: 16 bits 176 / 121 /
  // 120 / 125 / 128 us at a factor of 10 / 30 / 40 / 70 / 100, FP8 190 / 160 / 139 / 137 at
  // 12 / 20 / 35 / 50, 8-bit pages (20 rows beside two chunks) 74 / 41 / 38 at 5 / 20 / 35.
  const double share = 45.0 * c.S / std::max(1, c.T - c.S) * c.Hkv / c.Hq;
  const int ndec = ws_cnt ? std::clamp((int)(1024.0 * share), 64, kDecodeMfmaWGs) & ~7 : 0;
  hipLaunchKernelGGL(mixed_fn(c), dim3((unsigned)(items * c.Hkv * p.places + ndec)), dim3(256), 0, st, p, d, ndec);
}

}  // namespace emx
