// MFMA attention kernels over token-major caches and their launchers.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "decode_mfma.hpp"
#include "mfma_launch.hpp"

namespace emx {
namespace {

constexpr int kDecodeMfmaWGs = 512;  // persistent grid: two workgroups per compute unit

bool head_ok(int D) { return D == 64 || D == 128 || D == 256; }
int head_chunk(int Hq, int Hkv) { return std::min(Hq / Hkv, 16); }
int head_chunks(int Hq, int Hkv) { return (Hq / Hkv + head_chunk(Hq, Hkv) - 1) / head_chunk(Hq, Hkv); }
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

typedef void (*DecodeMfmaFn)(DecodeMfmaArgs);

template <class C>
DecodeMfmaFn pick_decode(int D) {
  return D == 64 ? decode_mfma<C, 64> : D == 128 ? decode_mfma<C, 128> : decode_mfma<C, 256>;
}

}  // namespace

bool token_major_ok(const TokenMajorCall& c) {
  // page_of() is exact for power-of-two pages, and for the others while position * bs < 2^32
  const bool pages = c.bs % 8 == 0 && ((c.bs & (c.bs - 1)) == 0 || (long long)c.max_blocks * c.bs * c.bs < (1LL << 32));
  return head_ok(c.D) && pages && (long long)c.max_blocks * c.bs < (1LL << 31) && c.S <= kMaxSeqs &&
         (long)c.S * c.Hkv * head_chunks(c.Hq, c.Hkv) <= kMaxUnits && aligned16(c.q) && aligned16(c.out) &&
         aligned16(c.k) && aligned16(c.v);
}

size_t decode_mfma_partial_bytes(int S, int Hq, int Hkv, int D) {
  if (!head_ok(D)) return 0;
  const size_t slots = kDecodeMfmaWGs + (size_t)S * Hkv * head_chunks(Hq, Hkv);
  return slots * head_chunk(Hq, Hkv) * (D + 2) * sizeof(float);
}

static DecodeMfmaArgs decode_args(const TokenMajorCall& c, int* ws_cnt, float* partials) {
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
  a.nt = kDecodeMfmaNT;
  A.hc = head_chunk(c.Hq, c.Hkv);
  A.nhc = head_chunks(c.Hq, c.Hkv);
  A.inv_bs = (uint32_t)(((1ULL << 32) + c.bs - 1) / c.bs);
  a.ws_cnt = ws_cnt;
  a.ws_o = partials;
  a.ws_ml = partials + (kDecodeMfmaWGs + (size_t)c.S * c.Hkv * A.nhc) * A.hc * c.D;
  return A;
}

void launch_decode_mfma(const TokenMajorCall& c, int* ws_cnt, float* partials, hipStream_t st) {
  const DecodeMfmaFn fn = c.kind == KvKind::f16    ? pick_decode<KvF16>(c.D)
                          : c.kind == KvKind::bf16 ? pick_decode<KvBF16>(c.D)
                                                   : pick_decode<KvFp8>(c.D);
  hipLaunchKernelGGL(fn, dim3(kDecodeMfmaWGs), dim3(256), 0, st, decode_args(c, ws_cnt, partials));
}

}  // namespace emx
