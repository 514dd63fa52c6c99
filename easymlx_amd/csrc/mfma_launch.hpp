// Launchers of the MFMA kernels over any cache (emx_mfma.hip, a translation unit of its
// own), called by the C entry points in emx_attn.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace emx {

enum class KvKind { f16, bf16, fp8, affine };

// One attention call, as the entry points receive it.
struct MfmaCall {
  KvKind kind;
  const void* q;
  void* out;
  const void* k;
  const void* v;
  const float *kps, *vps;        // FP8: scale per page
  const void *ks, *kb, *vs, *vb; // affine pages: scales and biases, bits, group size
  int bits, gs;
  const int32_t *block_tables, *kv_lens, *qsl;
  int T, S, Hq, Hkv, D, bs, nb, max_blocks;
  float scale_log2;
  int window;
};

// Shapes the kernels take: head_dim 64, 128 or 256 (whole MFMA k-slices and a power of
// two of dims per lane), pages of a multiple of 8 tokens (a quad of tokens in one page);
// over affine pages group 64 or 128 and pages that hold whole value tiles or are a power
// of two, of 16 tokens or more at 4 bits (the tokens of a lane's value words in one page);
// 16-byte aligned tensors, tables within the kernels' limits.  They were the faster side
// at every size tried within these (decode_mfma.hpp has figures).
bool mfma_ok(const MfmaCall& c);

// Bytes the decode's partials take after the workspace's fixed region (0: shape not taken).
size_t decode_mfma_partial_bytes(int S, int Hq, int Hkv, int D);
// ws_cnt: the workspace's unit counters; partials: decode_mfma_partial_bytes bytes.
void launch_decode_mfma(const MfmaCall& c, int* ws_cnt, float* partials, hipStream_t st);

// A ragged call (qsl given): rows of longer queries, and single-token rows beside them.
// ws_cnt null (no workspace): every row as a query tile, nothing cut.  part null: tiles
// are not cut; else mixed_mfma_part_bytes bytes (ws_part_cnt: their counters).
bool mixed_mfma_ok(const MfmaCall& c);
size_t mixed_mfma_part_bytes(int T, int S, int Hq, int Hkv, int D);
void launch_mixed_mfma(const MfmaCall& c, int* ws_cnt, float* partials, int* ws_part_cnt, float* part,
                       hipStream_t st);

}  // namespace emx
