// Ragged / causal paged attention (sequences with more than one query token), head_dim
// 64, 128 or 256, any GQA ratio up to 128, over token-major caches [nb, bs, Hkv, D]
// (unquantized fp16 / bf16, FP8 E4M3 with one fp32 scale per page; pages of a multiple of
// 8 tokens) and over affine pages.  MFMA.
//
// Replaces the ragged / causal Metal kernel of the reference
// (lib/python/easymlx/operations/kernels/unified_attention.py:290-465, causal limit
// :357-361, sliding window :369-376, FP8 :776-1102) and the single-sequence causal path
// (page_attention.py:84-133).
//
// Work: one workgroup (4 waves) per (sequence, kv head, tile of COLS / HG query tokens);
// a wave owns 16 CT query columns = (token, head) pairs, head fastest.  Keys are walked
// NT at a time up to the tile's causal limit.  A step's K and V rows are loaded once per
// workgroup, 16 bytes per lane and whole rows per 16 lanes, a step ahead into registers
// (their page ids another step ahead), and go to LDS token-major as 16-bit values (FP8:
// dec(code) * 2^-8, exact).  Each wave, on v_mfma 16x16x32:
//   S^T : A = K rows (16 keys), B = queries;
//   online softmax per column (base 2, fp32; the reference maximum moves only when a
//   score passes it by 2^kLazyMax, so the accumulator is rescaled rarely);
//   O^T += V^T P^T : A = V^T by the transposing LDS read (ds_read_b64_tr_b16: 4 tokens of
//   16 dims per 16 lanes), B = the probabilities of the lane's own keys in two fp16 or
//   three bf16 parts.
// Affine pages: K codes go to LDS as exact fp16 sub-normals and accumulate per
// quantization group, the (key, group) scale applied in fp32 and the bias term on the matrix
// unit (as in prefill_affine.hpp); value codes stay exact too, dim-major, the value scale
// entering the probability before it is split and sum p * v_bias kept in fp32 (the 128-wide
// prefill_affine rounds scale * code + bias to fp16 instead).  Keys sit in LDS in the order
// in which a lane's scores are then eight consecutive keys, those of its value operand.
// Tiles of many keys are cut into parts (MfmaRule), merged in
// part order by the wave that arrives last (as in prefill_affine.hpp).
//
// Bound by the matrix and vector units together (the probability parts double the PV
// products of fp16, triple those of bf16).  It took over from paged_generic, one wave per
// (token, kv head) on the VALU: four 512-token chunks beside 28 decode rows, bf16, D 128,
// pages of 16: 20.8 ms -> 110 us; a 1531-token prompt, fp16, D 256, window 700: 9.6 ms ->
// 51 us; three 203-token chunks beside 9 rows, 4-bit pages of 16: 5.47 ms -> 52 us.  Over 4-bit
// pages of 128 tokens prefill_affine (value codes dequantized to fp16 once per workgroup)
// remains the faster kernel where it applies.
#pragma once

#include "decode_mfma.hpp"
#include "prefill_affine.hpp"

namespace emx {

// As PrefillRule (prefill_affine.hpp): a third part only where all of three fit the 512 places of
// the chip.  3 / 2 / 1 parts, bf16 pages of 16, us: 16 tiles (a 64-token chunk after 9000) 110 / 156 /
// 292, 88 (330 tokens) 162 / 220 / 422, 256 (a 1000-token prompt) 38 / 39 / 57, 352 (2 x 700 beside
// 60 rows) 137 / 133 / 154, 512 (four 512-token chunks) 132 / 119 / 126, (beside 64 rows) 166 / 168 /
// 187, 656 (2 x 1300) 126 / 126 / 114, 752 (a 3000-token prompt) 167 / 163 / 168, 1024 (4 x 1000)
// 116 / 111 / 111, (eight chunks after up to 8192) 647 / 643 / 796, 1504 217 / 214 / 192, 2048
// 331 / 320 / 281; 4-bit pages of 16: 512 beside 28 rows 171 / 151 / 157, 1280 779 / 827 / 929.
constexpr int kTiles3 = 170;
static_assert(3 * kTiles3 <= 2 * kPrefillCutTiles, "the workspace holds either");
struct MfmaRule {
  static constexpr int kFew = kTiles3;
  static __host__ __device__ constexpr int most_parts(long tiles, float keys) {
    return tiles <= kTiles3 ? 3
           : tiles <= kPrefillFewTiles || (tiles <= kPrefillCutTiles && keys >= kPrefillLongKeys) ? 2
                                                                                                   : 1;
  }
};

struct PrefillMfmaArgs {
  DecodeArgs d;     // kc / vc: the caches; nt, ws_* unused
  uint32_t inv_bs;  // ceil(2^32 / bs)
  int min_q;        // sequences with fewer query tokens are not taken
  int tokb;         // query tokens per tile: columns / HG
  int T;            // query rows
  int items;        // tiles per kv head the grid has room for
  int places;       // workgroups the grid has for a tile (prefill_places), 1: no workspace for parts
  int* ws_cnt;      // [tiles * Hkv * 4], zero before and after every launch
  float* ws_part;   // [tiles * Hkv][parts][part bytes]
};

template <class C, int D, int CT>
struct PrefillMfmaCfg {
  static constexpr int EB = sizeof(typename C::ET);
  static constexpr int NT = D > 128 ? 32 : 64;        // keys per step
  static constexpr int KS = D / 32;                   // QK^T k-slices
  static constexpr int SB = D / 16;                   // PV dim sub-tiles
  static constexpr int COLS = 64 * CT;                // query columns per workgroup
  static constexpr int KSTR = D + 8;                  // halves per K row in LDS
  static constexpr int VSTR = D + 16;                 // halves per V row: 8 banks further each (D * 2 is 0 mod 256)
  static constexpr int PR = D * EB / 16;              // 16-byte pieces per row
  static constexpr int RP = 256 / PR;                 // rows per pass of the workgroup
  static constexpr int NP = NT / RP;                  // pieces per thread and step, of K and of V
  static constexpr int PARTB = 4 * (CT * SB + 1) * 64 * 16;  // bytes of one part's state
};

template <int BITS, int GS, int D, int CT>
struct PrefillMfmaCfg<KvAffine<BITS, GS>, D, CT> {
  static constexpr int NT = D > 128 ? 32 : 64, KS = D / 32, SB = D / 16, COLS = 64 * CT, G = D / GS;
  static constexpr int KSTR = D + 8;                    // halves per K row
  static constexpr int VSTR = NT + 8;                   // halves per V dim: 16 dims' reads on distinct banks
  static constexpr int RBK = D * BITS / 8;              // bytes of a key's codes
  static constexpr int PR = RBK / 16;                   // 16-byte pieces of them
  static constexpr int NPK = NT * PR;                   // K pieces of a step
  static constexpr int NP = (NPK + 255) / 256;
  static constexpr int UT = 64 / BITS, U = NT / UT;     // V units: 8 bytes, UT tokens of one dim
  static constexpr int NPV = D * U / 256;               // V units per thread
  static constexpr int NPS = 4 * G * NT / 8;            // 16-byte scale pieces of a step
  static constexpr int PARTB = 4 * (CT * SB + 1) * 64 * 16;
  static_assert(NPS <= 64 && D * U % 256 == 0, "one scale piece per lane, whole V units per thread");
};

// Where key k of a step sits in the K rows and scale arrays over affine pages: position
// 16 t + 4 q + e of its 32-key block for k = 8 q + 4 t + e.
__device__ __forceinline__ constexpr int affine_pos(int k) {
  return (k & ~31) | ((k & 4) << 2) | ((k & 24) >> 1) | (k & 3);
}

// 16-byte piece of the cache -> LDS row position, as 16-bit operand values.
template <class C>
__device__ __forceinline__ void put_piece(uint16_t* dst, const u32x4 x) {
  if constexpr (C::kFp8) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
      *reinterpret_cast<h16x8*>(dst + 8 * e) =
          as_h8(e4m3x2_to_h16x2(__builtin_amdgcn_perm(0u, x[2 * e], 0x0C010C00u)),
                e4m3x2_to_h16x2(__builtin_amdgcn_perm(0u, x[2 * e], 0x0C030C02u)),
                e4m3x2_to_h16x2(__builtin_amdgcn_perm(0u, x[2 * e + 1], 0x0C010C00u)),
                e4m3x2_to_h16x2(__builtin_amdgcn_perm(0u, x[2 * e + 1], 0x0C030C02u)));
  } else {
    *reinterpret_cast<u32x4*>(dst) = x;
  }
}

// Lane (i, jj): element i of the 16 dims at column d0 of rows row0 + 4 jj .. + 3.
__device__ __forceinline__ u32x2 read_tr(const uint16_t* v, const int stride, const int row0, const int d0,
                                         const int i, const int jj) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* lds4;
  const uint16_t* p = v + (row0 + 4 * jj + (i >> 2)) * stride + d0 + 4 * (i & 3);
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)p));
}

// Query rows that no sequence holds (before query_start_loc[0], a padded call's rows past the
// last entry) are zeros, as the reference's (unified_attention.py:341-344).  Written by the grid's
// workgroups past the last tile, `idx` of `n` (there are some whenever there are such rows: tile_items
// rounds the call's rows up to tiles, and counts one tile more for every sequence that can have tiles).
template <class QT>
__device__ void zero_other_rows(const DecodeArgs& a, const int T, const int D, const int idx, const int n) {
  const int lo = min(max(a.qsl[0], 0), T), hi = min(max(a.qsl[a.S], lo), T);
  const int per_row = a.Hq * D / 8;
  const size_t total = (size_t)(lo + T - hi) * per_row;
  for (size_t i = (size_t)idx * 256 + threadIdx.x; i < total; i += (size_t)n * 256) {
    const size_t r = i / per_row;
    reinterpret_cast<u32x4*>(a.out)[(r < lo ? r : r - lo + hi) * per_row + i % per_row] = u32x4{0u, 0u, 0u, 0u};
  }
}

template <class C, int D, int CT>
__device__ __forceinline__ void prefill_mfma_body(const PrefillMfmaArgs& A, const int bid) {
  using P = PrefillMfmaCfg<C, D, CT>;
  typedef typename C::Op Op;
  typedef typename C::QT QT;
  const DecodeArgs& a = A.d;
  constexpr int NT = P::NT;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, jj = lane >> 4;

  // LDS, carved from the shared arena
  constexpr bool AFF = C::kAffine;
  constexpr int G = [] {
    if constexpr (C::kAffine) return P::G;
    return 1;
  }();
  constexpr int oTcum = 0, oWred = lds_next(oTcum, 4 * (kMaxSeqs + 1)), oKe = lds_next(oWred, 48);
  constexpr int oVe = lds_next(oKe, 2 * NT * P::KSTR), oKsf = lds_next(oVe, 2 * (AFF ? D : NT) * P::VSTR);
  constexpr int oVsf = lds_next(oKsf, 4 * G * NT), oVbf = lds_next(oVsf, 4 * G * NT);
  constexpr int oKbe = lds_next(oVbf, AFF ? 4 * G * NT : 0), oEnd = lds_next(oKbe, AFF ? 16 * NT : 0);
  static_assert(oEnd <= kArenaBytes, "LDS arena too small");
  int(&tcum)[kMaxSeqs + 1] = lds_at<int[kMaxSeqs + 1]>(oTcum);
  int(&wred)[12] = lds_at<int[12]>(oWred);
  uint16_t* ke = &lds_at<uint16_t>(oKe);  // [key][KSTR]
  uint16_t* ve = &lds_at<uint16_t>(oVe);  // [key][VSTR]; affine: [dim][VSTR]
  float* ksf = &lds_at<float>(oKsf);      // key scale of each key; affine: [group][NT], * 2^kCodeExp
  float* vsf = &lds_at<float>(oVsf);      // value scales / 2^vexp
  float* vbf = &lds_at<float>(oVbf);      // affine: value biases
  h16* kbe = &lds_at<h16>(oKbe);          // affine: bias operand rows, key bias of group g at 2 g, 2 g + 1

  // ---- work item
  const int kvh = bid % a.Hkv;
  const TileItem ti = a.S <= 64 ? tile_item64<MfmaRule>(a.qsl, a.kv_lens, a.S, A.min_q, A.tokb, a.window, bid, a.Hkv,
                                                  A.places, A.T)
                          : tile_item_any<MfmaRule>(a.qsl, a.kv_lens, a.S, A.min_q, A.tokb, a.window, bid, a.Hkv,
                                                    A.places, tcum, wred, A.T);
  if (ti.tile < 0) {
    const int first = ti.total * a.Hkv * ti.places;
    zero_other_rows<QT>(a, A.T, D, bid - first, A.items * a.Hkv * A.places - first);
    return;
  }
  const int s = ti.s, tile = ti.tile, q0 = ti.q0, qlen = ti.qlen;
  const int kv_len = min(max(ti.kv_len, 0), a.max_blocks * a.bs);
  const int past = kv_len - qlen;  // query i sees keys [.., past + i]
  const int tok_lo = tile * A.tokb;
  const int HG = a.Hq / a.Hkv;

  // ---- this lane's query columns
  int ctok[CT], chead[CT], limit[CT], start[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int c = (wv * CT + ct) * 16 + col;
    const int t = c / HG;
    ctok[ct] = tok_lo + t;
    chead[ct] = c - t * HG;
    limit[ct] = min(past + ctok[ct], kv_len - 1);
    start[ct] = a.window > 0 ? max(0, past + ctok[ct] - a.window + 1) : 0;
    if (t >= A.tokb || ctok[ct] >= qlen || (unsigned)(q0 + ctok[ct]) >= (unsigned)A.T) ctok[ct] = -1;  // no such column
    if (ctok[ct] < 0) limit[ct] = -1;
  }
  const int t_last = min(tok_lo + A.tokb, min(qlen, A.T - q0)) - 1;
  const int k_hi = min(past + t_last, kv_len - 1);
  const int k_lo = a.window > 0 ? max(0, past + tok_lo - a.window + 1) : 0;
  const int steps_all = k_hi >= 0 ? max(k_hi / NT - k_lo / NT + 1, 0) : 0;
  const int item = ti.item, part = ti.part, nparts = prefill_parts(steps_all * NT, ti.most);
  if (part >= nparts) return;
  const int step_lo = k_lo / NT + part * steps_all / nparts;
  const int step_hi = k_lo / NT + (part + 1) * steps_all / nparts - 1;

  // ---- query operands (zeros for absent columns)
  Op qB[CT][P::KS];
  Op qbias[CT];  // affine, lane group 0: the query's sum over each group as fp16 hi + lo at 2 g, 2 g + 1
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const bool ok = ctok[ct] >= 0;
    const QT* qp = reinterpret_cast<const QT*>(a.q) +
                   ((size_t)(ok ? q0 + ctok[ct] : 0) * a.Hq + (size_t)kvh * HG + (ok ? chead[ct] : 0)) * D + 8 * jj;
    float gsum[G] = {};
#pragma unroll
    for (int w = 0; w < P::KS; ++w) {
      const u32x4 x = *reinterpret_cast<const u32x4*>(qp + 32 * w);
      const Op v = __builtin_bit_cast(Op, ok ? x : u32x4{0u, 0u, 0u, 0u});
      if constexpr (AFF) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          qB[ct][w][i] = v[slot_perm<C::kBits>(i)];  // the unpacked codes' order
          gsum[32 * w / C::kGS] += (float)v[i];
        }
      } else {
        qB[ct][w] = v;
      }
    }
    if constexpr (AFF) {
      qbias[ct] = Op{};
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float x = rows4_sum(gsum[g]);
        const h16 hi = (h16)x;
        if (jj == 0) {
          qbias[ct][2 * g] = hi;
          qbias[ct][2 * g + 1] = (h16)(x - (float)hi);
        }
      }
    }
  }

  // ---- pages: lane l holds the page id of key l of a step (positions past the tile's last key repeat it)
  const size_t rowb = (size_t)a.Hkv * D * sizeof(typename C::ET);  // token-major
  const char* kbase = reinterpret_cast<const char*>(a.kc) + (AFF ? 0 : (size_t)kvh * (D * sizeof(typename C::ET)));
  const char* vbase = reinterpret_cast<const char*>(a.vc) + (AFF ? 0 : (size_t)kvh * (D * sizeof(typename C::ET)));
  const int32_t* bt = a.block_tables + (size_t)s * a.max_blocks;
  auto page_id = [&](const int st) { return bt[page_of(min(st * NT + (lane & (NT - 1)), k_hi), A.inv_bs)]; };
  u32x4 rk[P::NP], rv[P::NP];  // the next step's pieces
  u32x2 ru[AFF ? 8 : 1];       // affine: its V units
  u32x4 rs;                    // affine: scale piece `lane` (every wave loads them: the largest scale is a wave's business)
  uint64_t okn = 0;            // keys of that step on a valid page
  float psk = 0.f, psv = 0.f;  // FP8: page scales of key `lane` of that step
  auto load_step = [&](const int st, const int blk) {
    const int pos = min(st * NT + (lane & (NT - 1)), k_hi);
    const bool ok = (unsigned)blk < (unsigned)a.nb;
    okn = __ballot(ok);
    const int b = ok ? blk : 0;
    const int off = pos - page_of(pos, A.inv_bs) * a.bs;
    if constexpr (AFF) {
      constexpr int B = C::kBits;
      const int row = (b * a.Hkv + kvh) * a.bs + off;
      {
        const int pc = min(lane, P::NPS - 1), seg = pc / (NT / 8), arr = seg / G, g = seg % G;
        const int r8 = __shfl(row, 8 * (pc % (NT / 8)), 64), o8 = __shfl(off, 8 * (pc % (NT / 8)), 64);
        const h16 *b_ks = a.ks, *b_kb = a.kb, *b_vs = a.vs, *b_vb = a.vb;
        asm("" : "+s"(b_ks), "+s"(b_kb), "+s"(b_vs), "+s"(b_vb));  // picked from registers, not by a vector load
        const h16* base = arr == 0 ? b_ks : arr == 1 ? b_kb : arr == 2 ? b_vs : b_vb;
        typedef const __attribute__((address_space(1))) u32x4* gu32x4;
        // (past the tile's last key the group's first token may repeat it: aligned down, inside the page)
        rs = *(gu32x4)(base + (size_t)G * (r8 - o8) + (size_t)g * a.bs + (o8 & ~7));
      }
#pragma unroll
      for (int n = 0; n < P::NP; ++n) {
        const int e = tid + 256 * n;  // (fewer than 256 pieces: the others repeat them)
        const int r = __shfl(row, (e / P::PR) & (NT - 1), 64);
        rk[n] = *reinterpret_cast<const u32x4*>(kbase + (size_t)r * P::RBK + 16 * (e % P::PR));
      }
      const int T = min(a.bs, 256 / B);  // tokens of a value tile (a power of two)
#pragma unroll
      for (int n = 0; n < P::NPV; ++n) {
        const int e = tid + 256 * n, u = e % P::U, dim = e / P::U;
        const int r = __shfl(row, u * P::UT, 64);
        const int o = (r & (T - 1)) & ~(P::UT - 1);
        ru[n] = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint32_t*>(vbase) +
                                                (size_t)(r & ~(T - 1)) * (D * B / 32) + (dim * T + o) * B / 32);
      }
    } else {
      const int row = b * a.bs + off;
      if constexpr (C::kFp8) {
        psk = a.kps[b];
        psv = a.vps[b];
      }
#pragma unroll
      for (int n = 0; n < P::NP; ++n) {
        const size_t o = (size_t)__shfl(row, tid / P::PR + n * P::RP, 64) * rowb + 16 * (tid % P::PR);
        rk[n] = *reinterpret_cast<const u32x4*>(kbase + o);
        rv[n] = *reinterpret_cast<const u32x4*>(vbase + o);
      }
    }
  };

  float m_run[CT], l_part[CT];
  f32x4 acc[CT][P::SB];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    m_run[ct] = -INFINITY;
    l_part[ct] = 0.f;
#pragma unroll
    for (int b = 0; b < P::SB; ++b) acc[ct][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float sl2 = a.scale_log2;
  int vexp = 0;          // FP8, affine: acc holds the sum / 2^vexp
  float pb[CT][G] = {};  // affine: sum p * v_bias
  if constexpr (AFF) {   // the bias operand's unused halves stay zero
    for (int i = tid; i < NT; i += 256) *reinterpret_cast<u32x4*>(kbe + 8 * i) = u32x4{0u, 0u, 0u, 0u};
  }

  int blk1 = 0;
  if (step_lo <= step_hi) {
    load_step(step_lo, page_id(step_lo));
    blk1 = page_id(min(step_lo + 1, step_hi));
  }
  for (int st = step_lo; st <= step_hi; ++st) {
    __syncthreads();  // the previous step's tiles are no longer read
    if constexpr (AFF) {
      constexpr int B = C::kBits;
#pragma unroll
      for (int n = 0; n < P::NP; ++n) {
        const int e = tid + 256 * n;
        uint16_t* kr = ke + affine_pos((e / P::PR) & (NT - 1)) * P::KSTR + (e % P::PR) * (128 / B);
        if (e < P::NPK) {
          if constexpr (B == 4) {
#pragma unroll
            for (int i = 0; i < 4; ++i) *reinterpret_cast<h16x8*>(kr + 8 * i) = unpack4_high(rk[n][i]);
          } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) *reinterpret_cast<h16x8*>(kr + 8 * i) = unpack8(rk[n][2 * i], rk[n][2 * i + 1]);
          }
        }
      }
#pragma unroll
      for (int n = 0; n < P::NPV; ++n) {
        const int e = tid + 256 * n;
        uint16_t* vr = ve + (e / P::U) * P::VSTR + (e % P::U) * P::UT;
        if constexpr (B == 4) {
          *reinterpret_cast<h16x8*>(vr) = unpack4_high(ru[n][0]);
          *reinterpret_cast<h16x8*>(vr + 8) = unpack4_high(ru[n][1]);
        } else {
          *reinterpret_cast<h16x8*>(vr) = unpack8(ru[n][0], ru[n][1]);
        }
      }
    } else {
#pragma unroll
      for (int n = 0; n < P::NP; ++n) {
        const int r = tid / P::PR + n * P::RP, c = (tid % P::PR) * (16 / P::EB);
        put_piece<C>(ke + r * P::KSTR + c, rk[n]);
        put_piece<C>(ve + r * P::VSTR + c, rv[n]);
      }
    }
    const uint64_t okm = okn;
    if constexpr (AFF) {
      // scales of keys past the tile's last one or on an invalid page (which may hold anything) as zeros
      const int pc = min(lane, P::NPS - 1), t8 = 8 * (pc % (NT / 8)), seg = pc / (NT / 8), arr = seg / G, g = seg % G;
      const int live = k_hi + 1 - st * NT - t8;
      u32x4 x = rs;
      if (live < 8 || !((okm >> t8) & 1)) {
        const int n = (okm >> t8) & 1 ? live : 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] &= (2 * e < n ? 0x0000FFFFu : 0u) | (2 * e + 1 < n ? 0xFFFF0000u : 0u);
      }
      int vm = 0;  // largest |v_scale|, as fp16 bits
      if (arr == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) vm = max(vm, (int)max(x[e] & 0x7FFFu, (x[e] >> 16) & 0x7FFFu));
      }
      // the accumulator's exponent follows the value scales' (exact powers of two; 6 binades of slack)
      const int ex = ((int)wave_max((float)vm) >> 10) - 15;
      if (ex > vexp || ex < vexp - 6) {
        const float f = __uint_as_float((uint32_t)(127 + vexp - ex) << 23);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int b = 0; b < P::SB; ++b) acc[ct][b] *= f;
        vexp = ex;
      }
      if (wv == 0 && lane < P::NPS) {
        const float down = __uint_as_float((uint32_t)(127 - vexp) << 23);
        const float f = arr == 0 ? (float)(1 << C::kCodeExp) : arr == 2 ? down : 1.f;
        const h16x8 hv = __builtin_bit_cast(h16x8, x);
        if (arr == 1) {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            *reinterpret_cast<h16x2*>(kbe + 8 * affine_pos(t8 + e) + 2 * g) = h16x2{hv[e], hv[e]};
        } else {
          float* dst = (arr == 0 ? ksf : arr == 2 ? vsf : vbf) + g * NT;
#pragma unroll
          for (int q = 0; q < 2; ++q)
            *reinterpret_cast<f32x4*>(dst + affine_pos(t8 + 4 * q)) =
                f32x4{(float)hv[4 * q] * f, (float)hv[4 * q + 1] * f, (float)hv[4 * q + 2] * f, (float)hv[4 * q + 3] * f};
        }
      }
    }
    float down = 1.f;
    if constexpr (C::kFp8) {
      // value scales enter with the probabilities, brought near 1 by a power of two that the
      // accumulator carries (exact; rescaled when the step's largest scale has another exponent)
      const float vmax = wave_max(psv);
      const int ex = min(max((int)((__float_as_uint(vmax) >> 23) & 0xFFu) - 127, -60), 60);
      if (ex != vexp) {
        const float f = __uint_as_float((uint32_t)(127 + min(max(vexp - ex, -126), 127)) << 23);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int b = 0; b < P::SB; ++b) acc[ct][b] *= f;
        vexp = ex;
      }
      down = __uint_as_float((uint32_t)(127 - ex) << 23);
      if (tid < NT) {
        ksf[tid] = psk * 256.f;
        vsf[tid] = psv * down;
      }
    }
    __syncthreads();
    if (st < step_hi) {
      load_step(st + 1, blk1);
      blk1 = page_id(min(st + 2, step_hi));
    }
    const int pos0 = st * NT;

#pragma unroll
    for (int h = 0; h < NT / 32; ++h) {
      // ---- S^T: lane (col, jj) gets keys 32 h + 16 t + 4 jj + r of its columns
      float sc[CT][8];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint16_t* kr = ke + (32 * h + 16 * t + col) * P::KSTR + 8 * jj;
        f32x4 c[CT][G];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int g = 0; g < G; ++g) c[ct][g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < P::KS; ++w) {
          const Op K = *reinterpret_cast<const Op*>(kr + 32 * w);
          const int g = w * G / P::KS;
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) c[ct][g] = mfma_op(K, qB[ct][w], c[ct][g]);
        }
        if constexpr (AFF) {
          // (the bias operand is zero outside lane group 0)
          const Op KB = *reinterpret_cast<const Op*>(kbe + 8 * (32 * h + 16 * t + col));
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            f32x4 v = mfma_op(KB, qbias[ct], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int g = 0; g < G; ++g) {
              const f32x4 ks4 = *reinterpret_cast<const f32x4*>(ksf + g * NT + 32 * h + 16 * t + 4 * jj);
#pragma unroll
              for (int r = 0; r < 4; ++r) v[r] = fmaf(c[ct][g][r], ks4[r], v[r]);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[ct][4 * t + r] = v[r];
          }
        } else {
          f32x4 ks4 = {1.f, 1.f, 1.f, 1.f};
          if constexpr (C::kFp8) ks4 = *reinterpret_cast<const f32x4*>(ksf + 32 * h + 16 * t + 4 * jj);
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[ct][4 * t + r] = C::kFp8 ? c[ct][0][r] * ks4[r] : c[ct][0][r];
        }
      }

      // ---- mask where a key of the half is not visible to every column
      const int kp = pos0 + 32 * h;
      const uint32_t okh = (uint32_t)(okm >> (32 * h));
      bool full = okh == 0xFFFFFFFFu;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) full = full && kp >= start[ct] && kp + 31 <= limit[ct];
      if (!full) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int k = AFF ? 8 * jj + e : 16 * (e >> 2) + 4 * jj + (e & 3);
            if (kp + k < start[ct] || kp + k > limit[ct] || !((okh >> k) & 1u)) sc[ct][e] = -INFINITY;
          }
      }

      // ---- online softmax
      float m_new[CT];
      bool grow = false;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        float tmax = -INFINITY;
#pragma unroll
        for (int e = 0; e < 8; ++e) tmax = fmaxf(tmax, sc[ct][e]);
        m_new[ct] = fmaxf(m_run[ct], rows4_max(tmax) * sl2);
        grow = grow || m_new[ct] > m_run[ct] + kLazyMax;
      }
      if (__any(grow)) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const bool up = m_new[ct] > m_run[ct] + kLazyMax;  // also the first finite maximum
          const float al = up ? __builtin_amdgcn_exp2f(m_run[ct] - m_new[ct]) : 1.f;
          l_part[ct] *= al;
#pragma unroll
          for (int b = 0; b < P::SB; ++b) acc[ct][b] *= al;
          if constexpr (AFF) {
#pragma unroll
            for (int g = 0; g < G; ++g) pb[ct][g] *= al;
          }
          if (up) m_run[ct] = m_new[ct];
        }
      }
      Op pB[CT][C::kParts];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        // p <= 2^(kLazyMax + 6), times a value scale below 2: inside fp16, and small p stay
        // clear of its sub-normals
        const float m_sub = fmaxf(m_run[ct], -3.0e38f) - 6.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          sc[ct][e] = __builtin_amdgcn_exp2f(fmaf(sc[ct][e], sl2, -m_sub));
          l_part[ct] += sc[ct][e];
        }
        if constexpr (C::kFp8) {
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const f32x4 vs4 = *reinterpret_cast<const f32x4*>(vsf + 32 * h + 16 * t + 4 * jj);
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[ct][4 * t + r] *= vs4[r];
          }
        }
        if constexpr (!AFF) split_p(sc[ct], pB[ct]);
      }

      // ---- O^T += V^T P^T
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if constexpr (AFF) {  // this group's operand: p * v_scale; the bias term in fp32
          f32x4 vs4[2], vb4[2];
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            vs4[t] = *reinterpret_cast<const f32x4*>(vsf + g * NT + 32 * h + 16 * t + 4 * jj);
            vb4[t] = *reinterpret_cast<const f32x4*>(vbf + g * NT + 32 * h + 16 * t + 4 * jj);
          }
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              x[e] = sc[ct][e] * vs4[e >> 2][e & 3];
              pb[ct][g] = fmaf(sc[ct][e], vb4[e >> 2][e & 3], pb[ct][g]);
            }
            split_p(x, pB[ct]);
          }
        }
#pragma unroll
        for (int b = g * P::SB / G; b < (g + 1) * P::SB / G; ++b) {
          Op V;
          if constexpr (AFF) {
            V = *reinterpret_cast<const Op*>(ve + (16 * b + col) * P::VSTR + 32 * h + 8 * jj);
          } else {
            const u32x2 v0 = read_tr(ve, P::VSTR, 32 * h, 16 * b, col, jj);
            const u32x2 v1 = read_tr(ve, P::VSTR, 32 * h + 16, 16 * b, col, jj);
            V = __builtin_bit_cast(Op, u32x4{v0[0], v0[1], v1[0], v1[1]});
          }
#pragma unroll
          for (int k = 0; k < C::kParts; ++k)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) acc[ct][b] = mfma_op(V, pB[ct][k], acc[ct][b]);
        }
      }
    }
  }
  if constexpr (AFF) {  // codes entered as code * 2^-kCodeExp; the bias term joins its group's dims
    const float f = __uint_as_float((uint32_t)(127 + vexp + C::kCodeExp) << 23);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int b = 0; b < P::SB; ++b) {
        const float bias = rows4_sum(pb[ct][b * G / P::SB]);
        acc[ct][b] = acc[ct][b] * f + bias;
      }
  }
  if constexpr (C::kFp8) {  // the codes entered as value * 2^-8
    const float f = __uint_as_float((uint32_t)(127 + vexp + 8) << 23);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int b = 0; b < P::SB; ++b) acc[ct][b] *= f;
  }

  // ---- a cut tile: store this wave's state; the wave arriving last among the parts merges
  if (nparts > 1) {
    const int u = item * a.Hkv + kvh;
    const __amdgpu_buffer_rsrc_t rp =
        uniform_rsrc(reinterpret_cast<uint8_t*>(A.ws_part) + (size_t)u * ti.most * P::PARTB, ti.most * P::PARTB);
    constexpr int NV = CT * P::SB;
    auto vo = [&](int k) { return ((wv * (NV + 1) + k) * 64 + lane) * 16; };
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int b = 0; b < P::SB; ++b) store_f32x4(acc[ct][b], rp, vo(P::SB * ct + b), part * P::PARTB);
    store_f32x4(f32x4{m_run[0], m_run[CT - 1], l_part[0], l_part[CT - 1]}, rp, vo(NV), part * P::PARTB);
    if (!arrive_last(A.ws_cnt + u * 4 + wv, nparts, lane)) return;
    // every part read back in part order: the result does not depend on the order of arrival
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      m_run[ct] = -INFINITY;
      l_part[ct] = 0.f;
#pragma unroll
      for (int b = 0; b < P::SB; ++b) acc[ct][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int q = 0; q < nparts; ++q) {
      const f32x4 ml = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(rp, vo(NV), q * P::PARTB, kCoherent));
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) {
        f32x4 o[P::SB];
#pragma unroll
        for (int b = 0; b < P::SB; ++b)
          o[b] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rp, vo(P::SB * ct + b), q * P::PARTB,
                                                                                 kCoherent));
        const float m1 = ml[ct], l1 = ml[2 + ct];
        const float mn = fmaxf(m_run[ct], m1);
        const float f0 = m_run[ct] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run[ct] - mn);
        const float f1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - mn);
#pragma unroll
        for (int b = 0; b < P::SB; ++b) acc[ct][b] = acc[ct][b] * f0 + o[b] * f1;
        l_part[ct] = l_part[ct] * f0 + l1 * f1;
        m_run[ct] = mn;
      }
    }
  }

  // ---- normalise and write: lane (col, jj) holds dims 16 b + 4 jj + r of its columns
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    float l = l_part[ct] + __shfl_xor(l_part[ct], 16, 64);
    l += __shfl_xor(l, 32, 64);
    const bool ok = ctok[ct] >= 0;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const size_t orow = ((size_t)(ok ? q0 + ctok[ct] : 0) * a.Hq + (size_t)kvh * HG + (ok ? chead[ct] : 0)) * D;
    QT* op = reinterpret_cast<QT*>(a.out) + orow;
    bool bad = not_finite(l);
#pragma unroll
    for (int b = 0; b < P::SB; ++b) {
      struct alignas(8) Four {
        QT x[4];
      } v;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        bad = bad || not_finite(acc[ct][b][r]);
        from_f32(acc[ct][b][r] * inv, &v.x[r]);
      }
      if (ok) *reinterpret_cast<Four*>(op + 16 * b + 4 * jj) = v;
    }
    // columns that are not finite: again in fp32 (attend_row)
    uint64_t todo = __ballot(bad && ok);
    todo = (todo | (todo >> 16) | (todo >> 32) | (todo >> 48)) & 0xFFFFu;
    while (todo) {
      const int c = __builtin_ctzll(todo);
      todo &= todo - 1;
      const int t = __builtin_amdgcn_readlane(ctok[ct], c), hh = __builtin_amdgcn_readlane(chead[ct], c);
      const int k0 = __builtin_amdgcn_readlane(start[ct], c), k1 = __builtin_amdgcn_readlane(limit[ct], c) + 1;
      const size_t ro = ((size_t)(q0 + t) * a.Hq + (size_t)kvh * HG + hh) * D;
      float mr, lr, x[D / 64];
      attend_row<C, D>(a, s, kvh, reinterpret_cast<const QT*>(a.q) + ro, k0, k1, mr, lr, x, lane);
      const float li = lr > 0.f ? 1.f / lr : 0.f;
#pragma unroll
      for (int i = 0; i < D / 64; ++i) from_f32(x[i] * li, reinterpret_cast<QT*>(a.out) + ro + lane + 64 * i);
    }
  }
}

// Workgroups [0, ndec) decode the single-token rows (decode_mfma.hpp), the rest take the
// query tiles: as unified.hpp does, the page streams run beside the matrix work.
// (Two workgroups per compute unit; at D 256, where the decode body alone takes 250 registers and
// more, the bound spills 7 to 117 of them, at D 128 over 4-bit group 64 34 and 8-bit pages 47 and 9.)
template <class C, int D, int CT>
__global__ __launch_bounds__(256, 2) void mixed_mfma(PrefillMfmaArgs p, DecodeMfmaArgs d, int ndec) {
  if ((int)blockIdx.x < ndec)
    decode_mfma_body<C, D>(d, blockIdx.x, ndec);
  else
    prefill_mfma_body<C, D, CT>(p, (int)blockIdx.x - ndec);
}

}  // namespace emx
