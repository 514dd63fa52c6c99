// Single-token paged decode, head_dim 64, 128 or 256, any GQA ratio, over token-major
// caches [nb, bs, Hkv, D] (unquantized fp16 / bf16, FP8 E4M3 with one fp32 scale per
// page; pages of a multiple of 8 tokens) and over affine pages.  MFMA, split-K, one
// launch.
//
// Replaces the reference's per-(seq, q_head) serial key loop
// (lib/python/easymlx/operations/kernels/unified_attention.py:467-609, head-256
// :611-775, FP8 :776-1268) and its split-K form (page_attention.py:1718-2059).
//
// Work: a unit is (sequence, kv head, up to 16 query heads), an item 128 tokens
// of one unit (32 per wave; 256 and 64 over 4-bit pages).  Items are ordered unit-major and workgroup w of NWG
// takes the range [w I / NWG, (w + 1) I / NWG); a unit inside one range goes
// straight to the output, a cut one leaves an fp32 partial per workgroup, merged
// by the workgroup that arrives last (counter per unit, zero before and after).
//
// Per 32-token item of a wave (lane l: i = l % 16, jj = l / 16)
//   QK^T : v_mfma 16x16x32, A row i of sub-tile t = token 16 t + i; a load
//          instruction reads 64 contiguous bytes of each of its 16 rows.  B column
//          i = query head i.  Lane (h, jj) gets the scores of tokens 16 t + 4 jj + r.
//   PV   : the k slot 8 jj + e is token 16 (e / 4) + 4 jj + e % 4, the eight scores
//          lane (h, jj) holds, so P needs no lane exchange.  Lane (i, jj) loads dims
//          D/16 i .. of those eight tokens (whole rows per 16 lanes) and sub-tile b
//          takes dim D/16 i + b, picked by byte permutes.
// Affine pages (as decode_affine.hpp, without its limits on head_dim and GQA): K rows are
// taken in the order token TPL (i / 4) + 4 t + i % 4, so that lane (h, jj) ends with the
// scores of TPL consecutive tokens, the tokens of the dim-major value words it loads; one
// accumulator per quantization group, scale and bias applied in fp32 after the MFMA; the
// value scale enters the probability before it is split, sum p * v_bias is kept in fp32.
// K of the next item is loaded as soon as QK^T has consumed this one's registers,
// V after PV: one register image, always in flight.
//
// Bound by HBM.  Against decode_split and its merge (VALU dot products, single-element
// loads, two launches), which ran these shapes before: batch 32, contexts of 512 to
// 4096, 8 kv heads, D 128, pages of 16: bf16 (311 MB) 121.7 -> 67 us, FP8 (136 MB)
// 330 -> 39 us; one context of 1024, D 64, fp16: 38.4 -> 11.4 us; 8-bit pages, D 256, 13
// contexts of 200 to 5000 (64 MB): 141 -> 30 us.  Slower than they: more than 1024 units of a few
// tokens at D 256 (96 contexts of 3 to 16, 16 heads: bf16 19.5 / 23.9, 4-bit 22.1 / 26.6 us), 4-bit D 256
// without GQA at 60 to 128 tokens (200 contexts of 16 heads 115 / 135).
#pragma once

#include "mfma_common.hpp"

namespace emx {

struct DecodeMfmaArgs {
  DecodeArgs d;      // kc / vc: the caches; nt: DecodeMfmaCfg::NT; ws_cnt, ws_o [slot][hc][D], ws_ml [slot][hc][2]
  int hc, nhc;       // query heads per unit (<= 16) and units per kv head
  uint32_t inv_bs;   // ceil(2^32 / bs)
  int T;             // query rows
};

// A unit that is cut costs its merge (a round trip through memory, the atomic and the
// partials: ~6 us, six items' time).  Ranges start at unit starts where no range of whole
// units is longer than an equal share of the items and this many more; else they are cut freely.
// Eight units of 64 items more than workgroups (65 contexts of 8192 tokens, 8 kv heads), where whole
// units put two into eight workgroups: FP8 292 -> 180 us, bf16 310 -> 226.
constexpr int kDecodeMfmaMergeItems = 6;

template <class C, int D>
struct DecodeMfmaCfg {
  static constexpr int EB = sizeof(typename C::ET);   // bytes per cache element (token-major)
  static constexpr int KS = D / 32;                   // QK^T k-slices
  static constexpr int SB = D / 16;                   // PV sub-tiles
  static constexpr int NTW = 32;                      // tokens of a wave's item
  static constexpr int NT = 4 * NTW;                  // tokens of an item
  static constexpr int NA = NTW / 16;                 // QK^T sub-tiles
  static constexpr int NV = NTW / 4;                  // scores per lane
  static constexpr int KL = D * EB / 64;              // 16-byte K loads per row (per lane)
  static constexpr int KW = KL * 4;                   // K words a lane holds per sub-tile
  static constexpr int VN = NTW / 4, VW = SB * EB / 4;  // tokens, words per token of V a lane holds
  static constexpr int NL = 4;                        // page lookups per item
  static constexpr int G = 1, SNI = 1, STAGE = 0;
  static constexpr int RD = D < 128 ? D : 128;        // dims combined per round
  static constexpr int XS = RD + 4;                   // LDS stride of a head's combined dims
};
template <int BITS, int GS, int D>
struct DecodeMfmaCfg<KvAffine<BITS, GS>, D> {
  static constexpr int KS = D / 32, SB = D / 16;
  static constexpr int NTW = 256 / BITS, NT = 4 * NTW, NA = NTW / 16, NV = NTW / 4;
  static constexpr int BD = GS < 64 ? GS : 64;        // dims of a K block: one quantization group
  static constexpr int LD = BD / 4;                   // dims of a block a lane holds
  static constexpr int BW = LD * BITS / 32;           // words of them
  static constexpr int KW = (D / BD) * BW;
  static constexpr int VN = SB, VW = 2;               // V: dims a lane holds, words of each (its NV tokens)
  static constexpr int G = D / GS;
  static constexpr int NP = 4 * G * NTW / 8;          // 16-byte scale pieces of an item
  static constexpr int SNI = (NP + 63) / 64;
  static constexpr int NL = 2 + SNI;
  static constexpr int STAGE = 4 * G * NTW;           // halves of a wave's scale slot
  static constexpr int RD = D < 128 ? D : 128, XS = RD + 4;
};

template <class C, int D>
struct DecodeMfmaLoads {
  using P = DecodeMfmaCfg<C, D>;
  uint32_t k[P::NA][P::KW];
  uint32_t v[P::VN][P::VW];
  u32x4 s[P::SNI];  // affine: scale pieces
};

// MFMA operand of K k-slice w from the loaded words of one row.  16-bit: load w
// holds dims 32 w + 8 jj ..; FP8: load w / 2 holds dims 64 (w / 2) + 16 jj .., its
// halves the slices w, w + 1 (the query operand follows the same order).
template <class C, int D>
__device__ __forceinline__ typename C::Op k_operand(const uint32_t* k, const int w) {
  if constexpr (C::kFp8) {
    const uint32_t d0 = k[2 * w], d1 = k[2 * w + 1];
    return as_h8(e4m3x2_to_h16x2(__builtin_amdgcn_perm(0u, d0, 0x0C010C00u)),
                 e4m3x2_to_h16x2(__builtin_amdgcn_perm(0u, d0, 0x0C030C02u)),
                 e4m3x2_to_h16x2(__builtin_amdgcn_perm(0u, d1, 0x0C010C00u)),
                 e4m3x2_to_h16x2(__builtin_amdgcn_perm(0u, d1, 0x0C030C02u)));
  } else {
    return __builtin_bit_cast(typename C::Op, u32x4{k[4 * w], k[4 * w + 1], k[4 * w + 2], k[4 * w + 3]});
  }
}

// PV operand of sub-tile b: element b of each of the eight tokens.
template <class C, int VW>
__device__ __forceinline__ typename C::Op v_operand(const uint32_t (&v)[8][VW], const int b) {
  uint32_t w[4];
  if constexpr (C::kFp8) {
    const uint32_t sel = 0x0C000C00u | (uint32_t)(b & 3) | ((uint32_t)(4 + (b & 3)) << 16);
#pragma unroll
    for (int m = 0; m < 4; ++m)
      w[m] = e4m3x2_to_h16x2(__builtin_amdgcn_perm(v[2 * m + 1][b >> 2], v[2 * m][b >> 2], sel));
  } else {
#pragma unroll
    for (int m = 0; m < 4; ++m)
      w[m] = __builtin_amdgcn_perm(v[2 * m + 1][b >> 1], v[2 * m][b >> 1], b & 1 ? 0x07060302u : 0x05040100u);
  }
  return __builtin_bit_cast(typename C::Op, u32x4{w[0], w[1], w[2], w[3]});
}

// O / L to four adjacent outputs (zeros for L = 0, a row without a live key);
// true when a value of O is not finite.
template <class QT>
__device__ __forceinline__ bool write4(const f32x4 O, const float L, QT* out) {
  struct alignas(8) Four {
    QT x[4];
  } v;
  bool bad = false;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    bad |= not_finite(O[k]);
    from_f32(L > 0.f ? O[k] / L : 0.f, &v.x[k]);
  }
  *reinterpret_cast<Four*>(out) = v;
  return bad;
}

// Per-sequence tables in LDS: cum[s] = items (of NT tokens, per unit) of the decoded
// sequences before s, kvl[s] = clamped kv_len (-1: not a single-token row of the call's T), qrw[s] = query row.
// (seq_table of decode_affine.hpp with a constant item size: its two divisions by a run-time
// one and the serial 64-bit range arithmetic were a third of a short call.)
template <int NT>
__device__ __forceinline__ void decode_mfma_table(const DecodeArgs& a, const int T, int* cum, int* kvl, int* qrw, int* wsum) {
  const int ch = (a.S + 255) / 256, s0 = threadIdx.x * ch;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int tsum = 0;
  for (int i = 0; i < ch; ++i) {
    const int s = s0 + i;
    if (s >= a.S) break;
    const int kl = max(min(a.kv_lens[s], a.max_blocks * a.bs), 0);
    const int q0 = a.qsl ? a.qsl[s] : s, q1 = a.qsl ? a.qsl[s + 1] : s + 1;
    const bool dec = q1 - q0 == 1 && (unsigned)q0 < (unsigned)T;
    const int st = a.window > 0 ? max(0, kl - a.window) : 0;
    const int n = dec && kl > 0 ? (kl - 1) / NT - st / NT + 1 : 0;
    kvl[s] = dec ? kl : -1;
    qrw[s] = q0;
    cum[s] = n;  // the count for now
    tsum += n;
  }
  int x = tsum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) wsum[wv] = x;
  __syncthreads();
  int run = x - tsum;
#pragma unroll
  for (int w = 0; w < 3; ++w) run += w < wv ? wsum[w] : 0;
  for (int i = 0; i < ch; ++i) {
    const int s = s0 + i;
    if (s >= a.S) break;
    const int n = cum[s];
    cum[s] = run;
    run += n;
  }
  if (threadIdx.x == 255) cum[a.S] = run;
  __syncthreads();
}

template <class C, int D>
__device__ __forceinline__ void decode_mfma_body(const DecodeMfmaArgs& A, const int bid, const int nblocks) {
  using P = DecodeMfmaCfg<C, D>;
  typedef typename C::Op Op;
  typedef typename C::QT QT;
  const DecodeArgs& a = A.d;
  constexpr int NT = P::NT;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, jj = lane >> 4;
  auto uru = [](int v) { return __builtin_amdgcn_readfirstlane(v); };

  // LDS, carved from the shared arena
  constexpr int oCum = 0, oKvl = lds_next(oCum, 4 * (kMaxSeqs + 1)), oQrw = lds_next(oKvl, 4 * kMaxSeqs);
  constexpr int oXo = lds_next(oQrw, 4 * kMaxSeqs), oXml = lds_next(oXo, 4 * 4 * 16 * P::XS);
  constexpr int oFlag = lds_next(oXml, 4 * 4 * 16 * 2), oEnd = lds_next(oFlag, 16);
  constexpr int oStage = oXo;  // (an item's scales are read before its unit's combine, on every wave)
  static_assert(oEnd <= kArenaBytes && 2 * 4 * P::STAGE <= oXml - oXo, "LDS arena too small");
  int(&cum)[kMaxSeqs + 1] = lds_at<int[kMaxSeqs + 1]>(oCum);
  int(&kvl)[kMaxSeqs] = lds_at<int[kMaxSeqs]>(oKvl);
  int(&qrw)[kMaxSeqs] = lds_at<int[kMaxSeqs]>(oQrw);
  float* xo = &lds_at<float>(oXo);      // [wave][head][XS]
  float* xml = &lds_at<float>(oXml);    // [wave][head][2]
  int& flag = lds_at<int>(oFlag);
  h16* stage = &lds_at<h16>(oStage) + wv * P::STAGE;  // affine: this wave's [array][group][token] scales
  decode_mfma_table<NT>(a, A.T, cum, kvl, qrw, reinterpret_cast<int*>(xml));
  const int S = a.S, HG = a.Hq / a.Hkv, Hu = a.Hkv * A.nhc;
  {  // decoded sequences without a live token produce zeros (the reference's l == 0 case)
    const int per_seq = a.Hq * D / 8;
    for (int i = bid * 256 + tid; i < S * per_seq; i += nblocks * 256) {
      const int si = i / per_seq;
      if (kvl[si] >= 0 && cum[si + 1] == cum[si])
        reinterpret_cast<u32x4*>(a.out)[(size_t)qrw[si] * per_seq + i % per_seq] = u32x4{0u, 0u, 0u, 0u};
    }
  }
  // (the host keeps the number of items below 2^31)
  const int I = Hu * uru(cum[S]);
  auto start_of = [&](int kl) { return a.window > 0 ? max(0, kl - a.window) : 0; };
  // The most items a unit has.  Solo: no unit's keys reach past one wave's tokens, and each takes units of
  // its own (a unit to a workgroup, with its three idle waves, the combine and the barriers, 3 to 10 us each:
  // 200 contexts of 3 to 16 tokens, 16 heads: bf16, D 64 27 -> 13 us, D 256 78 -> 41; 4-bit, D 256 135 -> 48).
  int nmax = 0;
  bool solo = true;
  for (int c = 0; c < S; c += 64) {
    const int si = c + lane;
    const int n = si < S ? cum[si + 1] - cum[si] : 0;
    nmax = max(nmax, n);
    if (n > 0) solo = solo && (kvl[si] - 1) / P::NTW == start_of(kvl[si]) / P::NTW;
  }
  nmax = uru((int)wave_max((float)nmax));
  solo = __all(solo);
  const int NW = min(solo ? 4 * nblocks : nblocks, I);
  const int worker = solo ? wv * nblocks + bid : bid;  // (solo: no barrier from here on)
  if (worker >= NW) return;
  const int per = (unsigned)I / (unsigned)NW, extra = I - per * NW;  // the first `extra` ranges hold one item more
  auto first_of = [&](int w) { return w * per + min(w, extra); };
  auto wg_of = [&](int g) {  // the workgroup whose range holds item g
    const int big = extra * (per + 1);
    return g < big ? (int)((unsigned)g / (unsigned)(per + 1)) : extra + (int)((unsigned)(g - big) / (unsigned)per);
  };
  // The sequence of item g.
  auto seq_of = [&](const int g) {
    int s = 0;
    for (int c = 0; c < S; c += 64) {
      const int si = c + lane;
      s += __builtin_popcountll(__ballot(si < S && Hu * cum[si + 1] <= g));
    }
    return uru(s);
  };
  bool cut = nmax > per + kDecodeMfmaMergeItems;  // (some range holds the longest unit)
  if (!cut && nmax > kDecodeMfmaMergeItems) {     // (no range exceeds per + nmax)
    // the longest range of whole units: those whose first item lies in an equal share
    auto ceil_at = [&](const int w) {
      const int g = first_of(w);
      if (g >= I) return I;
      int lo = 0, hi = S;  // the sequence of item g: the first s with Hu * cum[s + 1] > g
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (Hu * cum[mid + 1] > g) hi = mid;
        else lo = mid + 1;
      }
      const int b = Hu * cum[lo], n = cum[lo + 1] - cum[lo];
      return b + (int)((unsigned)(g - b + n - 1) / (unsigned)n) * n;
    };
    const int ch = (NW + 255) / 256, w0 = min(tid * ch, NW), w1 = min(w0 + ch, NW);
    int longest = 0, at = ceil_at(w0);
    for (int w = w0; w < w1; ++w) {
      const int next = ceil_at(w + 1);
      longest = max(longest, next - at);
      at = next;
    }
    int* red = reinterpret_cast<int*>(xml);
    const int x = (int)wave_max((float)longest);
    if (lane == 0) red[wv] = x;
    __syncthreads();
    cut = max(max(red[0], red[1]), max(red[2], red[3])) > per + kDecodeMfmaMergeItems;
    cut = uru(cut);
  }
  int g0 = first_of(worker), g1 = first_of(worker + 1);
  if (!cut) {  // whole units: those whose first item lies in the range
    auto unit_ceil = [&](const int g) {
      if (g >= I) return I;
      const int s = seq_of(g);
      const int b = Hu * uru(cum[s]), n = uru(cum[s + 1]) - uru(cum[s]);
      return b + uru((int)((unsigned)(g - b + n - 1) / (unsigned)n)) * n;
    };
    g0 = unit_ceil(g0);
    g1 = unit_ceil(g1);
    if (g0 >= g1) return;
  }

  // An item: item j of the n of unit y of sequence s; this wave's tokens start at tb.
  // (No bool: the compiler kept the bytes that pad it as arrays in LDS, whose index needs the workgroup's
  // size from the dispatch packet in host memory, 7 us and more before the first product with all compute
  // units at it: 25 contexts of 8 to 17 tokens, bf16, D 64, 19.1 -> 7.4 us; batch 32 over FP8 pages of 16
  // 46.6 -> 38.7.)
  struct Item {
    int s, y, j, n, kl, st, tb;
    int has;  // inside the range
  };
  auto tb_of = [&](int st, int jx) { return solo ? st / P::NTW * P::NTW : (st / NT + jx) * NT + P::NTW * wv; };
  Item it0;
  {
    it0.s = seq_of(g0);
    it0.n = uru(cum[it0.s + 1]) - uru(cum[it0.s]);
    const int r = g0 - Hu * uru(cum[it0.s]);
    it0.y = uru((int)((unsigned)r / (unsigned)it0.n));
    it0.j = r - it0.y * it0.n;
    it0.kl = uru(kvl[it0.s]);
    it0.st = start_of(it0.kl);
    it0.tb = tb_of(it0.st, it0.j);
    it0.has = true;
  }
  // the item after x, g being x's index; past the range x again with has = false
  auto after = [&](const Item& x, const int g) {
    Item r = x;
    r.has = g + 1 < g1;
    if (!r.has) return r;
    if (++r.j == r.n) {
      r.j = 0;
      if (++r.y == Hu) {
        r.y = 0;
        do {
          ++r.s;
        } while (uru(cum[r.s + 1]) == uru(cum[r.s]));
        r.n = uru(cum[r.s + 1]) - uru(cum[r.s]);
        r.kl = uru(kvl[r.s]);
        r.st = start_of(r.kl);
      }
    }
    r.tb = tb_of(r.st, r.j);
    return r;
  };

  const char* kbase = reinterpret_cast<const char*>(a.kc);
  const char* vbase = reinterpret_cast<const char*>(a.vc);
  auto ok_blk = [&](int b) { return (unsigned)b < (unsigned)a.nb; };

  // Page lookups of one item.  Token-major: K rows of tokens 16 t + i (n = 0, 1) and the
  // quads 16 t + 4 jj (n = 2, 3: V rows, FP8 page scales), positions past the end
  // repeating the last live token.  Affine: the NV tokens of the lane's K rows (n = 0), of its
  // value words (n = 1), the 8 tokens of its scale pieces (n = 2 ..); a group past the end
  // repeats the last live one.
  struct Look {
    int blk[P::NL];
  };
  // affine: scale piece i of the lane: segment (array, group), 8 tokens (lanes past the last repeat it)
  auto piece_of = [&](int i) {
    if constexpr (C::kAffine) return min(64 * i + lane, P::NP - 1);
    return 0;
  };
  auto pos_of = [&](const Item& x, int n) {
    if constexpr (C::kAffine) {
      if (n < 2) return min(x.tb + P::NV * (n == 0 ? col >> 2 : jj), (x.kl - 1) & ~(P::NV - 1));
      return min(x.tb + 8 * (piece_of(n - 2) % (P::NTW / 8)), (x.kl - 1) & ~7);
    } else {
      return min(x.tb + 16 * (n & 1) + (n < 2 ? col : 4 * jj), x.kl - 1);
    }
  };
  auto lookup = [&](Look& L, const Item& x) {
#pragma unroll
    for (int n = 0; n < P::NL; ++n)
      L.blk[n] = a.block_tables[(size_t)x.s * a.max_blocks + page_of(pos_of(x, n), A.inv_bs)];
  };

  // (an item past the range: every lane reads the cache's first bytes, one line; the loads are
  // issued on every path, so that the wait before a use never drains the ones behind it)
  DecodeMfmaLoads<C, D> ld;
  float ks[2] = {1.f, 1.f}, vs[2] = {1.f, 1.f}, ks1[2], vs1[2];  // FP8 page scales: this item's, the next one's
  // token-major: byte offset of the row of lookup n
  const size_t rowb = (size_t)a.Hkv * D * (C::kAffine ? 1 : sizeof(typename C::ET));
  auto row_of = [&](const Look& L, int n, const Item& x) {
    const int p = pos_of(x, n);
    const int b = ok_blk(L.blk[n]) ? L.blk[n] : 0;
    return ((size_t)b * a.bs + (p - page_of(p, A.inv_bs) * a.bs)) * rowb +
           (size_t)(x.y / A.nhc) * (D * sizeof(typename C::ET));
  };
  // affine: page-head and offset of lookup n's first token
  auto ph_of = [&](const Look& L, int n, const Item& x, int& off) {
    const int p = pos_of(x, n);
    off = p - page_of(p, A.inv_bs) * a.bs;
    return (size_t)(ok_blk(L.blk[n]) ? L.blk[n] : 0) * a.Hkv + x.y / A.nhc;
  };
  auto issue_k = [&](const Look& L, const Item& x) {
    if constexpr (C::kAffine) {
      constexpr int B = C::kBits;
#pragma unroll
      for (int i = 0; i < P::SNI; ++i) {
        const int seg = piece_of(i) / (P::NTW / 8), arr = seg / P::G, g = seg % P::G;
        int off;
        const size_t ph = ph_of(L, 2 + i, x, off);
        const h16 *b_ks = a.ks, *b_kb = a.kb, *b_vs = a.vs, *b_vb = a.vb;
        asm("" : "+s"(b_ks), "+s"(b_kb), "+s"(b_vs), "+s"(b_vb));  // picked from registers, not by a vector load
        const h16* base = arr == 0 ? b_ks : arr == 1 ? b_kb : arr == 2 ? b_vs : b_vb;
        typedef const __attribute__((address_space(1))) u32x4* gu32x4;
        ld.s[i] = *(gu32x4)(base + (x.has ? (ph * P::G + g) * a.bs + off : 0));
      }
      int off;
      const size_t ph = ph_of(L, 0, x, off);
      // K rows of tokens 4 t + i % 4 of the lane's group; a block's BD dims over the four lane groups
      const char* p = kbase + (x.has ? (ph * a.bs + off + (col & 3)) * (D * B / 8) + jj * (P::BW * 4) : 0);
#pragma unroll
      for (int t = 0; t < P::NA; ++t)
#pragma unroll
        for (int bl = 0; bl < D / P::BD; ++bl) {
          const char* q = p + (x.has ? 4 * t * (D * B / 8) + bl * (P::BD * B / 8) : 0);
          uint32_t* dst = &ld.k[t][bl * P::BW];
          if constexpr (P::BW == 4) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(q);
#pragma unroll
            for (int c = 0; c < 4; ++c) dst[c] = v[c];
          } else if constexpr (P::BW == 2) {
            const u32x2 v = *reinterpret_cast<const u32x2*>(q);
            dst[0] = v[0];
            dst[1] = v[1];
          } else {
            dst[0] = *reinterpret_cast<const uint32_t*>(q);
          }
        }
    } else {
      if constexpr (C::kFp8) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int b = ok_blk(L.blk[2 + t]) ? L.blk[2 + t] : 0;
          ks1[t] = a.kps[b];
          vs1[t] = a.vps[b];
        }
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const char* p = kbase + (x.has ? row_of(L, t, x) + 16 * jj : 0);
#pragma unroll
        for (int w = 0; w < P::KL; ++w) {
          const u32x4 v = *reinterpret_cast<const u32x4*>(p + (x.has ? 64 * w : 0));
#pragma unroll
          for (int c = 0; c < 4; ++c) ld.k[t][4 * w + c] = v[c];
        }
      }
    }
  };
  auto issue_v = [&](const Look& L, const Item& x) {
    if constexpr (C::kAffine) {
      // two words per dim 16 b + i: the lane's NV tokens (one page: bs % NV == 0)
      constexpr int B = C::kBits;
      int off;
      const size_t ph = ph_of(L, 1, x, off);
      const int T = min(a.bs, P::NTW);  // tokens of a value tile
      const size_t w0 = x.has ? v_word_index<B>(ph, off, col, D, a.bs) : 0;
#pragma unroll
      for (int b = 0; b < P::SB; ++b) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(a.vc + w0 + (x.has ? 16 * b * (T * B / 32) : 0));
        ld.v[b][0] = v[0];
        ld.v[b][1] = v[1];
      }
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        // the quad's tokens lie in one page (bs % 8 == 0); past the end they repeat the last live one
        const size_t r0 = x.has ? row_of(L, 2 + t, x) + (size_t)col * (4 * P::VW) : 0;
        const int left = x.has ? x.kl - 1 - pos_of(x, 2 + t) : 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const uint32_t* w = reinterpret_cast<const uint32_t*>(vbase + r0 + (size_t)min(r, left) * rowb);
          uint32_t(&dst)[P::VW] = ld.v[4 * t + r];
          if constexpr (P::VW == 1) {
            dst[0] = w[0];
          } else if constexpr (P::VW == 2) {
            const u32x2 v = *reinterpret_cast<const u32x2*>(w);
            dst[0] = v[0];
            dst[1] = v[1];
          } else {
#pragma unroll
            for (int c = 0; c < P::VW / 4; ++c) {
              const u32x4 v = *reinterpret_cast<const u32x4*>(w + 4 * c);
#pragma unroll
              for (int e = 0; e < 4; ++e) dst[4 * c + e] = v[e];
            }
          }
        }
      }
    }
  };

  // query operand of a unit: column h = query head h (zero past the unit's heads)
  Op qB[P::KS];
  float qsum[P::G] = {};  // affine: the query's sum over each quantization group
  auto load_q = [&](int si, int yy) {
    const int kh = yy / A.nhc, h0 = (yy % A.nhc) * A.hc;
    const int nh = min(A.hc, HG - h0);
    const QT* qp = reinterpret_cast<const QT*>(a.q) +
                   ((size_t)qrw[si] * a.Hq + (size_t)kh * HG + h0 + (col < nh ? col : 0)) * D;
    if constexpr (C::kAffine) {
#pragma unroll
      for (int g = 0; g < P::G; ++g) qsum[g] = 0.f;
    }
#pragma unroll
    for (int w = 0; w < P::KS; ++w) {
      int d;
      if constexpr (C::kAffine)
        d = P::BD * (w / (P::LD / 8)) + P::LD * jj + 8 * (w % (P::LD / 8));
      else
        d = C::kFp8 ? 64 * (w >> 1) + 16 * jj + 8 * (w & 1) : 32 * w + 8 * jj;
      const u32x4 x = *reinterpret_cast<const u32x4*>(qp + d);
      const Op v = __builtin_bit_cast(Op, col < nh ? x : u32x4{0u, 0u, 0u, 0u});
      if constexpr (C::kAffine) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          qB[w][i] = v[slot_perm<C::kBits>(i)];  // the unpacked codes' order
          qsum[32 * w / C::kGS] += (float)v[i];
        }
      } else {
        qB[w] = v;
      }
    }
    if constexpr (C::kAffine) {
#pragma unroll
      for (int g = 0; g < P::G; ++g) qsum[g] = rows4_sum(qsum[g]);
    }
  };

  float m_run = -INFINITY, l_part = 0.f;
  f32x4 acc[P::SB];
  float pb[P::G];  // affine: sum p * v_bias per group
  int vexp = 0;    // affine: acc holds the sum / 2^vexp
  auto clear = [&]() {
    m_run = -INFINITY;
    l_part = 0.f;
    vexp = -60;
#pragma unroll
    for (int g = 0; g < P::G; ++g) pb[g] = 0.f;
#pragma unroll
    for (int b = 0; b < P::SB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear();

  // In flight, oldest first: K of this item, the lookups of the next, V of this item.
  Item cur = it0, nxt = after(cur, g0);
  Look lc, ln, l2;
  lookup(lc, cur);
  load_q(cur.s, cur.y);
  // (kept in this order: one path with another order would make every wait the longest one)
  __builtin_amdgcn_sched_barrier(0);
  issue_k(lc, cur);
  __builtin_amdgcn_sched_barrier(0);
  lookup(ln, nxt);
  __builtin_amdgcn_sched_barrier(0);
  issue_v(lc, cur);
  __builtin_amdgcn_sched_barrier(0);
  int seg0 = g0;  // first item of the unit that this workgroup holds

  for (int g = g0; g < g1; ++g) {
    const int s = cur.s, y = cur.y, n_s = cur.n, tb = cur.tb, kv_len = cur.kl, start_k = cur.st;
    const Item n2 = nxt.has ? after(nxt, g + 1) : nxt;
    // ---- scores: lane (h, jj), element 4 t + r
    constexpr int NV = P::NV;
    float sc[NV];
    bool okp = ok_blk(lc.blk[1]);
#pragma unroll
    for (int n = 2; n < P::NL; ++n) okp = okp && ok_blk(lc.blk[n]);
    const bool full = tb >= start_k && tb + P::NTW <= kv_len && __all(okp);
    if constexpr (C::kAffine) {
      // ---- this item's scales to the wave's LDS slot; those of tokens outside
      // [start_k, kv_len) or on an invalid page (which may hold anything) as zeros
      int vmax = 0;  // largest |v_scale|, as fp16 bits
#pragma unroll
      for (int i = 0; i < P::SNI; ++i) {
        const int pc = piece_of(i), p0 = tb + 8 * (pc % (P::NTW / 8));
        u32x4 x = ld.s[i];
        if (!full) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool ok0 = p0 + 2 * e >= start_k && p0 + 2 * e < kv_len && ok_blk(lc.blk[2 + i]);
            const bool ok1 = p0 + 2 * e + 1 >= start_k && p0 + 2 * e + 1 < kv_len && ok_blk(lc.blk[2 + i]);
            x[e] &= (ok0 ? 0x0000FFFFu : 0u) | (ok1 ? 0xFFFF0000u : 0u);
          }
        }
        if (pc / (P::NTW / 8) / P::G == 2) {
#pragma unroll
          for (int e = 0; e < 4; ++e) vmax = max(vmax, (int)max(x[e] & 0x7FFFu, (x[e] >> 16) & 0x7FFFu));
        }
        if (64 * i + lane < P::NP) *reinterpret_cast<u32x4*>(stage + 8 * pc) = x;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      // the accumulator's exponent follows the value scales', so that p * v_scale keeps to the
      // middle of fp16's range (exact powers of two; 6 binades of slack below)
      const int ex = ((int)wave_max((float)vmax) >> 10) - 15;
      if (ex > vexp || ex < vexp - 6) {
        const float f = __uint_as_float((uint32_t)(127 + vexp - ex) << 23);
#pragma unroll
        for (int b = 0; b < P::SB; ++b) acc[b] *= f;
        vexp = ex;
      }
#pragma unroll
      for (int t = 0; t < P::NA; ++t) {
        f32x4 c[P::G];
#pragma unroll
        for (int g = 0; g < P::G; ++g) c[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < P::KS; ++w) {
          const uint32_t* k = &ld.k[t][w * C::kBits / 4];
          c[32 * w / C::kGS] = mfma_op(C::kBits == 4 ? unpack4_high(k[0]) : unpack8(k[0], k[1]), qB[w], c[32 * w / C::kGS]);
        }
        typedef h16 h16x4v __attribute__((ext_vector_type(4)));
        float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int g = 0; g < P::G; ++g) {
          const h16x4v ks4 = *reinterpret_cast<const h16x4v*>(stage + g * P::NTW + NV * jj + 4 * t);
          const h16x4v kb4 = *reinterpret_cast<const h16x4v*>(stage + (P::G + g) * P::NTW + NV * jj + 4 * t);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = fmaf(c[g][r] * (float)(1 << C::kCodeExp), (float)ks4[r], fmaf((float)kb4[r], qsum[g], v[r]));
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[4 * t + r] = v[r];
      }
    } else {
      if constexpr (C::kFp8) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          ks[t] = ks1[t];
          vs[t] = vs1[t];
        }
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < P::KS; ++w) c = mfma_op(k_operand<C, D>(ld.k[t], w), qB[w], c);
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[4 * t + r] = C::kFp8 ? c[r] * (ks[t] * 256.f) : c[r];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    issue_k(ln, nxt);
    __builtin_amdgcn_sched_barrier(0);
    lookup(l2, n2);
    __builtin_amdgcn_sched_barrier(0);
    const bool unit_end = !nxt.has || nxt.s != s || nxt.y != y;

    // ---- mask: outside [start_k, kv_len), or on a page with an invalid id
    if (!full) {
#pragma unroll
      for (int e = 0; e < NV; ++e) {
        const int p = tb + (C::kAffine ? NV * jj + e : 16 * (e >> 2) + 4 * jj + (e & 3));
        if (p < start_k || p >= kv_len || !ok_blk(lc.blk[C::kAffine ? 1 : 2 + (e >> 2)])) sc[e] = -INFINITY;
      }
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int e = 0; e < NV; ++e) tmax = fmaxf(tmax, sc[e]);
    tmax = rows4_max(tmax) * a.scale_log2;
    const float m_new = fmaxf(m_run, tmax);
    if (__any(m_new != m_run)) {
      const float alpha = m_run == m_new ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_part *= alpha;
#pragma unroll
      for (int b = 0; b < P::SB; ++b) acc[b] *= alpha;
#pragma unroll
      for (int g = 0; g < P::G; ++g) pb[g] *= alpha;
      m_run = m_new;
    }
    const float m_sub = fmaxf(m_run, -3.0e38f) - kPBias;
#pragma unroll
    for (int e = 0; e < NV; ++e) {
      sc[e] = __builtin_amdgcn_exp2f(fmaf(sc[e], a.scale_log2, -m_sub));
      l_part += sc[e];
    }
    if constexpr (C::kAffine) {
      const float down = __uint_as_float((uint32_t)(127 - vexp) << 23);
#pragma unroll
      for (int w = 0; w < NV / 8; ++w)
#pragma unroll
        for (int g = 0; g < P::G; ++g) {
          const h16x8 vs8 = *reinterpret_cast<const h16x8*>(stage + (2 * P::G + g) * P::NTW + NV * jj + 8 * w);
          const h16x8 vb8 = *reinterpret_cast<const h16x8*>(stage + (3 * P::G + g) * P::NTW + NV * jj + 8 * w);
          float x[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            x[i] = sc[8 * w + i] * ((float)vs8[i] * down);
            pb[g] = fmaf(sc[8 * w + i], (float)vb8[i], pb[g]);
          }
          Op pB[C::kParts];
          split_p(x, pB);
#pragma unroll
          for (int b = g * (C::kGS / 16); b < (g + 1) * (C::kGS / 16); ++b) {
            const Op V = C::kBits == 4 ? unpack4_high(ld.v[b][w]) : unpack8(ld.v[b][0], ld.v[b][1]);
#pragma unroll
            for (int k = 0; k < C::kParts; ++k) acc[b] = mfma_op(V, pB[k], acc[b]);
          }
        }
    } else {
      float post = 1.f;
      if constexpr (C::kFp8) {
        // p * (value page scale), brought near 1 by a power of two taken out after the MFMA
        const float vmax = rows4_max(fmaxf(vs[0], vs[1]));
        const int ex = min(max((int)((__float_as_uint(vmax) >> 23) & 0xFFu) - 127, -100), 100);
        const float down = __uint_as_float((uint32_t)(127 - ex) << 23);
        post = __uint_as_float((uint32_t)(127 + ex + 8) << 23);  // the codes enter as value * 2^-8
#pragma unroll
        for (int e = 0; e < 8; ++e) sc[e] *= vs[e >> 2] * down;
      }
      Op pB[C::kParts];
      split_p(sc, pB);
#pragma unroll
      for (int b = 0; b < P::SB; ++b) {
        const Op V = v_operand<C, P::VW>(ld.v, b);
        f32x4 t = C::kFp8 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[b];
#pragma unroll
        for (int k = 0; k < C::kParts; ++k) t = mfma_op(V, pB[k], t);
        if constexpr (C::kFp8) {
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[b][r] = fmaf(t[r], post, acc[b][r]);
        } else {
          acc[b] = t;
        }
      }
    }
    issue_v(ln, nxt);

    if (unit_end) {
      // ---- the waves' states through LDS (rounds of RD dims), all threads combining
      const int kvh = y / A.nhc, h0 = (y % A.nhc) * A.hc, nh = min(A.hc, HG - h0);
      const int u = s * Hu + y;
      const int unit_first = Hu * uru(cum[s]) + y * n_s;
      const bool whole = seg0 == unit_first && g + 1 == unit_first + n_s;
      int slot = 0, np = 1;
      if (!whole) {
        const int wf = uru(wg_of(unit_first));
        np = uru(wg_of(unit_first + n_s - 1)) - wf + 1;
        slot = uru(wf + u);  // the unit's pieces sit in slots wf + u ..
      }
      float l = l_part + __shfl_xor(l_part, 16, 64);
      l += __shfl_xor(l, 32, 64);
      if constexpr (C::kAffine) {  // codes entered as code * 2^-kCodeExp; the bias term joins its group's dims
        const float f = __uint_as_float((uint32_t)(127 + vexp + C::kCodeExp) << 23);
#pragma unroll
        for (int g = 0; g < P::G; ++g) {
          const float bias = rows4_sum(pb[g]);
#pragma unroll
          for (int b = g * (C::kGS / 16); b < (g + 1) * (C::kGS / 16); ++b) acc[b] = acc[b] * f + bias;
        }
      }
      bool bad = false;
      QT* out = reinterpret_cast<QT*>(a.out) + ((size_t)qrw[s] * a.Hq + (size_t)kvh * HG + h0) * D;
      if (solo) {  // this wave has the whole unit: its lanes write what they hold
        if (col < nh) {
          QT* o = out + (size_t)col * D;
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int b = 0; b < P::SB; b += 4) {
              if constexpr (C::kAffine)
                bad |= write4(acc[b + r], l, o + 16 * (b + r) + 4 * jj);
              else
                bad |= write4(f32x4{acc[b][r], acc[b + 1][r], acc[b + 2][r], acc[b + 3][r]}, l,
                              o + (4 * jj + r) * P::SB + b);
            }
        }
      }
      const __amdgpu_buffer_rsrc_t ro =
          uniform_rsrc(a.ws_o + (size_t)slot * (A.hc * D), whole ? 0 : np * A.hc * D * 4);
      const __amdgpu_buffer_rsrc_t rm = uniform_rsrc(a.ws_ml + (size_t)slot * (A.hc * 2), whole ? 0 : np * A.hc * 8);
      const int me = whole ? 0 : uru(bid + u - slot);
      if (!solo) {
#pragma unroll
        for (int rd = 0; rd < D / P::RD; ++rd) {
          __syncthreads();  // (the previous combine has been read)
          constexpr int BR = P::SB / (D / P::RD);  // sub-tiles of the round
          float* xw = xo + (wv * 16 + col) * P::XS;
          if constexpr (C::kAffine) {  // sub-tile b, row 4 jj + r: dim 16 b + 4 jj + r
            if (col < nh) {
#pragma unroll
              for (int b = 0; b < BR; ++b) *reinterpret_cast<f32x4*>(xw + 16 * b + 4 * jj) = acc[rd * BR + b];
            }
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
              for (int b = 0; b < BR; b += 4) {
                const f32x4 x = {acc[rd * BR + b][r], acc[rd * BR + b + 1][r], acc[rd * BR + b + 2][r],
                                 acc[rd * BR + b + 3][r]};
                if (col < nh) *reinterpret_cast<f32x4*>(xw + (4 * jj + r) * BR + b) = x;
              }
          }
          if (rd == 0 && jj == 0 && col < nh) {
            xml[(wv * 16 + col) * 2] = m_run;
            xml[(wv * 16 + col) * 2 + 1] = l;
          }
          __syncthreads();
          for (int e = tid; e < nh * (P::RD / 4); e += 256) {
            const int h = e / (P::RD / 4), c = e % (P::RD / 4);
            float M = -INFINITY;
#pragma unroll
            for (int w = 0; w < 4; ++w) M = fmaxf(M, xml[(w * 16 + h) * 2]);
            f32x4 O = {0.f, 0.f, 0.f, 0.f};
            float L = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
              const float mw = xml[(w * 16 + h) * 2];
              const float f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw - M);
              O += *reinterpret_cast<const f32x4*>(xo + (w * 16 + h) * P::XS + 4 * c) * f;
              L = fmaf(xml[(w * 16 + h) * 2 + 1], f, L);
            }
            // element 4 c + k of the round is dim SB * row + rd * BR + ..: contiguous in k
            const int dim = C::kAffine ? rd * P::RD + 4 * c : (4 * c / BR) * P::SB + rd * BR + (4 * c) % BR;
            if (whole) {
              bad |= write4(O, L, out + (size_t)h * D + dim);
            } else {
#pragma unroll
              for (int k = 0; k < 4; ++k) bad |= not_finite(O[k]);
              store_f32x4(O, ro, (h * D + dim) * 4, me * A.hc * D * 4);
              if (rd == 0 && c == 0)
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{M, L}), rm, h * 8, me * A.hc * 8,
                                                      kCoherent);
            }
          }
        }
      }
      // ---- rows that are not finite over this workgroup's keys: again in fp32 (attend_row)
      const bool again = solo ? __any(bad) : __syncthreads_or(bad);
      if (again) {
        __builtin_amdgcn_s_waitcnt(0);  // every wave's stores above come first
        if (!solo) __syncthreads();
        const int b0 = start_k / NT - unit_first;  // item g of the unit: tokens from (b0 + g) NT
        // (a piece's sums are of p = 2^(x - m + kPBias), as the others')
        const int k0 = max(start_k, (b0 + seg0) * NT), k1 = min(kv_len, (b0 + g + 1) * NT);
        for (int h = solo ? 0 : wv; h < nh; h += solo ? 1 : 4) {
          float mr, lr, x[D / 64];
          const QT* qp = reinterpret_cast<const QT*>(a.q) + ((size_t)qrw[s] * a.Hq + (size_t)kvh * HG + h0 + h) * D;
          attend_row<C, D>(a, s, kvh, qp, k0, k1, mr, lr, x, lane);
#pragma unroll
          for (int i = 0; i < D / 64; ++i) {
            if (whole)
              from_f32(lr > 0.f ? x[i] / lr : 0.f, out + (size_t)h * D + lane + 64 * i);
            else
              __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x[i] * kPScale), ro, (h * D + lane + 64 * i) * 4,
                                                    me * A.hc * D * 4, kCoherent);
          }
          if (!whole && lane == 0)
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{mr, lr * kPScale}), rm, h * 8, me * A.hc * 8,
                                                  kCoherent);
        }
      }
      if (!whole) {
        __builtin_amdgcn_s_waitcnt(0);  // this wave's stores are complete before the workgroup is counted
        __syncthreads();
        if (tid == 0) {
          const int old = __hip_atomic_fetch_add(a.ws_cnt + u, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (old == np - 1) __hip_atomic_store(a.ws_cnt + u, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          flag = old == np - 1;
        }
        __syncthreads();
        if (flag != 0) {
          // the workgroup counted last merges the pieces (page_attention.py:2006-2059):
          // NE float4 elements; with fewer than 256, groups of threads share the pieces
          const int NE = nh * (D / 4);
          const int ng = NE < 256 ? 256 / NE : 1;
          for (int e0 = 0; e0 < NE; e0 += 256) {
            const int e = NE < 256 ? tid % NE : e0 + tid;
            const int grp = NE < 256 ? tid / NE : 0;
            const bool act = e < NE && grp < ng;
            const int h = act ? 4 * e / D : 0;
            float M = -INFINITY, L = 0.f;
            f32x4 O = {0.f, 0.f, 0.f, 0.f};
            constexpr int NB = 4;  // pieces in flight per thread
            if (act) {
              for (int p0 = grp; p0 < np; p0 += NB * ng) {
                f32x4 o[NB];
                f32x2 ml[NB];
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                  const int p = min(p0 + k * ng, np - 1);
                  // (the piece's offset in the per-lane part: groups read different pieces)
                  o[k] = __builtin_bit_cast(
                      f32x4, __builtin_amdgcn_raw_buffer_load_b128(ro, (p * A.hc * D + 4 * e) * 4, 0, kCoherent));
                  ml[k] = __builtin_bit_cast(
                      f32x2, __builtin_amdgcn_raw_buffer_load_b64(rm, (p * A.hc + h) * 8, 0, kCoherent));
                }
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                  if (p0 + k * ng >= np) continue;
                  if (ml[k].x == -INFINITY) {  // no live key, or scores of NaN only
                    L += ml[k].y;
                    continue;
                  }
                  const float Mn = fmaxf(M, ml[k].x);
                  const float fo = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M - Mn);
                  const float fp = __builtin_amdgcn_exp2f(ml[k].x - Mn);
                  O = O * fo + o[k] * fp;
                  L = L * fo + ml[k].y * fp;
                  M = Mn;
                }
              }
            }
            if (ng > 1) {  // the groups' states through LDS (element-major: 6 floats each)
              if (act) {
                float* x = xo + (grp * NE + e) * 6;
                x[0] = M;
                x[1] = L;
#pragma unroll
                for (int k = 0; k < 4; ++k) x[2 + k] = O[k];
              }
              __syncthreads();
              if (act && grp == 0) {
                for (int q = 1; q < ng; ++q) {
                  const float* x = xo + (q * NE + e) * 6;
                  if (x[0] == -INFINITY) {
                    L += x[1];
                    continue;
                  }
                  const float Mn = fmaxf(M, x[0]);
                  const float fo = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M - Mn);
                  const float fp = __builtin_amdgcn_exp2f(x[0] - Mn);
#pragma unroll
                  for (int k = 0; k < 4; ++k) O[k] = O[k] * fo + x[2 + k] * fp;
                  L = L * fo + x[1] * fp;
                  M = Mn;
                }
              }
            }
            if (act && grp == 0) write4(O, L, out + 4 * e);
          }
        }
      }
      clear();
      seg0 = g + 1;
      if (nxt.has) load_q(nxt.s, nxt.y);
      // waited for here: a query load outstanding on this path only would make every item's first
      // product wait for all loads in flight
#pragma unroll
      for (int w = 0; w < P::KS; ++w) {
        u32x4 x = __builtin_bit_cast(u32x4, qB[w]);
        asm volatile("" : "+v"(x));
        qB[w] = __builtin_bit_cast(Op, x);
      }
    }
    cur = nxt;
    nxt = n2;
    lc = ln;
    ln = l2;
  }
}

// (D = 256 holds 64 words of V and 64 of K per lane: one workgroup per compute unit, no spills)
template <class C, int D>
__global__ __launch_bounds__(256, D == 256 ? 1 : 2) void decode_mfma(DecodeMfmaArgs a) {
  decode_mfma_body<C, D>(a, blockIdx.x, gridDim.x);
}

}  // namespace emx
