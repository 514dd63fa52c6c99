// Ragged / causal paged attention (sequences with more than one query token) over
// token-major caches [nb, bs, Hkv, D]: unquantized fp16 / bf16 and FP8 (E4M3, one
// fp32 scale per page), head_dim 64, 128 or 256, pages of a multiple of 8 tokens, any
// GQA ratio up to 128.  MFMA.
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
// Tiles of many keys are cut into up to kPrefillParts parts, merged in part order by the
// wave that arrives last (as in prefill_affine.hpp).
//
// Bound by the matrix and vector units together (the probability parts double the PV
// products of fp16, triple those of bf16).  It took over from paged_generic, one wave per
// (token, kv head) on the VALU: four 512-token chunks beside 28 decode rows, bf16, D 128,
// pages of 16: 20.7 ms -> 130 us; a 1531-token prompt, fp16, D 256, window 700: 9.7 ms ->
// 53 us.
#pragma once

#include "decode_mfma.hpp"
#include "prefill_affine.hpp"

namespace emx {

struct PrefillMfmaArgs {
  DecodeArgs d;     // kc / vc: the caches; nt, ws_* unused
  uint32_t inv_bs;  // ceil(2^32 / bs)
  int min_q;        // sequences with fewer query tokens are not taken
  int tokb;         // query tokens per tile: columns / HG
  int nparts, max_items;
  int* ws_cnt;      // [max_items * Hkv * 4], zero before and after every launch
  float* ws_part;   // [max_items * Hkv][kPrefillParts][part bytes]
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
  constexpr int oTcum = 0, oWred = lds_next(oTcum, 4 * (kMaxSeqs + 1)), oKe = lds_next(oWred, 16);
  constexpr int oVe = lds_next(oKe, 2 * NT * P::KSTR), oKsf = lds_next(oVe, 2 * NT * P::VSTR);
  constexpr int oVsf = lds_next(oKsf, 4 * NT), oEnd = lds_next(oVsf, 4 * NT);
  static_assert(oEnd <= kArenaBytes, "LDS arena too small");
  int(&tcum)[kMaxSeqs + 1] = lds_at<int[kMaxSeqs + 1]>(oTcum);
  int(&wred)[4] = lds_at<int[4]>(oWred);
  uint16_t* ke = &lds_at<uint16_t>(oKe);  // [key][KSTR]
  uint16_t* ve = &lds_at<uint16_t>(oVe);  // [key][VSTR]
  float* ksf = &lds_at<float>(oKsf);      // FP8: key / value scale of each key
  float* vsf = &lds_at<float>(oVsf);

  // ---- work item: tiles per sequence, scanned by the workgroup; the last tile (most keys) first
  {
    const int ch = (a.S + 255) / 256, s0 = tid * ch;
    int tsum = 0;
    for (int i = 0; i < ch; ++i) {
      const int si = s0 + i;
      if (si >= a.S) break;
      const int ql = a.qsl[si + 1] - a.qsl[si];
      const int n = ql >= A.min_q ? (ql + A.tokb - 1) / A.tokb : 0;
      tcum[si] = n;  // the count for now
      tsum += n;
    }
    int x = tsum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) wred[tid >> 6] = x;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < (tid >> 6); ++w) base += wred[w];
    int run = base + x - tsum;
    for (int i = 0; i < ch; ++i) {
      const int si = s0 + i;
      if (si >= a.S) break;
      const int n = tcum[si];
      tcum[si] = run;
      run += n;
    }
    if (tid == 255) tcum[a.S] = base + x;
  }
  __syncthreads();
  const int ntiles = tcum[a.S];
  const int kvh = bid % a.Hkv;
  const int part = (bid / a.Hkv) % A.nparts;
  const int item = bid / a.Hkv / A.nparts;
  if (item >= ntiles) return;
  int s = 0;
  for (int c = 0; c < a.S; c += 64) {
    const int si = c + lane;
    s += __builtin_popcountll(__ballot(si < a.S && tcum[si + 1] <= item));
  }
  s = __builtin_amdgcn_readfirstlane(s);
  const int nt_s = tcum[s + 1] - tcum[s];
  const int tile = __builtin_amdgcn_readfirstlane(nt_s - 1 - (item - tcum[s]));
  const int q0 = __builtin_amdgcn_readfirstlane(a.qsl[s]);
  const int qlen = __builtin_amdgcn_readfirstlane(a.qsl[s + 1]) - q0;
  const int kv_len = __builtin_amdgcn_readfirstlane(min(max(a.kv_lens[s], 0), a.max_blocks * a.bs));
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
    if (t >= A.tokb || ctok[ct] >= qlen) ctok[ct] = -1;  // no such column
    if (ctok[ct] < 0) limit[ct] = -1;
  }
  const int t_last = min(tok_lo + A.tokb, qlen) - 1;
  const int k_hi = min(past + t_last, kv_len - 1);
  const int k_lo = a.window > 0 ? max(0, past + tok_lo - a.window + 1) : 0;
  const int steps_all = k_hi >= 0 ? max(k_hi / NT - k_lo / NT + 1, 0) : 0;
  const int nparts = A.nparts > 1 && item < A.max_items
                         ? max(1, min(A.nparts, (steps_all * NT + kPrefillSplitKeys - 1) / kPrefillSplitKeys))
                         : 1;
  if (part >= nparts) return;
  const int step_lo = k_lo / NT + part * steps_all / nparts;
  const int step_hi = k_lo / NT + (part + 1) * steps_all / nparts - 1;

  // ---- query operands (zeros for absent columns)
  Op qB[CT][P::KS];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const bool ok = ctok[ct] >= 0;
    const QT* qp = reinterpret_cast<const QT*>(a.q) +
                   ((size_t)(q0 + (ok ? ctok[ct] : 0)) * a.Hq + (size_t)kvh * HG + (ok ? chead[ct] : 0)) * D + 8 * jj;
#pragma unroll
    for (int w = 0; w < P::KS; ++w) {
      const u32x4 x = *reinterpret_cast<const u32x4*>(qp + 32 * w);
      qB[ct][w] = __builtin_bit_cast(Op, ok ? x : u32x4{0u, 0u, 0u, 0u});
    }
  }

  // ---- pages: lane l holds the page id of key l of a step (positions past the tile's last key repeat it)
  const char* kbase = reinterpret_cast<const char*>(a.kc) + (size_t)kvh * (D * P::EB);
  const char* vbase = reinterpret_cast<const char*>(a.vc) + (size_t)kvh * (D * P::EB);
  const size_t rowb = (size_t)a.Hkv * D * P::EB;
  const int32_t* bt = a.block_tables + (size_t)s * a.max_blocks;
  auto page_id = [&](const int st) { return bt[page_of(min(st * NT + (lane & (NT - 1)), k_hi), A.inv_bs)]; };
  u32x4 rk[P::NP], rv[P::NP];  // the next step's pieces
  uint64_t okn = 0;            // keys of that step on a valid page
  float psk = 0.f, psv = 0.f;  // FP8: page scales of key `lane` of that step
  auto load_step = [&](const int st, const int blk) {
    const int pos = min(st * NT + (lane & (NT - 1)), k_hi);
    const bool ok = (unsigned)blk < (unsigned)a.nb;
    okn = __ballot(ok);
    const int b = ok ? blk : 0;
    const int row = b * a.bs + (pos - page_of(pos, A.inv_bs) * a.bs);
    if constexpr (C::kFp8) {
      psk = a.kps[b];
      psv = a.vps[b];
    }
#pragma unroll
    for (int n = 0; n < P::NP; ++n) {
      const size_t off = (size_t)__shfl(row, tid / P::PR + n * P::RP, 64) * rowb + 16 * (tid % P::PR);
      rk[n] = *reinterpret_cast<const u32x4*>(kbase + off);
      rv[n] = *reinterpret_cast<const u32x4*>(vbase + off);
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
  int vexp = 0;  // FP8: acc holds the sum / 2^vexp

  int blk1 = 0;
  if (step_lo <= step_hi) {
    load_step(step_lo, page_id(step_lo));
    blk1 = page_id(min(step_lo + 1, step_hi));
  }
  for (int st = step_lo; st <= step_hi; ++st) {
    __syncthreads();  // the previous step's tiles are no longer read
#pragma unroll
    for (int n = 0; n < P::NP; ++n) {
      const int r = tid / P::PR + n * P::RP, c = (tid % P::PR) * (16 / P::EB);
      put_piece<C>(ke + r * P::KSTR + c, rk[n]);
      put_piece<C>(ve + r * P::VSTR + c, rv[n]);
    }
    const uint64_t okm = okn;
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
        f32x4 c[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) c[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < P::KS; ++w) {
          const Op K = *reinterpret_cast<const Op*>(kr + 32 * w);
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) c[ct] = mfma_op(K, qB[ct][w], c[ct]);
        }
        f32x4 ks4 = {1.f, 1.f, 1.f, 1.f};
        if constexpr (C::kFp8) ks4 = *reinterpret_cast<const f32x4*>(ksf + 32 * h + 16 * t + 4 * jj);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[ct][4 * t + r] = C::kFp8 ? c[ct][r] * ks4[r] : c[ct][r];
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
            const int k = 16 * (e >> 2) + 4 * jj + (e & 3);
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
        split_p(sc[ct], pB[ct]);
      }

      // ---- O^T += V^T P^T
#pragma unroll
      for (int b = 0; b < P::SB; ++b) {
        const u32x2 v0 = read_tr(ve, P::VSTR, 32 * h, 16 * b, col, jj);
        const u32x2 v1 = read_tr(ve, P::VSTR, 32 * h + 16, 16 * b, col, jj);
        const Op V = __builtin_bit_cast(Op, u32x4{v0[0], v0[1], v1[0], v1[1]});
#pragma unroll
        for (int k = 0; k < C::kParts; ++k)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) acc[ct][b] = mfma_op(V, pB[ct][k], acc[ct][b]);
      }
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
        uniform_rsrc(reinterpret_cast<uint8_t*>(A.ws_part) + (size_t)u * kPrefillParts * P::PARTB,
                     kPrefillParts * P::PARTB);
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
    const size_t orow = ((size_t)(q0 + (ok ? ctok[ct] : 0)) * a.Hq + (size_t)kvh * HG + (ok ? chead[ct] : 0)) * D;
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
    // columns that are not finite: again in fp32, key by key (attend_row)
    uint64_t todo = __ballot(bad && ok);
    todo = (todo | (todo >> 16) | (todo >> 32) | (todo >> 48)) & 0xFFFFu;
    while (todo) {
      const int c = __builtin_ctzll(todo);
      todo &= todo - 1;
      const int t = __builtin_amdgcn_readlane(ctok[ct], c), hh = __builtin_amdgcn_readlane(chead[ct], c);
      const int k0 = __builtin_amdgcn_readlane(start[ct], c), k1 = __builtin_amdgcn_readlane(limit[ct], c) + 1;
      const size_t ro = ((size_t)(q0 + t) * a.Hq + (size_t)kvh * HG + hh) * D;
      float lr, x[D / 64];
      attend_row<C, D>(a, s, kvh, reinterpret_cast<const QT*>(a.q) + ro, k0, k1, lr, x, lane);
      const float li = lr > 0.f ? 1.f / lr : 0.f;
#pragma unroll
      for (int i = 0; i < D / 64; ++i) from_f32(x[i] * li, reinterpret_cast<QT*>(a.out) + ro + lane + 64 * i);
    }
  }
}

// Workgroups [0, ndec) decode the single-token rows (decode_mfma.hpp), the rest take the
// query tiles: as unified.hpp does, the page streams run beside the matrix work.
template <class C, int D, int CT>
__global__ __launch_bounds__(256, D > 128 && CT == 2 ? 1 : 2) void mixed_mfma(PrefillMfmaArgs p, DecodeMfmaArgs d,
                                                                             int ndec) {
  if ((int)blockIdx.x < ndec)
    decode_mfma_body<C, D>(d, blockIdx.x, ndec);
  else
    prefill_mfma_body<C, D, CT>(p, (int)blockIdx.x - ndec);
}

}  // namespace emx
