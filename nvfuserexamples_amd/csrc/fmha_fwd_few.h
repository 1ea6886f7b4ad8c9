// Forward kernel for launches of few workgroups (no mask, a per-key mask and / or the causal mask, valid key counts; no dropout or
// the Philox rule): the four (eight, one) waves of a workgroup share 32 queries and take their blocks of keys in turn.
//
// The other forward kernels give a workgroup 128 queries or more and walk its keys one tile after the other.  Where that makes
// fewer workgroups than the chip has room for, the launch lasts as long as one workgroup's row of tiles, about 1.5 us each for a
// wave that has its SIMD to itself.  Here the workgroups are four times as many and each wave has a quarter of a row.  A wave
// stages its own blocks (global -> registers -> LDS, one stage, so no barrier: LDS serves a wave's requests in order, and
// the next block's rows are on their way in registers while one is worked on); at the end the four partial rows meet in LDS.
// K and V are read once per 32 queries, which is what large launches cannot afford.  The rule and both sides' times are at few_waves in
// fmha_capi.hip; us, before -> now: BH 12 821 x 856 d 96 26.2 -> 15.5, BH 4 S 7937 d 128
// causal 139.4 -> 115.3, BH 1 S 2304 d 32 key counts 29.9 -> 11.3.
//
// A build with one wave per workgroup serves short key ranges of any number of heads: the other kernels' workgroups of 128 queries are mostly
// padding there, and their pipelines have nothing to run ahead of (BH 2460 S 24 d 32 22.0 -> 8.1 us, BH 1690 17 x 24 d 96 with dropout
// 34.0 -> 8.0, BH 3531 S 52 d 128 packed with dropout 87.6 -> 43.5, BH 3273 S 16 d 256 packed 96.1 -> 32.0).
//
// A build for pieces of the key range (few_chunk in fmha_capi.hip) serves launches whose 32-query groups leave most compute units idle, or
// each with a long row: a head is a (head, piece), the mask and the key counts stay the whole range's, and the normalised rows go out
// in fp32 with their log-sum-exps for a second launch to merge.  Bound by the piece's chain of blocks and the merge's 5 us; us, whole or in
// plain pieces -> so: BH 17 19 x 1 698 d 256 54.7 -> 16.8, BH 1 12 x 1 568 d 80 38.1 -> 9.5, BH 2 613 x 2 785 d 128 55.3 -> 16.2; 743 drawn
// launches (1 to 300 heads, 5 to 1 000 queries, 300 to 50 000 keys) 1.64 times as fast (least 0.92).
//
// Softmax as in fmha_fwd_mid.h: scores are scaled in fp32, the reference follows the row's maximum only where that has run ahead
// by more than 2^8, row sums are those of the rounded P.
#pragma once
#include "fmha_fwd_kernel.h"

namespace fmha {

template <int D, int NW_> struct FewCfg {
  static constexpr int BK = D <= 64 ? 64 : 32; // keys per block: what a lane holds of the next one fits beside the rest in 256 registers
  static constexpr int NW = NW_, NT = NW * 64, QT = 32;
  static constexpr int TILEB = BK * tile_cols(D) * 2;
  static constexpr int LDS_M = 2 * TILEB;            // (in a wave's stage) mask terms of the block's keys
  static constexpr int STAGEB = LDS_M + BK * 4;
  static constexpr int LDS_MERGE = NW * 32 * D * 4;  // over the stages: the waves' outputs
  static constexpr int LDS_ROWS = NW * STAGEB > LDS_MERGE ? NW * STAGEB : LDS_MERGE; // their rows' references and sums
  static constexpr int LDS_LAST = LDS_ROWS + NW * 2 * 32 * 4; // per wave: keys up to the last that is not hard-masked
  static constexpr int LDS_BYTES = LDS_LAST + NW * 4;
};

// PIECES: a head is a piece of the key range (FwdArgs::pieces; the mask and the key counts are the whole range's); o gets fp32 rows [bh, sq, dcols].
template <typename T, int D, int NW, int MASK, bool CAUSAL, int DROP, bool STRIDED, bool PIECES = false>
__global__ __launch_bounds__((FewCfg<D, NW>::NT), D == 256 ? 1 : 2) void fmha_fwd_few_kernel(const FwdArgs a) {
  using C = FewCfg<D, NW>;
  using E = Elem<T>;
  using v8 = typename E::v8;
  using RW = Rows<STRIDED, D>;
  constexpr int KS = D / 16, DB = D / 32, BK = C::BK, NSB = BK / 32;
  constexpr int CPT = BK * tile_cols(D) / 8 / 64; // 16-byte chunks per lane and block of K (of V)
  constexpr float NEG_INF = -__builtin_inff();

  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, ql = l & 31, h = l >> 5;

  // Of every 8 heads each XCD gets one with all its query tiles; causal: the longest tiles of all heads first.
  const int b0 = blockIdx.x, grouped = (a.bh & ~7) * a.nqt;
  int bh, qt;
  if (CAUSAL) {
    const int lg = head_groups_log2(a.bh), m = by_length(b0, (int)gridDim.x, lg), heads = a.bh >> lg;
    qt = m / heads;
    bh = ((m - qt * heads) << lg) + (b0 & ((1 << lg) - 1));
    qt = a.nqt - 1 - qt;
  } else {
    bh = b0 < grouped ? b0 / (8 * a.nqt) * 8 + (b0 & 7) : b0 / a.nqt;
    qt = b0 < grouped ? (b0 >> 3) % a.nqt : b0 % a.nqt;
  }
  const int q0 = qt * C::QT, q = q0 + ql;
  int piece = 0, head = bh;
  if constexpr (PIECES) { // (the first pieces of all heads, then the second ones: the last ones of short heads are empty, and else lie on few XCDs)
    const int heads = a.bh / a.pieces;
    piece = bh / heads;
    head = bh - piece * heads;
    bh = head * a.pieces + piece;
  }
  const T *Qr = (const T *)a.q + RW::head(a.mq, head, a.sq) + (size_t)(q < a.sq ? q : a.sq - 1) * RW::ss(a.mq) + h * 8;
  int kend = visible_keys<STRIDED>(a, head, piece);
  const int sk = kend > 0 ? kend : 1; // rows that may be read: those behind the head's count hold anything (a piece behind it: its first row)
  const T *Kb = (const T *)a.k + RW::head(a.mk, head, a.sk) + (PIECES ? piece * a.piece_stride : 0);
  const T *Vb = (const T *)a.v + RW::head(a.mv, head, a.sk) + (PIECES ? piece * a.piece_stride : 0);
  const T *mkey = MASK == kMaskPerKey ? (const T *)a.mask + (size_t)(head / a.mask_div) * a.mask_sb + (PIECES ? piece * a.sk : 0) : nullptr;
  const uint32_t ss = RW::ss(a.mk);
  const int cols = RW::cols(a);

  if (CAUSAL && kend > q0 + 32) kend = q0 + 32;

  // ---- a wave's block: its keys are b * BK .., chunk slot l + 64 i of the swizzled panel layout is this lane's
  char *stage = lds + w * C::STAGEB;
  float *fM = (float *)(stage + C::LDS_M);
  u32x4 kst[CPT], vst[CPT];
  T mraw = (T)0.f;
  auto load = [&](int b) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      int row, col;
      TileCopy<T, D, BK, 64>::slot(l + i * 64, row, col);
      int r = b * BK + row;
      r = r < sk ? r : sk - 1; // rows past the end: their scores get -inf, and P = 0 meets finite values
      const bool live = col * 8 < cols;
      const uint32_t at = (uint32_t)r * ss + (uint32_t)(live ? col * 8 : 0);
      kst[i] = *(const u32x4 *)(Kb + at);
      vst[i] = *(const u32x4 *)(Vb + at);
    }
    if (MASK == kMaskPerKey) mraw = mkey[b * BK + (l & (BK - 1)) < sk ? b * BK + (l & (BK - 1)) : sk - 1];
  };
  auto store = [&](int b) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      int row, col;
      TileCopy<T, D, BK, 64>::slot(l + i * 64, row, col);
      const bool live = col * 8 < cols;
      *(u32x4 *)(stage + (l + i * 64) * 16) = STRIDED ? chunk_or_zero(kst[i], live) : kst[i];
      *(u32x4 *)(stage + C::TILEB + (l + i * 64) * 16) = STRIDED ? chunk_or_zero(vst[i], live) : vst[i];
    }
    if (MASK == kMaskPerKey && l < BK) fM[l] = b * BK + l < kend ? fmaf((float)mraw, a.mask_a, a.mask_b) : NEG_INF;
  };
  auto fence = [&]() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };

  load(w);
  v8 qreg[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const bool live = ks * 16 + h * 8 < cols;
    qreg[ks] = as_v8<T>(STRIDED ? chunk_or_zero(*(const u32x4 *)(live ? Qr + ks * 16 : Qr), live) : *(const u32x4 *)(Qr + ks * 16));
  }
  if (MASK == kMaskPerKey && !(a.flags & kFwdFlagNoTrim)) { // hard-masked keys at the end need not be visited
    int *last = (int *)(lds + C::LDS_LAST), n = 0;
    for (int j = w * 64; j < kend; j += NW * 64) {
      const float mk = fmaf((float)mkey[j + l < sk ? j + l : sk - 1], a.mask_a, a.mask_b);
      const unsigned long long up = __builtin_amdgcn_ballot_w64(j + l < kend && mk > -9000.f * FMHA_LOG2E);
      if (up) n = j + 64 - (int)__builtin_clzll(up);
    }
    if (l == 0) last[w] = n;
    __syncthreads();
    n = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) n = last[i] > n ? last[i] : n;
    if (n) kend = __builtin_amdgcn_readfirstlane(n); // (a row without any live key keeps all its keys)
  }
  const int nkb = (kend + BK - 1) / BK;

  PanelLane pl;
  pl.init(l);
  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;
  float mref = NEG_INF, sum = 0.f, sum2 = 0.f; // softmax reference (of the scores in log2 units); row sum of the rounded P

  store(w);
  if (w + NW < nkb) load(w + NW);
  fence();
  for (int b = w; b < nkb; b += NW) {
    f32x16 x[NSB];
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int r = 0; r < 16; ++r) x[sb][r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb) x[sb] = E::mfma(panel_read_rows<T, BK>(stage, pl, sb, ks), qreg[ks], x[sb]);
    float mx = NEG_INF;
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb) {
      if (MASK == kMaskPerKey) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 mk = *(const f32x4 *)(fM + sb * 32 + 8 * g + 4 * h);
#pragma unroll
          for (int t = 0; t < 4; ++t) x[sb][4 * g + t] = fmaf(x[sb][4 * g + t], a.scale_l2, mk[t]);
        }
      } else if (b * BK + sb * 32 + 32 > kend) {
#pragma unroll
        for (int r = 0; r < 16; ++r) x[sb][r] = b * BK + sb * 32 + 8 * (r >> 2) + 4 * h + (r & 3) < kend ? x[sb][r] * a.scale_l2 : NEG_INF;
      } else { // (not folded into the exponent: key counts give the bits of the mask that hides the same keys)
#pragma unroll
        for (int r = 0; r < 16; ++r) x[sb][r] *= a.scale_l2;
      }
      if (CAUSAL && b * BK + sb * 32 + 31 > q0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) x[sb][r] = b * BK + sb * 32 + 8 * (r >> 2) + 4 * h + (r & 3) <= q ? x[sb][r] : NEG_INF;
      }
#pragma unroll
      for (int r = 0; r < 16; r += 2) mx = max3(mx, x[sb][r], x[sb][r + 1]);
    }
    mx = xhalf_max(mx);
    // the reference follows the row's maximum only where that has run ahead by more than 2^8
    if (__builtin_amdgcn_ballot_w64(mx > mref + 8.f)) {
      const float to = mx > mref + 8.f ? mx : mref, f = mref == NEG_INF ? 0.f : fast_exp2(mref - to);
      sum *= f;
      sum2 *= f;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= f;
      mref = to;
    }
    const float ref = mref == NEG_INF ? 0.f : mref;
    v8 pf[NSB][2];
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb) {
      uint32_t wd[4];
      if (DROP == 1) drop_words_q(a.drop, (uint32_t)bh, (uint32_t)q, (uint32_t)(b * BK + sb * 32), h, l, wd);
#pragma unroll
      for (int c = 0; c < 2; ++c) { // keys 16 c + 8 g + 4 h + t, g = 0, 1
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float p = fast_exp2(x[sb][8 * c + e] - ref);
          pf[sb][c][e] = (T)p;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sum_pair<T>(pf[sb][c], i, sum, sum2);
        if (DROP == 1) {
          u32x4 u = as_u32x4(pf[sb][c]);
          const uint32_t thr = ((a.drop.thr - 1u) & 0xffffu) * 0x00010001u; // (thr = 0 gives -1: everything kept)
          uint32_t r0 = u.x, r1 = u.y, r2 = u.z, r3 = u.w;
          drop_apply_pk4(wd[2 * c], thr, r0, r1);
          drop_apply_pk4(wd[2 * c + 1], thr, r2, r3);
          pf[sb][c] = as_v8<T>(u32x4{r0, r1, r2, r3});
        }
      }
    }
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] = E::mfma(panel_read_transposed<T, BK>(stage + C::TILEB, pl, sb, db, c), pf[sb][c], o[db]);
    fence();
    if (b + NW < nkb) {
      store(b + NW);
      if (b + 2 * NW < nkb) load(b + 2 * NW);
    }
    fence();
  }

  if constexpr (NW == 1) {
    sum = xhalf_sum(sum + sum2);
    if (q >= a.sq) return;
    const float out = sum > 0.f ? a.drop_scale / sum : 0.f;
    T *Or = (T *)a.o + RW::head(a.mo, bh, a.sq) + (size_t)q * RW::ss(a.mo);
#pragma unroll
    for (int db = 0; db < DB; ++db) store_acc_block_row<T>(Or + db * 32, o[db], out, h, cols - db * 32);
    if (a.lse && h == 0) a.lse[(size_t)bh * a.sq + q] = sum > 0.f ? (mref + fast_log2(sum)) * FMHA_LN2 : NEG_INF;
    return;
  }
  // ---- the waves' partial rows meet in LDS; wave i takes the columns 32 i .., 32 (i + 4) .. of the head
  sum = xhalf_sum(sum + sum2);
  __syncthreads();
  f32x4 *part = (f32x4 *)lds;
  float *rows = (float *)(lds + C::LDS_ROWS);
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      part[((w * DB + db) * 4 + g) * 64 + l] = f32x4{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]};
  if (h == 0) {
    rows[(w * 2 + 0) * 32 + ql] = mref;
    rows[(w * 2 + 1) * 32 + ql] = sum;
  }
  __syncthreads();
  if (w >= DB || q >= a.sq) return;
  float top = NEG_INF, wt[NW], lt = 0.f;
#pragma unroll
  for (int j = 0; j < NW; ++j) top = fmaxf(top, rows[j * 2 * 32 + ql]);
  const float ref = top == NEG_INF ? 0.f : top;
#pragma unroll
  for (int j = 0; j < NW; ++j) {
    wt[j] = fast_exp2(rows[j * 2 * 32 + ql] - ref);
    lt += wt[j] * rows[(j * 2 + 1) * 32 + ql];
  }
  const float out = lt > 0.f ? a.drop_scale / lt : 0.f;
  T *Or = (T *)a.o + RW::head(a.mo, bh, a.sq) + (size_t)q * RW::ss(a.mo);
#pragma unroll
  for (int d0 = 0; d0 < DB; d0 += NW) {
    const int db = d0 + w;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int j = 0; j < NW; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 v = part[((j * DB + db) * 4 + g) * 64 + l];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[4 * g + i] = fmaf(wt[j], v[i], acc[4 * g + i]);
      }
    if constexpr (PIECES) {
      float *dst = (float *)a.o + ((size_t)bh * a.sq + q) * cols + db * 32 + 4 * h;
#pragma unroll
      for (int g = 0; g < 4; ++g)
        if (db * 32 + 8 * g < cols) *(f32x4 *)(dst + 8 * g) = f32x4{acc[4 * g] * out, acc[4 * g + 1] * out, acc[4 * g + 2] * out, acc[4 * g + 3] * out};
    } else {
      store_acc_block_row<T>(Or + db * 32, acc, out, h, cols - db * 32);
    }
  }
  if (a.lse && h == 0 && w == 0) a.lse[(size_t)bh * a.sq + q] = lt > 0.f ? (ref + fast_log2(lt)) * FMHA_LN2 : NEG_INF;
}

} // namespace fmha
