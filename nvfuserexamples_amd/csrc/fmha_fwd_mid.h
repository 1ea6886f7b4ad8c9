// Forward kernel for 129 to 256 keys (head dim 64; no mask, a per-key mask and / or the causal mask, valid key counts; no dropout
// or the Philox rule): a head's K and V in LDS, copied once for up to 256 queries.
//
// The pipelined kernel (fmha_fwd_pipe.h) works on items of 128 queries and tiles of 64 keys: at 197 rows it computes 256 x 256
// scores for 197 x 197, and every 128 queries copy K and V again.  Here a wave owns 32 queries and walks blocks of 32 keys, as
// many as exist, are not hard-masked at the end and, under the causal mask, are seen; behind the one barrier, when the copies have
// landed, the waves run free.  Two workgroups share a compute unit (65 KB of LDS, eight waves each, at most 128 registers): one
// computes while the other loads or stores.  The next block's scores are formed beside this one's exponentials; the softmax
// reference follows the row's maximum only where that has run ahead by more than 2^8 (P stays within both element types); row
// sums are those of the rounded P.  Scores are scaled in fp32 (the pipelined kernel rounds Q * scale), so errors against 64 bits
// are smaller: 197 keys fp16 3.3e-5 for 4.1e-5 rms, scores three times as large 5.3e-4 for 1.6e-3.
//
// What bounds it: memory where workgroups overlap (BH 2048 S 197: 207 MB in 43 us, 4.8 TB/s, a copy's rate 5.0), elsewhere a
// workgroup's own chain of load, blocks and store.  Measured on rotated inputs (us, pipelined kernel -> this): BH 768 S 197 from
// packed rows 28.3 -> 25.7, folded under a padding mask with dropout 32.6 -> 25.0; BH 512 S 161 16.1 -> 14.6; BH 100 S 161 padding
// mask and dropout 10.4 -> 7.2; 8556 launches of its range 1.20 times as fast in the geometric mean.  It is behind with all eight
// key blocks in use and nothing masked (BH 512 S 240 17.3 -> 20.1, with dropout 22.0 -> 24.6) and where the pipelined kernel's rounds
// come out full (BH 768 S 197 folded 23.1 -> 23.9): mid_wanted of the dispatch has the line.
//
// NW: waves per workgroup.  8, 256 queries, or 4 where that still leaves a compute unit to each workgroup (BH 24 S 200 with
// dropout 9.9 us with eight, 7.3 with four; BH 300 S 160 9.6 / 11.8).
#pragma once
#include "fmha_fwd_kernel.h"

namespace fmha {

template <int NW_> struct MidCfg {
  static constexpr int D = 64, NW = NW_, NT = NW * 64, QT = NW * 32, SKMAX = 256;
  static constexpr int BT = 64, TILEB = BT * D * 2; // rows per copied tile
  static constexpr int BLOCKB = 32 * kPanelRowB;    // 32 keys
  static constexpr int LDS_V = SKMAX * kPanelRowB, LDS_M = 2 * LDS_V;
  static constexpr int LDS_BYTES = LDS_M + SKMAX * 4;
};

template <typename T, int NW, int MASK, bool CAUSAL, int DROP, bool STRIDED>
__global__ __launch_bounds__(MidCfg<NW>::NT) __attribute__((amdgpu_waves_per_eu(4, 4))) void fmha_fwd_mid_kernel(const FwdArgs a) {
  using C = MidCfg<NW>;
  using E = Elem<T>;
  using v8 = typename E::v8;
  constexpr int D = C::D, KS = D / 16, DB = D / 32;
  constexpr float NEG_INF = -__builtin_inff();
  using RW = Rows<STRIDED, D>;

  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, ql = l & 31, h = l >> 5;

  // one XCD (one L2) owns a contiguous range of heads
  int bid = blockIdx.x;
  const int nb = gridDim.x;
  if ((nb & 7) == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);
  const int bh = a.nqt == 1 ? bid : bid / a.nqt;
  const int q0w = (a.nqt == 1 ? 0 : bid - bh * a.nqt) * C::QT + __builtin_amdgcn_readfirstlane(w) * 32;
  const T *Qb = (const T *)a.q + RW::head(a.mq, bh, a.sq);
  const T *Kb = (const T *)a.k + RW::head(a.mk, bh, a.sk);
  const T *Vb = (const T *)a.v + RW::head(a.mv, bh, a.sk);

  // ---- every request up front
  float *fM = (float *)(lds + C::LDS_M); // mask term of key k in log2 units, -inf from the first invisible key on
  int kend = visible_keys<STRIDED>(a, bh, 0);
  static_assert(C::NT >= C::SKMAX, "a thread per key");
  T mraw = (T)0.f;
  if (MASK == kMaskPerKey && tid < C::SKMAX) {
    const int mhead = a.mask_div == 1 ? bh : bh / a.mask_div;
    mraw = ((const T *)a.mask + (size_t)mhead * a.mask_sb)[tid < a.sk ? tid : a.sk - 1];
  }
  TileCopy<T, D, C::BT, C::NT> tcopy;
  tcopy.init(tid, RW::ss(a.mk));
  const uint32_t lds0 = lds_address(lds);
  const int rows = kend > 0 ? kend : 1; // rows behind the head's count hold anything
  const int nt = (rows + C::BT - 1) / C::BT;
  for (int t = 0; t < nt; ++t) tcopy.issue(Kb, t * C::BT, rows, lds0 + (uint32_t)(t * C::TILEB), tid);
  for (int t = 0; t < nt; ++t) tcopy.issue(Vb, t * C::BT, rows, lds0 + (uint32_t)(C::LDS_V + t * C::TILEB), tid);
  const int q = q0w + ql;
  v8 qreg[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    qreg[ks] = as_v8<T>(*(const u32x4 *)(Qb + (size_t)(q < a.sq ? q : a.sq - 1) * RW::ss(a.mq) + ks * 16 + h * 8));
  dma_wait_all();
  if (MASK == kMaskPerKey && tid < C::SKMAX) fM[tid] = tid < kend ? fmaf((float)mraw, a.mask_a, a.mask_b) : NEG_INF;
  __syncthreads();
  if (q0w >= a.sq) return;

  if (MASK == kMaskPerKey && !(a.flags & kFwdFlagNoTrim)) { // hard-masked keys at the end need not be visited
    int last = -1;
#pragma unroll
    for (int c = 0; c < C::SKMAX / 64; ++c) {
      const unsigned long long bal = __builtin_amdgcn_ballot_w64(fM[c * 64 + l] > -9000.f * FMHA_LOG2E);
      if (bal) last = c * 64 + 63 - __builtin_clzll(bal);
    }
    if (last >= 0) kend = last + 1; // (a row without any live key keeps all its keys)
  }
  int nkb = (kend + 31) / 32;
  if (CAUSAL && nkb > q0w / 32 + 1) nkb = q0w / 32 + 1;

  PanelLane pl;
  pl.init(l);
  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;
  float mref = NEG_INF, sum = 0.f; // softmax reference (of the scores in log2 units); row sum of the rounded P

  // Scores of a block and their row maximum: in log2 units with their mask term (MASK), or as they are, the scale applied with
  // the reference.
  auto scores = [&](int b) -> f32x16 {
    f32x16 x;
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) x = E::mfma(panel_read_rows<T, 32>(lds + b * C::BLOCKB, pl, 0, ks), qreg[ks], x);
    return x;
  };
  auto masked_max = [&](int b, f32x16 &x) -> float {
    if (MASK == kMaskPerKey) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 mk = *(const f32x4 *)(fM + b * 32 + 8 * g + 4 * h);
#pragma unroll
        for (int t = 0; t < 4; ++t) x[4 * g + t] = fmaf(x[4 * g + t], a.scale_l2, mk[t]);
      }
    } else if (b * 32 + 32 > kend) {
#pragma unroll
      for (int r = 0; r < 16; ++r) x[r] = b * 32 + 8 * (r >> 2) + 4 * h + (r & 3) < kend ? x[r] : NEG_INF;
    }
    if (CAUSAL && b * 32 == q0w) {
#pragma unroll
      for (int r = 0; r < 16; ++r) x[r] = 8 * (r >> 2) + 4 * h + (r & 3) <= ql ? x[r] : NEG_INF;
    }
    float mx = NEG_INF;
#pragma unroll
    for (int r = 0; r < 16; r += 2) mx = max3(mx, x[r], x[r + 1]);
    mx = xhalf_max(mx);
    return MASK == kMaskPerKey ? mx : mx * a.scale_l2;
  };
  // The next block's scores are formed beside this one's exponentials.
  f32x16 x = scores(0);
  for (int b = 0; b < nkb; ++b) {
    const float mx = masked_max(b, x);
    // the reference follows the row's maximum only where that has run ahead by more than 2^8
    if (__builtin_amdgcn_ballot_w64(mx > mref + 8.f)) {
      const float to = mx > mref + 8.f ? mx : mref, f = mref == NEG_INF ? 0.f : fast_exp2(mref - to);
      sum *= f;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= f;
      mref = to;
    }
    const float ref = mref == NEG_INF ? 0.f : mref;
    const f32x16 xn = scores(b + 1 < nkb ? b + 1 : b);
    uint32_t wd[4];
    if (DROP == 1) drop_words_q(a.drop, (uint32_t)bh, (uint32_t)q, (uint32_t)(b * 32), h, l, wd);
    v8 pf[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) { // keys 16 c + 8 g + 4 h + t, g = 0, 1
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float p = fast_exp2(MASK == kMaskPerKey ? x[8 * c + e] - ref : fmaf(x[8 * c + e], a.scale_l2, -ref));
        pf[c][e] = (T)p;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) sum = dot2_ones<T>(pf[c], i, sum);
      if (DROP == 1) {
        u32x4 u = as_u32x4(pf[c]);
        const uint32_t thr = ((a.drop.thr - 1u) & 0xffffu) * 0x00010001u; // (thr = 0 gives -1: everything kept)
        uint32_t r0 = u.x, r1 = u.y, r2 = u.z, r3 = u.w;
        drop_apply_pk4(wd[2 * c], thr, r0, r1);
        drop_apply_pk4(wd[2 * c + 1], thr, r2, r3);
        pf[c] = as_v8<T>(u32x4{r0, r1, r2, r3});
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int db = 0; db < DB; ++db)
        o[db] = E::mfma(panel_read_transposed<T, 32>(lds + C::LDS_V + b * C::BLOCKB, pl, 0, db, c), pf[c], o[db]);
    x = xn;
  }

  const float lt = xhalf_sum(sum), out = lt > 0.f ? a.drop_scale / lt : 0.f;
  if (q < a.sq) {
    T *Ob = (T *)a.o + RW::head(a.mo, bh, a.sq) + (size_t)q * RW::ss(a.mo);
#pragma unroll
    for (int db = 0; db < DB; ++db) store_acc_block_row<T>(Ob + db * 32, o[db], out, h);
    if (a.lse && h == 0) a.lse[(size_t)bh * a.sq + q] = lt > 0.f ? (mref + fast_log2(lt)) * FMHA_LN2 : NEG_INF;
  }
}

} // namespace fmha
