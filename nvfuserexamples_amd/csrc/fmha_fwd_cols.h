// The reference's operators (a full [.., sq, sk] mask tensor, optionally a dropout tensor and the saved softmax and dropped softmax) with
// a workgroup per 32 queries and a wave per 64 keys.
//
// The streaming kernels give a workgroup 128 queries and walk the keys tile by tile: a launch of few heads is as long as that walk, with
// most compute units idle, and saving keeps one wave per SIMD because a wave holds all of a row's probabilities.  Here a wave has one block of
// 32 queries by 64 keys and everything of it in registers: all its requests go out at once (Q and K straight into the operand
// layout, V as a copy into an LDS tile of its own, mask and dropout rows as whole 128-byte segments), it forms its scores, its own
// maximum m_w and sum s_w, and its part of O = P V, and the waves meet once: every wave then knows
//   M = max m_w, S = sum 2^(m_w - M) s_w,
// adds a share of the partial outputs, and writes its segments of the saved tensors as p 2^(m_w - M) / S, rounded once.
// K and V are read again for every 32 queries, from L2: a head's workgroups share an XCD.
#pragma once
#include "fmha_fwd_kernel.h"

namespace fmha {

template <int D> struct ColsCfg {
  static constexpr int BK = 64, QT = 32;
  static constexpr int MAXW = D == 64 ? 10 : 7;     // waves per workgroup: what the LDS holds
  static constexpr int SKMAX = MAXW * BK;
  using Scratch = RowScratch<BK>;
  static constexpr int TILEB = BK * D * 2;          // a wave's V rows, then its part of the output (32 x D fp32: the same size)
  static constexpr int WAVEB = TILEB + Scratch::BYTES + 2 * QT * 4; // ... its scratch, its rows' maxima and sums
  static int lds_bytes(int nw) { return nw * WAVEB; }
};

template <typename T, int D, bool DROPT, bool SAVE, bool TAIL>
__global__ __launch_bounds__(ColsCfg<D>::MAXW * 64) __attribute__((amdgpu_waves_per_eu(D == 64 ? 3 : 2))) void fmha_fwd_cols_kernel(const FwdArgs a) {
  using E = Elem<T>;
  using v8 = typename E::v8;
  using v4 = typename E::v4;
  using C = ColsCfg<D>;
  constexpr int KS = D / 16, DB = D / 32, BK = C::BK, NSB = BK / 32;
  constexpr float NEG_INF = -__builtin_inff();
  static_assert(C::TILEB == 32 * D * 4, "a wave's part of the output takes the place of its V rows");

  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, ql = l & 31, h = l >> 5;
  const int nw = blockDim.x >> 6;

  // of every 8 heads each XCD gets one with all its query tiles
  const int b0 = blockIdx.x, grouped = (a.bh & ~7) * a.nqt;
  const int bh = b0 < grouped ? b0 / (8 * a.nqt) * 8 + (b0 & 7) : b0 / a.nqt;
  const int qt = b0 < grouped ? (b0 >> 3) % a.nqt : b0 % a.nqt;
  const int q0 = qt * C::QT, q = q0 + ql, k0 = w * BK;

  // ---- every request: Q, K, V, mask rows, dropout rows (they arrive in that order, and V with K)
  const T *Qr = (const T *)a.q + ((size_t)bh * a.sq + (q < a.sq ? q : a.sq - 1)) * D + h * 8;
  const T *Kb = (const T *)a.k + (size_t)bh * a.sk * D;
  const T *Vb = (const T *)a.v + (size_t)bh * a.sk * D;
  v8 qreg[KS], kreg[NSB][KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) qreg[ks] = as_v8<T>(*(const u32x4 *)(Qr + ks * 16));
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb) {
    const int key = k0 + sb * 32 + ql; // rows past the end re-read the last one: their scores become -inf
    const T *Kr = Kb + (uint32_t)((key < a.sk ? key : a.sk - 1) * D + h * 8);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kreg[sb][ks] = as_v8<T>(*(const u32x4 *)(Kr + ks * 16));
  }
  char *tile = lds + w * C::WAVEB;
  float *rows = (float *)(tile + C::TILEB + C::Scratch::BYTES); // this wave's maxima, then its sums
  TileCopy<T, D, BK, 64> vcopy;
  vcopy.init(l, D);
  vcopy.issue(Vb, k0, a.sk, lds_address(tile), l);
  typename C::Scratch scr;
  scr.init(tile + C::TILEB, l);
  u32x4 mreg[4], dreg[4];
  {
    const T *mb = (const T *)a.mask + (size_t)(bh / a.mask_div) * a.mask_sb;
    const T *db_ = DROPT ? (const T *)a.drop_mask + (size_t)bh * a.sq * a.sk : nullptr;
    const int koff = scr.template first_key<TAIL>(k0, a.sk);
    int qrow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) qrow[i] = q0 + 8 * i + scr.rsub < a.sq ? q0 + 8 * i + scr.rsub : a.sq - 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) mreg[i] = *(const u32x4_any *)(mb + (size_t)qrow[i] * a.mask_sq + koff);
    if (DROPT) {
#pragma unroll
      for (int i = 0; i < 4; ++i) dreg[i] = *(const u32x4_any *)(db_ + (size_t)qrow[i] * a.sk + koff);
    }
  }

  // ---- scores in log2 units
  f32x16 x[NSB];
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
    for (int r = 0; r < 16; ++r) x[sb][r] = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb) x[sb] = E::mfma(kreg[sb][ks], qreg[ks], x[sb]);
  if (TAIL) scr.place_tail(mreg, k0, a.sk);
  scr.rows_in(mreg);
  scr.turn();
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const v4 mv = as_v4<T>(scr.piece(sb, g));
#pragma unroll
      for (int i = 0; i < 4; ++i) x[sb][4 * g + i] = fmaf(x[sb][4 * g + i], a.scale_l2, fmaf((float)mv[i], a.mask_a, a.mask_b));
    }
  scr.turn();
  if (k0 + BK > a.sk) {
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int r = 0; r < 16; ++r) x[sb][r] = k0 + sb * 32 + 8 * (r >> 2) + 4 * h + (r & 3) < a.sk ? x[sb][r] : NEG_INF;
  }
  float mx = NEG_INF;
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
    for (int r = 0; r < 16; r += 2) mx = max3(mx, x[sb][r], x[sb][r + 1]);
  mx = xhalf_max(mx);
  const float ref = mx == NEG_INF ? 0.f : mx;
  float sum = 0.f;
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      x[sb][r] = fast_exp2(x[sb][r] - ref);
      sum += x[sb][r];
    }
  sum = xhalf_sum(sum);

  // ---- (dropped) probabilities in the element type, and this wave's part of O^T
  v4 dm[NSB][4];
  if (DROPT) {
    if (TAIL) scr.place_tail(dreg, k0, a.sk);
    scr.rows_in(dreg);
    scr.turn();
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int g = 0; g < 4; ++g) dm[sb][g] = as_v4<T>(scr.piece(sb, g));
    scr.turn();
  }
  dma_wait_all();
  PanelLane pl;
  pl.init(l);
  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;
#pragma unroll
  for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      v8 pf;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int r = 8 * c + e;
        pf[e] = (T)(DROPT ? x[sb][r] * (float)dm[sb][r >> 2][r & 3] : x[sb][r]);
      }
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] = E::mfma(panel_read_transposed<T, BK>(tile, pl, sb, db, c), pf, o[db]);
    }
  scr.turn(); // (the tile has been read)
  f32x4 *part = (f32x4 *)tile;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) part[(db * 4 + g) * 64 + l] = f32x4{o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]};
  if (h == 0) {
    rows[ql] = mx;
    rows[32 + ql] = sum;
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // ---- the row's maximum and sum
  auto row_of = [&](int j, int k) { return *(const float *)(lds + j * C::WAVEB + C::TILEB + C::Scratch::BYTES + (k * 32 + ql) * 4); };
  float top = NEG_INF, total = 0.f;
  for (int j = 0; j < nw; ++j) top = fmaxf(top, row_of(j, 0));
  const float base = top == NEG_INF ? 0.f : top;
  for (int j = 0; j < nw; ++j) total = fmaf(fast_exp2(row_of(j, 0) - base), row_of(j, 1), total);
  const float inv = total > 0.f ? 1.f / total : 0.f;

  if (SAVE) {
    const float f = fast_exp2(mx - base) * inv; // (a wave that saw no key: zero)
    auto rows_out = [&](void *out) {
      T *ob = (T *)out + (size_t)bh * a.sq * a.sk + k0 + scr.chunk * 8;
      scr.template rows_out<TAIL>([&](int qq) { return (char *)(ob + (size_t)qq * a.sk); }, q0, a.sq, k0, a.sk);
    };
    if (a.save_softmax) {
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          v4 s4;
#pragma unroll
          for (int i = 0; i < 4; ++i) s4[i] = (T)(x[sb][4 * g + i] * f);
          scr.template put_piece<T>(sb, g, s4);
        }
      scr.turn();
      rows_out(a.save_softmax);
      scr.turn();
    }
    if (a.save_dropout) {
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          v4 s4;
#pragma unroll
          for (int i = 0; i < 4; ++i) s4[i] = (T)(x[sb][4 * g + i] * f * ((float)dm[sb][g][i] * a.drop_scale));
          scr.template put_piece<T>(sb, g, s4);
        }
      scr.turn();
      rows_out(a.save_dropout);
    }
  }

  // ---- the partial outputs: wave w adds 16-column pieces w, w + nw, ..
  const float out = inv * a.drop_scale;
  T *Or = (T *)a.o + ((size_t)bh * a.sq + q) * D;
  for (int u = w; u < 2 * DB; u += nw) {
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    for (int j = 0; j < nw; ++j) {
      const float wt = fast_exp2(row_of(j, 0) - base);
      const f32x4 *pj = (const f32x4 *)(lds + j * C::WAVEB) + u * 2 * 64 + l;
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[g][i] = fmaf(wt, pj[g * 64][i], acc[g][i]);
    }
    if (q < a.sq) store_acc_pieces<T>(Or + u * 16, acc[0], acc[1], out, h);
  }
  if (a.lse && h == 0 && w == 0 && q < a.sq) a.lse[(size_t)bh * a.sq + q] = total > 0.f ? (base + fast_log2(total)) * FMHA_LN2 : NEG_INF;
}

} // namespace fmha
