// Forward kernel for long key ranges under a full [.., sq, sk] mask tensor (and, optionally, a dropout
// tensor of the same shape): the reference's operators beyond their own 128-key shape.
//
// With such tensors the forward is memory time at head dim 64 (BH 512, S 512: 34 GFLOP against
// 402 MB with the mask, 671 MB with mask and dropout tensor), so the kernel is built for streaming,
// like the kernel that writes the saved outputs: [.., sq, sk] rows arrive as whole 128-byte row
// segments (16 bytes per lane, 8 lanes per row; the last one of a row of any other length: TAIL), one
// tile ahead, and a wave-private LDS scratch per tensor turns them into the accumulator layout; K and V
// tiles are staged through registers with them, so every request of an iteration is in flight for a
// whole iteration.  (Two tiles ahead, with exact waits, measured 2 to 5 % slower with every compute unit
// busy: 91.1 -> 93.0 us at BH 512, S 512, 127.2 -> 134 with the dropout tensor.)  The softmax is the textbook
// online one (running row maximum, rescale on every tile, fp32 row sum): at two waves per SIMD the
// vector work hides under the memory time, which the lazily re-based, matrix-pipe-assisted softmax
// of the pipelined kernel is not needed for.
#pragma once
#include "fmha_fwd_kernel.h"

namespace fmha {

// MANY: the build for launches of more than two workgroups per compute unit, under the mask alone at head dim 64: one
// K / V stage instead of two, written between two barriers, which lets three workgroups share a compute unit.  BH 512,
// S 512: 87.5 -> 84.9 us, S 229: 28.4 -> 27.5; with fewer workgroups the second barrier only costs (BH 48, S 483: 13.7
// -> 14.7 us).  (With the dropout tensor three would need 54.6 KB of LDS each; the two scratches make it 55.3.)
// Head dim 128 has the one stage in any case: two would leave one workgroup per compute unit.
template <int D_, bool MANY> struct StreamCfg {
  static constexpr int D = D_;
  static constexpr int NW = 4;
  static constexpr int QT = NW * 32;
  static constexpr int BK = 64;
  static constexpr int ROWB = D * 2 + 16;          // padded K / V rows: conflict-free 16-byte and transpose reads
  static constexpr int TILEB = BK * ROWB;
  using Scratch = RowScratch<BK>;                  // wave-private: rows of a [.., sq, sk] tensor <-> accumulator layout
  static constexpr int NST = D == 64 && !MANY ? 2 : 1;
  static constexpr int OCC = MANY ? 3 : 2;
  static constexpr int nscr(bool dropt) { return dropt ? 2 : 1; }
  static constexpr int lds_bytes(bool dropt) { return NST * 2 * TILEB + NW * nscr(dropt) * Scratch::BYTES; } // {K, V} per stage + a wave's scratch
};

template <typename T, int D, bool DROPT, bool TAIL, bool MANY>
__global__ __launch_bounds__((StreamCfg<D, MANY>::NW * 64))
__attribute__((amdgpu_waves_per_eu(StreamCfg<D, MANY>::OCC, StreamCfg<D, MANY>::OCC)))
void fmha_fwd_stream_kernel(const FwdArgs a) {
  using E = Elem<T>;
  using v8 = typename E::v8;
  using v4 = typename E::v4;
  using C = StreamCfg<D, MANY>;
  static_assert(!MANY || (D == 64 && !DROPT), "three workgroups per compute unit: the mask alone at head dim 64");
  constexpr int KS = D / 16, DB = D / 32, BK = C::BK, NSB = BK / 32, NT = C::NW * 64, ROWB = C::ROWB;
  constexpr int TILEB = C::TILEB;
  constexpr int CPR = D / 8, CPT = BK * CPR / NT;
  constexpr float NEG_INF = -__builtin_inff();

  extern __shared__ __attribute__((aligned(16))) char lds[];

  const int tid = threadIdx.x;
  const int w = tid >> 6;
  const int l = tid & 63;
  const int ql = l & 31;
  const int h = l >> 5;

  int bid = blockIdx.x;
  const int nb = gridDim.x;
  if ((nb & 7) == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);
  const int bh = bid / a.nqt;
  const int qt = bid - bh * a.nqt;
  const int q0w = qt * C::QT + w * 32;

  const T *Qb = (const T *)a.q + (size_t)bh * a.sq * D;
  const T *Kb = (const T *)a.k + (size_t)bh * a.sk * D;
  const T *Vb = (const T *)a.v + (size_t)bh * a.sk * D;

  v8 qreg[KS];
  {
    int q = q0w + ql;
    q = q < a.sq ? q : a.sq - 1;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qreg[ks] = as_v8<T>(*(const u32x4 *)(Qb + (size_t)q * D + ks * 16 + h * 8));
  }

  // ---- staging.  K, V: global -> registers -> LDS (two stages).  [.., sq, sk] rows: instruction i covers
  // rows 8i .. 8i+7 of the wave's 32, eight lanes per row, 8 keys (16 bytes) per lane.
  typename C::Scratch scr, scrd; // mask rows, dropout rows
  scr.init(lds + C::NST * 2 * TILEB + w * C::nscr(DROPT) * C::Scratch::BYTES, l);
  scrd.init(lds + C::NST * 2 * TILEB + (w * C::nscr(DROPT) + C::nscr(DROPT) - 1) * C::Scratch::BYTES, l);
  const int rsub = scr.rsub, chunk = scr.chunk;
  int qrow[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = q0w + 8 * i + rsub;
    qrow[i] = q < a.sq ? q : a.sq - 1;
  }
  const T *mb = (const T *)a.mask + (size_t)(bh / a.mask_div) * a.mask_sb;
  const T *db_ = DROPT ? (const T *)a.drop_mask + (size_t)bh * a.sq * a.sk : nullptr;
  struct Stage {
    u32x4 k[CPT], v[CPT], m[4], d[4];
  };
  // Every load is unconditional (a load under a lane condition makes the compiler wait for it on the
  // spot): key rows past the end re-read the last row, chunks past sk re-read the row's last 8 keys;
  // those keys' scores are forced to -inf, so P = 0 meets finite values of V.
  auto gload = [&](int k0, Stage &st) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = tid + i * NT;
      int kr = k0 + c / CPR;
      kr = kr < a.sk ? kr : a.sk - 1;
      st.k[i] = *(const u32x4 *)(Kb + (size_t)kr * D + (c % CPR) * 8);
      st.v[i] = *(const u32x4 *)(Vb + (size_t)kr * D + (c % CPR) * 8);
    }
    const int koff = scr.template first_key<TAIL>(k0, a.sk);
#pragma unroll
    for (int i = 0; i < 4; ++i) st.m[i] = *(const u32x4_any *)(mb + (size_t)qrow[i] * a.mask_sq + koff);
    if (DROPT) {
#pragma unroll
      for (int i = 0; i < 4; ++i) st.d[i] = *(const u32x4_any *)(db_ + (size_t)qrow[i] * a.sk + koff);
    }
  };
  auto lstore = [&](int stage, const Stage &st) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = tid + i * NT;
      *(u32x4 *)(lds + stage * 2 * TILEB + (c / CPR) * ROWB + (c % CPR) * 16) = st.k[i];
      *(u32x4 *)(lds + stage * 2 * TILEB + TILEB + (c / CPR) * ROWB + (c % CPR) * 16) = st.v[i];
    }
  };

  auto rows_in = [&](int k0, Stage &st) {
    if (TAIL) scr.place_tail(st.m, k0, a.sk);
    scr.rows_in(st.m);
    if (DROPT) {
      if (TAIL) scrd.place_tail(st.d, k0, a.sk);
      scrd.rows_in(st.d);
    }
    scr.turn();
  };

  // ---- running state: row maximum m (log2 units), this lane's part of the row sum, unnormalised O^T
  float m = NEG_INF, lsum = 0.f;
  f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;

  const int nkt = (a.sk + BK - 1) / BK;
  Stage st;
  __builtin_amdgcn_sched_barrier(0);
  gload(0, st);
  lstore(0, st);
  rows_in(0, st);
  // (The compiler would wait for Q at its first use inside the loop, on every iteration, and with it for the
  // requests behind it.)
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qreg[ks]));
  __syncthreads();

  for (int t = 0; t < nkt; ++t) {
    const int k0 = t * BK;
    const char *ldsK = lds + (C::NST == 2 ? t & 1 : 0) * 2 * TILEB;
    const char *ldsV = ldsK + TILEB;
    const bool more = t + 1 < nkt; // workgroup-uniform
    if (more) gload(k0 + BK, st);

    // ---- scores in log2 units: x * scale + mask
    f32x16 x[NSB];
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) x[sb][r] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        x[sb] = E::mfma(as_v8<T>(*(const u32x4 *)(ldsK + (sb * 32 + ql) * ROWB + ks * 32 + h * 16)), qreg[ks], x[sb]);
    }
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const v4 mv = as_v4<T>(scr.piece(sb, g));
#pragma unroll
        for (int i = 0; i < 4; ++i)
          x[sb][4 * g + i] = fmaf(x[sb][4 * g + i], a.scale_l2, fmaf((float)mv[i], a.mask_a, a.mask_b));
      }
    scr.turn();
    if (k0 + BK > a.sk) { // only a partly filled last tile has keys to switch off (workgroup-uniform)
#pragma unroll
      for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kk = k0 + sb * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
          x[sb][r] = kk < a.sk ? x[sb][r] : NEG_INF;
        }
    }
    float tmax = NEG_INF;
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int r = 0; r < 16; r += 2) tmax = max3(tmax, x[sb][r], x[sb][r + 1]);

    // ---- online softmax: raise the maximum, rescale what has been accumulated under the old one
    tmax = xhalf_max(tmax);
    const float mnew = fmaxf(m, tmax);
    const float muse = mnew == NEG_INF ? 0.f : mnew;
    const float alpha = m == NEG_INF ? 0.f : fast_exp2(m - mnew);
    m = mnew;
    float rs = 0.f;
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = fast_exp2(x[sb][r] - muse);
        x[sb][r] = p;
        rs += p;
      }
    lsum = fmaf(lsum, alpha, rs);
    // (alpha is exactly one in every lane whose maximum stayed: the products are skipped when no lane's moved;
    // with the range check of the scores left to the one tile that needs it: BH 512 S 512 99.8 -> 95.3 us under
    // the mask alone, 136.9 -> 130.2 with the dropout tensor, BH 64 S 2048 167.3 -> 150.5 / 217.7 -> 199.2)
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
    }

    // ---- (dropped) probabilities in the element type: B operand of the second product
    v8 pfrag[NSB][2];
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float keep[4] = {1.f, 1.f, 1.f, 1.f};
        if (DROPT) {
          const v4 dm = as_v4<T>(scrd.piece(sb, g));
#pragma unroll
          for (int i = 0; i < 4; ++i) keep[i] = (float)dm[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) pfrag[sb][g >> 1][4 * (g & 1) + i] = (T)(x[sb][4 * g + i] * keep[i]);
      }
    if (DROPT) scr.turn();

    // ---- O^T += V^T . P^T
#pragma unroll
    for (int sb = 0; sb < NSB; ++sb)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int db = 0; db < DB; ++db)
          o[db] = E::mfma(lds_load_a_transposed<T, ROWB>(ldsV, sb * 32, db * 32, c, l), pfrag[sb][c], o[db]);

    if (C::NST == 1) __syncthreads(); // every wave is done with this tile
    if (more) {
      lstore(C::NST == 2 ? (t + 1) & 1 : 0, st);
      rows_in(k0 + BK, st);
    }
    __syncthreads();
  }

  // ---- epilogue
  const int q = q0w + ql;
  const float lt = xhalf_sum(lsum);
  const float inv = lt > 0.f ? a.drop_scale / lt : 0.f;
  if (q < a.sq) {
    T *Ob = (T *)a.o + ((size_t)bh * a.sq + q) * D;
#pragma unroll
    for (int db = 0; db < DB; ++db) store_acc_block_row<T>(Ob + db * 32, o[db], inv, h);
    if (a.lse && h == 0) a.lse[(size_t)bh * a.sq + q] = lt > 0.f ? (m + fast_log2(lt)) * FMHA_LN2 : NEG_INF;
  }
}

} // namespace fmha
