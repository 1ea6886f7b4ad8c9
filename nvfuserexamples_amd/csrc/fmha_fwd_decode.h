// Decode steps: one to four query rows per head against a long key range.
//
// Such a forward is memory time -- K and V are read once, 4*D bytes per key against 4*D flops per query row --
// so this kernel is built around the loads, not around the matrix pipe: a wave reads whole rows with 16-byte
// loads (D / 8 neighbouring lanes cover one row, so a load instruction fetches 64 / (D / 8) complete rows),
// keeps eight K loads and eight V loads in flight (up to 16 KB per wave, 128 KB per compute unit),
// and does the arithmetic on the vector pipe in fp32: dot products on v_dot2c_f32_f16 / _bf16 (exact products of
// the packed elements, fp32 sums; e4m3 rows as fp16, which holds every e4m3 value), summed over the lanes of a
// row by DPP additions, an online softmax per lane group, P.V by multiply-add.
// Nothing is staged in LDS and nothing is rounded on the way (scores, probabilities and sums are fp32).
//
// Several query rows, and short ranges of one, are bound by instructions, so no lane repeats another's: the 8 or 16 lanes of a row
// form two or four banks of four lanes, the sum over the lanes leaves a different score (query row, or key where rows are fewer) in each
// bank, and reference, exponential and sum are formed once a bank; P.V reads the probability of another bank through DPP.  Before, every
// lane had every score, and e4m3 rows were multiplied unpacked: a workgroup alone on its compute unit took 15.5 ns a key for four rows at
// D 128, now 13, 8.5 at D 64, now 6.3.  Whole steps of one, two and four rows at 746 drawn sizes are 1.09, 1.18 and 1.37 times as fast (with
// the lengths of the pieces that follow from this).
//
// Work split: a workgroup of four waves owns one (head, piece of the key range); its waves take the piece's
// blocks of keys in turn, and inside a wave the 64 / (D / 8) lane groups take every such-th key.  Each lane
// group runs its own online softmax over the keys it sees (running maximum m, sum l, 8 output columns per
// lane and query row); the 4 waves x lane groups meet once, at the end, through LDS.  With the key range in
// pieces (few heads: see the launch code) the piece's normalised output and log-sum-exp go to the caller's
// workspace as fp32 and a second kernel merges the pieces; otherwise O and the LSE are written directly.
#pragma once
#include "fmha_common.h"

namespace fmha {

// q, k and v may also hold e4m3 bytes (element type uint8_t here; o and the mask then have a 16-bit type of
// their own): the same kernel with 8-byte row loads, twice as many of them in flight, and the dequantisation
// factors folded into scale_l2 and out_scale.
struct DecodeArgs {
  const void *q, *k, *v;
  void *o;          // final output (element type), used when pieces == 1
  float *lse;       // optional final LSE [bh, sq], used when pieces == 1
  float *o_part;    // pieces > 1: [bh * pieces, sq, D] fp32
  float *lse_part;  // pieces > 1: [bh * pieces, sq]
  const void *mask; // optional per-key mask, element (b, j) at mask[(b / mask_div) * mask_sb + j]
  int64_t mask_sb;
  int32_t mask_div;
  float mask_a, mask_b; // mask term in log2 units = value * mask_a + mask_b
  const int32_t *kv_len;
  int32_t kv_div;
  int32_t bh, sq, sk;
  int32_t pieces, chunk; // pieces of `chunk` keys each (pieces == 1: chunk >= sk)
  float scale_l2;   // scale * log2(e) (times the dequantisation factors of q and k)
  float out_scale;  // 1 (the dequantisation factor of v)
  RowMap mq, mk, mv, mo;
};

constexpr int kDecodeWaves = 4;

// A lane's eight elements of a row: one 16-byte load of 16-bit elements, one 8-byte load of e4m3 bytes; how many K (and V) loads a
// wave keeps in flight per block (the same bytes either way); and the 16-bit type of the dot products (every e4m3 value is an fp16 value).
template <typename TI> struct DecodeIn {
  using Load = u32x4;
  using Dot = TI;
  static constexpr int LOADS = 8;
};
template <> struct DecodeIn<uint8_t> {
  using Load = u32x2;
  using Dot = _Float16;
  static constexpr int LOADS = 16;
};
FMHA_DEV u32x4 dot_form(u32x4 w) { return w; }
FMHA_DEV u32x4 dot_form(u32x2 w) { // eight e4m3 bytes as fp16
  return u32x4{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[0], 1.f, false)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[0], 1.f, true)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[1], 1.f, false)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[1], 1.f, true))};
}

template <typename T> FMHA_DEV void unpack8(u32x4 w, float (&x)[8]) {
  if constexpr (__is_same(T, _Float16)) {
    Pack16 p;
    p.u = w;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (float)p.h[e];
  } else { // bf16: the upper half of an fp32
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = __uint_as_float(w[i] << 16);
      x[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
}
template <typename T> FMHA_DEV void unpack8(u32x2 w, float (&x)[8]) { // e4m3
  static_assert(__is_same(T, uint8_t), "8-byte loads hold e4m3 bytes");
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[i], false), hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[i], true);
    x[4 * i] = lo[0];
    x[4 * i + 1] = lo[1];
    x[4 * i + 2] = hi[0];
    x[4 * i + 3] = hi[1];
  }
}

// c + a.x * b.x + a.y * b.y on a pair of 16-bit elements (fp32 products and sum).
template <typename T> FMHA_DEV float dot2(uint32_t a, uint32_t b, float c) {
  if constexpr (__is_same(T, _Float16)) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, a), __builtin_bit_cast(h2, b), c, false);
  } else {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, a), __builtin_bit_cast(b2, b), c, false);
  }
}

template <int V> struct Int {
  static constexpr int value = V;
};
template <int N, int I = 0, typename F> FMHA_DEV void static_for(const F &f) {
  if constexpr (I < N) {
    f(Int<I>{});
    static_for<N, I + 1>(f);
  }
}

// Among the LPR (8 or 16) neighbouring lanes that hold one row, the LPR / 4 fours of lanes are its banks.  score_banks sums LPR / 4
// values over those lanes at once and leaves value b in bank b, in all four of its lanes: what follows a score (reference, exponential,
// sum) is then done once per bank and not by every lane.
template <int CTRL> FMHA_DEV float dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
constexpr int DPP_ROW_MIRROR = 0x140, DPP_HALF_MIRROR = 0x141, DPP_ROR8 = 0x128, DPP_BCAST = 0x150; // (BCAST + n: lane n of each 16)
template <int LPR> FMHA_DEV float score_banks(const float (&v)[LPR / 4], bool odd_bank, bool upper) {
  float x, y;
  if constexpr (LPR == 16) {
    const float a = v[0] + dpp<DPP_ROW_MIRROR>(v[0]), b = v[1] + dpp<DPP_ROW_MIRROR>(v[1]);
    const float c = v[2] + dpp<DPP_ROW_MIRROR>(v[2]), d = v[3] + dpp<DPP_ROW_MIRROR>(v[3]);
    x = upper ? c : a;
    y = upper ? d : b;
  } else {
    x = v[0];
    y = v[1];
  }
  x += dpp<DPP_HALF_MIRROR>(x);
  y += dpp<DPP_HALF_MIRROR>(y);
  x = odd_bank ? y : x;
  x += dpp<0xB1>(x); // quad_perm [1,0,3,2]
  x += dpp<0x4E>(x); // quad_perm [2,3,0,1]
  return x;
}
// Bank b's value in every lane of the row (x is the same in the four lanes of a bank).
template <int LPR, int B> FMHA_DEV float from_bank(float x) {
  if constexpr (LPR == 16) return dpp<DPP_BCAST + 4 * B>(x);
  else {
    const int i = __builtin_bit_cast(int, x);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, DPP_HALF_MIRROR, 0xf, B == 0 ? 0xA : 0x5, false));
  }
}

// TI: element type of q, k, v (fp16, bf16 or uint8_t = e4m3); TO: of o and the mask (= TI unless TI is e4m3).
template <typename TI, typename TO, int D, int NQ, bool MASK>
// Two waves per SIMD at most, though fewer registers than 170 are needed: with three workgroups on some compute units and fewer on others the
// fullest one is waited for (e4m3, one row, BH 30 20 092 keys D 128: 33.4 us, with two 30.0; 700 drawn sizes 1.006 times as fast, 0.92 to 1.35).
__global__ __launch_bounds__(kDecodeWaves * 64) __attribute__((amdgpu_waves_per_eu(1, 2))) void fmha_fwd_decode_kernel(const DecodeArgs a) {
  using T = TI;
  using Load = typename DecodeIn<TI>::Load;
  constexpr int LPR = D / 8;       // lanes per row
  constexpr int NG = 64 / LPR;     // lane groups per wave = rows per load instruction
  using Dot = typename DecodeIn<TI>::Dot;
  constexpr int U = NQ >= 4 ? 8 : DecodeIn<TI>::LOADS; // (four query rows: fewer loads in flight, for the registers)
  constexpr int BANKS = LPR / 4;
  constexpr int RP = NQ < BANKS ? NQ : BANKS; // the banks' scores: RP query rows of
  constexpr int KP = BANKS / RP;              // KP keys (bank b: row b % RP, key b / RP)
  constexpr int RR = NQ / RP, JJ = U / KP;
  constexpr int BLK = U * NG;      // keys per wave and block
  constexpr int NS = kDecodeWaves * NG; // softmax states per workgroup
  constexpr float NEG_INF = -__builtin_inff();
  static_assert(D == 64 || D == 128, "rows of 8 or 16 lanes");

  __shared__ float s_m[NS][NQ], s_l[NS][NQ];
  __shared__ float s_acc[NS][NQ][D];

  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  const int g = l / LPR, c8 = l % LPR; // the lane's group and its 8 columns
  const bool odd_bank = l & 4, upper = l & 8;
  const int bank = c8 >> 2, koff = bank / RP;
  // The first pieces of all heads, then the second ones: with 8 pieces a head's would lie on one XCD each, and those of the last ones, which short
  // heads don't have, idle; the full ones start first (724 drawn steps, half of them with key counts, 1.02 times as fast).
  const int piece = blockIdx.x / a.bh, head = blockIdx.x - piece * a.bh, part = head * a.pieces + piece;

  // keys of this piece: [k0, k1)
  int n = a.sk;
  if (a.kv_len) {
    const int m = a.kv_len[head / a.kv_div];
    n = m < 0 ? 0 : (m < n ? m : n);
  }
  const int k0 = piece * a.chunk;
  int k1 = k0 + a.chunk;
  k1 = k1 < n ? k1 : n;

  const T *Kb = (const T *)a.k + a.mk.head(head) + c8 * 8;
  const T *Vb = (const T *)a.v + a.mv.head(head) + c8 * 8;
  const size_t kss = (size_t)a.mk.ss, vss = (size_t)a.mv.ss;
  const TO *mrow = MASK ? (const TO *)a.mask + (size_t)(head / a.mask_div) * (size_t)a.mask_sb : nullptr;

  // the lane's 8 columns of every query row, packed (the dot products run on v_dot2c_f32_*: exact products summed in fp32, and the
  // score is scaled afterwards)
  u32x4 qp[NQ];
#pragma unroll
  for (int r = 0; r < NQ; ++r) {
    const int qr = r < a.sq ? r : a.sq - 1;
    qp[r] = dot_form(*(const Load *)((const T *)a.q + a.mq.head(head) + (size_t)qr * (size_t)a.mq.ss + c8 * 8));
  }

  float m_run[RR], l_run[RR], acc[NQ][8];
#pragma unroll
  for (int rr = 0; rr < RR; ++rr) {
    m_run[rr] = NEG_INF;
    l_run[rr] = 0.f;
  }
#pragma unroll
  for (int r = 0; r < NQ; ++r) {
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[r][e] = 0.f;
  }

  // blocks of the piece: wave w takes blocks w, w + 4, ...; load j of a block covers keys kb + j*NG + g
  const int nblk = k1 > k0 ? (k1 - k0 + BLK - 1) / BLK : 0;
  // One set of registers per stream: the K loads of the wave's next block are issued as soon as this block's
  // scores are formed, its V loads as soon as this block's P.V is done, so that 8-16 loads per wave (and the other
  // waves of the SIMD) cover the trip to memory.
  Load kc[U], vc[U];
  float mc[JJ]; // (of the lane's bank)
  auto key_of = [&](int b, int j) {
    const int key = k0 + b * BLK + j * NG + g;
    return key < k1 ? key : k1 - 1; // keys past the end repeat the last one (their scores are set to -inf)
  };
  auto issue_k = [&](int b) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int key = key_of(b, j);
      kc[j] = *(const Load *)(Kb + (size_t)key * kss);
    }
    if constexpr (MASK) {
#pragma unroll
      for (int jj = 0; jj < JJ; ++jj) mc[jj] = (float)mrow[key_of(b, jj * KP + koff)];
    }
  };
  auto issue_v = [&](int b) {
#pragma unroll
    for (int j = 0; j < U; ++j) vc[j] = *(const Load *)(Vb + (size_t)key_of(b, j) * vss);
  };
  if (w < nblk) {
    issue_k(w);
    issue_v(w);
  }
  for (int b = w; b < nblk; b += kDecodeWaves) {
    const bool more = b + kDecodeWaves < nblk;
    const int kb = k0 + b * BLK;
    // scores of the group's U keys, all query rows
    float s[RR][JJ];
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj) {
      u32x4 x[KP];
#pragma unroll
      for (int kk = 0; kk < KP; ++kk) x[kk] = dot_form(kc[jj * KP + kk]);
      const bool live = kb + (jj * KP + koff) * NG + g < k1;
#pragma unroll
      for (int rr = 0; rr < RR; ++rr) {
        float v[BANKS];
#pragma unroll
        for (int bk = 0; bk < BANKS; ++bk) {
          float d = 0.f;
#pragma unroll
          for (int i = 0; i < 4; ++i) d = dot2<Dot>(qp[rr * RP + bk % RP][i], x[bk / RP][i], d);
          v[bk] = d;
        }
        float d = score_banks<LPR>(v, odd_bank, upper) * a.scale_l2;
        if constexpr (MASK) d += fmaf(mc[jj], a.mask_a, a.mask_b);
        s[rr][jj] = live ? d : NEG_INF;
      }
    }
    if (more) issue_k(b + kDecodeWaves);
    // online softmax: raise the reference, rescale, turn the scores into probabilities
    float alpha[RR];
#pragma unroll
    for (int rr = 0; rr < RR; ++rr) {
      float bm = s[rr][0];
#pragma unroll
      for (int jj = 1; jj < JJ; ++jj) bm = fmaxf(bm, s[rr][jj]);
      if constexpr (KP == 4 || (KP == 2 && LPR == 8)) bm = fmaxf(bm, dpp<DPP_HALF_MIRROR>(bm)); // one reference for the keys' banks
      if constexpr (KP > 1 && LPR == 16) bm = fmaxf(bm, dpp<DPP_ROR8>(bm));
      const float m_new = fmaxf(m_run[rr], bm);
      const float m_use = m_new == NEG_INF ? 0.f : m_new; // nothing visible yet: every probability is 0
      alpha[rr] = fast_exp2(m_run[rr] - m_use);           // (2^-inf = 0 at the start)
      m_run[rr] = m_new;
      float ps = 0.f;
#pragma unroll
      for (int jj = 0; jj < JJ; ++jj) {
        s[rr][jj] = fast_exp2(s[rr][jj] - m_use);
        ps += s[rr][jj];
      }
      l_run[rr] = l_run[rr] * alpha[rr] + ps; // (of the bank's keys)
    }
    static_for<RP>([&](auto rp) {
      constexpr int RI = decltype(rp)::value;
#pragma unroll
      for (int rr = 0; rr < RR; ++rr) {
        const float al = from_bank<LPR, RI>(alpha[rr]);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[rr * RP + RI][e] *= al;
      }
    });
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj) {
      static_for<KP>([&](auto kk) {
        constexpr int KI = decltype(kk)::value;
        float x[8];
        unpack8<T>(vc[jj * KP + KI], x);
        static_for<RP>([&](auto rp) {
          constexpr int RI = decltype(rp)::value;
#pragma unroll
          for (int rr = 0; rr < RR; ++rr) {
            const float p = from_bank<LPR, RI + RP * KI>(s[rr][jj]);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[rr * RP + RI][e] = fmaf(p, x[e], acc[rr * RP + RI][e]);
          }
        });
      });
    }
    if (more) issue_v(b + kDecodeWaves);
  }

  // ---- the workgroup's NS partial softmaxes meet in LDS
  const int st = w * NG + g;
#pragma unroll
  for (int rr = 0; rr < RR; ++rr) {
    float tot = l_run[rr];
    if constexpr (KP == 4 || (KP == 2 && LPR == 8)) tot += dpp<DPP_HALF_MIRROR>(tot);
    if constexpr (KP > 1 && LPR == 16) tot += dpp<DPP_ROR8>(tot);
    if ((c8 & 3) == 0 && koff == 0) {
      s_m[st][rr * RP + bank] = m_run[rr];
      s_l[st][rr * RP + bank] = tot;
    }
  }
#pragma unroll
  for (int r = 0; r < NQ; ++r) {
#pragma unroll
    for (int e = 0; e < 8; ++e) s_acc[st][r][c8 * 8 + e] = acc[r][e];
  }
  __syncthreads();
  // thread t: query row t / LPR, columns 8 * (t % LPR) .. +7
  const int r = tid / LPR;
  if (r < NQ && r < a.sq) {
    float M = NEG_INF;
#pragma unroll
    for (int i = 0; i < NS; ++i) M = fmaxf(M, s_m[i][r]);
    float tot = 0.f, out[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (M != NEG_INF) {
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const float f = fast_exp2(s_m[i][r] - M); // (an empty state: 2^-inf = 0)
        tot = fmaf(s_l[i][r], f, tot);
#pragma unroll
        for (int e = 0; e < 8; ++e) out[e] = fmaf(s_acc[i][r][c8 * 8 + e], f, out[e]);
      }
    }
    const float inv = tot > 0.f ? a.out_scale / tot : 0.f; // no visible key: O = 0, LSE = -inf
    const float lse = tot > 0.f ? (M + fast_log2(tot)) * FMHA_LN2 : NEG_INF;
    if (a.pieces > 1) {
      float *dst = a.o_part + ((size_t)part * a.sq + r) * D + c8 * 8;
      f32x4 lo = {out[0] * inv, out[1] * inv, out[2] * inv, out[3] * inv};
      f32x4 hi = {out[4] * inv, out[5] * inv, out[6] * inv, out[7] * inv};
      *(f32x4 *)dst = lo;
      *(f32x4 *)(dst + 4) = hi;
      if (c8 == 0) a.lse_part[(size_t)part * a.sq + r] = lse;
    } else {
      Pack16 y;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if constexpr (__is_same(TO, _Float16)) y.h[e] = (_Float16)(out[e] * inv);
        else y.b[e] = (__bf16)(out[e] * inv);
      }
      *(u32x4 *)((TO *)a.o + a.mo.head(head) + (size_t)r * (size_t)a.mo.ss + c8 * 8) = y.u;
      if (a.lse && c8 == 0) a.lse[(size_t)head * a.sq + r] = lse;
    }
  }
}

// Return 0 on success, 1 if the shape is not built, 2 if the launch failed.
int fwd_decode_dispatch(const DecodeArgs &a, int d, bool bf16, hipStream_t s);
// The same for e4m3 q, k, v (o and mask fp16 or bf16).
int fwd_decode_fp8_dispatch(const DecodeArgs &a, int d, bool out_bf16, hipStream_t s);

} // namespace fmha
