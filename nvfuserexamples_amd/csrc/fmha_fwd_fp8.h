// Forward attention on 8-bit floating point inputs (OCP e4m3): q, k, v hold e4m3 bytes with one
// dequantisation factor per tensor, both products run on v_mfma_f32_32x32x64_f8f6f4 (the K = 64 form, the
// only fp8 matrix instruction that runs at twice the 16-bit rate) with fp32 accumulation, the softmax is
// fp32, and the probabilities are rounded to e4m3 -- unnormalised, relative to an integer reference exponent
// near the row maximum, where e4m3 keeps its three mantissa bits down to 2^-6 -- before the second product.  O leaves as
// fp16 or bf16.  The reference is fp16 only (fmha/fmha_manual.cpp:120, Ampere_16_8_16).  Same
// transposed-product design as the 16-bit kernels, on a plain double-buffered loop:
//   S^T = K.Q^T   A = K rows from LDS (32 bytes per lane: keys l % 32, head-dim bytes 32 (l / 32) .. +31),
//                 B = Q in registers; lane = query
//   O^T = V^T.P^T A = V^T through the 8-bit LDS transpose read (ds_read_b64_tr_b8) from a V tile kept as it
//                 is in memory, B = the two accumulator tiles of the first product, rounded in place
// Feeding the accumulator tiles back: a lane's 32 contraction bytes are its 16 registers of key block 0, then
// of key block 1; register r of a lane (q, h) is key 8 (r / 4) + 4h + r % 4 of its block, so contraction byte
// j = 16 b + r of half-wave h stands for key 32 b + 8 (r / 4) + 4 h + r % 4, and the V^T operand is fetched in
// that order: transpose read (b, gp) covers the rows 32 b + 16 gp + 4 h + {0,1,2,3, 8,9,10,11}.
// The per-element vector work is what bounds the kernel: P = exp2(s x - M), s = scale * descale_q * descale_k *
// log2(e), is one fused multiply-add, one exponential and half a conversion per element (and an add for the LSE).
// A mask term or the end of the keys costs a tile that has one a bf16 32x32x16 step after the fp8 product,
//   A row of a key   (mk_hi, mk_mid, mk_lo, 0 ..)   mk = mask term / s, "-inf" for keys past the end
//   B col of a query (1, 1, 1, 0 ..)
// (three bf16 pieces: exact to fp32); tiles whose keys are all there and unmasked -- most of a padded batch --
// go without.  Key tiles of nothing but hard-masked keys at the end of a mask row are not visited where their
// weights are zero whatever the inputs (Fp8Args::trim).
// Counted at BH 156 S 2432 D 64: 163 vector instructions a tile and wave, 112 of them those above (an exponential and a
// packed conversion take the pipe about nine cycles, the others four), the vector pipe busy 74 % of the launch, the matrix
// pipe 25 %; clearing the conversions' registers, copies of the operand of ones and the first tile's second computation
// were the rest.  Without them 167 -> 154 us; BH 512 S 512 with masks whose lengths are spread over [256, 512] 38.0 -> 34.0,
// without a mask 38.4 -> 33.3.  (A loop that skews the products of the tiles before and after against a tile's exponentials
// inside a wave, at two waves a SIMD for its registers, lost: 154 -> 167, D 128 BH 384 S 960 138 -> 154.)
// The registers are held to four waves per SIMD at head dim 64, three where causal (a tighter budget spills in the loop).
// The row sums come out of the matrix pipe too:
// one more fp8 product of the rounded tile with an operand of ones gives every lane the sum of ITS row's
// rounded probabilities, so O = sum P~ v / sum P~ is a convex combination of the values (a row with one
// dominant key reproduces that key's value exactly, whatever the rounding did to its probability).  The row
// log-sum-exp, where the caller wants it, is accumulated from the unrounded probabilities (one add per element,
// in that case only).  M is the row's reference exponent, an INTEGER in log2 units, so that changing it
// rescales every probability by an exact power of two and the e4m3 rounding of P does not depend on when a
// maximum was met.  It is not a running maximum: it is set from the first tile a row sees (ceil of that tile's
// maximum) and raised only when a tile's row sum leaves the range in which no probability can exceed the e4m3
// range (sum of the rounded values > 256; a saturated 448 or a NaN fails the same test), the rare slow path
// that also rescales the accumulators; a common tile computes no maximum at all.
// ds_read_b64_tr_b8, as measured on the device: the 16 lanes of a group cover 8 rows x 16 byte columns; lane i
// supplies the address of row i / 2, byte columns 8 (i % 2) .. +7, and receives column i, rows 0..7.
#pragma once
#include "fmha_common.h"

namespace fmha {

struct Fp8Args {
  const uint8_t *q, *k, *v; // e4m3 bytes, [bh, s, d] contiguous
  void *o;                  // [bh, sq, d] fp16 / bf16
  float *lse;               // optional [bh, sq]
  const void *mask;         // optional per-key additive mask in O's element type: mask[(bh / mask_div) * mask_sb + key]
  int64_t mask_sb;
  int32_t mask_div;
  int32_t bh, sq, sk;
  float score_scale_l2;     // s = scale * descale_q * descale_k * log2(e)
  float inv_score_scale_l2; // 1 / s
  float out_scale;          // descale_v
  // Leave out the key tiles behind the last key whose mask term is above kFp8Hard, in rows that have a key at or above
  // kFp8Live.  The launch code sets it where  |score| <= 448^2 d scale descale_q descale_k <= kFp8TrimScore  for any
  // inputs: a hard-masked key's exponent is then at least 200 (288 in log2 units) below the row's reference, less the 8
  // that the reference may sit below the maximum, so its probability is 0 in fp32 and leaving it out changes nothing.
  int32_t trim;
  int32_t split; // the waves of a workgroup share 32 queries and take their key tiles in turn
};
constexpr float kFp8Hard = -9000.f, kFp8Live = -1000.f, kFp8TrimScore = 3900.f;

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x4v __attribute__((ext_vector_type(4)));
typedef int i32x2v __attribute__((ext_vector_type(2)));

// SPLIT: the four waves of a workgroup take the key tiles of the same 32 queries in turn instead of 32 queries each, every
// wave with an LDS stage of its own (no barrier), and their partial rows meet in LDS at the end.  A tile takes a wave
// that has its SIMD to itself 0.8 us from end to end, so a launch of few workgroups lasts as long as its longest row of
// tiles: four times the workgroups of a quarter of the tiles each use the idle units.  Large launches keep the other
// form (K and V are staged once per 128 queries there, not per 32; D 64 BH 512 S 512 34.5 / 52.8 us).  The line between them: fp8_split in
// fmha_capi.hip.  Before / now, us: BH 8 S 3712 D 64 causal 44.2 / 20.2, BH 16 S 2013 25.3 / 22.8, S 600 causal 10.0 / 6.8.
template <int D, bool SPLIT> struct Fp8Cfg {
  static constexpr int NW = 4, NT = NW * 64, QT = SPLIT ? 32 : NW * 32, BK = 64;
  static constexpr int PITCH = D + 16;              // bytes per key row of the K and V tiles (16 rows, 16 bank groups)
  static constexpr int TILEB = BK * PITCH;
  static constexpr int XROWB = 16;                  // extra-step row of a key: 8 bf16
  static constexpr int LDS_FLAG = 2 * TILEB + BK * XROWB; // (in a stage) whether the tile takes the extra step
  static constexpr int STAGEB = LDS_FLAG + 16;      // K tile, V tile, extra-step rows of the tile, flag
  static constexpr int NSTAGE = SPLIT ? NW : 2;     // one for each wave / two that all waves share
  static constexpr int LDS_MERGE = NW * 32 * D * 4; // SPLIT, over the stages: the waves' outputs, then their rows' sums
  static constexpr int LDS_TILES = SPLIT && NSTAGE * STAGEB < LDS_MERGE + NW * 3 * 32 * 4 ? LDS_MERGE + NW * 3 * 32 * 4 : NSTAGE * STAGEB;
  static constexpr int LDS_TRIM = LDS_TILES;        // per wave: keys up to its last live one, whether it saw a visible one
  static constexpr int LDS_BYTES = LDS_TRIM + 2 * NW * 4;
};

// 32x32 += (32 x 64 e4m3) . (64 x 32 e4m3); format selectors 0 = e4m3 for both operands, no block scaling
FMHA_DEV f32x16 mfma_fp8_k64(i32x8 a, i32x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}
// 16x16 = (16 x 128 e2m1) . (128 x 16 e4m3); the 4-bit operand takes the first half of its registers
FMHA_DEV f32x4 mfma_fp4_fp8_k128(i32x4v a, i32x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(i32x8{a.x, a.y, a.z, a.w, 0, 0, 0, 0}, b, c, 4, 0, 0, 0, 0, 0);
}
FMHA_DEV i32x2v lds_read_tr8(const char *lds_ptr) {
  typedef __attribute__((address_space(3))) i32x2v lds_vec;
  return __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_vec *)(lds_ptr));
}

// Four floats to four e4m3 bytes (round to nearest even), element 0 in the lowest byte.
FMHA_DEV int pack4_e4m3(float a, float b, float c, float d) {
  int w;
  asm("" : "=v"(w) : "v"(a)); // (any register: both halves are written, nothing has to be cleared first)
  w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, w, false);
  w = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
  return w;
}

// v = hi + mid + lo in bf16 pieces (24 bits together)
FMHA_DEV void split3_bf16(float v, __bf16 &hi, __bf16 &mid, __bf16 &lo) {
  hi = (__bf16)v;
  const float r = v - (float)hi;
  mid = (__bf16)r;
  lo = (__bf16)(r - (float)mid);
}

template <typename TO, int D, bool CAUSAL, bool MASK, bool SPLIT>
__global__ __launch_bounds__((Fp8Cfg<D, SPLIT>::NT), D == 64 ? (SPLIT || CAUSAL ? 3 : 4) : 2) void fmha_fwd_fp8_kernel(const Fp8Args a) {
  using C = Fp8Cfg<D, SPLIT>;
  constexpr int NT = C::NT, QT = C::QT, BK = C::BK, DS = D / 64, DB = D / 32, PITCH = C::PITCH, XROWB = C::XROWB;
  constexpr int CPR = D / 16;            // 16-byte chunks per row
  constexpr int TT = SPLIT ? 64 : NT;    // threads that stage a tile
  constexpr int CPT = BK * CPR / TT;     // chunks per thread and tile
  constexpr int STEP = SPLIT ? C::NW : 1; // a wave's tiles are this far apart
  static_assert(CPT >= 1, "tile must cover the workgroup");
  constexpr float NEG_INF = -__builtin_inff();
  constexpr float SUM_LIMIT = 256.f;     // a row sum up to here: every probability fits e4m3 (maximum 448)

  extern __shared__ __attribute__((aligned(16))) char lds[];

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, ql = l & 31, h = l >> 5;
  const int ts = SPLIT ? l : tid; // among the threads that stage a tile
  const int nqt = (a.sq + QT - 1) / QT;
  // Workgroups are dealt round-robin to the 8 XCDs: of every 8 heads each XCD gets one with all its query tiles, so a
  // head's keys go through one L2, and heads of different lengths stay spread evenly.  Causal: the longest tiles of all heads
  // first (us, against heads in turn with the order of tiles reversed from 32 workgroups of an XCD to the next: D 64 BH 20 S 4000
  // 65.9 / 48.6, BH 128 S 2048 76.9 / 62.0, BH 512 S 1024 79.2 / 71.3, BH 240 S 552 24.2 / 20.0; D 128 BH 64 S 1524 49.4 / 40.0, BH
  // 32 S 3616 97.1 / 81.9, BH 304 S 400 31.7 / 27.4, BH 8 S 8000 122 / 123).
  const int b = blockIdx.x, grouped = (a.bh & ~7) * nqt;
  int bh = b < grouped ? b / (8 * nqt) * 8 + (b & 7) : b / nqt;
  int qt = b < grouped ? (b >> 3) % nqt : b % nqt;
  if (CAUSAL) {
    const int lg = head_groups_log2(a.bh), m = by_length(b, (int)gridDim.x, lg), heads = a.bh >> lg;
    qt = m / heads;
    bh = ((m - qt * heads) << lg) + (b & ((1 << lg) - 1));
    qt = nqt - 1 - qt;
  }
  const int q0 = qt * QT + (SPLIT ? 0 : w * 32), q = q0 + ql;
  const int qc = q < a.sq ? q : a.sq - 1;
  const float s = a.score_scale_l2, inv_s = a.inv_score_scale_l2;
  // a masked key's term in raw score units: -1e25 in log2 units whatever the scale (kept inside the bf16 range)
  const float BIGNEG_RAW = -fminf(1e25f * inv_s, 1e37f);

  const uint8_t *Qb = a.q + (size_t)bh * a.sq * D;
  const uint8_t *Kb = a.k + (size_t)bh * a.sk * D;
  const uint8_t *Vb = a.v + (size_t)bh * a.sk * D;
  const TO *mkey = MASK ? (const TO *)a.mask + (size_t)(bh / a.mask_div) * a.mask_sb : nullptr;

  // Q as the B operand: column = this lane's query, contraction bytes 64 ds + 32 h .. +31
  i32x8 qreg[DS];
#pragma unroll
  for (int ds = 0; ds < DS; ++ds) {
    const u32x4 lo = *(const u32x4 *)(Qb + (size_t)qc * D + ds * 64 + h * 32);
    const u32x4 hi = *(const u32x4 *)(Qb + (size_t)qc * D + ds * 64 + h * 32 + 16);
    qreg[ds] = i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
  }

  int nkt = (a.sk + BK - 1) / BK;
  if (CAUSAL) {
    int qmax = qt * QT + QT - 1;
    if (qmax > a.sq - 1) qmax = a.sq - 1;
    const int need = qmax / BK + 1;
    if (need < nkt) nkt = need;
  }

  // tile staging: global -> registers -> LDS, both tiles as they are in memory; two LDS stages, or one of the wave's own
  u32x4 kst[CPT], vst[CPT];
  TO mraw = (TO)0.f; // this thread's key's mask value, as it is in memory: whatever is made of it here would wait for it here
  auto stage_of = [&](int kt) { return lds + (SPLIT ? w : kt & 1) * C::STAGEB; };
  auto gload = [&](int k0) {
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = ts + i * TT, row = c / CPR, col = c % CPR;
      int kr = k0 + row;
      kr = kr < a.sk ? kr : a.sk - 1; // keys past the end re-read the last row; their mask term is "-inf"
      const uint32_t at = (uint32_t)(kr * D + col * 16);
      kst[i] = *(const u32x4 *)(Kb + at);
      vst[i] = *(const u32x4 *)(Vb + at);
    }
    if (MASK && ts < BK) mraw = mkey[k0 + ts < a.sk ? k0 + ts : a.sk - 1];
  };
  auto lstore = [&](int kt) {
    char *kd = stage_of(kt);
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      const int c = ts + i * TT, row = c / CPR, col = c % CPR;
      *(u32x4 *)(kd + row * PITCH + col * 16) = kst[i];
      *(u32x4 *)(kd + C::TILEB + row * PITCH + col * 16) = vst[i];
    }
    if (ts < BK) { // (one wave) (mk_hi, mk_mid, mk_lo, 0 ...), the term in raw score units
      const float mk = (float)mraw;
      float mst = MASK ? (mk == NEG_INF ? BIGNEG_RAW : fmaxf(mk * (FMHA_LOG2E * inv_s), BIGNEG_RAW)) : 0.f;
      if (kt * BK + ts >= a.sk) mst = BIGNEG_RAW;
      const bool any = __builtin_amdgcn_ballot_w64(mst != 0.f) != 0;
      if (any) {
        __bf16 hi, mid, lo;
        split3_bf16(mst, hi, mid, lo);
        const uint32_t b0 = __builtin_bit_cast(uint16_t, hi), b1 = __builtin_bit_cast(uint16_t, mid), b2 = __builtin_bit_cast(uint16_t, lo);
        *(u32x4 *)(kd + 2 * C::TILEB + ts * XROWB) = u32x4{b0 | b1 << 16, b2, 0, 0};
      }
      if (ts == 0) *(int *)(kd + C::LDS_FLAG) = any;
    }
  };

  // transpose-read address of this lane inside a V tile: row 4h + {0,1,2,3, 8,9,10,11}[i16 / 2], byte column
  // (ql & 16) + 8 (i16 % 2) of a 32-column block
  const int i16 = l & 15;
  const int trofs = (4 * h + (i16 >> 1) + ((i16 >> 1) >= 4 ? 4 : 0)) * PITCH + (ql & 16) + 8 * (i16 & 1);

  f32x16 oacc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[db][r] = 0.f;
  float M = 0.f, l_run = 0.f, l_true = 0.f; // reference exponent (an integer); sums of the rounded / unrounded probabilities relative to it
  bool seen = false;          // M has been set from a tile with a live key
  // Row sums: the rounded tile's registers, read as the 128 x 16 operand of the 16x16 product, hold in column c and
  // lane group j (lane 16 j + c) the probabilities of query c + 16 (j & 1).  Rows 4 i .. 4 i + 3 of the other operand are ones
  // in the contraction indices of groups of i's parity, and come out in the lanes 16 i + c: every lane gets the whole sum of
  // its own row.  (As measured: index k belongs to group k / 16 % 4 in an 8-bit operand, to register k / 8 % 4 of group
  // k / 32 in a 4-bit one.)
  const int one0 = (l >> 2) & 1 ? 0 : 0x22222222, one1 = 0x22222222 - one0; // (1.0 in e2m1)
  const i32x4v ones = {one0, one0, one1, one1};
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // A NaN of query c times 0 is a NaN in the sum of query c + 16.  So where there may be one, rows with a NaN are cleared before
  // the product is formed; whether this lane's row was:
  auto clear_nan_row = [&](i32x8 &p) {
    int any = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) any |= (p[i] & 0x7f7f7f7f) + 0x01010101; // (e4m3: all seven bits)
    const auto both = __builtin_amdgcn_permlane32_swap(any, any, false, false);
    const bool nan = ((both[0] | both[1]) & 0x80808080) != 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = nan ? 0 : p[i];
    return nan;
  };
  // extra-step column of a query: bf16 (1, 1, 1, 0 ..); the other half-wave, which reads the same rows, takes zeros
  const uint32_t bx0 = h == 0 ? 0x3f803f80u : 0u, bx1 = h == 0 ? 0x3f80u : 0u;

  const int first = SPLIT ? w : 0; // this wave's first tile
  gload(first * BK);
  const bool trim = MASK && !CAUSAL && a.trim && nkt > 1;
  if (trim) {
    int last = 0, seen_live = 0;
    for (int j = w * 64; j < a.sk; j += NT) {
      const float mk = j + l < a.sk ? (float)mkey[j + l] : NEG_INF;
      const unsigned long long up = __builtin_amdgcn_ballot_w64(mk > kFp8Hard);
      if (up) last = j + 64 - (int)__builtin_clzll(up);
      seen_live |= __builtin_amdgcn_ballot_w64(mk >= kFp8Live) != 0;
    }
    if (l == 0) {
      ((int *)(lds + C::LDS_TRIM))[2 * w] = last;
      ((int *)(lds + C::LDS_TRIM))[2 * w + 1] = seen_live;
    }
  }
  lstore(first);
  if (first + STEP < nkt) gload((first + STEP) * BK);
  if (trim || !SPLIT) __syncthreads();
  else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // (as behind every later stage: other lanes read what this one wrote)
  if (trim) {
    int last = 0, seen_live = 0;
#pragma unroll
    for (int i = 0; i < C::NW; ++i) {
      const int n = ((const int *)(lds + C::LDS_TRIM))[2 * i];
      last = n > last ? n : last;
      seen_live |= ((const int *)(lds + C::LDS_TRIM))[2 * i + 1];
    }
    last = __builtin_amdgcn_readfirstlane(last);
    if (__builtin_amdgcn_readfirstlane(seen_live)) nkt = (last + BK - 1) / BK;
  }

  // The next tile goes to the other stage, whose last readers passed the barrier that ended the previous iteration; a wave
  // with a stage of its own overwrites it when it has read it (LDS serves a wave's requests in order).
  auto stage_next = [&](int kt) {
    if (kt + STEP < nkt) {
      lstore(kt + STEP);
      if (kt + 2 * STEP < nkt) gload((kt + 2 * STEP) * BK);
    }
  };
  // causal: the tiles that hold nothing up to this wave's own rows are left to the waves behind it
  int nktw = nkt;
  if (CAUSAL && !SPLIT) {
    const int own = (q0 + 31) / BK + 1;
    nktw = own < nkt ? own : nkt;
  }
  for (int kt = first; kt < nktw; kt += STEP) {
    const int k0 = kt * BK;
    const char *ldsK = stage_of(kt);
    const char *ldsV = ldsK + C::TILEB;
    const char *ldsX = ldsK + 2 * C::TILEB;

    const bool extra = MASK ? __builtin_amdgcn_readfirstlane(*(const int *)(ldsK + C::LDS_FLAG)) != 0 : k0 + BK > a.sk;

    // x = K.Q^T + mask[key] / s  for the two 32-key blocks of the tile
    f32x16 x[2];
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) x[sb][r] = 0.f;
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) {
        const char *kp = ldsK + (sb * 32 + ql) * PITCH + ds * 64 + h * 32;
        const u32x4 lo = *(const u32x4 *)kp, hi = *(const u32x4 *)(kp + 16);
        const i32x8 ka = {(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
        x[sb] = mfma_fp8_k64(ka, qreg[ds], x[sb]);
      }
    }
    if (extra) {
#pragma unroll
      for (int sb = 0; sb < 2; ++sb) {
        const bf16x8 xa = as_v8<__bf16>(*(const u32x4 *)(ldsX + (sb * 32 + ql) * XROWB));
        x[sb] = Elem<__bf16>::mfma(xa, as_v8<__bf16>(u32x4{bx0, bx1, 0, 0}), x[sb]);
      }
    }
    if (!SPLIT) stage_next(kt); // while this one is worked on
    // register r of block sb is key k0 + 32 sb + 8 (r / 4) + 4 h + r % 4
    const bool diag = CAUSAL && (k0 + BK - 1 > q0);
    const bool want_lse = a.lse != nullptr;
    const int own = q - k0 - 4 * h; // causal: the lane's last visible key, in its own order
    auto hide_later_keys = [&](f32x16 (&v)[2]) {
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          v[sb][r] = sb * 32 + 8 * (r / 4) + r % 4 <= own ? v[sb][r] : NEG_INF;
          asm volatile("" : "+v"(v[sb][r])); // (a branch: as selects every tile would pay two instructions per element)
        }
    };
    // the largest score of the tile in log2 units, mask term included
    auto row_max = [&](const f32x16 (&v)[2]) {
      float m0 = NEG_INF, m1 = NEG_INF;
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        m0 = max3(m0, v[0][r], v[0][r + 1]);
        m1 = max3(m1, v[1][r], v[1][r + 1]);
      }
      return xhalf_max(fmaxf(m0, m1)) * s;
    };
    // unrounded row sum (this half-wave's share), on four accumulators
    auto add_up = [&](const f32x16 (&v)[2]) {
      float t[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) t[r & 3] += v[sb][r];
      return (t[0] + t[1]) + (t[2] + t[3]);
    };
    if (diag) hide_later_keys(x);
    // a row's first tile with a key that is not masked out sets its reference (wave-uniform branch: as a rule the first tile's only)
    if (__builtin_amdgcn_ballot_w64(!seen)) {
      const float mx = row_max(x);
      if (!seen && mx > -1e20f) {
        M = __builtin_ceilf(mx); // (nothing has been accumulated before)
        seen = true;
      }
    }
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int r = 0; r < 16; ++r) x[sb][r] = fast_exp2(fmaf(x[sb][r], s, -M));
    float psum = 0.f;
    if (want_lse) psum = add_up(x);
    i32x8 pb;
#pragma unroll
    for (int sb = 0; sb < 2; ++sb)
#pragma unroll
      for (int g = 0; g < 4; ++g) pb[sb * 4 + g] = pack4_e4m3(x[sb][4 * g], x[sb][4 * g + 1], x[sb][4 * g + 2], x[sb][4 * g + 3]);
    float tsum = mfma_fp4_fp8_k128(ones, pb, zero)[0]; // of the rounded probabilities of this lane's row
    // Slow path, wave-uniform: a row sum beyond the range that guarantees representable probabilities (compared as
    // bit patterns: the sum is never negative, and a NaN from a saturated conversion must take this path although the
    // build tells the compiler that NaNs do not occur).  The scores are recomputed from the operands (the fast path has
    // overwritten them), the reference becomes ceil(max), everything is rescaled by the exact power of two.
    // Only the rows that need it change their reference (and take the recomputed probabilities): a row's result
    // depends on that row alone, whatever rows share its wave.
    if (__builtin_amdgcn_ballot_w64(__float_as_uint(tsum) > __float_as_uint(SUM_LIMIT))) {
      bool need = __float_as_uint(tsum) > __float_as_uint(SUM_LIMIT);
      if (__builtin_amdgcn_ballot_w64(__float_as_uint(tsum) > 0x7f800000u)) { // (wave-uniform, as the product wants all lanes)
        const bool over = clear_nan_row(pb);
        tsum = mfma_fp4_fp8_k128(ones, pb, zero)[0];
        need = over || tsum > SUM_LIMIT;
      }
      f32x16 y[2];
#pragma unroll
      for (int sb = 0; sb < 2; ++sb) {
#pragma unroll
        for (int r = 0; r < 16; ++r) y[sb][r] = 0.f;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
          const char *kp = ldsK + (sb * 32 + ql) * PITCH + ds * 64 + h * 32;
          const u32x4 lo = *(const u32x4 *)kp, hi = *(const u32x4 *)(kp + 16);
          const i32x8 ka = {(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
          y[sb] = mfma_fp8_k64(ka, qreg[ds], y[sb]);
        }
        if (extra) {
          const bf16x8 xa = as_v8<__bf16>(*(const u32x4 *)(ldsX + (sb * 32 + ql) * XROWB));
          y[sb] = Elem<__bf16>::mfma(xa, as_v8<__bf16>(u32x4{bx0, bx1, 0, 0}), y[sb]);
        }
      }
      if (diag) hide_later_keys(y);
      const float mx = row_max(y), Mn = need ? fmaxf(M, __builtin_ceilf(mx)) : M;
      const float alpha = fast_exp2(M - Mn); // (1 where the reference stays)
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int r = 0; r < 16; ++r) y[sb][r] = fast_exp2(fmaf(y[sb][r], s, -Mn));
      const float psum_new = add_up(y);
      psum = need ? psum_new : psum;
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int pn = pack4_e4m3(y[sb][4 * g], y[sb][4 * g + 1], y[sb][4 * g + 2], y[sb][4 * g + 3]);
          pb[sb * 4 + g] = need ? pn : pb[sb * 4 + g]; // (both half-waves of a row decide alike: the sums they test are the row's)
        }
      const bool lost = clear_nan_row(pb); // (a NaN among the inputs: the row's output is one)
      tsum = mfma_fp4_fp8_k128(ones, pb, zero)[0];
#pragma unroll
      for (int i = 0; i < 8; ++i) pb[i] = lost ? 0x7f7f7f7f : pb[i];
      l_run *= alpha;
      l_true *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[db][r] *= alpha;
      M = Mn;
    }
    l_run += tsum;
    if (want_lse) l_true += psum;
    // O^T += V^T.P^T: one K = 64 product per 32 head-dim columns
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      i32x8 va;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int gp = 0; gp < 2; ++gp) {
          const i32x2v t = lds_read_tr8(ldsV + trofs + (32 * b + 16 * gp) * PITCH + db * 32);
          va[4 * b + 2 * gp] = t.x;
          va[4 * b + 2 * gp + 1] = t.y;
        }
      oacc[db] = mfma_fp8_k64(va, pb, oacc[db]);
    }
    if (SPLIT) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      stage_next(kt);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    } else {
      __syncthreads(); // this stage is free again, the next one is complete
    }
  }
  if (!SPLIT) for (int kt = nktw; kt < nkt; ++kt) {
    stage_next(kt);
    __syncthreads();
  }

  l_true = xhalf_sum(l_true);
  TO *Or = (TO *)a.o + ((size_t)bh * a.sq + q) * D;
  if (SPLIT) {
    // The waves' partial rows meet in LDS: references are integers, so bringing them to the largest is exact.
    __syncthreads();
    f32x4 *part = (f32x4 *)lds;
    float *rows = (float *)(lds + C::LDS_MERGE);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        part[((w * DB + db) * 4 + g) * 64 + l] = f32x4{oacc[db][4 * g], oacc[db][4 * g + 1], oacc[db][4 * g + 2], oacc[db][4 * g + 3]};
    if (h == 0) {
      rows[(w * 3 + 0) * 32 + ql] = seen ? M : NEG_INF;
      rows[(w * 3 + 1) * 32 + ql] = l_run;
      rows[(w * 3 + 2) * 32 + ql] = l_true;
    }
    __syncthreads();
    if (w >= DB) return; // a wave for each 32 columns
    float top = NEG_INF, alpha[C::NW];
#pragma unroll
    for (int j = 0; j < C::NW; ++j) top = fmaxf(top, rows[j * 3 * 32 + ql]);
    M = top == NEG_INF ? 0.f : top;
    l_run = l_true = 0.f;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int j = 0; j < C::NW; ++j) {
      alpha[j] = fast_exp2(rows[j * 3 * 32 + ql] - M);
      l_run += alpha[j] * rows[(j * 3 + 1) * 32 + ql];
      l_true += alpha[j] * rows[(j * 3 + 2) * 32 + ql];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 v = part[((j * DB + w) * 4 + g) * 64 + l];
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[4 * g + i] += alpha[j] * v[i];
      }
    }
    if (q < a.sq) {
      const float inv = l_run > 0.f ? a.out_scale / l_run : 0.f;
      store_acc_block_row<TO>(Or + w * 32, acc, inv, h);
      if (a.lse && h == 0 && w == 0) a.lse[(size_t)bh * a.sq + q] = l_true > 0.f ? (M + fast_log2(l_true)) * FMHA_LN2 : NEG_INF;
    }
    return;
  }
  // normalise and store: in the accumulator layout lane (q, h) holds head-dim columns 8g + 4h .. +3 of each 32-block
  if (q < a.sq) {
    const float inv = l_run > 0.f ? a.out_scale / l_run : 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) store_acc_block_row<TO>(Or + db * 32, oacc[db], inv, h);
    if (a.lse && h == 0) a.lse[(size_t)bh * a.sq + q] = l_true > 0.f ? (M + fast_log2(l_true)) * FMHA_LN2 : NEG_INF;
  }
}

} // namespace fmha
