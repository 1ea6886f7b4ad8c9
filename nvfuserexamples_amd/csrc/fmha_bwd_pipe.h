// Software-pipelined backward kernels for head dims up to 128 (96: dQ), and dQ at 256 (no mask or a per-key mask; full mask tensors stay on
// fmha_bwd_kernel.h).  Mathematics, register layouts and the extra contraction step are those of fmha_bwd_kernel.h, whose
// header describes them; what changes is the order of work and how tiles arrive:
//
//   * 32-row tiles, four resident per operand.  The copies of tile t + 3 are spread over iteration t, one instruction
//     every few matrix instructions (in one burst behind the barrier they stall the issuing waves: 226 -> 216 us for dQ at
//     BH 256 S 1024 D 128), and are waited for two iterations later with a count (`vmcnt(N)`), so no iteration waits for
//     memory it has just asked for.  Tiles past the end re-read the last row instead of being skipped: every iteration
//     issues the same number of copies and the counts are constants.  The first tiles are asked for before anything else.
//   * Iteration t is one hand-ordered stream: the first products of tile t + 1 beside the exponentials of tile t (two sets
//     of score / dP accumulators), then the gradient products of tile t, with the Philox call of tile t + 1 beside them.
//     LDS operands are requested three or four matrix instructions ahead.  A scheduling barrier closes every slot and
//     values are pinned to theirs (the compiler sinks exponentials towards their use otherwise).
//   * Causal: a wave leaves out the tiles on the masked side of its own diagonal, and only the tile on it compares indexes.
//   * The per-key mask terms (dQ) and the rows (-LSE, -delta) (dK / dV) of the whole head are staged in LDS once, in
//     segments of 4096 keys / 1024 queries, instead of per tile through registers: a load that the compiler waits for
//     would also wait for every copy issued ahead of it.  (Where there is more than one segment, the second tile of a
//     causal pair stages its first one again: the other tile's pass has overwritten it.)
//   * Gradients leave as whole rows (store_acc_rows).
//
// Measured against the two-stage, phase-by-phase kernels on one card (kernel times, us, dQ / dK+dV, fp16 unless said): BH 64
// S 2048 D 64 without dropout 126.9 / 159.3 -> 116.6 / 153.1, with dropout 140.0 / 194.5 -> 135.9 / 174.7; BH 192 S 1024 D 64
// causal 84.3 / 98.2 -> 66.4 / 81.9; BH 32 S 4096 D 128 causal 280 / 335 -> 225 / 304 (bf16 272 / 329 -> 214 / 275); BH 512
// S 1024 D 128 causal bf16 285 / 455 -> 293 / 413, before dQ there lost the registers that spilled into its stream (300 -> 246 on another
// card; the lines between the two kinds of kernel at head dim 128: fmha_bwd.hip).
// What bounds them: at head dim 64 the issue slots (a matrix instruction takes the vector pipe for about 21 cycles, a
// vector instruction for 2.5, and the sum of both is what two waves per SIMD need); at head dim 128 the board's power
// (dQ on random data: 1.57 GHz, on zeros 2.19 GHz) and, for dK / dV at one wave per SIMD, the start and the stores of
// workgroups that all compute units run in step (without stores 328 -> 255 us at BH 256 S 1024).
#pragma once
#include "fmha_bwd_kernel.h"

namespace fmha {

FMHA_DEV void bwd_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
template <int N> FMHA_DEV void bwd_vm_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

template <int D> struct BwdPipeCfg {
  static constexpr int BT = 32, NST = 4; // rows per tile, tiles resident per operand
  static constexpr int KS = D / 16, DB = D / 32;
  static constexpr int TILEB = BT * tile_cols(D) * 2, STAGEB = 2 * TILEB;
  static constexpr bool TURNED = D == 64 || D == 128;                       // register operands are read as whole rows (RowOperands)
  static constexpr int OFF_T = (NST - 1) * STAGEB, TURNB = 32 * kPanelRowB; // ... and turned here, in the last stage, a panel per wave
  static constexpr int OFF_X = D == 64 ? OFF_T + 4 * TURNB : NST * STAGEB;
  static_assert(!TURNED || 4 * TURNB + OFF_T <= OFF_X, "a panel for each of four waves");
  static_assert(4 * RowStore<D>::BYTES <= OFF_X, "the output rows are turned in the tiles' LDS");
  static constexpr int MSEG = 4096;             // per-key mask terms staged at once
  static constexpr int QSEG = 1024;             // queries whose extra-step rows are staged at once (dK / dV)
  static int dkdv_lds_bytes(int drop, int sq) { return OFF_X + 64 + (sq < QSEG ? (16 + (drop ? 4 : 0)) * ((sq + 31) / 32 * 32) : (16 + (drop ? 8 : 0)) * QSEG); }
  static int dq_lds_bytes(int mask, int sk) { return OFF_X + (mask == kMaskPerKey ? 4 * (sk < MSEG ? (sk + 31) / 32 * 32 : MSEG) : 0) + 64; }
};

// Copies of 32-row tiles of a row-major [rows][D] matrix into swizzled LDS tiles, one instruction at a time so that
// they can be spread over an instruction stream: rows past the end re-read the last one (a minimum on the byte offset,
// no branch), so tiles that do not exist may be asked for and every tile costs the same number of copies.  Columns a
// row does not have are filled with its first ones: they meet zeros in the register operand, or land in output columns
// that are not stored.
template <typename T, int D, int NT> struct PipeCopy {
  static constexpr int BT = 32, CPT = BT * tile_cols(D) / 8 / NT;
  static_assert(CPT * NT * 8 == BT * tile_cols(D), "tile must divide evenly over the workgroup");
  uint32_t voff[CPT], lim[CPT], dst;
  uint32_t tile_step; // bytes between the first rows of consecutive tiles
  FMHA_DEV void init(int tid, int64_t row_stride, int rend, int dv) {
    const uint32_t ss2 = (uint32_t)row_stride * 2u;
    tile_step = ss2 * BT;
    dst = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6) * 1024u;
#pragma unroll
    for (int i = 0; i < CPT; ++i) {
      int row, col;
      TileCopy<T, D, BT, NT>::slot(tid + i * NT, row, col);
      const uint32_t cb = col * 8 < dv ? (uint32_t)col * 16u : 0u;
      voff[i] = (uint32_t)row * ss2 + cb;
      lim[i] = (uint32_t)(rend - 1) * ss2 + cb;
    }
  }
  FMHA_DEV void issue(const T *base, int tile, uint32_t lds_tile, int i) const {
    const uint32_t o = voff[i] + (uint32_t)tile * tile_step;
    dma_global_to_lds_b128(base, o < lim[i] ? o : lim[i], lds_tile + dst + (uint32_t)(i * NT * 16));
  }
};

// A wave's 32 rows as register operands: lane (row l % 32, half l / 32) gets columns 16 ks + 8 (l / 32) .. +7.  Loaded as they are
// wanted, an instruction touches 32 rows, 32 bytes of each.  Here whole panel rows are loaded, eight lanes a row, and turned through a
// panel of the wave's own LDS.  Backward, us, loaded as wanted / so: D 128 BH 512 S 1024 bf16 causal 642 / 623, S 384 169 / 166, packed
// with dropout S 512 369 / 358; D 64 BH 512 S 1024 causal 343 / 331, packed S 512 170 / 166, BH 256 S 800 with dropout 234 / 229,
// BH 100 S 400 31.8 / 30.6; level to 1.5 % behind on whole rows without mask and dropout, BH 512 S 512 157 / 158.
// Rows of 33 to 63 columns that follow on each other (heads folded) fill the lines they are in as they are, and short heads of them pay for
// the way through LDS: without a causal mask they are loaded as wanted (D 48, 16 to 128
// heads of 64 to 320 rows 4 to 6 % less, 512 heads level).  Under one the kernels have no registers for both ways (D 48
// and 112 10 to 12 % behind), and at head dim 128 the way through LDS is level to 1 % ahead.
template <typename T, int D> struct RowOperands {
  static constexpr int NI = 32 * tile_cols(D) / 8 / 64;
  u32x4 v[NI];
  FMHA_DEV void load(const T *base, uint32_t ss, int row0, int rend, int cols, int l) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      int row, col;
      TileCopy<T, D, 32, 64>::slot(l + i * 64, row, col);
      int r = row0 + row;
      r = r < rend ? r : rend - 1;
      v[i] = *(const u32x4 *)(base + (size_t)(uint32_t)r * ss + (col * 8 < cols ? col * 8 : 0)); // (as in PipeCopy)
    }
  }
  FMHA_DEV void turn(char *panel, const PanelLane &pl, int l, u32x4 (&out)[D / 16]) const {
#pragma unroll
    for (int p = 0; p < NI / 4; ++p) {
      asm volatile("" ::: "memory"); // (a wave's LDS accesses execute in order)
#pragma unroll
      for (int i = 0; i < 4; ++i) *(u32x4 *)(panel + (l + i * 64) * 16) = v[4 * p + i];
      asm volatile("" ::: "memory");
#pragma unroll
      for (int ks = 4 * p; ks < 4 * p + 4 && ks < D / 16; ++ks) out[ks] = as_u32x4(panel_read_rows<T, 32>(panel, pl, 0, ks & 3));
    }
    asm volatile("" ::: "memory");
  }
};

// Products on score / dP accumulators that stay in the first half of the register file, where the vector pipe reads them.  Left to
// the compiler, all accumulators of a kernel that needs both halves go to the second one, and 32 moves a tile bring these back
// (backward at head dim 128, us, so / with these: BH 512 S 1024 causal bf16 637 / 606, with dropout 769 / 722, BH 256 S 1024 482 / 469,
// BH 32 S 4096 821 / 803, BH 512 S 512 under a padding mask with dropout 339 / 329).  The compiler does not see into them: behind
// the last one `settle` before anything but another product reads the result.
template <typename T> struct MfmaV;
template <> struct MfmaV<_Float16> {
  static FMHA_DEV void start(f16x8 a, f16x8 b, f32x16 &c) { asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b)); }
  static FMHA_DEV void add(f16x8 a, f16x8 b, f32x16 &c) { asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
};
template <> struct MfmaV<__bf16> {
  static FMHA_DEV void start(bf16x8 a, bf16x8 b, f32x16 &c) { asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b)); }
  static FMHA_DEV void add(bf16x8 a, bf16x8 b, f32x16 &c) { asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
};
FMHA_DEV void settle(f32x16 &x, f32x16 &g) { asm volatile("s_nop 15" : "+v"(x), "+v"(g)); } // (twelve wait states are due, this is sixteen)

// One Philox4x32-10 call in slices that can be spread over an instruction stream.
struct PhiloxSlices {
  uint32_t c[4];
  // Both halves of a product are wanted, one round apart: said so, it is one v_mad_u64_u32 (the compiler made v_mul_lo and v_mul_hi,
  // each as dear, of half of them).
  static FMHA_DEV uint64_t product(uint32_t c, uint32_t m) {
    uint64_t p = (uint64_t)c * m;
    asm volatile("" ::"v"(p));
    return p;
  }
  // With round 0: its offset is the same for all lanes like the key, and so is what round 1 adds to c[3].  These scalars meet here: the
  // instruction of `round` reads one scalar at most, and copies of the others in vector registers, kept across the loop around it, made
  // dQ at head dim 128 reload five spilled registers a turn, each behind all copies in flight (backward with dropout, us, as copies / so:
  // D 128 BH 96 S 700 causal packed under a padding mask 97.9 / 95.0, BH 64 S 2048 causal 314 / 309, BH 256 S 1024 556 / 550; D 64 BH 512
  // S 512 under a padding mask 184.6 / 180.1; D 32 BH 512 S 512 135 / 132).
  FMHA_DEV void start(const DropCtx &d, uint32_t bh, uint32_t q4, uint32_t k4) {
    const uint64_t blk = ((uint64_t)bh * d.qb4 + q4) * d.kb4 + k4;
    const uint64_t p0 = (uint64_t)Philox::M0 * d.off_lo, p1 = product((uint32_t)blk, Philox::M1);
    c[0] = (uint32_t)(p1 >> 32) ^ (d.off_hi ^ d.seed_lo);
    c[1] = (uint32_t)p1;
    c[2] = (uint32_t)(blk >> 32) ^ ((uint32_t)(p0 >> 32) ^ d.seed_hi);
    c[3] = (uint32_t)p0 ^ (d.seed_hi + Philox::W1);
  }
  FMHA_DEV void round(const DropCtx &d, int r) {
    if (r == 0) return;
    const uint32_t k0 = d.seed_lo + (uint32_t)r * Philox::W0, k1 = r == 1 ? 0u : d.seed_hi + (uint32_t)r * Philox::W1;
    const uint64_t p0 = product(c[0], Philox::M0), p1 = product(c[2], Philox::M1);
    const uint32_t n0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c[1], k0, 0x96);
    const uint32_t n2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c[3], k1, 0x96);
    c[0] = n0;
    c[1] = (uint32_t)p1;
    c[2] = n2;
    c[3] = (uint32_t)p0;
  }
};

// ------------------------------------------------------------------------------ dQ
// (waves per SIMD: at head dim 256 a wave needs about 400 registers, and the tiles leave room for one workgroup; at 32 without a
// causal mask three waves have the 150 it needs: with dK / dV at three as well BH 512 S 512 backward 96 -> 89 us, BH 1760 S 64 under a padding mask 35 -> 29)
template <int D, bool CAUSAL> constexpr int bwd_dq_pipe_occ() { return D == 256 ? 1 : D == 32 && !CAUSAL ? 3 : 2; }
// A query's LSE and delta are constants of its lane: where registers have room for 32 copies, the products of x and g start from them,
// and neither an extra contraction step (two of a tile's 14 matrix instructions at head dim 64, and the only one left is a mask's) nor
// a subtraction per element brings them in.  Backward, us, before / so: D 64 BH 64 S 2048 239.6 / 234.4, with dropout 295.7 / 290.7, key
// counts 201.3 / 196.4, BH 512 S 512 packed with dropout 184.9 / 182.2, BH 192 S 1024 bf16 causal 120.4 / 118.0; D 96 BH 64 S 2048 363.7 /
// 353.2, BH 512 S 512 under a padding mask 220.3 / 213.3; D 32 BH 512 S 512 causal 77.7 / 75.8; up to 700 queries of 24 heads level.
// No room: D 32 at three waves and D 96, each with dropout (16 to 20 registers spill), and D 128.
template <int D, bool CAUSAL, int DROP> constexpr bool bwd_dq_pipe_constants() { return D == 64 || (D == 96 && DROP == 0) || (D == 32 && (CAUSAL || DROP == 0)); }
template <typename T, int D, int NW, int MASK, bool CAUSAL, int DROP, bool STRIDED>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(bwd_dq_pipe_occ<D, CAUSAL>(), bwd_dq_pipe_occ<D, CAUSAL>()))) void fmha_bwd_dq_pipe_kernel(const BwdArgs a) {
  using RW = Rows<STRIDED, D>;
  using E = Elem<T>;
  using v8 = typename E::v8;
  using C = BwdPipeCfg<D>;
  constexpr int BT = C::BT, NST = C::NST, KS = C::KS, DB = C::DB, TILEB = C::TILEB, STAGEB = C::STAGEB;
  constexpr int NT = NW * 64, QT = NW * 32;
  constexpr float NEG_INF = -__builtin_inff();
  constexpr float BIGNEG = -60000.f;
  static_assert(MASK != kMaskFull, "full mask tensors: fmha_bwd_dq_kernel");
  // Rank-one terms that the products do not start from (CI): at head dims up to 64 the vector pipe is the busier one and they ride in
  // an extra contraction step (XS, GX); above it is the matrix pipe, and a subtraction per element costs less.  A per-key mask always
  // rides in one.
  constexpr bool CI = bwd_dq_pipe_constants<D, CAUSAL, DROP>();
  constexpr bool XS = (D <= 64 && !CI) || MASK == kMaskPerKey, GX = D <= 64 && !CI; // x, g have an extra step
  constexpr bool GS = D <= 64 || CI, LS = GS;                                       // they come with delta, with the LSE

  extern __shared__ __attribute__((aligned(16))) char lds[];
  uint32_t *ldsM = (uint32_t *)(lds + C::OFF_X + 64); // (mask_hi, mask_lo) per key of the current segment
  int *ldsR = (int *)(lds + C::OFF_X);

  const int tid = threadIdx.x;
  const int w = tid >> 6, l = tid & 63, ql = l & 31, h = l >> 5;

  int bh, pi, npass;
  bwd_item<CAUSAL, bwd_dq_pipe_occ<D, CAUSAL>() == 2, !CAUSAL>(a, bh, pi, npass);

  const T *Qb = (const T *)a.q + RW::head(a.mq, bh, a.sq);
  const T *Ob = (const T *)a.o + RW::head(a.mo, bh, a.sq);
  const T *dOb = (const T *)a.dout + RW::head(a.mdo, bh, a.sq);
  const T *Kb = (const T *)a.k + RW::head(a.mk, bh, a.sk);
  const T *Vb = (const T *)a.v + RW::head(a.mv, bh, a.sk);
  const T *mkey = (MASK == kMaskPerKey) ? (const T *)a.mask + (size_t)(bh / a.mask_div) * a.mask_sb : nullptr;
  const int skv0 = bwd_valid_keys(a, bh);
  int skv = skv0; // keys worth visiting

  // Terms of a segment of the mask row -> LDS; returns (uniform) the number of keys up to the last one that is not
  // hard-masked.
  auto stage_mask = [&](int seg0) -> int {
    constexpr float kHardMask = -9000.f * FMHA_LOG2E;
    const int n = a.sk - seg0 < C::MSEG ? a.sk - seg0 : C::MSEG;
    int last = -1;
    for (int base = 0; base < n; base += 4 * NT) {
      T v[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int key = seg0 + base + c * NT + tid;
        v[c] = mkey[key < a.sk ? key : a.sk - 1];
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int i = base + c * NT + tid;
        float mk = fmaf((float)v[c], a.mask_a, a.mask_b);
        const bool live = i < n && mk > kHardMask;
        const unsigned long long bal = __builtin_amdgcn_ballot_w64(live);
        if (bal) last = base + c * NT + (tid & ~63) + 63 - __builtin_clzll(bal);
        if (seg0 + i >= skv0) mk = BIGNEG;
        T hl[2];
        split_hi_lo<T>(mk, hl[0], hl[1]);
        if (i < (n + 31) / 32 * 32) ldsM[i] = __builtin_bit_cast(uint32_t, *(const __attribute__((ext_vector_type(2))) T *)hl);
      }
    }
    if ((tid & 63) == 0) ldsR[w] = last;
    __syncthreads();
    int top = -1;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) top = ldsR[ww] > top ? ldsR[ww] : top;
    return __builtin_amdgcn_readfirstlane(top) + 1;
  };

  for (int pass = 0; pass < npass; ++pass) {
    // (From head dim 64 on set up for each pass, from an index that the compiler cannot trace: kept from one pass to the next, what a lane
    // addresses had 33 to 59 registers spilled into the stream at 128, and would have up to 9 at 64.  Backward, us: BH 512 S 1024 bf16 698 -> 649, with dropout 836 -> 776,
    // BH 128 S 900 167 -> 154, BH 32 S 4096 497 -> 485.  Where nothing spills it costs the second pass 1 to 2 %.)
    int tid = threadIdx.x;
    if (CAUSAL && D >= 64) asm volatile("" : "+v"(tid));
    const int w = tid >> 6, l = tid & 63, ql = l & 31, h = l >> 5;
    const int qt = CAUSAL ? (pass == 0 ? a.ntile - 1 - pi : pi) : pi;
    const int q0w = qt * QT + w * 32;
    const int q = q0w + ql;

    // ---- tiles 0..2 on their way, ahead of everything that waits for memory
    const uint32_t lds_base = lds_address(lds);
    PipeCopy<T, D, NT> tcopy;
    tcopy.init(tid, RW::ss(a.mk), a.sk, RW::cols(a));
    constexpr int VPT = 2 * PipeCopy<T, D, NT>::CPT; // copies per tile pair and wave
    auto dma_one = [&](int kt, int i) { // copy i of the K and V tiles kt
      const uint32_t dst = lds_base + (uint32_t)(kt & (NST - 1)) * STAGEB;
      if (i < VPT / 2) tcopy.issue(Kb, kt, dst, i);
      else tcopy.issue(Vb, kt, dst + TILEB, i - VPT / 2);
    };
    auto dma_kv = [&](int kt) {
#pragma unroll
      for (int i = 0; i < VPT; ++i) dma_one(kt, i);
    };
#pragma unroll
    for (int t = 0; t < NST - 1; ++t) dma_kv(t);

    PanelLane pl;
    pl.init(l);
    // ---- per-row operands (all loads unconditional, see fmha_bwd_dq_kernel)
    v8 qreg[KS], doreg[KS], bxs, bxd;
    float delta, nlse;
    {
      const int qc = q < a.sq ? q : a.sq - 1;
      u32x4 tq[KS], td[KS], to[KS];
      const bool turned = C::TURNED && (CAUSAL || D != 64 || !STRIDED || RW::ss(a.mq) != (uint32_t)RW::cols(a)); // (see RowOperands)
      RowOperands<T, D> rq, rd, ro;
      if (turned) {
        rq.load(Qb, RW::ss(a.mq), q0w, a.sq, RW::cols(a), l);
        rd.load(dOb, RW::ss(a.mdo), q0w, a.sq, RW::cols(a), l);
        ro.load(Ob, RW::ss(a.mo), q0w, a.sq, RW::cols(a), l);
      } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const size_t col = ks * 16 + h * 8 < RW::cols(a) ? ks * 16 + h * 8 : 0;
          tq[ks] = *(const u32x4 *)(Qb + (size_t)qc * RW::ss(a.mq) + col);
          td[ks] = *(const u32x4 *)(dOb + (size_t)qc * RW::ss(a.mdo) + col);
          to[ks] = *(const u32x4 *)(Ob + (size_t)qc * RW::ss(a.mo) + col);
        }
      }
      float lse_q = a.lse[(size_t)bh * a.sq + qc];
      if (MASK == kMaskPerKey && (pass == 0 || a.sk > C::MSEG)) { // (with more than one segment the first pass leaves a later one)
        const int n = stage_mask(0); // (its loads share the trip to memory)
        const bool trim = a.sk > 128 && a.sk <= C::MSEG && !(a.flags & kBwdFlagNoTrim);
        if (trim && n > 0 && n < skv) skv = n; // a row without any live key keeps all its keys
      }
      if (turned) {
        char *panel = lds + C::OFF_T + w * C::TURNB;
        rq.turn(panel, pl, l, tq);
        rd.turn(panel, pl, l, td);
        ro.turn(panel, pl, l, to);
      }
      asm volatile("" : "+v"(lse_q));
      float dsum = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bool live = ks * 16 + h * 8 < RW::cols(a);
        const v8 qraw = as_v8<T>(chunk_or_zero(tq[ks], live));
        const v8 doraw = as_v8<T>(chunk_or_zero(td[ks], live));
        const v8 ov = as_v8<T>(to[ks]);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          qreg[ks][j] = (T)((float)qraw[j] * a.scale_l2);
          doreg[ks][j] = DROP == 1 ? (T)((float)doraw[j] * a.drop_scale) : doraw[j];
          dsum = fmaf((float)doraw[j], (float)ov[j], dsum);
        }
      }
      dsum = xhalf_sum(dsum);
      delta = dsum;
      float nl = BIGNEG; // rows past the end and fully masked rows get P = 0
      if (q < a.sq) {
        if (lse_q != NEG_INF) nl = -lse_q * FMHA_LOG2E;
        if (h == 0) a.delta[(size_t)bh * a.sq + q] = dsum;
      }
      nlse = nl;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        bxs[j] = (T)0.f;
        bxd[j] = (T)0.f;
      }
      if (h == 0) {
        T hi, lo;
        split_hi_lo<T>(LS && !CI ? nl : 0.f, hi, lo);
        bxs[0] = hi;
        bxs[1] = lo;
        bxs[2] = (T)1.f;
        bxs[3] = (T)1.f;
        split_hi_lo<T>(-dsum, hi, lo);
        bxd[0] = hi;
        bxd[1] = lo;
      }
    }

    int nkt = (skv + BT - 1) / BT;
    if (nkt < 1) nkt = 1;
    if (CAUSAL) {
      int qmax = qt * QT + QT - 1;
      if (qmax > a.sq - 1) qmax = a.sq - 1;
      const int need = qmax / BT + 1;
      if (need < nkt) nkt = need;
    }
    const int kend = nkt * BT < skv ? nkt * BT : skv;
    const int last_key = CAUSAL && q < kend - 1 ? q : kend - 1; // of this lane's row
    // causal: tiles past the one that holds this wave's own diagonal are all masked for it
    const int ws = __builtin_amdgcn_readfirstlane(w);
    int nktw = nkt;
    if (CAUSAL) {
      const int own = (qt * QT + ws * 32) / BT + 1;
      nktw = own < nkt ? own : nkt;
    }

    constexpr uint32_t ONES = std::is_same<T, _Float16>::value ? 0x3c003c00u : 0x3f803f80u;
    constexpr uint32_t BIGPAIR = std::is_same<T, _Float16>::value ? 0x0000fb53u : 0x0000c76au; // (-60000 in T, 0)
    auto hl_of = [&](int kt) -> uint32_t { // (mask_hi, mask_lo) of key (l % 32) of a tile
      const int key = kt * BT + ql;
      if (MASK == kMaskPerKey) {
        const uint32_t m = ldsM[key & (C::MSEG - 1)];
        return key < kend ? m : BIGPAIR;
      }
      return key < kend ? 0u : BIGPAIR;
    };
    auto xa_of = [&](uint32_t hl) -> v8 { return as_v8<T>(u32x4{ONES, hl, 0u, 0u}); };

    f32x16 cx, cg; // what the products of x and g start from
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      cx[r] = CI ? nlse : 0.f;
      cg[r] = CI ? -delta : 0.f;
    }
    if (CI) asm volatile("" : "+v"(cx), "+v"(cg)); // (left alone the compiler forms them anew for each tile)

    f32x16 dq[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) dq[db][r] = 0.f;

    f32x16 xA, gA, xB, gB;
    uint32_t wdA[4], wdB[4];
    PhiloxSlices ph;

    // The stream of one tile: first products of tile kt + 1 into (xn, gn) beside the softmax of tile kt (xc, gc),
    // then dQ^T += K(kt)^T.dS(kt)^T; the Philox call of tile kt + 1 behind the softmax.
    auto step = [&](auto next_tag, auto guard_tag, int kt, uint32_t hl, const f32x16 &xc, const f32x16 &gc,
                    const uint32_t (&wc)[4], f32x16 &xn, f32x16 &gn, uint32_t (&wn)[4]) {
      constexpr bool NEXT = decltype(next_tag)::value, GUARD = decltype(guard_tag)::value;
      constexpr int NX = NEXT ? (XS ? 1 : 0) + (GX ? 1 : 0) : 0, NA = NEXT ? 2 * KS : 0, NC = 2 * DB, NO = NA + NC, NM = NX + NO;
      constexpr int AHEAD = 3;
      constexpr int NS = 10;                                  // softmax slots: 8 pairs, two to drain
      constexpr int NP = DROP == 1 && NEXT ? 14 : 0;          // Philox slots
      constexpr int JS = NEXT ? NX + NA : 0;                  // the softmax is done before matrix instruction JS
      const char *ldsN = lds + ((kt + 1) & (NST - 1)) * STAGEB;
      const char *ldsC = lds + (kt & (NST - 1)) * STAGEB;
      const int k0 = kt * BT;
      auto fetch = [&](int j) -> v8 {
        if (j < NA) return panel_read_rows<T, BT>(ldsN + (j & 1) * TILEB, pl, 0, j >> 1);
        const int i = j - NA;
        return panel_read_transposed<T, BT>(ldsC, pl, 0, i % DB, i / DB);
      };
      float p[16];
      bool keep[16];
      v8 frag[2];
      auto softmax = [&](int s) {
        if (s < 8) {
#pragma unroll
          for (int e = 2 * s; e < 2 * s + 2; ++e) {
            float xv = xc[e];
            if (!LS) xv += nlse;
            if (GUARD) xv = (k0 + 8 * (e / 4) + 4 * h + e % 4 <= last_key) ? xv : BIGNEG;
            p[e] = fast_exp2(xv);
            asm volatile("" : "+v"(p[e])); // (stays in this slot: left alone the compiler sinks it towards its use)
            if (DROP == 1) keep[e] = drop_keep_byte(wc[e / 4], e % 4, a.drop.thr); // (used one slot on: no wait for it)
          }
        }
        if (s >= 1 && s < 9) {
#pragma unroll
          for (int e = 2 * (s - 1); e < 2 * s; ++e) {
            float gv = gc[e];
            if (DROP == 1) gv = keep[e] ? gv : (GS ? -delta : 0.f);
            if (!GS) gv -= delta;
            p[e] *= gv;
            asm volatile("" : "+v"(p[e]));
          }
        }
        if (s >= 2) {
#pragma unroll
          for (int e = 2 * (s - 2); e < 2 * (s - 1); ++e) frag[e / 8][e % 8] = (T)p[e];
        }
      };
      auto philox = [&](int s) {
        if (s == 0) ph.start(a.drop, (uint32_t)bh, (uint32_t)q >> 2, (uint32_t)((k0 + BT) >> 2) + (uint32_t)h + 2u * ((uint32_t)l & 3u));
        else if (s <= 10) ph.round(a.drop, s - 1);
        else if (s == 11) {
#pragma unroll
          for (int i = 0; i < 4; ++i) wn[i] = ph.c[i];
          quad_transpose4(wn, l);
        }
      };
      v8 opnd[NO];
#pragma unroll
      for (int j = 0; j < AHEAD && j < NO; ++j) opnd[j] = fetch(j);
      int done = 0;
      if (!NEXT) {
#pragma unroll
        for (; done < NS; ++done) softmax(done);
      }
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        if (m < NX) {
          const v8 xa = xa_of(hl);
          if (XS && m == 0) xn = E::mfma(xa, bxs, cx);
          else gn = E::mfma(xa, bxd, cg);
        } else {
          const int j = m - NX;
          if (j + AHEAD < NO) opnd[j + AHEAD] = fetch(j + AHEAD);
          if (j < NA) {
            if ((j & 1) == 0) xn = E::mfma(opnd[j], qreg[j >> 1], !XS && j == 0 ? cx : xn);
            else gn = E::mfma(opnd[j], doreg[j >> 1], !GX && j == 1 ? cg : gn);
          } else {
            const int i = j - NA;
            dq[i % DB] = E::mfma(opnd[j], frag[i / DB], dq[i % DB]);
          }
        }
        if (m % (NM / VPT) == NM / VPT - 1 && m / (NM / VPT) < VPT) dma_one(kt + NST - 1, m / (NM / VPT));
        const int upto = m < JS ? (m + 1) * NS / (JS ? JS : 1) : NS + (m - JS + 1) * NP / (NM - JS);
#pragma unroll
        for (; done < upto; ++done) {
          if (done < NS) softmax(done);
          else philox(done - NS);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    using Yes = std::true_type;
    using No = std::false_type;

    // ---- first products of tile 0 (its wait covers the loads above too: they are younger than its copies)
    uint32_t wd0[4];
    if (DROP == 1) drop_words_q(a.drop, (uint32_t)bh, (uint32_t)q, 0u, h, l, wd0); // (while the tiles are on their way)
    bwd_vm_wait<0>();
    bwd_lds_barrier();
    auto first = [&](auto odd, f32x16 &x, f32x16 &g, uint32_t (&wd)[4]) {
      asm volatile("" ::"n"(decltype(odd)::value) : "memory"); // (its reads stay on either side of the branch below: ahead of it they spill)
#pragma unroll
      for (int i = 0; i < 4 && DROP == 1; ++i) wd[i] = wd0[i];
      const v8 xa = xa_of(hl_of(0));
      constexpr int AHEAD = 2; // (operand pairs asked for ahead of their products)
      v8 ox[KS], og[KS];
      auto fetch = [&](int ks) {
        ox[ks] = panel_read_rows<T, BT>(lds, pl, 0, ks);
        og[ks] = panel_read_rows<T, BT>(lds + TILEB, pl, 0, ks);
      };
#pragma unroll
      for (int ks = 0; ks < AHEAD && ks < KS; ++ks) fetch(ks);
      x = XS ? E::mfma(xa, bxs, cx) : cx;
      g = GX ? E::mfma(xa, bxd, cg) : cg;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + AHEAD < KS) fetch(ks + AHEAD);
        x = E::mfma(ox[ks], qreg[ks], x);
        g = E::mfma(og[ks], doreg[ks], g);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // top of the iteration of tile kt: tile kt + 1 has landed, tile kt + 3 goes on its way
    // (`No`: for a wave's last tile, behind which nothing is read: the head may have no mask terms there, nor LDS for them)
    auto turn = [&](auto next_tag, int kt) -> uint32_t {
      if (MASK == kMaskPerKey && ((kt + 1) * BT & (C::MSEG - 1)) == 0 && kt + 1 < nkt) stage_mask((kt + 1) * BT); // (4096 keys on)
      uint32_t hl = 0u;
      if constexpr (decltype(next_tag)::value) hl = hl_of(kt + 1);
      bwd_vm_wait<(NST - 3) * VPT>();
      bwd_lds_barrier(); // ... everybody's part of it, and tile kt - 1 is no longer read
      return hl;
    };
    auto mid = [&](int kt, const f32x16 &xc, const f32x16 &gc, const uint32_t (&wc)[4], f32x16 &xn, f32x16 &gn, uint32_t (&wn)[4]) {
      const uint32_t hl = turn(Yes{}, kt);
      step(Yes{}, No{}, kt, hl, xc, gc, wc, xn, gn, wn);
    };
    int kt = 0;
    const int nmid = nktw - 1;
    if (nmid & 1) {
      first(Yes{}, xB, gB, wdB);
      mid(0, xB, gB, wdB, xA, gA, wdA);
      kt = 1;
    } else {
      first(No{}, xA, gA, wdA);
    }
    for (; kt < nmid; kt += 2) {
      mid(kt, xA, gA, wdA, xB, gB, wdB);
      mid(kt + 1, xB, gB, wdB, xA, gA, wdA);
    }
    {
      turn(No{}, kt);
      step(No{}, std::integral_constant<bool, CAUSAL || !XS>{}, kt, 0u, xA, gA, wdA, xB, gB, wdB);
      for (++kt; kt < nkt; ++kt) {
        turn(No{}, kt);
        dma_kv(kt + NST - 1);
      } // (causal: tiles that only later waves of the workgroup need)
    }

    bwd_vm_wait<0>(); // no copy may still be on its way into LDS when the wave ends, or the next pass starts
    bwd_lds_barrier(); // (every wave is done with the tiles: their LDS turns the output rows)
    {
      T *dQb = (T *)a.dq + RW::head(a.mdq, bh, a.sq) + (size_t)q0w * RW::ss(a.mdq);
      store_acc_rows<T, D>(lds + w * RowStore<D>::BYTES, dq, a.scale, dQb, RW::ss(a.mdq), a.sq - q0w, RW::cols(a), l);
    }
    __syncthreads(); // the next pass refills the tiles
  }
}

// --------------------------------------------------------------------------- dK, dV
// (with dropout three waves would spill 16 registers: head dim 32 BH 208 S 1602 487 -> 554 us)
template <int D, bool CAUSAL, int DROP> constexpr int bwd_dkdv_pipe_occ() { return D == 32 && !CAUSAL && DROP == 0 ? 3 : D <= 64 ? 2 : 1; }

template <typename T, int D, int NW, int MASK, bool CAUSAL, int DROP, bool STRIDED>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(bwd_dkdv_pipe_occ<D, CAUSAL, DROP>(), bwd_dkdv_pipe_occ<D, CAUSAL, DROP>()))) void fmha_bwd_dkdv_pipe_kernel(const BwdArgs a) {
  using RW = Rows<STRIDED, D>;
  using E = Elem<T>;
  using v8 = typename E::v8;
  using C = BwdPipeCfg<D>;
  constexpr int BT = C::BT, NST = C::NST, KS = C::KS, DB = C::DB, TILEB = C::TILEB, STAGEB = C::STAGEB;
  constexpr int NT = NW * 64, KT = NW * 32;
  constexpr float NEG_INF = -__builtin_inff();
  constexpr float BIGNEG = -60000.f;
  static_assert(MASK != kMaskFull, "full mask tensors: fmha_bwd_dkdv_kernel");

  extern __shared__ __attribute__((aligned(16))) char lds[];
  int *ldsR = (int *)(lds + C::OFF_X);
  u32x4 *ldsX = (u32x4 *)(lds + C::OFF_X + 64); // per query of the segment: (-L_hi, -L_lo, 1, 1, -delta_hi, -delta_lo, 0, 0)
  const int nseg = a.sq < C::QSEG ? (a.sq + 31) / 32 * 32 : C::QSEG;
  float *ldsD = (float *)(ldsX + nseg);         // -delta (dropout)

  const int tid = threadIdx.x;
  const int w = tid >> 6, l = tid & 63, kl = l & 31, h = l >> 5;

  int bh, pi, npass;
  bwd_item<CAUSAL, bwd_dkdv_pipe_occ<D, CAUSAL, DROP>() == 2, !CAUSAL>(a, bh, pi, npass);

  const T *Qb = (const T *)a.q + RW::head(a.mq, bh, a.sq);
  const T *dOb = (const T *)a.dout + RW::head(a.mdo, bh, a.sq);
  const T *Kb = (const T *)a.k + RW::head(a.mk, bh, a.sk);
  const T *Vb = (const T *)a.v + RW::head(a.mv, bh, a.sk);
  const float *lseb = a.lse + (size_t)bh * a.sq;
  const float *delb = a.delta + (size_t)bh * a.sq;
  const int skv = bwd_valid_keys(a, bh); // keys at or past it are invalid: their dK, dV rows are zero
  MaskTail<T, NT> tail;
  int live_keys = a.sk;
  if (MASK == kMaskPerKey) tail.issue(a, (const T *)a.mask + (size_t)(bh / a.mask_div) * a.mask_sb, tid);

  auto stage_rows = [&](int seg0) { // extra-step rows of queries seg0 .. seg0 + nseg - 1
    for (int base = 0; base < nseg; base += 4 * NT) {
      float lr[4], dr[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int q = seg0 + base + c * NT + tid, qc = q < a.sq ? q : a.sq - 1;
        lr[c] = lseb[qc];
        dr[c] = delb[qc];
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int i = base + c * NT + tid;
        const bool ok = seg0 + i < a.sq && lr[c] != NEG_INF; // rows past the end and fully masked rows: P = 0
        const float nl = ok ? -lr[c] * FMHA_LOG2E : BIGNEG, nd = ok ? -dr[c] : 0.f;
        v8 x;
        split_hi_lo<T>(nl, ((T *)&x)[0], ((T *)&x)[1]);
        x[2] = (T)1.f;
        x[3] = (T)1.f;
        split_hi_lo<T>(nd, ((T *)&x)[4], ((T *)&x)[5]);
        x[6] = (T)0.f;
        x[7] = (T)0.f;
        if (i < nseg) {
          ldsX[i] = as_u32x4(x);
          if (DROP == 1) ldsD[(seg0 + i) & (2 * C::QSEG - 1)] = nd; // (the previous segment's stay: its last tile is still to come)
        }
      }
    }
  };

  for (int pass = 0; pass < npass; ++pass) {
    // (where registers spilled set up for each pass, see dQ: backward, us, BH 600 S 380 D 64 packed with dropout 134.6 -> 131.8; BH 512 S 512
    // with dropout 146 -> 142, S 1024 bf16 405 -> 398; on whole rows without dropout, where nothing spills, 1 to 2 % behind)
    int tid = threadIdx.x;
    if (CAUSAL && (D > 64 || STRIDED || DROP == 1)) asm volatile("" : "+v"(tid));
    const int w = tid >> 6, l = tid & 63, kl = l & 31, h = l >> 5;
    const int ktile = pass == 0 ? pi : a.ntile - 1 - pi;
    const int k0w = ktile * KT + w * 32;
    const int key = k0w + kl;
    const int nqt = (a.sq + BT - 1) / BT;
    const int qt0 = CAUSAL ? ktile * KT / BT : 0; // first query tile that sees any of these keys

    // ---- the first three tiles on their way
    const uint32_t lds_base = lds_address(lds);
    PipeCopy<T, D, NT> qcopy, dcopy; // Q and dO rows need not be equally far apart
    qcopy.init(tid, RW::ss(a.mq), a.sq, RW::cols(a));
    dcopy.init(tid, RW::ss(a.mdo), a.sq, RW::cols(a));
    constexpr int VPT = 2 * PipeCopy<T, D, NT>::CPT;
    auto dma_one = [&](int qt, int i) {
      const uint32_t dst = lds_base + (uint32_t)(qt & (NST - 1)) * STAGEB;
      if (i < VPT / 2) qcopy.issue(Qb, qt, dst, i);
      else dcopy.issue(dOb, qt, dst + TILEB, i - VPT / 2);
    };
    auto dma_qdo = [&](int qt) {
#pragma unroll
      for (int i = 0; i < VPT; ++i) dma_one(qt, i);
    };
#pragma unroll
    for (int t = 0; t < NST - 1; ++t) dma_qdo(qt0 + t);

    PanelLane pl;
    pl.init(l);
    // ---- per-key operands
    v8 kreg[KS], vreg[KS], bxs, bxd;
    {
      const int kc = key < a.sk ? key : a.sk - 1;
      u32x4 tk[KS], tv[KS];
      const bool turned = C::TURNED && (CAUSAL || D != 64 || !STRIDED || RW::ss(a.mk) != (uint32_t)RW::cols(a)); // (see RowOperands)
      RowOperands<T, D> rk, rv;
      if (turned) {
        rk.load(Kb, RW::ss(a.mk), k0w, a.sk, RW::cols(a), l);
        rv.load(Vb, RW::ss(a.mv), k0w, a.sk, RW::cols(a), l);
      } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const size_t col = ks * 16 + h * 8 < RW::cols(a) ? ks * 16 + h * 8 : 0;
          tk[ks] = *(const u32x4 *)(Kb + (size_t)kc * RW::ss(a.mk) + col);
          tv[ks] = *(const u32x4 *)(Vb + (size_t)kc * RW::ss(a.mv) + col);
        }
      }
      T mraw = (T)0.f;
      if (MASK == kMaskPerKey) mraw = ((const T *)a.mask)[(size_t)(bh / a.mask_div) * a.mask_sb + kc];
      if (pass == 0 || a.sq > C::QSEG) stage_rows(qt0 * BT / C::QSEG * C::QSEG);
      if (turned) {
        char *panel = lds + C::OFF_T + w * C::TURNB; // (the first tiles go to the other stages: qt0 is a multiple of four)
        rk.turn(panel, pl, l, tk);
        rv.turn(panel, pl, l, tv);
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bool live = ks * 16 + h * 8 < RW::cols(a);
        const v8 kraw = as_v8<T>(chunk_or_zero(tk[ks], live));
        const v8 vraw = as_v8<T>(chunk_or_zero(tv[ks], live));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          kreg[ks][j] = (T)((float)kraw[j] * a.scale_l2);
          vreg[ks][j] = DROP == 1 ? (T)((float)vraw[j] * a.drop_scale) : vraw[j];
        }
      }
      float mk = 0.f;
      if (MASK == kMaskPerKey) mk = fmaf((float)mraw, a.mask_a, a.mask_b);
      if (key >= skv) mk = BIGNEG;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        bxs[j] = (T)0.f;
        bxd[j] = (T)0.f;
      }
      if (h == 0) {
        bxs[0] = (T)1.f;
        bxs[1] = (T)1.f;
        T hi, lo;
        split_hi_lo<T>(mk, hi, lo);
        bxs[2] = hi;
        bxs[3] = lo;
        bxd[4] = (T)1.f;
        bxd[5] = (T)1.f;
      }
    }
    if (MASK == kMaskPerKey && pass == 0) live_keys = tail.finish(a, ldsR, tid);
    const bool dead = ktile * KT >= (live_keys < skv ? live_keys : skv); // the whole key tile is invalid

    f32x16 dk[DB], dv[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        dk[db][r] = 0.f;
        dv[db][r] = 0.f;
      }

    f32x16 xA, gA, xB, gB;
    uint32_t rbA[4], rbB[4];
    PhiloxSlices ph;
    const uint32_t sel1 = (l & 1) ? 0x03070105u : 0x06020400u, sel2 = (l & 2) ? 0x03020706u : 0x05040100u; // see drop_bytes_k

    constexpr bool VFORM = D > 64;
    auto begin = [&](const v8 &p, const v8 &q, f32x16 &c) {
      if constexpr (VFORM) {
        MfmaV<T>::start(p, q, c);
      } else {
        f32x16 z;
#pragma unroll
        for (int r = 0; r < 16; ++r) z[r] = 0.f;
        c = E::mfma(p, q, z);
      }
    };
    auto add = [&](const v8 &p, const v8 &q, f32x16 &c) {
      if constexpr (VFORM) MfmaV<T>::add(p, q, c);
      else c = E::mfma(p, q, c);
    };
    auto xrow = [&](int qt) -> v8 { return as_v8<T>(ldsX[(qt * BT + kl) & (C::QSEG - 1)]); };
    auto step = [&](auto next_tag, auto guard_tag, int qt, const f32x16 &xc, const f32x16 &gc, const uint32_t (&rc)[4],
                    f32x16 &xn, f32x16 &gn, uint32_t (&rn)[4]) {
      constexpr bool NEXT = decltype(next_tag)::value, GUARD = decltype(guard_tag)::value;
      constexpr int NX = NEXT ? 2 : 0, NA = NEXT ? 2 * KS : 0, NC = 4 * DB, NO = NA + NC, NM = NX + NO;
      constexpr int AHEAD = D > 64 ? 4 : 3;
      constexpr bool SWAP = D > 64;
      constexpr int NS = 10;
      constexpr int NP = DROP == 1 && NEXT ? 15 : 0;
      constexpr int JS = NEXT ? NX + NA : 0;
      const char *ldsN = lds + ((qt + 1) & (NST - 1)) * STAGEB;
      const char *ldsC = lds + (qt & (NST - 1)) * STAGEB;
      const int q0 = qt * BT;
      auto fetch = [&](int j) -> v8 {
        if (j < NA) return panel_read_rows<T, BT>(ldsN + (j & 1) * TILEB, pl, 0, j >> 1);
        const int i = j - NA; // dO^T and Q^T alternate
        return panel_read_transposed<T, BT>(ldsC + ((i & 1) ^ 1) * TILEB, pl, 0, (i >> 1) % DB, (i >> 1) / DB);
      };
      float p[16], ds[16];
      bool keep[16];
      f32x4 Dl[4];
      v8 pf[2], df[2];
      auto softmax = [&](int s) {
        if (s < 8) {
          if (DROP == 1 && s % 2 == 0) Dl[s / 2] = *(const f32x4 *)(ldsD + ((q0 + 8 * (s / 2) + 4 * h) & (2 * C::QSEG - 1)));
#pragma unroll
          for (int e = 2 * s; e < 2 * s + 2; ++e) {
            float xv = xc[e];
            if (GUARD) xv = (key <= q0 + 8 * (e / 4) + 4 * h + e % 4) ? xv : BIGNEG;
            p[e] = fast_exp2(xv);
            asm volatile("" : "+v"(p[e])); // (stays in this slot)
            if (DROP == 1) keep[e] = drop_keep_byte(rc[e % 4], e / 4, a.drop.thr);
          }
        }
        if (s >= 1 && s < 9) {
#pragma unroll
          for (int e = 2 * (s - 1); e < 2 * s; ++e) {
            float gv = gc[e];
            if (DROP == 1) gv = keep[e] ? gv : Dl[e / 4][e % 4];
            ds[e] = p[e] * gv;
            if (DROP == 1) p[e] = keep[e] ? p[e] : 0.f; // (drop_scale multiplies dV once, on store)
            asm volatile("" : "+v"(ds[e]), "+v"(p[e]));
          }
        }
        if (s >= 2) {
#pragma unroll
          for (int e = 2 * (s - 2); e < 2 * (s - 1); ++e) {
            pf[e / 8][e % 8] = (T)p[e];
            df[e / 8][e % 8] = (T)ds[e];
          }
        }
      };
      auto philox = [&](int s) {
        if (s == 0) ph.start(a.drop, (uint32_t)bh, (uint32_t)((q0 + BT) >> 2) + (uint32_t)h + 2u * ((uint32_t)l & 3u), (uint32_t)key >> 2);
        else if (s <= 10) ph.round(a.drop, s - 1);
        else {
          const int t = s - 11;
          const uint32_t a1 = __builtin_amdgcn_perm(quad_perm<0xB1>(ph.c[t]), ph.c[t], sel1);
          rn[t] = __builtin_amdgcn_perm(quad_perm<0x4E>(a1), a1, sel2);
        }
      };
      v8 opnd[NO], xa;
      if (NEXT) xa = xrow(qt + 1);
#pragma unroll
      for (int j = 0; j < AHEAD && j < NO; ++j) opnd[j] = fetch(j);
      int done = 0;
      if (!NEXT) {
#pragma unroll
        for (; done < NS; ++done) softmax(done);
      }
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        if (m < NX) {
          if (m == 0) begin(xa, bxs, xn);
          else begin(xa, bxd, gn);
        } else {
          const int j = m - NX;
          if (j + AHEAD < NO) opnd[j + AHEAD] = fetch(j + AHEAD);
          const int u = SWAP ? j ^ 1 : j; // (the later one of a pair first: its wait covers the other)
          if (u < NA) {
            if ((u & 1) == 0) add(opnd[u], kreg[u >> 1], xn);
            else add(opnd[u], vreg[u >> 1], gn);
          } else {
            const int i = u - NA, db = (i >> 1) % DB, c = (i >> 1) / DB;
            f32x16 &acc = (i & 1) ? dk[db] : dv[db];
            const v8 fr = (i & 1) ? df[c] : pf[c];
            acc = E::mfma(opnd[u], fr, acc);
          }
        }
        if (m % (NM / VPT) == NM / VPT - 1 && m / (NM / VPT) < VPT) dma_one(qt + NST - 1, m / (NM / VPT));
        const int upto = m < JS ? (m + 1) * NS / (JS ? JS : 1) : NS + (m - JS + 1) * NP / (NM - JS);
#pragma unroll
        for (; done < upto; ++done) {
          if (done < NS) softmax(done);
          else philox(done - NS);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    using Yes = std::true_type;
    using No = std::false_type;
    using Guard = std::integral_constant<bool, CAUSAL>;

    // causal: query tiles ahead of the one that holds this wave's own diagonal see none of its keys
    const int t_own = CAUSAL ? (ktile * KT + __builtin_amdgcn_readfirstlane(w) * 32) / BT : qt0;
    uint32_t rb0[4];
    if (DROP == 1) drop_bytes_k(a.drop, (uint32_t)bh, (uint32_t)(t_own * BT), (uint32_t)key, h, l, rb0); // (while the tiles are on their way)
    auto first = [&](int qt, f32x16 &x, f32x16 &g, uint32_t (&rb)[4]) {
      const char *t = lds + (qt & (NST - 1)) * STAGEB;
#pragma unroll
      for (int i = 0; i < 4 && DROP == 1; ++i) rb[i] = rb0[i];
      const v8 xa = xrow(qt);
      constexpr int AHEAD = 2; // (operand pairs asked for ahead of their products)
      v8 ox[KS], og[KS];
      auto fetch = [&](int ks) {
        ox[ks] = panel_read_rows<T, BT>(t, pl, 0, ks);
        og[ks] = panel_read_rows<T, BT>(t + TILEB, pl, 0, ks);
      };
#pragma unroll
      for (int ks = 0; ks < AHEAD && ks < KS; ++ks) fetch(ks);
      if (VFORM) asm volatile("s_nop 4"); // (the operands may just have been written)
      begin(xa, bxs, x);
      begin(xa, bxd, g);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + AHEAD < KS) fetch(ks + AHEAD);
        add(ox[ks], kreg[ks], x);
        add(og[ks], vreg[ks], g);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (VFORM) settle(x, g);
    };
    // top of the iteration of tile qt: tile qt + 1 has landed, tile qt - 1 is no longer read
    auto turn = [&](int qt) {
      if (a.sq > C::QSEG && ((qt + 1) * BT & (C::QSEG - 1)) == 0 && qt + 1 < nqt) { // the next segment's extra-step rows
        bwd_lds_barrier();
        stage_rows((qt + 1) * BT);
      }
      bwd_vm_wait<(NST - 3) * VPT>();
      bwd_lds_barrier();
    };
    bwd_vm_wait<0>();
    bwd_lds_barrier();
    if (!dead && qt0 < nqt) {
      int t0 = qt0;
      if (CAUSAL) {
        const int stop = t_own < nqt ? t_own : nqt; // (no query at all may see them)
        for (; t0 < stop; ++t0) {
          turn(t0);
          dma_qdo(t0 + NST - 1);
        }
      }
      if (t0 < nqt) {
        const int nmid = nqt - 1 - t0;
        int qt = t0;
        if (nmid & 1) {
          first(qt, xB, gB, rbB);
          turn(qt);
          step(Yes{}, Guard{}, qt, xB, gB, rbB, xA, gA, rbA);
          ++qt;
        } else {
          first(qt, xA, gA, rbA);
          if (CAUSAL && nmid > 0) {
            turn(qt);
            step(Yes{}, Guard{}, qt, xA, gA, rbA, xB, gB, rbB);
            turn(qt + 1);
            step(Yes{}, No{}, qt + 1, xB, gB, rbB, xA, gA, rbA);
            qt += 2;
          }
        }
        for (; qt < nqt - 1; qt += 2) {
          turn(qt);
          step(Yes{}, No{}, qt, xA, gA, rbA, xB, gB, rbB);
          turn(qt + 1);
          step(Yes{}, No{}, qt + 1, xB, gB, rbB, xA, gA, rbA);
        }
        turn(qt);
        if (CAUSAL && nmid == 0) step(No{}, Guard{}, qt, xA, gA, rbA, xB, gB, rbB);
        else step(No{}, No{}, qt, xA, gA, rbA, xB, gB, rbB);
      }
    }
    bwd_vm_wait<0>(); // no copy may still be on its way into LDS when the wave ends, or the next pass starts

    bwd_lds_barrier(); // (every wave is done with the tiles: their LDS turns the output rows)
    {
      T *dKb = (T *)a.dk + RW::head(a.mdk, bh, a.sk) + (size_t)k0w * RW::ss(a.mdk);
      T *dVb = (T *)a.dv + RW::head(a.mdv, bh, a.sk) + (size_t)k0w * RW::ss(a.mdv);
      char *scratch = lds + w * RowStore<D>::BYTES;
      store_acc_rows<T, D>(scratch, dk, a.scale, dKb, RW::ss(a.mdk), a.sk - k0w, RW::cols(a), l);
      store_acc_rows<T, D>(scratch, dv, DROP == 1 ? a.drop_scale : 1.f, dVb, RW::ss(a.mdv), a.sk - k0w, RW::cols(a), l);
    }
    __syncthreads(); // the next pass refills the tiles
  }
}

} // namespace fmha
