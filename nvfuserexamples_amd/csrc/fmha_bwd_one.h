// One-pass backward for heads of up to 256 queries and keys (head dim 64; no mask, a per-key mask and / or the causal mask), where
// there are more heads than compute units.
//
// The kernel for short heads (fmha_bwd_short.h) forms the score and dP products, the exponentials and the dropout decisions
// twice, once with a lane per query (dQ) and once with a lane per key (dK, dV): 7 tile products instead of 5; and a compute
// unit holds one workgroup of it at 256 rows, so each head's copies wait for the last head's stores.  Here:
//
//   * A persistent workgroup of eight waves per compute unit walks a list of heads.  A wave owns 32 keys (K and V rows as
//     register operands, dK^T and dV^T accumulators resident) and walks the query tiles of 32 rows:
//       x = Q.K^T + (mask - LSE) / scale, g = dO.V^T - delta, P = exp2(scale x), dS = P o (kept ? g : -delta),
//       dV^T += dO^T.(P o Z), dK^T += Q^T.dS, formulas and dropout rule as in fmha_bwd_kernel.h.
//   * dQ needs dS with the keys as the contraction index, and the sum over all waves' keys.  Each wave writes its rounded 32 x 32
//     block of dS^T to LDS; behind the next barrier wave w forms ONE 16 x 16 block of dQ^T (16 queries, 16 columns) over all
//     256 keys, 8 v_mfma_f32_16x16x32: B = dS by the transpose read, A = K^T, loaded once per head into 32 registers.  So
//     every element of dQ is complete in one wave: no atomics, no partial sums, and one barrier per query tile, because the
//     blocks alternate between two buffers and dQ of tile t runs beside the exponentials of tile t + 1.
//   * Q, dO and O rows stream through LDS, five tiles (O: four) resident, asked for four tiles ahead and on into the next
//     head; delta of tile t + 1 is formed from the O and dO tiles while tile t is computed, and stays in LDS.  The next head's
//     K and V rows are copied meanwhile.
//   * The rank-one terms ride in one extra contraction step in bf16, three pieces to a value: exact to fp32, and with the
//     range that (mask - LSE) / scale of a fully masked row needs.  K and V stay as they are (scale and the dropout factor are
//     applied in fp32), so nothing is rounded that the kernel for short heads does not round.
//   * No register may spill: a reload waits for every copy in flight.  Lane addresses are set up anew for each head (Lane).
//
// LDS of dS: row = key, 64 bytes = 32 queries in pieces of 4; piece u of row k at position u ^ (bits 2, 3, 4 of k, reversed):
// conflict-free both for the rows' writes (8 bytes per lane, 32 rows) and for the transpose read (8 rows x 4 pieces per
// half wave, rows 4g..4g+3 and 16+4g..16+4g+3 for lane group g).
//
// Measured (us; kernel for short heads -> this): BH 768 S 197 bf16 63.2 -> 52.6, from packed rows 65.0 -> 56.2; BH 512 S 256
// fp16 53.4 -> 44.5, with dropout 64.1 -> 49.7, causal 46.8 -> 40.0, causal with dropout 53.8 -> 44.5; BH 1000 S 130 55.0 -> 49.1.
// A tile takes 1.7 us (about 3450 cycles: 1580 of the matrix pipe, 900 of the vector pipe, 1200 of LDS, which two waves
// per SIMD overlap only in part), the step between heads 2.5 us, a start 5 us.  Without its stores BH 1024 S 256 takes 69
// instead of 82 us, without operand reads 74, without dQ 72, without exponentials 79, without barriers 78, on zeros (power) 68:
// no one part bounds it.  Tried and level: four waves of 64 keys (66 us at BH 768 S 197), half of the waves a phase behind the
// others, wave priorities, operands two, three or four products ahead, dK and dV straight from the accumulator layout.
#pragma once
#include <utility>

#include "fmha_bwd_persist.h"

namespace fmha {

struct BwdOneCfg {
  static constexpr int D = 64, NW = 8, KEYS = NW * 32;
  static constexpr int KS = D / 16, DB = D / 32;
  static constexpr int TILEB = 32 * D * 2;                        // 32 rows
  static constexpr int NST = 5, NSO = 4;                          // tiles resident of Q and dO; of O and LSE
  static constexpr int OFF_O = NST * 2 * TILEB;                   // O tiles
  static constexpr int OFF_K = OFF_O + NSO * TILEB;               // K rows of a head, 32 per wave
  static constexpr int OFF_V = OFF_K + NW * TILEB;                // V rows; per wave, also the way out of its dK and dV rows
  static constexpr int VB = RowStore<D>::BYTES;
  static constexpr int OFF_S = OFF_V + NW * VB;                   // dS, two buffers of [256 keys][32 queries]
  static constexpr int SB = KEYS * 64;
  static constexpr int OFF_X = OFF_S + 2 * SB;                    // extra-step rows of a tile, two buffers
  static constexpr int OFF_L = OFF_X + 2 * 32 * 32;               // LSE of a tile
  static constexpr int OFF_D = OFF_L + NSO * 128;                 // -delta (dropout), two buffers
  static constexpr int OFF_M = OFF_D + 2 * 128;                   // mask values of a head's keys, a dword each
  static constexpr int LDS_BYTES = OFF_M + (KEYS + 32) * 4;
  static_assert(VB >= TILEB && LDS_BYTES <= 160 * 1024, "does not fit the LDS of a compute unit");
};

// f(0), f(1), ... f(N - 1) with the index as a constant
template <typename F, int... I> FMHA_DEV void unrolled(F &&f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }

template <typename T> struct Mfma16;
template <> struct Mfma16<_Float16> {
  static FMHA_DEV f32x4 k32(f16x8 a, f16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <> struct Mfma16<__bf16> {
  static FMHA_DEV f32x4 k32(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};

// One 16-bit value per lane, zero-extended: lane i's lands as a dword at LDS byte address lds_wave_base + 4*i.
FMHA_DEV void dma_global_to_lds_u16(const void *uniform_base, uint32_t lane_offset, uint32_t lds_wave_base) {
  lds_wave_base = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_wave_base);
  const uint64_t b = (uint64_t)uniform_base;
  const uint64_t ub = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32) |
                      (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, %2" ::"s"(lds_wave_base), "v"(lane_offset), "s"(ub) : "memory");
}

// v as the sum of three bf16 values (exact to fp32 but for subnormal remainders)
FMHA_DEV void split_bf16x3(float v, __bf16 &a, __bf16 &b, __bf16 &c) {
  a = (__bf16)v;
  v -= (float)a;
  b = (__bf16)v;
  c = (__bf16)(v - (float)b);
}

template <typename T, int DROP, bool CAUSAL, bool STRIDED>
__global__ __launch_bounds__(BwdOneCfg::NW * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void fmha_bwd_one_kernel(const BwdArgs a) {
  using C = BwdOneCfg;
  constexpr int D = C::D, NW = C::NW, KS = C::KS, DB = C::DB, TILEB = C::TILEB;
  using RW = Rows<STRIDED, D>;
  using E = Elem<T>;
  using v8 = typename E::v8;
  using v4 = typename E::v4;
  constexpr float NEG_INF = -__builtin_inff();
  constexpr float BIGNEG = -3.0e38f; // of an unscaled score: P = 0 at any scale (two of them add up to -inf, which does the same)

  extern __shared__ __attribute__((aligned(16))) char lds[];
  const uint32_t lds_base = lds_address(lds);
  const int l = threadIdx.x & 63, ws = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const float inv_scale = 1.f / a.scale_l2, l2_per_score = FMHA_LOG2E * inv_scale; // (of an LSE in the units of an unscaled score)
  const float inv_drop = DROP == 1 ? 1.f / a.drop_scale : 1.f;
  const int nqt = (a.sq + 31) / 32, ntl = nqt < 4 ? 4 : nqt; // query tiles, and turns a head takes (the stream looks one head ahead at most)
  const int G = gridDim.x;

  // What a lane addresses.  It is set up for each head from a lane index that the compiler cannot trace back to the last head's,
  // so that none of it is kept (or spilled) across the step between two heads, where the registers are full.
  const int qi = ws & 1, di = ws >> 1; // of dQ: this wave's 16 queries and 16 columns of a tile
  struct Lane {
    int l, kl, h, g16, i16, drow;
    uint32_t dofs, xofs, sofs0, sofs1, wpos;
    PanelLane pl;
    PipeCopy<T, D, 256> copy1, copyo;
    FMHA_DEV void init(int l0, int ws) {
      l = l0;
      asm volatile("" : "+v"(l));
      kl = l & 31, h = l >> 5, g16 = l >> 4, i16 = l & 15;
      pl.init(l);
      // delta and the extra-step row of the 32 queries of a tile: 16 lanes per row, 4 columns each
      drow = ws * 4 + g16;
      const int dcol = i16 * 4;
      dofs = (uint32_t)(drow * kPanelRowB + (((dcol >> 3) ^ ((drow >> 1) & 7)) << 4) + (dcol & 4) * 2);
      xofs = (uint32_t)(kl * 32 + h * 16);
      // dS operand of dQ; the position flip of rows 16 + 4 g16 .. +3 is one more than that of rows 4 g16 .. +3
      const uint32_t srev = (uint32_t)((g16 & 1) * 4 + (g16 >> 1) * 2), piece = (uint32_t)(4 * (ws & 1) + (i16 & 3));
      const uint32_t srow = (uint32_t)((4 * g16 + (i16 >> 2)) * 64);
      sofs0 = srow + ((piece ^ srev) << 3), sofs1 = srow + 16 * 64 + ((piece ^ (srev | 1u)) << 3);
      // dS block of this wave: lane = key, registers = queries 8g + 4h + t; of g = 0, the others flip bits 4 and 5
      const uint32_t wrev = (uint32_t)(((kl >> 2) & 1) * 4 + ((kl >> 3) & 1) * 2 + (kl >> 4));
      wpos = (uint32_t)(ws * 2048 + kl * 64) + (((uint32_t)h ^ wrev) << 3);
    }
  };
  auto copies_init = [&](Lane &n) {
    n.copy1.init((ws & 3) * 64 + n.l, (ws < 4) ? RW::ss(a.mq) : RW::ss(a.mdo), a.sq, D);
    n.copyo.init((ws & 3) * 64 + n.l, RW::ss(a.mo), a.sq, D);
  };

  // ---- copies.  Per tile: waves 0-3 a quarter of the Q and of the O tile each, waves 4-7 of the dO tile, and LSE.
  const bool qside = ws < 4;
  constexpr int VPT = 2;
  struct {
    const T *p1; // Q or dO
    const T *po; // O
    const float *pl;
    int tile, left;
  } cs = {nullptr, nullptr, nullptr, 0, 0};
  auto from_head = [&](int bh) {
    cs.p1 = qside ? (const T *)a.q + RW::head(a.mq, bh, a.sq) : (const T *)a.dout + RW::head(a.mdo, bh, a.sq);
    cs.po = (const T *)a.o + RW::head(a.mo, bh, a.sq);
    cs.pl = a.lse + (size_t)bh * a.sq;
  };
  auto copy_first = [&](const Lane &n, int s5) { n.copy1.issue(cs.p1, cs.tile, lds_base + (uint32_t)(s5 * 2 * TILEB + (qside ? 0 : TILEB)), 0); };
  auto copy_second = [&](const Lane &n, int s4) {
    if (qside) n.copyo.issue(cs.po, cs.tile, lds_base + (uint32_t)(C::OFF_O + s4 * TILEB), 0);
    else if (n.l < 32) {
      int q = cs.tile * 32 + n.l;
      q = q < a.sq ? q : a.sq - 1;
      dma_global_to_lds_b32(cs.pl, (uint32_t)q * 4u, lds_base + (uint32_t)(C::OFF_L + s4 * 128)); // (four waves the same values)
    }
    ++cs.tile;
  };
  auto own_lane = [&]() -> int { // (for what is needed once per head, as in Lane)
    int x = l;
    asm volatile("" : "+v"(x));
    return x;
  };
  auto copy_kv = [&](int bh) { // this wave's 32 rows (past the last key: that one again), and their mask values
    const int lx = own_lane();
    const T *Kb = (const T *)a.k + RW::head(a.mk, bh, a.sk), *Vb = (const T *)a.v + RW::head(a.mv, bh, a.sk);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int row, col;
      TileCopy<T, D, 32, 64>::slot(lx + i * 64, row, col);
      int key = ws * 32 + row;
      key = key < a.sk ? key : a.sk - 1;
      const uint32_t off = (uint32_t)key * (RW::ss(a.mk) * 2u) + (uint32_t)col * 16u;
      dma_global_to_lds_b128(Kb, off, lds_base + (uint32_t)(C::OFF_K + ws * TILEB + i * 1024));
      dma_global_to_lds_b128(Vb, off, lds_base + (uint32_t)(C::OFF_V + ws * C::VB + i * 1024));
    }
    if (a.mask) { // (lanes 32 .. 63: what the next wave writes there itself)
      int key = ws * 32 + lx;
      key = key < a.sk ? key : a.sk - 1;
      dma_global_to_lds_u16((const T *)a.mask + (size_t)(bh / a.mask_div) * a.mask_sb, (uint32_t)key * 2u, lds_base + (uint32_t)(C::OFF_M + ws * 128));
    }
  };
  constexpr int VKV = 8; // (there is one more with a mask)

  struct DeltaRows { // of one tile, in steps that can be spread over an instruction stream
    u32x2 o, d;
    float s, ls;
  };
  auto delta_step = [&](auto step, const Lane &n, DeltaRows &r, int q0, int s5, int s4, int buf) {
    constexpr int S = decltype(step)::value;
    auto plus = [&](uint32_t x) { r.s += __builtin_bit_cast(float, x); };
    if constexpr (S == 0) {
      r.o = *(const u32x2 *)(lds + C::OFF_O + s4 * TILEB + n.dofs);
      r.d = *(const u32x2 *)(lds + s5 * 2 * TILEB + TILEB + n.dofs);
      r.ls = *(const float *)(lds + C::OFF_L + s4 * 128 + n.drow * 4);
    } else if constexpr (S == 1) {
      const v4 ov = as_v4<T>(r.o), dv = as_v4<T>(r.d);
      r.s = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) r.s = fmaf((float)ov[j], (float)dv[j], r.s);
    } else if constexpr (S == 2) plus(quad_perm<0xB1>(__builtin_bit_cast(uint32_t, r.s)));  // lane ^ 1
    else if constexpr (S == 3) plus(quad_perm<0x4E>(__builtin_bit_cast(uint32_t, r.s)));    // lane ^ 2
    else if constexpr (S == 4) plus(quad_perm<0x141>(__builtin_bit_cast(uint32_t, r.s)));   // mirrored within 8 lanes
    else if constexpr (S == 5) plus(quad_perm<0x140>(__builtin_bit_cast(uint32_t, r.s)));   // mirrored within 16 lanes
    else {
      const bool ok = q0 + n.drow < a.sq && r.ls != NEG_INF; // rows past the end and fully masked rows: P = 0
      const float nl = ok ? -r.ls * l2_per_score : BIGNEG;
      const float nd = ok ? -r.s * inv_drop : 0.f;
      bf16x8 x, d;
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = d[j] = (__bf16)0.f;
      split_bf16x3(nl, ((__bf16 *)&x)[0], ((__bf16 *)&x)[1], ((__bf16 *)&x)[2]);
      x[3] = x[4] = x[5] = (__bf16)1.f;
      split_bf16x3(nd, ((__bf16 *)&d)[0], ((__bf16 *)&d)[1], ((__bf16 *)&d)[2]);
      char *dst = lds + C::OFF_X + buf * 1024 + n.drow * 32;
      if (n.i16 == 0) {
        *(u32x4 *)dst = as_u32x4(x);
        *(u32x4 *)(dst + 16) = as_u32x4(d);
        if (DROP == 1) *(float *)(lds + C::OFF_D + buf * 128 + n.drow * 4) = nd;
      }
    }
  };
  constexpr int DELTA_STEPS = 7;

  auto ds_operand = [&](const Lane &n, const char *buf, int kb) -> v8 {
    const u32x2 lo = lds_read_tr16(buf + kb * 2048 + n.sofs0), hi = lds_read_tr16(buf + kb * 2048 + n.sofs1);
    return as_v8<T>(u32x4{lo.x, lo.y, hi.x, hi.y});
  };
  auto store_dq = [&](const Lane &n, int bh, int tile, const f32x4 &acc) {
    const int q = tile * 32 + 16 * qi + n.i16, col = 16 * di + 4 * n.g16;
    const float sc = DROP == 1 ? a.scale * a.drop_scale : a.scale;
    typename E::v4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = (T)(acc[r] * sc);
    Pack8 p;
    if constexpr (std::is_same<T, _Float16>::value) p.h = o;
    else p.b = o;
    if (q < a.sq) *(u32x2 *)((T *)a.dq + RW::head(a.mdq, bh, a.sq) + (size_t)q * RW::ss(a.mdq) + col) = p.u;
  };
  auto put_ds = [&](const Lane &n, int buf, int g, u32x2 v) { *(u32x2 *)(lds + C::OFF_S + ((n.wpos + (uint32_t)(buf * C::SB)) ^ (uint32_t)(g << 4))) = v; };

  v8 kt[NW]; // K^T: 16 columns of 32 keys each
  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      dk[db][r] = 0.f;
      dv[db][r] = 0.f;
    }
  auto dq_alone = [&](int bh, int tile, int sb) { // (the head's last tile: behind its barrier)
    const char *buf = lds + C::OFF_S + sb * C::SB;
    Lane n;
    n.init(l, ws);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < NW; ++kb) acc = Mfma16<T>::k32(kt[kb], ds_operand(n, buf, kb), acc);
    store_dq(n, bh, tile, acc);
  };
  auto store_head = [&](int bh) {
    asm volatile("" ::: "memory"); // (the rows go where the V rows have been read: no access may move past the other kind)
    const int k0w = ws * 32, lx = own_lane();
    if (k0w < a.sk) {
      T *dKb = (T *)a.dk + RW::head(a.mdk, bh, a.sk) + (size_t)k0w * RW::ss(a.mdk);
      T *dVb = (T *)a.dv + RW::head(a.mdv, bh, a.sk) + (size_t)k0w * RW::ss(a.mdv);
      char *scratch = lds + C::OFF_V + ws * C::VB;
      store_acc_rows<T, D>(scratch, dk, DROP == 1 ? a.scale * a.drop_scale : a.scale, dKb, RW::ss(a.mdk), a.sk - k0w, D, lx);
      store_acc_rows<T, D>(scratch, dv, DROP == 1 ? a.drop_scale : 1.f, dVb, RW::ss(a.mdv), a.sk - k0w, D, lx);
    }
  };

  // ---- start: the first head's rows, and delta of its first tile
  int bh = blockIdx.x, pbh = -1;
  int s5 = 0, s4 = 0; // stages of the current tile
  from_head(bh);
  {
    Lane n;
    n.init(l, ws);
    copies_init(n);
    copy_kv(bh);
    for (int t = 0; t < 4; ++t) {
      copy_first(n, t);
      copy_second(n, t);
    }
    bwd_vm_wait<3 * VPT>(); // (tiles 1 to 3 may still be on their way)
    bwd_lds_barrier();
    DeltaRows r;
    unrolled([&](auto i) { delta_step(i, n, r, 0, 0, 0, 0); }, std::make_integer_sequence<int, DELTA_STEPS>{});
  }
  int xb = 0, sb = 0; // buffers of the current tile's extra-step rows and dS

  for (; bh < a.bh; bh += G) {
    const bool more = bh + G < a.bh;
    const int kend = bwd_valid_keys(a, bh);
    from_head(bh);
    cs.tile = 4;
    cs.left = ntl - 4;
    auto turn = [&](int j) { // top of turn j: tile j + 1 has landed, tile j - 1 is no longer read; tile j + 4 goes on its way
      if ((j == 2 || j == 3) && more) bwd_vm_wait<2 * VPT + VKV>(); // (the next head's K and V rows are younger)
      else bwd_vm_wait<2 * VPT>();
      bwd_lds_barrier();
      if (j == 1 && more) copy_kv(bh + G); // (every wave has this head's operands)
    };
    // the copies of a turn, in two parts that the stream puts apart (all waves' at once, behind the barrier, they stall)
    auto ahead_first = [&]() {
      if (cs.left == 0) {
        if (more) {
          from_head(bh + G);
          cs.tile = 0;
        }
        cs.left = 0x7fffffff;
      }
      --cs.left;
    };
    auto advance = [&]() {
      s5 = s5 == C::NST - 1 ? 0 : s5 + 1;
      s4 = (s4 + 1) & 3;
      xb ^= 1;
    };
    // ---- between two heads: the last one's dQ of its last tile, then this one's operands
    turn(0);
    if (pbh >= 0) dq_alone(pbh, nqt - 1, sb ^ 1);
    const int lx = own_lane();
    PanelLane plx;
    plx.init(lx);
    const int hx = lx >> 5, keyx = ws * 32 + (lx & 31);
    v8 kreg[KS], vreg[KS];
    bf16x8 bxs, bxd;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      kreg[ks] = panel_read_rows<T, 32>(lds + C::OFF_K + ws * TILEB, plx, 0, ks);
      vreg[ks] = panel_read_rows<T, 32>(lds + C::OFF_V + ws * C::VB, plx, 0, ks);
    }
    {
      const int r0 = 4 * (lx >> 4) + ((lx & 15) >> 2), chunk = 2 * di + ((lx & 3) >> 1);
      const char *p0 = lds + C::OFF_K + r0 * kPanelRowB + ((chunk ^ ((r0 >> 1) & 7)) << 4) + 8 * (lx & 1);
#pragma unroll
      for (int kb = 0; kb < NW; ++kb) { // (rows 16 on: the same position, (row >> 1) & 7 repeats)
        const u32x2 lo = lds_read_tr16(p0 + kb * TILEB), hi = lds_read_tr16(p0 + kb * TILEB + 16 * kPanelRowB);
        kt[kb] = as_v8<T>(u32x4{lo.x, lo.y, hi.x, hi.y});
      }
      float mk = 0.f;
      if (a.mask) {
        const uint32_t raw = *(const uint32_t *)(lds + C::OFF_M + keyx * 4);
        mk = fmaf((float)__builtin_bit_cast(T, (unsigned short)raw), a.mask_a, a.mask_b) * inv_scale;
        mk = mk > BIGNEG ? mk : BIGNEG;
      }
      if (keyx >= kend) mk = BIGNEG;
#pragma unroll
      for (int j = 0; j < 8; ++j) bxs[j] = bxd[j] = (__bf16)0.f;
      if (hx == 0) {
        bxs[0] = bxs[1] = bxs[2] = (__bf16)1.f;
        split_bf16x3(mk, ((__bf16 *)&bxs)[3], ((__bf16 *)&bxs)[4], ((__bf16 *)&bxs)[5]);
      } else {
        bxd[0] = bxd[1] = bxd[2] = (__bf16)1.f;
      }
    }
    if (pbh >= 0) store_head(pbh);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        dk[db][r] = 0.f;
        dv[db][r] = 0.f;
      }
    pbh = bh;

    Lane n;
    n.init(l, ws);
    copies_init(n);
    const int key = ws * 32 + n.kl;
    const uint32_t sel1 = (n.l & 1) ? 0x03070105u : 0x06020400u, sel2 = (n.l & 2) ? 0x03020706u : 0x05040100u; // see drop_bytes_k
    auto ahead_copy = [&]() { copy_first(n, s5 == 0 ? C::NST - 1 : s5 - 1); };
    auto ahead_second = [&]() { copy_second(n, s4); };
    // delta of the stream's next tile: this head's, or the first of the next one (where there is neither nobody reads it)
    auto next_delta = [&](auto step, DeltaRows &r, int j) {
      delta_step(step, n, r, j + 1 < nqt ? (j + 1) * 32 : 0, s5 == C::NST - 1 ? 0 : s5 + 1, (s4 + 1) & 3, xb ^ 1);
    };
    auto whole_delta = [&](int j) {
      DeltaRows r;
      unrolled([&](auto i) { next_delta(i, r, j); }, std::make_integer_sequence<int, DELTA_STEPS>{});
    };
    constexpr int NA = 2 * KS, NB = NW, NC = 4 * DB, NS = 10;
    constexpr int NPRE = 2;
    v8 next[NPRE]; // the next phase's first operands
    // A phase is `count` products.  Their operands are asked for K products ahead, the first ones by the phase before.
    auto phase = [&](auto count, auto ahead, auto &&fetch, auto &&fetch_next, auto &&product) {
      constexpr int N = decltype(count)::value, K = decltype(ahead)::value;
      v8 op[N + NPRE];
#pragma unroll
      for (int i = 0; i < NPRE; ++i) op[i] = next[i];
      unrolled([&](auto mt) {
        constexpr int m = decltype(mt)::value, from = m == 0 ? NPRE : K + m > N + NPRE ? N + NPRE : K + m, to = K + m + 1 > N + NPRE ? N + NPRE : K + m + 1;
        unrolled([&](auto it) {
          constexpr int i = from + decltype(it)::value;
          op[i] = i < N ? fetch(i) : fetch_next(i - N);
        }, std::make_integer_sequence<int, (to > from ? to - from : 0)>{});
        product(mt, op[m]);
        __builtin_amdgcn_sched_barrier(0);
      }, std::make_integer_sequence<int, N>{});
#pragma unroll
      for (int i = 0; i < NPRE; ++i) next[i] = op[N + i];
    };
    auto tile_at = [&](int s) -> const char * { return lds + s * 2 * TILEB; };
    auto operand_a = [&](const char *t, int m) -> v8 { return panel_read_rows<T, 32>(t + (m & 1) * TILEB, n.pl, 0, m >> 1); };
    auto operand_c = [&](const char *t, int i) -> v8 { // dO^T and Q^T alternate
      return panel_read_transposed<T, 32>(t + ((i & 1) ^ 1) * TILEB, n.pl, 0, (i >> 1) % DB, (i >> 1) / DB);
    };
    v8 pf[2], df[2]; // P o Z and dS of a tile
    // x, g, P, dS of a tile, with dQ of the tile before it beside the exponentials (of tile 0: of whatever is in that buffer, and
    // nothing is stored)
    auto scores = [&](int j) -> f32x4 {
      const char *tq = tile_at(s5), *pbuf = lds + C::OFF_S + (sb ^ 1) * C::SB;
      const float *fD = (const float *)(lds + C::OFF_D + xb * 128);
      const int q0 = j * 32;
      f32x16 x, g;
      f32x4 dq = {0.f, 0.f, 0.f, 0.f};
      float p[16], ds[16];
      bool keep[16];
      f32x4 Dl[4];
      uint32_t rb[4];
      PhiloxSlices ph;
      auto philox = [&](int s) {
        if (s == 0) ph.start(a.drop, (uint32_t)bh, (uint32_t)(q0 >> 2) + (uint32_t)n.h + 2u * ((uint32_t)n.l & 3u), (uint32_t)key >> 2);
        else if (s <= 10) ph.round(a.drop, s - 1);
        else if (s < 15) {
          const int t = s - 11;
          const uint32_t a1 = __builtin_amdgcn_perm(quad_perm<0xB1>(ph.c[t]), ph.c[t], sel1);
          rb[t] = __builtin_amdgcn_perm(quad_perm<0x4E>(a1), a1, sel2);
        }
      };
      auto softmax = [&](int s) {
        if (s < 8) {
          if (DROP == 1 && s % 2 == 0) Dl[s / 2] = *(const f32x4 *)(fD + 8 * (s / 2) + 4 * n.h);
#pragma unroll
          for (int e = 2 * s; e < 2 * s + 2; ++e) {
            p[e] = fast_exp2(x[e] * a.scale_l2);
            asm volatile("" : "+v"(p[e])); // (stays in this slot)
            if (DROP == 1) keep[e] = drop_keep_byte(rb[e % 4], e / 4, a.drop.thr);
          }
        }
        if (s >= 1 && s < 9) {
#pragma unroll
          for (int e = 2 * (s - 1); e < 2 * s; ++e) {
            float gv = g[e];
            if (DROP == 1) gv = keep[e] ? gv : Dl[e / 4][e % 4];
            ds[e] = p[e] * gv;
            if (DROP == 1) p[e] = keep[e] ? p[e] : 0.f;
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
      const bf16x8 xa = as_v8<__bf16>(*(const u32x4 *)(lds + C::OFF_X + xb * 1024 + n.xofs));
#pragma unroll
      for (int r = 0; r < 16; ++r) x[r] = g[r] = 0.f;
      phase(std::integral_constant<int, NA>{}, std::integral_constant<int, 4>{}, [&](int m) { return operand_a(tq, m); }, [&](int m) { return ds_operand(n, pbuf, m); },
            [&](auto mt, const v8 &op) {
              constexpr int m = decltype(mt)::value;
              if constexpr (m == 4) { // (by now the row has come)
                x = Elem<__bf16>::mfma(xa, bxs, x);
                g = Elem<__bf16>::mfma(xa, bxd, g);
              }
              if constexpr ((m & 1) == 0) x = E::mfma(op, kreg[m >> 1], x);
              else g = E::mfma(op, vreg[m >> 1], g);
              if (DROP == 1) {
                philox(2 * m);
                if (2 * m + 1 < 15) philox(2 * m + 1);
              }
              if constexpr (m == 5) ahead_copy();
            });
      if (CAUSAL) { // (in every tile: a branch here would split the stream)
        const int rel = key - q0 - 4 * n.h;
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = rel <= 8 * (r / 4) + r % 4 ? x[r] : BIGNEG;
      }
      softmax(0); // (alone: the last products are still on their way)
      phase(std::integral_constant<int, NB>{}, std::integral_constant<int, 2>{}, [&](int m) { return ds_operand(n, pbuf, m); }, [&](int m) { return operand_c(tq, m); },
            [&](auto mt, const v8 &op) {
              constexpr int m = decltype(mt)::value;
              dq = Mfma16<T>::k32(kt[m], op, dq);
              asm volatile("" : "+v"(dq)); // (stays in this slot)
              softmax(m + 1);
            });
      static_assert(NS == NB + 2, "");
      softmax(NS - 1);
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const u32x4 u = as_u32x4(df[gq >> 1]);
        put_ds(n, sb, gq, (gq & 1) ? u32x2{u.z, u.w} : u32x2{u.x, u.y});
      }
      return dq;
    };
    // dV and dK, beside delta of the next tile
    auto gradients = [&](int j) {
      const char *tq = tile_at(s5), *tnext = tile_at(s5 == C::NST - 1 ? 0 : s5 + 1);
      DeltaRows dr;
      phase(std::integral_constant<int, NC>{}, std::integral_constant<int, 4>{}, [&](int m) { return operand_c(tq, m); }, [&](int m) { return operand_a(tnext, m); },
            [&](auto it, const v8 &op) {
              constexpr int i = decltype(it)::value, db = (i >> 1) % DB, c = (i >> 1) / DB;
              f32x16 &acc = (i & 1) ? dk[db] : dv[db];
              acc = E::mfma(op, (i & 1) ? df[c] : pf[c], acc);
              constexpr int at[DELTA_STEPS] = {0, 3, 4, 4, 5, 5, 6}; // (the rows take a while to come)
              unrolled([&](auto st) {
                if constexpr (at[decltype(st)::value] == i) next_delta(st, dr, j);
              }, std::make_integer_sequence<int, DELTA_STEPS>{});
            });
    };
    // a tile none of this wave's keys takes part in
    auto idle_tile = [&](int j) {
      ahead_first();
      ahead_copy();
      if (j > 0) dq_alone(bh, j - 1, sb ^ 1);
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) put_ds(n, sb, gq, u32x2{0, 0});
      whole_delta(j);
      ahead_second();
    };
    const int busy_from = ws * 32 >= kend ? nqt : CAUSAL ? ws : 0; // (the first query tile that sees one of them)
    int j = 0;
    for (; j < nqt && j < busy_from; ++j) {
      if (j > 0) turn(j);
      idle_tile(j);
      advance();
      sb ^= 1;
    }
#pragma unroll
    for (int i = 0; i < NPRE; ++i) next[i] = operand_a(tile_at(s5), i);
    for (; j < nqt; ++j) {
      if (j > 0) turn(j);
      ahead_first();
      const f32x4 dq = scores(j);
      gradients(j);
      if (j > 0) store_dq(n, bh, j - 1, dq);
      ahead_second();
      advance();
      sb ^= 1;
    }
    for (int j = nqt; j < ntl; ++j) { // (heads of fewer than four query tiles)
      turn(j);
      ahead_first();
      ahead_copy();
      whole_delta(j);
      ahead_second();
      advance();
    }
  }
  bwd_vm_wait<0>(); // no copy may still be on its way into LDS when the wave ends
  bwd_lds_barrier();
  dq_alone(pbh, nqt - 1, sb ^ 1);
  store_head(pbh);
}

} // namespace fmha
