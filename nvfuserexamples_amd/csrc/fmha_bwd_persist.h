// Persistent dK / dV kernel for head dim 128 without mask and key counts (with either: fmha_bwd_pipe.h and fmha_bwd_kernel.h).
// Mathematics, register layouts and the hand-ordered stream of an iteration are those of fmha_bwd_dkdv_pipe_kernel
// (fmha_bwd_pipe.h).  At head dim 128 a wave's accumulators and operands take both halves of the register file, so there is one
// wave per SIMD and one workgroup per compute unit: nothing ran while a workgroup fetched its K and V rows and first tiles, nor
// while its gradients left, and as all compute units run in step the memory idled in between (9.8 of the 51 us that a
// workgroup's two tiles took at BH 512 S 1024 causal).  Here a workgroup stays and walks a list of items (a head's 128 keys):
//
//   * The stream of query tiles runs on into the next item; its K and V rows and its rows (LSE, delta) are copied into LDS of
//     their own while this item is computed.  Between two items a wave turns what has landed into registers and hands the last
//     item's gradients, whole rows through its own part of that LDS, to stores that nobody waits for before two tiles later.
//   * The list is dealt in advance and evens out causal tiles.  A mask's hidden tiles it cannot know: with masks it measured 2 to
//     6 % behind the plain kernels, whose workgroups come and go as there is work.
//   * At head dim 64 there are two workgroups per compute unit, and one's start and stores run under the other's products
//     already; the same kernel there measured level (BH 512 S 512) to 8 % behind (causal), so it is built for 128 only.
//
// Kernel times on one card, us, plain pipelined kernel (without causal mask and dropout: phase by phase) -> this one: BH 512
// S 1024 causal bf16 415 -> 369, BH 300 S 400 causal 91 -> 62, BH 64 S 1500 causal 110 -> 91, BH 256 S 1024 341 -> 291, BH 32
// S 4096 507 -> 466, causal 265 -> 253.  What bounds it now: at long sequences the board's power (BH 32 S 4096 causal on
// zeros 231); at short ones the turn from item to item, about 5 us of which 2 are the gradients' way through LDS and 1.5 the
// issue of the next item's copies behind their stores.  (Spread over the first turns those copies cost more than they hid:
// 291 -> 303 us at BH 256 S 1024.)
#pragma once
#include "fmha_bwd_pipe.h"

namespace fmha {

template <int D> struct BwdPersistCfg {
  static constexpr int NW = 4;
  static constexpr int BT = 32, NST = 4; // rows per tile, tiles resident per operand
  static constexpr int KS = D / 16, DB = D / 32;
  static constexpr int TILEB = BT * tile_cols(D) * 2, STAGEB = 2 * TILEB;
  static constexpr int QSEG = 1024;                 // queries whose extra-step rows are staged at once
  // tiles, then the K and V rows of the next item (a wave's 32 of each), then the extra-step rows, the raw (LSE, delta) of the
  // segment that comes next, and -delta (dropout; with more than one segment of two, see stage_rows)
  static constexpr int OFF_KV = NST * STAGEB, OFF_Q = OFF_KV + NW * 2 * TILEB;
  static constexpr int MAX_LDS = OFF_Q + 32 * QSEG;
  static int lds_bytes(int drop, int sq) { return OFF_Q + (sq <= QSEG ? (24 + (drop ? 4 : 0)) * ((sq + 63) / 64 * 64) : (24 + (drop ? 8 : 0)) * QSEG); }
};

// One dword per lane: lane i's lands at LDS byte address lds_wave_base + 4*i.
FMHA_DEV void dma_global_to_lds_b32(const void *uniform_base, uint32_t lane_offset, uint32_t lds_wave_base) {
  lds_wave_base = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_wave_base);
  const uint64_t b = (uint64_t)uniform_base;
  const uint64_t ub = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32) |
                      (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds_wave_base), "v"(lane_offset), "s"(ub) : "memory");
}

template <typename T, int D, int NW, bool CAUSAL, int DROP, bool STRIDED>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(1, 1))) void fmha_bwd_dkdv_persist_kernel(const BwdArgs a) {
  using RW = Rows<STRIDED, D>;
  using E = Elem<T>;
  using M = MfmaV<T>;
  using v8 = typename E::v8;
  using C = BwdPersistCfg<D>;
  constexpr int BT = C::BT, NST = C::NST, KS = C::KS, DB = C::DB, TILEB = C::TILEB, STAGEB = C::STAGEB;
  constexpr int NT = NW * 64, KT = NW * 32;
  constexpr float NEG_INF = -__builtin_inff();
  constexpr float BIGNEG = -60000.f;
  static_assert(NW == C::NW && RowStore<D>::BYTES <= 2 * TILEB, "a wave's K and V rows share their LDS with its output rows");
  static_assert(KT / BT == 4 && NST == 4, "the counts of copies in flight below");

  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int nseg = a.sq <= C::QSEG ? (a.sq + 63) / 64 * 64 : C::QSEG;
  u32x4 *ldsX = (u32x4 *)(lds + C::OFF_Q); // per query of the segment: (-L_hi, -L_lo, 1, 1, -delta_hi, -delta_lo, 0, 0)
  float *ldsRaw = (float *)(ldsX + nseg);  // LSE, then delta of the segment that comes next
  float *ldsD = ldsRaw + 2 * nseg;         // -delta (dropout)

  const int tid = threadIdx.x;
  const int w = tid >> 6, l = tid & 63, kl = l & 31, h = l >> 5;
  const int ws = __builtin_amdgcn_readfirstlane(w);
  char *ldsKV = lds + C::OFF_KV + ws * 2 * TILEB; // this wave's own part

  // ---- schedule: in round r this workgroup takes unit r * G + lb, a key tile or a causal pair of them.  Workgroups of one XCD
  // (every eighth one) work on neighbouring units, so a head's Q and dO rows are read through one L2.
  const int G = gridDim.x;
  const bool paired = CAUSAL && a.pair == kTilesPaired, by_length = CAUSAL && !paired;
  int lb = blockIdx.x;
  if (!by_length && (G & 7) == 0) lb = (lb & 7) * (G >> 3) + (lb >> 3);
  const int npair = paired ? (a.ntile + 1) / 2 : a.ntile;
  const int nunit = a.bh * npair;
  const int nqt = (a.sq + BT - 1) / BT;
  int base = 0, pass = 0; // of the item that is looked at next: its round's first unit, and which tile of a pair
  // Causal without pairs (few heads): the longest tiles of all heads come first, and the order of the workgroups turns from
  // round to round, so that who had a long one gets a short one next.  (With a multiple of eight heads the tiles of one stay
  // on its XCD.)
  auto unit_of = [&]() -> int { return base + (by_length && (base / G & 1) ? G - 1 - lb : lb); };
  auto locate = [&](int &bh, int &kt) {
    const int unit = unit_of(), n = by_length ? a.bh : npair, hi = unit / n, lo = unit - hi * n;
    bh = by_length ? lo : hi;
    kt = by_length ? hi : lo;
    if (paired && pass) kt = a.ntile - 1 - kt;
  };

  int nbh = 0, nkt = 0;                // the next item
  bool more = false;
  // -> (nbh, nkt, more).  Causal key tiles behind every query get their zeros on the way.
  auto seek = [&]() {
    more = false;
    for (; base < nunit;) {
      if (unit_of() >= nunit) { // (the last round need not be full)
        base += G;
        continue;
      }
      locate(nbh, nkt);
      if (paired && pass == 0 && a.ntile - 1 - nkt != nkt) pass = 1;
      else {
        pass = 0;
        base += G;
      }
      if (!CAUSAL || nkt * KT < nqt * BT) {
        more = true;
        return;
      }
      T *dKb = (T *)a.dk + RW::head(a.mdk, nbh, a.sk), *dVb = (T *)a.dv + RW::head(a.mdv, nbh, a.sk);
      for (int c = tid; c < KT * D / 8; c += NT) {
        const int key = nkt * KT + c / (D / 8), col = c % (D / 8) * 8;
        if (key < a.sk && col < RW::cols(a)) {
          *(u32x4 *)(dKb + (uint32_t)key * RW::ss(a.mdk) + col) = u32x4{0u, 0u, 0u, 0u};
          *(u32x4 *)(dVb + (uint32_t)key * RW::ss(a.mdv) + col) = u32x4{0u, 0u, 0u, 0u};
        }
      }
    }
  };

  // ---- copies
  const uint32_t lds_base = lds_address(lds);
  PipeCopy<T, D, NT> qcopy, dcopy; // Q and dO rows need not be equally far apart
  qcopy.init(tid, RW::ss(a.mq), a.sq, RW::cols(a));
  dcopy.init(tid, RW::ss(a.mdo), a.sq, RW::cols(a));
  constexpr int VPT = 2 * PipeCopy<T, D, NT>::CPT; // copies per tile pair and wave
  constexpr int VKV = 2 * (32 * tile_cols(D) / 8 / 64);       // copies of a wave's K and V rows
  // the stream of tiles: the one that is copied next; behind an item's last turn come the next item's first tiles
  struct {
    const T *q, *d;
    int tile, left; // ... and how many more of this item
  } cs = {nullptr, nullptr, 0, 0};
  auto copy_one = [&](uint32_t dst, int i) {
    if (i < VPT / 2) qcopy.issue(cs.q, cs.tile, dst, i);
    else dcopy.issue(cs.d, cs.tile, dst + TILEB, i - VPT / 2);
  };
  auto from_item = [&](int bh, int tile) {
    cs.q = (const T *)a.q + RW::head(a.mq, bh, a.sq);
    cs.d = (const T *)a.dout + RW::head(a.mdo, bh, a.sq);
    cs.tile = tile;
  };
  auto copy_kv = [&](int bh, int kt) { // this wave's rows (past the last key: that one again)
    const T *Kb = (const T *)a.k + RW::head(a.mk, bh, a.sk), *Vb = (const T *)a.v + RW::head(a.mv, bh, a.sk);
    const uint32_t dst = lds_base + C::OFF_KV + (uint32_t)ws * 2 * TILEB;
#pragma unroll
    for (int i = 0; i < VKV / 2; ++i) {
      int row, col;
      TileCopy<T, D, 32, 64>::slot(l + i * 64, row, col);
      int key = kt * KT + ws * 32 + row;
      key = key < a.sk ? key : a.sk - 1;
      const uint32_t cb = col * 8 < RW::cols(a) ? (uint32_t)col * 16u : 0u;
      dma_global_to_lds_b128(Kb, (uint32_t)key * (RW::ss(a.mk) * 2u) + cb, dst + (uint32_t)i * 1024u);
      dma_global_to_lds_b128(Vb, (uint32_t)key * (RW::ss(a.mv) * 2u) + cb, dst + TILEB + (uint32_t)i * 1024u);
    }
  };
  auto copy_raw = [&](int bh, int seg0) { // LSE and delta of queries seg0 .. seg0 + nseg - 1 (past the last one: that one again)
    const uint32_t dst = lds_base + C::OFF_Q + (uint32_t)nseg * 16u;
    for (int i = ws * 64; i < nseg; i += NT) {
      int q = seg0 + i + l;
      q = q < a.sq ? q : a.sq - 1;
      dma_global_to_lds_b32(a.lse + (size_t)bh * a.sq, (uint32_t)q * 4u, dst + (uint32_t)i * 4u);
      dma_global_to_lds_b32(a.delta + (size_t)bh * a.sq, (uint32_t)q * 4u, dst + (uint32_t)(nseg + i) * 4u);
    }
  };
  auto stage_rows = [&](int seg0) { // raw rows -> extra-step rows
    for (int i0 = tid; i0 < nseg; i0 += 4 * NT) { // (four rows at a time: their reads share one trip)
      float lr[4], dr[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int i = i0 + c * NT < nseg ? i0 + c * NT : i0;
        lr[c] = ldsRaw[i];
        dr[c] = ldsRaw[nseg + i];
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int i = i0 + c * NT;
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
  auto first_tile = [&](int kt) { return CAUSAL ? kt * KT / BT : 0; }; // the first query tile that sees any key of tile kt
  auto first_seg = [&](int kt) { return first_tile(kt) * BT / C::QSEG * C::QSEG; };
  auto start_item = [&](int bh, int kt) { // everything it begins with
    from_item(bh, first_tile(kt));
    for (int j = 0; j < NST - 1; ++j, ++cs.tile) {
#pragma unroll
      for (int i = 0; i < VPT; ++i) copy_one(lds_base + (uint32_t)j * STAGEB, i);
    }
    copy_kv(bh, kt);
    copy_raw(bh, first_seg(kt));
  };

  seek();
  if (!more) return;
  start_item(nbh, nkt);

  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      dk[db][r] = 0.f;
      dv[db][r] = 0.f;
    }
  int pbh = -1, pkt = 0; // the item whose gradients are still in the accumulators
  auto store_item = [&]() {
    asm volatile("" ::: "memory"); // (the rows go where the K and V rows have been read: no access may move past the other kind)
    const int k0w = pkt * KT + ws * 32;
    T *dKb = (T *)a.dk + RW::head(a.mdk, pbh, a.sk) + (size_t)k0w * RW::ss(a.mdk);
    T *dVb = (T *)a.dv + RW::head(a.mdv, pbh, a.sk) + (size_t)k0w * RW::ss(a.mdv);
    store_acc_rows<T, D>(ldsKV, dk, a.scale, dKb, RW::ss(a.mdk), a.sk - k0w, RW::cols(a), l);
    store_acc_rows<T, D>(ldsKV, dv, DROP == 1 ? a.drop_scale : 1.f, dVb, RW::ss(a.mdv), a.sk - k0w, RW::cols(a), l);
  };
  PanelLane pl;
  pl.init(l);
  int s0 = 0; // stream position of the item's first tile: tile j of it is in stage (s0 + j) % NST

  for (;;) {
    const int bh = nbh, ktile = nkt;
    const int key = ktile * KT + w * 32 + kl;
    const int qt0 = first_tile(ktile);
    const int nj = nqt - qt0;             // query tiles it walks
    const int ntl = nj < 3 ? 3 : nj;      // turns it takes: at least three, so that the stream looks one item ahead at most
    seek();
    bwd_vm_wait<0>();
    bwd_lds_barrier(); // tiles 0 .. 2, the K and V rows and the raw rows are there, and nobody reads the last item's any more

    // ---- per-key operands
    v8 kreg[KS], vreg[KS], bxs, bxd;
    {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bool live = ks * 16 + h * 8 < RW::cols(a);
        const v8 kraw = as_v8<T>(chunk_or_zero(as_u32x4(panel_read_rows<T, 32>(ldsKV, pl, 0, ks)), live));
        const v8 vraw = as_v8<T>(chunk_or_zero(as_u32x4(panel_read_rows<T, 32>(ldsKV + TILEB, pl, 0, ks)), live));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          kreg[ks][j] = (T)((float)kraw[j] * a.scale_l2);
          vreg[ks][j] = DROP == 1 ? (T)((float)vraw[j] * a.drop_scale) : vraw[j];
        }
      }
      const float mk = key < a.sk ? 0.f : BIGNEG;
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
    stage_rows(first_seg(ktile));
    if (pbh >= 0) { // the previous item's gradients leave under this one's products
      store_item();
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          dk[db][r] = 0.f;
          dv[db][r] = 0.f;
        }
    }
    pbh = bh;
    pkt = ktile;
    bwd_lds_barrier(); // the extra-step rows are there, and the raw ones free
    auto next_raw = [&](int seg0) { // behind the staging of segment seg0
      if (seg0 + C::QSEG < a.sq) copy_raw(bh, seg0 + C::QSEG);
      else if (more) copy_raw(nbh, first_seg(nkt));
    };
    next_raw(first_seg(ktile));

    if (more) copy_kv(nbh, nkt); // (this item's have become registers, and the last item's output rows have gone through there)
    from_item(bh, qt0 + NST - 1);
    cs.left = ntl - (NST - 1);
    auto next_copy = [&]() { // before the copies of a turn
      if (cs.left == 0) { // (a branch, taken once per item: nothing of it is kept in registers meanwhile)
        if (more) from_item(nbh, first_tile(nkt)); // (without a next item tiles past the end: rows of the last one)
        cs.left = 0x7fffffff;
      }
      --cs.left;
    };
    auto dst_of = [&](int j) -> uint32_t { return lds_base + (uint32_t)((s0 + j) & (NST - 1)) * STAGEB; };
    auto copy_tile = [&](int j) {
      next_copy();
#pragma unroll
      for (int i = 0; i < VPT; ++i) copy_one(dst_of(j), i);
      ++cs.tile;
    };
    auto stage_of = [&](int j) -> const char * { return lds + ((s0 + j) & (NST - 1)) * STAGEB; };

    f32x16 xA, gA, xB, gB;
    uint32_t rbA[4], rbB[4];
    PhiloxSlices ph;
    const uint32_t sel1 = (l & 1) ? 0x03070105u : 0x06020400u, sel2 = (l & 2) ? 0x03020706u : 0x05040100u; // see drop_bytes_k

    auto xrow = [&](int j) -> v8 { return as_v8<T>(ldsX[((qt0 + j) * BT + kl) & (C::QSEG - 1)]); };
    auto step = [&](auto next_tag, int tj, const f32x16 &xc, const f32x16 &gc, const uint32_t (&rc)[4],
                    f32x16 &xn, f32x16 &gn, uint32_t (&rn)[4]) {
      constexpr bool NEXT = decltype(next_tag)::value;
      constexpr int NX = NEXT ? 2 : 0, NA = NEXT ? 2 * KS : 0, NC = 4 * DB, NO = NA + NC, NM = NX + NO;
      constexpr int AHEAD = 4;
      constexpr int NS = 10;
      constexpr int NP = DROP == 1 && NEXT ? 15 : 0;
      constexpr int JS = NEXT ? NX + NA : 0;
      const char *ldsN = stage_of(tj + 1);
      const char *ldsC = stage_of(tj);
      next_copy();
      const uint32_t dst = dst_of(tj + NST - 1);
      const int q0 = (qt0 + tj) * BT;
      DropCtx dctx = a.drop; // (the ten rounds' keys are formed where they are used: kept for the whole kernel they would not fit)
      if (DROP == 1) asm volatile("" : "+s"(dctx.seed_lo), "+s"(dctx.seed_hi));
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
            p[e] = fast_exp2(xc[e]);
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
        if (s == 0) ph.start(dctx, (uint32_t)bh, (uint32_t)((q0 + BT) >> 2) + (uint32_t)h + 2u * ((uint32_t)l & 3u), (uint32_t)key >> 2);
        else if (s <= 10) ph.round(dctx, s - 1);
        else {
          const int t = s - 11;
          const uint32_t a1 = __builtin_amdgcn_perm(quad_perm<0xB1>(ph.c[t]), ph.c[t], sel1);
          rn[t] = __builtin_amdgcn_perm(quad_perm<0x4E>(a1), a1, sel2);
        }
      };
      v8 opnd[NO], xa;
      if (NEXT) xa = xrow(tj + 1);
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
          if (m == 0) M::start(xa, bxs, xn);
          else M::start(xa, bxd, gn);
        } else {
          const int j = m - NX;
          if (j + AHEAD < NO) opnd[j + AHEAD] = fetch(j + AHEAD);
          const int u = j ^ 1; // (the later one of a pair first: its wait covers the other)
          if (u < NA) {
            if ((u & 1) == 0) M::add(opnd[u], kreg[u >> 1], xn);
            else M::add(opnd[u], vreg[u >> 1], gn);
          } else {
            const int i = u - NA, db = (i >> 1) % DB, c = (i >> 1) / DB;
            f32x16 &acc = (i & 1) ? dk[db] : dv[db];
            const v8 fr = (i & 1) ? df[c] : pf[c];
            acc = E::mfma(opnd[u], fr, acc);
          }
        }
        if (m % (NM / VPT) == NM / VPT - 1 && m / (NM / VPT) < VPT) copy_one(dst, m / (NM / VPT));
        const int upto = m < JS ? (m + 1) * NS / (JS ? JS : 1) : NS + (m - JS + 1) * NP / (NM - JS);
#pragma unroll
        for (; done < upto; ++done) {
          if (done < NS) softmax(done);
          else philox(done - NS);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      ++cs.tile;
    };
    using Yes = std::true_type;
    using No = std::false_type;

    auto first = [&](int tj, f32x16 &x, f32x16 &g, uint32_t (&rb)[4]) {
      const char *t = stage_of(tj);
      if (DROP == 1) drop_bytes_k(a.drop, (uint32_t)bh, (uint32_t)((qt0 + tj) * BT), (uint32_t)key, h, l, rb);
      const v8 xa = xrow(tj);
      constexpr int AHEAD = 2; // (operand pairs asked for ahead of their products)
      v8 ox[KS], og[KS];
      auto fetch = [&](int ks) {
        ox[ks] = panel_read_rows<T, BT>(t, pl, 0, ks);
        og[ks] = panel_read_rows<T, BT>(t + TILEB, pl, 0, ks);
      };
#pragma unroll
      for (int ks = 0; ks < AHEAD; ++ks) fetch(ks);
      asm volatile("s_nop 4"); // (the operands may just have been written)
      M::start(xa, bxs, x);
      M::start(xa, bxd, g);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + AHEAD < KS) fetch(ks + AHEAD);
        M::add(ox[ks], kreg[ks], x);
        M::add(og[ks], vreg[ks], g);
        __builtin_amdgcn_sched_barrier(0);
      }
      settle(x, g);
      if (CAUSAL) { // the wave's first tile is the one on its diagonal
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = key <= (qt0 + tj) * BT + 8 * (r / 4) + 4 * h + r % 4 ? x[r] : BIGNEG;
      }
    };
    // top of the iteration of tile j: tile j + 1 has landed, tile j - 1 is no longer read.  Copies land in the order in which
    // they were asked for.  (Tiles 0 .. 2 were waited for between the items.)
    auto turn = [&](int j) {
      if (j >= 2) bwd_vm_wait<VPT>();
      bwd_lds_barrier();
      if (a.sq > C::QSEG && ((qt0 + j + 1) * BT & (C::QSEG - 1)) == 0 && j + 1 < nj) { // (j >= 3: the raw rows are older than tile 3)
        stage_rows((qt0 + j + 1) * BT);
        bwd_lds_barrier();
        next_raw((qt0 + j + 1) * BT);
      }
    };
    int j = 0;
    // causal: query tiles ahead of the one that holds this wave's own diagonal see none of its keys
    if (CAUSAL) {
      for (; j < (ws < nj ? ws : nj); ++j) {
        turn(j);
        copy_tile(j + NST - 1);
      }
    }
    if (j < nj) {
      const int nmid = nj - 1 - j;
      if (nmid & 1) {
        first(j, xB, gB, rbB);
        turn(j);
        step(Yes{}, j, xB, gB, rbB, xA, gA, rbA);
        ++j;
      } else {
        first(j, xA, gA, rbA);
      }
      for (; j < nj - 1; j += 2) {
        turn(j);
        step(Yes{}, j, xA, gA, rbA, xB, gB, rbB);
        turn(j + 1);
        step(Yes{}, j + 1, xB, gB, rbB, xA, gA, rbA);
      }
      turn(j);
      step(No{}, j, xA, gA, rbA, xB, gB, rbB);
      ++j;
    }
    for (; j < ntl; ++j) { // (heads of one or two query tiles)
      turn(j);
      copy_tile(j + NST - 1);
    }
    s0 += ntl;
    if (!more) break;
  }
  bwd_vm_wait<0>(); // no copy may still be on its way into LDS when the wave ends
  store_item();
}

} // namespace fmha
