// Instantiates the backward kernels for one (element type, head dim, row layout kind) triple, chosen
// with -DFMHA_TU_BF16={0,1} -DFMHA_TU_D={32,64,96,128,256} -DFMHA_TU_STRIDED={0,1}, and exports their dispatcher.
#include "fmha_launch.h"
#ifndef FMHA_TU_STRIDED
#define FMHA_TU_STRIDED 0
#endif
#if FMHA_TU_D == 64
#define FMHA_TU_SHORT 1
#include "fmha_bwd_short.h"
#else
#define FMHA_TU_SHORT 0
#endif
#if FMHA_TU_D == 256 || defined(FMHA_BWD_FORCE_WIDE) // (the second: development builds, to measure the wave-pair kernel at narrower heads)
#define FMHA_TU_WIDE 1
#include "fmha_bwd_wide.h"
#else
#define FMHA_TU_WIDE 0
#endif

#if FMHA_TU_BF16
#define FMHA_TU_T __bf16
#define FMHA_TU_TNAME bf16
#else
#define FMHA_TU_T _Float16
#define FMHA_TU_TNAME f16
#endif
#if FMHA_TU_STRIDED
#define FMHA_CAT3(a, b, c) a##b##_d##c##_strided
#else
#define FMHA_CAT3(a, b, c) a##b##_d##c
#endif
#define FMHA_NAME(t, d) FMHA_CAT3(bwd_dispatch_, t, d)
#define FMHA_PIPE_NAME(t, d) FMHA_CAT3(bwd_pipe_launch_, t, d)
#define FMHA_ONE_NAME(t, d) FMHA_CAT3(bwd_one_launch_, t, d)

namespace fmha {
namespace {

constexpr int kNW = 4;
constexpr int kQB = 1; // 32-query blocks per wave in the dQ kernel
constexpr int kKB = 1; // 32-key blocks per wave in the dK/dV kernel
constexpr bool kStrided = FMHA_TU_STRIDED != 0;

template <typename K> int set_lds(K kern, int bytes) {
  return hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                             bytes) == hipSuccess ? 0 : 2;
}

// The pipelined kernels (fmha_bwd_pipe.hip) take everything but full mask tensors and, at head dim 256, dK / dV -- at head dims 128
// and 256 from a number of queries on, because their prologue costs more.
// Kernel times, us, pipelined / phase by phase, 512 heads, D 128, fp16, S queries and keys:
//   dQ, no causal mask     S 61 13 / 11, S 128 20 / 21, S 256 58 / 62, S 512 131 / 131, S 1024 402 / 418
//     with dropout         S 61 15 / 13, S 128 22 / 22, S 256 59 / 59, S 512 147 / 152, S 1024 455 / 471
//   dK+dV (persistent)     S 61 16 / 13, S 128 23 / 23, S 192 44 / 48, S 256 56 / 62, 2048 heads S 128 80 / 104
//     with dropout         S 61 19 / 17, S 128 27 / 31
//   dK+dV, causal          S 128 27 / 30, S 192 43 / 56, S 256 55 / 71, 2048 heads S 128 with dropout 101 / 126
//   dK+dV of few heads (one round of workgroups, the plain pipelined kernel): 64 heads S 200 12 / 17, causal 14 / 16
// The line is 128 queries (192 for causal dK / dV that is not persistent, see fmha_bwd_pipe.hip).
// At head dim 96 dK / dV is never pipelined: phase by phase on 32-row tiles it has the
// registers for two waves per SIMD, pipelined it does not (backward, us, persistent or pipelined / so: BH 512 S 512 padding mask and
// dropout 316 / 270, without either 265 / 245; causal BH 608 S 365 181 / 158, BH 128 S 1024 with dropout 171 / 154, BH 32 S 3000 232 /
// 228; BH 576 S 120 56 / 49).
template <int MASK, bool CAUSAL, int DROP> constexpr bool pipe_built() { return FMHA_TU_D != 256 && MASK != kMaskFull; }
static inline bool pipe_wanted(const BwdArgs &a) { return FMHA_TU_D <= 64 || a.sq >= 128; }
// dQ of causal heads at head dim 128 follows the same line (backward, us, phase by phase / pipelined, 512 heads: S 160 bf16 73.1 / 72.1,
// S 256 106.8 / 105.7, S 384 169.4 / 163.8, S 512 248 / 244, S 768 446 / 418, S 895 fp16 627 / 573; with dropout S 200 107 / 103, S 640
// fp16 423 / 387; BH 64 S 512 47.9 / 41.4, BH 100 S 700 87.6 / 87.7, BH 40 S 800 with dropout 76.4 / 61.3).
// dQ at head dim 256, one wave per SIMD: from 128 queries on as well (us, pipelined / phase by phase: BH 128 S 2048 750 / 1041,
// causal 440 / 616; BH 64 S 1000 with dropout 118 / 140; BH 300 S 512 bf16 causal with dropout 174 / 244; BH 512 S 256 119 / 126,
// causal 113 / 126, S 128 42.6 / 43.7; BH 1000 S 129 causal 164 / 174; BH 8 S 1750 59 / 102).
template <typename K> int launch_one(K kern, BwdArgs &a, long long nblk, int threads, int lds, hipStream_t s) {
  if (nblk > 0x7fffffffLL) return 2;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(threads), lds, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

template <int MASK, bool CAUSAL, int DROP> int launch_dq(BwdArgs &a, const BwdVariant &v, long long nblk, hipStream_t s) {
  if constexpr (MASK != kMaskFull) { // (pipe_built, or head dim 256, where it is built for dQ only)
    if (pipe_wanted(a)) return FMHA_PIPE_NAME(FMHA_TU_TNAME, FMHA_TU_D)(a, v, false, nblk, s);
  }
  if constexpr (!(pipe_built<MASK, CAUSAL, DROP>() && FMHA_TU_D <= 64)) { // (there the pipelined kernel takes all)
    constexpr int kLds = BwdCfg<FMHA_TU_D, bwd_dq_tile_rows<FMHA_TU_D>()>::LDS_BYTES;
    static_assert(kLds <= 160 * 1024, "tiles do not fit the LDS of a compute unit");
    auto kern = fmha_bwd_dq_kernel<FMHA_TU_T, FMHA_TU_D, kQB, kNW, MASK, CAUSAL, DROP, kStrided>;
    static const int attr = set_lds(kern, kLds);
    return attr ? 2 : launch_one(kern, a, nblk, kNW * 64, kLds, s);
  }
  return 1;
}

template <int MASK, bool CAUSAL, int DROP> int launch_dkdv(BwdArgs &a, const BwdVariant &v, long long nblk, hipStream_t s) {
#if FMHA_TU_WIDE
  // head dim 256: the dK / dV work of a key block is split between two waves (fmha_bwd_wide.h; at head
  // dims 128 and 64 the same kernel measured level with and a third slower than the one-wave kernel)
  using Cfg = BwdWideCfg<FMHA_TU_D, MASK>;
  static_assert(Cfg::LDS_BYTES <= 160 * 1024, "tiles do not fit the LDS of a compute unit");
  auto kern = fmha_bwd_dkdv_wide_kernel<FMHA_TU_T, FMHA_TU_D, MASK, CAUSAL, DROP, kStrided>;
  static const int attr = set_lds(kern, Cfg::LDS_BYTES);
  return attr ? 2 : launch_one(kern, a, nblk, Cfg::NW * 64, Cfg::LDS_BYTES, s);
#else
  constexpr bool kPipe = pipe_built<MASK, CAUSAL, DROP>();
  // One exception: under a mask or key counts, without causal mask and dropout, short heads' dK / dV at head dim 128 stays on 32-row
  // tiles at two waves per SIMD, which overlap one workgroup's start and stores with another's arithmetic as the persistent
  // kernel does where there is neither: below 192 queries, and up to 384 of rows shorter than the kernel's.  Backward under padding
  // masks / key counts, us, so / pipelined: BH 512 S 128 48.3 / 51.0, 45.6 / 50.8, S 160 level; S 197 110.9 / 100.3, S 258 156 / 133, 135
  // / 129, S 512 417 / 329, 316 / 307, packed 464 / 342, 460 / 325; BH 256 S 1024 702 / 524, 503 / 491, packed 796 / 527, 785 / 503; 112
  // to 120 columns BH 192 S 320 65.3 / 66.6, 65.9 / 64.4, S 384 87.7 / 92.2, 84.5 / 87.5, BH 512 S 416 270 / 251, 278 / 245, BH 64 S 2048
  // 502 / 430, 476 / 377.  (Whole folded rows under key counts of 192 to 256 queries: 64 to 128 heads a fifth less, BH 256 S 256 50.2 / 52.1, BH 512
  // S 256 95.8 / 100.3; the line must not depend on the number of heads, with which a head's gradients would change.)
  constexpr bool kTwoWaves = bwd_dkdv_small_tiles<FMHA_TU_D, CAUSAL, DROP>();
  if constexpr (kPipe && FMHA_TU_D != 96) { // (see pipe_wanted)
    const bool two_waves = kTwoWaves && (MASK != kMaskNone || a.kv_len) && (a.dcols < FMHA_TU_D ? a.sq <= 384 : a.sq < 192);
    if (pipe_wanted(a) && !two_waves) {
      const int rc = FMHA_PIPE_NAME(FMHA_TU_TNAME, FMHA_TU_D)(a, v, true, nblk, s);
      if (FMHA_TU_D <= 64 || rc != kBwdNotHere) return rc;
    }
  }
  if constexpr (!(kPipe && FMHA_TU_D <= 64)) {
    using Cfg = BwdCfg<FMHA_TU_D, bwd_dkdv_tile_rows<FMHA_TU_D, CAUSAL, DROP>()>;
    constexpr int kLds = Cfg::LDS_BYTES + (MASK == kMaskFull ? Cfg::MASK_BYTES : 0);
    static_assert(kLds <= 160 * 1024, "tiles do not fit the LDS of a compute unit");
    auto kern = fmha_bwd_dkdv_kernel<FMHA_TU_T, FMHA_TU_D, kKB, kNW, MASK, CAUSAL, DROP, kStrided>;
    static const int attr = set_lds(kern, kLds);
    return attr ? 2 : launch_one(kern, a, nblk, kNW * 64, kLds, s);
  }
  return 1;
#endif
}

template <int MASK, bool CAUSAL, int DROP> int launch(BwdArgs &a, const BwdVariant &v, hipStream_t s) {
#if FMHA_TU_WIDE
  constexpr int KT = BwdWideCfg<FMHA_TU_D, MASK>::KT;
#else
  constexpr int KT = kNW * kKB * 32;
#endif
  constexpr int QT = kNW * kQB * 32;
  // Causal: workgroups take pairs of tiles (see bwd_item) when that leaves at least two rounds of workgroups for the device, but not
  // of three tiles, where the middle one is left alone with half a pair's work (us, paired / one by one, longest first: D 64
  // BH 1000 S 300 dQ 70.7 / 63.6, dK / dV 74.3 / 63.8, BH 1500 S 380 with dropout 138 / 120 and 170 / 145; D 128 BH 600 S 380 109 / 93
  // and 128 / 105).  Otherwise the longest tiles of all heads go first, except where three or five tiles leave two or three rounds:
  // there a head's tiles beside each other, which read its rows from one L2, are ahead, for dK / dV without dropout only (backward, us,
  // longest first / so, bf16: BH 448 S 380 packed 92.5 / 85.0, D 32 78.2 / 68.4, BH 320 S 640 packed 127.9 / 115.8, folded 113.5 / 107.0,
  // BH 600 S 300 with dropout 96.7 / 93.1), and where a handful of tiles start a second round (D 64 BH 104 S 640 packed 46.2 / 42.6,
  // D 32 43.4 / 38.5; but with eleven tiles, BH 48 S 1368, 57 / 68).
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      n = 0;
    return n;
  }();
  const int qtiles = (a.sq + QT - 1) / QT, ktiles = (a.sk + KT - 1) / KT;
  const bool uneven = !CAUSAL && (MASK == kMaskPerKey || (MASK == kMaskNone && a.kv_len));
  const bool share = rows_share_lines(a.mq.heads, a.mq.sh, a.mq.ss) || rows_share_lines(a.mk.heads, a.mk.sh, a.mk.ss);
  const bool dealt = uneven && bwd_heads_dealt(share, a.bh, qtiles, ktiles);
  // dQ of short heads at head dim 256 is dealt alone from four rounds of workgroups on (backward: BH 1024 S 128 both kernels dealt 3 to 6 % less
  // than ranges, dQ alone 1.5 to 4 % less than both; BH 2240 S 56 and S 24 level).
  const bool one = FMHA_TU_D == 256 && uneven && !share && qtiles == 1 && a.bh >= 4 * cus;
  auto blocks = [&](int ntile, bool dq) -> long long {
    const long long tiles = (long long)a.bh * ntile, pairs = (long long)a.bh * ((ntile + 1) / 2), over = tiles - 2LL * cus;
    const bool by_head = (ntile == 3 || ntile == 5) && ((tiles >= (ntile + 1LL) * cus && (dq || DROP == 0)) || (FMHA_TU_D <= 64 && over > 0 && 16 * over <= cus));
    a.ntile = ntile;
    a.pair = kTilesByLength;
    if (CAUSAL && v.pair >= 0) a.pair = v.pair;
    else if (CAUSAL && ntile != 3 && pairs >= 4LL * cus) a.pair = kTilesPaired;
    else if (CAUSAL && by_head) a.pair = kTilesByHead;
    a.lg = head_groups_log2(a.bh);
    a.units = !CAUSAL || a.pair == kTilesByHead ? ntile : a.pair == kTilesPaired ? (ntile + 1) / 2 : a.bh >> a.lg;
    a.dealt = dealt || (one && dq) ? bwd_dealt_blocks(a.bh, ntile) : 0;
    a.range = bwd_range_blocks(a.pair == kTilesPaired ? pairs : tiles, a.dealt);
    return a.pair == kTilesPaired ? pairs : tiles;
  };
  // dQ first: it also writes delta, which the dK/dV kernel reads (same stream => ordered)
  const long long nq = blocks(qtiles, true);
  if (const int rc = launch_dq<MASK, CAUSAL, DROP>(a, v, nq, s)) return rc;
  const long long nk = blocks(ktiles, false);
  return launch_dkdv<MASK, CAUSAL, DROP>(a, v, nk, s);
}

#if FMHA_TU_SHORT
// sq, sk <= 128: one workgroup per head computes dQ, dK and dV from one copy of the head in LDS
template <int DROP, int SMAX, bool CAUSAL> int launch_short(BwdArgs &a, hipStream_t s) {
  using Cfg = BwdShortCfg<SMAX>;
  auto kern = fmha_bwd_short_kernel<FMHA_TU_T, DROP, SMAX, CAUSAL, kStrided>;
  static const int attr = set_lds(kern, Cfg::LDS_BYTES);
  if (attr) return 2;
  hipLaunchKernelGGL(kern, dim3((unsigned)a.bh), dim3(Cfg::NW * 64), Cfg::LDS_BYTES, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}
#endif

template <int MASK, bool CAUSAL> int by_drop(BwdArgs &a, const BwdVariant &v, hipStream_t s) {
  if (v.drop == 0) return launch<MASK, CAUSAL, 0>(a, v, s);
  if (v.drop == 1) return launch<MASK, CAUSAL, 1>(a, v, s);
  return 1;
}

} // namespace

int FMHA_NAME(FMHA_TU_TNAME, FMHA_TU_D)(BwdArgs &a, const BwdVariant &v, hipStream_t s) {
#if FMHA_TU_SHORT
  if (v.short_seq) {
    // Beyond 128 rows a launch of more heads than the device holds at once goes to the one-pass kernel, which forms the scores
    // once and has the next head's rows on their way (us, one-pass / this kernel, S 256 BH 300 38.1 / 41.5, S 130 BH 300 with
    // dropout 28.1 / 31.3, S 200 BH 257 causal 29.4 / 31.3; more in fmha_bwd_one.h).  Where every head has a compute unit to
    // itself there is no next head, and its longer start shows: S 130 BH 256 15.2 / 14.3, S 200 BH 100 17.2 / 16.5, S 256
    // BH 64 18.7 / 18.2, though S 256 BH 256 25.4 / 27.0.
    const bool small = a.sq <= 128 && a.sk <= 128;
    if (!small) {
      const int rc = FMHA_ONE_NAME(FMHA_TU_TNAME, FMHA_TU_D)(a, v, s);
      if (rc != kBwdNotHere) return rc;
    }
    if (v.causal) {
      if (small) return v.drop == 1 ? launch_short<1, 128, true>(a, s) : launch_short<0, 128, true>(a, s);
      return v.drop == 1 ? launch_short<1, 256, true>(a, s) : launch_short<0, 256, true>(a, s);
    }
    if (small) return v.drop == 1 ? launch_short<1, 128, false>(a, s) : launch_short<0, 128, false>(a, s);
    return v.drop == 1 ? launch_short<1, 256, false>(a, s) : launch_short<0, 256, false>(a, s);
  }
#else
  if (v.short_seq) return 1;
#endif
  if (v.mask == kMaskPerKey)
    return v.causal ? by_drop<kMaskPerKey, true>(a, v, s) : by_drop<kMaskPerKey, false>(a, v, s);
#if FMHA_TU_D % 64 == 0
  if (v.mask == kMaskFull)
    return v.causal ? by_drop<kMaskFull, true>(a, v, s) : by_drop<kMaskFull, false>(a, v, s);
#else // (full mask tensors: the next whole panel's kernels)
  if (v.mask == kMaskFull) return 1;
#endif
  return v.causal ? by_drop<kMaskNone, true>(a, v, s) : by_drop<kMaskNone, false>(a, v, s);
}

} // namespace fmha
