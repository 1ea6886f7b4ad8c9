// Instantiates the forward kernel for one (element type, head dim, row layout kind) triple, chosen
// with -DFMHA_TU_BF16={0,1} -DFMHA_TU_D={32,64,96,128,256} -DFMHA_TU_STRIDED={0,1}, and exports its dispatcher.
#include "fmha_launch.h"
#include "fmha_fwd_pipe.h"
#ifndef FMHA_TU_STRIDED
#define FMHA_TU_STRIDED 0
#endif
#if FMHA_TU_D != 256 && !FMHA_TU_STRIDED
#define FMHA_TU_ROWS 1 // the kernels that move [.., sq, sk] tensors as whole rows
#include "fmha_fwd_save.h"
#include "fmha_fwd_stream.h"
#include "fmha_fwd_stream_save.h"
#include "fmha_fwd_cols.h"
#else
#define FMHA_TU_ROWS 0
#endif
#if FMHA_TU_D == 64 && !FMHA_TU_STRIDED
#define FMHA_TU_SHORT 1
#include "fmha_fwd_short.h"
#include "fmha_fwd_head.h"
#include "fmha_fwd_mid.h"
#else
#define FMHA_TU_SHORT 0
#if FMHA_TU_D == 64
#include "fmha_fwd_short.h" // run-time row layouts: its builds without a full mask tensor
#include "fmha_fwd_head.h"  // the whole-head kernel
#include "fmha_fwd_mid.h"   // and the one for 129 to 256 keys
#endif
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
#define FMHA_NAME(t, d) FMHA_CAT3(fwd_dispatch_, t, d)

namespace fmha {
namespace {

#ifndef FMHA_FWD_NW
#define FMHA_FWD_NW 4
#endif
constexpr int kNW = FMHA_FWD_NW;
constexpr bool kStrided = FMHA_TU_STRIDED != 0;

template <int QB, int MASK, bool CAUSAL, int DROP, bool kPipe = (DROP != 2)> int launch(FwdArgs &a, hipStream_t s) {
  constexpr int kLds = kPipe ? PipeCfg<FMHA_TU_D, QB>::lds_bytes(kNW) : FwdCfg<FMHA_TU_D>::LDS_BYTES;
  // the save pass (and tensor dropout at head dim 128) runs on the plain loop; everything else is
  // software-pipelined
  auto kern = [] {
    if constexpr (!kPipe) return fmha_fwd_kernel<FMHA_TU_T, FMHA_TU_D, QB, kNW, MASK, CAUSAL, DROP, kStrided && FMHA_TU_D == 256>;
    else return fmha_fwd_pipe_kernel<FMHA_TU_T, FMHA_TU_D, QB, kNW, MASK, CAUSAL, DROP, kStrided>;
  }();
  // once per kernel: allow the dynamic LDS size, and for the persistent kernel find how many
  // workgroups the device keeps resident (that is its grid size)
  static const int resident = [&]() -> int {
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds) !=
        hipSuccess)
      return -1;
    if (!kPipe) return 0;
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(kern), kNW * 64, kLds) !=
            hipSuccess ||
        cus <= 0 || per_cu <= 0)
      return -1;
    return cus * per_cu;
  }();
  if (resident < 0) return 2;
  constexpr int QT = kNW * QB * 32;
  a.nqt = (a.sq + QT - 1) / QT;
  long long nblk = (long long)a.bh * a.nqt;
  if (nblk > 0x7fffffffLL) return 2;
  if (kPipe && nblk > resident) nblk = resident;
  // Causal items, from half a round to four: by length, unless the rounds pair a head's tiles exactly anyway (whole heads in an
  // even number of rounds).  A head's items in turn met as they came, and a workgroup with two long ones ended the launch (us,
  // bf16, in turn / by length): D 64 16 heads S 5573 169 / 90, 84 heads S 1562 74 / 46, 88 heads S 2368 132 / 90, 300 heads S 512
  // 31.8 / 26.8; D 128 32 heads S 4286 240 / 155, 48 heads S 2194 101 / 74, 12 heads S 3584 85 / 72, 40 heads S 1000 33.3 / 27.9.
  // Exact pairs keep a head on fewer compute units at a time (32 heads S 4001), beyond four rounds little is left to gain.  At head dim 128
  // a head's rows are worth more and it ends at three and a quarter (us, by length / in turn: 472 heads S 512 80 / 72, 236 heads S 900 104 / 96, but 188
  // heads S 1024 ahead by 5 %), with up to three tiles at two and a quarter (528 heads S 384 packed 81 / 75); dropout on packed
  // rows keeps four (472 heads S 512 ahead by 6 %).
  a.deal = a.deal_heads = 0;
  if (kPipe && CAUSAL && MASK == kMaskNone && a.sk_whole == 0) {
    const long long items = (long long)a.bh * a.nqt, G = nblk;
    constexpr bool kWhole = (FMHA_TU_D != 96 && FMHA_TU_D != 128) || (DROP != 0 && kStrided);
    const int quarters = kWhole ? 16 : DROP == 0 && a.nqt <= 3 ? 9 : 13;
    if (2 * items > resident && 4 * items < quarters * G && !(G % a.nqt == 0 && items % (2 * G) == 0)) {
      int lg = 0;
      while (G % 8 == 0 && lg < 3 && a.bh % (2 << lg) == 0) ++lg;
      a.deal = lg + 1;
      a.deal_heads = a.bh >> lg;
    }
  }
  a.bal_rows = 0;
  if (kPipe && MASK == kMaskPerKey && !CAUSAL && a.mask_div > 0 && a.bh % a.mask_div == 0) {
    // shapes whose mask rows can be dealt to the workgroups by length (see FwdArgs::bal_rows): an
    // additive mask (its values are compared as they are), rows of whole 16-byte pieces, at most 64
    // pieces of 512 keys in all
    const long long items = (long long)a.bh * a.nqt, ipr = (long long)a.mask_div * a.nqt, rows = a.bh / a.mask_div;
    const bool shape = nblk % ipr == 0 && items % nblk == 0 && items / nblk >= 2 && items / nblk <= 4 &&
                       rows == items / nblk * (nblk / ipr);
    const bool mask_ok = a.mask_a == FMHA_LOG2E && a.mask_b == 0.f && a.sk % 8 == 0 && a.sk > 128 && a.sk <= 1024 &&
                         rows * ((a.sk + 511) / 512) <= 64 && a.mask_sb % 8 == 0 &&
                         (reinterpret_cast<uintptr_t>(a.mask) & 15) == 0;
    if (shape && mask_ok && !a.kv_len && a.sk_whole == 0 && !(a.flags & kFwdFlagNoTrim)) {
      a.bal_rows = (int32_t)rows;
      a.bal_ipr = (int32_t)ipr;
      a.bal_R = (int32_t)(nblk / ipr);
      a.bal_inv_ipr = 1.f / (float)ipr;
    }
  }
  if constexpr (kPipe && CAUSAL && MASK == kMaskNone) {
    if (a.deal) {
      auto dealt = fmha_fwd_pipe_kernel<FMHA_TU_T, FMHA_TU_D, QB, kNW, MASK, CAUSAL, DROP, kStrided, true>;
      static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void *>(dealt), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                    kLds) == hipSuccess;
      if (!ready) return 2;
      hipLaunchKernelGGL(dealt, dim3((unsigned)nblk), dim3(kNW * 64), kLds, s, a);
      return hipGetLastError() == hipSuccess ? 0 : 2;
    }
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(kNW * 64), kLds, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

#if FMHA_TU_D == 64
// short key ranges in one pass: under a full mask tensor (the reference's operators at their own shape), and under
// no mask / a per-key mask / valid key counts, without dropout or with the Philox rule
template <int MASK, int DROP, bool SAVE, bool FULL, bool TAIL = false> int launch_short_as(FwdArgs &a, hipStream_t s) {
  static_assert(MASK != kMaskFull || !kStrided, "full mask tensors: folded layout only");
  auto kern = [] {
    if constexpr (MASK == kMaskFull && TAIL) return fmha_fwd_short_tail_kernel<FMHA_TU_T, DROP, SAVE, FULL>;
    else if constexpr (MASK == kMaskFull) return fmha_fwd_short_kernel<FMHA_TU_T, DROP, SAVE, FULL>;
    else return fmha_fwd_short_kernel_keymask<FMHA_TU_T, MASK, DROP, FULL, kStrided>;
  }();
  constexpr int kLds = MASK == kMaskFull ? ShortCfg::LDS_BYTES : ShortCfg::LDS_BYTES_KEYMASK;
  static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                hipFuncAttributeMaxDynamicSharedMemorySize, kLds) == hipSuccess;
  if (!ready) return 2;
  a.nqt = (a.sq + ShortCfg::QT - 1) / ShortCfg::QT;
  const long long nblk = (long long)a.bh * a.nqt;
  if (nblk > 0x7fffffffLL) return 2;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(ShortCfg::NW * 64), kLds, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}
// (more than 96 keys: every 32-key block exists, and the kernel is built without the conditions around them)
template <int MASK, int DROP, bool SAVE> int launch_short(FwdArgs &a, hipStream_t s) {
  if constexpr (MASK == kMaskFull)
    if (a.sk & 7) // rows that end within a 16-byte piece
      return a.sk > ShortCfg::SKMAX - 32 ? launch_short_as<MASK, DROP, SAVE, true, true>(a, s)
                                         : launch_short_as<MASK, DROP, SAVE, false, true>(a, s);
  return a.sk > ShortCfg::SKMAX - 32 ? launch_short_as<MASK, DROP, SAVE, true>(a, s)
                                     : launch_short_as<MASK, DROP, SAVE, false>(a, s);
}
#endif

#if FMHA_TU_D == 64
// 129 to 256 keys
template <int NW, int MASK, bool CAUSAL, int DROP> int launch_mid_as(FwdArgs &a, hipStream_t s) {
  using MidCfg = fmha::MidCfg<NW>;
  auto kern = fmha_fwd_mid_kernel<FMHA_TU_T, NW, MASK, CAUSAL, DROP, kStrided>;
  static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                hipFuncAttributeMaxDynamicSharedMemorySize, MidCfg::LDS_BYTES) == hipSuccess;
  if (!ready) return 2;
  if (a.sk > MidCfg::SKMAX) return 1;
  a.nqt = (a.sq + MidCfg::QT - 1) / MidCfg::QT;
  const long long nblk = (long long)a.bh * a.nqt;
  if (nblk > 0x7fffffffLL) return 2;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(MidCfg::NT), MidCfg::LDS_BYTES, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}
template <int NW, int MASK> int launch_mid(FwdArgs &a, const FwdVariant &v, hipStream_t s) {
  if (v.causal) return v.drop == 1 ? launch_mid_as<NW, MASK, true, 1>(a, s) : launch_mid_as<NW, MASK, true, 0>(a, s);
  return v.drop == 1 ? launch_mid_as<NW, MASK, false, 1>(a, s) : launch_mid_as<NW, MASK, false, 0>(a, s);
}
#endif

#if FMHA_TU_ROWS
// the saved outputs of the save-intermediates operator, from the row log-sum-exp of a forward launch
template <bool TAIL> int launch_save_as(FwdArgs &a, hipStream_t s) {
  using SaveCfg = fmha::SaveCfg<FMHA_TU_D>;
  auto kern = fmha_fwd_save_kernel<FMHA_TU_T, FMHA_TU_D, TAIL>;
  static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                hipFuncAttributeMaxDynamicSharedMemorySize, SaveCfg::LDS_BYTES) == hipSuccess;
  if (!ready) return 2;
  a.nqt = (a.sq + SaveCfg::QT - 1) / SaveCfg::QT;
  const long long nblk = (long long)a.bh * a.nqt;
  if (nblk > 0x7fffffffLL) return 2;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(SaveCfg::NW * 64), SaveCfg::LDS_BYTES, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

int launch_save(FwdArgs &a, hipStream_t s) { return a.sk & 7 ? launch_save_as<true>(a, s) : launch_save_as<false>(a, s); }

// long key ranges under a full mask tensor (and a dropout tensor): the streaming forward
template <bool DROPT, bool TAIL, bool MANY> int launch_stream_as(FwdArgs &a, hipStream_t s) {
  using StreamCfg = fmha::StreamCfg<FMHA_TU_D, MANY>;
  auto kern = fmha_fwd_stream_kernel<FMHA_TU_T, FMHA_TU_D, DROPT, TAIL, MANY>;
  constexpr int kLds = StreamCfg::lds_bytes(DROPT);
  static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                hipFuncAttributeMaxDynamicSharedMemorySize, kLds) == hipSuccess;
  if (!ready) return 2;
  a.nqt = (a.sq + StreamCfg::QT - 1) / StreamCfg::QT;
  const long long nblk = (long long)a.bh * a.nqt;
  if (nblk > 0x7fffffffLL) return 2;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(StreamCfg::NW * 64), kLds, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

// TAIL: rows that end within a 16-byte piece; MANY: more than two workgroups per compute unit
template <bool DROPT> int launch_stream(FwdArgs &a, const FwdVariant &v, hipStream_t s) {
  if constexpr (FMHA_TU_D == 64 && !DROPT)
    if (v.many) return a.sk & 7 ? launch_stream_as<false, true, true>(a, s) : launch_stream_as<false, false, true>(a, s);
  return a.sk & 7 ? launch_stream_as<DROPT, true, false>(a, s) : launch_stream_as<DROPT, false, false>(a, s);
}

// the save-intermediates operator for up to 512 keys in one launch (one wave per SIMD: the whole register file)
template <bool TAIL, int NTILE> int launch_stream_save_as(FwdArgs &a, hipStream_t s) {
  using StreamSaveCfg = fmha::StreamSaveCfg<FMHA_TU_D, NTILE>;
  auto kern = fmha_fwd_stream_save_kernel<FMHA_TU_T, FMHA_TU_D, TAIL, NTILE>;
  constexpr int kLds = StreamSaveCfg::lds_bytes(TAIL || FMHA_TU_D != 64);
  static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                hipFuncAttributeMaxDynamicSharedMemorySize, kLds) == hipSuccess;
  if (!ready) return 2;
  if (a.sk > StreamSaveCfg::SKMAX) return 1;
  a.nqt = (a.sq + StreamSaveCfg::QT - 1) / StreamSaveCfg::QT;
  const long long nblk = (long long)a.bh * a.nqt;
  if (nblk > 0x7fffffffLL) return 2;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(StreamSaveCfg::NW * 64), kLds, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}
int launch_stream_save(FwdArgs &a, hipStream_t s) {
  // Few tiles leave the registers for two waves per SIMD (us, one wave / two): three at head dim 64 BH 352 S 173 52.4 / 41.0, BH 800 S 192
  // 95.5 / 70.4, BH 96 S 144 13.9 / 12.7; one at 128 BH 504 S 40 16.3 / 10.7, BH 1500 S 64 51.5 / 34.7; two at 128 spill 50 registers
  // and pay where workgroups share compute units: BH 504 S 72 28.9 / 25.3, BH 1500 S 128 104.7 / 103.0, but BH 150 S 100 15.4 / 17.2.
  // (Four at 64 spill 45 and do not: BH 352 S 240 56.4 / 62.1.)
  constexpr int kFew = FMHA_TU_D == 64 ? 3 : 1, kMost = FMHA_TU_D == 64 ? 8 : 7;
  if (a.sk <= kFew * 64) return a.sk & 7 ? launch_stream_save_as<true, kFew>(a, s) : launch_stream_save_as<false, kFew>(a, s);
#if FMHA_TU_D == 128
  if (a.sk <= 128 && (long long)a.bh * ((a.sq + 127) / 128) > kCUs)
    return a.sk & 7 ? launch_stream_save_as<true, 2>(a, s) : launch_stream_save_as<false, 2>(a, s);
#endif
  return a.sk & 7 ? launch_stream_save_as<true, kMost>(a, s) : launch_stream_save_as<false, kMost>(a, s);
}
#endif

#if FMHA_TU_ROWS
// 32 queries a workgroup, 64 keys a wave
template <bool DROPT, bool SAVE, bool TAIL> int launch_cols_as(FwdArgs &a, hipStream_t s) {
  using ColsCfg = fmha::ColsCfg<FMHA_TU_D>;
  auto kern = fmha_fwd_cols_kernel<FMHA_TU_T, FMHA_TU_D, DROPT, SAVE, TAIL>;
  static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                ColsCfg::lds_bytes(ColsCfg::MAXW)) == hipSuccess;
  if (!ready) return 2;
  if (a.sk > ColsCfg::SKMAX || (DROPT && !a.drop_mask)) return 1;
  a.nqt = (a.sq + ColsCfg::QT - 1) / ColsCfg::QT;
  const long long nblk = (long long)a.bh * a.nqt;
  if (nblk > 0x7fffffffLL) return 2;
  const int nw = (a.sk + ColsCfg::BK - 1) / ColsCfg::BK;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(nw * 64), ColsCfg::lds_bytes(nw), s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}
template <bool DROPT, bool SAVE> int launch_cols(FwdArgs &a, hipStream_t s) {
  return a.sk & 7 ? launch_cols_as<DROPT, SAVE, true>(a, s) : launch_cols_as<DROPT, SAVE, false>(a, s);
}
#endif

#if FMHA_TU_D == 64
// a whole head's K and V resident in LDS: one persistent workgroup per compute unit
#ifndef FMHA_HEAD_QB
#define FMHA_HEAD_QB 2
#endif
template <int MASK, int DROP> int launch_head(FwdArgs &a, hipStream_t s) {
  using HC = HeadCfgT<FMHA_HEAD_QB>;
  auto kern = fmha_fwd_head_kernel<FMHA_TU_T, FMHA_HEAD_QB, MASK, DROP, kStrided>;
  static const int resident = [&]() -> int {
    if (hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                            HC::LDS_BYTES) != hipSuccess)
      return -1;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
      return -1;
    return cus;
  }();
  if (resident < 0) return 2;
  if (a.sk > HC::MAXK) return 1;
  a.nqt = (a.sq + HC::QT - 1) / HC::QT;
  long long nblk = (long long)a.bh * a.nqt;
  if (nblk > 0x7fffffffLL) return 2;
  if (nblk > resident) nblk = resident;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(HC::NT), HC::LDS_BYTES, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}
#endif

template <int QB, int MASK, bool CAUSAL> int by_drop(FwdArgs &a, int drop, hipStream_t s) {
  if (drop == 0) return launch<QB, MASK, CAUSAL, 0>(a, s);
  if (drop == 1) return launch<QB, MASK, CAUSAL, 1>(a, s);
  return 1;
}

template <int QB, int MASK> int by_causal(FwdArgs &a, const FwdVariant &v, hipStream_t s) {
  return v.causal ? by_drop<QB, MASK, true>(a, v.drop, s) : by_drop<QB, MASK, false>(a, v.drop, s);
}

#ifdef FMHA_DEV_MINIMAL
// development builds: only the variants the headline benchmark uses
template <int QB> int by_mask(FwdArgs &a, const FwdVariant &v, hipStream_t s) {
  if (v.causal || v.drop) return 1;
  if (v.mask == kMaskPerKey) return launch<1, kMaskPerKey, false, 0>(a, s);
  if (v.mask == kMaskNone) return launch<1, kMaskNone, false, 0>(a, s);
  return 1;
}
#else
template <int QB> int by_mask(FwdArgs &a, const FwdVariant &v, hipStream_t s) {
  if (v.mask == kMaskPerKey) return by_causal<QB, kMaskPerKey>(a, v, s);
#if FMHA_TU_D % 64 == 0
  if (v.mask == kMaskFull) return by_causal<QB, kMaskFull>(a, v, s);
#else // (full mask tensors: the next whole panel's kernels)
  if (v.mask == kMaskFull) return 1;
#endif
  return by_causal<QB, kMaskNone>(a, v, s);
}
#endif

} // namespace

#if FMHA_TU_D == 256
// Head dim 256, one wave per SIMD: the output accumulators alone take 128 registers per lane, all in all about 400 of the 512 that
// a wave then has.  The pipelined loop (132 KB of LDS) takes what needs no [.., sq, sk] tensor and has more than one key tile;
// us, pipelined / plain loop: BH 128 S 2048 631 / 911, causal 372 / 624; BH 72 S 1408 bf16 188 / 299; BH 300 S 512 causal with
// dropout 106 / 193; BH 512 S 256 padding mask 70 / 97; BH 512 S 100 24.2 / 33.5; BH 12 S 500 21.5 / 31.6; rows of 200 elements
// BH 64 S 2048 262 / 405.  One tile has nothing to overlap: BH 1900 S 31 60.4 / 58.8, 64 keys level.  Nor has a single round of
// workgroups much where tiles are few, or an odd number (the loop takes two at a time): there run-time row layouts, whose addresses
// the prologue works out, stay with the plain loop at three tiles (of 256 columns only causal ones) and, causal, masked or with
// key counts, at two and five (us, pipelined / plain: BH 64 rows of 200 elements S 65 13.4 / 12.1, S 160 causal under a padding mask 21.3 / 16.3,
// S 300 26.6 / 23.6, BH 400 S 160 ahead by 8 %; BH 64 S 160 packed causal 10 to 14 % behind; S 256 level to 10 % ahead).
namespace { // (per translation unit: the element type differs between units of the same name)
bool d256_plain_ahead(const FwdArgs &a, bool causal, bool mask) {
  if (!kStrided || (long long)a.bh * ((a.sq + 127) / 128) > kCUs) return false;
  const int tiles = (a.sk + 63) / 64;
  if (a.dcols == FMHA_TU_D) return causal && tiles == 3;
  return tiles == 3 || ((tiles == 2 || tiles == 5) && (causal || mask || a.kv_len));
}

template <int MASK, bool CAUSAL> int d256_by_drop(FwdArgs &a, int drop, hipStream_t s) {
  if constexpr (MASK != kMaskFull) {
    if (a.sk > 64 && drop < 2 && !d256_plain_ahead(a, CAUSAL, MASK == kMaskPerKey))
      return drop == 1 ? launch<1, MASK, CAUSAL, 1>(a, s) : launch<1, MASK, CAUSAL, 0>(a, s);
  }
  if (drop == 0) return launch<1, MASK, CAUSAL, 0, false>(a, s);
  if (drop == 1) return launch<1, MASK, CAUSAL, 1, false>(a, s);
  if (drop == 2 && !CAUSAL) return launch<1, MASK, false, 2, false>(a, s);
  return 1;
}
} // namespace

int FMHA_NAME(FMHA_TU_TNAME, FMHA_TU_D)(FwdArgs &a, const FwdVariant &v, hipStream_t s) {
  if (v.qb == 2 || v.short_keys || v.save_split || v.save_once || v.stream || v.head || (kStrided && v.drop == 2)) return 1;
  if (v.mask == kMaskPerKey)
    return v.causal ? d256_by_drop<kMaskPerKey, true>(a, v.drop, s) : d256_by_drop<kMaskPerKey, false>(a, v.drop, s);
  if (v.mask == kMaskFull)
    return v.causal ? d256_by_drop<kMaskFull, true>(a, v.drop, s) : d256_by_drop<kMaskFull, false>(a, v.drop, s);
  return v.causal ? d256_by_drop<kMaskNone, true>(a, v.drop, s) : d256_by_drop<kMaskNone, false>(a, v.drop, s);
}
#else
int FMHA_NAME(FMHA_TU_TNAME, FMHA_TU_D)(FwdArgs &a, const FwdVariant &v, hipStream_t s) {
#if defined(FMHA_DEV_MINIMAL) || FMHA_TU_STRIDED
  if (v.drop == 2 || v.qb == 2) return 1; // folded layout only
#endif
#if FMHA_TU_D == 64
  if (v.mid) {
    if (v.drop == 2 || v.mask == kMaskFull) return 1;
    if (v.mid == 4) return v.mask == kMaskPerKey ? launch_mid<4, kMaskPerKey>(a, v, s) : launch_mid<4, kMaskNone>(a, v, s);
    return v.mask == kMaskPerKey ? launch_mid<8, kMaskPerKey>(a, v, s) : launch_mid<8, kMaskNone>(a, v, s);
  }
#endif
#if FMHA_TU_D == 64 && FMHA_TU_STRIDED
  if (v.head && !v.short_keys) { // run-time row layouts: the whole-head kernel
    if (v.causal || v.drop == 2 || v.mask == kMaskFull) return 1;
    if (v.mask == kMaskPerKey) return v.drop ? launch_head<kMaskPerKey, 1>(a, s) : launch_head<kMaskPerKey, 0>(a, s);
    return v.drop ? launch_head<kMaskNone, 1>(a, s) : launch_head<kMaskNone, 0>(a, s);
  }
  if (v.short_keys) { // run-time row layouts: the one-pass kernel's builds without a full mask tensor
    if (v.causal || v.mask == kMaskFull || v.drop == 2 || v.saving) return 1;
    if (v.mask == kMaskPerKey)
      return v.drop == 1 ? launch_short<kMaskPerKey, 1, false>(a, s) : launch_short<kMaskPerKey, 0, false>(a, s);
    return v.drop == 1 ? launch_short<kMaskNone, 1, false>(a, s) : launch_short<kMaskNone, 0, false>(a, s);
  }
#endif
#if FMHA_TU_SHORT
  if (v.short_keys) {
    if (v.causal) return 1;
    if (v.mask == kMaskFull) {
      if (v.drop == 1) return 1;
      if (v.saving) return launch_short<kMaskFull, 2, true>(a, s);
      return v.drop == 2 ? launch_short<kMaskFull, 2, false>(a, s) : launch_short<kMaskFull, 0, false>(a, s);
    }
    if (v.drop == 2 || v.saving) return 1;
    if (v.mask == kMaskPerKey)
      return v.drop == 1 ? launch_short<kMaskPerKey, 1, false>(a, s) : launch_short<kMaskPerKey, 0, false>(a, s);
    return v.drop == 1 ? launch_short<kMaskNone, 1, false>(a, s) : launch_short<kMaskNone, 0, false>(a, s);
  }
  if (v.head) {
    if (v.causal || v.drop == 2 || v.mask == kMaskFull) return 1;
    if (v.mask == kMaskPerKey) return v.drop ? launch_head<kMaskPerKey, 1>(a, s) : launch_head<kMaskPerKey, 0>(a, s);
    return v.drop ? launch_head<kMaskNone, 1>(a, s) : launch_head<kMaskNone, 0>(a, s);
  }
#else
  if (v.short_keys || v.head) return 1;
#endif
#if FMHA_TU_ROWS
  if (v.cols) return v.drop != 2 ? launch_cols<false, false>(a, s) : a.save_softmax || a.save_dropout ? launch_cols<true, true>(a, s) : launch_cols<true, false>(a, s);
  if (v.save_once) return launch_stream_save(a, s);
  if (v.save_split) { // forward with LSE, then the saved outputs from that LSE
    const int rc = v.stream ? launch_stream<true>(a, v, s) : launch<1, kMaskFull, false, 2, FMHA_TU_D == 64>(a, s);
    return rc ? rc : launch_save(a, s);
  }
  if (v.stream) return v.drop == 2 ? launch_stream<true>(a, v, s) : launch_stream<false>(a, v, s);
#else
  if (v.save_split || v.save_once || v.stream || v.cols) return 1;
#endif
#if !FMHA_TU_STRIDED
  if (v.drop == 2) { // tensor dropout / save-intermediates: the legacy ops' shape class
    if (v.causal) return 1;
#if FMHA_TU_D == 64
    if (!v.saving) { // dropout tensor alone: pipelined kernel
      if (v.mask == kMaskPerKey) return launch<1, kMaskPerKey, false, 2, true>(a, s);
      if (v.mask == kMaskFull) return launch<1, kMaskFull, false, 2, true>(a, s);
      return launch<1, kMaskNone, false, 2, true>(a, s);
    }
#endif
    if (v.mask == kMaskPerKey) return launch<1, kMaskPerKey, false, 2>(a, s);
    if (v.mask == kMaskFull) return launch<1, kMaskFull, false, 2>(a, s);
    return launch<1, kMaskNone, false, 2>(a, s);
  }
#endif
#if FMHA_TU_D == 64
  // two query blocks per wave: only where their accumulators fit the register file and only
  // for the variants the host ever selects them for
  if (v.qb == 2) {
    if (v.causal || v.drop != 0 || v.mask == kMaskFull) return 1;
    return v.mask == kMaskPerKey ? launch<2, kMaskPerKey, false, 0>(a, s) : launch<2, kMaskNone, false, 0>(a, s);
  }
#endif
  return by_mask<1>(a, v, s);
}
#endif

} // namespace fmha
