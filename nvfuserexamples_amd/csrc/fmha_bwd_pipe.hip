// Instantiates the software-pipelined backward kernels for one (element type, head dim, row layout kind) triple, chosen
// with -DFMHA_TU_BF16={0,1} -DFMHA_TU_D={32,64,96,128,256} -DFMHA_TU_STRIDED={0,1}, and exports their launcher.
#include "fmha_launch.h"
#include "fmha_bwd_persist.h"
#ifndef FMHA_TU_STRIDED
#define FMHA_TU_STRIDED 0
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
#define FMHA_PIPE_NAME(t, d) FMHA_CAT3(bwd_pipe_launch_, t, d)

namespace fmha {
namespace {

constexpr int kNW = 4;
constexpr bool kStrided = FMHA_TU_STRIDED != 0;
using Cfg = BwdPipeCfg<FMHA_TU_D>;

#if FMHA_TU_D == 128
// From how many half rounds of workgroups on the persistent dK / dV kernel is taken.  A single round has nothing to run ahead of, and
// the plain kernel starts sooner: 16 heads, S 1024 causal 33.6 us persistent, 31.7 plain.  From one and a half on it is ahead for whole
// rows; not yet where a tile's own work is long beside what is hidden (dropout decisions on long heads), or where rows are shorter
// than the kernel's and there is less to hide.  Backward, us, persistent / plain, bf16: BH 96 S 512 96 columns with dropout 81.9 /
// 76.9, BH 684 S 384 305 / 317; BH 224 S 160 46.4 / 43.3; BH 512 S 128 51.1 / 52.4; BH 56 S 1536 128 columns 295 / 285; BH 320 S 256
// 86.6 / 88.6; BH 224 S 192 96 columns without dropout 43.5 / 42.1.  Over 1536 launches (128 to 2048 rows, 1.5 to 8 rounds) 25 are
// more than 2 % behind the plain kernel, with one and a half rounds for all 215.
int persist_half_rounds(const BwdArgs &a, bool causal, bool drop) {
  const bool narrow = a.dcols < FMHA_TU_D;
  if (!drop) return narrow ? 4 : 3;
  if (causal) return a.sq > 1024 ? (narrow ? 16 : 6) : narrow && a.sq < 160 ? 6 : 3;
  return a.sq > 512 ? (narrow ? 16 : 6) : a.sq >= 160 ? (narrow ? 8 : 4) : narrow ? 4 : 3;
}
#endif

template <int MASK, bool CAUSAL, int DROP> int launch(const BwdArgs &a, bool dkdv, long long nblk, hipStream_t s) {
  if (nblk > 0x7fffffffLL) return 2;
#if FMHA_TU_D == 96 || FMHA_TU_D == 256 // (dQ only)
  if (dkdv) return 1;
#else
  if (dkdv) {
#if FMHA_TU_D == 128
    if constexpr (MASK == kMaskNone) {
      // From some rounds of workgroups on (persist_half_rounds): persistent ones, as many as the device keeps resident (by the
      // current device at the first call).
      using PCfg = BwdPersistCfg<FMHA_TU_D>;
      static_assert(PCfg::MAX_LDS <= 160 * 1024, "does not fit the LDS of a compute unit");
      auto persist = fmha_bwd_dkdv_persist_kernel<FMHA_TU_T, FMHA_TU_D, kNW, CAUSAL, DROP, kStrided>;
      static const int resident = [&]() -> int {
        const void *f = reinterpret_cast<const void *>(persist);
        int dev = 0, cus = 0, per_cu = 0;
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, PCfg::MAX_LDS) != hipSuccess || hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, kNW * 64, PCfg::MAX_LDS) != hipSuccess || cus < 1 || per_cu < 1)
          return -1;
        return cus * per_cu;
      }();
      if (resident < 0) return 2;
      if (2 * nblk >= persist_half_rounds(a, CAUSAL, DROP != 0) * (long long)resident && !a.kv_len) {
        hipLaunchKernelGGL(persist, dim3((unsigned)resident), dim3(kNW * 64), PCfg::lds_bytes(DROP, a.sq), s, a);
        return hipGetLastError() == hipSuccess ? 0 : 2;
      }
    }
    // Short causal heads that the persistent kernel does not take: phase by phase (backward, us, this kernel / that one: S 128
    // BH 350 43.4 / 40.6; under a padding mask BH 512 S 128 54.2 / 51.2, S 176 95.1 / 91.3, S 160 level; S 200 103.4 / 105.5).
    if (CAUSAL && a.sq < 192) return kBwdNotHere;
#endif
    auto kern = fmha_bwd_dkdv_pipe_kernel<FMHA_TU_T, FMHA_TU_D, kNW, MASK, CAUSAL, DROP, kStrided>;
    static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                  Cfg::dkdv_lds_bytes(DROP, Cfg::QSEG)) == hipSuccess;
    if (!ready) return 2;
    hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(kNW * 64), Cfg::dkdv_lds_bytes(DROP, a.sq), s, a);
  } else
#endif
  {
    static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void *>(fmha_bwd_dq_pipe_kernel<FMHA_TU_T, FMHA_TU_D, kNW, MASK, CAUSAL, DROP, kStrided>),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::dq_lds_bytes(MASK, Cfg::MSEG)) == hipSuccess;
    if (!ready) return 2;
    hipLaunchKernelGGL((fmha_bwd_dq_pipe_kernel<FMHA_TU_T, FMHA_TU_D, kNW, MASK, CAUSAL, DROP, kStrided>), dim3((unsigned)nblk),
                       dim3(kNW * 64), Cfg::dq_lds_bytes(MASK, a.sk), s, a);
  }
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

template <int MASK> int by_mask(const BwdArgs &a, const BwdVariant &v, bool dkdv, long long nblk, hipStream_t s) {
  if (v.causal) return v.drop ? launch<MASK, true, 1>(a, dkdv, nblk, s) : launch<MASK, true, 0>(a, dkdv, nblk, s);
  return v.drop ? launch<MASK, false, 1>(a, dkdv, nblk, s) : launch<MASK, false, 0>(a, dkdv, nblk, s);
}

} // namespace

int FMHA_PIPE_NAME(FMHA_TU_TNAME, FMHA_TU_D)(const BwdArgs &a, const BwdVariant &v, bool dkdv, long long nblk, hipStream_t s) {
  if (v.mask == kMaskPerKey) return by_mask<kMaskPerKey>(a, v, dkdv, nblk, s);
  if (v.mask == kMaskNone) return by_mask<kMaskNone>(a, v, dkdv, nblk, s);
  return 1;
}

} // namespace fmha
