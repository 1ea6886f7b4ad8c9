// Instantiates the one-pass backward for short heads for one (element type, row layout kind) pair, chosen with
// -DFMHA_TU_BF16={0,1} -DFMHA_TU_STRIDED={0,1}, and exports its launcher.
#include "fmha_launch.h"
#include "fmha_bwd_one.h"
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
#define FMHA_CAT(a, b) a##b##_d64_strided
#else
#define FMHA_CAT(a, b) a##b##_d64
#endif
#define FMHA_ONE_NAME(t) FMHA_CAT(bwd_one_launch_, t)

namespace fmha {
namespace {

constexpr bool kStrided = FMHA_TU_STRIDED != 0;

template <int DROP, bool CAUSAL> int launch(const BwdArgs &a, hipStream_t s) {
  using Cfg = BwdOneCfg;
  auto kern = fmha_bwd_one_kernel<FMHA_TU_T, DROP, CAUSAL, kStrided>;
  // as many workgroups as the device keeps resident (by the current device at the first call)
  static const int resident = [&]() -> int {
    const void *f = reinterpret_cast<const void *>(kern);
    int dev = 0, cus = 0, per_cu = 0;
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES) != hipSuccess || hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, Cfg::NW * 64, Cfg::LDS_BYTES) != hipSuccess || cus < 1 || per_cu < 1)
      return -1;
    return cus * per_cu;
  }();
  if (resident < 0) return 2;
  if (a.bh <= resident) return kBwdNotHere;
  hipLaunchKernelGGL(kern, dim3((unsigned)resident), dim3(Cfg::NW * 64), Cfg::LDS_BYTES, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

} // namespace

int FMHA_ONE_NAME(FMHA_TU_TNAME)(const BwdArgs &a, const BwdVariant &v, hipStream_t s) {
  if (a.sq > BwdOneCfg::KEYS || a.sk > BwdOneCfg::KEYS) return 1;
  // The copies number bytes within a head in 32 bits, also those of the rows that fill up the last tile (at least four tiles).
  const int64_t rows = a.sq > 96 ? (a.sq + 31) / 32 * 32 : 128;
  for (const RowMap *m : {&a.mq, &a.mo, &a.mdo})
    if (kStrided && rows * m->ss >= (1ll << 31)) return kBwdNotHere;
  if (v.causal) return v.drop ? launch<1, true>(a, s) : launch<0, true>(a, s);
  return v.drop ? launch<1, false>(a, s) : launch<0, false>(a, s);
}

} // namespace fmha
