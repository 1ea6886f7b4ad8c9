// The forward whose waves share 32 queries (fmha_fwd_few.h) for one (element type, head dim, row layout kind) triple, chosen with
// -DFMHA_TU_BF16={0,1} -DFMHA_TU_D={32,64,96,128,256} -DFMHA_TU_STRIDED={0,1}, and its dispatcher.
// The rules (few_waves, few_chunk) reach every build: four and eight waves each mask, causal or not, with and without dropout (training forwards), at head
// dim 256 four only; one wave the same, at head dim 64 causal launches, dropout on many heads and query rows too far apart for the one-pass
// kernel; pieces without causal mask and dropout from run-time row layouts (folded tensors are one).
#include "fmha_launch.h"

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
#define FMHA_NAME(t, d) FMHA_CAT3(fwd_few_launch_, t, d)
#include "fmha_fwd_few.h"

namespace fmha {
namespace {

template <int NW, int MASK, bool CAUSAL, int DROP, bool PIECES = false> int launch_as(FwdArgs &a, hipStream_t s) {
  using C = FewCfg<FMHA_TU_D, NW>;
  auto kern = fmha_fwd_few_kernel<FMHA_TU_T, FMHA_TU_D, NW, MASK, CAUSAL, DROP, FMHA_TU_STRIDED != 0, PIECES>;
  static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                C::LDS_BYTES) == hipSuccess;
  if (!ready) return 2;
  a.nqt = (a.sq + C::QT - 1) / C::QT;
  const long long nblk = (long long)a.bh * a.nqt;
  if (nblk > 0x7fffffffLL) return 2;
  hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(C::NT), C::LDS_BYTES, s, a);
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

template <int MASK, bool CAUSAL, int DROP> int launch(FwdArgs &a, int nw, hipStream_t s) {
#if FMHA_TU_D != 256
  if (nw == 8) return launch_as<8, MASK, CAUSAL, DROP>(a, s);
#endif
  if (nw == 1) return launch_as<1, MASK, CAUSAL, DROP>(a, s);
  return launch_as<4, MASK, CAUSAL, DROP>(a, s);
}

template <int MASK> int by_variant(FwdArgs &a, const FwdVariant &v, hipStream_t s) {
  if (v.causal) return v.drop ? launch<MASK, true, 1>(a, v.few, s) : launch<MASK, true, 0>(a, v.few, s);
  return v.drop ? launch<MASK, false, 1>(a, v.few, s) : launch<MASK, false, 0>(a, v.few, s);
}

} // namespace

int FMHA_NAME(FMHA_TU_TNAME, FMHA_TU_D)(FwdArgs &a, const FwdVariant &v, hipStream_t s) {
  if (v.mask == kMaskFull || v.drop == 2) return 1;
  if (a.sk_whole != 0) {
#if FMHA_TU_STRIDED
    if (!v.causal && !v.drop) return v.mask == kMaskPerKey ? launch_as<4, kMaskPerKey, false, 0, true>(a, s) : launch_as<4, kMaskNone, false, 0, true>(a, s);
#endif
    return 1;
  }
  return v.mask == kMaskPerKey ? by_variant<kMaskPerKey>(a, v, s) : by_variant<kMaskNone>(a, v, s);
}

} // namespace fmha
