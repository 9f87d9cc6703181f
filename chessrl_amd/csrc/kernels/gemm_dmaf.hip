// Instances of the 256x256 GEMM whose waves take turns (gemm_dmaf_kernel.hpp), in a translation unit of their own.
#include "gemm_dmaf_kernel.hpp"

namespace crl {

// false: no instance for this combination (the caller falls back to gemm_dma_kernel.hpp).
bool gemm_dmaf_has(int in_dt, int out_dt, bool res_norm) {
  if (res_norm) return in_dt == DT_FP8 && out_dt == DT_BF16;
  if (in_dt == DT_FP8) return true;
  if (in_dt == DT_BF16 && out_dt == DT_F32) return true;   // (an fp32 residual stream, fp32 logits)
  return in_dt == out_dt && (in_dt == DT_BF16 || in_dt == DT_F16);
}

hipError_t launch_gemm_dmaf(const GemmArgs& a, int in_dt, int out_dt, int cus, hipStream_t st) {
  const int epi = dmaf_epilogue(a, in_dt, out_dt);
  if (a.res_stats) {
    if (in_dt != DT_FP8 || out_dt != DT_BF16 || !a.res || a.res_dtype != DT_BF16 || !a.res_gamma || a.res_rows > 0 || a.alpha == 0.f || (a.M & 1))
      return hipErrorInvalidValue;
    return epi == DMAF_RESNORM ? launch_dmaf<DT_FP8, DT_BF16, DMAF_RESNORM>(a, cus, st) : launch_dmaf<DT_FP8, DT_BF16, DMAF_GENERAL_NORM>(a, cus, st);
  }
#define DMAF(IN, OUT, EPI, ACT) launch_dmaf<IN, OUT, EPI, ACT>(a, cus, st)
  if (in_dt == DT_FP8) {
    switch (out_dt) {
      case DT_BF16:
        if (epi == DMAF_PLAIN) return a.act == ACT_MISH ? DMAF(DT_FP8, DT_BF16, DMAF_PLAIN, ACT_MISH) : DMAF(DT_FP8, DT_BF16, DMAF_PLAIN, ACT_NONE);
        return epi == DMAF_RES16 ? DMAF(DT_FP8, DT_BF16, DMAF_RES16, ACT_NONE) : DMAF(DT_FP8, DT_BF16, DMAF_GENERAL, ACT_NONE);
      case DT_F16: return DMAF(DT_FP8, DT_F16, DMAF_GENERAL, ACT_NONE);
      case DT_F32: if (epi == DMAF_PLAIN) return DMAF(DT_FP8, DT_F32, DMAF_PLAIN, ACT_NONE);
        return epi == DMAF_RES32 ? DMAF(DT_FP8, DT_F32, DMAF_RES32, ACT_NONE) : DMAF(DT_FP8, DT_F32, DMAF_GENERAL, ACT_NONE);
      case DT_FP8:
        if (epi == DMAF_PLAIN) return a.act == ACT_MISH ? DMAF(DT_FP8, DT_FP8, DMAF_PLAIN, ACT_MISH) : DMAF(DT_FP8, DT_FP8, DMAF_PLAIN, ACT_GELU);
        return DMAF(DT_FP8, DT_FP8, DMAF_GENERAL, ACT_NONE);
    }
  }
  if (in_dt == DT_BF16 && out_dt == DT_BF16) {
    if (epi == DMAF_PLAIN)
      return a.act == ACT_GELU ? DMAF(DT_BF16, DT_BF16, DMAF_PLAIN, ACT_GELU) : a.act == ACT_MISH ? DMAF(DT_BF16, DT_BF16, DMAF_PLAIN, ACT_MISH) : DMAF(DT_BF16, DT_BF16, DMAF_PLAIN, ACT_NONE);
    if (epi == DMAF_RES16) return a.act == ACT_GELU ? DMAF(DT_BF16, DT_BF16, DMAF_RES16, ACT_GELU) : DMAF(DT_BF16, DT_BF16, DMAF_RES16, ACT_NONE);
    return DMAF(DT_BF16, DT_BF16, DMAF_GENERAL, ACT_NONE);
  }
  if (in_dt == DT_F16 && out_dt == DT_F16) {
    if (epi == DMAF_PLAIN) return a.act == ACT_MISH ? DMAF(DT_F16, DT_F16, DMAF_PLAIN, ACT_MISH) : DMAF(DT_F16, DT_F16, DMAF_PLAIN, ACT_NONE);
    return epi == DMAF_RES16 ? DMAF(DT_F16, DT_F16, DMAF_RES16, ACT_NONE) : DMAF(DT_F16, DT_F16, DMAF_GENERAL, ACT_NONE);
  }
  if (in_dt == DT_BF16 && out_dt == DT_F32 && epi == DMAF_PLAIN) return DMAF(DT_BF16, DT_F32, DMAF_PLAIN, ACT_NONE);
  if (in_dt == DT_BF16 && out_dt == DT_F32) return epi == DMAF_RES32 ? DMAF(DT_BF16, DT_F32, DMAF_RES32, ACT_NONE) : DMAF(DT_BF16, DT_F32, DMAF_GENERAL, ACT_NONE);
#undef DMAF
  return hipErrorInvalidValue;
}

}  // namespace crl
