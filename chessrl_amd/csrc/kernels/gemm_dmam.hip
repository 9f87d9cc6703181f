// Instances of the 128x128 GEMM with loading and multiplying waves (gemm_dmam_kernel.hpp), in a translation unit of their own.
#include "gemm_dmam_kernel.hpp"

namespace crl {

// false: no instance for this combination (the caller keeps the register-staged kernel).
bool gemm_dmam_has(int in_dt, int out_dt) {
  if (in_dt == DT_FP8) return out_dt == DT_BF16 || out_dt == DT_F16 || out_dt == DT_FP8;
  if (in_dt == DT_BF16 && out_dt == DT_F32) return true;   // (an fp32 residual stream, fp32 logits)
  return in_dt == out_dt && (in_dt == DT_BF16 || in_dt == DT_F16);
}

// Tiles of 128x192: outputs of the operands' type, or bf16 of e4m3 operands, without a residual (its registers spill beside twelve multiplying waves: BT4-class bf16 at 150 positions
// 3661 -> 3903 us with it), rows of W no further apart than 192 of them can be addressed (128x128 tiles reach half as far again: they serve what lies between).
bool gemm_dmam_wide_can(const GemmArgs& a, int in_dt, int out_dt) {
  if (a.res_stats || !dmam_reaches(a, in_dt == DT_FP8 ? 1 : 2, 192) || (long)((a.M + 127) / 128) * ((a.N + 191) / 192) >= 65536 || dmaf_epilogue(a, in_dt, out_dt, 192) != DMAF_PLAIN) return false;
  if (in_dt == DT_FP8) return (out_dt == DT_FP8 && a.act == ACT_MISH) || (out_dt == DT_BF16 && a.act == ACT_NONE);
  return in_dt == out_dt && (in_dt == DT_BF16 || in_dt == DT_F16) && (a.act == ACT_NONE || a.act == ACT_MISH || (a.act == ACT_GELU && in_dt == DT_BF16));
}

hipError_t launch_gemm_dmam_wide(const GemmArgs& a, int in_dt, int out_dt, int cus, hipStream_t st) {
  if (!gemm_dmam_wide_can(a, in_dt, out_dt)) return hipErrorInvalidValue;
#define WIDE(IN, OUT, ACT) launch_dmam<IN, OUT, DMAF_PLAIN, ACT, 192>(a, cus, st)
  if (in_dt == DT_FP8) return out_dt == DT_FP8 ? WIDE(DT_FP8, DT_FP8, ACT_MISH) : WIDE(DT_FP8, DT_BF16, ACT_NONE);
  if (in_dt == DT_F16) return a.act == ACT_MISH ? WIDE(DT_F16, DT_F16, ACT_MISH) : WIDE(DT_F16, DT_F16, ACT_NONE);
  return a.act == ACT_GELU ? WIDE(DT_BF16, DT_BF16, ACT_GELU) : a.act == ACT_MISH ? WIDE(DT_BF16, DT_BF16, ACT_MISH) : WIDE(DT_BF16, DT_BF16, ACT_NONE);
#undef WIDE
}

hipError_t launch_gemm_dmam(const GemmArgs& a, int in_dt, int out_dt, int cus, hipStream_t st) {
  // (the conditions of the 256x256 tile, and a column split on this tile's boundary)
  const int epi = dmaf_epilogue(a, in_dt, out_dt, DmamCfg::BN);
#define DMAM(IN, OUT, EPI, ACT) launch_dmam<IN, OUT, EPI, ACT>(a, cus, st)
  if (a.res_stats) {
    if (in_dt != DT_FP8 || out_dt != DT_BF16 || !a.res || a.res_dtype != DT_BF16 || !a.res_gamma || a.res_rows > 0 || a.alpha == 0.f) return hipErrorInvalidValue;
    return epi == DMAF_RESNORM ? DMAM(DT_FP8, DT_BF16, DMAF_RESNORM, ACT_NONE) : DMAM(DT_FP8, DT_BF16, DMAF_GENERAL_NORM, ACT_NONE);
  }
  if (in_dt == DT_FP8) {
    switch (out_dt) {
      case DT_BF16:
        if (epi == DMAF_PLAIN && a.act == ACT_NONE) return DMAM(DT_FP8, DT_BF16, DMAF_PLAIN, ACT_NONE);
        return epi == DMAF_RES16 ? DMAM(DT_FP8, DT_BF16, DMAF_RES16, ACT_NONE) : DMAM(DT_FP8, DT_BF16, DMAF_GENERAL, ACT_NONE);
      case DT_F16: return DMAM(DT_FP8, DT_F16, DMAF_GENERAL, ACT_NONE);
      case DT_FP8:
        if (epi == DMAF_PLAIN) return a.act == ACT_MISH ? DMAM(DT_FP8, DT_FP8, DMAF_PLAIN, ACT_MISH) : DMAM(DT_FP8, DT_FP8, DMAF_PLAIN, ACT_GELU);
        return DMAM(DT_FP8, DT_FP8, DMAF_GENERAL, ACT_NONE);
    }
  }
  if (in_dt == DT_BF16 && out_dt == DT_BF16) {
    if (epi == DMAF_PLAIN)
      return a.act == ACT_GELU ? DMAM(DT_BF16, DT_BF16, DMAF_PLAIN, ACT_GELU) : a.act == ACT_MISH ? DMAM(DT_BF16, DT_BF16, DMAF_PLAIN, ACT_MISH) : DMAM(DT_BF16, DT_BF16, DMAF_PLAIN, ACT_NONE);
    if (epi == DMAF_RES16) return a.act == ACT_GELU ? DMAM(DT_BF16, DT_BF16, DMAF_RES16, ACT_GELU) : DMAM(DT_BF16, DT_BF16, DMAF_RES16, ACT_NONE);
    return DMAM(DT_BF16, DT_BF16, DMAF_GENERAL, ACT_NONE);
  }
  if (in_dt == DT_F16 && out_dt == DT_F16) {
    if (epi == DMAF_PLAIN) return a.act == ACT_MISH ? DMAM(DT_F16, DT_F16, DMAF_PLAIN, ACT_MISH) : DMAM(DT_F16, DT_F16, DMAF_PLAIN, ACT_NONE);
    return epi == DMAF_RES16 ? DMAM(DT_F16, DT_F16, DMAF_RES16, ACT_NONE) : DMAM(DT_F16, DT_F16, DMAF_GENERAL, ACT_NONE);
  }
  if (in_dt == DT_BF16 && out_dt == DT_F32 && epi == DMAF_PLAIN) return DMAM(DT_BF16, DT_F32, DMAF_PLAIN, ACT_NONE);
  if (in_dt == DT_BF16 && out_dt == DT_F32) return epi == DMAF_RES32 ? DMAM(DT_BF16, DT_F32, DMAF_RES32, ACT_NONE) : DMAM(DT_BF16, DT_F32, DMAF_GENERAL, ACT_NONE);
#undef DMAM
  return hipErrorInvalidValue;
}

}  // namespace crl
