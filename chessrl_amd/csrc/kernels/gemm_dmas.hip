// Instances of the 64x64 and 32x32 GEMMs of gemm_dmas_kernel.hpp, in a translation unit of their own.
#include "gemm_dmas_kernel.hpp"

namespace crl {

template <typename S>
static hipError_t launch_small(const GemmArgs& a, int in_dt, int out_dt, hipStream_t st) {
  if (in_dt == DT_FP8) {
    switch (out_dt) {
      case DT_BF16: return launch_dmas<S, DT_FP8, DT_BF16>(a, st);
      case DT_F16: return launch_dmas<S, DT_FP8, DT_F16>(a, st);
      case DT_FP8: return launch_dmas<S, DT_FP8, DT_FP8>(a, st);
    }
  }
  if (in_dt == DT_BF16 && out_dt == DT_BF16) return launch_dmas<S, DT_BF16, DT_BF16>(a, st);
  if (in_dt == DT_F16 && out_dt == DT_F16) return launch_dmas<S, DT_F16, DT_F16>(a, st);
  if (in_dt == DT_BF16 && out_dt == DT_F32) return launch_dmas<S, DT_BF16, DT_F32>(a, st);
  return hipErrorInvalidValue;
}

// tile_size: 64 (eight stages) or 32 (sixteen); the operand types are those of gemm_dmam_has. With k_parallel set the 32x32 tile spreads K over four waves.
hipError_t launch_gemm_dmas(const GemmArgs& a, int in_dt, int out_dt, hipStream_t st, int tile_size) {
  if (tile_size == 64) return launch_small<DmasCfg<64>>(a, in_dt, out_dt, st);
  return a.k_parallel ? launch_small<DmasCfg<32, 4>>(a, in_dt, out_dt, st) : launch_small<DmasCfg<32>>(a, in_dt, out_dt, st);
}

// K in 4 n equal shares (SLICED), 16-bit operands: the raw fp32 sums of share y in rows y M .. of C.
hipError_t launch_gemm_dmas_sliced(const GemmArgs& a, int in_dt, hipStream_t st, int tile_size, int shares) {
  if (in_dt == DT_BF16)
    return tile_size == 64 ? launch_dmas<DmasCfg<64>, DT_BF16, DT_F32, 0, 1>(a, st, shares) : launch_dmas<DmasCfg<32>, DT_BF16, DT_F32, 0, 1>(a, st, shares);
  if (in_dt == DT_F16)
    return tile_size == 64 ? launch_dmas<DmasCfg<64>, DT_F16, DT_F32, 0, 1>(a, st, shares) : launch_dmas<DmasCfg<32>, DT_F16, DT_F32, 0, 1>(a, st, shares);
  return hipErrorInvalidValue;
}

}  // namespace crl
