// Instances of the 64x64 and 32x32 GEMMs of gemm_dmas_kernel.hpp, in a translation unit of their own.
#include "gemm_dmas_kernel.hpp"

namespace crl {

// (S8: the form of e4m3 operands)
template <typename S, typename S8>
static hipError_t launch_small(const GemmArgs& a, int in_dt, int out_dt, hipStream_t st, SmallTile t) {
#define SMALL(CFG, IN, OUT) launch_dmas<CFG, IN, OUT>(a, st, 1, t.bm, t.bn)
  if (in_dt == DT_FP8) {
    switch (out_dt) {
      case DT_BF16: return SMALL(S8, DT_FP8, DT_BF16);
      case DT_F16: return SMALL(S8, DT_FP8, DT_F16);
      case DT_FP8: return SMALL(S8, DT_FP8, DT_FP8);
    }
  }
  if (in_dt == DT_BF16 && out_dt == DT_BF16) return SMALL(S, DT_BF16, DT_BF16);
  if (in_dt == DT_F16 && out_dt == DT_F16) return SMALL(S, DT_F16, DT_F16);
  if (in_dt == DT_BF16 && out_dt == DT_F32) return SMALL(S, DT_BF16, DT_F32);
#undef SMALL
  return hipErrorInvalidValue;
}

// tile_size: 64 (eight stages) or 32 (sixteen, and tiles of fewer rows or columns where there are CUs for them); the operand types are those of gemm_dmam_has.
hipError_t launch_gemm_dmas(const GemmArgs& a, int in_dt, int out_dt, hipStream_t st, int tile_size) {
  if (tile_size == 64) return launch_small<DmasCfg<64>, DmasCfg<64>>(a, in_dt, out_dt, st, {64, 64});
  const SmallTile t = small_tile(a.M, a.N, device_cus());
  if (t.bm <= 16 && t.bn <= 16)
    return t.bm + t.bn <= 16 ? launch_small<DmasCfg<32, 1, 14, 1>, DmasCfg<32, 0, 14>>(a, in_dt, out_dt, st, t) : launch_small<DmasCfg<32, 1, 8, 1>, DmasCfg<32, 0, 14>>(a, in_dt, out_dt, st, t);
  if (t.bm + t.bn <= 40) return launch_small<DmasCfg<32, 1, 14>, DmasCfg<32, 0, 14>>(a, in_dt, out_dt, st, t);
  return launch_small<DmasCfg<32, 1, 8>, DmasCfg<32>>(a, in_dt, out_dt, st, t);
}

// K in 4 n equal shares (SLICED), 16-bit operands: the raw fp32 sums of share y in rows y M .. of C.
hipError_t launch_gemm_dmas_sliced(const GemmArgs& a, int in_dt, hipStream_t st, int tile_size, int shares) {
  if (in_dt == DT_BF16)
    return tile_size == 64 ? launch_dmas<DmasCfg<64>, DT_BF16, DT_F32, 0, 1>(a, st, shares) : launch_dmas<DmasCfg<32, 1>, DT_BF16, DT_F32, 0, 1>(a, st, shares);
  if (in_dt == DT_F16)
    return tile_size == 64 ? launch_dmas<DmasCfg<64>, DT_F16, DT_F32, 0, 1>(a, st, shares) : launch_dmas<DmasCfg<32, 1>, DT_F16, DT_F32, 0, 1>(a, st, shares);
  return hipErrorInvalidValue;
}

}  // namespace crl
