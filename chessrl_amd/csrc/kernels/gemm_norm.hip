// Launches of the norm-and-product kernel (gemm_norm_kernel.hpp).
#include "gemm_norm_kernel.hpp"

namespace crl {

template <int IN_DT, int BN, int KP>
static hipError_t launch_norm(const NormGemmArgs& a, hipStream_t st) {
  static std::atomic<bool> attr_set[16] = {};
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2;
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto kern = gemm_norm_kernel<IN_DT, BN, KP>;
  if (dev < 0 || dev >= 16 || !attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 16) attr_set[dev] = true;
  }
  NormGemmKArgs k;
  k.a = a;
  k.nslab = a.K * ESZ / 128;
  k.tiles_m = (a.M + 31) / 32;
  k.m_tm = dmaf_magic(k.tiles_m);
  const int tiles = k.tiles_m * ((a.N + BN - 1) / BN);
  if (tiles >= 65536) return hipErrorInvalidValue;
  k.per_xcd = tiles >> 3;
  const int lds = std::max((32 + BN) * a.K * ESZ + 9216, 8 * 4096);   // operands, gain and offset, the spare kilobyte; the patches of the sums
  hipLaunchKernelGGL(kern, dim3(tiles), dim3(1024), lds, st, k);
  return hipGetLastError();
}

// Tile width for this call: 64 columns, 32, or 0 where the kernel does not serve it. Every tile has to have a CU of its own; of
// the two widths the smaller one that leaves it one (fewer weight rows per CU), and both operands have to fit LDS.
int gemm_norm_width(int M, int N, int K, int in_dt, int cus) {
  const long kb = (long)K * (in_dt == DT_FP8 ? 1 : 2), tm = (M + 31) / 32;
  if (M <= 0 || N <= 0 || kb % 128 || K > 1024 || K % 256) return 0;
  if (tm * ((N + 31) / 32) <= cus && 64 * kb + 9216 <= 160 * 1024) return 32;
  if (tm * ((N + 63) / 64) <= cus && 96 * kb + 9216 <= 160 * 1024) return 64;
  return 0;
}

hipError_t launch_gemm_norm(NormGemmArgs a, int in_dt, int width, bool k_parallel, hipStream_t st) {
  const int esz = in_dt == DT_FP8 ? 1 : 2, osz = a.out_dtype == DT_F32 ? 4 : a.out_dtype == DT_FP8 ? 1 : 2;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (gemm_norm_width(a.M, a.N, a.K, in_dt, 1 << 16) == 0 || (width != 32 && width != 64) || a.ldx % 4 || !al16(a.x) || !al16(a.gamma) || (a.beta && !al16(a.beta)) ||
      !al16(a.W) || (a.ldw * esz) % 16 || a.ldw * esz * 64 >= (1L << 31) ||
      (32 + width) * a.K * esz + 9216 > 160 * 1024)
    return hipErrorInvalidValue;
  if (a.nsplit <= 0 || a.nsplit > a.N || !a.out2) { a.nsplit = a.N; a.out2 = a.out; a.ldo2 = a.ldo; }
  if (a.rms) a.beta = nullptr;
  // groups of four columns: aligned, and on one side of the split
  a.vec_ok = al16(a.out) && al16(a.out2) && (a.ldo * osz) % 16 == 0 && (a.ldo2 * osz) % 16 == 0 && (a.nsplit == a.N || a.nsplit % 4 == 0);
#define NORM(DT) (width == 32 ? (k_parallel ? launch_norm<DT, 32, 4>(a, st) : launch_norm<DT, 32, 1>(a, st)) : (k_parallel ? launch_norm<DT, 64, 4>(a, st) : launch_norm<DT, 64, 1>(a, st)))
  switch (in_dt) {
    case DT_BF16: return NORM(DT_BF16);
    case DT_F16: return NORM(DT_F16);
    case DT_FP8: return NORM(DT_FP8);
  }
#undef NORM
  return hipErrorInvalidValue;
}

}  // namespace crl
