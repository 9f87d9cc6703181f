// Launches of the norm-and-product kernel (gemm_norm_kernel.hpp).
#include "gemm_norm_kernel.hpp"

namespace crl {

constexpr int NORM_SPARE = 9216, NORM_LDS = 160 * 1024;   // gain and offset, the spare kilobyte

template <int IN_DT, int BM, bool X16>
static hipError_t launch_norm(const NormGemmArgs& a, int bn, hipStream_t st) {
  static std::atomic<bool> attr_set[16] = {};
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2;
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto kern = gemm_norm_kernel<IN_DT, BM, X16>;
  if (dev < 0 || dev >= 16 || !attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, NORM_LDS);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 16) attr_set[dev] = true;
  }
  NormGemmKArgs k;
  k.a = a;
  k.nslab = a.K * ESZ / 128;
  k.tiles_m = (a.M + BM - 1) / BM;
  k.m_tm = dmaf_magic(k.tiles_m);
  const int tiles = k.tiles_m * ((a.N + bn - 1) / bn), rg = bn / 8;
  if (tiles >= 65536) return hipErrorInvalidValue;
  k.per_xcd = tiles >> 3;
  k.bn = bn; k.m_bn2 = dmaf_magic(bn / 2);
  k.w_div = 16 / rg; k.w_mod = 16 % rg; k.loads = (rg * k.nslab + 15) / 16;
  if (k.loads > 9 || BM * bn > 2048) return hipErrorInvalidValue;
  // operands, gain and offset, the spare kilobyte; the patches of the sums; what is read ahead of the last slab of W
  const int lds = std::max({(BM + bn) * a.K * ESZ + NORM_SPARE, (bn + 31) / 32 * 4096, (k.nslab + 3) * bn * 128 + 4096});
  if (lds > NORM_LDS) return hipErrorInvalidValue;
  hipLaunchKernelGGL(kern, dim3(tiles), dim3(1024), lds, st, k);
  return hipGetLastError();
}

// Rows and columns of a tile for this call, or no columns where the kernel does not serve it: every tile has a CU of its own and both operands fit LDS.
// 16 rows, whose norm is half the work of 32, where the columns allow it; then the fewest columns, i.e. weight rows, per CU. (Which calls are
// served at all is decided by tiles of 32 rows.)
NormTile gemm_norm_tile(int M, int N, int K, int in_dt, int cus) {
  const long kb = (long)K * (in_dt == DT_FP8 ? 1 : 2);
  if (M <= 0 || N <= 0 || kb % 128 || K > 1024 || K % 256) return {0, 0};
  auto fits = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn) <= cus && (bm + bn) * kb + NORM_SPARE <= NORM_LDS && bn * kb <= 9 * 16 * 1024 && (kb / 128 + 3) * bn * 128 + 4096 <= NORM_LDS; };
  if (!fits(32, 64) && !fits(32, 32)) return {0, 0};
  for (int bm = 16; bm <= 32; bm += 16)
    for (int bn = 8; bn <= (bm == 16 ? 96 : 64); bn += 8)
      if (fits(bm, bn)) return {bm, bn};
  return {0, 0};
}

hipError_t launch_gemm_norm(NormGemmArgs a, int in_dt, NormTile t, hipStream_t st) {
  const int esz = in_dt == DT_FP8 ? 1 : 2, osz = a.out_dtype == DT_F32 ? 4 : a.out_dtype == DT_FP8 ? 1 : 2;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (gemm_norm_tile(a.M, a.N, a.K, in_dt, 1 << 16).bn == 0 || (t.bm != 16 && t.bm != 32) || t.bn < 8 || t.bn % 8 || a.ldx % 4 || !al16(a.x) || !al16(a.gamma) || (a.beta && !al16(a.beta)) ||
      !al16(a.W) || (a.ldw * esz) % 16 || a.ldw * esz * 96 >= (1L << 31) ||
      (t.bm + t.bn) * a.K * esz + NORM_SPARE > NORM_LDS)
    return hipErrorInvalidValue;
  if (a.nsplit <= 0 || a.nsplit > a.N || !a.out2) { a.nsplit = a.N; a.out2 = a.out; a.ldo2 = a.ldo; }
  if (a.rms) a.beta = nullptr;
  // groups of four columns: aligned, and on one side of the split
  a.vec_ok = al16(a.out) && al16(a.out2) && (a.ldo * osz) % 16 == 0 && (a.ldo2 * osz) % 16 == 0 && (a.nsplit == a.N || a.nsplit % 4 == 0);
  if (a.x_dtype != DT_F32 && (a.x_dtype != in_dt || in_dt == DT_FP8 || a.K % 512 || a.ldx % 8 || !al16(a.x) || (a.norm_out && (a.ld_norm % 8 || !al16(a.norm_out))))) return hipErrorInvalidValue;
  if (a.x_dtype == DT_F32 && a.norm_out) return hipErrorInvalidValue;
#define NORM(DT, X) (t.bm == 16 ? launch_norm<DT, 16, X>(a, t.bn, st) : launch_norm<DT, 32, X>(a, t.bn, st))
  switch (in_dt) {
    case DT_BF16: return a.x_dtype == DT_F32 ? NORM(DT_BF16, false) : NORM(DT_BF16, true);
    case DT_F16: return a.x_dtype == DT_F32 ? NORM(DT_F16, false) : NORM(DT_F16, true);
    case DT_FP8: return NORM(DT_FP8, false);
  }
#undef NORM
  return hipErrorInvalidValue;
}

}  // namespace crl
