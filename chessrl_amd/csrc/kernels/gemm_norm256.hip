// Launches of the attention-bias generator's norms with the products behind them (gemm_norm256_kernel.hpp).
#include "gemm_norm256_kernel.hpp"

namespace crl {

template <int X_DT, int IN_DT, int RB, bool GROUPED>
static hipError_t launch_n256(Norm256KArgs k, int cus, hipStream_t st) {
  k.groups = (k.M + 32 * RB - 1) / (32 * RB);
  k.tiles = k.N / 64;
  // Slices of N: one workgroup fits a CU (its stages and operand are 74 or 139 KB), so the call takes rounds of workgroups, each its slice's steps long and
  // some four steps more for launch, norm and first weights. One row block: one tile each.
  const long slots = cus > 0 ? cus : 256;
  k.steps = 1;
  if (RB > 1) {
    long best = -1;
    for (int steps = 1; steps <= k.tiles; ++steps) {
      const long units = (long)k.groups * ((k.tiles + steps - 1) / steps), cost = (units + slots - 1) / slots * (steps + 4);
      if (best < 0 || cost < best) { best = cost; k.steps = steps; }
    }
  }
  const int grid = k.groups * ((k.tiles + k.steps - 1) / k.steps);
  if (grid >= 65536) return hipErrorInvalidValue;
  k.m_groups = dmaf_magic(k.groups);
  k.per_xcd = grid >> 3;
  hipLaunchKernelGGL((gemm_norm256_kernel<X_DT, IN_DT, RB, GROUPED>), dim3(grid), dim3(512), 0, st, k);
  return hipGetLastError();
}

bool gemm_norm256_can(const Norm256Args& a) {
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if ((a.x_dtype != DT_BF16 && a.x_dtype != DT_F16) || (a.in_dtype != a.x_dtype && a.in_dtype != DT_FP8)) return false;
  if (a.M <= 0 || a.M > 65536 || a.N <= 0 || a.N % 64 || !a.gamma || !a.beta || !a.x || !a.W || !a.out) return false;
  if (a.grouped ? a.M % 32 != 0 || a.ldx != 256 || a.bias : a.in_dtype == DT_FP8 || !a.bias) return false;
  return a.ldx >= 256 && a.ldx % 8 == 0 && a.ldo >= a.N && a.ldo % 8 == 0 && al16(a.x) && al16(a.gamma) && al16(a.beta) && al16(a.W) &&
         al16(a.out) && (!a.bias || al16(a.bias)) && (long)a.N * 512 < (1L << 31);
}

hipError_t launch_gemm_norm256(const Norm256Args& a, hipStream_t st) {
  if (!gemm_norm256_can(a)) return hipErrorInvalidValue;
  Norm256KArgs k{};
  k.x = a.x; k.ldx = a.ldx; k.gamma = a.gamma; k.beta = a.beta; k.W = a.W; k.bias = a.bias; k.out = a.out; k.ldo = a.ldo;
  k.M = a.M; k.N = a.N; k.eps = a.eps; k.x_scale = a.x_scale; k.descale = a.descale;
  const int cus = device_cus();
  // 32 rows while every tile of 32 x 64 has a CU, else 64.
  const bool small = (long)((a.M + 31) / 32) * (a.N / 64) <= cus;
#define N256(X, IN, G) (small ? launch_n256<X, IN, 1, G>(k, cus, st) : launch_n256<X, IN, 2, G>(k, cus, st))
  if (!a.grouped) return a.x_dtype == DT_BF16 ? N256(DT_BF16, DT_BF16, false) : N256(DT_F16, DT_F16, false);
  if (a.in_dtype == DT_FP8) return a.x_dtype == DT_BF16 ? N256(DT_BF16, DT_FP8, true) : N256(DT_F16, DT_FP8, true);
  return a.x_dtype == DT_BF16 ? N256(DT_BF16, DT_BF16, true) : N256(DT_F16, DT_F16, true);
#undef N256
}

}  // namespace crl
