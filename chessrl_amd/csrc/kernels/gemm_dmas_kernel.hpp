// C[M,N] = epilogue(A[M,K] · W[N,K]^T) on a 64x64 or 32x32 workgroup tile fed by direct-to-LDS loads through a ring of stages
// (loads, ring and K order are those of gemm_dmam_kernel.hpp): the kernel for products so small that every tile has a CU of
// its own, the products of one to a few positions and of the token steps of generation. Such a launch is a few
// microseconds of latency in a row, and nothing on the CU hides any of it, so this kernel is built to shorten the row:
//  * the fragments of slab s + 1 are read from LDS while the MFMAs of slab s run (a 32x32 wave tile is one chain of
//    dependent MFMAs; read, wait, multiply in turn cost 0.18 us per slab);
//  * the residual is requested before anything else and waits in registers (read in the epilogue it was a trip to memory
//    with nothing beside it);
//  * the code is short and straight: the epilogue's branches that such a call does not take lie outside the path, the ring is
//    filled by a loop (a cold instruction cache fetches every line of what runs, and a forward pass changes kernels 200
//    times).
// Same K order and same arithmetic per element as the other tiled kernels: bit-equal results.
#pragma once
#include "gemm_dmaf_kernel.hpp"

namespace crl {

// BT = 64: four waves of 32x32, eight stages of 16 KB. BT = 32: one wave computes and fills the weight rows, a second one fills the
// activation rows; sixteen stages of 8 KB (K = 1024 16-bit elements are in flight whole). A wave fills 32 of a stage's rows
// with four load instructions.
template <int BT>
struct DmasCfg {
  static_assert(BT == 64 || BT == 32, "two tile sizes");
  static constexpr int BM = BT, BN = BT, WGM = BT / 32, WGN = BT / 32;
  static constexpr int NCOMP = WGM * WGN;                      // waves that compute
  static constexpr int NW = BT == 64 ? 4 : 2, NT = 64 * NW;    // waves that load: all of them
  static constexpr int ROWB = 128, NSTAGE = 512 / BT, LOADS = 4;
  static constexpr int PART_BYTES = NSTAGE * BN * ROWB;        // 64 KB: the weight rows of all stages, then the activation rows
  static constexpr int RING_BYTES = 2 * PART_BYTES;            // 128 KB
  static constexpr int COLS_OFF = RING_BYTES;                  // bias: [wave][64]
  static constexpr int LDS_BYTES = COLS_OFF + NW * 64 * 4;
  static_assert((NSTAGE - 2) * LOADS + 1 < 64, "the counted waits fit the counter");
};

__device__ __forceinline__ void dmas_barrier() { asm volatile("s_barrier" ::: "memory"); }
// (a function of its own, like dmam_load16: inside a kernel template this builtin makes the host pass drop the kernel's stub)
__device__ __forceinline__ void dmas_load16(__amdgpu_buffer_rsrc_t r, uint8_t* dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
}
// All LDS reads issued so far have returned (known to the compiler, which then adds no waits of its own).
__device__ __forceinline__ void dmas_wait_lds() { __builtin_amdgcn_s_waitcnt(0xC07F); }

// The epilogue of one 32x32 wave tile, as gemm_epilogue does it for WM = WN = 32: through an LDS patch a lane gets eight
// consecutive columns of two rows. A tile whose columns lie inside C and on one side of the column split, with aligned
// rows (small_full, uniform), has its residual requested before the main loop (small_load_res); the others go element by
// element in a loop (small_epilogue_edge).
struct SmallRes { uint4 r[2][2]; };   // [row][low, high half]: 16 bytes of a 16-bit residual, 32 of an fp32 one
__device__ __forceinline__ bool small_full(const GemmArgs& a, int nw0) {
  return a.vec_ok && nw0 + 32 <= a.N && (nw0 >= a.nsplit || nw0 + 32 <= a.nsplit);
}
__device__ __forceinline__ void small_load_res(const GemmArgs& a, int mw0, int nw0, int lane, SmallRes& s) {
  const int sz = a.res_dtype == DT_F32 ? 4 : 2;
  const char* const base = reinterpret_cast<const char*>(a.res) + (long)(nw0 + (lane & 3) * 8) * sz;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    int m = mw0 + (lane >> 2) + 16 * it;
    m = m < a.M ? m : a.M - 1;   // (a row past the end reads the last one; nothing of it is stored)
    if (__builtin_expect(a.res_rows > 0, 0)) m = m % a.res_rows;
    const char* p = base + m * (a.ldr * sz);
    s.r[it][0] = *reinterpret_cast<const uint4*>(p);
    if (sz == 4) s.r[it][1] = *reinterpret_cast<const uint4*>(p + 16);
  }
}
// (as in gemm_epilogue: e4m3(out_scale * mish(...)) with nothing else asked for has an activation of its own)
template <int OUT_DT>
__device__ __forceinline__ bool small_fused_mish(const GemmArgs& a) { return OUT_DT == DT_FP8 && a.act == ACT_MISH && !a.res && a.alpha == 1.f && !a.amax; }
__device__ __forceinline__ float small_mish8(const GemmArgs& a, float acc, float bias, float x) {
  constexpr float L2E = 1.4426950408889634f;
  const float nexp = __builtin_amdgcn_exp2f(fmaf(acc, a.descale * L2E, bias * L2E));
  return x * fmaf(fast_rcp(fmaf(nexp, nexp + 2.f, 2.f)), -2.f * a.out_scale, a.out_scale);
}

template <int OUT_DT>
__device__ __forceinline__ void small_epilogue_edge(const GemmArgs& a, const float* sC, int mw0, int nw0, int lane) {
  const int r = lane & 31, m = mw0 + r;
  float am = 0.f;
#pragma unroll 1
  for (int c = lane >> 5; c < 32; c += 2) {
    const int n = nw0 + c;
    if (m >= a.M || n >= a.N) continue;
    const float acc = sC[r * 32 + (((c >> 2) ^ (r & 7)) << 2) + (c & 3)];
    const float bias = a.bias ? a.bias[n] : 0.f;
    float v = fmaf(acc, a.descale, bias);
    if (small_fused_mish<OUT_DT>(a)) {
      v = small_mish8(a, acc, bias, v);
    } else {
      v = apply_act(v, a.act);
      if (a.res) {
        const long o = (long)(a.res_rows > 0 ? m % a.res_rows : m) * a.ldr + n;
        const float rv = a.res_dtype == DT_F32 ? reinterpret_cast<const float*>(a.res)[o]
                         : a.res_dtype == DT_F16 ? f16_bits_to_f32(reinterpret_cast<const uint16_t*>(a.res)[o])
                                                 : bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(a.res)[o]);
        v = fmaf(v, a.alpha, rv);
      } else if (a.alpha != 1.f) {
        v *= a.alpha;
      }
      am = fmaxf(am, fabsf(v));
      if constexpr (OUT_DT == DT_FP8) v *= a.out_scale;
    }
    if (n < a.nsplit) store1<OUT_DT>(a.C, (long)m * a.ldc + n, v);
    else store1<OUT_DT>(a.C2, (long)m * a.ldc2 + (n - a.nsplit), v);
  }
  if (a.amax) {
    am = wave_max(am);
    if (lane == 0) atomic_amax(a.amax, am);
  }
}

template <int OUT_DT>
__device__ __forceinline__ void small_epilogue(const GemmArgs& a, const f32x16_t& acc, float* sC, int mw0, int nw0, int lane, const float* sCols,
                                               const SmallRes& res) {
  const int lr = lane & 31, g = lane >> 5, ec = lane & 3, er = lane >> 2;
#pragma unroll
  for (int rq = 0; rq < 4; ++rq)
    *reinterpret_cast<f32x4_t*>(sC + lr * 32 + (((2 * rq + g) ^ (lr & 7)) << 2)) = f32x4_t{acc[4 * rq], acc[4 * rq + 1], acc[4 * rq + 2], acc[4 * rq + 3]};
  wave_lds_fence();
  if (__builtin_expect(!small_full(a, nw0), 0)) {
    small_epilogue_edge<OUT_DT>(a, sC, mw0, nw0, lane);
    return;
  }
  const int n = nw0 + ec * 8;
  const float descale = a.descale, alpha = a.alpha;
  float bias8[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) bias8[e] = 0.f;
  if (a.bias) {
    const f32x4_t b0 = *reinterpret_cast<const f32x4_t*>(sCols + ec * 8), b1 = *reinterpret_cast<const f32x4_t*>(sCols + ec * 8 + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { bias8[e] = b0[e]; bias8[4 + e] = b1[e]; }
  }
  float v[2][8];
  const bool fused_mish = small_fused_mish<OUT_DT>(a);
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int r = er + 16 * it;
    const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(sC + r * 32 + (((2 * ec) ^ (r & 7)) << 2));
    const f32x4_t hi = *reinterpret_cast<const f32x4_t*>(sC + r * 32 + (((2 * ec + 1) ^ (r & 7)) << 2));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[it][e] = fmaf(lo[e], descale, bias8[e]);
      v[it][4 + e] = fmaf(hi[e], descale, bias8[4 + e]);
    }
    if (fused_mish) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[it][e] = small_mish8(a, e < 4 ? lo[e] : hi[e - 4], bias8[e], v[it][e]);
    }
  }
  if (!fused_mish) {
    switch (a.act) {   // uniform
      case ACT_GELU:
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i >> 3][i & 7] = act_gelu(v[i >> 3][i & 7]);
        break;
      case ACT_MISH:
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i >> 3][i & 7] = act_mish(v[i >> 3][i & 7]);
        break;
      case ACT_SWISH:
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i >> 3][i & 7] = act_swish(v[i >> 3][i & 7]);
        break;
      default: break;
    }
    if (a.res) {
#pragma unroll
      for (int it = 0; it < 2; ++it) {
        const uint4 lo = res.r[it][0], hi = res.r[it][1];
        const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        float rv[8];
        if (a.res_dtype == DT_F32) {
#pragma unroll
          for (int e = 0; e < 8; ++e) rv[e] = __uint_as_float(w[e]);
        } else if (a.res_dtype == DT_F16) {
#pragma unroll
          for (int e = 0; e < 8; ++e) rv[e] = f16_bits_to_f32((uint16_t)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffff)));
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) rv[e] = __uint_as_float((e & 1) ? (w[e >> 1] & 0xffff0000u) : (w[e >> 1] << 16));
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) v[it][e] = fmaf(v[it][e], alpha, rv[e]);
      }
    } else if (alpha != 1.f) {
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i >> 3][i & 7] *= alpha;
    }
    if (__builtin_expect(a.amax != nullptr, 0)) {
      float am = 0.f;
#pragma unroll
      for (int it = 0; it < 2; ++it)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (mw0 + er + 16 * it < a.M) am = fmaxf(am, fabsf(v[it][e]));
      am = wave_max(am);
      if (lane == 0) atomic_amax(a.amax, am);
    }
    if constexpr (OUT_DT == DT_FP8) {
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i >> 3][i & 7] *= a.out_scale;
    }
  }
  constexpr int OUT_SZ = OUT_DT == DT_F32 ? 4 : OUT_DT == DT_FP8 ? 1 : 2;
  const bool first = nw0 < a.nsplit;
  char* const out = reinterpret_cast<char*>(first ? a.C : a.C2) + (long)(first ? n : n - a.nsplit) * OUT_SZ;
  const long stride = (first ? a.ldc : a.ldc2) * OUT_SZ;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int m = mw0 + er + 16 * it;
    if (m < a.M) store8<OUT_DT, 0>(out + m * stride, 0, v[it]);
  }
}

template <typename Cfg, int IN_DT, int OUT_DT>
__global__ void __launch_bounds__(Cfg::NT) gemm_dmas_kernel(const GemmArgs a, const DmafWalk wk) {
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2;                      // bytes per operand element
  constexpr int KSTEPS = Cfg::ROWB / (IN_DT == DT_FP8 ? 64 : 32);   // MFMA K steps per slab
  constexpr int BM = Cfg::BM, BN = Cfg::BN, LOADS = Cfg::LOADS, NSTAGE = Cfg::NSTAGE;
  constexpr int STAGE = BN * Cfg::ROWB;   // bytes of one operand's rows in one stage
  extern __shared__ __align__(16) uint8_t smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % Cfg::WGM, wn = (wave / Cfg::WGM) % Cfg::WGN;
  const int lr = lane & 31, g = lane >> 5;

  // Workgroup b runs on XCD b & 7, which owns a contiguous range of the row-major tile order.
  int pid = blockIdx.x;
  {
    const int per = gridDim.x >> 3;
    if (pid < (per << 3)) pid = (pid & 7) * per + (pid >> 3);
  }
  const int tile_m = dmaf_div(pid, wk.m_tn), tile_n = pid - tile_m * wk.tiles_n;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int mw0 = m0 + wm * 32, nw0 = n0 + wn * 32;
  const int nslab = a.K * ESZ / Cfg::ROWB;  // the launcher sends only whole slabs of K here
  const bool wave_active = wave < Cfg::NCOMP && mw0 < a.M && nw0 < a.N;

  // The residual of this wave's tile, ahead of the ring's loads (so the counted waits below cover it).
  SmallRes res;
  if (a.res && wave_active && small_full(a, nw0)) small_load_res(a, mw0, nw0, lane, res);
  __builtin_amdgcn_sched_barrier(0);

  // Loader role: the first half of the waves fills the weight rows of a stage, the second half the activation rows, 32
  // consecutive rows each: 8 rows per wave-instruction, eight 16-byte chunks per row, the swizzle applied on the global
  // side (row r = rbase + 8 i + lane / 8 has swizzle lds_swizzle(r) = (lane / 8) ^ ((rbase / 8 + i) & 7)).
  const bool loads_a = wave >= Cfg::NW / 2;
  const int rbase = (wave & (Cfg::NW / 2 - 1)) * 32;
  const int ld = (loads_a ? a.lda : a.ldw) * ESZ;   // row stride in bytes
  const int rows_left = loads_a ? a.M - m0 : a.N - n0;
  uint32_t voff[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    int r = rbase + 8 * i + (lane >> 3);
    r = r < rows_left ? r : rows_left - 1;
    voff[i] = (uint32_t)r * (uint32_t)ld + (((lane & 7) ^ (lane >> 3) ^ ((rbase / 8 + i) & 7)) << 4);
  }
  const long span = (long)(rows_left < BM ? rows_left : BM) * ld;
  const uint8_t* origin = loads_a ? reinterpret_cast<const uint8_t*>(a.A) + (long)m0 * a.lda * ESZ
                                  : reinterpret_cast<const uint8_t*>(a.W) + (long)n0 * a.ldw * ESZ;
  const __amdgpu_buffer_rsrc_t rsrc_mine = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(origin), 0, (int)(span < 0x7fffffffL ? span : 0x7fffffffL), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_none = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.A), 0, 0, 0x00020000);
  const uint32_t lds_load0 = (loads_a ? Cfg::PART_BYTES : 0) + rbase * Cfg::ROWB;   // stage 0
  auto issue_slab = [&](int slab) {
    const __amdgpu_buffer_rsrc_t r = slab < nslab ? rsrc_mine : rsrc_none;
    uint8_t* dst = smem + lds_load0 + (slab & (NSTAGE - 1)) * STAGE;
    static_for<0, LOADS>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      dmas_load16(r, dst + i * 1024, (int)voff[i], slab * Cfg::ROWB);
    });
  };
#pragma unroll 1
  for (int s0 = 0; s0 < NSTAGE - 1; ++s0) issue_slab(s0);
  __builtin_amdgcn_sched_barrier(0);

  // Bias of this wave's 32 columns (and the 32 behind them, which nothing reads), one column per lane, landed outside the
  // ring; columns past N repeat the last one. Issued behind the first slabs: the first waits allow for it.
  if (a.bias) {
    int n = nw0 + lane;
    n = n < a.N ? n : a.N - 1;
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a.bias + n),
                                     (__attribute__((address_space(3))) void*)(smem + Cfg::COLS_OFF + wave * 256), 4, 0, 0);
  }

  // Fragment addresses, as in gemm_dmaf_kernel.hpp: chunk Kc ^ L with L = (2g or g) ^ swizzle(row) per lane and a
  // compile-time Kc that takes four values.
  const int LW = (IN_DT == DT_FP8 ? 2 * g : g) ^ lds_swizzle(wn * 32 + lr);
  const int LX = (IN_DT == DT_FP8 ? 2 * g : g) ^ lds_swizzle(wm * 32 + lr);
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)smem);
  uint32_t wb0[4], xb0[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int kc = IN_DT == DT_FP8 ? ((k & 1) | ((k >> 1) << 2)) : 2 * k;
    wb0[k] = lds0 + (wn * 32 + lr) * Cfg::ROWB + ((kc ^ LW) << 4);
    xb0[k] = lds0 + Cfg::PART_BYTES + (wm * 32 + lr) * Cfg::ROWB + ((kc ^ LX) << 4);
  }

  f32x16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  struct Frags { Frag<IN_DT> w[KSTEPS], x[KSTEPS]; };
  auto read_slab = [&](int slab, Frags& f) {
    const uint32_t soff = (slab & (NSTAGE - 1)) * STAGE;
    auto piece = [&](uint32_t base) -> i32x4_t { return *reinterpret_cast<const __attribute__((address_space(3))) i32x4_t*>(base + soff); };
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
      if constexpr (IN_DT == DT_FP8) {
        // chunks 4 ks and 4 ks + 1 of the slab: lane addresses 2 ks and 2 ks + 1
        f.w[ks].lo = piece(wb0[2 * ks]); f.w[ks].hi = piece(wb0[2 * ks + 1]);
        f.x[ks].lo = piece(xb0[2 * ks]); f.x[ks].hi = piece(xb0[2 * ks + 1]);
      } else {
        f.w[ks].lo = piece(wb0[ks]);
        f.x[ks].lo = piece(xb0[ks]);
      }
    }
  };
  auto mfma_slab = [&](const Frags& f) {
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) acc = mfma_frag<IN_DT>(f.w[ks], f.x[ks], acc);
  };

  // Slab 0 of this wave's loads has landed (NSTAGE - 2 slabs behind it and the bias may be in flight); past the barrier everybody's has.
  if (a.bias) wait_vmcnt<(NSTAGE - 2) * LOADS + 1>();
  else wait_vmcnt<(NSTAGE - 2) * LOADS>();
  dmas_barrier();
  if (wave_active) {
    Frags f0, f1;
    read_slab(0, f0);
    auto step = [&](int slab, Frags& cur, Frags& nxt) {
      // Slab + 1 has landed (NSTAGE - 3 slabs behind it may be in flight). Past the barrier every wave has the fragments of
      // slab - 1 in registers (it waited for them before the MFMAs), so that slab's stage is refilled.
      wait_vmcnt<(NSTAGE - 3) * LOADS>();
      dmas_wait_lds();
      dmas_barrier();
      issue_slab(slab + NSTAGE - 1);
      read_slab(slab + 1, nxt);   // (past the last slab: what the stage holds; nothing uses it)
      __builtin_amdgcn_sched_barrier(0);
      mfma_slab(cur);
      __builtin_amdgcn_sched_barrier(0);
    };
    int slab = 0;
    for (; slab + 1 < nslab; slab += 2) {
      step(slab, f0, f1);
      step(slab + 1, f1, f0);
    }
    if (slab < nslab) step(slab, f0, f1);
  } else {
    for (int slab = 0; slab < nslab; ++slab) {   // (a wave that only loads: the same waits, barriers and loads)
      wait_vmcnt<(NSTAGE - 3) * LOADS>();
      dmas_barrier();
      issue_slab(slab + NSTAGE - 1);
    }
  }

  wait_vmcnt<0>();
  dmas_wait_lds();
  dmas_barrier();  // every wave is done with the ring, and the empty loads past the end of K have retired
  if (!wave_active) return;
  small_epilogue<OUT_DT>(a, acc, reinterpret_cast<float*>(smem) + wave * (32 * 32), mw0, nw0, lane,
                         reinterpret_cast<const float*>(smem + Cfg::COLS_OFF) + wave * 64, res);
}

template <typename Cfg, int IN_DT, int OUT_DT>
static hipError_t launch_dmas(const GemmArgs& a, hipStream_t st) {
  static std::atomic<bool> attr_set[16] = {};
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2;
  if ((a.K * ESZ) % Cfg::ROWB != 0 || a.K <= 0 || a.res_stats || (long)a.lda * ESZ * 64 >= (1L << 31) || (long)a.ldw * ESZ * 64 >= (1L << 31))
    return hipErrorInvalidValue;
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto kern = gemm_dmas_kernel<Cfg, IN_DT, OUT_DT>;
  if (dev < 0 || dev >= 16 || !attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 16) attr_set[dev] = true;
  }
  const int tiles_n = (a.N + Cfg::BN - 1) / Cfg::BN;
  const int tiles = ((a.M + Cfg::BM - 1) / Cfg::BM) * tiles_n;
  if (tiles >= 65536) return hipErrorInvalidValue;
  DmafWalk wk{};
  wk.tiles_n = tiles_n;
  wk.m_tn = dmaf_magic(tiles_n);
  hipLaunchKernelGGL(kern, dim3(tiles), dim3(Cfg::NT), Cfg::LDS_BYTES, st, a, wk);
  return hipGetLastError();
}

}  // namespace crl
