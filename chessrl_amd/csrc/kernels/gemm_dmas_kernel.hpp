// C[M,N] = epilogue(A[M,K] · W[N,K]^T) on a 64x64 or 32x32 workgroup tile fed by direct-to-LDS loads through a ring of stages: the
// kernel for products so small that every tile has a CU of its own, the products of one to a few positions and of the
// token steps of generation. Such a launch is a few microseconds of latency in a row and nothing else on the CU hides any
// of it, so the kernel is built to shorten the row:
//  * Loading and computing waves are different waves. A load instruction of 64 x 16 bytes holds its wave for 100 to 150
//    cycles, and a CU moves 64 bytes per clock into LDS at most: eight waves that do nothing else reach that (146 GB/s; one
//    wave pulls 23), the computing ones start on the first slab while the later ones are still being requested.
//  * The fragments of slab s + 1 are read from LDS between the MFMAs of slab s, which are one chain, and a wave issues in order.
//  * The epilogue belongs to the loading waves: 512 threads need a third of the time one wave needs for a tile of 1024 elements,
//    which is a chain of some 300 instructions there. Residual and bias are brought into LDS meanwhile by a wave of their own.
//  * Everything the kernel needs to know travels in 144 bytes of arguments, requested at once (they are read from memory, cold,
//    before the first address can be formed).
// Measured inside passes of one position (bf16, by the workgroups' own clock from their first to their last instruction, of which the first slab takes 1900 to 2800 cycles and the epilogue
// 1000; launch and drain, which the profiler's trace counts too, come on top: 4.4 to 5.0 us a launch of one position there): M = 64, N = 1024, K = 1024 2.5 us
// where the memory-side cache has the weights and 2.9 past it (3.0 and 4.1 on 32x32 tiles with 32x32x16 MFMAs), K = 1536 3.0 and 3.3 (3.7 and 5.6), N = 768, K = 3072 4.1 (5.7);
// M = 128, N = 768, K = 3072 4.8 (7.3 with four waves on K). One position of 15 layers 685 -> 643 us, of GPT 182 -> 171; token steps of 128 sequences 51.1 -> 48.5 ms a rollout.
// Same K order and same arithmetic per element as the other tiled kernels: bit-equal results.
#pragma once
#include "gemm_dmaf_kernel.hpp"

namespace crl {

// BT = 64: eight stages of 16 KB, four computing waves of 32x32; BT = 32: sixteen stages of 8 KB. Eight loading waves either way (twelve delay the first slab: GPT one position
// 217 -> 228 us), which keep AHEAD stages requested, and one wave that fetches what the epilogue needs. AHEAD is some 64 KB, all that a CU has in flight: the first slab is
// announced when AHEAD have been asked for, and 14 stages of 64 rows put that at 4400 cycles instead of 2500 (one position 684 -> 711 us), of 32 rows
// (PAIRS) K = 1536 past the caches at 3900 instead of 2560.
// QUADS (BT = 32, 16-bit operands): four computing waves, a quarter of the tile each, with 16x16x32 MFMAs. Those add K exactly as two 32x32x16 do (checked on sums of
// normal, wide-ranged and all-positive values: the same bits), but follow each other in at most 32 cycles where two of the other take 97: a slab 136 cycles with its barrier
// instead of 208. (e4m3 has no such pair: 16x16x128 differs from two 32x32x64 in one sum of eight.)
// PAIRS (tiles of at most 16 x 16): a stage holds two slabs, the second in rows 16 to 31 of either operand: a barrier for two slabs, 105 cycles each.
template <int BT, int QUADS_ = 0, int AHEAD_ = 6, int PAIRS_ = 0>
struct DmasCfg {
  static_assert(BT == 64 || BT == 32, "two tile sizes");
  static constexpr bool QUADS = QUADS_ != 0;
  static_assert(!QUADS || BT == 32, "quarters of 16x16");
  static constexpr bool PAIRS = PAIRS_ != 0;
  static_assert(!PAIRS || QUADS, "one quarter");
  static constexpr int BM = BT, BN = BT, WGM = QUADS ? 2 : BT / 32, WGN = QUADS ? 2 : BT / 32, WT = QUADS ? 16 : 32;   // rows and columns of a computing wave
  static constexpr int NCOMP = WGM * WGN, NLOAD = 8, NT = 64 * (NCOMP + NLOAD + 1);
  static constexpr int ROWB = 128, NSTAGE = 512 / BT, AHEAD = AHEAD_;
  static constexpr int LOADS = 2 * BT / (8 * NLOAD);           // load instructions (8 rows each) of a wave per stage
  static constexpr int STAGE = BN * ROWB;                      // bytes of one operand's rows in one stage
  static constexpr int PART_BYTES = NSTAGE * STAGE;            // 64 KB: the weight rows of all stages, then the activation rows
  static constexpr int RES_OFF = 2 * PART_BYTES;               // residual of the tile as it lies in memory, row by row
  static constexpr int BIAS_OFF = RES_OFF + BM * BN * 4;
  static constexpr int LDS_BYTES = BIAS_OFF + 64 * 4;
  static constexpr int EV = BM * BN / (64 * NLOAD);            // elements of an epilogue thread: 2 or 8 consecutive columns of one row
  // The sums of 32x32 block w on their way to the epilogue: a patch in the weight rows of the stage(s) behind the last
  // slab's, which held slab nslab - NSTAGE and which nothing is loaded into any more.
  static __device__ __forceinline__ int patch_off(int nslab, int w) {
    return ((nslab + w * 4096 / STAGE) & (NSTAGE - 1)) * STAGE + w * 4096 % STAGE;
  }
  static_assert(AHEAD * LOADS < 64 && AHEAD + 2 <= NSTAGE, "the counted waits fit the counter; a stage is read before it is refilled");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS of a CU");
};

struct SmallArgs {
  const void* A; const void* W; void* C; void* C2; const float* bias; const void* res; float* amax;
  int lda_b, ldw_b;            // row strides in bytes
  int ldc, ldc2, ldr;          // in elements
  int M, N, nslab, nsplit;
  int act, res_dtype, res_rows, vec_ok;
  float descale, alpha, out_scale;
  int inner; uint32_t m_inner; // tiles along the direction that is walked first, and the magic of dividing by them
  int by_cols;                 // 1: that direction is down a column of tiles
  int per_xcd;                 // workgroups per XCD
  int bm, bn;                  // rows and columns of C a workgroup makes: BT, or fewer in multiples of eight
};

__device__ __forceinline__ void dmas_barrier() { asm volatile("s_barrier" ::: "memory"); }

// The epilogue of one thread: EV consecutive columns of one row, arithmetic as in gemm_epilogue. small_full: the tile's columns
// lie inside C and on one side of the column split, with aligned rows (uniform): vector accesses, residual and bias from LDS.
// small_edge: element by element.
__device__ __forceinline__ bool small_tile_full(const SmallArgs& s, int n0, int bn) { return s.vec_ok && n0 + bn <= s.N && (n0 >= s.nsplit || n0 + bn <= s.nsplit); }
// e4m3(out_scale * mish(...)) with nothing else asked for has an activation of its own, as in gemm_epilogue
template <int OUT_DT>
__device__ __forceinline__ bool small_fused_mish(const SmallArgs& s) { return OUT_DT == DT_FP8 && s.act == ACT_MISH && !s.res && s.alpha == 1.f && !s.amax; }
__device__ __forceinline__ float small_mish8(const SmallArgs& s, float acc, float bias, float x) {
  constexpr float L2E = 1.4426950408889634f;
  const float nexp = __builtin_amdgcn_exp2f(fmaf(acc, s.descale * L2E, bias * L2E));
  return x * fmaf(fast_rcp(fmaf(nexp, nexp + 2.f, 2.f)), -2.f * s.out_scale, s.out_scale);
}

template <int OUT_DT>
__device__ __forceinline__ void small_edge(const SmallArgs& s, const float* acc, int ev, int m, int n0) {
  float am = 0.f;
#pragma unroll 1
  for (int e = 0; e < ev; ++e) {
    const int n = n0 + e;
    if (m >= s.M || n >= s.N) break;
    const float x = acc[e], bias = s.bias ? s.bias[n] : 0.f;
    float v = fmaf(x, s.descale, bias);
    if (small_fused_mish<OUT_DT>(s)) {
      v = small_mish8(s, x, bias, v);
    } else {
      v = apply_act(v, s.act);
      if (s.res) {
        const long o = (long)(s.res_rows > 0 ? m % s.res_rows : m) * s.ldr + n;
        const float rv = s.res_dtype == DT_F32 ? reinterpret_cast<const float*>(s.res)[o]
                         : s.res_dtype == DT_F16 ? f16_bits_to_f32(reinterpret_cast<const uint16_t*>(s.res)[o])
                                                 : bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(s.res)[o]);
        v = fmaf(v, s.alpha, rv);
      } else if (s.alpha != 1.f) {
        v *= s.alpha;
      }
      am = fmaxf(am, fabsf(v));
      if constexpr (OUT_DT == DT_FP8) v *= s.out_scale;
    }
    if (n < s.nsplit) store1<OUT_DT>(s.C, (long)m * s.ldc + n, v);
    else store1<OUT_DT>(s.C2, (long)m * s.ldc2 + (n - s.nsplit), v);
  }
  if (s.amax) {
    am = wave_max(am);
    if ((threadIdx.x & 63) == 0) atomic_amax(s.amax, am);
  }
}

template <int OUT_DT, int EV>
__device__ __forceinline__ void small_full(const SmallArgs& s, const float (&acc)[EV], int m, int n, bool first, const float* bias_lds, const uint8_t* res_lds) {
  float v[EV], bias[EV];
  uint32_t res[EV];   // raw: EV fp32 words, or EV / 2 words of 16-bit pairs
#pragma unroll
  for (int e = 0; e < EV; ++e) { bias[e] = 0.f; res[e] = 0; }
  if (s.bias) {
#pragma unroll
    for (int e = 0; e < EV; ++e) bias[e] = bias_lds[e];
  }
  if (s.res) {
    const uint32_t* p = reinterpret_cast<const uint32_t*>(res_lds);
    if (s.res_dtype == DT_F32) {
#pragma unroll
      for (int e = 0; e < EV; ++e) res[e] = p[e];
    } else {
#pragma unroll
      for (int e = 0; e < EV / 2; ++e) res[e] = p[e];
    }
  }
#pragma unroll
  for (int e = 0; e < EV; ++e) v[e] = fmaf(acc[e], s.descale, bias[e]);
  if (small_fused_mish<OUT_DT>(s)) {
#pragma unroll
    for (int e = 0; e < EV; ++e) v[e] = small_mish8(s, acc[e], bias[e], v[e]);
  } else {
    switch (s.act) {   // uniform
      case ACT_GELU:
#pragma unroll
        for (int e = 0; e < EV; ++e) v[e] = act_gelu(v[e]);
        break;
      case ACT_MISH:
#pragma unroll
        for (int e = 0; e < EV; ++e) v[e] = act_mish(v[e]);
        break;
      case ACT_SWISH:
#pragma unroll
        for (int e = 0; e < EV; ++e) v[e] = act_swish(v[e]);
        break;
      default: break;
    }
    if (s.res) {
#pragma unroll
      for (int e = 0; e < EV; ++e) {
        const uint32_t w = s.res_dtype == DT_F32 ? res[e] : (e & 1) ? res[e >> 1] >> 16 : res[e >> 1] & 0xffff;
        const float rv = s.res_dtype == DT_F32 ? __uint_as_float(w) : s.res_dtype == DT_F16 ? f16_bits_to_f32((uint16_t)w) : bf16_bits_to_f32((uint16_t)w);
        v[e] = fmaf(v[e], s.alpha, rv);
      }
    } else if (s.alpha != 1.f) {
#pragma unroll
      for (int e = 0; e < EV; ++e) v[e] *= s.alpha;
    }
    if (__builtin_expect(s.amax != nullptr, 0)) {
      float am = 0.f;
#pragma unroll
      for (int e = 0; e < EV; ++e)
        if (m < s.M) am = fmaxf(am, fabsf(v[e]));
      am = wave_max(am);
      if ((threadIdx.x & 63) == 0) atomic_amax(s.amax, am);
    }
    if constexpr (OUT_DT == DT_FP8) {
#pragma unroll
      for (int e = 0; e < EV; ++e) v[e] *= s.out_scale;
    }
  }
  if (m >= s.M) return;
  const long o = first ? (long)m * s.ldc + n : (long)m * s.ldc2 + (n - s.nsplit);
  void* const out = first ? s.C : s.C2;
  if constexpr (EV == 8) {
    store8<OUT_DT, 0>(out, o, v);
  } else if constexpr (OUT_DT == DT_F32) {
    *reinterpret_cast<float2*>(reinterpret_cast<float*>(out) + o) = make_float2(v[0], v[1]);
  } else if constexpr (OUT_DT == DT_BF16) {
    *reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(out) + o) = pack_bf16x2(v[0], v[1]);
  } else if constexpr (OUT_DT == DT_F16) {
    *reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(out) + o) = (uint32_t)f32_to_f16_bits(v[0]) | ((uint32_t)f32_to_f16_bits(v[1]) << 16);
  } else {
    *reinterpret_cast<uint16_t*>(reinterpret_cast<uint8_t*>(out) + o) = (uint16_t)pack_fp8x4(v[0], v[1], v[0], v[1]);
  }
}

// ONCE: GemmArgs::w_once (an instance of its own: a branch at every load cost a call of one position 2 %)
// SLICED: the fp32 sums of K share y = blockIdx.y go to rows y M .. y M + M - 1 of C. Share y is what group y % 4 of a four-group workgroup walks of slice
// y / 4 of K: nslab slabs, every fourth one.
template <typename Cfg, int IN_DT, int OUT_DT, int ONCE = 0, int SLICED = 0>
__global__ void __launch_bounds__(Cfg::NT) gemm_dmas_kernel(const SmallArgs s_in) {
  SmallArgs s = s_in;
  if constexpr (SLICED) s.C = reinterpret_cast<float*>(s.C) + (long)blockIdx.y * s.M * s.ldc;
  constexpr int KSTEPS = Cfg::ROWB / (IN_DT == DT_FP8 ? 64 : 32);   // MFMA K steps per slab
  constexpr int BM = Cfg::BM, BN = Cfg::BN, LOADS = Cfg::LOADS, NSTAGE = Cfg::NSTAGE, AHEAD = Cfg::AHEAD, EV = Cfg::EV;
  constexpr int STAGE = Cfg::STAGE;
  extern __shared__ __align__(16) uint8_t smem[];

  // (all arguments in registers at this point: left alone, the compiler asks for them in four batches, one wait after the other)
  asm volatile("" ::"s"(s.A), "s"(s.W), "s"(s.C), "s"(s.bias), "s"(s.res), "s"(s.amax), "s"(s.lda_b), "s"(s.ldr), "s"(s.nsplit), "s"(s.vec_ok), "s"(s.per_xcd));
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nslab = Cfg::PAIRS ? (s.nslab + 1) >> 1 : s.nslab;   // stages to fill

  // Workgroup b runs on XCD b & 7, which owns a contiguous range of the tile order (rows or columns first, see the launch).
  int pid = blockIdx.x;
  if (pid < (s.per_xcd << 3)) pid = (pid & 7) * s.per_xcd + (pid >> 3);
  const int outer = dmaf_div(pid, s.m_inner), inner = pid - outer * s.inner;
  const int tile_m = s.by_cols ? inner : outer, tile_n = s.by_cols ? outer : inner;
  const int bm = BM == 32 ? s.bm : BM, bn = BM == 32 ? s.bn : BN;
  const int m0 = tile_m * bm, n0 = tile_n * bn;

  // Barrier i (0 .. nslab - 1) of the workgroup says that slab i has landed, barrier nslab that sums, residual and bias
  // lie in LDS. Every wave passes all of them.
  if (wave == Cfg::NCOMP + Cfg::NLOAD) {
    if (small_tile_full(s, n0, bn)) {
      if (s.bias) {
        int n = n0 + lane;
        n = n < s.N ? n : s.N - 1;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(s.bias + n), (__attribute__((address_space(3))) void*)(smem + Cfg::BIAS_OFF), 4, 0, 0);
      }
      if (s.res) {
        // 16 bytes per lane: 64 / lpr rows per instruction (a row past the end reads the last one, a column past the tile the first ones; nothing of either is stored)
        const int rowb = s.res_dtype == DT_F32 ? BN * 4 : BN * 2, lpr = rowb >> 4;
        const int sh = 31 - __builtin_clz(lpr);
        const int chunk = (lane & (lpr - 1)) << 4;
        const char* const base = reinterpret_cast<const char*>(s.res) + ((long)n0 << (s.res_dtype == DT_F32 ? 2 : 1)) + (chunk < bn << (s.res_dtype == DT_F32 ? 2 : 1) ? chunk : 0);
        const long ldr_b = (long)s.ldr << (s.res_dtype == DT_F32 ? 2 : 1);
#pragma unroll 1
        for (int i = 0; i < (bm * lpr + 63) / 64; ++i) {
          int m = m0 + i * (64 >> sh) + (lane >> sh);
          m = m < s.M ? m : s.M - 1;
          if (__builtin_expect(s.res_rows > 0, 0)) m = m % s.res_rows;
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base + m * ldr_b),
                                           (__attribute__((address_space(3))) void*)(smem + Cfg::RES_OFF + i * 1024), 16, 0, 0);
        }
      }
    }
#pragma unroll 1
    for (int i = 0; i < nslab; ++i) dmas_barrier();
    wait_vmcnt<0>();
    dmas_barrier();
    return;
  }
  if (wave >= Cfg::NCOMP) {
    // Loading waves: the first half fills the weight rows of a stage, the second half the activation rows, 8 LOADS consecutive
    // rows each: 8 rows per wave-instruction, eight 16-byte chunks per row, the swizzle applied on the global side.
    const int lw = wave - Cfg::NCOMP;
    const bool loads_a = lw >= Cfg::NLOAD / 2;
    const int rbase = (lw & (Cfg::NLOAD / 2 - 1)) * (8 * LOADS);
    const int ld = loads_a ? s.lda_b : s.ldw_b;
    int rows_left = loads_a ? s.M - m0 : s.N - n0;
    if constexpr (BM == 32) rows_left = min(rows_left, loads_a ? bm : bn);
    const bool idle = BM == 32 && (Cfg::PAIRS ? rbase & 15 : rbase) >= (loads_a ? bm : bn);   // (a narrower tile has fewer groups of eight rows)
    uint32_t voff[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int r = (Cfg::PAIRS ? rbase & 15 : rbase + 8 * i) + (lane >> 3);
      r = r < rows_left ? r : rows_left - 1;
      voff[i] = (uint32_t)r * (uint32_t)ld + (Cfg::PAIRS ? (rbase >> 4) * Cfg::ROWB : 0) + (((lane & 7) ^ lds_swizzle16(rbase + 8 * i + (lane >> 3))) << 4);
    }
    // (the rows of a tile span less than 2 GB: the launcher checks; they end with K, which the second slab of a last pair may lie behind)
    const uint8_t* origin = reinterpret_cast<const uint8_t*>(loads_a ? s.A : s.W) + (long)(loads_a ? m0 : n0) * ld + (SLICED ? (long)((blockIdx.y >> 2) * 4 * nslab + (blockIdx.y & 3)) * Cfg::ROWB : 0);
    const __amdgpu_buffer_rsrc_t rsrc_mine = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(origin), 0, SLICED ? (rows_left < BM ? rows_left : BM) * ld : ((rows_left < BM ? rows_left : BM) - 1) * ld + s.nslab * Cfg::ROWB, 0x00020000);
    const uint32_t lds_load0 = (loads_a ? Cfg::PART_BYTES : 0) + rbase * Cfg::ROWB;   // stage 0
    auto issue_slab = [&](int slab) {
      if (idle) return;
      uint8_t* dst = smem + lds_load0 + (slab & (NSTAGE - 1)) * STAGE;
      static_for<0, LOADS>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        constexpr int STEP = SLICED ? 4 * Cfg::ROWB : Cfg::PAIRS ? 2 * Cfg::ROWB : Cfg::ROWB;
        if (ONCE && !loads_a) dmaf_load16_nt(rsrc_mine, dst + i * 1024, (int)voff[i], slab * STEP);
        else dmaf_load16(rsrc_mine, dst + i * 1024, (int)voff[i], slab * STEP);
      });
    };
#pragma unroll
    for (int s0 = 0; s0 < AHEAD; ++s0)
      if (s0 < nslab) issue_slab(s0);
    {
      int slab = 0;
#pragma unroll 1
      for (; slab + AHEAD < nslab; ++slab) {
        wait_vmcnt<(AHEAD - 1) * LOADS>();
        dmas_barrier();
        // (stage slab + AHEAD - NSTAGE <= slab - 2, whose fragments the computing waves had in registers before they came here)
        issue_slab(slab + AHEAD);
      }
      // The last AHEAD slabs, or all there are: nothing is issued any more, so each wait leaves one slab less in flight.
      static_for<0, AHEAD>([&](auto ic) {
        constexpr int left = AHEAD - decltype(ic)::value;   // slabs still to be announced
        if (nslab - slab >= left) {
          wait_vmcnt<(left - 1) * LOADS>();
          dmas_barrier();
          ++slab;
        }
      });
    }
    dmas_barrier();
    // This thread's part of the epilogue: row er, columns ec .. ec + EV - 1 of the tile.
    constexpr int TPR = BN / EV;   // threads per row
    const int et = tid - 64 * Cfg::NCOMP, er = et / TPR, ec = (et % TPR) * EV;
    const int pr = er & 31, pc = ec & 31;
    float acc[EV];
    const float* const patch = reinterpret_cast<const float*>(smem + Cfg::patch_off(nslab, (er >> 5) + (ec >> 5) * (BM / 32))) + pr * 32;
    if constexpr (EV == 8) {
      const f32x4_t lo = *reinterpret_cast<const f32x4_t*>(patch + (((pc >> 2) ^ (pr & 7)) << 2));
      const f32x4_t hi = *reinterpret_cast<const f32x4_t*>(patch + ((((pc >> 2) + 1) ^ (pr & 7)) << 2));
#pragma unroll
      for (int e = 0; e < 4; ++e) { acc[e] = lo[e]; acc[4 + e] = hi[e]; }
    } else {
      const float2 p2 = *reinterpret_cast<const float2*>(patch + (((pc >> 2) ^ (pr & 7)) << 2) + (pc & 3));
      acc[0] = p2.x; acc[1] = p2.y;
    }
    const int m = BM == 32 && (er >= bm || ec >= bn) ? s.M : m0 + er;   // (M: nothing is stored)
    if (__builtin_expect(small_tile_full(s, n0, bn), 1))
      small_full<OUT_DT, EV>(s, acc, m, n0 + ec, n0 < s.nsplit, reinterpret_cast<const float*>(smem + Cfg::BIAS_OFF) + ec,
                             smem + Cfg::RES_OFF + (er * BN + ec) * (s.res_dtype == DT_F32 ? 4 : 2));
    else small_edge<OUT_DT>(s, acc, EV, m, n0 + ec);
    return;
  }

  const int wm = wave % Cfg::WGM, wn = wave / Cfg::WGM;
  constexpr int WT = Cfg::WT;
  if (m0 + wm * WT >= s.M || n0 + wn * WT >= s.N || (BM == 32 && (wm * WT >= bm || wn * WT >= bn))) {
    for (int i = 0; i <= nslab; ++i) dmas_barrier();
    return;
  }
  // Fragment addresses, as in gemm_dmaf_kernel.hpp: lane group g (of 64 / WT) holds chunks (16 bytes of a row's 128; e4m3: pairs of them) g and on, one step of K behind
  // the other; chunk Kc ^ L with L per lane and a compile-time Kc that takes four values, two in quarters.
  constexpr int STEPS = Cfg::PAIRS ? 4 : Cfg::QUADS ? 2 : KSTEPS;   // of a stage
  const int lr = lane & (WT - 1), g = lane / WT;
  const int LW = (IN_DT == DT_FP8 ? 2 * g : g) ^ lds_swizzle16(wn * WT + lr);
  const int LX = (IN_DT == DT_FP8 ? 2 * g : g) ^ lds_swizzle16(wm * WT + lr);
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)smem);
  constexpr int NB = Cfg::QUADS && !Cfg::PAIRS ? 2 : 4;
  uint32_t wb0[NB], xb0[NB];
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    // (pairs: steps 2 and 3 are those of rows 16 further, whose swizzle has bit 1 flipped)
    const int kc = Cfg::PAIRS ? (4 * (k & 1)) ^ (k & 2) : Cfg::QUADS ? 4 * k : IN_DT == DT_FP8 ? ((k & 1) | ((k >> 1) << 2)) : 2 * k;
    const int second = Cfg::PAIRS && k >= 2 ? 16 * Cfg::ROWB : 0;
    wb0[k] = lds0 + (wn * WT + lr) * Cfg::ROWB + second + ((kc ^ LW) << 4);
    xb0[k] = lds0 + Cfg::PART_BYTES + (wm * WT + lr) * Cfg::ROWB + second + ((kc ^ LX) << 4);
  }
  typedef std::conditional_t<Cfg::QUADS, f32x4_t, f32x16_t> Acc;
  Acc acc{};
  struct Frags { Frag<IN_DT> w[STEPS], x[STEPS]; };
  auto read_step = [&](uint32_t soff, Frags& f, auto ksc) {
    constexpr int ks = decltype(ksc)::value;
    auto piece = [&](uint32_t base) -> i32x4_t { return *reinterpret_cast<const __attribute__((address_space(3))) i32x4_t*>(base + soff); };
    if constexpr (IN_DT == DT_FP8) {
      // chunks 4 ks and 4 ks + 1 of the slab: lane addresses 2 ks and 2 ks + 1
      f.w[ks].lo = piece(wb0[2 * ks]); f.w[ks].hi = piece(wb0[2 * ks + 1]);
      f.x[ks].lo = piece(xb0[2 * ks]); f.x[ks].hi = piece(xb0[2 * ks + 1]);
    } else {
      f.w[ks].lo = piece(wb0[ks]);
      f.x[ks].lo = piece(xb0[ks]);
    }
  };
  auto mul_step = [&](const Frags& f, auto ksc) {
    constexpr int ks = decltype(ksc)::value;
    if constexpr (Cfg::QUADS) acc = mfma_quad<IN_DT>(f.w[ks], f.x[ks], acc);
    else acc = mfma_frag<IN_DT>(f.w[ks], f.x[ks], acc);
  };
  __builtin_amdgcn_s_setprio(2);
  Frags f0, f1;
  auto last_step = [&](Frags& cur) {   // (the last pair may be a single slab)
    static_for<0, Cfg::PAIRS ? 2 : STEPS>([&](auto ksc) { mul_step(cur, ksc); });
    if (Cfg::PAIRS && (s.nslab & 1) == 0) static_for<2, STEPS>([&](auto ksc) { mul_step(cur, ksc); });
  };
  dmas_barrier();
  static_for<0, STEPS>([&](auto ksc) { read_step(0, f0, ksc); });
  auto step = [&](int slab, Frags& cur, Frags& nxt) {
    dmas_barrier();    // slab + 1 has landed
    const uint32_t soff = ((slab + 1) & (NSTAGE - 1)) * STAGE;
    static_for<0, STEPS>([&](auto ksc) {
      mul_step(cur, ksc);
      __builtin_amdgcn_sched_barrier(0);
      read_step(soff, nxt, ksc);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  int slab = 0;
  for (; slab + 2 < nslab; slab += 2) {
    step(slab, f0, f1);
    step(slab + 1, f1, f0);
  }
  if (slab + 1 < nslab) {
    step(slab, f0, f1);
    last_step(f1);
  } else {
    last_step(f0);
  }
  // The sums go to a 32x32 block's patch, rows of 32 floats in 16-byte chunks swizzled by row: acc[4 rq + e] is column 8 rq + 4 g + e of row lr (in quarters: column 4 g + e).
  if constexpr (Cfg::QUADS) {
    const int row = wm * WT + lr;
    float* const patch = reinterpret_cast<float*>(smem + Cfg::patch_off(nslab, 0));
    *reinterpret_cast<f32x4_t*>(patch + row * 32 + (((4 * wn + g) ^ (row & 7)) << 2)) = acc;
  } else {
    float* const patch = reinterpret_cast<float*>(smem + Cfg::patch_off(nslab, wave));
#pragma unroll
    for (int rq = 0; rq < 4; ++rq)
      *reinterpret_cast<f32x4_t*>(patch + lr * 32 + (((2 * rq + g) ^ (lr & 7)) << 2)) = f32x4_t{acc[4 * rq], acc[4 * rq + 1], acc[4 * rq + 2], acc[4 * rq + 3]};
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the patch is written
  dmas_barrier();
}

// Rows and columns of C per workgroup of the 32x32 form: of the tiles that leave every one a CU, the one whose workgroup reads the fewest rows of both
// operands. A CU gets 30 bytes a cycle from memory (some 64 KB in flight at 2000 cycles and more), less than half of what it gets from L2: the walk of 32 + 32
// rows over weights that come from memory takes 310 cycles a slab. The same 64 rows by 1024 columns on 256 workgroups of 16x16 instead of
// 64 of 32x32 read half as much each. MFMA lanes past the tile multiply whatever lies in LDS there; nothing of theirs is stored.
struct SmallTile { int bm, bn; };
inline SmallTile small_tile(int M, int N, int cus) {
  SmallTile best{32, 32};
  for (int bm = 8; bm <= 32; bm += 8)
    for (int bn = 8; bn <= 32; bn += 8) {
      if ((long)((M + bm - 1) / bm) * ((N + bn - 1) / bn) > cus) continue;
      if (bm + bn < best.bm + best.bn || (bm + bn == best.bm + best.bn && bm * bn > best.bm * best.bn)) best = {bm, bn};
    }
  return best;
}

template <typename Cfg, int IN_DT, int OUT_DT, int ONCE = 0, int SLICED = 0>
static hipError_t launch_dmas(const GemmArgs& a, hipStream_t st, int shares = 1, int bm = Cfg::BM, int bn = Cfg::BN) {
  static_assert(!SLICED || OUT_DT == DT_F32, "a share's sums as they are");
  if constexpr (!ONCE && !SLICED) {
    // (up to 512 rows: the weight rows that more tiles share do better kept in L2; 8 positions 1062 -> 1013 us, 12 the same, 16 1222 -> 1262)
    if (a.w_once && a.M <= 512) return launch_dmas<Cfg, IN_DT, OUT_DT, 1>(a, st, 1, bm, bn);
  }
  static std::atomic<bool> attr_set[16] = {};
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2;
  auto fits = [](long v) { return v >= 0 && v < (1L << 31); };
  if ((a.K * ESZ) % (Cfg::ROWB * shares) != 0 || a.K <= 0 || a.res_stats || !fits(a.lda * ESZ * 64) || !fits(a.ldw * ESZ * 64) || !fits(a.ldc) || !fits(a.ldc2) || (a.res && !fits(a.ldr)))
    return hipErrorInvalidValue;
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto kern = gemm_dmas_kernel<Cfg, IN_DT, OUT_DT, ONCE, SLICED>;
  if (dev < 0 || dev >= 16 || !attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 16) attr_set[dev] = true;
  }
  const int tiles_n = (a.N + bn - 1) / bn;
  const int tiles = ((a.M + bm - 1) / bm) * tiles_n;
  if (tiles >= 65536) return hipErrorInvalidValue;
  SmallArgs s{};
  s.A = a.A; s.W = a.W; s.C = a.C; s.C2 = a.C2; s.bias = a.bias; s.res = a.res; s.amax = a.amax;
  s.lda_b = (int)(a.lda * ESZ); s.ldw_b = (int)(a.ldw * ESZ); s.ldc = (int)a.ldc; s.ldc2 = (int)a.ldc2; s.ldr = (int)a.ldr;
  s.M = a.M; s.N = a.N; s.nslab = a.K * ESZ / Cfg::ROWB / shares; s.nsplit = a.nsplit;
  s.act = a.act; s.res_dtype = a.res_dtype; s.res_rows = a.res_rows; s.vec_ok = a.vec_ok;
  s.descale = a.descale; s.alpha = a.alpha; s.out_scale = a.out_scale;
  // Rows or columns of tiles first, whichever lets an XCD read fewer rows of both operands: each XCD's L2 fetches its own copy (BT4-class bf16, whole calls
  // of 2, 4 and 8 positions: 850 -> 835, 912 -> 868, 1083 -> 1065 us). Two rows of tiles gain nothing.
  const int tiles_m = tiles / tiles_n, per = std::max(tiles >> 3, 1);
  const int by_rows = (per + tiles_n - 1) / tiles_n * bm + std::min(per, tiles_n) * bn, by_cols = (per + tiles_m - 1) / tiles_m * bn + std::min(per, tiles_m) * bm;
  s.by_cols = tiles_m >= 4 && by_cols < by_rows;
  s.inner = s.by_cols ? tiles_m : tiles_n;
  s.m_inner = dmaf_magic(s.inner); s.per_xcd = tiles >> 3; s.bm = bm; s.bn = bn;
  hipLaunchKernelGGL(kern, dim3(tiles, shares), dim3(Cfg::NT), Cfg::LDS_BYTES, st, s);
  return hipGetLastError();
}

}  // namespace crl
