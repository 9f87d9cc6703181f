// C[M,N] = epilogue(A[M,K] · W[N,K]^T) on a 128x128 workgroup tile, K a whole number of 128-byte slabs: the kernel of batches
// whose 256x256 tiles would leave CUs idle (a batch of 16 to 64 positions).
// Four waves load and eight multiply. A load instruction holds its wave for 100 cycles and more; eight waves that loaded and
// multiplied in turn took 1.3 times the sum of both (M = 4096, N = 1024, K = 1024, one tile per CU: 16.0 us, of which
// 3.4 are loads and 3.5 MFMAs). The loading waves keep all but one of the ring's four stages of 32 KB (three of 40) requested; slab s is announced by a workgroup barrier, at
// which the multiplying waves are through with slab s - 1, so its stage is the next to be filled. They read the fragments
// of a slab from LDS between the MFMAs of the one before.
// Workgroups are persistent, one per CU, where the epilogue below serves the call: the loading waves run on into the next tile while the
// multiplying ones finish theirs, each for itself, in the accumulator layout and through 2 KB of LDS of its own outside the ring (as in
// gemm_dmaf_kernel.hpp). Residuals are requested half way through a tile's walk over K.
// Measured (bf16, M = 4096): N = 1024, K = 1024 with residual 16.5 -> 13.9 us, K = 1536 21.3 -> 18.1, N = 1536 with mish 27.9 -> 20.9 (register-staged before);
// 128x192 tiles (twelve multiplying waves, three stages of 40 KB) do the work of 1.5 tiles in 1.25 of their time: M = 4096, N = 1536, K = 1024 one round instead of two, 20.9 -> 19 us,
// M = 2816 19.5 -> 14.
// e4m3, M = 2112: N = 3104 16.4 -> 11.8. A slab takes 680 cycles where its MFMAs take 512; weights that come from memory add 3000 cycles to a tile.
// Same K order and same arithmetic per element as the other tiled kernels: bit-equal results.
#pragma once
#include "gemm_dmaf_kernel.hpp"

namespace crl {

template <int BN_>
struct DmamCfgN {
  static constexpr int BM = 128, BN = BN_, WGM = 2, WGN = BN / 32, NCOMP = WGM * WGN, NLOAD = 4, NT = 64 * (NCOMP + NLOAD);
  static constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 32;       // 64x32 per wave
  static constexpr int ROWB = 128, NSTAGE = BN == 128 ? 4 : 3, AHEAD = NSTAGE - 1;
  static constexpr int LOADS = (BM + BN) / 32;                           // load instructions of a loading wave per slab
  static constexpr int STAGE = (BM + BN) * ROWB;                         // weight rows, then activation rows
  static constexpr int PATCH_OFF = NSTAGE * STAGE, PATCH = 2048;         // a wave's patch: 32 rows of 64 bytes
  static constexpr int COLS_OFF = PATCH_OFF + NCOMP * PATCH;             // per-column constants: [wave][bias, gain, offset][64] (a load lands 64)
  static constexpr int LDS_BYTES = COLS_OFF + NCOMP * 3 * 64 * 4;
  static_assert(LDS_BYTES <= 160 * 1024 && AHEAD * LOADS < 64 && AHEAD < NSTAGE && NT <= 1024, "LDS of a CU; the counted waits; the ring; a workgroup");
};
typedef DmamCfgN<128> DmamCfg;

// A bare barrier: the waits it needs are written out in front of it (a __syncthreads waits for every outstanding memory
// operation, i.e. for the slabs that are meant to stay in flight).
__device__ __forceinline__ void dmam_barrier() { asm volatile("s_barrier" ::: "memory"); }

// The order of the tiles: columns in groups of up to gw, inside a group row by row.
struct DmamWalk {
  int gw, lastw, per_group, ngroups;        // columns of a group, of the last one; tiles of a group
  uint32_t m_group, m_gw, m_lastw;          // magics
  __device__ __forceinline__ void pos(int t, int& tm, int& tn) const {
    const int g = dmaf_div(t, m_group), r = t - g * per_group;
    const bool last = g + 1 == ngroups;
    tm = dmaf_div(r, last ? m_lastw : m_gw);
    tn = g * gw + r - tm * (last ? lastw : gw);
  }
};
inline DmamWalk dmam_walk(int tiles_m, int tiles_n) {
  DmamWalk w{};
  w.ngroups = (tiles_n + 5) / 6;
  w.gw = (tiles_n + w.ngroups - 1) / w.ngroups;
  w.ngroups = (tiles_n + w.gw - 1) / w.gw;
  w.lastw = tiles_n - (w.ngroups - 1) * w.gw;
  w.per_group = tiles_m * w.gw;
  w.m_group = dmaf_magic(w.per_group); w.m_gw = dmaf_magic(w.gw); w.m_lastw = dmaf_magic(w.lastw);
  return w;
}

// EPI, ACT: as in gemm_dmaf_kernel.hpp.
template <int IN_DT, int OUT_DT, int EPI, int ACT = ACT_NONE, int TILE_N = 128>
__global__ void __launch_bounds__(DmamCfgN<TILE_N>::NT) gemm_dmam_kernel(const GemmArgs a, const int tiles, const DmamWalk walk) {
  typedef DmamCfgN<TILE_N> Cfg;
  constexpr bool PERSIST = EPI >= DMAF_PLAIN;
  constexpr bool HAS_RES = EPI == DMAF_RES16 || EPI == DMAF_RESNORM || EPI == DMAF_RES32;
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2, OSZ = OUT_DT == DT_F32 ? 4 : OUT_DT == DT_FP8 ? 1 : 2, RSZ = EPI == DMAF_RES32 ? 4 : 2;
  constexpr int KSTEPS = Cfg::ROWB / (IN_DT == DT_FP8 ? 64 : 32);   // MFMA K steps per slab
  constexpr int TM = Cfg::TM, BM = Cfg::BM, BN = Cfg::BN;
  extern __shared__ __align__(16) uint8_t smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nslab = a.K * ESZ / Cfg::ROWB;
  // Workgroup b runs on XCD b & 7, which owns a contiguous range of the row-major tile order. With fewer workgroups than
  // tiles (a multiple of eight then) an XCD's workgroups take its tiles in turn.
  int tile = blockIdx.x, hi = tiles, step = tiles;
  if ((int)gridDim.x < tiles) {
    const int xcd = blockIdx.x & 7;
    tile = (int)((long)tiles * xcd >> 3) + ((int)blockIdx.x >> 3);
    hi = (int)((long)tiles * (xcd + 1) >> 3);
    step = (int)gridDim.x >> 3;
    if (tile >= hi) return;
  } else {
    const int per = tiles >> 3;
    if (tile < (per << 3)) tile = (tile & 7) * per + (tile >> 3);
  }

  if (wave >= Cfg::NCOMP) {
    // ---- loading waves, a quarter of a slab's weight rows and of its activation rows each: 8 rows per
    // wave-instruction, eight 16-byte chunks per row, the swizzle applied on the global side. They announce slab s (barrier s) and then request
    // slab s + AHEAD, whose stage is the one slab s - 1 has left. Past the last slab the requests are out of bounds: they keep the counts.
    const int lw = wave - Cfg::NCOMP, l8 = lane >> 3;
    constexpr int LW = Cfg::BN / 32, LA = Cfg::BM / 32;   // load instructions: of weight rows, of activation rows
    uint32_t voff[Cfg::LOADS];
    __amdgpu_buffer_rsrc_t rw, ra;
    int l_tile = tile, l_slab = 0, l_stage = 0;
    auto stream_tile = [&]() {
      int tm, tn;
      walk.pos(l_tile, tm, tn);
      const int m0 = tm * BM, n0 = tn * BN;
      const int left_w = a.N - n0 < BN ? a.N - n0 : BN, left_a = a.M - m0 < BM ? a.M - m0 : BM;
      const int ldw = (int)a.ldw * ESZ, lda = (int)a.lda * ESZ;
#pragma unroll
      for (int i = 0; i < Cfg::LOADS; ++i) {
        const int q = i < LW ? lw * LW + i : lw * LA + i - LW, left = i < LW ? left_w : left_a;
        int r = q * 8 + l8;
        r = r < left ? r : left - 1;
        voff[i] = (uint32_t)r * (uint32_t)(i < LW ? ldw : lda) + (((lane & 7) ^ l8 ^ (q & 7)) << 4);
      }
      rw = dmaf_rsrc(reinterpret_cast<const uint8_t*>(a.W) + (long)n0 * ldw, (long)left_w * ldw);
      ra = dmaf_rsrc(reinterpret_cast<const uint8_t*>(a.A) + (long)m0 * lda, (long)left_a * lda);
    };
    auto request = [&]() {
      if (l_slab == nslab) {
        l_slab = 0;
        l_tile += step;
        if (l_tile < hi) stream_tile();
        else rw = ra = dmaf_rsrc(a.A, 0);
      }
      uint8_t* const dst = smem + l_stage * Cfg::STAGE;
      static_for<0, Cfg::LOADS>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if constexpr (i < LW) dmaf_load16(rw, dst + (lw * LW + i) * 1024, (int)voff[i], l_slab * Cfg::ROWB);
        else dmaf_load16(ra, dst + BN * Cfg::ROWB + (lw * LA + i - LW) * 1024, (int)voff[i], l_slab * Cfg::ROWB);
      });
      ++l_slab;
      l_stage = l_stage + 1 == Cfg::NSTAGE ? 0 : l_stage + 1;
    };
    stream_tile();
#pragma unroll
    for (int s = 0; s < Cfg::AHEAD; ++s) request();
    const int mine = (hi - tile + step - 1) / step;   // tiles of this workgroup
#pragma unroll 1
    for (int s = mine * nslab; s > 0; --s) {
      wait_vmcnt<(Cfg::AHEAD - 1) * Cfg::LOADS>();
      dmam_barrier();
      request();
    }
    wait_vmcnt<0>();   // (before the ring becomes epilogue scratch, and before the workgroup's LDS is another's)
    if constexpr (!PERSIST) dmam_barrier();
    return;
  }

  // ---- multiplying waves
  const int wm = wave % Cfg::WGM, wn = wave / Cfg::WGM, lr = lane & 31, g = lane >> 5;
  // Fragment addresses, as in gemm_dmaf_kernel.hpp: chunk Kc ^ L with L = (2g or g) ^ swizzle(row) per lane and a compile-time Kc that
  // takes four values; the swizzle has the period of 64 rows.
  const int wrow = wn * Cfg::WN + lr;
  const int LW = (IN_DT == DT_FP8 ? 2 * g : g) ^ lds_swizzle(wrow & 63), LX = (IN_DT == DT_FP8 ? 2 * g : g) ^ lds_swizzle(lr);
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)smem);
  uint32_t wb[4], xb[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int kc = IN_DT == DT_FP8 ? ((k & 1) | ((k >> 1) << 2)) : 2 * k;
    wb[k] = lds0 + wrow * Cfg::ROWB + ((kc ^ LW) << 4);
    xb[k] = lds0 + (BN + wm * Cfg::WM + lr) * Cfg::ROWB + ((kc ^ LX) << 4);
  }
  struct Frags { Frag<IN_DT> w[KSTEPS], x[KSTEPS][TM]; };
  auto lds_piece = [](uint32_t addr) -> i32x4_t { return *reinterpret_cast<const __attribute__((address_space(3))) i32x4_t*>(addr); };
  // (row block 1 of the activations: rows + 32, whose swizzle has bit 2 flipped: another of the four lane addresses)
  auto x_piece = [&](uint32_t soff, int t, int ks, int half) -> i32x4_t {
    const int kc = (IN_DT == DT_FP8 ? 4 * ks + half : 2 * ks) ^ (4 * (t & 1));
    const int k = IN_DT == DT_FP8 ? ((kc & 1) | ((kc >> 2) << 1)) : kc >> 1;
    return lds_piece(xb[k] + soff + t * 32 * Cfg::ROWB);
  };
  auto read_step = [&](uint32_t soff, Frags& f, auto ksc) {
    constexpr int ks = decltype(ksc)::value;
    if constexpr (IN_DT == DT_FP8) {
      f.w[ks].lo = lds_piece(wb[2 * ks] + soff); f.w[ks].hi = lds_piece(wb[2 * ks + 1] + soff);
    } else {
      f.w[ks].lo = lds_piece(wb[ks] + soff);
    }
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      f.x[ks][t].lo = x_piece(soff, t, ks, 0);
      if constexpr (IN_DT == DT_FP8) f.x[ks][t].hi = x_piece(soff, t, ks, 1);
    }
  };
  f32x16_t acc[1][TM];
  auto mul_step = [&](Frags& f, auto ksc) {
    constexpr int ks = decltype(ksc)::value;
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[0][t] = mfma_frag<IN_DT>(f.w[ks], f.x[ks][t], acc[0][t]);
  };
  int r_stage = 0;
  Frags f;

  uint8_t* const patch = smem + Cfg::PATCH_OFF + wave * Cfg::PATCH;
  const float* const cols = reinterpret_cast<const float*>(smem + Cfg::COLS_OFF) + wave * (3 * 64);
  // 16-byte chunk c of patch row r; chunks are swizzled over groups of four rows (256 bytes are a pass of all banks)
  auto at = [&](int r, int c) -> uint8_t* { return patch + r * 64 + ((c ^ ((r >> 2) & 3)) << 4); };
  // store layout (16 bytes per lane): rows er + 16 it of a row block, chunk ec of a 64-byte row (e4m3: er + 32 it, of a 32-byte one)
  constexpr int EPR = OUT_DT == DT_FP8 ? 2 : 4;
  constexpr int NRES = EPI == DMAF_RES32 ? 8 : 4;        // residual loads of 16 bytes per lane
  u32x4_t res[HAS_RES ? NRES : 1];
  u32x2_t row_st[EPI == DMAF_RESNORM ? TM : 1];

  for (;;) {
    int tm0, tn0;
    walk.pos(tile, tm0, tn0);
    const int m0 = tm0 * BM, n0 = tn0 * BN;
    const bool wave_active = (m0 + wm * Cfg::WM < a.M) && (n0 + wn * Cfg::WN < a.N);
    const int rows = a.M - m0 < BM ? a.M - m0 : BM;
    {
      int n = n0 + wn * Cfg::WN + lane;
      n = n < a.N ? n : a.N - 1;
      uint8_t* c = smem + Cfg::COLS_OFF + wave * (3 * 64 * 4);
      if (a.bias) __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a.bias + n), (__attribute__((address_space(3))) void*)c, 4, 0, 0);
      else if constexpr (PERSIST) reinterpret_cast<float*>(c)[lane] = 0.f;   // (so that the epilogue reads the constants without asking)
      if constexpr (EPI == DMAF_RESNORM || EPI == DMAF_GENERAL_NORM) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a.res_gamma + n), (__attribute__((address_space(3))) void*)(c + 256), 4, 0, 0);
        if (a.res_beta)
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a.res_beta + n), (__attribute__((address_space(3))) void*)(c + 512), 4, 0, 0);
      }
    }
    auto res_load = [&]() {
      if constexpr (HAS_RES) {
        const int ln = dmaf_here(lane), ldrb = (int)a.ldr * RSZ, left = a.N - n0 < BN ? a.N - n0 : BN;
        const __amdgpu_buffer_rsrc_t rr = dmaf_rsrc(reinterpret_cast<const char*>(a.res) + (long)m0 * ldrb + (long)n0 * RSZ, (long)(rows - 1) * ldrb + (long)left * RSZ);
        const int v = (wm * Cfg::WM + (ln >> 2)) * ldrb + wn * Cfg::WN * RSZ + (ln & 3) * 16;
        // 16-bit: [row block][it]; fp32: [column half][row block][it]
#pragma unroll
        for (int j = 0; j < NRES; ++j) res[j] = dmaf_get16(rr, v + (j >> 2) * 64 + (j & 3) * 16 * ldrb);
        if constexpr (EPI == DMAF_RESNORM) {
          const __amdgpu_buffer_rsrc_t rs = dmaf_rsrc(a.res_stats + 2 * (long)m0, (long)rows * 8);
#pragma unroll
          for (int t = 0; t < TM; ++t) row_st[t] = dmaf_get8(rs, (wm * Cfg::WM + t * 32 + (ln & 31)) * 8);
        }
      }
    };
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][t][r] = 0.f;

    // A fragment of slab s + 1 is read as soon as the MFMAs that used its registers for slab s are issued; at a barrier every read before it has returned.
    auto landed = [&]() -> uint32_t {
      __builtin_amdgcn_s_waitcnt(0xC07F);
      dmam_barrier();
      const uint32_t soff = r_stage * Cfg::STAGE;
      r_stage = r_stage + 1 == Cfg::NSTAGE ? 0 : r_stage + 1;
      return soff;
    };
    {
      const uint32_t soff = landed();
      if (wave_active) static_for<0, KSTEPS>([&](auto ksc) { read_step(soff, f, ksc); });
    }
#pragma unroll 1
    for (int slab = 1; slab < nslab; ++slab) {
      const uint32_t soff = landed();
      // (half way: a CU's requests are answered in order, so the first slabs would wait behind a residual that comes from memory)
      if constexpr (HAS_RES) {
        if (slab == (nslab + 1) >> 1) res_load();
      }
      if (!wave_active) continue;
      static_for<0, KSTEPS>([&](auto ksc) {
        mul_step(f, ksc);
        __builtin_amdgcn_sched_barrier(0);
        read_step(soff, f, ksc);
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    if (HAS_RES && nslab == 1) res_load();
    if (wave_active) static_for<0, KSTEPS>([&](auto ksc) { mul_step(f, ksc); });

    if constexpr (!PERSIST) {
      __builtin_amdgcn_s_waitcnt(0xC07F);
      wait_vmcnt<0>();     // the column constants
      dmam_barrier();      // every wave has read the last slab, and nothing is on its way into the ring any more
      gemm_epilogue<Cfg::WM, Cfg::WN, OUT_DT, EPI == DMAF_GENERAL_NORM ? 1 : 0, 0>(a, acc, reinterpret_cast<float*>(smem) + wave * (32 * Cfg::WN), m0 + wm * Cfg::WM, n0 + wn * Cfg::WN, lane,
                                                         reinterpret_cast<float*>(smem + Cfg::STAGE) + wave * (2 * Cfg::WM), nullptr);
      return;
    } else {
      wait_vmcnt<0>();     // column constants and residual (requested a tile's walk ago), and the stores of the tile before
      const int ln = dmaf_here(lane), er = ln / EPR, ec = ln % EPR, el = ln & 31, eg = ln >> 5;
      const bool first = n0 < a.nsplit;      // (a tile lies on one side of the split: the launcher checks)
      const int ldob = (int)(first ? a.ldc : a.ldc2) * OSZ;
      int left = (first ? a.nsplit : a.N) - n0;
      left = left < BN ? left : BN;
      const __amdgpu_buffer_rsrc_t rsrc_o = dmaf_rsrc(reinterpret_cast<char*>(first ? a.C : a.C2) + (long)m0 * ldob + (long)(first ? n0 : n0 - a.nsplit) * OSZ,
                                                      (long)(rows - 1) * ldob + (long)left * OSZ);
      constexpr int NOWHERE = (int)0x80000000u, CPL = 16 / OSZ, NST = OUT_DT == DT_FP8 ? 1 : 2;     // columns per lane in the store layout, stores of a row block
      const bool nt = a.stream_out != 0 && (OUT_DT != DT_F32 || ldob % 128 == 0);
      // (one branch on the hint per row block, as in gemm_dmaf_kernel.hpp)
      auto put = [&](const u32x4_t (&v)[NST], int row, int col) {
        const int off = wn * Cfg::WN + col + (OUT_DT == DT_F32 && !HAS_RES ? 3 : 0) < left ? (wm * Cfg::WM + row) * ldob + (wn * Cfg::WN + col) * OSZ : NOWHERE;
        if (nt) {
#pragma unroll
          for (int it = 0; it < NST; ++it) dmaf_put16_nt(v[it], rsrc_o, off + it * (64 / EPR) * ldob);
        } else {
#pragma unroll
          for (int it = 0; it < NST; ++it) dmaf_put16(v[it], rsrc_o, off + it * (64 / EPR) * ldob);
        }
      };
      auto col_const = [&](const float* c, float (&o)[16]) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4_t v = *reinterpret_cast<const f32x4_t*>(c + 8 * q + 4 * eg);
#pragma unroll
          for (int e = 0; e < 4; ++e) o[4 * q + e] = v[e];
        }
      };
      auto activate = [&](float v) -> float {
        if constexpr (ACT == ACT_GELU) return act_gelu(v);
        else if constexpr (ACT == ACT_MISH) return act_mish(v);
        else return v;
      };
      if constexpr (OUT_DT == DT_F32) {
        // raw sums through the patch, 16 columns at a time; the rest in the store layout (4 columns per lane)
        static_for<0, 2 * TM>([&](auto sc) {
          constexpr int st = decltype(sc)::value, half = st / TM, t = st % TM;
          const f32x4_t bv = *reinterpret_cast<const f32x4_t*>(cols + half * 16 + ec * 4);
#pragma unroll
          for (int qq = 0; qq < 2; ++qq) {
            const int r0 = 4 * (2 * half + qq);
            *reinterpret_cast<f32x4_t*>(at(el, 2 * qq + eg)) = f32x4_t{acc[0][t][r0], acc[0][t][r0 + 1], acc[0][t][r0 + 2], acc[0][t][r0 + 3]};
          }
          wave_lds_fence();
          u32x4_t o[2];
#pragma unroll
          for (int it = 0; it < 2; ++it) o[it] = *reinterpret_cast<const u32x4_t*>(at(er + 16 * it, ec));
#pragma unroll
          for (int it = 0; it < 2; ++it)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float v = activate(fmaf(__uint_as_float(o[it][e]), a.descale, bv[e]));
              if constexpr (HAS_RES) v = fmaf(v, a.alpha, __uint_as_float(res[(half * TM + t) * 2 + it][e]));
              o[it][e] = __float_as_uint(v);
            }
          put(o, t * 32 + er, half * 16 + ec * 4);
          if constexpr (!HAS_RES) {
            const int col = wn * Cfg::WN + half * 16 + ec * 4;
            if (left & 3)
#pragma unroll
              for (int it = 0; it < 2; ++it) dmaf_put_part(o[it], rsrc_o, (wm * Cfg::WM + t * 32 + er + 16 * it) * ldob + col * 4, left - col);
          }
          wave_lds_fence();
        });
      } else {
        float bias16[16], gain16[16];
        col_const(cols, bias16);
        if constexpr (EPI == DMAF_RESNORM) {
          col_const(cols + 64, gain16);
          if (a.res_beta) {   // the offset joins the bias (which is multiplied by alpha)
            const float inv_alpha = 1.0f / a.alpha;
            float off16[16];
            col_const(cols + 128, off16);
#pragma unroll
            for (int i = 0; i < 16; ++i) bias16[i] += off16[i] * inv_alpha;
          }
        }
        static_for<0, TM>([&](auto tc) {
          constexpr int t = decltype(tc)::value;
          uint32_t resw[8];
          if constexpr (HAS_RES) {   // the residual from the store layout to the accumulator layout
#pragma unroll
            for (int it = 0; it < 2; ++it) *reinterpret_cast<u32x4_t*>(at(er + 16 * it, ec)) = res[2 * t + it];
            wave_lds_fence();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const u32x2_t x = *reinterpret_cast<const u32x2_t*>(at(el, q) + 8 * eg);
              resw[2 * q] = x[0]; resw[2 * q + 1] = x[1];
            }
            wave_lds_fence();
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int i = 4 * q + e;
              const float s = acc[0][t][i];
              v[e] = fmaf(s, a.descale, bias16[i]);
              if constexpr (OUT_DT == DT_FP8 && ACT == ACT_MISH) {   // the fused form of gemm_epilogue
                constexpr float L2E = 1.4426950408889634f;
                const float nexp = __builtin_amdgcn_exp2f(fmaf(s, a.descale * L2E, bias16[i] * L2E));
                v[e] *= fmaf(fast_rcp(fmaf(nexp, nexp + 2.f, 2.f)), -2.f * a.out_scale, a.out_scale);
              } else {
                v[e] = activate(v[e]);
                if constexpr (OUT_DT == DT_FP8) v[e] *= a.out_scale;
              }
              if constexpr (HAS_RES) {
                const uint32_t rw = resw[i >> 1];
                const float r = OUT_DT == DT_F16 ? f16_bits_to_f32((uint16_t)((e & 1) ? (rw >> 16) : (rw & 0xffff)))
                                                 : __uint_as_float((e & 1) ? (rw & 0xffff0000u) : (rw << 16));
                if constexpr (EPI == DMAF_RESNORM) v[e] = fmaf(v[e], a.alpha, fmaf(r, __uint_as_float(row_st[t][0]), __uint_as_float(row_st[t][1])) * gain16[i]);
                else v[e] = fmaf(v[e], a.alpha, r);
              }
              if constexpr (OUT_DT == DT_F16) asm volatile("" : "+v"(v[e]));   // (rounded to fp32 first, as everywhere else)
            }
            if constexpr (OUT_DT == DT_FP8) {   // a 32-byte row: chunks 0 and 1
              *reinterpret_cast<uint32_t*>(at(el, q >> 1) + 8 * (q & 1) + 4 * eg) = pack_fp8x4(v[0], v[1], v[2], v[3]);
            } else {
              u32x2_t w;
              if constexpr (OUT_DT == DT_F16) {
                w[0] = (uint32_t)f32_to_f16_bits(v[0]) | ((uint32_t)f32_to_f16_bits(v[1]) << 16);
                w[1] = (uint32_t)f32_to_f16_bits(v[2]) | ((uint32_t)f32_to_f16_bits(v[3]) << 16);
              } else {
                w[0] = pack_bf16x2(v[0], v[1]);
                w[1] = pack_bf16x2(v[2], v[3]);
              }
              *reinterpret_cast<u32x2_t*>(at(el, q) + 8 * eg) = w;
            }
          }
          wave_lds_fence();
          u32x4_t o[NST];
#pragma unroll
          for (int it = 0; it < NST; ++it) o[it] = *reinterpret_cast<const u32x4_t*>(at(er + (64 / EPR) * it, ec));
          put(o, t * 32 + er, ec * CPL);
          wave_lds_fence();
        });
      }
      tile += step;
      if (tile >= hi) return;
    }
  }
}

// The rows of a tile's operands lie within the 31-bit offsets of a buffer descriptor.
inline bool dmam_reaches(const GemmArgs& a, int esz, int tile_n) {
  return (long)a.lda * esz * DmamCfg::BM < (1L << 31) && (long)a.ldw * esz * tile_n < (1L << 31);
}

template <int IN_DT, int OUT_DT, int EPI, int ACT = ACT_NONE, int TILE_N = 128>
static hipError_t launch_dmam(const GemmArgs& a, int cus, hipStream_t st) {
  static std::atomic<bool> attr_set[16] = {};
  typedef DmamCfgN<TILE_N> Cfg;
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2;
  if ((a.K * ESZ) % Cfg::ROWB != 0 || a.K <= 0 || !dmam_reaches(a, ESZ, TILE_N)) return hipErrorInvalidValue;
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto kern = gemm_dmam_kernel<IN_DT, OUT_DT, EPI, ACT, TILE_N>;
  if (dev < 0 || dev >= 16 || !attr_set[dev]) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::LDS_BYTES);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 16) attr_set[dev] = true;
  }
  const int tiles_n = (a.N + Cfg::BN - 1) / Cfg::BN, tiles_m = (a.M + Cfg::BM - 1) / Cfg::BM, tiles = tiles_m * tiles_n;
  if (tiles >= 65536) return hipErrorInvalidValue;
  const int slots = cus >= 8 ? cus & ~7 : 256;
  const int grid = EPI >= DMAF_PLAIN && tiles > slots ? slots : tiles;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(Cfg::NT), Cfg::LDS_BYTES, st, a, tiles, dmam_walk(tiles_m, tiles_n));
  return hipGetLastError();
}

}  // namespace crl
