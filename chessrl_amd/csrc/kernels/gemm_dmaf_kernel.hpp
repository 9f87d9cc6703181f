// C[M,N] = epilogue(A[M,K] . W[N,K]^T), e4m3 or 16-bit operands, K a whole number of 128-byte slabs: the 256x256 workgroup tile of
// the large products. Eight waves (two per SIMD) of 128x64 outputs, two LDS stages of 64 KB filled by direct-to-LDS loads.
//
// The two waves of a SIMD take turns: waves 0-3 (group 0) multiply while waves 4-7 (group 1) read fragments and request slabs,
// and the other way round, with a workgroup barrier at every change. A load instruction of 64 x 16 bytes holds its wave for 100
// cycles and more; with both waves of a SIMD loading first and multiplying afterwards (this kernel's earlier form) a slab took the
// load time plus the MFMA time, 1.8-2.1 us, and the matrix pipe stood still for half of it. In turns a slab of 2048 MFMA cycles
// takes 2360-2540 (e4m3, K = 16384: 2.67 -> 2.95 PFLOP/s; bf16, M = 64000, N = 3072, K = 1024: 1.02 -> 1.11).
//
// A slab is two phases. Phase 0 reads the weight fragments of the slab and the activation fragments of row blocks 0 and 1,
// phase 1 those of row blocks 2 and 3; 16 of the slab's 24 LDS rows per 8 are free after phase 0. Requests follow: phase 1 asks
// for six eighths of the slab after next (weights and row blocks 0, 1), the next phase 0 for the last two. No wait ever drains
// the queue: eight loads of a wave stay in flight across every barrier.
//
// Workgroups are persistent (one per CU) where the epilogue below exists for the call, and the stream of requested slabs runs on
// across tiles: the first slab and a half of the next tile is on its way while a tile's results are written, which took 3200
// cycles of prologue and 1800 of workgroup turnover off each tile's 29000 (e4m3, K = 1024) to 49000 (bf16). The epilogue
// therefore lives outside the ring, in 2 KB of LDS per wave: results are finished in the accumulator layout (four consecutive
// columns of one row), converted, and turned through LDS in their output type, so that a store writes 64-byte row segments
// (32-byte ones cost three times as much: 5200 against 1550 cycles per tile). A 16-bit residual takes the same way in reverse.
// The epilogue's stream is kept free of branches and of work that repeats: constants read from LDS without asking whether there are any, one branch on
// the store hint per row block (with one per store every LDS read of the turn waited for the store before it), a tile's first products added to zero
// instead of to cleared registers (M = 262144, N = 3072, K = 1024, e4m3 in, bf16 out: 723 -> 706 us; M = 64000, bf16: 322 -> 316; M = 96000, N = 3072,
// K = 768, gelu: 491 -> 483; the residual products, which wait for memory there, within 1 %).
// Stores and residual loads go through buffer descriptors that end with the tile, so ragged M and N need no branches, and every
// wave issues the same number of them, which the counted waits rely on.
//
// Same K order and same arithmetic per element as the other tiled kernels: the outputs are bit-equal.
#pragma once
#include "gemm_dma_kernel.hpp"

namespace crl {

struct DmafCfg {
  static constexpr int BM = 256, BN = 256, WGM = 2, WGN = 4, NW = 8, NT = 512;
  static constexpr int WM = 128, WN = 64, TM = 4, TN = 2;
  static constexpr int ROWB = 128, LOADS = 8, FIRST = 6;    // load instructions of a wave per slab; those of phase 1
  static constexpr int RING_BYTES = 2 * (BM + BN) * ROWB;   // 128 KB: weight rows of both stages, then activation rows
  static constexpr int PATCH_OFF = RING_BYTES, PATCH = 2048;           // a wave's patch: 32 rows of 64 bytes
  static constexpr int COLS_OFF = PATCH_OFF + NW * PATCH;              // per-column constants: [wave][bias, gain, offset][WN]
  static constexpr int LDS_BYTES = COLS_OFF + NW * 3 * WN * 4;
  static_assert(LDS_BYTES <= 160 * 1024, "LDS of a CU");
};

// The tile walk's constants, worked out once on the host: the walk divides a workgroup index by six launch constants,
// and as generic integer divisions those were most of the ~410 instructions a workgroup issued before its first load.
// q = n / d for n, d < 65536 is the high half of n * ceil(2^32 / d) (d = 1: n itself).
struct DmafWalk {
  int tiles_n, grouped, wb, extra, big;
  uint32_t m_tn, m_8tn, m_8w1, m_8w0, m_w1, m_w0;   // magics of tiles_n, 8 tiles_n, 8 (wb+1), 8 wb, wb+1, wb
};
inline uint32_t dmaf_magic(uint32_t d) { return d <= 1 ? 0u : (uint32_t)(((1ull << 32) + d - 1) / d); }
__device__ __forceinline__ int dmaf_div(int n, uint32_t magic) { return magic ? (int)__umulhi((uint32_t)n, magic) : n; }
inline DmafWalk dmaf_walk(int M, int N, bool fp8) {
  DmafWalk w{};
  const int tiles_n = (N + 255) / 256, tiles_m = (M + 255) / 256;
  w.tiles_n = tiles_n;
  // (16-bit operands keep the plain row-major order unless the columns divide by four, as in gemm_dma_kernel.hpp)
  w.grouped = tiles_m % 8 == 0 && (fp8 || tiles_n % 4 == 0);
  const int ngrp = (tiles_n + 3) >> 2;
  w.wb = tiles_n / ngrp;
  w.extra = tiles_n - w.wb * ngrp;
  w.big = 8 * (w.wb + 1) * w.extra;
  w.m_tn = dmaf_magic(tiles_n); w.m_8tn = dmaf_magic(8 * tiles_n);
  w.m_8w1 = dmaf_magic(8 * (w.wb + 1)); w.m_8w0 = dmaf_magic(8 * w.wb);
  w.m_w1 = dmaf_magic(w.wb + 1); w.m_w0 = dmaf_magic(w.wb);
  return w;
}


// What happens to the sums of a tile (all but DMAF_GENERAL persistent):
enum {
  DMAF_GENERAL = 0,       // anything: gemm_epilogue through the ring, one tile per workgroup
  DMAF_GENERAL_NORM = 1,  // the same with a residual normalised on the fly
  DMAF_PLAIN = 2,         // no residual, alpha = 1
  DMAF_RES16 = 3,         // 16-bit residual
  DMAF_RESNORM = 4,       // 16-bit residual normalised on the fly
  DMAF_RES32 = 5          // fp32 residual, fp32 output
};

template <int N>
__device__ __forceinline__ void wait_vmcnt_lgkm0() { __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4)); }
__device__ __forceinline__ void dmaf_barrier() { asm volatile("s_barrier" ::: "memory"); }
// (functions of their own, not lambdas: inside a kernel template, where an argument depends on a template parameter, the load builtin makes the host pass drop the
// kernel's stub without a diagnostic; the library then fails to load over the unresolved name, which the build checks for)
__device__ __forceinline__ void dmaf_load16(__amdgpu_buffer_rsrc_t r, uint8_t* dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void dmaf_load16_nt(__amdgpu_buffer_rsrc_t r, uint8_t* dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 2);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t dmaf_rsrc(const void* base, long span) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)(span < 0x7fffffffL ? span : 0x7fffffffL), 0x00020000);
}
// The value, in a register the compiler cannot trace back: address arithmetic built on it stays where it is written instead of
// being hoisted out of the tile loop into registers of its own.
__device__ __forceinline__ int dmaf_here(int x) {
  asm volatile("" : "+v"(x));
  return x;
}
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u32x2_t dmaf_get8(__amdgpu_buffer_rsrc_t r, int off) { return __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0); }
__device__ __forceinline__ u32x4_t dmaf_get16(__amdgpu_buffer_rsrc_t r, int off) { return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0); }
__device__ __forceinline__ u32x4_t dmaf_get16_nt(__amdgpu_buffer_rsrc_t r, int off) { return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 2); }
__device__ __forceinline__ void dmaf_put16_nt(u32x4_t v, __amdgpu_buffer_rsrc_t r, int off) { __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, 2); }
__device__ __forceinline__ void dmaf_put16(u32x4_t v, __amdgpu_buffer_rsrc_t r, int off) { __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, 0); }

// The 1 to 3 columns of a 16-byte chunk that a ragged row still has (have; otherwise nothing is stored).
__device__ __forceinline__ void dmaf_put_part(u32x4_t v, __amdgpu_buffer_rsrc_t r, int off, int have) {
#pragma unroll
  for (int e = 0; e < 3; ++e) __builtin_amdgcn_raw_buffer_store_b32(v[e], r, e < have && have < 4 ? off + 4 * e : (int)0x80000000u, 0, 0);
}

template <int IN_DT, int OUT_DT, int EPI, int ACT = ACT_NONE>
__global__ void __launch_bounds__(DmafCfg::NT, 2) gemm_dmaf_kernel(const GemmArgs a, const DmafWalk wk, const int tiles) {
  typedef DmafCfg Cfg;
  constexpr bool PERSIST = EPI >= DMAF_PLAIN;
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2;                      // bytes per operand element
  constexpr int OSZ = OUT_DT == DT_F32 ? 4 : OUT_DT == DT_FP8 ? 1 : 2;
  constexpr int KSTEPS = Cfg::ROWB / (IN_DT == DT_FP8 ? 64 : 32);   // MFMA K steps per slab
  constexpr int BM = Cfg::BM, BN = Cfg::BN, TM = Cfg::TM, TN = Cfg::TN, LOADS = Cfg::LOADS, FIRST = Cfg::FIRST;
  extern __shared__ __align__(16) uint8_t smem[];

  // (the wave index as a scalar: everything derived from it, LDS destinations and descriptors, stays in scalar registers)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % Cfg::WGM, wn = wave / Cfg::WGM, grp = wave >> 2;
  const int lr = lane & 31, g = lane >> 5;
  const int nslab = a.K * ESZ / Cfg::ROWB;  // the launcher sends only whole slabs of K here

  // Workgroup b runs on XCD b & 7, which owns a contiguous range of the tile order. With fewer workgroups than tiles (a
  // multiple of eight then) an XCD's workgroups take its tiles in turn.
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

  // Tiles are walked from the last row of tiles to the first. The kernels around a product (norms, attention) walk their
  // rows upwards, so this product starts on the rows its producer wrote last and ends on the rows its consumer reads first,
  // which are the ones the memory-side cache still holds (measured on a 4096-position pass: -0.4 ms over its 60 launches).
  // Inside an XCD's range: groups of 8 x w tiles (M x N), w = 3 or 4, as in gemm_dma_kernel.hpp.
  auto tile_pos = [&](int t, int& tm, int& tn) {
    const int pid = tiles - 1 - t;
    if (wk.grouped) {
      constexpr int GM = 8;
      const int sr = dmaf_div(pid, wk.m_8tn), rem = pid - sr * (GM * wk.tiles_n);
      int gi, r2, rq, gw;
      if (rem < wk.big) { gw = wk.wb + 1; gi = dmaf_div(rem, wk.m_8w1); r2 = rem - gi * GM * gw; rq = dmaf_div(r2, wk.m_w1); tn = gi * gw; }
      else { gw = wk.wb; const int rem2 = rem - wk.big; gi = dmaf_div(rem2, wk.m_8w0); r2 = rem2 - gi * GM * gw; rq = dmaf_div(r2, wk.m_w0); tn = (gi + wk.extra) * gw + wk.extra; }
      tm = sr * GM + rq;
      tn += r2 - rq * gw;
    } else {
      tm = dmaf_div(pid, wk.m_tn);
      tn = pid - tm * wk.tiles_n;
    }
  };

  // ---- the stream of requested slabs (l_*: where it stands; it runs up to two slabs ahead, across tiles)
  // Load i of a wave, 8 rows of 128 bytes: weight rows 32 wave + 8 i (i < 4); activation rows 16 (wave & 3) + 8 (i & 1) of
  // the 64 that row blocks 0, 1 (i = 4, 5) or 2, 3 (i = 6, 7) of wave row wave / 4 have. The swizzle is applied on the global side.
  uint32_t voff[LOADS];
  __amdgpu_buffer_rsrc_t rsrc_w, rsrc_x;
  const int ldab = (int)a.lda * ESZ, ldwb = (int)a.ldw * ESZ;
  int l_tile = tile, l_slab = 0;
  uint32_t l_stage = 0;
  auto stream_tile = [&]() {
    int tm, tn;
    tile_pos(l_tile, tm, tn);
    const int ln = dmaf_here(lane);
    const int m0 = tm * BM, n0 = tn * BN, leftx = a.M - m0, leftw = a.N - n0, l8 = ln >> 3;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int r = i >= 4 ? (wave >> 2) * 128 + (wave & 3) * 16 + ((i & 2) ? 64 : 0) + 8 * (i & 1) + l8 : wave * 32 + 8 * i + l8;
      const int sw = l8 ^ ((i >= 4 ? 2 * (wave & 3) + (i & 1) : 4 * (wave & 1) + i) & 7);
      const int left = i >= 4 ? leftx : leftw;
      r = r < left ? r : left - 1;
      voff[i] = (uint32_t)r * (uint32_t)(i >= 4 ? ldab : ldwb) + (((ln & 7) ^ sw) << 4);
    }
    rsrc_w = dmaf_rsrc(reinterpret_cast<const uint8_t*>(a.W) + (long)n0 * ldwb, (long)(leftw < 256 ? leftw : 256) * ldwb);
    rsrc_x = dmaf_rsrc(reinterpret_cast<const uint8_t*>(a.A) + (long)m0 * ldab, (long)(leftx < 256 ? leftx : 256) * ldab);
  };
  auto issue = [&](auto ic) {
    constexpr int i = decltype(ic)::value;
    const uint32_t d = i >= 4 ? 65536u + ((wave >> 2) * 128 + (wave & 3) * 16 + ((i & 2) ? 64 : 0) + 8 * (i & 1)) * 128u : (wave * 32 + 8 * i) * 128u;
    dmaf_load16(i >= 4 ? rsrc_x : rsrc_w, smem + (d ^ l_stage), (int)voff[i], l_slab * Cfg::ROWB);
  };
  auto request_first = [&]() {   // weights and row blocks 0, 1 of the stream's next slab
    if (l_slab == nslab) {
      l_slab = 0;
      l_tile += step;
      if (PERSIST && l_tile < hi) stream_tile();
      else rsrc_w = rsrc_x = dmaf_rsrc(a.A, 0);   // past the end: loads that move nothing keep the counts
    }
    static_for<0, FIRST>(issue);
  };
  auto request_rest = [&]() {    // its row blocks 2, 3
    static_for<FIRST, LOADS>(issue);
    ++l_slab;
    l_stage ^= 32768u;
  };
  stream_tile();
  request_first();
  request_rest();
  request_first();
  __builtin_amdgcn_sched_barrier(0);

  int tm0, tn0;
  tile_pos(tile, tm0, tn0);
  int m0 = tm0 * BM, n0 = tn0 * BN;
  // The per-column constants of the epilogue (bias; gain and offset of a residual normalised on the fly) for this wave's
  // 64 columns, one column per lane. Columns past N repeat the last one; nothing of theirs is stored.
  auto load_cols = [&]() {
    int n = n0 + wn * Cfg::WN + lane;
    n = n < a.N ? n : a.N - 1;
    uint8_t* cols = smem + Cfg::COLS_OFF + wave * (3 * Cfg::WN * 4);
    if (a.bias)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a.bias + n), (__attribute__((address_space(3))) void*)cols, 4, 0, 0);
    else if constexpr (PERSIST)
      reinterpret_cast<float*>(cols)[lane] = 0.f;   // (so that the epilogue reads the constants without asking)
    if constexpr (EPI == DMAF_RESNORM || EPI == DMAF_GENERAL_NORM) {
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a.res_gamma + n),
                                       (__attribute__((address_space(3))) void*)(cols + Cfg::WN * 4), 4, 0, 0);
      if (a.res_beta)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(a.res_beta + n),
                                         (__attribute__((address_space(3))) void*)(cols + 2 * Cfg::WN * 4), 4, 0, 0);
    }
  };

  f32x16_t acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // Fragment addresses. A lane's 16-byte piece of row 32 t + lr of a wave's block sits at chunk c ^ swizzle(row) with
  // c = 4 ks + half + 2g for e4m3 (two pieces per K step of 64 bytes) and c = 2 ks + g for 16-bit operands (one piece
  // per K step of 32 bytes), and swizzle(row) = swizzle(lr) ^ 4 (t & 1). With L = (2g or g) ^ swizzle(lr) the chunk is
  // Kc ^ L for a compile-time Kc that takes four values (0, 1, 4, 5 or 0, 2, 4, 6): four lane addresses per operand
  // plus the immediate 4096 t cover every read of a stage. A stage is bit 15 of an address.
  const int L0 = (IN_DT == DT_FP8 ? 2 * g : g) ^ lds_swizzle(lr);
  const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)smem);
  uint32_t wb[4], xb[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int kc = IN_DT == DT_FP8 ? ((k & 1) | ((k >> 1) << 2)) : 2 * k;
    wb[k] = lds0 + (wn * Cfg::WN + lr) * Cfg::ROWB + ((kc ^ L0) << 4);
    xb[k] = lds0 + 65536 + (wm * Cfg::WM + lr) * Cfg::ROWB + ((kc ^ L0) << 4);
  }
  auto lds_piece = [](uint32_t addr) -> i32x4_t { return *reinterpret_cast<const __attribute__((address_space(3))) i32x4_t*>(addr); };
  auto read_piece = [&](const uint32_t (&b)[4], int t, int ks, int half) -> i32x4_t {
    const int kc = (IN_DT == DT_FP8 ? 4 * ks + half : 2 * ks) ^ (4 * (t & 1));
    const int k = IN_DT == DT_FP8 ? ((kc & 1) | ((kc >> 2) << 1)) : kc >> 1;
    return lds_piece(b[k] + t * 32 * Cfg::ROWB);
  };
  auto read_frag = [&](const uint32_t (&b)[4], int t, auto ksc) {
    constexpr int ks = decltype(ksc)::value;
    Frag<IN_DT> f;
    f.lo = read_piece(b, t, ks, 0);
    if constexpr (IN_DT == DT_FP8) f.hi = read_piece(b, t, ks, 1);
    return f;
  };
  Frag<IN_DT> wf[KSTEPS][TN], xf[KSTEPS][2];

  // A wave whose 128x64 part lies wholly outside C still takes its share of the loads and every barrier.
  bool wave_active = (m0 + wm * Cfg::WM < a.M) && (n0 + wn * Cfg::WN < a.N);

  auto read_phase = [&](auto pc) {
    constexpr int p = decltype(pc)::value;
    static_for<0, KSTEPS>([&](auto ksc) {
      constexpr int ks = decltype(ksc)::value;
      if constexpr (p == 0) {
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) wf[ks][tn] = read_frag(wb, tn, ksc);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) xf[ks][t] = read_frag(xb, 2 * p + t, ksc);
    });
  };
  // (fresh: a tile's first slab, whose products are added to zero instead of to the sums, so that no tile has to clear 128 registers of a lane)
  auto multiply_phase = [&](auto pc, bool fresh) {
    constexpr int p = decltype(pc)::value;
    auto multiply = [&](auto fc) {
      static_for<0, KSTEPS>([&](auto ksc) {
        constexpr int ks = decltype(ksc)::value;
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            if constexpr (decltype(fc)::value && ks == 0) acc[tn][2 * p + t] = mfma_frag<IN_DT>(wf[ks][tn], xf[ks][t], f32x16_t{});
            else acc[tn][2 * p + t] = mfma_frag<IN_DT>(wf[ks][tn], xf[ks][t], acc[tn][2 * p + t]);
          }
      });
    };
    __builtin_amdgcn_sched_barrier(0);
    dmaf_barrier();
    __builtin_amdgcn_s_setprio(1);
    if (wave_active) {
      if (fresh) multiply(std::true_type{});
      else multiply(std::false_type{});
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
  };
  typedef std::integral_constant<int, 0> P0;
  typedef std::integral_constant<int, 1> P1;

  // ---- epilogue of the persistent instances
  // Accumulator layout: acc[tn][tm][4 q + e] is row 32 tm + lr, column 32 tn + 8 q + 4 g + e of the wave's 128x64 part.
  // Store layout (16 bytes per lane): rows er + 8 it of a row block, 16-byte chunk ec of a 128-byte row segment (e4m3: rows
  // er + 16 it, chunk ec of a 64-byte one). A wave's patch is two halves of 32 rows of 64 bytes, column blocks 0 and 1: its own
  // 2 KB and 2 KB of the ring, row blocks 2 and 3 of the last slab's stage, which nothing is requested into until every wave is
  // through with its epilogue. 16-byte chunks are swizzled over groups of four rows (256 bytes are one pass of all banks).
  constexpr int EPR = OUT_DT == DT_FP8 ? 4 : 8, ITS = 32 * EPR / 64;   // lanes per row, store instructions per row block
  constexpr bool HAS_RES = EPI == DMAF_RES16 || EPI == DMAF_RESNORM || EPI == DMAF_RES32;
  constexpr int RSZ = EPI == DMAF_RES32 ? 4 : 2;
  // A step of the epilogue: a row block (its 64 columns), with fp32 outputs the half of one, 32 columns.
  constexpr int NSTEP = OUT_DT == DT_F32 ? 2 * TM : TM;
  uint8_t* const patch0 = smem + Cfg::PATCH_OFF + wave * Cfg::PATCH;
  const float* const cols = reinterpret_cast<const float*>(smem + Cfg::COLS_OFF) + wave * (3 * Cfg::WN);
  u32x4_t res[HAS_RES ? 2 : 1][ITS];        // residual of the next two steps
  u32x2_t row_st[EPI == DMAF_RESNORM ? 2 : 1];   // 1/std and -mean/std of the lane's row in them
  __amdgpu_buffer_rsrc_t rsrc_r = dmaf_rsrc(a.A, 0);
  int vres = 0, res_step = 0;
  auto res_begin = [&]() {
    const int ln = dmaf_here(lane);
    const int rows = a.M - m0 < BM ? a.M - m0 : BM, left = a.N - n0 < BN ? a.N - n0 : BN;
    res_step = (int)a.ldr * RSZ;
    rsrc_r = dmaf_rsrc(reinterpret_cast<const char*>(a.res) + (long)m0 * res_step + (long)n0 * RSZ, (long)(rows - 1) * res_step + (long)left * RSZ);
    vres = (wm * Cfg::WM + ln / EPR) * res_step + wn * Cfg::WN * RSZ + (ln % EPR) * 16;
  };
  auto res_load = [&](auto sc) {
    constexpr int st = decltype(sc)::value, tm = st % TM, half = st / TM;
    if constexpr (HAS_RES && st < NSTEP) {
      // (fp32 rows go past the caches where the output does, by the launcher's rule; 768 columns, K = 768, back to back, with and without the
      // hint: 96000 rows 173 and 191 us, 32768 rows, which the memory-side cache holds, 70 and 60)
      if (OUT_DT != DT_F32 || a.stream_out != 0) {
#pragma unroll
        for (int it = 0; it < ITS; ++it) res[st & 1][it] = dmaf_get16_nt(rsrc_r, vres + half * 128 + (tm * 32 + it * (64 / EPR)) * res_step);
      } else {
#pragma unroll
        for (int it = 0; it < ITS; ++it) res[st & 1][it] = dmaf_get16(rsrc_r, vres + half * 128 + (tm * 32 + it * (64 / EPR)) * res_step);
      }
      if constexpr (EPI == DMAF_RESNORM)
        row_st[st & 1] = dmaf_get8(dmaf_rsrc(a.res_stats + 2 * (long)m0, (long)(a.M - m0) * 8), (wm * Cfg::WM + tm * 32 + (dmaf_here(lane) & 31)) * 8);
    }
  };
  auto activate = [&](float v) -> float {
    if constexpr (ACT == ACT_GELU) return act_gelu(v);
    else if constexpr (ACT == ACT_MISH) return act_mish(v);
    else return v;
  };
  // e4m3(out_scale * mish(x)) in the fused form of gemm_epilogue
  auto mish8 = [&](float accv, float bias, float v) -> float {
    constexpr float L2E = 1.4426950408889634f;
    const float nexp = __builtin_amdgcn_exp2f(fmaf(accv, a.descale * L2E, bias * L2E));
    return v * fmaf(fast_rcp(fmaf(nexp, nexp + 2.f, 2.f)), -2.f * a.out_scale, a.out_scale);
  };
  auto epilogue = [&](uint32_t last_stage) {
    const int ln = dmaf_here(lane), er = ln / EPR, ec = ln % EPR, lr = ln & 31, g = ln >> 5;
    const bool first = n0 < a.nsplit;      // (a tile lies on one side of the split: the launcher checks)
    const int ldob = (int)(first ? a.ldc : a.ldc2) * OSZ, rows = a.M - m0 < BM ? a.M - m0 : BM;
    int left = (first ? a.nsplit : a.N) - n0;
    left = left < BN ? left : BN;
    const __amdgpu_buffer_rsrc_t rsrc_o = dmaf_rsrc(reinterpret_cast<char*>(first ? a.C : a.C2) + (long)m0 * ldob + (long)(first ? n0 : n0 - a.nsplit) * OSZ,
                                                    (long)(rows - 1) * ldob + (long)left * OSZ);
    const int vout = (wm * Cfg::WM + er) * ldob + wn * Cfg::WN * OSZ + ec * 16;
    constexpr int NOWHERE = (int)0x80000000u;
    const bool nt = a.stream_out != 0 && (OUT_DT != DT_F32 || ldob % 128 == 0);   // (part of a line with the hint takes three times as long)
    // A row block's stores, off + it * step: one branch on the hint for all of them. With a branch at each store the LDS read in
    // front of it could not start before the store of the one before had been issued.
    auto put = [&](const u32x4_t (&v)[ITS], int off, int step) {
      if (nt) {
#pragma unroll
        for (int it = 0; it < ITS; ++it) dmaf_put16_nt(v[it], rsrc_o, off + it * step);
      } else {
#pragma unroll
        for (int it = 0; it < ITS; ++it) dmaf_put16(v[it], rsrc_o, off + it * step);
      }
    };
    uint8_t* const patch1 = smem + 65536 + last_stage + (wave >> 2) * 16384 + 8192 + (wave & 3) * 2048;
    auto at = [&](uint8_t* half, int r, int c) -> uint8_t* { return half + r * 64 + ((c ^ ((r >> 2) & 3)) << 4); };
    // this lane's chunk of row er + 8 it in the store layout
    uint8_t* const mine = ec < 4 ? patch0 : patch1;
    auto turned = [&](u32x4_t (&v)[ITS]) {
#pragma unroll
      for (int it = 0; it < ITS; ++it) v[it] = *reinterpret_cast<const u32x4_t*>(at(mine, er + it * (64 / EPR), ec & 3));
    };
    auto col_const = [&](const float* c, int base, float (&o)[16]) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(c + base + 8 * q + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[4 * q + e] = v[e];
      }
    };
    if constexpr (EPI == DMAF_RESNORM) {   // the residual norm's offset joins the bias (which is multiplied by alpha), once per column
      if (a.res_beta) {
        float* const c = const_cast<float*>(cols) + ln;
        *c = fmaf(c[2 * Cfg::WN], 1.0f / a.alpha, *c);
        wave_lds_fence();
      }
    }
    if constexpr (OUT_DT == DT_FP8) {
      const int v0 = wn * Cfg::WN + ec * 16 < left ? vout : NOWHERE;
      float bias16[2][16];
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) col_const(cols, tn * 32, bias16[tn]);
      static_for<0, TM>([&](auto tmc) {
        constexpr int tm = decltype(tmc)::value;
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float s = acc[tn][tm][4 * q + e];
              v[e] = fmaf(s, a.descale, bias16[tn][4 * q + e]);
              if constexpr (ACT == ACT_MISH) v[e] = mish8(s, bias16[tn][4 * q + e], v[e]);
              else v[e] = activate(v[e]) * a.out_scale;
            }
            *reinterpret_cast<uint32_t*>(at(patch0, lr, 2 * tn + (q >> 1)) + 8 * (q & 1) + 4 * g) = pack_fp8x4(v[0], v[1], v[2], v[3]);
          }
        wave_lds_fence();
        u32x4_t o[ITS];
        turned(o);
        put(o, v0 + tm * 32 * ldob, 16 * ldob);
        wave_lds_fence();
      });
    } else if constexpr (OUT_DT == DT_F32) {
      // Raw sums through the patch, 32 columns at a time; bias, activation and residual in the store layout (4 columns per lane).
      // Without a residual the rows may have any length (16-byte stores need 4-byte alignment only): the 1929 logits of 32768 rows,
      // K = 768, took 260 us through the general epilogue and 128 here.
      static_for<0, NSTEP>([&](auto sc) {
        constexpr int st = decltype(sc)::value, tn = st / TM, tm = st % TM;
        const int have = left - (wn * Cfg::WN + tn * 32 + ec * 4);
        const int v0 = have >= (HAS_RES ? 1 : 4) ? vout + tn * 128 : NOWHERE;
        const f32x4_t bv = *reinterpret_cast<const f32x4_t*>(cols + tn * 32 + ec * 4);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<f32x4_t*>(at(q < 2 ? patch0 : patch1, lr, 2 * (q & 1) + g)) = f32x4_t{acc[tn][tm][4 * q], acc[tn][tm][4 * q + 1], acc[tn][tm][4 * q + 2], acc[tn][tm][4 * q + 3]};
        wave_lds_fence();
        u32x4_t o[ITS];
        turned(o);
#pragma unroll
        for (int it = 0; it < ITS; ++it)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v = activate(fmaf(__uint_as_float(o[it][e]), a.descale, bv[e]));
            if constexpr (HAS_RES) v = fmaf(v, a.alpha, __uint_as_float(res[st & 1][it][e]));
            o[it][e] = __float_as_uint(v);
          }
        put(o, v0 + tm * 32 * ldob, 8 * ldob);
        if constexpr (!HAS_RES) {
          if (left & 3)
#pragma unroll
            for (int it = 0; it < ITS; ++it) dmaf_put_part(o[it], rsrc_o, vout + tn * 128 + (tm * 32 + it * 8) * ldob, have);
        }
        wave_lds_fence();
        res_load(std::integral_constant<int, st + 2>{});
      });
    } else {
      const int v0 = wn * Cfg::WN + ec * 8 < left ? vout : NOWHERE;
      static_for<0, NSTEP>([&](auto sc) {
        constexpr int tm = decltype(sc)::value;
        if constexpr (HAS_RES) {   // the residual from the store layout to the accumulator layout
#pragma unroll
          for (int it = 0; it < ITS; ++it) *reinterpret_cast<u32x4_t*>(at(mine, er + it * 8, ec & 3)) = res[tm & 1][it];
          wave_lds_fence();
        }
        float st0 = 0.f, st1 = 0.f;
        if constexpr (EPI == DMAF_RESNORM) { st0 = __uint_as_float(row_st[tm & 1][0]); st1 = __uint_as_float(row_st[tm & 1][1]); }
        res_load(std::integral_constant<int, tm + 2>{});
        static_for<0, TN>([&](auto tc) {
          constexpr int tn = decltype(tc)::value;
          uint8_t* const half = tn ? patch1 : patch0;
          uint32_t resw[8];
          if constexpr (HAS_RES) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const u32x2_t x = *reinterpret_cast<const u32x2_t*>(at(half, lr, q) + 8 * g);
              resw[2 * q] = x[0]; resw[2 * q + 1] = x[1];
            }
          }
          float bias16[16], gain16[16];
          col_const(cols, tn * 32, bias16);
          if constexpr (EPI == DMAF_RESNORM) col_const(cols + Cfg::WN, tn * 32, gain16);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int i = 4 * q + e;
              v[e] = activate(fmaf(acc[tn][tm][i], a.descale, bias16[i]));
              if constexpr (HAS_RES) {
                const uint32_t rw = resw[i >> 1];
                const float r = OUT_DT == DT_F16 ? f16_bits_to_f32((uint16_t)((e & 1) ? (rw >> 16) : (rw & 0xffff)))
                                                 : __uint_as_float((e & 1) ? (rw & 0xffff0000u) : (rw << 16));
                if constexpr (EPI == DMAF_RESNORM)
                  v[e] = fmaf(v[e], a.alpha, fmaf(r, st0, st1) * gain16[i]);
                else
                  v[e] = fmaf(v[e], a.alpha, r);
              }
              // (a multiply-add that rounds straight to f16 would skip the rounding to fp32 that the other tiles' epilogues make)
              if constexpr (OUT_DT == DT_F16) asm volatile("" : "+v"(v[e]));
            }
            u32x2_t w;
            if constexpr (OUT_DT == DT_F16) {
              w[0] = (uint32_t)f32_to_f16_bits(v[0]) | ((uint32_t)f32_to_f16_bits(v[1]) << 16);
              w[1] = (uint32_t)f32_to_f16_bits(v[2]) | ((uint32_t)f32_to_f16_bits(v[3]) << 16);
            } else {
              w[0] = pack_bf16x2(v[0], v[1]);
              w[1] = pack_bf16x2(v[2], v[3]);
            }
            *reinterpret_cast<u32x2_t*>(at(half, lr, q) + 8 * g) = w;
          }
        });
        wave_lds_fence();
        u32x4_t o[ITS];
        turned(o);
        put(o, v0 + tm * 32 * ldob, 8 * ldob);
        wave_lds_fence();
      });
    }
  };
  // Stores an epilogue issues behind its last load (a wave waits past them for the slabs requested before).
  constexpr int ESTORES = PERSIST ? NSTEP * ITS : 0;
  constexpr int INFLIGHT = LOADS;   // FIRST of the slab after next and LOADS - FIRST of the next one

  wait_vmcnt<INFLIGHT>();
  dmaf_barrier();
  uint32_t r_stage = 0;   // stage of the slab being read
  bool later = false;   // a tile before this one has left stores in flight
  for (;;) {
    if (grp) dmaf_barrier();   // group 1 runs one phase behind
    for (int slab = 0; slab < nslab; ++slab) {
      const bool last = slab + 1 == nslab;
      read_phase(P0{});
      __builtin_amdgcn_sched_barrier(0);
      request_rest();
      if (slab == 0) load_cols();
      __builtin_amdgcn_sched_barrier(0);
      // Row blocks 2, 3 of this slab: requested before the last INFLIGHT loads (and before the previous tile's stores).
      if (slab == 0 && later) wait_vmcnt_lgkm0<INFLIGHT + ESTORES>();
      else wait_vmcnt_lgkm0<INFLIGHT>();
      multiply_phase(P0{}, PERSIST && slab == 0);
      dmaf_barrier();
      __builtin_amdgcn_sched_barrier(0);
      read_phase(P1{});
      __builtin_amdgcn_sched_barrier(0);
      request_first();
      r_stage ^= 32768u;
#pragma unroll
      for (int k = 0; k < 4; ++k) { wb[k] ^= 32768u; xb[k] ^= 32768u; }
      if constexpr (HAS_RES) {
        if (last) { res_begin(); res_load(P0{}); }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (!PERSIST && last) wait_vmcnt_lgkm0<0>();   // (the ring becomes epilogue scratch)
      else if (slab == 0 && later) wait_vmcnt_lgkm0<INFLIGHT + ESTORES>();
      else if (HAS_RES && last) wait_vmcnt_lgkm0<INFLIGHT + ITS + (EPI == DMAF_RESNORM ? 1 : 0)>();
      else wait_vmcnt_lgkm0<INFLIGHT>();
      multiply_phase(P1{}, PERSIST && slab == 0);
      if (!(last && grp)) dmaf_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!PERSIST) break;
    res_load(P1{});
    epilogue(r_stage ^ 32768u);
    tile += step;
    if (tile >= hi) break;
    tile_pos(tile, tm0, tn0);
    m0 = tm0 * BM; n0 = tn0 * BN;
    wave_active = (m0 + wm * Cfg::WM < a.M) && (n0 + wn * Cfg::WN < a.N);
    later = true;
    dmaf_barrier();
  }
  if constexpr (!PERSIST) {
    // (every wave's ring reads and loads are behind the last barrier of group 0 and the last but one of group 1)
    gemm_epilogue<Cfg::WM, Cfg::WN, OUT_DT, EPI == DMAF_GENERAL_NORM ? 1 : 0, 0>(a, acc, reinterpret_cast<float*>(smem) + wave * (32 * Cfg::WN),
                                                     m0 + wm * Cfg::WM, n0 + wn * Cfg::WN, lane,
                                                     reinterpret_cast<float*>(smem + 65536) + wave * (2 * Cfg::WM), cols);
  } else {
    wait_vmcnt<0>();   // no load to LDS outlives its workgroup
  }
}

// Which instance serves a call. 0 / 1: the general ones.
inline int dmaf_epilogue(const GemmArgs& a, int in_dt, int out_dt, int tile_cols = DmafCfg::BN) {
  // (fp32 rows without a residual: any length, see the epilogue)
  if (out_dt == DT_F32 && !a.res && !a.res_stats && a.alpha == 1.f && a.act == ACT_NONE && a.nsplit >= a.N && !a.amax && !a.ln_out && a.res_rows == 0 &&
      (in_dt == DT_BF16 || in_dt == DT_FP8) && (long)a.K * (in_dt == DT_FP8 ? 1 : 2) >= 2 * DmafCfg::ROWB && a.ldc * 4 * 256 < (1L << 31))
    return DMAF_PLAIN;
  const int general = a.res_stats ? DMAF_GENERAL_NORM : DMAF_GENERAL, osz = out_dt == DT_F32 ? 4 : out_dt == DT_FP8 ? 1 : 2;
  // 16-byte stores of whole column groups inside one tile, offsets inside a tile that fit 31 bits, two slabs at least (the
  // constants of a tile land during its second slab)
  if (!a.vec_ok || a.N % (out_dt == DT_FP8 ? 16 : 8) || (a.nsplit < a.N && a.nsplit % tile_cols) || a.amax || a.res_rows > 0 || a.ln_out) return general;
  if ((long)a.K * (in_dt == DT_FP8 ? 1 : 2) < 2 * DmafCfg::ROWB) return general;
  if (a.ldc * osz * 256 >= (1L << 31) || a.ldc2 * osz * 256 >= (1L << 31) || (a.res && a.ldr * 4 * 256 >= (1L << 31)) || a.ldc < a.nsplit) return general;
  if (a.res_stats) return a.act == ACT_NONE && out_dt == DT_BF16 ? DMAF_RESNORM : general;
  if (!a.res) {
    if (a.alpha != 1.f || out_dt == DT_F32) return general;
    if (out_dt == DT_FP8) return a.act == ACT_MISH || a.act == ACT_GELU ? DMAF_PLAIN : general;
    return a.act == ACT_NONE || a.act == ACT_MISH || (a.act == ACT_GELU && out_dt == DT_BF16 && in_dt == DT_BF16) ? DMAF_PLAIN : general;
  }
  if (out_dt == DT_F32) return a.res_dtype == DT_F32 && a.act == ACT_NONE ? DMAF_RES32 : general;
  if (out_dt == DT_FP8 || a.res_dtype != out_dt) return general;
  return a.act == ACT_NONE || (a.act == ACT_GELU && out_dt == DT_BF16 && in_dt == DT_BF16) ? DMAF_RES16 : general;
}

template <int IN_DT, int OUT_DT, int EPI, int ACT = ACT_NONE>
static hipError_t launch_dmaf(const GemmArgs& a, int cus, hipStream_t st) {
  static std::atomic<bool> attr_set[16] = {};
  hipError_t e = hipSuccess;
  // Whole slabs of K only, and lane offsets inside a tile's 256 rows that fit 31 bits.
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2;
  if ((a.K * ESZ) % DmafCfg::ROWB != 0 || a.K <= 0 || (long)a.lda * ESZ * 256 >= (1L << 31) || (long)a.ldw * ESZ * 256 >= (1L << 31)) return hipErrorInvalidValue;
  int dev = 0;
  (void)hipGetDevice(&dev);
  auto kern = gemm_dmaf_kernel<IN_DT, OUT_DT, EPI, ACT>;
  constexpr int LDS = DmafCfg::LDS_BYTES;
  if (dev < 0 || dev >= 16 || !attr_set[dev]) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return e;
    if (dev >= 0 && dev < 16) attr_set[dev] = true;
  }
  const int tiles_n = (a.N + DmafCfg::BN - 1) / DmafCfg::BN;
  const int tiles = ((a.M + DmafCfg::BM - 1) / DmafCfg::BM) * tiles_n;
  if (tiles >= 65536) return hipErrorInvalidValue;   // (the walk's divisions are exact below that; the caller has another kernel)
  // One workgroup per CU walks the tiles (a multiple of eight, so that every XCD has its share), or one per tile.
  const int slots = cus >= 8 ? cus & ~7 : 256;
  const int grid = EPI >= DMAF_PLAIN && tiles > slots ? slots : tiles;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(DmafCfg::NT), LDS, st, a, dmaf_walk(a.M, a.N, IN_DT == DT_FP8), tiles);
  return hipGetLastError();
}

}  // namespace crl
