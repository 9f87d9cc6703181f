// C[M,N] = act(descale * norm(X)[M,K] · W[N,K]^T + bias): a LayerNorm (or RMSNorm) of fp32 or 16-bit rows of K <= 1024 columns and the product that
// reads it as one launch, for products so small that every tile of 16 or 32 rows has a CU of its own (GPT and the post-norm trunks on one to a few
// positions, the token steps of generation). There a norm is a launch of 4 us around a handful of rows. Here every workgroup normalises
// its rows itself: sixteen waves take one or two rows each, requested before anything is waited for, the workgroup's weight rows
// follow straight to LDS, and the normalised rows go to LDS as the operand. With both operands whole in LDS (at most
// 150 KB) there is no ring; one barrier stands between gain and offset and their use, one between the operands and the product.
// Bound by the norm's own vector instructions, which every tile column repeats (four waves share a SIMD: 70 of them for a row's statistics are 1300 cycles), by the CU's
// load rate before them (every wave's requests are issued after 2600 of 9000 cycles) and by the chain of a tile's MFMAs behind (1600). Hence 16 rows where the columns
// then still fit: one position, K = 768, N = 2304 and 3072: 32x32 tiles 11100 cycles, 16x40 and 16x48 10400 and 10800, with 16x16x32 MFMAs 9000 and 9400; the last layer's one row
// 10800, 9600 and 8000; vocabulary 10800, 9000, 7500 (whole call 186.0 -> 182.3 us, 171.0 -> 163.7).
// One counted wait behind the last request lets the statistics run under the weight loads; the normalised rows wait for
// them all the same, because the compiler drains every load into LDS in front of the first write to it. Measured in place: K = 768, N = 2304, 128 rows 8.4 us (12.4 for the norm riding on the K-sliced product before it and the
// product), 64 rows 7.3 us (8.5 for two launches). 16-bit rows of 1024 columns (BT4-class, one position, tiles
// of 16 rows, N = 3104 and 1536) 7.3 us on average inside the call, two launches 8.2 and the gap of 1.2 between them (whole call 659 -> 621). Taken back: the weights requested behind a barrier, so
// that no wave's rows queue behind another's weights, LDS writes that do not wait for the weights, 16-bit rows straight to LDS (each wave then waits for all the others first): one
// position 621 -> 637 us for the call.
// The norm's arithmetic is that of layernorm_kernel row by row and the product adds K in the order of the other tiled kernels: bit-equal to
// the two launches.
#pragma once
#include "gemm_dmaf_kernel.hpp"
#include "norm_rows.hpp"

namespace crl {

struct NormGemmKArgs {
  NormGemmArgs a;
  int nslab, tiles_m;
  uint32_t m_tm, m_bn2;        // magics of tiles_m and bn / 2
  int per_xcd;
  int bn;                      // columns of a tile, a multiple of eight
  int w_div, w_mod, loads;     // 16 / (bn / 8) and 16 % (bn / 8); weight requests of a wave
};

template <int N>
__device__ __forceinline__ void norm_wait(int loads) {   // all requests but the last `loads` (uniform, at most N) are there
  if constexpr (N > 0) {
    if (loads == N) wait_vmcnt_lgkm0<N>();
    else norm_wait<N - 1>(loads);
  } else {
    wait_vmcnt_lgkm0<0>();
  }
}

// X16: the rows are of the operands' 16-bit type, whole groups of 512 columns, and the normalised ones are also left in memory (by the first tile column).
template <int IN_DT, int BM, bool X16>
__global__ void __launch_bounds__(1024) gemm_norm_kernel(const NormGemmKArgs s) {
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2, ROWB = 128, RW = BM / 16;   // rows of X that a wave normalises
  constexpr int KSTEPS = ROWB / (IN_DT == DT_FP8 ? 64 : 32);
  const int bn = s.bn;
  extern __shared__ __align__(16) uint8_t smem[];
  const NormGemmArgs& a = s.a;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nslab = s.nslab;
  // Workgroup b runs on XCD b & 7, which owns a contiguous range of the column-major tile order: the tiles that share weight rows sit together.
  int pid = blockIdx.x;
  if (pid < (s.per_xcd << 3)) pid = (pid & 7) * s.per_xcd + (pid >> 3);
  const int tile_n = dmaf_div(pid, s.m_tm), tile_m = pid - tile_n * s.tiles_m;
  const int m0 = tile_m * BM, n0 = tile_n * bn;
  uint8_t* const lds_w = smem;                                   // [slab][bn rows][128 bytes]
  uint8_t* const lds_a = smem + nslab * bn * ROWB;               // [slab][BM rows][128 bytes]

  float* const lds_g = reinterpret_cast<float*>(lds_a + nslab * BM * ROWB);   // [K] gain, then [K] offset

  // ---- rows of X: wave w takes rows RW w and on. A lane's 16 columns are those of layernorm_kernel (norm_columns).
  const int C = a.K;
  float x[RW][2][8];
  i32x4_t raw[RW][2];
  auto has = [&](int i, int h) { return (X16 ? i * 512 : (2 * i + h) * 256) < C; };   // (whole groups of columns: the same for all lanes)
  // Gain and offset first.
  // 256 columns per wave-instruction, waves 0-3 and 4-7
  if (wave < 8) {
    const float* src = wave < 4 ? a.gamma : a.beta;
    const int c = (wave & 3) * 256 + lane * 4;
    if (src && (wave & 3) * 256 < C)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + (c < C ? c : 0)),
                                       (__attribute__((address_space(3))) void*)(lds_g + (wave >> 2) * 1024 + (wave & 3) * 256), 16, 0, 0);
    else if (!src) *reinterpret_cast<f32x4_t*>(lds_g + 1024 + (wave & 3) * 256 + lane * 4) = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    int m = m0 + wave * RW + r;
    m = m < a.M ? m : a.M - 1;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (X16) {
        if (has(i, 0)) raw[r][i] = *reinterpret_cast<const i32x4_t*>(reinterpret_cast<const uint16_t*>(a.x) + (long)m * a.ldx + norm_column(false, i, 0, lane));
      } else {
        load_norm8<DT_F32>(a.x, (long)m * a.ldx, i, lane, C, x[r][i]);
      }
    }
  }
  // the bias of this thread's columns: two consecutive ones of row er (threads past the tile have nothing to store)
  constexpr int EV = 2;
  const int er = dmaf_div(tid, s.m_bn2), ec = (tid - er * (bn >> 1)) * 2;
  float bias[EV];
#pragma unroll
  for (int e = 0; e < EV; ++e) {
    const int n = n0 + ec + e;
    bias[e] = a.bias ? a.bias[n < a.N ? n : a.N - 1] : 0.f;
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- weight rows: 8 rows of 128 bytes per instruction, the swizzle applied on the global side
  {
    const int rg = bn >> 3, ldb = (int)a.ldw * ESZ, left = a.N - n0 < bn ? a.N - n0 : bn, l8 = lane >> 3;   // (row groups of a slab)
    int sl = 0, grp = wave;
    while (grp >= rg) { grp -= rg; ++sl; }
    const __amdgpu_buffer_rsrc_t rs = dmaf_rsrc(reinterpret_cast<const uint8_t*>(a.W) + (long)n0 * ldb, (long)left * ldb);
    // (every wave asks as often, past K out of bounds and into a spare kilobyte: the wait for what was requested before counts past them)
    const __amdgpu_buffer_rsrc_t none = dmaf_rsrc(a.W, 0);
    auto request = [&](auto once) {
#pragma unroll 1
      for (int j = 0; j < s.loads; ++j) {
        int r = grp * 8 + l8;
        r = r < left ? r : left - 1;
        const int voff = r * ldb + (((lane & 7) ^ lds_swizzle16(grp * 8 + l8)) << 4);
        uint8_t* const dst = sl < nslab ? lds_w + (sl * bn + grp * 8) * ROWB : reinterpret_cast<uint8_t*>(lds_g) + 8192;
        if constexpr (decltype(once)::value) dmaf_load16_nt(sl < nslab ? rs : none, dst, voff, sl * ROWB);
        else dmaf_load16(sl < nslab ? rs : none, dst, voff, sl * ROWB);
        sl += s.w_div;
        grp += s.w_mod;
        if (grp >= rg) { grp -= rg; ++sl; }
      }
    };
    if (a.w_once) request(std::true_type{});
    else request(std::false_type{});
  }
  __builtin_amdgcn_sched_barrier(0);
  // Everything requested before the weight rows is there: this wave's rows and bias, and its share of gain and offset (the zeros in the place of
  // an offset are a write to LDS), which the barrier behind the statistics then hands to every wave; the barrier itself waits for nothing.
  norm_wait<9>(s.loads);
  __builtin_amdgcn_sched_barrier(0);
  // ---- the norm
  const float inv_c = fast_rcp((float)C);
  if constexpr (X16) {
#pragma unroll
    for (int r = 0; r < RW; ++r)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t w = (uint32_t)raw[r][i][e];
          x[r][i][2 * e] = IN_DT == DT_F16 ? f16_bits_to_f32((uint16_t)(w & 0xffff)) : bf16_bits_to_f32((uint16_t)(w & 0xffff));
          x[r][i][2 * e + 1] = IN_DT == DT_F16 ? f16_bits_to_f32((uint16_t)(w >> 16)) : bf16_bits_to_f32((uint16_t)(w >> 16));
        }
  }
  float mean[RW], rstd[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (has(i, h)) {
#pragma unroll
          for (int e = 0; e < 4; ++e) sum += x[r][i][4 * h + e];
        }
    mean[r] = a.rms ? 0.f : wave_sum(sum) * inv_c;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (has(i, h)) {
#pragma unroll
          for (int e = 0; e < 4; ++e) { x[r][i][4 * h + e] -= mean[r]; q += x[r][i][4 * h + e] * x[r][i][4 * h + e]; }   // (from here on x - mean)
        }
    rstd[r] = rsqrtf(wave_sum(q) * inv_c + a.eps);
  }
  __builtin_amdgcn_sched_barrier(0);
  dmaf_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const int row = wave * RW + r;
    // A lane's place in the operand: 16-byte chunk of the column's 128-byte slab row; further groups of columns lie whole slabs behind.
    constexpr int GB = (X16 ? 8 : 4) * ESZ;       // bytes of the lane's consecutive columns
    const int lb = lane * GB;
    uint8_t* const dst = lds_a + ((lb >> 7) * BM + row) * ROWB + ((((lb & 127) >> 4) ^ lds_swizzle16(row)) << 4) + (lb & 15);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (has(i, h)) {
          const int col = norm_column(!X16, i, h, lane);
          const f32x4_t gv = *reinterpret_cast<const f32x4_t*>(lds_g + col), bv = *reinterpret_cast<const f32x4_t*>(lds_g + 1024 + col);
          float y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = x[r][i][4 * h + e] * rstd[r] * gv[e] + bv[e];
          if constexpr (IN_DT == DT_F16) {   // (rounded to fp32 first, as layernorm_kernel does: a multiply-add straight to f16 rounds once)
#pragma unroll
            for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(y[e]));
          }
          uint8_t* const d = X16 ? dst + i * 64 * GB / 128 * (BM * ROWB) + 8 * h : dst + (2 * i + h) * 64 * GB / 128 * (BM * ROWB);
          if constexpr (X16) {
            uint2 w;
            if constexpr (IN_DT == DT_BF16) w = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
            else w = make_uint2((uint32_t)f32_to_f16_bits(y[0]) | ((uint32_t)f32_to_f16_bits(y[1]) << 16), (uint32_t)f32_to_f16_bits(y[2]) | ((uint32_t)f32_to_f16_bits(y[3]) << 16));
            raw[r][i][2 * h] = (int)w.x; raw[r][i][2 * h + 1] = (int)w.y;
            if (h == 1) *reinterpret_cast<i32x4_t*>(d - 8) = raw[r][i];
          } else if constexpr (IN_DT == DT_FP8) *reinterpret_cast<uint32_t*>(d) = pack_fp8x4(y[0] * a.x_scale, y[1] * a.x_scale, y[2] * a.x_scale, y[3] * a.x_scale);
          else if constexpr (IN_DT == DT_BF16) *reinterpret_cast<uint2*>(d) = make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
          else
            *reinterpret_cast<uint2*>(d) = make_uint2((uint32_t)f32_to_f16_bits(y[0]) | ((uint32_t)f32_to_f16_bits(y[1]) << 16),
                                                      (uint32_t)f32_to_f16_bits(y[2]) | ((uint32_t)f32_to_f16_bits(y[3]) << 16));
        }
  }
  wait_vmcnt_lgkm0<0>();
  dmaf_barrier();      // the operands are there
  if constexpr (X16) {
    if (a.norm_out && tile_n == 0)
#pragma unroll
      for (int r = 0; r < RW; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (has(i, 0) && m0 + wave * RW + r < a.M)
            *reinterpret_cast<i32x4_t*>(reinterpret_cast<uint16_t*>(a.norm_out) + (long)(m0 + wave * RW + r) * a.ld_norm + norm_column(false, i, 0, lane)) = raw[r][i];
  }


  // ---- the product: a wave per block of WT x WT. 16-bit operands: 16x16x32 MFMAs (the same bits as 32x32x16 and a shorter chain, see gemm_dmas_kernel.hpp).
  // What a wave issues between two MFMAs of its chain counts: two blocks to a wave, whose fragments of X they share, with offsets worked out read by read took 2600 cycles
  // for K = 768, a block to a wave with offsets that run on 1500, 32x32x16 3000.
  // (rows of a block past the tile, and slabs read ahead past the last, are what lies behind: only sums that are not stored read them)
  constexpr bool QUADS = IN_DT != DT_FP8;
  constexpr int WT = QUADS ? 16 : 32, WROWS = (BM + WT - 1) / WT, STEPS = QUADS ? 2 : KSTEPS, NB = QUADS ? 2 : 4;
  const int wm = wave % WROWS, nb = wave / WROWS;
  typedef std::conditional_t<QUADS, f32x4_t, f32x16_t> Acc;
  Acc acc{};
  const bool multiplies = nb * WT < bn && n0 + nb * WT < a.N;
  const int lr = lane & (WT - 1), g = lane / WT;
  if (multiplies) {
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)smem);
    uint32_t wb[NB], xb[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int kc = QUADS ? 4 * k : (k & 1) | ((k >> 1) << 2), c = (QUADS ? g : 2 * g) ^ kc;
      wb[k] = lds0 + (nb * WT + lr) * ROWB + ((c ^ lds_swizzle16(nb * WT + lr)) << 4);
      xb[k] = lds0 + nslab * bn * ROWB + (wm * WT + lr) * ROWB + ((c ^ lds_swizzle16(wm * WT + lr)) << 4);
    }
    struct Frags { Frag<IN_DT> w[STEPS], x[STEPS]; };
    auto piece = [](uint32_t at) -> i32x4_t { return *reinterpret_cast<const __attribute__((address_space(3))) i32x4_t*>(at); };
    constexpr int SETS = BM == 16 && QUADS ? 4 : 2;   // slabs whose fragments are in registers or on their way; K is whole 256s, i.e. a multiple of them
    // (fragments of the slab the addresses stand at, and `ahead` slabs on for X; the addresses of W move on by a slab, those of X by a round of SETS)
    const uint32_t w_step = bn * ROWB;
    auto read_slab = [&](Frags& f, auto ahead) {
      constexpr int off = decltype(ahead)::value * BM * ROWB;
#pragma unroll
      for (int ks = 0; ks < STEPS; ++ks) {
        if constexpr (IN_DT == DT_FP8) {
          f.w[ks].lo = piece(wb[2 * ks]); f.w[ks].hi = piece(wb[2 * ks + 1]);
          f.x[ks].lo = piece(xb[2 * ks] + off); f.x[ks].hi = piece(xb[2 * ks + 1] + off);
        } else {
          f.w[ks].lo = piece(wb[ks]);
          f.x[ks].lo = piece(xb[ks] + off);
        }
      }
#pragma unroll
      for (int k = 0; k < NB; ++k) wb[k] += w_step;
    };
    auto mul_slab = [&](const Frags& f) {
#pragma unroll
      for (int ks = 0; ks < STEPS; ++ks) {
        if constexpr (QUADS) acc = mfma_quad<IN_DT>(f.w[ks], f.x[ks], acc);
        else acc = mfma_frag<IN_DT>(f.w[ks], f.x[ks], acc);
      }
    };
    Frags f[SETS];
    static_for<0, SETS - 1>([&](auto jc) { read_slab(f[decltype(jc)::value], jc); });
    for (int slab = 0; slab < nslab; slab += SETS) {
      static_for<0, SETS>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        read_slab(f[(j + SETS - 1) % SETS], std::integral_constant<int, j + SETS - 1>{});
        __builtin_amdgcn_sched_barrier(0);
        mul_slab(f[j]);
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int k = 0; k < NB; ++k) xb[k] += SETS * BM * ROWB;
    }
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
  dmaf_barrier();   // both operands are read: their space becomes the patches of the sums, one per 32 columns
  if (multiplies) {
    if constexpr (QUADS) {
      const int row = wm * WT + lr;
      *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(smem) + (nb >> 1) * 1024 + row * 32 + (((4 * (nb & 1) + g) ^ (row & 7)) << 2)) = acc;
    } else {
      float* const patch = reinterpret_cast<float*>(smem) + nb * 1024;
#pragma unroll
      for (int rq = 0; rq < 4; ++rq)
        *reinterpret_cast<f32x4_t*>(patch + lr * 32 + (((2 * rq + g) ^ (lr & 7)) << 2)) = f32x4_t{acc[4 * rq], acc[4 * rq + 1], acc[4 * rq + 2], acc[4 * rq + 3]};
    }
  }
  __syncthreads();
  // ---- epilogue: row er, columns ec .. ec + EV - 1
  const int m = m0 + er, n = n0 + ec;
  if (er >= BM || m >= a.M || n >= a.N) return;
  float v[EV];
  {
    const float* patch = reinterpret_cast<const float*>(smem) + (ec >> 5) * 1024 + er * 32 + ((((ec & 31) >> 2) ^ (er & 7)) << 2) + (ec & 3);
#pragma unroll
    for (int e = 0; e < EV; ++e) v[e] = patch[e];
  }
  const bool fused_mish = a.out_dtype == DT_FP8 && a.act == ACT_MISH;   // as in gemm_epilogue
#pragma unroll
  for (int e = 0; e < EV; ++e) {
    const float sum = v[e];
    v[e] = fmaf(sum, a.descale, bias[e]);
    if (fused_mish) {
      constexpr float L2E = 1.4426950408889634f;
      const float nexp = __builtin_amdgcn_exp2f(fmaf(sum, a.descale * L2E, bias[e] * L2E));
      v[e] *= fmaf(fast_rcp(fmaf(nexp, nexp + 2.f, 2.f)), -2.f * a.out_scale, a.out_scale);
    } else {
      v[e] = apply_act(v[e], a.act);
      if (a.out_dtype == DT_FP8) v[e] *= a.out_scale;
    }
    if (a.out_dtype == DT_F16) asm volatile("" : "+v"(v[e]));   // (rounded to fp32 first, as everywhere else)
  }
  const bool first = n < a.nsplit;
  void* const out = first ? a.out : a.out2;
  const long o = first ? (long)m * a.ldo + n : (long)m * a.ldo2 + (n - a.nsplit);
  {
    if (a.vec_ok && n + EV <= a.N) {
      if (a.out_dtype == DT_F32) *reinterpret_cast<float2*>(reinterpret_cast<float*>(out) + o) = make_float2(v[0], v[1]);
      else if (a.out_dtype == DT_FP8) *reinterpret_cast<uint16_t*>(reinterpret_cast<uint8_t*>(out) + o) = (uint16_t)pack_fp8x4(v[0], v[1], v[0], v[1]);
      else *reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(out) + o) = a.out_dtype == DT_BF16 ? pack_bf16x2(v[0], v[1]) : (uint32_t)f32_to_f16_bits(v[0]) | ((uint32_t)f32_to_f16_bits(v[1]) << 16);
      return;
    }
  }
#pragma unroll
  for (int e = 0; e < EV; ++e) {
    const int c = n + e;
    if (c >= a.N) break;
    void* const d = c < a.nsplit ? a.out : a.out2;
    const long at = c < a.nsplit ? (long)m * a.ldo + c : (long)m * a.ldo2 + (c - a.nsplit);
    switch (a.out_dtype) {
      case DT_F32: reinterpret_cast<float*>(d)[at] = v[e]; break;
      case DT_BF16: reinterpret_cast<uint16_t*>(d)[at] = f32_to_bf16_bits(v[e]); break;
      case DT_F16: reinterpret_cast<uint16_t*>(d)[at] = f32_to_f16_bits(v[e]); break;
      default: reinterpret_cast<uint8_t*>(d)[at] = f32_to_fp8(v[e]); break;
    }
  }
}

}  // namespace crl
