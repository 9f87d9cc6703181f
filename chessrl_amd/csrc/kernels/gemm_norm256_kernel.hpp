// C[M,N] = swish(norm(X)[M,256] · W[N,256]^T + bias) or descale * norm(X)[M,256] · W[N,256]^T: the two norms of the attention-bias generator, each with the product behind it, as one
// launch: 256 16-bit columns per row, normalised row by row (the hidden layer, M = positions) or 32 rows together (the 8192 values of a
// position, which are its 32 heads' rows of the product behind).
// On few positions the norms were launches of 3.2 and 5.4 us around a handful of rows, between products of 3.6 us. Here a workgroup normalises
// its 32 or 64 rows itself, keeps them as the MFMA operand in registers and walks a slice of N in steps of 64 columns, whose weights four waves
// bring into a ring of three LDS stages; the first stage, on which a call of one position waits, is requested by all eight waves,
// behind the rows, gains and offsets of the norm and ahead of its arithmetic.
// The 256 columns and the 32 rows of a position are the generator's sizes at 1024 channels and 32 heads; other sizes take two launches.
// Bound by the load latencies in a row (rows, then weights) on one position: 4.0 and 4.6 us where the two kernels took 6.3 and 8.3, and a launch more. On many
// rows by the weights' way into LDS: 64 KB in flight per CU and some 0.95 us a step of 64 x 64 outputs, of which the 16 MFMAs in one chain are 0.4
// (256 bf16 positions: 31.6 us a launch, 33.9 before; results stored 8 bytes per lane and row, or finished behind the MFMAs instead of in the shadow of the
// next tile's: 54 and 40 us). 32 rows a workgroup while every tile of 32 x 64 has a CU: that form has one stage and no loop.
// The norms' arithmetic is that of layernorm_kernel and layernorm_wide_kernel, the products add K in the order of the tiled kernels: bit-equal to
// the launches this replaces.
#pragma once
#include "gemm_dmaf_kernel.hpp"
#include "norm_rows.hpp"

namespace crl {

struct Norm256KArgs {
  const void* x; long ldx;            // rows of 256 16-bit values; GROUPED: dense
  const float* gamma; const float* beta;   // [256]; GROUPED: [8192]
  const void* W; const float* bias;   // [N, 256] dense; [N] or null
  void* out; long ldo;
  int M, N;
  int groups, tiles, steps;           // row groups of 32 RB, column tiles of 64, tiles of a workgroup's slice
  float eps, x_scale, descale;
  uint32_t m_groups;
  int per_xcd;
};

// Sum over the 32 lanes of a half wave, in the order of wave_sum (whose last step adds the other half).
__device__ __forceinline__ float half_wave_sum(float v) {
  v += dpp_move<DPP_XOR1>(v);
  v += dpp_move<DPP_XOR2>(v);
  v += dpp_move<DPP_HALF_MIRROR>(v);
  v += dpp_move<DPP_MIRROR>(v);
  return add_xor16(v);
}

// X_DT: type of X and of the output; IN_DT: operand type (X_DT or e4m3); RB: row blocks of 32 per workgroup.
template <int X_DT, int IN_DT, int RB, bool GROUPED>
__global__ void __launch_bounds__(512) gemm_norm256_kernel(const Norm256KArgs a) {
  constexpr int ESZ = IN_DT == DT_FP8 ? 1 : 2, ROWB = 128, NSLAB = 256 * ESZ / ROWB, KSTEPS = ROWB / (IN_DT == DT_FP8 ? 64 : 32);
  constexpr int ROWS = 32 * RB, BN = 64, NST = RB == 1 ? 1 : 3, STAGE = BN * 256 * ESZ, A_BYTES = ROWS * 256 * ESZ;
  constexpr int LOADS = STAGE / 1024;                 // load instructions of a stage
  __shared__ __align__(16) uint8_t s_a[A_BYTES];      // [slab][row][128 bytes]
  __shared__ __align__(16) uint8_t s_w[NST * STAGE];  // [stage][slab][64 rows][128 bytes]
  __shared__ __align__(16) uint8_t s_out[2 * RB][2048];   // a multiplying wave's results: 32 rows of 64 bytes
  __shared__ float s_red[2][2][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Slices outermost: workgroup b runs on XCD b & 7, which owns a contiguous range, so that an XCD reads its part of the weights only.
  int pid = blockIdx.x;
  if (pid < (a.per_xcd << 3)) pid = (pid & 7) * a.per_xcd + (pid >> 3);
  const int slice = dmaf_div(pid, a.m_groups), group = pid - slice * a.groups;
  const int m0 = group * ROWS, t0 = slice * a.steps;
  const int steps = a.tiles - t0 < a.steps ? a.tiles - t0 : a.steps;

  // ---- everything the norm reads, then the first stage
  // GROUPED: thread t of 256 holds columns (256 i + t) * 8 .. + 7 of the position's 8192 (i = 0 .. 3), as in layernorm_wide_kernel; waves 0-3 have the
  // first position, 4-7 the second. Row by row: a half wave holds a row, eight columns a lane, 16 rows in a pass of the workgroup.
  constexpr int VPT = GROUPED ? 4 : ROWS / 16;
  const int t256 = tid & 255, hl = lane & 31;
  const bool norms = !GROUPED || (tid >> 8) < RB;
  float x[VPT][8], gv[GROUPED ? VPT : 1][8], bv[GROUPED ? VPT : 1][8];
  if constexpr (GROUPED) {
    if (norms) {
      long pos = (long)group * RB + (tid >> 8);
      const long last = a.M / 32 - 1;
      pos = pos < last ? pos : last;
#pragma unroll
      for (int i = 0; i < VPT; ++i) load8<X_DT>(a.x, pos * 8192 + (i * 256 + t256) * 8, x[i]);
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        load8<DT_F32>(a.gamma, (i * 256 + t256) * 8, gv[i]);
        load8<DT_F32>(a.beta, (i * 256 + t256) * 8, bv[i]);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      int m = m0 + i * 16 + wave * 2 + (lane >> 5);
      m = m < a.M ? m : a.M - 1;
      load8<X_DT>(a.x, (long)m * a.ldx + hl * 8, x[i]);
    }
    load8<DT_F32>(a.gamma, hl * 8, gv[0]);
    load8<DT_F32>(a.beta, hl * 8, bv[0]);
  }
  __builtin_amdgcn_sched_barrier(0);
  // Load i of a stage: 8 rows of a slab, the swizzle applied on the global side. (N is whole tiles: no row past the end.)
  const int l8 = lane >> 3;
  const __amdgpu_buffer_rsrc_t rs = dmaf_rsrc(reinterpret_cast<const uint8_t*>(a.W) + (long)t0 * BN * 256 * ESZ, (long)steps * BN * 256 * ESZ);
  auto load = [&](int t, int stage, int i) {
    const int slab = i >> 3, rg = i & 7;
    dmaf_load16(rs, s_w + stage * STAGE + i * 1024, (rg * 8 + l8) * 256 * ESZ + (((lane & 7) ^ l8 ^ rg) << 4), t * (BN * 256 * ESZ) + slab * ROWB);
  };
#pragma unroll
  for (int i = 0; i < LOADS / 8; ++i) load(0, 0, wave * (LOADS / 8) + i);
  __builtin_amdgcn_sched_barrier(0);

  // ---- the norm, and the normalised rows as the operand
  auto put = [&](int row, int col, const float (&y)[8]) {   // eight columns of one row
    const int b = col * ESZ;
    uint8_t* const d = s_a + ((b >> 7) * ROWS + row) * ROWB + ((((b & 127) >> 4) ^ lds_swizzle(row)) << 4) + (b & 15);
    if constexpr (IN_DT == DT_FP8) {
      *reinterpret_cast<uint2*>(d) = make_uint2(pack_fp8x4(y[0] * a.x_scale, y[1] * a.x_scale, y[2] * a.x_scale, y[3] * a.x_scale),
                                                pack_fp8x4(y[4] * a.x_scale, y[5] * a.x_scale, y[6] * a.x_scale, y[7] * a.x_scale));
    } else {
      store8(d, 0, y, IN_DT);
    }
  };
  auto affine = [&](float xm, float rstd, float g, float b) -> float {
    float y = xm * rstd * g + b;
    if constexpr (IN_DT == DT_F16) asm volatile("" : "+v"(y));   // (rounded to fp32 first, as the norm kernels do: a multiply-add straight to f16 rounds once)
    return y;
  };
  if constexpr (GROUPED) {
    float s = 0.f;
    const int half = tid >> 8, w4 = wave & 3;
    if (norms) {
#pragma unroll
      for (int i = 0; i < VPT; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) s += x[i][e];
      s = wave_sum(s);
      if (lane == 0) s_red[half][0][w4] = s;
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    dmaf_barrier();
    float mean = 0.f, q = 0.f;
    if (norms) {
      const float* r = s_red[half][0];
      mean = (((r[0] + r[1]) + r[2]) + r[3]) / 8192.f;
#pragma unroll
      for (int i = 0; i < VPT; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) { const float d = x[i][e] - mean; q += d * d; }
      q = wave_sum(q);
      if (lane == 0) s_red[half][1][w4] = q;
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);
    dmaf_barrier();
    if (norms) {
      const float* r = s_red[half][1];
      const float rstd = rsqrtf((((r[0] + r[1]) + r[2]) + r[3]) / 8192.f + a.eps);
#pragma unroll
      for (int i = 0; i < VPT; ++i) {
        float y[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = affine(x[i][e] - mean, rstd, gv[i][e], bv[i][e]);
        put(32 * half + 8 * i + (t256 >> 5), (t256 & 31) * 8, y);
      }
    }
  } else {
    const float inv_c = fast_rcp(256.f);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) s += x[i][e];
      const float mean = half_wave_sum(s) * inv_c;
      float q = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) { const float d = x[i][e] - mean; q += d * d; }
      const float rstd = rsqrtf(half_wave_sum(q) * inv_c + a.eps);
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = affine(x[i][e] - mean, rstd, gv[0][e], bv[0][e]);
      put(i * 16 + wave * 2 + (lane >> 5), hl * 8, y);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  wait_vmcnt_lgkm0<0>();   // the operand's rows and this wave's part of the first stage

  // ---- loading waves: barrier t says that stage t has landed (barrier 0: and the operand), and that every fragment of stage t - 1 is in registers
  if (wave >= 4) {
    auto stage = [&](int t) {
#pragma unroll
      for (int i = 0; i < LOADS / 4; ++i) load(t, t % NST, (wave - 4) * (LOADS / 4) + i);
    };
    if (RB > 1 && steps > 1) stage(1);
    if (RB > 1 && steps > 2) stage(2);
    dmaf_barrier();
    for (int t = 1; RB > 1 && t < steps; ++t) {
      if (t + 1 < steps) wait_vmcnt<LOADS / 4>();
      else wait_vmcnt<0>();
      dmaf_barrier();
      if (t + 2 < steps) stage(t + 2);   // into the place of stage t - 1
    }
    return;
  }
  dmaf_barrier();
  if (wave >= 2 * RB) return;

  // ---- multiplying waves: row block rb, columns 32 cb .. + 31 of every tile
  const int rb = wave % RB, cb = wave / RB, lr = lane & 31, g = lane >> 5;
  const int arow = rb * 32 + lr, wrow = cb * 32 + lr;
  auto piece = [](const uint8_t* p) -> i32x4_t { return *reinterpret_cast<const i32x4_t*>(p); };
  auto frag = [&](const uint8_t* row, int sw, auto ksc) -> Frag<IN_DT> {
    constexpr int ks = decltype(ksc)::value;
    Frag<IN_DT> f;
    if constexpr (IN_DT == DT_FP8) {
      f.lo = piece(row + (((4 * ks + 2 * g) ^ sw) << 4));
      f.hi = piece(row + (((4 * ks + 2 * g + 1) ^ sw) << 4));
    } else {
      f.lo = piece(row + (((2 * ks + g) ^ sw) << 4));
    }
    return f;
  };
  const int swx = lds_swizzle(arow), sww = lds_swizzle(wrow);
  struct Slab { Frag<IN_DT> f[KSTEPS]; };
  Slab xf[NSLAB], wf[2];
  auto read_w = [&](int stage, int slab, Slab& s) {
    const uint8_t* row = s_w + stage * STAGE + (slab * BN + wrow) * ROWB;
    static_for<0, KSTEPS>([&](auto ksc) { s.f[decltype(ksc)::value] = frag(row, sww, ksc); });
  };
  read_w(0, 0, wf[0]);
  static_for<0, NSLAB>([&](auto sc) {
    constexpr int sl = decltype(sc)::value;
    static_for<0, KSTEPS>([&](auto ksc) { xf[sl].f[decltype(ksc)::value] = frag(s_a + (sl * ROWS + arow) * ROWB, swx, ksc); });
  });
  // Results leave through a patch: 16 rows of 64 bytes per store (8 bytes per lane and row, straight from the accumulators, took 1.6 us a step).
  uint8_t* const patch = s_out[wave];
  const int er = lane >> 2, ec = lane & 3;
  const int mo = m0 + rb * 32 + er;
  uint16_t* const orow = reinterpret_cast<uint16_t*>(a.out) + (long)mo * a.ldo + t0 * BN + cb * 32 + 8 * ec;
  const float* const bcol = a.bias + t0 * BN + cb * 32 + 4 * g;   // (row by row only)
  // The results of a tile are finished in the shadow of the next tile's MFMAs, a piece behind each: four times four columns of the lane's row into the
  // patch, the patch read back by rows, two stores. One copy of each in the code: a call of one position fetches its instructions from memory, and every
  // jump to a line that nothing has asked for yet is a round trip.
  constexpr int NM = NSLAB * KSTEPS, PIECES = 16;
  i32x4_t back0, back1;
  f32x16_t done = {};
  f32x4_t bias[2][4];   // of this tile, of the one before
#pragma unroll
  for (int rq = 0; rq < 4; ++rq) bias[0][rq] = bias[1][rq] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto finish = [&](auto pc, int t) {
    constexpr int p = decltype(pc)::value;
    if constexpr (p < 4) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = fmaf(done[4 * p + e], a.descale, bias[1][p][e]);
        if constexpr (!GROUPED) v[e] = act_swish(v[e]);
        if constexpr (X_DT == DT_F16) asm volatile("" : "+v"(v[e]));
      }
      uint2 w;
      if constexpr (X_DT == DT_BF16) w = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
      else w = make_uint2((uint32_t)f32_to_f16_bits(v[0]) | ((uint32_t)f32_to_f16_bits(v[1]) << 16), (uint32_t)f32_to_f16_bits(v[2]) | ((uint32_t)f32_to_f16_bits(v[3]) << 16));
      *reinterpret_cast<uint2*>(patch + lr * 64 + ((p ^ ((lr >> 2) & 3)) << 4) + 8 * g) = w;
    } else if constexpr (p == 5) {
      wave_lds_fence();
      back0 = *reinterpret_cast<const i32x4_t*>(patch + er * 64 + ((ec ^ ((er >> 2) & 3)) << 4));
      back1 = *reinterpret_cast<const i32x4_t*>(patch + (er + 16) * 64 + ((ec ^ ((er >> 2) & 3)) << 4));
      wave_lds_fence();
    } else if constexpr (p == 9) {
      if (t >= 0 && mo < a.M) *reinterpret_cast<i32x4_t*>(orow + t * BN) = back0;
      if (t >= 0 && mo + 16 < a.M) *reinterpret_cast<i32x4_t*>(orow + 16L * a.ldo + t * BN) = back1;
    }
  };
  int st = 0;
#pragma unroll 1
  for (int t = 0; t < steps; ++t) {
    const int nx = st == NST - 1 ? 0 : st + 1;
    if constexpr (!GROUPED) {
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) bias[0][rq] = *reinterpret_cast<const f32x4_t*>(bcol + t * BN + 8 * rq);
    }
    f32x16_t acc;
    static_for<0, NSLAB>([&](auto sc) {
      constexpr int sl = decltype(sc)::value;
      Slab& cur = wf[sl & 1];
      Slab& next = wf[(sl + 1) & 1];
      if constexpr (sl + 1 == NSLAB) {
        if (RB > 1 && t + 1 < steps) {
          __builtin_amdgcn_sched_barrier(0);
          __builtin_amdgcn_s_waitcnt(0xC07F);   // this stage's last fragments
          dmaf_barrier();
          __builtin_amdgcn_sched_barrier(0);
          read_w(nx, 0, next);
        }
      } else {
        read_w(st, sl + 1, next);
      }
      static_for<0, KSTEPS>([&](auto ksc) {
        constexpr int ks = decltype(ksc)::value, i = sl * KSTEPS + ks;
        if constexpr (i == 0) acc = mfma_frag<IN_DT>(cur.f[ks], xf[sl].f[ks], f32x16_t{});
        else acc = mfma_frag<IN_DT>(cur.f[ks], xf[sl].f[ks], acc);
        if constexpr (RB > 1) {   // (one row block: one tile)
          __builtin_amdgcn_sched_barrier(0);
          static_for<i * PIECES / NM, (i + 1) * PIECES / NM>([&](auto pc) { finish(pc, t - 1); });
          __builtin_amdgcn_sched_barrier(0);
        }
      });
    });
    static_assert(NSLAB % 2 == 0, "the next tile's first fragments lie where this tile's did");
    st = nx;
    done = acc;
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) bias[1][rq] = bias[0][rq];
    if constexpr (RB == 1) break;
  }
  static_for<0, PIECES>([&](auto pc) { finish(pc, steps - 1); });
}

}  // namespace crl
