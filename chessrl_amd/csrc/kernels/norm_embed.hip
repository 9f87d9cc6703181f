// Row-wise LayerNorm and the board-token embedding.
//
// LayerNorm replaces F.layer_norm / nn.LayerNorm (eps 1e-5, affine) at
// model_bis.py:34, new_paradigm/value.py:36-37,134 and utils/fen_encoder.py:57; the
// residual sum it normalises is produced by the preceding GEMM's epilogue. It can
// also emit an e4m3 copy of its output (value * scale) so the next fp8 GEMM needs no
// separate quantise pass.
//
// The embedding kernel is FenEncoder.forward (utils/fen_encoder.py:61-67) and the
// identical stem of BT4.forward (new_paradigm/value.py:159-167): Linear(19->C), GELU,
// LayerNorm, x*exp(a)+b gating, plus the fixed sinusoid rows of model_bis.py:362-366
// when a table is supplied.
//
// One 64-lane wave owns one row; a lane keeps VPL vectors of 8 consecutive columns in
// registers, so a row is read once and the statistics are two wave reductions.
#include "norm_rows.hpp"

namespace crl {

// (fp32 rows: a lane's columns are two groups of four per vector, see norm_column; 16-bit rows: eight consecutive ones)
// Bound by memory at many rows, by one wave's trips to it at few: everything a wave reads (RPW rows, then scale and offset, which the rows share) is
// requested before the first reduction. 97344 rows of 512 bf16 41.7 -> 35.0 us (5.7 TB/s), 32768 of 768 fp32 27.8 -> 25.5, 96000 73.7 -> 69.4, against one
// row per wave with scale and offset read behind the reductions; four rows per wave 39.3 for the first.
// ONCE: the rows are read past the caches (see the launch).
template <int IN_DT, int VPL, bool FULL = false, int RPW = 1, bool ONCE = false>
__global__ void __launch_bounds__(256) layernorm_kernel(const LayerNormArgs a) {
  constexpr bool F32 = IN_DT == DT_F32;
  const int lane = threadIdx.x & 63;
  const long row0 = ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * RPW;
  if (row0 >= a.rows) return;
  const int C = FULL ? VPL * 512 : a.C;
  auto has = [&](int i, int h) { return FULL || norm_column(F32, i, h, lane) < C; };
  const bool rms = a.rms != 0;
  const float* const beta = rms ? nullptr : a.beta;
  float x[RPW][VPL][8], g[VPL][8], b[VPL][8];
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    const long row = RPW > 1 && row0 + r >= a.rows ? a.rows - 1 : row0 + r;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      if constexpr (ONCE) {
        static_assert(!F32, "16-bit rows");
        if (has(i, 0)) {
          const i32x4_t raw = __builtin_nontemporal_load(reinterpret_cast<const i32x4_t*>(reinterpret_cast<const uint16_t*>(a.x) + row * a.ldx + norm_column(false, i, 0, lane)));
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint16_t lo = (uint16_t)((uint32_t)raw[e] & 0xffff), hi = (uint16_t)((uint32_t)raw[e] >> 16);
            x[r][i][2 * e] = IN_DT == DT_BF16 ? bf16_bits_to_f32(lo) : f16_bits_to_f32(lo);
            x[r][i][2 * e + 1] = IN_DT == DT_BF16 ? bf16_bits_to_f32(hi) : f16_bits_to_f32(hi);
          }
        }
      } else {
        load_norm8<IN_DT>(a.x, row * a.ldx, i, lane, C, x[r][i]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < VPL; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int e = 0; e < 4; ++e) g[i][4 * h + e] = b[i][4 * h + e] = 0.f;
      if (has(i, h)) {
        const int col = norm_column(F32, i, h, lane);
        const float4 gv = *reinterpret_cast<const float4*>(a.gamma + col);
        g[i][4 * h] = gv.x; g[i][4 * h + 1] = gv.y; g[i][4 * h + 2] = gv.z; g[i][4 * h + 3] = gv.w;
        if (beta) {
          const float4 bv = *reinterpret_cast<const float4*>(beta + col);
          b[i][4 * h] = bv.x; b[i][4 * h + 1] = bv.y; b[i][4 * h + 2] = bv.z; b[i][4 * h + 3] = bv.w;
        }
      }
    }
  if constexpr (RPW > 1) __builtin_amdgcn_sched_barrier(0);   // (no use of a loaded value, and so no wait, moves up between the loads)
  // (1 / C by the hardware reciprocal, exact for the power-of-two widths and within one unit in the last place otherwise:
  // two IEEE divisions are 22 of a row's ~400 instructions)
  const float inv_c = fast_rcp((float)C);
  float am = 0.f;
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    const long row = row0 + r;
    if (RPW > 1 && row >= a.rows) break;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (has(i, h)) {
#pragma unroll
          for (int e = 0; e < 4; ++e) s += x[r][i][4 * h + e];
        }
    const float mean = rms ? 0.f : wave_sum(s) * inv_c;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (has(i, h)) {
#pragma unroll
          for (int e = 0; e < 4; ++e) { const float d = x[r][i][4 * h + e] - mean; q += d * d; }
        }
    const float rstd = rsqrtf(wave_sum(q) * inv_c + a.eps);
    if (a.stats && lane == 0) *reinterpret_cast<float2*>(a.stats + 2 * row) = make_float2(rstd, -mean * rstd);   // (x - mean) * rstd = x * s0 + s1
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      float y[8];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (has(i, h)) {
          const int col = norm_column(F32, i, h, lane);
#pragma unroll
          for (int e = 0; e < 4; ++e) y[4 * h + e] = (x[r][i][4 * h + e] - mean) * rstd * g[i][4 * h + e] + b[i][4 * h + e];
          if (a.amax) {
#pragma unroll
            for (int e = 0; e < 4; ++e) am = fmaxf(am, fabsf(y[4 * h + e]));
          }
          if constexpr (F32) {
            const long off = row * a.ldo + col;
            if (a.out) store4(a.out, off, y + 4 * h, a.out_dtype);
            if (a.out_b) store4(a.out_b, off, y + 4 * h, a.out_b_dtype);
            if (a.out_fp8) store4_fp8(a.out_fp8, off, y + 4 * h, a.fp8_scale);
          }
        }
      if constexpr (!F32) {
        if (has(i, 0)) {
          const long off = row * a.ldo + norm_column(false, i, 0, lane);
          if (a.out) store8(a.out, off, y, a.out_dtype);
          if (a.out_b) store8(a.out_b, off, y, a.out_b_dtype);
          if (a.out_fp8) store8_fp8(a.out_fp8, off, y, a.fp8_scale);
        }
      }
    }
  }
  if (a.amax) {
    am = wave_max(am);
    if (lane == 0) atomic_amax(a.amax, am);
  }
}

// The trunk's norm: bf16 rows of exactly 1024 elements, LayerNorm with offset, outputs bf16 and/or e4m3. Same arithmetic per
// row as layernorm_kernel (same order of additions, same roundings), but with everything about the call fixed at compile
// time and all of a wave's loads (RPW rows, then scale and offset, which RPW rows share) issued before the first
// reduction, so that a wave waits for memory once instead of three times.
template <bool OUT16, bool OUT8, int RPW>
__global__ void __launch_bounds__(256) layernorm_trunk_kernel(const LayerNormArgs a) {
  const int lane = threadIdx.x & 63;
  const long row0 = ((long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * RPW;
  if (row0 >= a.rows) return;
  float x[RPW][2][8], g[2][8], b[2][8];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    load8<DT_F32>(a.gamma, (i * 64 + lane) * 8, g[i]);
    load8<DT_F32>(a.beta, (i * 64 + lane) * 8, b[i]);
  }
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      // (read once: with the non-temporal hint the row does not displace what the products around this launch keep in
      // the caches; measured on a 4096-position pass: this kernel -2.8 %, the pass -0.6 ms)
      typedef int i32x4_nt __attribute__((ext_vector_type(4)));
      const i32x4_nt raw = __builtin_nontemporal_load(reinterpret_cast<const i32x4_nt*>(reinterpret_cast<const uint16_t*>(a.x) + (row0 + r) * a.ldx + (i * 64 + lane) * 8));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[r][i][2 * e] = bf16_bits_to_f32((uint16_t)((uint32_t)raw[e] & 0xffff));
        x[r][i][2 * e + 1] = bf16_bits_to_f32((uint16_t)((uint32_t)raw[e] >> 16));
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);   // (no use of a loaded value, and so no wait, moves up between the loads)
  const float inv_c = fast_rcp(1024.f);
  float am = 0.f;
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int e = 0; e < 8; ++e) s += x[r][i][e];
    }
    const float mean = wave_sum(s) * inv_c;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int e = 0; e < 8; ++e) { const float d = x[r][i][e] - mean; q += d * d; }
    }
    const float rstd = rsqrtf(wave_sum(q) * inv_c + a.eps);
    if (a.stats && lane == 0) *reinterpret_cast<float2*>(a.stats + 2 * (row0 + r)) = make_float2(rstd, -mean * rstd);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float y[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = (x[r][i][e] - mean) * rstd * g[i][e] + b[i][e];
      const long off = (row0 + r) * a.ldo + (i * 64 + lane) * 8;
      if constexpr (OUT16) store8(a.out, off, y, DT_BF16);
      if constexpr (OUT8) store8_fp8(a.out_fp8, off, y, a.fp8_scale);
      if (a.amax) {
#pragma unroll
        for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(y[e]));
      }
    }
  }
  if (a.amax) {
    am = wave_max(am);
    if (lane == 0) atomic_amax(a.amax, am);
  }
}

template <int RPW>
static void launch_ln_trunk(const LayerNormArgs& a, int waves, hipStream_t st) {
  const dim3 grid((a.rows / RPW + waves - 1) / waves), block(64 * waves);
  if (a.out && a.out_fp8) hipLaunchKernelGGL((layernorm_trunk_kernel<true, true, RPW>), grid, block, 0, st, a);
  else if (a.out) hipLaunchKernelGGL((layernorm_trunk_kernel<true, false, RPW>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((layernorm_trunk_kernel<false, true, RPW>), grid, block, 0, st, a);
}

// Rows longer than 2048 elements (the 8192-wide norm of the bias generator): the four waves of a workgroup share one
// row, 8 elements per thread and step of 2048, and meet through LDS for the two reductions (wave sums added in wave
// order). Chosen by the row length alone, so a row's result does not depend on how many rows the call has; with one
// row per position it also puts four times as many waves on a small batch as one wave per row would.
template <int IN_DT>
__global__ void __launch_bounds__(256) layernorm_wide_kernel(const LayerNormArgs a) {
  constexpr int VPT = 4;
  __shared__ float s_red[2][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const long row = blockIdx.x;
  float x[VPT][8];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int col = (i * 256 + tid) * 8;
    if (col < a.C) {
      load8<IN_DT>(a.x, row * a.ldx + col, x[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += x[i][e];
    }
  }
  s = wave_sum(s);
  if (lane == 0) s_red[0][wave] = s;
  __syncthreads();
  const bool rms = a.rms != 0;
  const float mean = rms ? 0.f : (((s_red[0][0] + s_red[0][1]) + s_red[0][2]) + s_red[0][3]) / (float)a.C;
  const float* beta = rms ? nullptr : a.beta;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    if ((i * 256 + tid) * 8 < a.C) {
#pragma unroll
      for (int e = 0; e < 8; ++e) { const float d = x[i][e] - mean; q += d * d; }
    }
  }
  q = wave_sum(q);
  if (lane == 0) s_red[1][wave] = q;
  __syncthreads();
  const float rstd = rsqrtf((((s_red[1][0] + s_red[1][1]) + s_red[1][2]) + s_red[1][3]) / (float)a.C + a.eps);
  float am = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int col = (i * 256 + tid) * 8;
    if (col < a.C) {
      float gv[8], bv[8], y[8];
      load8<DT_F32>(a.gamma, col, gv);
      if (beta) load8<DT_F32>(beta, col, bv);
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = (x[i][e] - mean) * rstd * gv[e] + (beta ? bv[e] : 0.f);
      if (a.out) store8(a.out, row * a.ldo + col, y, a.out_dtype);
      if (a.out_b) store8(a.out_b, row * a.ldo + col, y, a.out_b_dtype);
      if (a.out_fp8) store8_fp8(a.out_fp8, row * a.ldo + col, y, a.fp8_scale);
      if (a.amax) {
#pragma unroll
        for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(y[e]));
      }
    }
  }
  if (a.amax) {
    am = wave_max(am);
    if (lane == 0) atomic_amax(a.amax, am);
  }
}

template <int IN_DT, bool ONCE>
static hipError_t launch_ln_two_rows(const LayerNormArgs& a, int vecs, hipStream_t st) {
  const dim3 grid((a.rows + 7) / 8), block(256);
  if (vecs <= 1) hipLaunchKernelGGL((layernorm_kernel<IN_DT, 1, false, 2, ONCE>), grid, block, 0, st, a);
  else if (a.C == 1024) hipLaunchKernelGGL((layernorm_kernel<IN_DT, 2, true, 2, ONCE>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((layernorm_kernel<IN_DT, 2, false, 2, ONCE>), grid, block, 0, st, a);
  return hipGetLastError();
}

template <int IN_DT>
static hipError_t launch_ln_dt(const LayerNormArgs& a, hipStream_t st) {
  const dim3 grid((a.rows + 3) / 4), block(256);
  const int vecs = (a.C / 8 + 63) / 64;
  if constexpr (IN_DT == DT_BF16) {
    if (a.C == 1024 && !a.rms && a.beta && !a.out_b && (a.out || a.out_fp8) && (!a.out || a.out_dtype == DT_BF16)) {
      // (two rows per wave: 18 % faster than one at 262144 rows, and no slower than four; per-row arithmetic is the same)
      // (few rows: the launch is one wave's chain of latencies, and a row's wave alone on its compute unit has the shortest; 64 rows 3.45 us with
      // two rows per wave, 3.0 with one, 2.7 in workgroups of one wave)
      const int cus = device_cus();
      if (a.rows <= 2 * cus) launch_ln_trunk<1>(a, 1, st);
      else if (a.rows % 2 || a.rows <= 16 * cus) launch_ln_trunk<1>(a, 4, st);
      else launch_ln_trunk<2>(a, 4, st);
      return hipGetLastError();
    }
  }
  // Two rows per wave from where that leaves enough waves in flight (10 layers of 512 channels: 16000 rows 1.224 -> 1.234 ms, 22400 1.81 -> 1.79; 1024
  // channels, f16: 4096 rows 2.23 -> 2.22 ms, 16000 5.79 -> 5.70).
  if (vecs <= 2 && a.rows > (vecs == 1 ? 80 : 16) * device_cus()) {
    if constexpr (IN_DT != DT_F32) {
      // Rows of more than 80 MB, with what the products around this launch read and write, are past what the 256 MB cache on the memory side holds from
      // one launch to the next: with the non-temporal hint they leave it to the others (10 layers of 512 channels: 97344 rows 5.99 -> 5.91 ms, 128000
      // 7.93 -> 7.69, 256000 15.7 -> 15.1; 64000 rows 4.06 -> 4.08; set on this one model, and only time depends on it).
      if ((long)a.rows * a.C * 2 > 80L << 20) return launch_ln_two_rows<IN_DT, true>(a, vecs, st);
    }
    return launch_ln_two_rows<IN_DT, false>(a, vecs, st);
  }
  if (vecs <= 1) hipLaunchKernelGGL((layernorm_kernel<IN_DT, 1>), grid, block, 0, st, a);
  else if (a.C == 1024) hipLaunchKernelGGL((layernorm_kernel<IN_DT, 2, true>), grid, block, 0, st, a);   // (the trunk's width: no column guards)
  else if (vecs <= 2) hipLaunchKernelGGL((layernorm_kernel<IN_DT, 2>), grid, block, 0, st, a);
  else if (vecs <= 4) hipLaunchKernelGGL((layernorm_kernel<IN_DT, 4>), grid, block, 0, st, a);
  else if (vecs <= 16) hipLaunchKernelGGL((layernorm_wide_kernel<IN_DT>), dim3(a.rows), block, 0, st, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_layernorm(const LayerNormArgs& a, hipStream_t st) {
  if (a.rows <= 0) return hipSuccess;
  if (a.C % 8 || a.ldx % 8 || a.ldo % 8 || a.C > 8192) return hipErrorInvalidValue;
  if ((a.out && a.out_dtype == DT_FP8) || (a.out_b && a.out_b_dtype == DT_FP8)) return hipErrorInvalidValue;   // e4m3 goes through out_fp8
  if (a.stats && a.C > 2048) return hipErrorInvalidValue;   // the four-waves-per-row kernel does not write them
  switch (a.in_dtype) {
    case DT_F32: return launch_ln_dt<DT_F32>(a, st);
    case DT_BF16: return launch_ln_dt<DT_BF16>(a, st);
    case DT_F16: return launch_ln_dt<DT_F16>(a, st);
  }
  return hipErrorInvalidValue;
}

// ---- embedding ------------------------------------------------------------------------
// A wave per token; lane p holds feature p. At few tokens the launch is one wave's trips to memory, beyond them the activation and the
// norm on the vector units. The weight rows of the features that are not zero (3 to 8 of 19) are requested EMB_ROWS at a time, all vectors of
// a row together (one by one, each behind a branch and its own wait: 8.6 us for 64 tokens of 1024, 12.2 for 4096, 89 for 64000; now 6.4,
// 9.7 and 81). Two rows at a time and scale, offset and gates read where they are used keep six or more waves on a SIMD: with four rows and
// those reads up front 64 tokens take 6.1 but 64000 105 us; a wave that keeps them in registers and walks a square of several
// positions was no faster anywhere.
constexpr int EMB_ROWS = 2;
template <int VPL>
__global__ void __launch_bounds__(256) embed_kernel(const EmbedArgs a) {
  const int lane = threadIdx.x & 63;
  const int tok = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (tok >= a.tokens) return;
  const int sqr = tok & 63;
  float f = 0.f;
  if (a.planes) {
    if (lane < 19) f = a.planes[(long)tok * 19 + lane];
  } else {
    const int id = a.ids[tok];
    const uint8_t* fl = a.flags + (tok >> 6) * 4;
    if (lane < 12) f = id == lane + 1 ? 1.f : 0.f;
    else if (lane == 12) f = fl[0] ? 1.f : 0.f;
    else if (lane == 13) f = fl[2] == sqr ? 1.f : 0.f;
    else if (lane < 18) f = (fl[1] >> (lane - 14)) & 1 ? 1.f : 0.f;
    else if (lane == 18) f = fminf((float)fl[3] / 100.0f, 1.0f);
  }
  float x[VPL][8];
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int col = (i * 64 + lane) * 8;
    if (col < a.C) load8<DT_F32>(a.b1, col, x[i]);
  }
  uint32_t left = (uint32_t)__ballot(f != 0.f);   // the features that are not zero, added in their order
  while (left) {
    float w[EMB_ROWS][VPL][8], fv[EMB_ROWS];
    int cnt = 0;
#pragma unroll
    for (int k = 0; k < EMB_ROWS; ++k)
      if (left) {
        const int p = __builtin_ctz(left);
        left &= left - 1;
        cnt = k + 1;
        fv[k] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), p));
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
          const int col = (i * 64 + lane) * 8;
          if (col < a.C) load8<DT_F32>(a.w1t, (long)p * a.C + col, w[k][i]);
        }
      }
#pragma unroll
    for (int k = 0; k < EMB_ROWS; ++k)
      if (k < cnt) {
#pragma unroll
        for (int i = 0; i < VPL; ++i)
          if ((i * 64 + lane) * 8 < a.C) {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[i][e] = fmaf(fv[k], w[k][i][e], x[i][e]);
          }
      }
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; ++i)
    if ((i * 64 + lane) * 8 < a.C) {
#pragma unroll
      for (int e = 0; e < 8; ++e) { x[i][e] = apply_act(x[i][e], a.act); s += x[i][e]; }
    }
  // (1 / C by the hardware reciprocal, exact for the power-of-two widths and within one unit in the last place otherwise)
  const float inv_c = fast_rcp((float)a.C);
  const float mean = wave_sum(s) * inv_c;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; ++i)
    if ((i * 64 + lane) * 8 < a.C) {
#pragma unroll
      for (int e = 0; e < 8; ++e) { const float d = x[i][e] - mean; q += d * d; }
    }
  const float rstd = rsqrtf(wave_sum(q) * inv_c + a.eps);
  const long orow = a.out_T > 64 ? (long)(tok >> 6) * a.out_T + sqr : (long)tok;
  float am = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int col = (i * 64 + lane) * 8;
    if (col < a.C) {
      float y[8];
      float lg[8], lb[8], ga[8], gb[8];
      load8<DT_F32>(a.ln_g, col, lg);
      load8<DT_F32>(a.ln_b, col, lb);
      load8<DT_F32>(a.gate_a_exp, (long)sqr * a.C + col, ga);
      load8<DT_F32>(a.gate_b, (long)sqr * a.C + col, gb);
#pragma unroll
      for (int e = 0; e < 8; ++e) y[e] = ((x[i][e] - mean) * rstd * lg[e] + lb[e]) * ga[e] + gb[e];
      if (a.pe) {
        float pe[8];
        load8<DT_F32>(a.pe, (long)sqr * a.C + col, pe);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] += pe[e];
      }
      store8(a.out, orow * a.C + col, y, a.out_dtype);
      if (a.out_b) store8(a.out_b, orow * a.C + col, y, a.out_b_dtype);
      if (a.out_fp8) store8_fp8(a.out_fp8, orow * a.C + col, y, a.fp8_scale);
      if (a.amax) {
#pragma unroll
        for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(y[e]));
      }
    }
  }
  if (a.amax) {
    am = wave_max(am);
    if (lane == 0) atomic_amax(a.amax, am);
  }
}

// One workgroup per (position, move token).
__global__ void __launch_bounds__(256) token_embed_kernel(const TokenEmbedArgs a) {
  const int b = blockIdx.x / a.t, j = blockIdx.x - b * a.t;
  long id = a.idx[(long)b * a.t + j];
  id = id < 0 ? 0 : id >= a.V ? a.V - 1 : id;
  const float* w = a.wte + id * a.C;
  const float* pe = a.pe + (long)(64 + j) * a.C;
  const long row = (long)b * a.T + 64 + j;
  for (int c = threadIdx.x; c < a.C; c += 256) {
    const float v = w[c] + pe[c];
    if (a.out_dtype == DT_F32) reinterpret_cast<float*>(a.out)[row * a.C + c] = v;
    else if (a.out_dtype == DT_BF16) reinterpret_cast<uint16_t*>(a.out)[row * a.C + c] = f32_to_bf16_bits(v);
    else reinterpret_cast<uint16_t*>(a.out)[row * a.C + c] = f32_to_f16_bits(v);
  }
}

hipError_t launch_token_embed(const TokenEmbedArgs& a, hipStream_t st) {
  if (a.B <= 0 || a.t <= 0) return hipSuccess;
  if (!a.idx || !a.wte || !a.pe || !a.out || a.T != 64 + a.t || a.out_dtype == DT_FP8) return hipErrorInvalidValue;
  hipLaunchKernelGGL(token_embed_kernel, dim3(a.B * a.t), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_embed(const EmbedArgs& a, hipStream_t st) {
  if (a.tokens <= 0) return hipSuccess;
  if (a.C % 8 || a.C > 2048) return hipErrorInvalidValue;
  const int vecs = (a.C / 8 + 63) / 64;
  const int waves = a.tokens <= 2 * device_cus() ? 1 : 4;   // (few tokens: a wave alone on its compute unit has the shortest chain)
  const dim3 grid((a.tokens + waves - 1) / waves), block(64 * waves);
  if (vecs <= 1) hipLaunchKernelGGL((embed_kernel<1>), grid, block, 0, st, a);
  else if (vecs <= 2) hipLaunchKernelGGL((embed_kernel<2>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((embed_kernel<4>), grid, block, 0, st, a);
  return hipGetLastError();
}

}  // namespace crl
