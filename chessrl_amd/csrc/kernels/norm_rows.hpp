// Eight consecutive elements of a row, in and out of fp32: what the norm kernels and the product with a norm in front share.
#pragma once
#include "common.hpp"

namespace crl {

template <int DT>
__device__ __forceinline__ void load8(const void* base, long off, float v[8]) {
  if constexpr (DT == DT_F32) {
    const float4* p = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(base) + off);
    float4 a = p[0], b = p[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  } else {
    uint4 u = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(base) + off);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (DT == DT_BF16) {
        v[2 * i] = bf16_bits_to_f32((uint16_t)(w[i] & 0xffff));
        v[2 * i + 1] = bf16_bits_to_f32((uint16_t)(w[i] >> 16));
      } else {
        v[2 * i] = f16_bits_to_f32((uint16_t)(w[i] & 0xffff));
        v[2 * i + 1] = f16_bits_to_f32((uint16_t)(w[i] >> 16));
      }
    }
  }
}

__device__ __forceinline__ void store8(void* base, long off, const float v[8], int dt) {
  if (dt == DT_F32) {
    float4* p = reinterpret_cast<float4*>(reinterpret_cast<float*>(base) + off);
    p[0] = make_float4(v[0], v[1], v[2], v[3]);
    p[1] = make_float4(v[4], v[5], v[6], v[7]);
  } else if (dt == DT_BF16) {
    uint4 u = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
    *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(base) + off) = u;
  } else {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = (uint32_t)f32_to_f16_bits(v[2 * i]) | ((uint32_t)f32_to_f16_bits(v[2 * i + 1]) << 16);
    *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(base) + off) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

__device__ __forceinline__ void store8_fp8(uint8_t* base, long off, const float v[8], float scale) {
  uint2 u = make_uint2(pack_fp8x4(v[0] * scale, v[1] * scale, v[2] * scale, v[3] * scale),
                       pack_fp8x4(v[4] * scale, v[5] * scale, v[6] * scale, v[7] * scale));
  *reinterpret_cast<uint2*>(base + off) = u;
}

// Which columns a lane holds of a row spread over a wave, four consecutive ones at a time (i: vector of eight, h: its half). 16-bit rows:
// eight consecutive columns, one 16-byte access. fp32 rows: two accesses of 16 bytes per lane, each over 1 KB without gaps.
__device__ __forceinline__ int norm_column(bool f32, int i, int h, int lane) { return f32 ? ((2 * i + h) * 64 + lane) * 4 : (i * 64 + lane) * 8 + 4 * h; }

// The eight values of vector i (columns past C are left alone).
template <int DT>
__device__ __forceinline__ void load_norm8(const void* base, long row_off, int i, int lane, int C, float (&v)[8]) {
  if constexpr (DT == DT_F32) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int col = norm_column(true, i, h, lane);
      if (col < C) {
        const float4 u = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(base) + row_off + col);
        v[4 * h] = u.x; v[4 * h + 1] = u.y; v[4 * h + 2] = u.z; v[4 * h + 3] = u.w;
      }
    }
  } else {
    const int col = norm_column(false, i, 0, lane);
    if (col < C) load8<DT>(base, row_off + col, v);
  }
}

__device__ __forceinline__ void store4(void* base, long off, const float* v, int dt) {
  if (dt == DT_F32) *reinterpret_cast<float4*>(reinterpret_cast<float*>(base) + off) = make_float4(v[0], v[1], v[2], v[3]);
  else if (dt == DT_BF16) *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(base) + off) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  else
    *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(base) + off) =
        make_uint2((uint32_t)f32_to_f16_bits(v[0]) | ((uint32_t)f32_to_f16_bits(v[1]) << 16), (uint32_t)f32_to_f16_bits(v[2]) | ((uint32_t)f32_to_f16_bits(v[3]) << 16));
}
__device__ __forceinline__ void store4_fp8(uint8_t* base, long off, const float* v, float scale) {
  *reinterpret_cast<uint32_t*>(base + off) = pack_fp8x4(v[0] * scale, v[1] * scale, v[2] * scale, v[3] * scale);
}

}  // namespace crl
