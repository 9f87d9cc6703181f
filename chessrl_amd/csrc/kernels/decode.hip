// Incremental decoding for the GPT model: the kernels that let one new token per sequence be
// processed against cached keys and values instead of re-running the whole prefix, plus the
// on-device sampling step. Replaces the per-step full recomputation of
// GPT.generate_sequence / generate_sequence_raw (model_bis.py:213-263, 266-311).
#include "common.hpp"

namespace crl {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// ---- K|V of a freshly computed prefix into the cache ------------------------------------------
// qkv [B*T, 3C] (q|k|v per row) -> cache [B, Tmax, 2C] (k|v per row), 16-bit elements, 16 bytes per thread.
__global__ void __launch_bounds__(256) kv_store_kernel(const uint16_t* qkv, uint16_t* cache, int B, int T, int Tmax, int C) {
  const int chunks = 2 * C / 8;
  const long n = (long)B * T * chunks;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
    const long row = i / chunks;
    const int c = (int)(i - row * chunks);
    const int b = (int)(row / T), s = (int)(row - (long)b * T);
    const uint4 v = *reinterpret_cast<const uint4*>(qkv + row * 3 * C + C + 8 * c);
    *reinterpret_cast<uint4*>(cache + ((long)b * Tmax + s) * 2 * C + 8 * c) = v;
  }
}

hipError_t launch_kv_store(const void* qkv, void* cache, int B, int T, int Tmax, int C, hipStream_t st) {
  if (B <= 0 || T <= 0) return hipSuccess;
  if (C % 8 || T > Tmax) return hipErrorInvalidValue;
  const long n = (long)B * T * (2 * C / 8);
  const int grid = (int)std::min<long>((n + 255) / 256, 8192);
  hipLaunchKernelGGL(kv_store_kernel, dim3(grid), dim3(256), 0, st, reinterpret_cast<const uint16_t*>(qkv), reinterpret_cast<uint16_t*>(cache), B, T, Tmax, C);
  return hipGetLastError();
}

// staging [B, 2C] (k|v of the newest token) -> its row of every sequence's cache
__global__ void __launch_bounds__(256) kv_append_kernel(const uint16_t* staging, uint16_t* cache, int B, int Tmax, int C, int pos, const int* dyn_k) {
  const int row = dyn_k ? 64 + dyn_k[0] : pos;
  const int chunks = 2 * C / 8;
  const int n = B * chunks;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    const int b = i / chunks, c = i - b * chunks;
    *reinterpret_cast<uint4*>(cache + ((long)b * Tmax + row) * 2 * C + 8 * c) = *reinterpret_cast<const uint4*>(staging + (long)b * 2 * C + 8 * c);
  }
}

hipError_t launch_kv_append(const void* staging, void* cache, int B, int Tmax, int C, int pos, const int* dyn_k, hipStream_t st) {
  if (B <= 0) return hipSuccess;
  if (C % 8 || (!dyn_k && (pos < 0 || pos >= Tmax))) return hipErrorInvalidValue;
  const int n = B * (2 * C / 8);
  hipLaunchKernelGGL(kv_append_kernel, dim3(std::min((n + 255) / 256, 1024)), dim3(256), 0, st, reinterpret_cast<const uint16_t*>(staging),
                     reinterpret_cast<uint16_t*>(cache), B, Tmax, C, pos, dyn_k);
  return hipGetLastError();
}

__global__ void add_int_kernel(int* p, int v) { p[0] += v; }
hipError_t launch_add_int(int* p, int v, hipStream_t st) {
  hipLaunchKernelGGL(add_int_kernel, dim3(1), dim3(1), 0, st, p, v);
  return hipGetLastError();
}

// ---- one query against the cache -------------------------------------------------------------------
// One workgroup of four waves per (sequence, head). A key or value row of the head (HS elements) is read by HS/8
// neighbouring lanes, 16 bytes each, so a wave instruction covers 64/(HS/8) whole rows; the waves take such row groups
// in turn. Scores go to LDS, every wave derives the same max and sum from them, each wave accumulates p*V over its own
// rows, and the four partial outputs are added in wave order.
// Bound by memory (128 sequences of 160 tokens, 12 heads of 64: 63 MB). A lane's first 256 tokens are requested at once, keys in front of the scores and values in front
// of the softmax, eight loads in flight per wave either way in the same registers; both in front of the scores takes 64 registers more and a third of the waves (whole rollout of
// 128 sequences, 191 tokens: 54.7 ms with the values asked for behind the softmax, 55.0 both in front, 54.3 as it is).
// NT: the rows are read with the non-temporal hint (past).
constexpr int DEC_TMAX = 1024;

template <bool NT>
__device__ __forceinline__ u32x4_t kv_rows(__amdgpu_buffer_rsrc_t r, int off) { return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, NT ? 2 : 0); }

template <int HS, int IN_DT, bool NT>
__global__ void __launch_bounds__(256) decode_attention_kernel(const uint16_t* q, long ldq, const uint16_t* cache, int Tmax, int C, int n_arg,
                                                               const int* dyn_k, uint16_t* out, long ldo, int B, int H, float scale) {
  constexpr int LPK = HS / 8, KPI = 64 / LPK;    // lanes per key row, key rows per wave instruction
  constexpr int AHEAD = 256 / (4 * KPI);         // 256 tokens
  static_assert(LPK == 4 || LPK == 8, "head sizes 32 and 64");
  __shared__ float s_p[DEC_TMAX];
  __shared__ float s_acc[4][HS];
  const int n = dyn_k ? 65 + dyn_k[0] : n_arg;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int sub = lane % LPK, kin = lane / LPK;
  const int unit = blockIdx.x;
  const int b = unit / H, h = unit - b * H;
  auto unpack = [](const u32x4_t w, float (&f)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint16_t x = (uint16_t)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffff));
      f[e] = IN_DT == DT_BF16 ? bf16_bits_to_f32(x) : f16_bits_to_f32(x);
    }
  };
  float qv[8];
  // This lane's key and value rows j0 = wave KPI + kin + 4 KPI i, through descriptors that end with row n - 1 (zeros behind it), so that no branch stands between the requests.
  const uint16_t* const kbase = cache + (long)b * Tmax * 2 * C + h * HS;
  const int row_b = 4 * C, span = (n - 1) * row_b + HS * 2, j_first = wave * KPI + kin, voff = j_first * row_b + sub * 16;
  const __amdgpu_buffer_rsrc_t krows = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kbase), 0, span, 0x00020000);
  const __amdgpu_buffer_rsrc_t vrows = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kbase + C), 0, span, 0x00020000);
  u32x4_t kr[AHEAD], vr[AHEAD];
  const u32x4_t qu = *reinterpret_cast<const u32x4_t*>(q + (long)b * ldq + h * HS + sub * 8);
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) kr[i] = kv_rows<NT>(krows, voff + i * 4 * KPI * row_b);
  __builtin_amdgcn_sched_barrier(0);
  unpack(qu, qv);
  auto score = [&](int j, const u32x4_t& u) {
    float kv[8], s = 0.f;
    unpack(u, kv);
#pragma unroll
    for (int e = 0; e < 8; ++e) s = fmaf(qv[e], kv[e], s);
    s += dpp_move<DPP_XOR1>(s);
    s += dpp_move<DPP_XOR2>(s);
    if constexpr (LPK == 8) s += dpp_move<DPP_HALF_MIRROR>(s);
    if (sub == 0 && j < n) s_p[j] = s * scale;
  };
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
    if (i * 4 * KPI < n) score(j_first + i * 4 * KPI, kr[i]);
#pragma unroll 4
  for (int j = j_first + AHEAD * 4 * KPI; j - kin < n; j += 4 * KPI) score(j, kv_rows<NT>(krows, j * row_b + sub * 16));
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) vr[i] = kv_rows<NT>(vrows, voff + i * 4 * KPI * row_b);
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  float mx = -INFINITY;
  for (int j = lane; j < n; j += 64) mx = fmaxf(mx, s_p[j]);
  mx = wave_max(mx);
  float sum = 0.f;
  for (int j = lane; j < n; j += 64) sum += __expf(s_p[j] - mx);
  sum = wave_sum(sum);

  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  auto add = [&](int j, const u32x4_t& u) {
    if (j < n) {
      const float pj = __expf(s_p[j] - mx);
      float vv[8];
      unpack(u, vv);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] = fmaf(pj, vv[e], acc[e]);
    }
  };
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
    if (i * 4 * KPI < n) add(j_first + i * 4 * KPI, vr[i]);
#pragma unroll 4
  for (int j = j_first + AHEAD * 4 * KPI; j - kin < n; j += 4 * KPI) add(j, kv_rows<NT>(vrows, j * row_b + sub * 16));
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    // (distances LPK = 4 or 8, then 8, 16 and 32; at distance 4 the sums of a lane's neighbours are other dims', so no mirrored lane)
    if constexpr (LPK == 4) acc[e] += __shfl_xor(acc[e], 4, 64);
    acc[e] += dpp_move<DPP_XOR8>(acc[e]);
    acc[e] = add_xor32(add_xor16(acc[e]));
  }
  if (kin == 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) s_acc[wave][sub * 8 + e] = acc[e];
  }
  __syncthreads();
  if (threadIdx.x < HS) {
    const int d = threadIdx.x;
    const float v = (((s_acc[0][d] + s_acc[1][d]) + s_acc[2][d]) + s_acc[3][d]) / sum;
    out[(long)b * ldo + h * HS + d] = IN_DT == DT_BF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v);
  }
}

hipError_t launch_decode_attention(const void* q, long ldq, const void* cache, int Tmax, int C, int n, const int* dyn_k, void* out, long ldo,
                                   int B, int H, int head_dim, int in_dtype, float scale, bool past, hipStream_t st) {
  if (B <= 0) return hipSuccess;
  if (Tmax > DEC_TMAX || C % 8 || ldq % 8 || (reinterpret_cast<uintptr_t>(q) & 15) || (reinterpret_cast<uintptr_t>(cache) & 15) || (in_dtype != DT_BF16 && in_dtype != DT_F16)) return hipErrorInvalidValue;
  if (!dyn_k && (n < 1 || n > Tmax)) return hipErrorInvalidValue;
  const dim3 grid(B * H), block(256);
  const uint16_t* qp = reinterpret_cast<const uint16_t*>(q);
  const uint16_t* cp = reinterpret_cast<const uint16_t*>(cache);
  uint16_t* op = reinterpret_cast<uint16_t*>(out);
#define DEC_LAUNCH(HS, DT) hipLaunchKernelGGL((past ? decode_attention_kernel<HS, DT, true> : decode_attention_kernel<HS, DT, false>), grid, block, 0, st, qp, ldq, cp, Tmax, C, n, dyn_k, op, ldo, B, H, scale)
  if (head_dim == 32 && in_dtype == DT_BF16) DEC_LAUNCH(32, DT_BF16);
  else if (head_dim == 32) DEC_LAUNCH(32, DT_F16);
  else if (head_dim == 64 && in_dtype == DT_BF16) DEC_LAUNCH(64, DT_BF16);
  else if (head_dim == 64) DEC_LAUNCH(64, DT_F16);
  else return hipErrorInvalidValue;
#undef DEC_LAUNCH
  return hipGetLastError();
}

// ---- sampling ------------------------------------------------------------------------------------------
// One workgroup per sequence: softmax(logits/T) and one draw by inverse CDF (arg-max for T == 0), then the
// forced tokens of generate_sequence (model_bis.py:252-259) when rules != 0:
//   five end_variation tokens so far -> </thinking>; the token two places after </thinking> -> end.
// and, where asked for, the embedding of the token, wte[tok] + pe[64 + k] (model_bis.py:224, 233-235 for the last position only).
// Wave 0 draws: its lane l owns the contiguous classes [l*CH, l*CH+CH), so the CDF is a lane-level scan plus a short walk. The logits come
// in and the probabilities go out over all four waves, class by class; read and written by the owning lanes, each access touching
// 64 lines, the step took 15.9 us for 128 sequences and its embedding another 4.0; together they took 9.8, and 9.0 with what the rules and the
// embedding read requested beside the logits and the searches without the LDS crossbar.
constexpr int SAMPLE_CH = 32;

__device__ __forceinline__ float uniform01(uint64_t seed, uint64_t a, uint64_t b) {
  uint64_t z = seed + 0x9E3779B97F4A7C15ull * (a * 0x100000001B3ull + b + 1);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (float)(z >> 40) * (1.0f / 16777216.0f);
}

__global__ void __launch_bounds__(256) sample_kernel(const SampleArgs a) {
  __shared__ float s_v[64 * (SAMPLE_CH + 1)];
  __shared__ float s_max[4];
  __shared__ int s_idx[4];
  __shared__ float s_total;
  __shared__ long s_tok;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int b = blockIdx.x;
  const int k = a.dyn_k ? a.dyn_k[0] : a.k;
  const int step = a.dyn_k ? k : a.step;
  const float* x = a.logits + (long)b * a.ldl;
  const int ch = (a.V + 63) / 64;
  // class c of lane c / ch; an odd pitch keeps the lanes' walks through their classes off each other's banks
  const bool odd = (ch & 1) != 0;
  const int pitch = ch | 1;
  auto at = [&](int c) { return odd ? c : c + c / ch; };
  const float invT = a.temperature > 0.f ? 1.0f / a.temperature : 1.0f;
  constexpr int VPT = 64 * SAMPLE_CH / 256;
  float v[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = i * 256 + tid;
    v[i] = c < a.V ? x[c] * invT : -INFINITY;
  }
  // What the rules and the embedding read besides the draw, requested with the logits: behind the draw each would be a trip to memory of its own.
  int nz = 0;
  long two_back = -1;
  if (a.rules && tid == 0) {
    nz = a.num_zeros[b];
    if (k >= 2) two_back = a.seq[(long)b * a.ld_seq + k - 2];
  }
  float4 pe0 = make_float4(0.f, 0.f, 0.f, 0.f);
  if (a.emb_out && tid * 4 < a.emb_C) pe0 = *reinterpret_cast<const float4*>(a.pe + (long)(64 + k) * a.emb_C + tid * 4);
  float wmx = -INFINITY;
  int wi = 0x7fffffff;
#pragma unroll
  for (int i = 0; i < VPT; ++i)
    if (v[i] > wmx) { wmx = v[i]; wi = i * 256 + tid; }
  // arg-max with the lowest index among equals
  lowest_argmax(wmx, wi);
  if (lane == 0) { s_max[wave] = wmx; s_idx[wave] = wi; }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float om = s_max[w];
    const int oi = s_idx[w];
    if (om > wmx || (om == wmx && oi < wi)) { wmx = om; wi = oi; }
  }
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    v[i] = __expf(v[i] - wmx);
    const int c = i * 256 + tid;
    if (c < a.V) s_v[at(c)] = v[i];
  }
  __syncthreads();
  if (wave == 0) {
    float u[SAMPLE_CH];
    float lsum = 0.f;
#pragma unroll
    for (int i = 0; i < SAMPLE_CH; ++i) u[i] = (i < ch && lane * ch + i < a.V) ? s_v[lane * pitch + i] : 0.f;
#pragma unroll
    for (int i = 0; i < SAMPLE_CH; ++i) lsum += u[i];
    // inclusive scan of the lane sums
    float incl = lsum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float t = __shfl_up(incl, o, 64);
      if (lane >= o) incl += t;
    }
    const float total = __shfl(incl, 63, 64);
    long tok = wi;
    if (a.temperature > 0.f) {
      const float target = uniform01(a.seed, (uint64_t)b, (uint64_t)step) * total;
      const float excl = incl - lsum;
      // the first lane whose inclusive sum exceeds the target holds the draw
      const bool mine = target < incl && target >= excl;
      int pick = -1;
      if (mine) {
        float run = excl;
        pick = lane * ch;
#pragma unroll
        for (int i = 0; i < SAMPLE_CH; ++i) {
          if (i < ch && lane * ch + i < a.V) {
            if (u[i] > 0.f) pick = lane * ch + i;    // last class with mass at or before the crossing
            run += u[i];
            if (run > target) break;
          }
        }
      }
      // the last lane that has one; rounding can leave none (target == total): fall back to the arg-max
      const uint64_t have = __ballot(pick >= 0);
      if (have) tok = __builtin_amdgcn_readlane(pick, 63 - __builtin_clzll(have));
    }
    if (lane == 0) {
      if (a.rules) {
        if (nz == 5) { tok = a.end_think; nz = 6; }
        if (k >= 2 && two_back == a.end_think) tok = a.end_tok;
        nz += (tok == a.end_variation) ? 1 : 0;
        a.num_zeros[b] = nz;
      }
      a.seq[(long)b * a.ld_seq + k] = tok;
      a.tok_out[b] = tok;
      s_tok = tok;
      s_total = total;
    }
  }
  if (!a.step_out && !a.emb_out) return;
  __syncthreads();
  if (a.emb_out) {
    const long id = s_tok < 0 ? 0 : s_tok >= a.V ? a.V - 1 : s_tok;
    const float* wte = a.wte + id * a.emb_C;
    const float* pe = a.pe + (long)(64 + k) * a.emb_C;
    for (int c = tid * 4; c < a.emb_C; c += 1024) {
      const float4 w = *reinterpret_cast<const float4*>(wte + c), p = c == tid * 4 ? pe0 : *reinterpret_cast<const float4*>(pe + c);
      const float4 r = make_float4(w.x + p.x, w.y + p.y, w.z + p.z, w.w + p.w);
      const long o = (long)b * a.emb_C + c;
      if (a.emb_dtype == DT_F32) *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.emb_out) + o) = r;
      else if (a.emb_dtype == DT_BF16) *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.emb_out) + o) = make_uint2(pack_bf16x2(r.x, r.y), pack_bf16x2(r.z, r.w));
      else
        *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.emb_out) + o) =
            make_uint2((uint32_t)f32_to_f16_bits(r.x) | ((uint32_t)f32_to_f16_bits(r.y) << 16), (uint32_t)f32_to_f16_bits(r.z) | ((uint32_t)f32_to_f16_bits(r.w) << 16));
    }
  }
  if (a.step_out) {
    float* o = a.step_out + (long)b * a.ld_out + (a.dyn_k ? (long)(k - 1) * a.V : 0);
    const float inv = 1.0f / s_total;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int c = i * 256 + tid;
      if (c < a.V) o[c] = a.out_logits ? x[c] : v[i] * inv;
    }
  }
}

hipError_t launch_sample(const SampleArgs& a, hipStream_t st) {
  if (a.B <= 0) return hipSuccess;
  if (!a.logits || !a.seq || !a.tok_out || a.V <= 0 || a.V > 64 * SAMPLE_CH || (a.rules && !a.num_zeros)) return hipErrorInvalidValue;
  if (a.emb_out && (!a.wte || !a.pe || a.emb_C % 4 || a.emb_dtype == DT_FP8)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(sample_kernel, dim3(a.B), dim3(256), 0, st, a);
  return hipGetLastError();
}

}  // namespace crl
