// Fused 64-token multi-head attention: one 64-lane wave per unit, i.e. (position, head); two where there are few of them.
//
// Replaces F.scaled_dot_product_attention(q,k,v,is_causal=True) of model_bis.py:71 and
// the score/softmax/context chain of RelativeMultiHeadAttention2.forward
// (new_paradigm/attn.py:507-521), including the pad-and-reshape relative shift of
// new_paradigm/attn.py:525-533. A third mode adds a generated per-head 64x64 bias
// before the softmax (the BT4-class configuration).
//
// The wave computes the TRANSPOSED score tile S^T[j][i] = K[j]·Q[i] with 32x32x16
// MFMAs whose operands are 16-byte row segments read straight from global memory
// (both Q and K are head-dim contiguous). In the accumulator layout a lane then owns
// one query i and 32 of its 64 keys j, so the softmax over keys is a reduction over
// the lane's own registers plus one exchange with lane^32. The probabilities are
// re-used in place as the column operand of the second product O^T = V^T · P^T; only V
// needs a transpose, which goes through a wave-private LDS patch.
#include "common.hpp"

#include <type_traits>

namespace crl {

constexpr int VT_STRIDE = 68;   // bf16 elements per V^T row (64 keys + 4 padding: rows 8 apart land 16 banks apart, so the transposing
                                // 8-byte writes and the fragment reads of a wave touch every bank twice, the minimum; with 72 it was eight and four times)
constexpr int SP_STRIDE = 66;   // floats per row of the positional score patch: the shifted read-back of a wave walks it in steps of one less, an odd number
                                // (with 65 all 32 rows of a read lay in one bank: 71 us per layer of 496 positions of 8 heads, 49 with the other)

// Storage order of a 64x64 bias tile so that each lane reads its accumulator
// registers as 16-byte vectors: element (query i, key j) lives at
//   ((((i/32)*2 + j/32)*2 + rh)*64 + lane)*8 + e
// with lane = (i%32) + 32*g, j%32 = 8*(2*rh + e/4) + 4*g + e%4.
__host__ __device__ inline int attn_bias_slot(int i, int j) {
  const int it = i >> 5, jt = j >> 5, jj = j & 31;
  const int q4 = jj >> 3, g = (jj >> 2) & 1, e0 = jj & 3;
  const int rh = q4 >> 1, e = ((q4 & 1) << 2) | e0;
  const int lane = (i & 31) + 32 * g;
  return ((((it * 2 + jt) * 2 + rh) * 64 + lane) << 3) + e;
}

// The two 16-bit element types the kernel runs in.
template <int DT>
struct Half16;
template <>
struct Half16<DT_BF16> {
  typedef bf16x8_t vec;
  typedef __bf16 elem;
  static __device__ __forceinline__ f32x16_t mfma(vec a, vec b, f32x16_t c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ float to_f32(uint16_t h) { return bf16_bits_to_f32(h); }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) { return pack_bf16x2(lo, hi); }
};
template <>
struct Half16<DT_F16> {
  typedef f16x8_t vec;
  typedef _Float16 elem;
  static __device__ __forceinline__ f32x16_t mfma(vec a, vec b, f32x16_t c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
  static __device__ __forceinline__ float to_f32(uint16_t h) { return f16_bits_to_f32(h); }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) { return (uint32_t)f32_to_f16_bits(lo) | ((uint32_t)f32_to_f16_bits(hi) << 16); }
};

// This wave's LDS writes are done and seen by its later reads.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename H>
__device__ __forceinline__ typename H::vec add_bias_h(typename H::vec q, const float* bias8) {
  typename H::vec r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = (typename H::elem)((float)q[e] + bias8[e]);
  return r;
}

// Waves per workgroup (of the form with one wave per unit). With a generated bias a workgroup takes eight
// heads of a position (eight waves): per token row it then reads 512 contiguous bytes of each of q, k and v, its bias is
// 2 KB pieces of the blocked layout and its e4m3 output rows are two whole lines (measured 9.07 -> 8.53 ms per
// 4096-position forward against four waves; sixteen waves, one workgroup per CU, 9.71 ms).
template <int MODE>
struct AttnWaves { static constexpr int N = MODE == ATTN_BIAS ? 8 : 4; };

// Waves per SIMD the register allocation is held to (0: the compiler's own choice). The kernel is a chain of load,
// compute and store phases, so resident waves are what hides its memory latency: at head size 32 with a generated
// bias it fits 4 waves in 122 registers without spilling (152 and 3 waves left alone; measured 10.8 -> 9.6 ms per
// 4096-position forward; 5 waves spill and are slower). The other instances spill at that bound and keep theirs.
// 16 bytes that the kernel reads once: loaded with the non-temporal hint so that they do not displace what other kernels
// will want from the caches.
__device__ __forceinline__ uint4 attn_load_once(const void* p) {
  typedef int i32x4_nt __attribute__((ext_vector_type(4)));
  const i32x4_nt v = __builtin_nontemporal_load(reinterpret_cast<const i32x4_nt*>(p));
  return make_uint4((uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]);
}

template <int HS, int MODE>
struct AttnMinWaves { static constexpr int N = (HS == 32 && MODE == ATTN_BIAS) ? 4 : 0; };

// OUT_FP8: write e4m3 (value*out_scale) instead of the input element type.
// COOP: the workgroup's outputs leave through an LDS tile as whole row segments (see s_out below; the launcher says when).
// SPLIT: a workgroup is one unit, its two waves take a query tile each and transpose half of V each.
// LAST (ATTN_CAUSAL): only token 63's output is wanted: the query tile of tokens 32..63 alone runs and that one row is stored, at row b.
template <int HS, int MODE, int OUT_FP8, int IN_DT, int COOP = 0, int LAST = 0, int SPLIT = 0>
__global__ void __launch_bounds__(SPLIT ? 128 : 64 * AttnWaves<MODE>::N, (SPLIT ? 0 : AttnMinWaves<HS, MODE>::N)) attention_kernel(const AttnArgs a) {
  typedef Half16<IN_DT> H16;
  typedef typename H16::vec hvec;
  constexpr int KS = HS / 16;   // k-steps of the score product
  constexpr int DT_TILES = HS / 32;
  constexpr int NW = SPLIT ? 1 : AttnWaves<MODE>::N;   // units of the workgroup
  __shared__ __align__(16) uint16_t s_vt[NW][HS * VT_STRIDE];
  // Output tile of the workgroup's NW heads (head size 32): 64 rows of NW * HS elements, 16 bytes of padding
  // per row. A wave's own output is 64 row pieces of 32 (e4m3) or 64 bytes, which it would have to store 16 bytes per
  // lane and row, a quarter or an eighth of a line at a time; gathered here, the workgroup stores whole lines (measured
  // on 4096 positions x 32 heads in e4m3: the stores were 9 % of the kernel's bytes and 21 % of its time).
  static_assert(!LAST || (MODE == ATTN_CAUSAL && !COOP), "one-row form");
  static_assert(!SPLIT || (!COOP && !LAST), "one query tile per wave");
  static_assert(MODE != ATTN_RELSHIFT, "the relative mode has a kernel of its own");
  constexpr int NIT = LAST || SPLIT ? 1 : 2;   // query tiles of a wave
  static_assert(!COOP || (HS == 32 && (NW == 4 || NW == 8 || NW == 16)), "the output tile is laid out for head size 32");
  constexpr int OSZ = OUT_FP8 ? 1 : 2;
  constexpr int OROW = NW * HS * OSZ, OSTRIDE = OROW + 16;
  __shared__ __align__(16) uint8_t s_out[COOP ? 64 * OSTRIDE : 16];

  // A wave that starts gets its loads out ahead of its neighbours' arithmetic: raised priority until the score product
  // begins (which also keeps every load above that point: 8.49 -> 8.31 ms per 4096-position forward).
  if constexpr (MODE == ATTN_BIAS) __builtin_amdgcn_s_setprio(3);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lr = lane & 31, g = lane >> 5;
  // (workgroup indices go round the eight XCDs: renumbered so that each XCD walks a contiguous range of units)
  int bid = blockIdx.x;
  {
    const int per = gridDim.x >> 3;
    if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
  }
  const int unit = SPLIT ? bid : bid * NW + wave;
  const int it0 = LAST ? 1 : SPLIT ? wave : 0;   // the first of them
  if (unit >= a.B * a.H) return;
  const int b = unit / a.H, h = unit - b * a.H;
  constexpr bool coop = COOP != 0;

  const int qk_hst = a.qk_hstride ? a.qk_hstride : HS;
  const bool qk_once = a.qk_hstride != 0;   // q and k of a head share lines with nobody else
  const uint16_t* qp = reinterpret_cast<const uint16_t*>(a.q) + (long)b * 64 * a.ldq + h * qk_hst;
  const uint16_t* kp = reinterpret_cast<const uint16_t*>(a.k) + (long)b * 64 * a.ldk + h * qk_hst;
  const uint16_t* vp = reinterpret_cast<const uint16_t*>(a.v) + (long)b * 64 * a.ldv + h * HS;

  // ---- V -> V^T in LDS ------------------------------------------------------------
  uint16_t* vt = s_vt[SPLIT ? 0 : wave];
  // V rows of this wave (SPLIT: half of the unit's each; with a single pass half the lanes of each wave), four of one 16-byte chunk a lane and pass.
  constexpr int DC = HS / 8;            // 16-byte chunks per V row
  constexpr int PASSES = (16 * DC) / 64, MYP = SPLIT && PASSES > 1 ? PASSES / 2 : PASSES;
  i32x4_t vrow4[MYP][4];
  const bool v_mine = !(SPLIT && PASSES == 1 && g);
  auto v_id = [&](int p) { return SPLIT ? (PASSES == 1 ? 32 * wave + lr : (wave * MYP + p) * 64 + lane) : p * 64 + lane; };
  auto v_load = [&]() {
#pragma unroll
    for (int p = 0; p < MYP; ++p)
      if (v_mine) {
        const int id = v_id(p), jq = id / DC, dc = id - jq * DC;
#pragma unroll
        for (int t = 0; t < 4; ++t) vrow4[p][t] = *reinterpret_cast<const i32x4_t*>(vp + (long)(4 * jq + t) * a.ldv + 8 * dc);
      }
  };
  auto v_write = [&]() {
#pragma unroll
    for (int p = 0; p < MYP; ++p)
      if (v_mine) {
        const int id = v_id(p), jq = id / DC, dc = id - jq * DC;
#pragma unroll
        for (int e2 = 0; e2 < 4; ++e2) {
          // d = 8dc + 2e2 (low halves) and d+1 (high halves)
          const uint32_t w0 = (uint32_t)vrow4[p][0][e2], w1 = (uint32_t)vrow4[p][1][e2], w2 = (uint32_t)vrow4[p][2][e2], w3 = (uint32_t)vrow4[p][3][e2];
          *reinterpret_cast<uint2*>(vt + (8 * dc + 2 * e2) * VT_STRIDE + 4 * jq) = make_uint2((w0 & 0xffffu) | (w1 << 16), (w2 & 0xffffu) | (w3 << 16));
          *reinterpret_cast<uint2*>(vt + (8 * dc + 2 * e2 + 1) * VT_STRIDE + 4 * jq) = make_uint2((w0 >> 16) | (w1 & 0xffff0000u), (w2 >> 16) | (w3 & 0xffff0000u));
        }
      }
  };
  // VPAIR: the two waves of a pair of neighbouring heads (a token's V rows of the two are one whole 128-byte line) take
  // half the tokens each, for both heads: every line is read by one wave, once, with the non-temporal hint, and lands
  // transposed in the patch of the head it belongs to; the workgroup meets at a barrier before the second product.
  constexpr bool VPAIR = COOP != 0 && MODE == ATTN_BIAS && HS == 32 && NW % 2 == 0;
  if constexpr (VPAIR) {
    const int half = wave & 1;
    const uint16_t* vp2 = vp - half * HS;
    const int dc8 = lane & 7, jq8 = lane >> 3;
    uint4 rows[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) rows[t] = attn_load_once(vp2 + (long)(32 * half + 4 * jq8 + t) * a.ldv + 8 * dc8);
    uint16_t* vt2 = s_vt[(wave & ~1) + (dc8 >> 2)];
    const int dc = dc8 & 3, jq = 8 * half + jq8;
    const uint32_t* w0 = reinterpret_cast<const uint32_t*>(&rows[0]);
    const uint32_t* w1 = reinterpret_cast<const uint32_t*>(&rows[1]);
    const uint32_t* w2 = reinterpret_cast<const uint32_t*>(&rows[2]);
    const uint32_t* w3 = reinterpret_cast<const uint32_t*>(&rows[3]);
#pragma unroll
    for (int e2 = 0; e2 < 4; ++e2) {
      uint2 lo = make_uint2((w0[e2] & 0xffffu) | (w1[e2] << 16), (w2[e2] & 0xffffu) | (w3[e2] << 16));
      uint2 hi = make_uint2((w0[e2] >> 16) | (w1[e2] & 0xffff0000u), (w2[e2] >> 16) | (w3[e2] & 0xffff0000u));
      *reinterpret_cast<uint2*>(vt2 + (8 * dc + 2 * e2) * VT_STRIDE + 4 * jq) = lo;
      *reinterpret_cast<uint2*>(vt2 + (8 * dc + 2 * e2 + 1) * VT_STRIDE + 4 * jq) = hi;
    }
  } else {
    v_load();
    v_write();
  }

  // ---- scores -----------------------------------------------------------------------
  hvec qf[NIT][KS], kf[2][KS];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const uint16_t* ka = kp + (long)(32 * t + lr) * a.ldk + 16 * ks + 8 * g;
      if (t < NIT) {
        const uint16_t* qa = qp + (long)(32 * (it0 + t) + lr) * a.ldq + 16 * ks + 8 * g;
        qf[t][ks] = qk_once ? __builtin_bit_cast(hvec, attn_load_once(qa)) : *reinterpret_cast<const hvec*>(qa);
      }
      kf[t][ks] = qk_once ? __builtin_bit_cast(hvec, attn_load_once(ka)) : *reinterpret_cast<const hvec*>(ka);
    }

  // The bias tile (8 KB per wave), requested behind V, q and k: loads return in the order of their issue, which is now
  // the order of their use, and all twenty are out before the first of them is waited for.
  uint4 braw[NIT][2][2];
  if constexpr (MODE == ATTN_BIAS) {
    // Element k = 512 L + 8 lane + e of the unit's 4096 (L = (it, jt, rh)): row-major, or in blocks of 256 units x 128
    // elements (the layout the bias generator's GEMM writes fastest), where a load of 1 KB is four pieces of 256 bytes.
    const uint16_t* bp = reinterpret_cast<const uint16_t*>(a.bias);
    long lstride = 512;
    if (a.bias_blocked) {
      bp += (long)(unit >> 8) * (256 * 4096) + ((long)(lane >> 4) * 256 + (unit & 255)) * 128 + ((lane & 15) << 3);
      lstride = 4 * 256 * 128;
    } else {
      bp += (long)unit * 4096 + (lane << 3);
    }
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int jt = 0; jt < 2; ++jt)
#pragma unroll
        for (int rh = 0; rh < 2; ++rh)
          braw[it][jt][rh] = attn_load_once(bp + (((it0 + it) * 2 + jt) * 2 + rh) * lstride);
  }

  if constexpr (MODE == ATTN_BIAS) __builtin_amdgcn_s_setprio(0);
  f32x16_t s[2][NIT];  // [jt][it]
#pragma unroll
  for (int jt = 0; jt < 2; ++jt)
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[jt][it][r] = 0.f;

  {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int jt = 0; jt < 2; ++jt)
#pragma unroll
        for (int it = 0; it < NIT; ++it)
          s[jt][it] = H16::mfma(kf[jt][ks], qf[it][ks], s[jt][it]);

    if constexpr (MODE == ATTN_BIAS) {
#pragma unroll
      for (int it = 0; it < NIT; ++it)
#pragma unroll
        for (int jt = 0; jt < 2; ++jt)
#pragma unroll
          for (int rh = 0; rh < 2; ++rh) {
            const uint4 u = braw[it][jt][rh];
            const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float bv = H16::to_f32((uint16_t)((e & 1) ? (w[e >> 1] >> 16) : (w[e >> 1] & 0xffff)));
              s[jt][it][8 * rh + e] = s[jt][it][8 * rh + e] * a.scale + bv;
            }
          }
    }
  }

  // ---- softmax over keys (registers + lane^32) ------------------------------------------
  // tc: the query tile, which the causal test wants as a constant: keys of a later tile than the queries' have no weight, those of an earlier one are all
  // seen, and only in between is there anything to test. Every instance multiplies and subtracts in the same steps (a fused multiply-add where
  // the scaled score is not changed in between), so that a row does not depend on the instance.
  float inv_l[NIT];
  auto softmax = [&](int it, auto tc) {
    constexpr int TILE = decltype(tc)::value;
    constexpr bool SCALED = MODE == ATTN_BIAS;   // (the scores are finished)
    constexpr int JT = MODE == ATTN_CAUSAL ? TILE + 1 : 2;
    float mx = -INFINITY;
#pragma unroll
    for (int jt = 0; jt < JT; ++jt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float x = s[jt][it][r];
        if constexpr (!SCALED) {
          x *= a.scale;
          if (MODE == ATTN_CAUSAL && jt == TILE) {
            const int j = 8 * (r >> 2) + 4 * g + (r & 3);   // (within the tile)
            if (j > lr) x = -INFINITY;
            s[jt][it][r] = x;
          }
        }
        mx = fmaxf(mx, x);
      }
    mx = max_xor32(mx);
    float sum = 0.f;
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float p = 0.f;
        if (jt < JT) p = __expf(SCALED || (MODE == ATTN_CAUSAL && jt == TILE) ? s[jt][it][r] - mx : fmaf(s[jt][it][r], a.scale, -mx));
        s[jt][it][r] = p;
        sum += p;
      }
    sum = add_xor32(sum);
    inv_l[it] = 1.0f / sum;
  };
  typedef std::integral_constant<int, 0> T0;
  typedef std::integral_constant<int, 1> T1;
  if constexpr (NIT == 2) {
    softmax(0, T0{});
    softmax(1, T1{});
  } else if (it0 == 1 && MODE == ATTN_CAUSAL) {
    softmax(0, T1{});
  } else {
    softmax(0, T0{});
  }

  // ---- O^T = V^T · P^T ------------------------------------------------------------------
  if constexpr (VPAIR || SPLIT) {
    __syncthreads();   // (the other wave of the pair wrote half of this head's V^T)
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  f32x16_t o[DT_TILES][NIT];
#pragma unroll
  for (int dt = 0; dt < DT_TILES; ++dt)
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][it][r] = 0.f;

#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const int jt = kb >> 1, kh = kb & 1;
    hvec pf[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it)
#pragma unroll
      for (int e = 0; e < 8; ++e) pf[it][e] = (typename H16::elem)s[jt][it][8 * kh + e];
#pragma unroll
    for (int dt = 0; dt < DT_TILES; ++dt) {
      const uint16_t* vrow = vt + (32 * dt + lr) * VT_STRIDE + 16 * kb + 4 * g;
      const uint2 lo = *reinterpret_cast<const uint2*>(vrow);
      const uint2 hi = *reinterpret_cast<const uint2*>(vrow + 8);
      const uint4 packed = make_uint4(lo.x, lo.y, hi.x, hi.y);
      const hvec vf = __builtin_bit_cast(hvec, packed);
#pragma unroll
      for (int it = 0; it < NIT; ++it) o[dt][it] = H16::mfma(vf, pf[it], o[dt][it]);
    }
  }

  // ---- normalise and store ----------------------------------------------------------------
  float am = 0.f;
#pragma unroll
  for (int it = 0; it < NIT; ++it) {
    const long row = LAST ? (long)b : (long)b * 64 + 32 * (it0 + it) + lr;
    const bool keep_row = !LAST || lr == 31;
#pragma unroll
    for (int dt = 0; dt < DT_TILES; ++dt)
#pragma unroll
      for (int rp = 0; rp < 2; ++rp) {
        // A lane holds dims 8rq + 4g .. +3 of its row for rq = 0..3; the lane 32 away holds the other four of each
        // group of eight. The two swap one half per pair of groups, so each stores 8 consecutive dims of the row
        // (8 bytes of e4m3 or 16 bytes of 16-bit elements) and a row receives 16 or 32 contiguous bytes per instruction.
        uint32_t pk[2][2];   // [rq - 2rp][word]: e4m3 uses word 0 only
#pragma unroll
        for (int q2 = 0; q2 < 2; ++q2) {
          const int rq = 2 * rp + q2;
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = o[dt][it][4 * rq + e] * inv_l[it];
            am = fmaxf(am, fabsf(v[e]));
          }
          if constexpr (OUT_FP8) {
            pk[q2][0] = pack_fp8x4(v[0] * a.out_scale, v[1] * a.out_scale, v[2] * a.out_scale, v[3] * a.out_scale);
            pk[q2][1] = 0;
          } else {
            pk[q2][0] = H16::pack2(v[0], v[1]);
            pk[q2][1] = H16::pack2(v[2], v[3]);
          }
        }
        // g = 0 keeps group 2rp and receives the partner's half of it; g = 1 keeps group 2rp+1.
        lanes_swap32(pk[0][0], pk[1][0]);
        const int d = 32 * dt + 16 * rp + 8 * g;
        const long off = row * a.ldo + h * HS + d;
        if constexpr (OUT_FP8) {
          const uint2 w = make_uint2(pk[0][0], pk[1][0]);
          if constexpr (coop) *reinterpret_cast<uint2*>(s_out + (32 * it + lr) * OSTRIDE + (wave * HS + d) * OSZ) = w;
          else if (keep_row) *reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(a.out) + off) = w;
        } else {
          lanes_swap32(pk[0][1], pk[1][1]);
          const uint4 w = make_uint4(pk[0][0], pk[0][1], pk[1][0], pk[1][1]);
          if constexpr (coop) *reinterpret_cast<uint4*>(s_out + (32 * it + lr) * OSTRIDE + (wave * HS + d) * OSZ) = w;
          else if (keep_row) *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(a.out) + off) = w;
        }
      }
  }
  if constexpr (COOP) {
    {
      __syncthreads();
      // 16-byte chunks of the tile, row by row: a wave-instruction stores 8 (e4m3) or 4 (16-bit) whole row segments.
      constexpr int CPR = OROW / 16;   // chunks per row
      char* const ob = reinterpret_cast<char*>(a.out) + ((long)b * 64 * a.ldo + (h - wave) * HS) * OSZ;
      const long ldo_b = a.ldo * OSZ;
#pragma unroll
      for (int i = 0; i < 64 * CPR / (64 * NW); ++i) {
        const int id = i * (64 * NW) + threadIdx.x;
        const int row = id / CPR, c = id % CPR;
        const uint4 w = *reinterpret_cast<const uint4*>(s_out + row * OSTRIDE + c * 16);
        *reinterpret_cast<uint4*>(ob + row * ldo_b + c * 16) = w;
      }
    }
  }
  if (a.amax) {
    am = wave_max(am);
    if (lane == 0) atomic_amax(a.amax, am);
  }
}

// Relative-position attention of 64 tokens (new_paradigm/attn.py:507-533): two waves per unit, one per query tile; a workgroup keeps one head and walks positions.
// content = (q+u)·k, position = (q+v)·p, both with the bias folded into the query, the second shifted (pad and reshape) through LDS.
// With a workgroup per unit and operands read as the MFMAs hold them (a lane per row: 64 lanes of a load on 32 rows, which holds it for 190 cycles, and stores of 32 bytes a row)
// a unit took 11300 cycles, 2300 of them to issue the loads, 1900 the stores. Here queries and keys go straight to LDS and results leave through it, whole rows at a time, the
// keys once for both waves; the next position's are requested behind the shift, its values once V is transposed, and the positional table's fragments
// stay in registers. 496 positions of 8 heads of 64 40.1 -> 34.4 us (bytes: 26), 1521 122.9 -> 89.7 (81). Registers alone, without LDS: 40.8 and 113.4.
// Requests past the last position go through empty descriptors and move nothing. 50 KB of LDS: three workgroups a CU.
// FAR: rows further apart than the 31-bit offsets inside a position reach (2^24 elements), or in descending order: 64-bit addresses; past the last position the last one is read again.
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_any_t __attribute__((ext_vector_type(4), aligned(1)));   // output rows start wherever the caller's pointer and stride (a multiple of four elements) put them
__device__ __forceinline__ void attn_load_lds(__amdgpu_buffer_rsrc_t r, uint8_t* dst, int off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, off, 0, 0, 0);
}
template <int HS, int OUT_FP8, int IN_DT, bool FAR>
__global__ void __launch_bounds__(128, 2) relshift_kernel(const AttnArgs a, const int slices) {
  typedef Half16<IN_DT> H16;
  typedef typename H16::vec hvec;
  constexpr int KS = HS / 16, DT_TILES = HS / 32;
  constexpr int ROWB = HS * 2, CPR = ROWB / 16, QK_LOADS = 2 * 64 * ROWB / 1024 / 2;   // bytes and 16-byte chunks of a row, requests of a wave for q and k
  constexpr int ORB = HS * (OUT_FP8 ? 1 : 2), OCH = ORB / 16, NST = 32 * ORB / 1024;    // an output row's bytes and chunks; stores of a wave's tile
  __shared__ __align__(16) uint8_t s_qk[2][64 * ROWB];
  __shared__ __align__(16) uint8_t s_out[2][32 * ORB];
  __shared__ __align__(16) uint16_t s_vt[HS * VT_STRIDE];
  __shared__ float s_sp[64 * SP_STRIDE];
  __shared__ __align__(16) float s_uv[2][2 * HS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lr = lane & 31, g = lane >> 5;
  // (workgroup indices go round the eight XCDs: renumbered so that the heads of a position sit together)
  int bid = blockIdx.x;
  {
    const int per = gridDim.x >> 3;
    if (bid < (per << 3)) bid = (bid & 7) * per + (bid >> 3);
  }
  const int h = bid % a.H, b0 = bid / a.H;
  const int i = 32 * wave + lr;   // this lane's query

  hvec pf[2][KS];
  {
    const uint16_t* pp = reinterpret_cast<const uint16_t*>(a.pos) + h * HS;
    const long ldp = (long)a.H * HS;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) pf[t][ks] = *reinterpret_cast<const hvec*>(pp + (long)(32 * t + lr) * ldp + 16 * ks + 8 * g);
  }
  float* const uv = s_uv[wave];   // u, then v (a wave's own copy)
  if (lane < HS) { uv[lane] = a.u_bias[h * HS + lane]; uv[HS + lane] = a.v_bias[h * HS + lane]; }

  // ---- requests: offsets inside a position's 64 rows, the same for every position
  typedef std::conditional_t<FAR, long, int> Off;
  const Off ldq2 = (Off)a.ldq * 2, ldk2 = (Off)a.ldk * 2, ldv2 = (Off)a.ldv * 2;
  auto unit = [&](const void* base, int b, Off ld2) { return reinterpret_cast<const char*>(base) + (long)b * 64 * ld2 + h * (HS * 2); };
  auto rows = [&](const void* base, int b, Off ld2) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(unit(base, b, ld2)), 0, b < a.B ? 63 * (int)ld2 + HS * 2 : 0, 0x00020000);
  };
  // Queries and keys straight into LDS, whole rows at a time (64 lanes of 32 rows, as the MFMAs want them, hold a load for 190 cycles and a store for more: 2300 and 1900 of a
  // unit's 11300): wave 0 the queries, wave 1 the keys, 16-byte chunks swizzled by row on the global side.
  auto swz = [](int row) { return CPR == 8 ? (row ^ (row >> 3)) & 7 : (row >> 1) & 3; };
  const Off ldw2 = wave ? ldk2 : ldq2;
  Off wo[QK_LOADS];
#pragma unroll
  for (int j = 0; j < QK_LOADS; ++j) {
    const int row = j * (64 / CPR) + lane / CPR;
    wo[j] = row * ldw2 + (((lane % CPR) ^ swz(row)) << 4);
  }
  auto qk_load = [&](int b) {
    if constexpr (FAR) {
      const char* const p = unit(wave ? a.k : a.q, b < a.B ? b : a.B - 1, ldw2);
#pragma unroll
      for (int j = 0; j < QK_LOADS; ++j)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(p + wo[j]), (__attribute__((address_space(3))) void*)(s_qk[wave] + j * 1024), 16, 0, 0);
    } else {
      const __amdgpu_buffer_rsrc_t r = rows(wave ? a.k : a.q, b, ldw2);
#pragma unroll
      for (int j = 0; j < QK_LOADS; ++j) attn_load_lds(r, s_qk[wave] + j * 1024, wo[j]);
    }
  };
  auto frag = [&](const uint8_t* rows_, int row, int ks) -> hvec {
    return *reinterpret_cast<const hvec*>(rows_ + row * ROWB + (((2 * ks + g) ^ swz(row)) << 4));
  };
  // V rows of this wave, half of the unit's: four of one 16-byte chunk a lane (head size 32: half the lanes)
  constexpr int DC = HS / 8, PASSES = (16 * DC) / 64;
  static_assert(PASSES == 1 || PASSES == 2, "head sizes 32 and 64");
  const bool v_mine = PASSES == 2 || !g;
  const int v_id = PASSES == 2 ? wave * 64 + lane : 32 * wave + lr, jq = v_id / DC, dc = v_id - jq * DC;
  const Off vo = 4 * jq * ldv2 + 16 * dc;
  u32x4_t vrow[4];
  auto v_load = [&](int b) {
    if constexpr (FAR) {
      const char* const p = unit(a.v, b < a.B ? b : a.B - 1, ldv2) + vo;
#pragma unroll
      for (int t = 0; t < 4; ++t) vrow[t] = *reinterpret_cast<const u32x4_t*>(p + t * ldv2);
    } else {
      const __amdgpu_buffer_rsrc_t rv = rows(a.v, b, ldv2);
#pragma unroll
      for (int t = 0; t < 4; ++t) vrow[t] = __builtin_amdgcn_raw_buffer_load_b128(rv, vo + t * ldv2, 0, 0);
    }
  };
  auto barrier = [&]() {   // (a bare one: a __syncthreads may wait for what is meant to stay in flight)
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("s_barrier" ::: "memory");
  };

  v_load(b0);
  qk_load(b0);
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  float am = 0.f;
#pragma unroll 1
  for (int b = b0; b < a.B; b += slices) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70 | NST);   // everything but the last position's stores, which follow this one's requests (loads and stores retire in order of issue): its queries or keys are there
    barrier();                                  // and the other wave's part; it is also through with the last position's shift and values
    __builtin_amdgcn_sched_barrier(0);
    f32x16_t s[2], sp[2];
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[jt][r] = sp[jt][r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      float ub[8], vb[8];
      const hvec qf = frag(s_qk[0], i, ks);
#pragma unroll
      for (int e = 0; e < 8; ++e) { ub[e] = uv[16 * ks + 8 * g + e]; vb[e] = uv[HS + 16 * ks + 8 * g + e]; }
      const hvec qu = add_bias_h<H16>(qf, ub);
      const hvec qv = add_bias_h<H16>(qf, vb);
#pragma unroll
      for (int jt = 0; jt < 2; ++jt) {
        s[jt] = H16::mfma(frag(s_qk[1], 32 * jt + lr, ks), qu, s[jt]);
        sp[jt] = H16::mfma(pf[jt][ks], qv, sp[jt]);
      }
    }
    if (v_mine) {
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        // d = 8dc + 2e2 (low halves) and d+1 (high halves)
        const uint32_t w0 = vrow[0][e2], w1 = vrow[1][e2], w2 = vrow[2][e2], w3 = vrow[3][e2];
        *reinterpret_cast<uint2*>(s_vt + (8 * dc + 2 * e2) * VT_STRIDE + 4 * jq) = make_uint2((w0 & 0xffffu) | (w1 << 16), (w2 & 0xffffu) | (w3 << 16));
        *reinterpret_cast<uint2*>(s_vt + (8 * dc + 2 * e2 + 1) * VT_STRIDE + 4 * jq) = make_uint2((w0 >> 16) | (w1 & 0xffff0000u), (w2 >> 16) | (w3 & 0xffff0000u));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    v_load(b + slices);
    __builtin_amdgcn_sched_barrier(0);
    // Shifted read-back (new_paradigm/attn.py:525-533): with T=64,
    //   out[i][j] = P[i][63-i+j] (j<=i), 0 (j==i+1), P[i+1][j-i-2] (j>i+1).
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int r = 0; r < 16; ++r) s_sp[i * SP_STRIDE + 32 * jt + 8 * (r >> 2) + 4 * g + (r & 3)] = sp[jt][r];
    barrier();   // (row 32 of the shift is the other wave's, as is half of V^T; both have read their queries and keys)
    __builtin_amdgcn_sched_barrier(0);
    qk_load(b + slices);
    __builtin_amdgcn_sched_barrier(0);
    // (both cases at one address but for a constant; the element between them is zero; all reads ahead of their use)
    const float* const back = s_sp + i * (SP_STRIDE - 1) + 63 + 4 * g;
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int j0 = 32 * jt + 8 * (r >> 2) + (r & 3);
        sp[jt][r] = back[j0 + (j0 + 4 * g > i ? SP_STRIDE - 65 : 0)];
      }
    __builtin_amdgcn_sched_barrier(0);
    float mx = -INFINITY;
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pv = 32 * jt + 8 * (r >> 2) + 4 * g + (r & 3) == i + 1 ? 0.f : sp[jt][r];
        s[jt][r] = (s[jt][r] + pv) * a.scale;
        mx = fmaxf(mx, s[jt][r]);
      }
    // softmax over keys (registers + lane^32)
    mx = max_xor32(mx);
    float sum = 0.f;
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float p = __expf(s[jt][r] - mx);
        s[jt][r] = p;
        sum += p;
      }
    sum = add_xor32(sum);
    const float inv_l = 1.0f / sum;

    // O^T = V^T · P^T
    f32x16_t o[DT_TILES];
#pragma unroll
    for (int dt = 0; dt < DT_TILES; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      hvec p8;
#pragma unroll
      for (int e = 0; e < 8; ++e) p8[e] = (typename H16::elem)s[kb >> 1][8 * (kb & 1) + e];
#pragma unroll
      for (int dt = 0; dt < DT_TILES; ++dt) {
        const uint16_t* vrow_t = s_vt + (32 * dt + lr) * VT_STRIDE + 16 * kb + 4 * g;
        const uint2 lo = *reinterpret_cast<const uint2*>(vrow_t);
        const uint2 hi = *reinterpret_cast<const uint2*>(vrow_t + 8);
        const uint4 packed = make_uint4(lo.x, lo.y, hi.x, hi.y);
        o[dt] = H16::mfma(__builtin_bit_cast(hvec, packed), p8, o[dt]);
      }
    }
    // normalise and store, as in attention_kernel
#pragma unroll
    for (int dt = 0; dt < DT_TILES; ++dt)
#pragma unroll
      for (int rp = 0; rp < 2; ++rp) {
        uint32_t pk[2][2];
#pragma unroll
        for (int q2 = 0; q2 < 2; ++q2) {
          const int rq = 2 * rp + q2;
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = o[dt][4 * rq + e] * inv_l;
            am = fmaxf(am, fabsf(v[e]));
          }
          if constexpr (OUT_FP8) {
            pk[q2][0] = pack_fp8x4(v[0] * a.out_scale, v[1] * a.out_scale, v[2] * a.out_scale, v[3] * a.out_scale);
            pk[q2][1] = 0;
          } else {
            pk[q2][0] = H16::pack2(v[0], v[1]);
            pk[q2][1] = H16::pack2(v[2], v[3]);
          }
        }
        lanes_swap32(pk[0][0], pk[1][0]);
        // through the wave's own patch, so that a store writes whole rows; chunks swizzled by row
        const int piece = 4 * dt + 2 * rp + g, chunk = OUT_FP8 ? piece >> 1 : piece;
        uint8_t* const d = s_out[wave] + lr * ORB + ((chunk ^ (lr & (OCH - 1))) << 4);
        if constexpr (OUT_FP8) {
          *reinterpret_cast<uint2*>(d + 8 * (piece & 1)) = make_uint2(pk[0][0], pk[1][0]);
        } else {
          lanes_swap32(pk[0][1], pk[1][1]);
          *reinterpret_cast<uint4*>(d) = make_uint4(pk[0][0], pk[0][1], pk[1][0], pk[1][1]);
        }
      }
    wave_fence();
    {
      uint8_t* const ob = reinterpret_cast<uint8_t*>(a.out) + ((long)b * 64 + 32 * wave) * a.ldo * (OUT_FP8 ? 1 : 2) + h * ORB;
#pragma unroll
      for (int j = 0; j < NST; ++j) {
        const int row = j * (64 / OCH) + lane / OCH, c = lane % OCH;
        *reinterpret_cast<u32x4_any_t*>(ob + row * (a.ldo * (OUT_FP8 ? 1 : 2)) + c * 16) = *reinterpret_cast<const u32x4_t*>(s_out[wave] + row * ORB + ((c ^ (row & (OCH - 1))) << 4));
      }
    }
  }
  if (a.amax) {
    am = wave_max(am);
    if (lane == 0) atomic_amax(a.amax, am);
  }
}

template <int HS, int IN_DT, bool FAR>
static hipError_t launch_relshift_dt(const AttnArgs& a, hipStream_t st) {
  // Three workgroups fit a CU: the positions of a head in as many slices as that gives, evened out.
  const int cus = device_cus() > 0 ? device_cus() : 256, most = std::max(3 * cus / a.H, 1), each = (a.B + most - 1) / most, slices = (a.B + each - 1) / each;
  const dim3 grid(slices * a.H), block(128);
  if (a.out_dtype == DT_FP8) hipLaunchKernelGGL((relshift_kernel<HS, 1, IN_DT, FAR>), grid, block, 0, st, a, slices);
  else if (a.out_dtype == IN_DT) hipLaunchKernelGGL((relshift_kernel<HS, 0, IN_DT, FAR>), grid, block, 0, st, a, slices);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}
template <int HS>
static hipError_t launch_relshift(const AttnArgs& a, hipStream_t st) {
  if (a.qk_hstride) return hipErrorInvalidValue;
  auto near = [](long ld) { return ld >= 0 && ld < 1L << 24; };
  const bool far = !near(a.ldq) || !near(a.ldk) || !near(a.ldv);
  if (a.in_dtype == DT_F16) return far ? launch_relshift_dt<HS, DT_F16, true>(a, st) : launch_relshift_dt<HS, DT_F16, false>(a, st);
  if (a.in_dtype == DT_BF16) return far ? launch_relshift_dt<HS, DT_BF16, true>(a, st) : launch_relshift_dt<HS, DT_BF16, false>(a, st);
  return hipErrorInvalidValue;
}

// Causal attention over T > 64 tokens per position (the board tokens followed by move tokens,
// model_bis.py:171-199 with F.scaled_dot_product_attention(is_causal=True) at :71). One wave per
// (position, head, block of 64 queries) walks the key blocks 0..own block with the running
// maximum and sum of a streaming softmax. In the transposed layout a lane owns one query in the
// score tile and in the output tile alike, so the rescale of the running output is one
// multiply per register with the lane's own factor.
template <int HS, int OUT_FP8, int IN_DT>
__global__ void __launch_bounds__(256) causal_long_kernel(const AttnArgs a) {
  typedef Half16<IN_DT> H16;
  typedef typename H16::vec hvec;
  constexpr int KS = HS / 16;
  constexpr int DT_TILES = HS / 32;
  __shared__ __align__(16) uint16_t s_vt[4][HS * VT_STRIDE];

  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lr = lane & 31, g = lane >> 5;
  const int T = a.T, nqb = (T + 63) >> 6;
  const int unit = blockIdx.x * 4 + wave;
  if (unit >= a.B * a.H * (a.last_row ? 1 : nqb)) return;
  // Longest units (last query block) first: they walk the most key blocks.
  const int qb = nqb - 1 - unit / (a.B * a.H);
  const int bh = unit % (a.B * a.H);
  const int b = bh / a.H, h = bh - b * a.H;
  const long row0 = (long)b * T;

  const uint16_t* qp = reinterpret_cast<const uint16_t*>(a.q) + row0 * a.ldq + h * HS;
  const uint16_t* kp = reinterpret_cast<const uint16_t*>(a.k) + row0 * a.ldk + h * HS;
  const uint16_t* vp = reinterpret_cast<const uint16_t*>(a.v) + row0 * a.ldv + h * HS;
  uint16_t* vt = s_vt[wave];
  auto clampT = [&](int t) { return t < T ? t : T - 1; };   // rows past the end re-read the last token

  hvec qf[2][KS];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[t][ks] = *reinterpret_cast<const hvec*>(qp + (long)clampT(64 * qb + 32 * t + lr) * a.ldq + 16 * ks + 8 * g);

  float run_m[2] = {-INFINITY, -INFINITY}, run_l[2] = {0.f, 0.f};
  f32x16_t o[DT_TILES][2];
#pragma unroll
  for (int dt = 0; dt < DT_TILES; ++dt)
#pragma unroll
    for (int it = 0; it < 2; ++it)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][it][r] = 0.f;

  // V rows and keys of a block are requested into the registers the block before has just left: V once it is transposed into
  // LDS, the keys once they are multiplied, each a softmax and an output product ahead of its use. A wave's chain of load,
  // product, softmax and product bounds the kernel (two or three waves share a SIMD), so the loads leave it: scoring 128
  // sequences of 256 tokens with two 6x768 models, 12 of these launches, went from 8.95 to 8.76 ms.
  constexpr int DC = HS / 8;                 // 16-byte chunks per V row
  constexpr int PASSES = (16 * DC) / 64;
  uint4 vrow4[PASSES][4];
  hvec kf[2][KS];
  auto request_v = [&](int kb) {
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int id = p * 64 + lane, jq = id / DC, dc = id - jq * DC;
#pragma unroll
      for (int t = 0; t < 4; ++t) vrow4[p][t] = *reinterpret_cast<const uint4*>(vp + (long)clampT(64 * kb + 4 * jq + t) * a.ldv + 8 * dc);
    }
  };
  auto request_k = [&](int kb) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        kf[t][ks] = *reinterpret_cast<const hvec*>(kp + (long)clampT(64 * kb + 32 * t + lr) * a.ldk + 16 * ks + 8 * g);
  };
  request_v(0);
  request_k(0);

  // (the diagonal block alone needs the causal test; keys past T sit in it too)
  auto key_block = [&](int kb, auto edge_c) {
    constexpr bool edge = decltype(edge_c)::value;
    // ---- V block -> V^T in LDS (the previous block's reads are complete: same wave, in order)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int id = p * 64 + lane, jq = id / DC, dc = id - jq * DC;
      const uint32_t* w0 = reinterpret_cast<const uint32_t*>(&vrow4[p][0]);
      const uint32_t* w1 = reinterpret_cast<const uint32_t*>(&vrow4[p][1]);
      const uint32_t* w2 = reinterpret_cast<const uint32_t*>(&vrow4[p][2]);
      const uint32_t* w3 = reinterpret_cast<const uint32_t*>(&vrow4[p][3]);
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        uint2 lo = make_uint2((w0[e2] & 0xffffu) | (w1[e2] << 16), (w2[e2] & 0xffffu) | (w3[e2] << 16));
        uint2 hi = make_uint2((w0[e2] >> 16) | (w1[e2] & 0xffff0000u), (w2[e2] >> 16) | (w3[e2] & 0xffff0000u));
        *reinterpret_cast<uint2*>(vt + (8 * dc + 2 * e2) * VT_STRIDE + 4 * jq) = lo;
        *reinterpret_cast<uint2*>(vt + (8 * dc + 2 * e2 + 1) * VT_STRIDE + 4 * jq) = hi;
      }
    }
    if constexpr (!edge) request_v(kb + 1);
    // ---- scores of this key block
    f32x16_t s[2][2];
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int it = 0; it < 2; ++it) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[jt][it][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s[jt][it] = H16::mfma(kf[jt][ks], qf[it][ks], s[jt][it]);
      }
    if constexpr (!edge) request_k(kb + 1);
    __builtin_amdgcn_sched_barrier(0);   // (the requests stay above the softmax)
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int i = 64 * qb + 32 * it + lr;
      float mx = run_m[it];
#pragma unroll
      for (int jt = 0; jt < 2; ++jt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = 64 * kb + 32 * jt + 8 * (r >> 2) + 4 * g + (r & 3);
          float x = s[jt][it][r] * a.scale;
          if constexpr (edge) {
            if (j > i || j >= T) x = -INFINITY;
            s[jt][it][r] = x;
          }
          mx = fmaxf(mx, x);
        }
      mx = max_xor32(mx);
      // Key 0 is visible to every query, so mx is finite from the first block on.
      const float alpha = __expf(run_m[it] - mx);
      float sum = 0.f;
#pragma unroll
      for (int jt = 0; jt < 2; ++jt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = __expf(edge ? s[jt][it][r] - mx : fmaf(s[jt][it][r], a.scale, -mx));
          s[jt][it][r] = p;
          sum += p;
        }
      sum = add_xor32(sum);
      run_l[it] = run_l[it] * alpha + sum;
      run_m[it] = mx;
#pragma unroll
      for (int dt = 0; dt < DT_TILES; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][it][r] *= alpha;
    }
    // ---- O^T += V^T · P^T
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int k4 = 0; k4 < 4; ++k4) {
      const int jt = k4 >> 1, kh = k4 & 1;
      hvec pf[2];
#pragma unroll
      for (int it = 0; it < 2; ++it)
#pragma unroll
        for (int e = 0; e < 8; ++e) pf[it][e] = (typename H16::elem)s[jt][it][8 * kh + e];
#pragma unroll
      for (int dt = 0; dt < DT_TILES; ++dt) {
        const uint16_t* vrow = vt + (32 * dt + lr) * VT_STRIDE + 16 * k4 + 4 * g;
        const uint2 lo = *reinterpret_cast<const uint2*>(vrow);
        const uint2 hi = *reinterpret_cast<const uint2*>(vrow + 8);
        const uint4 packed = make_uint4(lo.x, lo.y, hi.x, hi.y);
        const hvec vf = __builtin_bit_cast(hvec, packed);
#pragma unroll
        for (int it = 0; it < 2; ++it) o[dt][it] = H16::mfma(vf, pf[it], o[dt][it]);
      }
    }
  };
#pragma unroll 1
  for (int kb = 0; kb < qb; ++kb) key_block(kb, std::false_type{});
  key_block(qb, std::true_type{});

  float am = 0.f;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int i = 64 * qb + 32 * it + lr;
    if (i >= T || (a.last_row && i != T - 1)) continue;
    const float inv_l = 1.0f / run_l[it];
    const long row = a.last_row ? (long)b : row0 + i;
#pragma unroll
    for (int dt = 0; dt < DT_TILES; ++dt)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const int d = 32 * dt + 8 * rq + 4 * g;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = o[dt][it][4 * rq + e] * inv_l;
          am = fmaxf(am, fabsf(v[e]));
        }
        const long off = row * a.ldo + h * HS + d;
        if constexpr (OUT_FP8) {
          *reinterpret_cast<uint32_t*>(reinterpret_cast<uint8_t*>(a.out) + off) =
              pack_fp8x4(v[0] * a.out_scale, v[1] * a.out_scale, v[2] * a.out_scale, v[3] * a.out_scale);
        } else {
          *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.out) + off) = make_uint2(H16::pack2(v[0], v[1]), H16::pack2(v[2], v[3]));
        }
      }
  }
  if (a.amax) {
    am = wave_max(am);
    if (lane == 0) atomic_amax(a.amax, am);
  }
}

// The same for up to 256 tokens, all rows wanted: one workgroup of four waves per (position, head). V is transposed into LDS once for all of them, a block of
// 64 keys per wave; then every wave takes two tiles of 32 queries, the wave-th from the end and, of what is left, the one that makes the waves' key
// blocks equal (256 tokens: 5 each). A wave's state is half of the other form's, which at 402 registers left a SIMD with one wave that waited for its own
// chain: 128 sequences of 256 tokens, 12 heads of 64, 80.6 us a launch there, 68 here (71 at the compiler's own 248 registers, 101 held to 128; leaving out the half
// of a diagonal block that an even tile cannot see changes nothing); of 65 tokens 27 and 21. Vector instructions are 36 % of it, the rest is waits between
// dependent ones; bytes 40 us at the rate of a large copy.
constexpr int CG_BLOCKS = 4;
template <int HS, int OUT_FP8, int IN_DT>
__global__ void __launch_bounds__(256, 3) causal_group_kernel(const AttnArgs a) {
  typedef Half16<IN_DT> H16;
  typedef typename H16::vec hvec;
  constexpr int KS = HS / 16, DT_TILES = HS / 32;
  __shared__ __align__(16) uint16_t s_vt[CG_BLOCKS][HS * VT_STRIDE];

  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lr = lane & 31, g = lane >> 5;
  const int T = a.T, nblk = (T + 63) >> 6, ntile = (T + 31) >> 5;
  int unit = blockIdx.x;   // (as in attention_kernel: each XCD walks a contiguous range)
  {
    const int per = gridDim.x >> 3;
    if (unit < (per << 3)) unit = (unit & 7) * per + (unit >> 3);
  }
  const int b = unit / a.H, h = unit - b * a.H;
  const long row0 = (long)b * T;
  const uint16_t* qp = reinterpret_cast<const uint16_t*>(a.q) + row0 * a.ldq + h * HS;
  const uint16_t* kp = reinterpret_cast<const uint16_t*>(a.k) + row0 * a.ldk + h * HS;
  const uint16_t* vp = reinterpret_cast<const uint16_t*>(a.v) + row0 * a.ldv + h * HS;
  auto clampT = [&](int t) { return t < T ? t : T - 1; };   // rows past the end re-read the last token

  hvec qf[KS], kf[2][KS];
  auto request_q = [&](int tile) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const hvec*>(qp + (long)clampT(32 * tile + lr) * a.ldq + 16 * ks + 8 * g);
  };
  auto request_k = [&](int kb) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[t][ks] = *reinterpret_cast<const hvec*>(kp + (long)clampT(64 * kb + 32 * t + lr) * a.ldk + 16 * ks + 8 * g);
  };
  int tile = ntile - 1 - wave;
  constexpr int DC = HS / 8, PASSES = (16 * DC) / 64;
  i32x4_t vrow4[PASSES][4];
  if (wave < nblk) {
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int id = p * 64 + lane, jq = id / DC, dc = id - jq * DC;
#pragma unroll
      for (int t = 0; t < 4; ++t) vrow4[p][t] = *reinterpret_cast<const i32x4_t*>(vp + (long)clampT(64 * wave + 4 * jq + t) * a.ldv + 8 * dc);
    }
  }
  if (tile >= 0) { request_q(tile); request_k(0); }
  __builtin_amdgcn_sched_barrier(0);
  if (wave < nblk) {
    uint16_t* vt = s_vt[wave];
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int id = p * 64 + lane, jq = id / DC, dc = id - jq * DC;
#pragma unroll
      for (int e2 = 0; e2 < 4; ++e2) {
        const uint32_t w0 = (uint32_t)vrow4[p][0][e2], w1 = (uint32_t)vrow4[p][1][e2], w2 = (uint32_t)vrow4[p][2][e2], w3 = (uint32_t)vrow4[p][3][e2];
        *reinterpret_cast<uint2*>(vt + (8 * dc + 2 * e2) * VT_STRIDE + 4 * jq) = make_uint2((w0 & 0xffffu) | (w1 << 16), (w2 & 0xffffu) | (w3 << 16));
        *reinterpret_cast<uint2*>(vt + (8 * dc + 2 * e2 + 1) * VT_STRIDE + 4 * jq) = make_uint2((w0 >> 16) | (w1 & 0xffff0000u), (w2 >> 16) | (w3 & 0xffff0000u));
      }
    }
  }
  __syncthreads();

  float am = 0.f;
#pragma unroll 1
  for (int part = 0; part < 2; ++part) {
    if (part == 1) {
      tile = wave + ntile - 8;
      if (tile >= 0) { request_q(tile); request_k(0); }
    }
    if (tile < 0) continue;
    const int qb = tile >> 1, i = 32 * tile + lr;
    float run_m = -INFINITY, run_l = 0.f;
    f32x16_t o[DT_TILES];
#pragma unroll
    for (int dt = 0; dt < DT_TILES; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
    // (the diagonal block alone needs the causal test; keys past T sit in it too)
    auto key_block = [&](int kb, auto edge_c) {
      constexpr bool edge = decltype(edge_c)::value;
      f32x16_t s[2];
#pragma unroll
      for (int jt = 0; jt < 2; ++jt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[jt][r] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s[jt] = H16::mfma(kf[jt][ks], qf[ks], s[jt]);
      }
      if constexpr (!edge) request_k(kb + 1);
      __builtin_amdgcn_sched_barrier(0);   // (the requests stay above the softmax)
      float mx = run_m;
#pragma unroll
      for (int jt = 0; jt < 2; ++jt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float x = s[jt][r] * a.scale;
          if constexpr (edge) {
            const int j = 64 * kb + 32 * jt + 8 * (r >> 2) + 4 * g + (r & 3);
            if (j > i || j >= T) x = -INFINITY;
            s[jt][r] = x;
          }
          mx = fmaxf(mx, x);
        }
      mx = max_xor32(mx);
      // Key 0 is visible to every query, so mx is finite from the first block on.
      const float alpha = __expf(run_m - mx);
      float sum = 0.f;
#pragma unroll
      for (int jt = 0; jt < 2; ++jt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = __expf(edge ? s[jt][r] - mx : fmaf(s[jt][r], a.scale, -mx));
          s[jt][r] = p;
          sum += p;
        }
      sum = add_xor32(sum);
      run_l = run_l * alpha + sum;
      run_m = mx;
#pragma unroll
      for (int dt = 0; dt < DT_TILES; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
      // ---- O^T += V^T · P^T
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4) {
        const int jt = k4 >> 1, kh = k4 & 1;
        hvec pf;
#pragma unroll
        for (int e = 0; e < 8; ++e) pf[e] = (typename H16::elem)s[jt][8 * kh + e];
#pragma unroll
        for (int dt = 0; dt < DT_TILES; ++dt) {
          const uint16_t* vrow = s_vt[kb] + (32 * dt + lr) * VT_STRIDE + 16 * k4 + 4 * g;
          const uint2 lo = *reinterpret_cast<const uint2*>(vrow);
          const uint2 hi = *reinterpret_cast<const uint2*>(vrow + 8);
          const uint4 packed = make_uint4(lo.x, lo.y, hi.x, hi.y);
          o[dt] = H16::mfma(__builtin_bit_cast(hvec, packed), pf, o[dt]);
        }
      }
    };
#pragma unroll 1
    for (int kb = 0; kb < qb; ++kb) key_block(kb, std::false_type{});
    key_block(qb, std::true_type{});

    // Two lanes of a row exchange halves, as in attention_kernel: each stores eight consecutive dims. (Rows past the end take part and store nothing.)
    const float inv_l = 1.0f / run_l;
    const bool keep_row = i < T;
#pragma unroll
    for (int dt = 0; dt < DT_TILES; ++dt)
#pragma unroll
      for (int rp = 0; rp < 2; ++rp) {
        uint32_t pk[2][2];
#pragma unroll
        for (int q2 = 0; q2 < 2; ++q2) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = o[dt][4 * (2 * rp + q2) + e] * inv_l;
            if (keep_row) am = fmaxf(am, fabsf(v[e]));
          }
          if constexpr (OUT_FP8) {
            pk[q2][0] = pack_fp8x4(v[0] * a.out_scale, v[1] * a.out_scale, v[2] * a.out_scale, v[3] * a.out_scale);
            pk[q2][1] = 0;
          } else {
            pk[q2][0] = H16::pack2(v[0], v[1]);
            pk[q2][1] = H16::pack2(v[2], v[3]);
          }
        }
        lanes_swap32(pk[0][0], pk[1][0]);
        const long off = (row0 + i) * a.ldo + h * HS + 32 * dt + 16 * rp + 8 * g;
        if constexpr (OUT_FP8) {
          if (keep_row) *reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(a.out) + off) = make_uint2(pk[0][0], pk[1][0]);
        } else {
          lanes_swap32(pk[0][1], pk[1][1]);
          if (keep_row) *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(a.out) + off) = make_uint4(pk[0][0], pk[0][1], pk[1][0], pk[1][1]);
        }
      }
  }
  if (a.amax) {
    am = wave_max(am);
    if (lane == 0) atomic_amax(a.amax, am);
  }
}

template <int HS, int IN_DT>
static hipError_t launch_causal_long_dt(const AttnArgs& a, hipStream_t st) {
  // (16-byte stores of the one with the shared V need rows and base aligned to that)
  const int osz = a.out_dtype == DT_FP8 ? 1 : 2;
  if (a.T > 64 && a.T <= 64 * CG_BLOCKS && !a.last_row && (a.ldo * osz) % 16 == 0 && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0) {
    const dim3 grid((unsigned)(a.B * a.H)), block(256);
    if (a.out_dtype == DT_FP8) hipLaunchKernelGGL((causal_group_kernel<HS, 1, IN_DT>), grid, block, 0, st, a);
    else if (a.out_dtype == IN_DT) hipLaunchKernelGGL((causal_group_kernel<HS, 0, IN_DT>), grid, block, 0, st, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
  }
  const long units = (long)a.B * a.H * (a.last_row ? 1 : (a.T + 63) / 64);   // (the last token sits in the block that is walked first)
  const dim3 grid((unsigned)((units + 3) / 4)), block(256);
  if (a.out_dtype == DT_FP8) hipLaunchKernelGGL((causal_long_kernel<HS, 1, IN_DT>), grid, block, 0, st, a);
  else if (a.out_dtype == IN_DT) hipLaunchKernelGGL((causal_long_kernel<HS, 0, IN_DT>), grid, block, 0, st, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}
template <int HS>
static hipError_t launch_causal_long(const AttnArgs& a, hipStream_t st) {
  if (a.in_dtype == DT_F16) return launch_causal_long_dt<HS, DT_F16>(a, st);
  if (a.in_dtype == DT_BF16) return launch_causal_long_dt<HS, DT_BF16>(a, st);
  return hipErrorInvalidValue;
}

template <int HS, int MODE, int IN_DT>
static hipError_t launch_attn_dt(const AttnArgs& a, hipStream_t st) {
  constexpr int NW = AttnWaves<MODE>::N;
  const dim3 grid((a.B * a.H + NW - 1) / NW), block(64 * NW);
  // Few units: two waves for each, one per query tile (bit-equal; the shift of the relative mode crosses the tiles). The wave's chain of loads, scores,
  // softmax and output bounds a call that does not fill the chip, and this halves all of it but the loads: 15 layers of 32 heads of 32, one
  // position 6.8 -> 4.2 us a launch, 8 positions 7.2 -> 4.5, 33 9.0 -> 7.9, 64 the same, 250 +10 %; 6 layers of 12 heads of 64, one position 6.9 -> 4.8 us,
  // 16 7.2 -> 5.0, 32 -0.6 us, 64 +0.4, 256 +9. Beyond the lines the second reading of the keys costs more than the shorter chain gives.
  if (!a.last_row && 2L * a.B * a.H <= (HS == 32 ? 9L : 4L) * device_cus()) {
    const dim3 units(a.B * a.H), two(128);
    if (a.out_dtype == DT_FP8) hipLaunchKernelGGL((attention_kernel<HS, MODE, 1, IN_DT, 0, 0, 1>), units, two, 0, st, a);
    else if (a.out_dtype == IN_DT) hipLaunchKernelGGL((attention_kernel<HS, MODE, 0, IN_DT, 0, 0, 1>), units, two, 0, st, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
  }
  if constexpr (HS == 32 && (NW == 4 || NW == 8 || NW == 16)) {
    // Whole workgroups only: H a multiple of 4 puts four heads of one position in every workgroup and leaves none partly
    // filled; 16-byte stores need rows and base aligned to that.
    const int osz = a.out_dtype == DT_FP8 ? 1 : 2;
    if (!a.last_row && a.H % NW == 0 && (a.ldo * osz) % 16 == 0 && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0) {
      if (a.out_dtype == DT_FP8) hipLaunchKernelGGL((attention_kernel<HS, MODE, 1, IN_DT, 1>), grid, block, 0, st, a);
      else if (a.out_dtype == IN_DT) hipLaunchKernelGGL((attention_kernel<HS, MODE, 0, IN_DT, 1>), grid, block, 0, st, a);
      else return hipErrorInvalidValue;
      return hipGetLastError();
    }
  }
  if constexpr (MODE == ATTN_CAUSAL) {
    if (a.last_row) {
      if (a.out_dtype == DT_FP8) hipLaunchKernelGGL((attention_kernel<HS, MODE, 1, IN_DT, 0, 1>), grid, block, 0, st, a);
      else if (a.out_dtype == IN_DT) hipLaunchKernelGGL((attention_kernel<HS, MODE, 0, IN_DT, 0, 1>), grid, block, 0, st, a);
      else return hipErrorInvalidValue;
      return hipGetLastError();
    }
  }
  if (a.out_dtype == DT_FP8) hipLaunchKernelGGL((attention_kernel<HS, MODE, 1, IN_DT>), grid, block, 0, st, a);
  else if (a.out_dtype == IN_DT) hipLaunchKernelGGL((attention_kernel<HS, MODE, 0, IN_DT>), grid, block, 0, st, a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

template <int HS, int MODE>
static hipError_t launch_attn_mode(const AttnArgs& a, hipStream_t st) {
  if (a.in_dtype == DT_F16) return launch_attn_dt<HS, MODE, DT_F16>(a, st);
  if (a.in_dtype == DT_BF16) return launch_attn_dt<HS, MODE, DT_BF16>(a, st);
  return hipErrorInvalidValue;
}

template <int HS>
static hipError_t launch_attn_hs(const AttnArgs& a, hipStream_t st) {
  switch (a.mode) {
    case ATTN_PLAIN: return launch_attn_mode<HS, ATTN_PLAIN>(a, st);
    case ATTN_CAUSAL: return launch_attn_mode<HS, ATTN_CAUSAL>(a, st);
    case ATTN_BIAS: return launch_attn_mode<HS, ATTN_BIAS>(a, st);
    case ATTN_RELSHIFT: return launch_relshift<HS>(a, st);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_attention(const AttnArgs& a, int head_dim, hipStream_t st) {
  if (a.B <= 0) return hipSuccess;
  // 16-byte row-segment loads: strides and bases must be multiples of 8 elements.
  if (a.ldq % 8 || a.ldk % 8 || a.ldv % 8 || a.ldo % 4 || a.qk_hstride % 8 || (a.qk_hstride && (a.qk_hstride < head_dim || (a.T != 0 && a.T != 64))) ||
      (reinterpret_cast<uintptr_t>(a.q) & 15) || (reinterpret_cast<uintptr_t>(a.k) & 15) || (reinterpret_cast<uintptr_t>(a.v) & 15))
    return hipErrorInvalidValue;
  if (a.last_row && (a.mode != ATTN_CAUSAL || a.amax)) return hipErrorInvalidValue;
  if (a.mode == ATTN_BIAS && !a.bias) return hipErrorInvalidValue;
  if (a.mode == ATTN_BIAS && a.bias_blocked && ((long)a.B * a.H) % 256 != 0) return hipErrorInvalidValue;
  if (a.mode == ATTN_RELSHIFT && (!a.pos || !a.u_bias || !a.v_bias)) return hipErrorInvalidValue;
  if (a.T != 0 && a.T != 64) {
    if (a.mode != ATTN_CAUSAL || a.T < 1 || a.T > 4096) return hipErrorInvalidValue;
    if (head_dim == 32) return launch_causal_long<32>(a, st);
    if (head_dim == 64) return launch_causal_long<64>(a, st);
    return hipErrorInvalidValue;
  }
  if (head_dim == 32) return launch_attn_hs<32>(a, st);
  if (head_dim == 64) return launch_attn_hs<64>(a, st);
  return hipErrorInvalidValue;
}

int attn_bias_slot_host(int i, int j) { return attn_bias_slot(i, j); }

}  // namespace crl
