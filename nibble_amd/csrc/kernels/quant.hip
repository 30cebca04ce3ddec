// Quantized weight matmuls and dequantization on gfx950: Backend::matmul / matmul_multi / embed for the ggml block
// formats Q4_0, Q5_0, Q5_1, Q8_0, Q4_K, Q5_K, Q6_K (src/quant.h), bit-exact with the reference's scalar kernels
// src/quant.cpp (itself llama.cpp's generic code) and hence with its AVX2 tier.
//
// A matmul never dequantizes the weights (ref_ops.cpp:109-135): each activation row is quantized to the weight
// type's companion format (Q8_0, Q8_1 or Q8_K), and y[t, r] = sum over blocks b of a per-block term, summed in block
// order. The integer part of every term is exact, so it is computed in any order (here with v_dot4 where it
// applies); the float part - the scale products and the running sum over blocks - is the reference's expression,
// in its order, with no multiply-add contraction (this file is compiled with -ffp-contract=off, as the reference's
// quant.cpp is; the __f*_rn spellings only mark the rounding points):
//   Q4_0  sum += (float(isum) * d_w) * d_a          quant.cpp:309-325
//   Q8_0  sum += float(isum) * (d_w * d_a)          :329-342
//   Q5_0  sum += (d_w * d_a) * float(isum)          :346-365
//   Q5_1  sum += (d_w * d_a) * float(isum) + m_w * s_a  :369-390
//   Q4_K / Q5_K (quant.cpp:118-144) and Q6_K (:394-416): eight int32 lanes (element e feeds lane e % 8) per
//   super-block, sums[l] += (d_w * d_a) * float(aux[l]) in super-block order, Q4_K / Q5_K also sumf -= (dmin_w *
//   d_a) * float(sumi) per super-block, and the eight sums added to sumf last.
//
// qgemv_kernel (n <= 16 activation rows): a 64-lane wave takes RW weight rows; its lanes take (row, block) pairs -
// a legacy block or a whole K super-block each - and write each pair's float term(s) to LDS; then one lane per
// (row, activation row) adds its terms in block order. K quants are stored in residue order (quant_layout.h), so a
// sub-block's eight integer lanes are eight v_dot4. With up to 4 activation rows the rows are quantized inside the
// launch (into LDS, once per wave and block), with the same bits as the standalone quantizer. K types at up to 4 rows
// take kgemv_kernel instead (a workgroup quantizes the rows once), longer calls of either kind the tiled kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "backend/hip/kernel_timing.h"
#include "kernels/quant_layout.h"
#include "nibble_hip_shim.h"

namespace {

using namespace nbh_quant;

struct QW {
  const uint8_t* q;
  const uint8_t* h;
  const uint8_t* s;
  const uint16_t* d;
  const uint16_t* m;
  int64_t rows, nb;
};
struct QA {
  const int8_t* qs;
  const float* d;
  const float* s;
  const int16_t* bsums;
  int64_t nb;
};

__device__ __forceinline__ float h2f(uint16_t h) { return float(__builtin_bit_cast(_Float16, h)); }
__device__ __forceinline__ uint16_t f2h(float f) { return __builtin_bit_cast(uint16_t, _Float16(f)); }  // RNE

// v as a float in a register, opaque to the optimizer. fp16(a * b) is otherwise compiled to one v_fma_mix, which
// rounds the exact product to fp16 once; the reference rounds to float first and then to fp16, and the two differ
// when the float product lands on an fp16 tie.
__device__ __forceinline__ float opaque(float v) {
  asm volatile("" : "+v"(v));
  return v;
}

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
// Quant words as native vectors (a uint4 copy is a memcpy that keeps the value in scratch).
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// Orders a wave's LDS operations across its lanes: the writes of every lane before it are seen by the reads of every lane
// after it, and none of them moves across it. The LDS unit completes one wave's operations in order, so wavefront-scope
// fences keep the compiler to that order and cost no wait; the barrier alone orders no memory access.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lane exchanges on the VALU (DPP), a few cycles each where a __shfl goes through LDS: within quads, and mirrored within
// 8 and 16 lanes. In this order they are the steps of a reduction over 16 lanes.
template <int CTRL>
__device__ __forceinline__ int dpp(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, dpp<CTRL>(__builtin_bit_cast(int, v)));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E, kMirror8 = 0x141, kMirror16 = 0x140;
__device__ __forceinline__ int lane_int(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// The first element of largest magnitude of a quantization block sets the sign of its scale: every lane gives its own
// largest magnitude (NaN never counts) and 2 * (its first element of that magnitude) + (that element's sign bit).
// Returns the block's value; KEYS lanes (8 consecutive ones, or the wave's 64) share a block.
template <int KEYS>
__device__ __forceinline__ float block_max(float amax, int key, float& out_amax) {
  float m = amax;
  m = fmaxf(m, dpp<kQuadXor1>(m));
  m = fmaxf(m, dpp<kQuadXor2>(m));
  m = fmaxf(m, dpp<kMirror8>(m));
  if constexpr (KEYS == 64) {
    m = fmaxf(m, dpp<kMirror16>(m));
    const int b = __builtin_bit_cast(int, m);
    m = fmaxf(fmaxf(__builtin_bit_cast(float, lane_int(b, 0)), __builtin_bit_cast(float, lane_int(b, 16))),
              fmaxf(__builtin_bit_cast(float, lane_int(b, 32)), __builtin_bit_cast(float, lane_int(b, 48))));
  }
  int k = amax == m ? key : 0x7FFFFFFF;
  k = min(k, dpp<kQuadXor1>(k));
  k = min(k, dpp<kQuadXor2>(k));
  k = min(k, dpp<kMirror8>(k));
  if constexpr (KEYS == 64) {
    k = min(k, dpp<kMirror16>(k));
    k = min(min(lane_int(k, 0), lane_int(k, 16)), min(lane_int(k, 32), lane_int(k, 48)));
  }
  out_amax = m;
  return k & 1 ? -m : m;
}

__device__ __forceinline__ int sdot4(uint32_t a, uint32_t b, int c) {
  return __builtin_amdgcn_sdot4(int(a), int(b), c, false);
}

// ---- activation quantizers (quant.cpp:37-49, 245-303) ----

// One thread per 32-element block of row t: Q8_0 (and Q8_1's sum term when Q81).
template <bool Q81>
__global__ __launch_bounds__(256) void quantize_q8_kernel(const float* __restrict__ x, int64_t in, int64_t n,
                                                          int8_t* __restrict__ qs, float* __restrict__ dq,
                                                          float* __restrict__ sq) {
  const int64_t nb = in / 32;
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n * nb) return;
  const float* xb = x + (i / nb) * in + (i % nb) * 32;
  float v[32];
  float amax = 0.f;
  bool nan = false;
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    v[j] = xb[j];
    amax = fmaxf(amax, fabsf(v[j]));
    nan |= v[j] != v[j];
  }
  const float d = nan ? __builtin_nanf("") : __fdiv_rn(amax, 127.f);
  const float id = d != 0.f ? __fdiv_rn(1.0f, d) : 0.0f;
  int sum = 0;
  uint32_t packed[8];
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    uint32_t word = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float r = roundf(__fmul_rn(v[4 * w + e], id));
      const int q = r != r ? 0 : int(fminf(127.f, fmaxf(-127.f, r)));
      sum += q;
      word |= uint32_t(q & 0xFF) << (8 * e);
    }
    packed[w] = word;
  }
  uint4* o = reinterpret_cast<uint4*>(qs + i * 32);
  o[0] = make_uint4(packed[0], packed[1], packed[2], packed[3]);
  o[1] = make_uint4(packed[4], packed[5], packed[6], packed[7]);
  dq[i] = h2f(f2h(d));
  if constexpr (Q81) sq[i] = h2f(f2h(opaque(__fmul_rn(float(sum), d))));
}

// ggml nearest_int (quant.cpp:146-152): round half to even through the float mantissa.
__device__ __forceinline__ int nearest_int(float f) {
  const float val = __fadd_rn(f, 12582912.f);
  return (__float_as_int(val) & 0x007fffff) - 0x00400000;
}

// quantize_row_q8_K (quant.cpp:273-303) of one super-block by a wave; lane l = 8k + w holds elements 32k + w + 8i
// (i < 4) of sub-block k, at xb[8 i]: its four quants, its sub-block's two 16-sums and the block's scale.
__device__ __forceinline__ void q8k_lane(const float* xb, int lane, int (&q)[4], int& b0, int& b1, float& d) {
  const int k = lane >> 3, w = lane & 7;
  const float v[4] = {xb[0], xb[8], xb[16], xb[24]};
  float own = 0.f, amax;
  int key = 0;
  bool nan = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float ax = fabsf(v[e]);
    if (ax > own) own = ax, key = 2 * (32 * k + w + 8 * e) + (v[e] < 0.f ? 1 : 0);
    nan |= v[e] != v[e];
  }
  const float mx = block_max<64>(own, key, amax);
  nan = __builtin_amdgcn_ballot_w64(nan) != 0;
  d = 0.f;
  q[0] = q[1] = q[2] = q[3] = 0;
  if (amax != 0.f) {
    const float iscale = __fdiv_rn(-127.f, mx);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float sv = __fmul_rn(iscale, v[e]);
      q[e] = sv != sv ? 0 : nearest_int(fminf(127.f, fmaxf(-127.f, sv)));
    }
    d = __fdiv_rn(1.f, iscale);
  }
  if (nan) d = __builtin_nanf("");
  // the sub-block's two 16-sums (elements w, w + 8 | w + 16, w + 24 of each lane)
  b0 = q[0] + q[1], b1 = q[2] + q[3];
  b0 += dpp<kQuadXor1>(b0), b1 += dpp<kQuadXor1>(b1);
  b0 += dpp<kQuadXor2>(b0), b1 += dpp<kQuadXor2>(b1);
  b0 += dpp<kMirror8>(b0), b1 += dpp<kMirror8>(b1);
}

// One wave per super-block; a lane's four quants are residue word w of its sub-block, which it stores as word w of the
// sub-block (residue order, quant_layout.h).
// RM: the tiled K kernels' operand form instead (quant_layout.h, kActQ8_K16): 16 times each quant as fp16, residue
// by residue, and each sub-block's sum of its quants as two fp16 digits.
template <bool RM>
__global__ __launch_bounds__(64) void quantize_q8k_kernel(const float* __restrict__ x, int64_t in,
                                                          int8_t* __restrict__ qs, float* __restrict__ dq,
                                                          int16_t* __restrict__ bsums) {
  const int64_t nb = in / 256, i = blockIdx.x;
  const int lane = threadIdx.x, k = lane >> 3, w = lane & 7;
  int q[4], b0, b1;
  float d;
  q8k_lane(x + (i / nb) * in + (i % nb) * 256 + 32 * k + w, lane, q, b0, b1, d);
  if constexpr (RM) {
    // chunk k / 2 of residue w: sub-block k's elements (0, 2) at halves 2 (k % 2), (1, 3) at 4 + 2 (k % 2)
    _Float16* o = reinterpret_cast<_Float16*>(qs) + i * 256 + 32 * w + 8 * (k >> 1) + 2 * (k & 1);
    *reinterpret_cast<half2_t*>(o) = half2_t{_Float16(16 * q[0]), _Float16(16 * q[2])};
    *reinterpret_cast<half2_t*>(o + 4) = half2_t{_Float16(16 * q[1]), _Float16(16 * q[3])};
    if (w == 0) {
      _Float16* bs = reinterpret_cast<_Float16*>(bsums) + i * 16;
      const int sum = b0 + b1;
      const int at = (k & 4) | ((k & 1) << 1) | ((k >> 1) & 1);  // 0, 2, 1, 3 of each four
      bs[at] = _Float16(sum & 63);
      bs[8 + at] = _Float16(sum >> 6);
    }
  } else {
    uint32_t word = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) word |= uint32_t(q[e] & 0xFF) << (8 * e);
    reinterpret_cast<uint32_t*>(qs + i * 256)[lane] = word;
    if (w == 0) bsums[i * 16 + 2 * k] = int16_t(b0), bsums[i * 16 + 2 * k + 1] = int16_t(b1);
  }
  if (lane == 0) dq[i] = d;
}

// ---- activation blocks ----

// One legacy activation block: 32 quants as 8 words, the scale d (fp16-rounded, widened), Q8_1's s, and the sum
// of the quants (for the Q4_0 / Q5_0 offsets).
struct ActL {
  uint32_t a[8];
  float d, s;
  int sum;
};

__device__ __forceinline__ ActL load_act_l(const QA& A, int64_t t, int64_t b) {
  ActL r;
  const int64_t ab = t * A.nb + b;
  const uint4* ap = reinterpret_cast<const uint4*>(A.qs + ab * 32);
  const uint4 a0 = ap[0], a1 = ap[1];
  r.a[0] = a0.x, r.a[1] = a0.y, r.a[2] = a0.z, r.a[3] = a0.w, r.a[4] = a1.x, r.a[5] = a1.y, r.a[6] = a1.z,
  r.a[7] = a1.w;
  r.d = A.d[ab];
  r.s = A.s ? A.s[ab] : 0.f;
  r.sum = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) r.sum = sdot4(r.a[i], 0x01010101u, r.sum);
  return r;
}

// quantize_block_q8 (quant.cpp:37-49) of the 32 floats at xb (16-byte aligned), in registers: the same bits
// quantize_q8_kernel writes.
template <bool Q81>
__device__ __forceinline__ ActL quant_act_l(const float* xb) {
  float v[32];
  float amax = 0.f;
  bool nan = false;
#pragma unroll
  for (int j = 0; j < 32; j += 4) {
    const float4 f = *reinterpret_cast<const float4*>(xb + j);
    v[j] = f.x, v[j + 1] = f.y, v[j + 2] = f.z, v[j + 3] = f.w;
  }
#pragma unroll
  for (int j = 0; j < 32; ++j) {
    amax = fmaxf(amax, fabsf(v[j]));
    nan |= v[j] != v[j];
  }
  const float d = nan ? __builtin_nanf("") : __fdiv_rn(amax, 127.f);
  const float id = d != 0.f ? __fdiv_rn(1.0f, d) : 0.0f;
  ActL r;
  r.sum = 0;
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    uint32_t word = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float q = roundf(__fmul_rn(v[4 * w + e], id));
      const int qi = q != q ? 0 : int(fminf(127.f, fmaxf(-127.f, q)));
      r.sum += qi;
      word |= uint32_t(qi & 0xFF) << (8 * e);
    }
    r.a[w] = word;
  }
  r.d = h2f(f2h(d));
  r.s = Q81 ? h2f(f2h(opaque(__fmul_rn(float(r.sum), d)))) : 0.f;
  return r;
}

// quantize_row_q8_K (quant.cpp:273-303) of one super-block spread over the 8 lanes of this lane's group (lane k
// holds elements 32k..32k+31 at xs, 16-byte aligned): the first element of largest magnitude sets the scale.
// Returns sub-block k's words in residue order and its two 16-sums; every lane of the wave must call it.
__device__ __forceinline__ void quant_act_k(const float* xs, int k, uint32_t (&aw)[8], int& bs0, int& bs1, float& d) {
  float v[32];
#pragma unroll
  for (int j = 0; j < 32; j += 4) {
    const float4 f = *reinterpret_cast<const float4*>(xs + j);
    v[j] = f.x, v[j + 1] = f.y, v[j + 2] = f.z, v[j + 3] = f.w;
  }
  float own = 0.f, amax;
  int key = 0, nanf = 0;
#pragma unroll
  for (int e = 0; e < 32; ++e) {
    const float ax = fabsf(v[e]);
    if (ax > own) own = ax, key = 2 * (32 * k + e) + (v[e] < 0.f ? 1 : 0);
    nanf |= v[e] != v[e];
  }
  const float mx = block_max<8>(own, key, amax);
  nanf |= dpp<kQuadXor1>(nanf);
  nanf |= dpp<kQuadXor2>(nanf);
  nanf |= dpp<kMirror8>(nanf);
  int q[32];
  d = 0.f;
  bs0 = bs1 = 0;
  if (amax != 0.f) {
    const float iscale = __fdiv_rn(-127.f, mx);
#pragma unroll
    for (int e = 0; e < 32; ++e) {
      const float sv = __fmul_rn(iscale, v[e]);
      q[e] = sv != sv ? 0 : nearest_int(fminf(127.f, fmaxf(-127.f, sv)));
      if (e < 16) bs0 += q[e]; else bs1 += q[e];
    }
    d = __fdiv_rn(1.f, iscale);
  } else {
#pragma unroll
    for (int e = 0; e < 32; ++e) q[e] = 0;
  }
#pragma unroll
  for (int w = 0; w < 8; ++w)
    aw[w] = uint32_t(q[w] & 0xFF) | uint32_t(q[w + 8] & 0xFF) << 8 | uint32_t(q[w + 16] & 0xFF) << 16 |
            uint32_t(q[w + 24] & 0xFF) << 24;
  if (nanf) d = __builtin_nanf("");
}

// ---- block terms ----

// Legacy block b of weight row rr against one activation block: the block's float term (header comment).
template <int T>
__device__ __forceinline__ float legacy_term(const QW& W, int64_t rr, int64_t b, const ActL& A) {
  const int64_t wb = rr * W.nb + b;
  const float dw = h2f(W.d[wb]), da = A.d;
  if constexpr (T == kQ8_0) {
    const uint4* wp = reinterpret_cast<const uint4*>(W.q + wb * 32);
    const uint4 w0 = wp[0], w1 = wp[1];
    int s = sdot4(w0.x, A.a[0], 0);
    s = sdot4(w0.y, A.a[1], s), s = sdot4(w0.z, A.a[2], s), s = sdot4(w0.w, A.a[3], s);
    s = sdot4(w1.x, A.a[4], s), s = sdot4(w1.y, A.a[5], s), s = sdot4(w1.z, A.a[6], s), s = sdot4(w1.w, A.a[7], s);
    return __fmul_rn(float(s), __fmul_rn(dw, da));
  } else {
    const uint4 wv = *reinterpret_cast<const uint4*>(W.q + wb * 16);
    const uint32_t w[4] = {wv.x, wv.y, wv.z, wv.w};
    // element j of the block: low nibble of byte j (j < 16), high nibble of byte j - 16 (j >= 16)
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) lo[i] = w[i] & 0x0F0F0F0Fu, hi[i] = (w[i] >> 4) & 0x0F0F0F0Fu;
    if constexpr (T == kQ5_0 || T == kQ5_1) {
      const uint32_t qh = *reinterpret_cast<const uint32_t*>(W.h + wb * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = 4 * i + e;
          lo[i] |= ((qh >> j) & 1u) << (8 * e + 4);
          hi[i] |= ((qh >> (j + 16)) & 1u) << (8 * e + 4);
        }
    }
    int s = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) s = sdot4(lo[i], A.a[i], s), s = sdot4(hi[i], A.a[i + 4], s);
    if constexpr (T == kQ4_0) return __fmul_rn(__fmul_rn(float(s - 8 * A.sum), dw), da);
    if constexpr (T == kQ5_0) return __fmul_rn(__fmul_rn(dw, da), float(s - 16 * A.sum));
    if constexpr (T == kQ5_1) return __fadd_rn(__fmul_rn(__fmul_rn(dw, da), float(s)), __fmul_rn(h2f(W.m[wb]), A.s));
  }
  return 0.f;
}

// A legacy weight block in registers (loaded ahead of the activation work that hides its latency).
struct WBlk {
  uint4 q0, q1;  // quants (q1: Q8_0's second half)
  uint32_t h;    // Q5_0 / Q5_1 high bits
  uint16_t d, m;
};

template <int T>
__device__ __forceinline__ WBlk load_wblk(const QW& W, int64_t rr, int64_t b) {
  const int64_t wb = rr * W.nb + b;
  WBlk k;
  if constexpr (T == kQ8_0) {
    const uint4* wp = reinterpret_cast<const uint4*>(W.q + wb * 32);
    k.q0 = wp[0], k.q1 = wp[1];
  } else {
    k.q0 = *reinterpret_cast<const uint4*>(W.q + wb * 16);
  }
  if constexpr (T == kQ5_0 || T == kQ5_1) k.h = reinterpret_cast<const uint32_t*>(W.h)[wb];
  k.d = W.d[wb];
  if constexpr (T == kQ5_1) k.m = W.m[wb];
  return k;
}

// legacy_term on a preloaded weight block.
template <int T>
__device__ __forceinline__ float wblk_term(const WBlk& k, const ActL& A) {
  const float dw = h2f(k.d), da = A.d;
  if constexpr (T == kQ8_0) {
    int s = sdot4(k.q0.x, A.a[0], 0);
    s = sdot4(k.q0.y, A.a[1], s), s = sdot4(k.q0.z, A.a[2], s), s = sdot4(k.q0.w, A.a[3], s);
    s = sdot4(k.q1.x, A.a[4], s), s = sdot4(k.q1.y, A.a[5], s), s = sdot4(k.q1.z, A.a[6], s), s = sdot4(k.q1.w, A.a[7], s);
    return __fmul_rn(float(s), __fmul_rn(dw, da));
  } else {
    const uint32_t w[4] = {k.q0.x, k.q0.y, k.q0.z, k.q0.w};
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) lo[i] = w[i] & 0x0F0F0F0Fu, hi[i] = (w[i] >> 4) & 0x0F0F0F0Fu;
    if constexpr (T == kQ5_0 || T == kQ5_1) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = 4 * i + e;
          lo[i] |= ((k.h >> j) & 1u) << (8 * e + 4);
          hi[i] |= ((k.h >> (j + 16)) & 1u) << (8 * e + 4);
        }
    }
    int s = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) s = sdot4(lo[i], A.a[i], s), s = sdot4(hi[i], A.a[i + 4], s);
    if constexpr (T == kQ4_0) return __fmul_rn(__fmul_rn(float(s - 8 * A.sum), dw), da);
    if constexpr (T == kQ5_0) return __fmul_rn(__fmul_rn(dw, da), float(s - 16 * A.sum));
    if constexpr (T == kQ5_1) return __fadd_rn(__fmul_rn(__fmul_rn(dw, da), float(s)), __fmul_rn(h2f(k.m), A.s));
  }
  return 0.f;
}

// ggml get_scale_min_k4 (quant.cpp:52-61)
__device__ __forceinline__ void scale_min_k4(int j, const uint8_t* q, int& d, int& m) {
  if (j < 4) {
    d = q[j] & 63;
    m = q[j + 4] & 63;
  } else {
    d = (q[j + 4] & 0xF) | ((q[j - 4] >> 6) << 4);
    m = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
  }
}

__device__ __forceinline__ void load32(const uint8_t* p, uint32_t (&w)[8]) {
  const uint4 a = reinterpret_cast<const uint4*>(p)[0], b = reinterpret_cast<const uint4*>(p)[1];
  w[0] = a.x, w[1] = a.y, w[2] = a.z, w[3] = a.w, w[4] = b.x, w[5] = b.y, w[6] = b.z, w[7] = b.w;
}

// The integer lanes of super-block sb of row rr against an activation super-block whose sub-block k words are
// act(k, w) (residue order) and 16-sums bsum(g): aux[w] = sum over the block's elements e with e % 8 == w of
// scale(e) * (a_e * q_e) (quant.cpp:118-144, 394-416), and for Q4_K / Q5_K sumi = sum_k (bsums) * m_k.
// SPL > 1: this lane takes part `part` of SPL equal shares of the sub-blocks (the same code for every part, only
// the data offsets differ, so lanes of different parts do not diverge); the integer results of the parts add up
// to the whole block's (exactly: integer sums).
template <int T, int SPL = 1, class ActW, class BSum>
__device__ __forceinline__ void k_lanes(const QW& W, int64_t rr, int64_t sb, ActW act, BSum bsum, int (&aux)[8],
                                        int& sumi, int part = 0) {
  const int64_t wb = rr * W.nb + sb;
#pragma unroll
  for (int w = 0; w < 8; ++w) aux[w] = 0;
  sumi = 0;
  const uint8_t* sc = W.s + wb * 16;
  if constexpr (T == kQ4_K || T == kQ5_K) {
    uint32_t hw[8];
    if constexpr (T == kQ5_K) load32(W.h + wb * 32, hw);
#pragma unroll
    for (int cc = 0; cc < 4 / SPL; ++cc) {
      const int c = cc + (4 / SPL) * part;
      uint32_t qw[8];
      load32(W.q + wb * 128 + 32 * c, qw);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int k = 2 * c + half;
        int s, m;
        scale_min_k4(k, sc, s, m);
        sumi += (bsum(2 * k) + bsum(2 * k + 1)) * m;
#pragma unroll
        for (int w = 0; w < 8; ++w) {
          uint32_t v = (qw[w] >> (4 * half)) & 0x0F0F0F0Fu;
          if constexpr (T == kQ5_K) v |= ((hw[w] >> k) & 0x01010101u) << 4;
          aux[w] += s * sdot4(v, act(k, w), 0);
        }
      }
    }
  } else {  // Q6_K: sub-block k = 4h + g of the 128-element half h; values 0..63 less 32 (quant.cpp:84-96)
    const int8_t* scl = reinterpret_cast<const int8_t*>(sc);
#pragma unroll
    for (int hh = 0; hh < 2 / SPL; ++hh) {
      const int h = hh + (2 / SPL) * part;
      uint32_t hw[8];
      load32(W.h + wb * 64 + 32 * h, hw);
#pragma unroll
      for (int lg = 0; lg < 2; ++lg) {  // ql group: bytes 64h + 32lg .. +31 (sub-blocks g = lg and lg + 2)
        uint32_t lw[8];
        load32(W.q + wb * 128 + 64 * h + 32 * lg, lw);
#pragma unroll
        for (int sel = 0; sel < 2; ++sel) {
          const int g = lg + 2 * sel, k = 4 * h + g;
          const int s_lo = scl[2 * k], s_hi = scl[2 * k + 1];
#pragma unroll
          for (int w = 0; w < 8; ++w) {
            const uint32_t v = ((lw[w] >> (4 * sel)) & 0x0F0F0F0Fu) | (((hw[w] >> (2 * g)) & 0x03030303u) << 4);
            const uint32_t a = act(k, w);
            // bytes 0, 1 of a residue word are elements w, w + 8 (the first 16: scale s_lo); bytes 2, 3 the rest
            const int dlo = sdot4(v & 0x0000FFFFu, a, 0) - 32 * sdot4(0x00000101u, a, 0);
            const int dhi = sdot4(v & 0xFFFF0000u, a, 0) - 32 * sdot4(0x01010000u, a, 0);
            aux[w] += s_lo * dlo + s_hi * dhi;
          }
        }
      }
    }
  }
}

// ---- the matmul ----

constexpr int kMaxQWeights = NBHS_GEMV_MAX_WEIGHTS;
struct QBatch {  // weights of one type sharing one input; wave0: first wave of each weight's rows
  QW w[kMaxQWeights];
  float* y[kMaxQWeights];
  int64_t wave0[kMaxQWeights];
  int n_w;
};

// Weight rows per wave: a legacy row has a block per lane (in = 2048: 64 blocks), a K row a super-block per lane
// (in = 2048: 8), so K waves take twice the rows; with 16 activation rows a wave's outputs are capped at 64. A
// single-row launch over many rows (an FFN's 16384) takes 16 rows per wave: the activation row each wave quantizes
// is then shared by more weight rows, and there are still a thousand or more waves.
constexpr int rows_per_wave(bool k, int NT, bool wide) {
  return NT > 4 ? 4 : k ? (NT == 1 && !wide ? 4 : 8) : wide && NT == 1 ? 16 : 4;
}
// K types with one activation row in a launch of QKV size: each (row, super-block) pair is split over two adjacent
// lanes (half the sub-blocks each), which halves the serial integer chain per lane and doubles the waves. Wide
// launches (an FFN's 16384 rows) have waves enough and lose more to the activation quantization each wave repeats.
constexpr int k_split(bool k, int NT, bool wide) { return k && NT == 1 && !wide ? 2 : 1; }
constexpr int64_t kWideRows = 16384;  // total rows of a launch from which single-row launches go wide

// A K activation super-block staged in LDS on the fused path: 256 quants in residue order, d, the 16-sums.
struct LdsActK {
  uint32_t a[64];
  float d;
  int bs[16];
};

// FUSED: the activation rows are quantized here, from x (NT <= 4), instead of read from A.
template <int T, int NT, bool FUSED, bool WIDE>
__global__ __launch_bounds__(64) void qgemv_kernel(QBatch B, QA A, const float* __restrict__ x, int64_t in, int n) {
  constexpr bool K = T == kQ4_K || T == kQ5_K || T == kQ6_K;
  constexpr int RW = rows_per_wave(K, NT, WIDE);
  constexpr int O = RW * NT;  // outputs of this wave
  constexpr int CH = K ? 8 : 64;  // blocks per chunk
  constexpr int TERMS = K ? 9 : 1;
  static_assert(O <= 64, "one lane per output in the ordered sum");
  static_assert(!FUSED || NT <= 4, "fused activation quantization stages at most 4 rows");
  __shared__ float terms[O][CH][TERMS];
  __shared__ LdsActK acts[K && FUSED ? NT : 1][K ? CH : 1];
  const int lane = threadIdx.x;
  int wi = 0;
  for (int j = 1; j < B.n_w; ++j)
    if (int64_t(blockIdx.x) >= B.wave0[j]) wi = j;
  const QW& W = B.w[wi];
  float* __restrict__ y = B.y[wi];
  const int64_t r0 = (int64_t(blockIdx.x) - B.wave0[wi]) * RW;
  const int nr = int(W.rows - r0 < RW ? W.rows - r0 : RW);
  float acc = 0.f, sums[8];
#pragma unroll
  for (int l = 0; l < 8; ++l) sums[l] = 0.f;
  for (int64_t c0 = 0; c0 < W.nb; c0 += CH) {
    const int nc = int(W.nb - c0 < CH ? W.nb - c0 : CH);
    if constexpr (FUSED && K) {  // quantize this chunk's activation super-blocks once, into LDS
      const int sbl = lane >> 3, k = lane & 7;
      const int64_t sb = c0 + (sbl < nc ? sbl : 0);
      for (int t = 0; t < NT; ++t) {
        if (t >= n) break;
        uint32_t aw[8];
        int bs0, bs1;
        float d;
        quant_act_k(x + int64_t(t) * in + sb * 256 + 32 * k, k, aw, bs0, bs1, d);
        if (sbl < nc) {
          LdsActK& o = acts[t][sbl];
#pragma unroll
          for (int w = 0; w < 8; ++w) o.a[8 * k + w] = aw[w];
          o.bs[2 * k] = bs0, o.bs[2 * k + 1] = bs1;
          if (k == 0) o.d = d;
        }
      }
      __syncthreads();
    }
    // phase 1: the term(s) of every (row, block) pair, for each activation row
    if constexpr (!K) {  // a block per lane; its activation block (quantized here when fused) serves every row
      if (lane < nc) {
        const int64_t b = c0 + lane;
        // every row's weight block is requested before the activation work, which hides the loads' latency
        WBlk wk[RW];
#pragma unroll
        for (int r = 0; r < RW; ++r) wk[r] = load_wblk<T>(W, r0 + (r < nr ? r : nr - 1), b);
        for (int t = 0; t < NT; ++t) {
          if (t >= n) break;
          ActL a;
          if constexpr (FUSED)
            a = quant_act_l<T == kQ5_1>(x + int64_t(t) * in + b * 32);
          else
            a = load_act_l(A, t, b);
#pragma unroll
          for (int r = 0; r < RW; ++r) terms[r * NT + t][lane][0] = wblk_term<T>(wk[r], a);
        }
      }
    } else {
      constexpr int SPL = k_split(K, NT, WIDE);
      // RW * nc * SPL <= 64 (nc <= 8), so the two lanes of a split pair are always in the same pass
      for (int p = lane; p < RW * nc * SPL; p += 64) {
        const int pair = p / SPL, part = p % SPL;
        const int r = pair / nc, bl = pair % nc;
        const int64_t rr = r0 + (r < nr ? r : nr - 1), b = c0 + bl;
        for (int t = 0; t < NT; ++t) {
          if (t >= n) break;
          int aux[8], sumi;
          float da;
          if constexpr (FUSED) {
            const LdsActK& s = acts[t][bl];
            k_lanes<T, SPL>(W, rr, b, [&](int k, int w) { return s.a[8 * k + w]; }, [&](int g) { return s.bs[g]; },
                            aux, sumi, part);
            da = s.d;
          } else {
            const int64_t ab = int64_t(t) * A.nb + b;
            const uint32_t* aq = reinterpret_cast<const uint32_t*>(A.qs + ab * 256);
            const int16_t* bs = A.bsums + ab * 16;
            k_lanes<T, SPL>(W, rr, b, [&](int k, int w) { return aq[8 * k + w]; }, [&](int g) { return int(bs[g]); },
                            aux, sumi, part);
            da = A.d[ab];
          }
          if constexpr (SPL == 2) {  // the partner lane (p ^ 1) holds the other half
#pragma unroll
            for (int l = 0; l < 8; ++l) aux[l] += __shfl_xor(aux[l], 1, 64);
            sumi += __shfl_xor(sumi, 1, 64);
            if (part != 0) continue;
          }
          const int64_t wb = rr * W.nb + b;
          const float d = __fmul_rn(h2f(W.d[wb]), da);
#pragma unroll
          for (int l = 0; l < 8; ++l) terms[r * NT + t][bl][l] = __fmul_rn(d, float(aux[l]));
          terms[r * NT + t][bl][8] = T == kQ6_K ? 0.f : __fmul_rn(__fmul_rn(h2f(W.m[wb]), da), float(sumi));
        }
      }
    }
    __syncthreads();
    // phase 2: each output adds its terms in block order
    if (lane < O) {
      if constexpr (!K) {
        for (int b = 0; b < nc; ++b) acc = __fadd_rn(acc, terms[lane][b][0]);
      } else {
        for (int b = 0; b < nc; ++b) {
#pragma unroll
          for (int l = 0; l < 8; ++l) sums[l] = __fadd_rn(sums[l], terms[lane][b][l]);
          if constexpr (T != kQ6_K) acc = __fsub_rn(acc, terms[lane][b][8]);
        }
      }
    }
    __syncthreads();
  }
  if (lane < O) {
    if constexpr (K) {
#pragma unroll
      for (int l = 0; l < 8; ++l) acc = __fadd_rn(acc, sums[l]);
    }
    const int r = lane / NT, t = lane % NT;
    if (r < nr && t < n) y[int64_t(t) * W.rows + r0 + r] = acc;
  }
}

// ---- the K types with up to 4 activation rows ----
//
// kgemv_kernel: a workgroup of four waves quantizes the activation rows into LDS once, together, and each wave then
// takes weight rows of its own. Four lanes share a (row, super-block) pair: lane c takes the 32-byte chunk c of its quants
// (sub-blocks 2 c and 2 c + 1; Q6_K: sub-blocks k and k + 2, k = 4 (c / 2) + c % 2), so a wave's 16 pairs are 16 whole
// super-blocks read contiguously, and its two sub-blocks' activation words stay in registers for every row. The four
// lanes' integer lane sums are added exactly by DPP, lane c keeping aux[2 c] and aux[2 c + 1]; their float terms go to
// the wave's LDS slice and are then added in super-block order, a lane per (row, integer lane) chain: the reference's
// operations in its order (quant.cpp:118-144, 394-416).
// A pass of 16 pairs is 2.3-3.4 KB per wave, so P passes are requested before any is computed. What bounds it by its
// counters: VALU issue at many rows (131072 rows, K = 2048, one activation row: the VALU busy 67 % of the time with Q6_K at
// 4.5 TB/s, 58 % with Q4_K; waves wait 35-42 % of their time to issue and 26-30 % for loads), the loads' latency at few
// (2048 rows, K = 8192: the VALU busy 18 %, 47 % of the time waiting for loads). Two activation rows have an instance of
// their own, whose LDS leaves room for up to four workgroups on a CU; the one for four rows holds two. us a call: 131072
// weight rows, K = 2048, Q6_K 48, Q4_K 32; 2048 rows, K = 8192, Q6_K 9.9, Q4_K 8.8; 3072 rows, K = 2048, Q4_K 6.1, three
// activation rows 9.8.
constexpr int kGemvChunk = 16;  // super-blocks of a pass
constexpr int kgemv_max_sb(int nt) { return nt == 1 ? 64 : 32; }  // super-blocks of a row, at most (LDS)

// Sum over the four lanes of a quad, lane c keeping values 2 c and 2 c + 1 of 8.
__device__ __forceinline__ void quad_reduce(const int (&v)[8], int c, int& r0, int& r1) {
  int h[4];
  const bool hi = (c & 2) != 0, odd = (c & 1) != 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) h[i] = (hi ? v[4 + i] : v[i]) + dpp<kQuadXor2>(hi ? v[i] : v[4 + i]);
  r0 = (odd ? h[2] : h[0]) + dpp<kQuadXor1>(odd ? h[0] : h[2]);
  r1 = (odd ? h[3] : h[1]) + dpp<kQuadXor1>(odd ? h[1] : h[3]);
}

template <int T>
struct KChunk {  // a lane's share of a (row, super-block) pair, as loaded
  u32x4_t q[2], h[2];
  u32x4_t sc;   // Q4_K / Q5_K: the 12 packed bytes; Q6_K: words 0, 1 hold the 8 scales of half c / 2
  uint16_t d, m;
  __device__ __forceinline__ void load(const QW& W, int64_t wb, int c) {
    const u32x4_t* qp = reinterpret_cast<const u32x4_t*>(W.q + wb * 128 + 32 * c);
    q[0] = __builtin_nontemporal_load(qp), q[1] = __builtin_nontemporal_load(qp + 1);
    if constexpr (T == kQ5_K) {
      const u32x4_t* hp = reinterpret_cast<const u32x4_t*>(W.h + wb * 32);
      h[0] = hp[0], h[1] = hp[1];
    }
    if constexpr (T == kQ6_K) {
      const u32x4_t* hp = reinterpret_cast<const u32x4_t*>(W.h + wb * 64 + 32 * (c >> 1));
      h[0] = hp[0], h[1] = hp[1];
      const u32x2_t s = *reinterpret_cast<const u32x2_t*>(W.s + wb * 16 + 8 * (c >> 1));
      sc[0] = s[0], sc[1] = s[1];
    } else {
      sc = *reinterpret_cast<const u32x4_t*>(W.s + wb * 16);
      m = W.m[wb];
    }
    d = W.d[wb];
  }
};

// NT activation rows at most, super-blocks per row at most MAXSB, P passes in flight.
template <int T, int NT, int P>
__global__ __launch_bounds__(256) void kgemv_kernel(QBatch B, const float* __restrict__ x, int64_t in, int n, int batches) {
  constexpr int MAXSB = kgemv_max_sb(NT);
  constexpr int TS = kGemvChunk + 1;  // floats per chain of terms (one of padding)
  constexpr int CH = T == kQ6_K ? 8 : 9;
  __shared__ __align__(16) uint32_t qs[NT][MAXSB][64];
  __shared__ float ad[NT][MAXSB];
  __shared__ int bsum[NT][T == kQ6_K ? 1 : MAXSB][8];
  constexpr int RB = 8;  // rows of a wave's batch, at most: a lane per (row, integer lane)
  __shared__ float terms[4][RB][CH][TS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 3;
  int wi = 0;
  for (int j = 1; j < B.n_w; ++j)
    if (int64_t(blockIdx.x) >= B.wave0[j]) wi = j;
  const QW W = B.w[wi];
  float* __restrict__ y = B.y[wi];
  const int nb = int(W.nb), nbc = nb < kGemvChunk ? nb : kGemvChunk, rp = kGemvChunk / nbc;  // rows of a pass
  const int rb = P * rp < RB ? P * rp : RB, np = (rb + rp - 1) / rp;                          // rows, passes of a batch
  const int u = lane >> 2, ur = u / nbc, us = u - ur * nbc;  // this lane's row and super-block within a pass
  const int64_t r00 = ((int64_t(blockIdx.x) - B.wave0[wi]) * 4 + wave) * rb * batches;
  // the first weight loads, ahead of the activation work
  KChunk<T> k[P];
  auto load_pass = [&](int64_t r0, int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int64_t r = r0 + p * rp + ur;
      k[p].load(W, (r < W.rows ? r : W.rows - 1) * nb + (s0 + us < nb ? s0 + us : nb - 1), c);
    }
  };
  load_pass(r00, 0);
  // quantize_row_q8_K (quant.cpp:273-303), the same bits either way: few super-blocks a wave each, four elements per
  // lane; many eight lanes each, 32 elements per lane. A wave each against eight lanes each, us a call with 2048-4096 weight
  // rows: 8 super-blocks 5.4 / 6.4, 16 (two rows of 8) 7.0 / 6.9, 24 8.8 / 7.5, 32 11.3 / 8.8.
  if (n * nb <= 16) {
    for (int i = wave; i < n * nb; i += 4) {
      const int t = i / nb, sb = i - t * nb, kk = lane >> 3, w = lane & 7;
      int q[4], b0, b1;
      float d;
      q8k_lane(x + int64_t(t) * in + sb * 256 + 32 * kk + w, lane, q, b0, b1, d);
      qs[t][sb][lane] = uint32_t(q[0] & 0xFF) | uint32_t(q[1] & 0xFF) << 8 | uint32_t(q[2] & 0xFF) << 16 |
                        uint32_t(q[3] & 0xFF) << 24;
      if (T != kQ6_K && w == 0) bsum[t][T == kQ6_K ? 0 : sb][kk] = b0 + b1;
      if (lane == 0) ad[t][sb] = d;
    }
  } else {
    for (int i0 = 0; i0 < n * nb; i0 += 32) {
      const int i = i0 + (tid >> 3), kk = lane & 7, ic = i < n * nb ? i : 0;
      const int t = ic / nb, sb = ic - t * nb;
      uint32_t aw[8];
      int b0, b1;
      float d;
      quant_act_k(x + int64_t(t) * in + sb * 256 + 32 * kk, kk, aw, b0, b1, d);
      if (i < n * nb) {
#pragma unroll
        for (int w = 0; w < 8; ++w) qs[t][sb][8 * kk + w] = aw[w];
        if constexpr (T != kQ6_K) bsum[t][sb][kk] = b0 + b1;
        if (kk == 0) ad[t][sb] = d;
      }
    }
  }
  __syncthreads();
  const int k0 = T == kQ6_K ? 4 * (c >> 1) + (c & 1) : 2 * c, k1 = T == kQ6_K ? k0 + 2 : k0 + 1;  // its sub-blocks
  const int cr = lane >> 3, cl = lane & 7;  // the chain this lane adds: row of the batch, integer lane
  for (int b = 0; b < batches; ++b) {
    const int64_t r0 = r00 + int64_t(b) * rb;
    if (r0 >= W.rows) break;  // (a wave leaves alone: no workgroup barrier follows)
    float sum[NT], acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) sum[t] = acc[t] = 0.f;
    for (int s0 = 0; s0 < nb; s0 += kGemvChunk) {
      if (b > 0 || s0 > 0) load_pass(r0, s0);
      const int sb = s0 + us < nb ? s0 + us : nb - 1;
      const int nc = nb - s0 < kGemvChunk ? nb - s0 : kGemvChunk;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (t >= n) break;
        uint32_t a0[8], a1[8];
        load32(reinterpret_cast<const uint8_t*>(&qs[t][sb][8 * k0]), a0);
        load32(reinterpret_cast<const uint8_t*>(&qs[t][sb][8 * k1]), a1);
        const float da = ad[t][sb];
#pragma unroll
        for (int p = 0; p < P; ++p) {
          if (p >= np) break;
          const KChunk<T>& K = k[p];
          int aux[8], sumi = 0;
          if constexpr (T == kQ6_K) {
            const int sh = 16 * (c & 1);  // scales of sub-block k0: bytes 2 (c % 2), + 1 of the half; of k1: + 4
            const int s0l = int8_t(K.sc[0] >> sh), s0h = int8_t(K.sc[0] >> (sh + 8));
            const int s1l = int8_t(K.sc[1] >> sh), s1h = int8_t(K.sc[1] >> (sh + 8));
            const int hs = 2 * (c & 1);  // bits of sub-block k0 in a high-bit byte; of k1: + 4
#pragma unroll
            for (int w = 0; w < 8; ++w) {
              const uint32_t qw = K.q[w >> 2][w & 3], hw = K.h[w >> 2][w & 3] >> hs;
              // values less 32, bytewise: (v | 128) - 32 never borrows, and the top bit flips back
              const uint32_t v0 = (((qw & 0x0F0F0F0Fu) | ((hw & 0x03030303u) << 4) | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
              const uint32_t v1 =
                  ((((qw >> 4) & 0x0F0F0F0Fu) | (hw & 0x30303030u) | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
              aux[w] = s0l * sdot4(v0 & 0xFFFFu, a0[w], 0) + s0h * sdot4(v0 & 0xFFFF0000u, a0[w], 0) +
                       s1l * sdot4(v1 & 0xFFFFu, a1[w], 0) + s1h * sdot4(v1 & 0xFFFF0000u, a1[w], 0);
            }
          } else {
            const uint32_t hi = c >= 2 ? ~0u : 0u;  // get_scale_min_k4 (quant.cpp:52-61), four sub-blocks to a word
            const uint32_t d4 =
                (((K.sc[2] & 0x0F0F0F0Fu) | ((K.sc[0] >> 2) & 0x30303030u)) & hi) | (K.sc[0] & 0x3F3F3F3Fu & ~hi);
            const uint32_t m4 =
                ((((K.sc[2] >> 4) & 0x0F0F0F0Fu) | ((K.sc[1] >> 2) & 0x30303030u)) & hi) | (K.sc[1] & 0x3F3F3F3Fu & ~hi);
            const int sh = 16 * (c & 1);
            const int s0_ = int((d4 >> sh) & 0xFFu), s1_ = int((d4 >> (sh + 8)) & 0xFFu);
#pragma unroll
            for (int w = 0; w < 8; ++w) {
              const uint32_t qw = K.q[w >> 2][w & 3];
              uint32_t v0 = qw & 0x0F0F0F0Fu, v1 = (qw >> 4) & 0x0F0F0F0Fu;
              if constexpr (T == kQ5_K) {
                const uint32_t hw = K.h[w >> 2][w & 3] >> (2 * c);
                v0 |= (hw & 0x01010101u) << 4;
                v1 |= (hw & 0x02020202u) << 3;
              }
              aux[w] = s0_ * sdot4(v0, a0[w], 0) + s1_ * sdot4(v1, a1[w], 0);
            }
            sumi = bsum[t][T == kQ6_K ? 0 : sb][2 * c] * int((m4 >> sh) & 0xFFu) +
                   bsum[t][T == kQ6_K ? 0 : sb][2 * c + 1] * int((m4 >> (sh + 8)) & 0xFFu);
          }
          int x0, x1;
          quad_reduce(aux, c, x0, x1);
          const float d = __fmul_rn(h2f(K.d), da);
          const int br = p * rp + ur;  // row of the batch
          if (ur < rp && br < rb) {
            float* o = &terms[wave][br][0][us];
            o[(2 * c) * TS] = __fmul_rn(d, float(x0));
            o[(2 * c + 1) * TS] = __fmul_rn(d, float(x1));
          }
          if constexpr (T != kQ6_K) {
            sumi += dpp<kQuadXor1>(sumi);
            sumi += dpp<kQuadXor2>(sumi);
            if (c == 0 && ur < rp && br < rb) terms[wave][br][CH - 1][us] = __fmul_rn(__fmul_rn(h2f(K.m), da), float(sumi));
          }
        }
        // the wave's terms of this chunk, in super-block order
        wave_lds_sync();
        const float* tp = &terms[wave][cr][cl][0];
        const float* mp = &terms[wave][cr][CH - 1][0];
        float tv[kGemvChunk], mv[kGemvChunk];
#pragma unroll
        for (int i = 0; i < kGemvChunk; ++i) {  // (past nc: read, not added)
          tv[i] = tp[i];
          if constexpr (T != kQ6_K) mv[i] = mp[i];
        }
#pragma unroll
        for (int i = 0; i < kGemvChunk; ++i) {
          if (i < nc) {
            sum[t] = __fadd_rn(sum[t], tv[i]);
            if constexpr (T != kQ6_K) acc[t] = __fsub_rn(acc[t], mv[i]);
          }
        }
        wave_lds_sync();
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (t >= n) break;
      float o = acc[t];
#pragma unroll
      for (int l = 0; l < 8; ++l) o = __fadd_rn(o, __shfl(sum[t], (lane & 56) + l, 64));
      if (cl == 0 && cr < rb && r0 + cr < W.rows) y[int64_t(t) * W.rows + r0 + cr] = o;
    }
  }
}

// ---- the tiled matmul for longer calls (prefill chunks) ----
//
// qgemm_legacy_kernel: a 256-thread workgroup computes 64 weight rows x 16 TJ activation rows on the int8 matrix
// cores. A legacy block is 32 elements, exactly the contraction of one v_mfma_i32_16x16x32_i8, so each (16 weight
// rows, 16 activation rows, block) is one MFMA from zero: the block's exact integer dots (Q4_0 / Q5_0 as
// sum q_w q_a, the offset term -8 or -16 times the activation block's quant sum applied after, exactly). Every output
// then adds its block's float term - the reference's expression, in block order - so the outputs are bit-exact with
// the v_dot4 path and with quant.cpp. Waves: 2 x 2 over 64 x 64 (TJ = 4), 4 x 1 over 64 x 32 (TJ = 2) or, with
// WRT = 32 weight rows, 2 x 2 over 32 x 32; each lane holds the MFMA result layout's 4 weight rows of one
// activation row per 16 x 16 pair. Chunks of 8 blocks of
// both operands are staged in LDS (one 16-byte pad per row: conflict-free fragment reads); the next chunk's share of
// each thread is loaded into registers while the current one is computed, the weight scales are widened to float
// and an activation block's quant sum taken once at staging. One launch covers the weights of one type that share
// the input (a layer's Q, K and V): grid x runs over the row tiles of all of them, so small weights do not leave
// most CUs idle; TJ = 2 doubles the workgroups of a launch that would otherwise leave most SIMDs with one wave.
constexpr int kGemmCB = 8;  // blocks per staged chunk

struct QGemmBatch {  // weights of one type sharing one input; tile0[i]: first row tile of weight i
  QW w[kMaxQWeights];
  float* y[kMaxQWeights];
  int tile0[kMaxQWeights];
  int n_w;
};

typedef int i32x4_t __attribute__((ext_vector_type(4)));  // an integer MFMA result

// UB: blocks whose LDS reads and MFMAs a wave has in flight.
template <int T, int TJ, int WRT = 64, int UB = 1>
__global__ __launch_bounds__(256) void qgemm_legacy_kernel(QGemmBatch B, QA A, int64_t n) {
  int wi = 0;
  for (int i = 1; i < B.n_w; ++i)
    if (int(blockIdx.x) >= B.tile0[i]) wi = i;
  const QW W = B.w[wi];
  float* __restrict__ y = B.y[wi];
  constexpr int QB = T == kQ8_0 ? 32 : 16;           // quant bytes per block
  constexpr int QW4 = QB / 16;                        // u32x4_t per block
  constexpr int WROW = kGemmCB * QW4 + 1;             // u32x4_t per staged weight row (one of padding: spreads banks)
  constexpr int AROW = 2 * kGemmCB + 1;               // u32x4_t per staged activation row (likewise)
  constexpr int AR = 16 * TJ;                         // activation rows per workgroup
  constexpr int NWQ = WRT * kGemmCB * QW4 / 256;       // weight u32x4_t a thread stages per chunk
  constexpr int NWM = WRT * kGemmCB / 256;             // weight block headers a thread stages per chunk
  constexpr int NA = (AR * kGemmCB + 255) / 256;      // activation blocks a thread stages per chunk (at most)
  static_assert(NWQ * 256 == WRT * kGemmCB * QW4 && NWM * 256 == WRT * kGemmCB, "chunks split evenly");
  // Per wave: WM 16-row weight groups x 2 16-row activation groups, one v_mfma_i32_16x16x32_i8 per pair and block
  // (a legacy block is exactly the MFMA's 32-deep contraction). TJ = 4: waves 2 x 2 over 64 x 64; TJ = 2: waves
  // 4 x 1 over 64 x 32.
  constexpr int WM = TJ == 4 && WRT == 64 ? 2 : 1;
  constexpr int WN = WRT == 64 ? 2 : 1;  // 16-row activation groups per wave (32 x 32 tiles: waves 2 x 2 of 16 x 16)
  __shared__ u32x4_t wq[WRT * WROW];
  __shared__ float wdf[kGemmCB][WRT], wmf[kGemmCB][WRT];
  __shared__ uint32_t wh[WRT][kGemmCB];
  __shared__ u32x4_t aq[AR * AROW];
  __shared__ float ad[kGemmCB][AR], as_[kGemmCB][AR];
  __shared__ int asum[kGemmCB][AR];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ml = lane & 15, kg = lane >> 4;  // operand row / column of the lane and its 8-deep k group
  const int wr0 = WRT == 32 ? 16 * (wave & 1) : TJ == 4 ? 32 * (wave & 1) : 16 * wave;
  const int ac0 = WRT == 32 ? 16 * (wave >> 1) : TJ == 4 ? 32 * (wave >> 1) : 0;
  const int64_t row0 = int64_t(int(blockIdx.x) - B.tile0[wi]) * WRT, t0 = int64_t(blockIdx.y) * AR;
  // acc[i][j][v]: weight row wr0 + 16 i + 4 kg + v, activation row ac0 + 16 j + ml (the MFMA's result layout)
  float acc[WM][WN][4];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.f;
  // A thread's share of one chunk, in registers: rows and activation rows past the ends, and blocks past the
  // chunk's end, load clamped (staged but never used).
  struct Share {
    u32x4_t q[NWQ];
    uint32_t d[NWM], m[NWM], h[NWM];
    u32x4_t a0[NA], a1[NA];
    float ad[NA], as[NA];
  };
  auto load_share = [&](int64_t c0, Share& sh) __attribute__((always_inline)) {
    const int nc = int(W.nb - c0 < kGemmCB ? W.nb - c0 : kGemmCB);
#pragma unroll
    for (int u = 0; u < NWQ; ++u) {
      const int e = tid + 256 * u;
      const int r = e / (kGemmCB * QW4), rem = e % (kGemmCB * QW4), b = rem / QW4, part = rem % QW4;
      const int64_t rr = min(row0 + r, W.rows - 1), bb = c0 + min(b, nc - 1);
      sh.q[u] = reinterpret_cast<const u32x4_t*>(W.q + (rr * W.nb + bb) * QB)[part];
    }
#pragma unroll
    for (int u = 0; u < NWM; ++u) {
      const int e = tid + 256 * u;
      const int r = e / kGemmCB, b = e % kGemmCB;
      const int64_t wb = min(row0 + r, W.rows - 1) * W.nb + c0 + min(b, nc - 1);
      sh.d[u] = W.d[wb];
      if constexpr (T == kQ5_1) sh.m[u] = W.m[wb];
      if constexpr (T == kQ5_0 || T == kQ5_1) sh.h[u] = reinterpret_cast<const uint32_t*>(W.h)[wb];
    }
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      const int e = tid + 256 * u;
      if (e < AR * kGemmCB) {
        const int r = e / kGemmCB, b = e % kGemmCB;
        const int64_t ab = min(t0 + r, n - 1) * A.nb + c0 + min(b, nc - 1);
        sh.ad[u] = A.d[ab];
        if constexpr (T == kQ5_1) sh.as[u] = A.s[ab];
        const u32x4_t* ap = reinterpret_cast<const u32x4_t*>(A.qs + ab * 32);
        sh.a0[u] = ap[0];
        sh.a1[u] = ap[1];
      }
    }
  };
  auto store_share = [&](const Share& sh) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < NWQ; ++u) {
      const int e = tid + 256 * u;
      const int r = e / (kGemmCB * QW4), rem = e % (kGemmCB * QW4);
      wq[r * WROW + rem] = sh.q[u];
    }
#pragma unroll
    for (int u = 0; u < NWM; ++u) {
      const int e = tid + 256 * u;
      const int r = e / kGemmCB, b = e % kGemmCB;
      wdf[b][r] = h2f(uint16_t(sh.d[u]));
      if constexpr (T == kQ5_1) wmf[b][r] = h2f(uint16_t(sh.m[u]));
      if constexpr (T == kQ5_0 || T == kQ5_1) wh[r][b] = sh.h[u];
    }
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      const int e = tid + 256 * u;
      if (e < AR * kGemmCB) {
        const int r = e / kGemmCB, b = e % kGemmCB;
        ad[b][r] = sh.ad[u];
        if constexpr (T == kQ5_1) as_[b][r] = sh.as[u];
        aq[r * AROW + 2 * b] = sh.a0[u];
        aq[r * AROW + 2 * b + 1] = sh.a1[u];
        if constexpr (T == kQ4_0 || T == kQ5_0) {
          int sum = 0;
#pragma unroll
          for (int w = 0; w < 4; ++w) sum = sdot4(sh.a0[u][w], 0x01010101u, sum);
#pragma unroll
          for (int w = 0; w < 4; ++w) sum = sdot4(sh.a1[u][w], 0x01010101u, sum);
          asum[b][r] = sum;
        }
      }
    }
  };
  // The lane's A operand (weight row wr0 + 16 i + ml, block elements 8 kg .. 8 kg + 7) as int8 values: element e of
  // a 4/5-bit block is the low nibble of byte e (e < 16) or the high nibble of byte e - 16, plus bit e of qh as
  // bit 4 for the 5-bit types; Q8_0 bytes are the values.
  auto a_operand = [&](int r, int b) __attribute__((always_inline)) {
    const uint32_t* wr = reinterpret_cast<const uint32_t*>(&wq[r * WROW + QW4 * b]);
    uint32_t lo, hi;
    if constexpr (T == kQ8_0) {
      lo = wr[2 * kg], hi = wr[2 * kg + 1];
    } else {
      const int sh = 4 * (kg >> 1);
      lo = (wr[2 * (kg & 1)] >> sh) & 0x0F0F0F0Fu;
      hi = (wr[2 * (kg & 1) + 1] >> sh) & 0x0F0F0F0Fu;
      if constexpr (T == kQ5_0 || T == kQ5_1) {
        const uint32_t bits = (wh[r][b] >> (8 * kg)) & 0xFFu;  // qh bits of elements 8 kg .. 8 kg + 7
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          lo |= ((bits >> e) & 1u) << (8 * e + 4);
          hi |= ((bits >> (e + 4)) & 1u) << (8 * e + 4);
        }
      }
    }
    return long((uint64_t(hi) << 32) | uint64_t(lo));
  };
  Share cur;
  load_share(0, cur);
  for (int64_t c0 = 0; c0 < W.nb; c0 += kGemmCB) {
    const int nc = int(W.nb - c0 < kGemmCB ? W.nb - c0 : kGemmCB);
    store_share(cur);
    __syncthreads();
    // the next chunk's share, in flight while this one is computed (the last chunk loads itself again, unused)
    load_share(c0 + kGemmCB < W.nb ? c0 + kGemmCB : c0, cur);
    auto block = [&](int b) __attribute__((always_inline)) {
      long bop[WN];
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        const uint32_t* ar = reinterpret_cast<const uint32_t*>(&aq[(ac0 + 16 * j + ml) * AROW + 2 * b]);
        bop[j] = long((uint64_t(ar[2 * kg + 1]) << 32) | uint64_t(ar[2 * kg]));
      }
#pragma unroll
      for (int i = 0; i < WM; ++i) {
        const int rb = wr0 + 16 * i;
        const long aop = a_operand(rb + ml, b);
        const float4 dw4 = *reinterpret_cast<const float4*>(&wdf[b][rb + 4 * kg]);
        const float dw[4] = {dw4.x, dw4.y, dw4.z, dw4.w};
        float mw[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (T == kQ5_1) {
          const float4 m4 = *reinterpret_cast<const float4*>(&wmf[b][rb + 4 * kg]);
          mw[0] = m4.x, mw[1] = m4.y, mw[2] = m4.z, mw[3] = m4.w;
        }
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          const i32x4_t c = __builtin_amdgcn_mfma_i32_16x16x32_i8(aop, bop[j], i32x4_t{0, 0, 0, 0}, 0, 0, 0);
          const int t = ac0 + 16 * j + ml;
          const float da = ad[b][t];
          const int sum = T == kQ4_0 || T == kQ5_0 ? asum[b][t] : 0;
          const float sa = T == kQ5_1 ? as_[b][t] : 0.f;
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int s = c[v];
            float term;
            if constexpr (T == kQ8_0) term = __fmul_rn(float(s), __fmul_rn(dw[v], da));
            if constexpr (T == kQ4_0) term = __fmul_rn(__fmul_rn(float(s - 8 * sum), dw[v]), da);
            if constexpr (T == kQ5_0) term = __fmul_rn(__fmul_rn(dw[v], da), float(s - 16 * sum));
            if constexpr (T == kQ5_1) term = __fadd_rn(__fmul_rn(__fmul_rn(dw[v], da), float(s)), __fmul_rn(mw[v], sa));
            acc[i][j][v] = __fadd_rn(acc[i][j][v], term);
          }
        }
      }
    };
    int b = 0;
    if constexpr (UB > 1)
      for (; b + UB <= nc; b += UB) {
#pragma unroll
        for (int u = 0; u < UB; ++u) block(b + u);
      }
    for (; b < nc; ++b) block(b);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t r = row0 + wr0 + 16 * i + 4 * kg + v, t = t0 + ac0 + 16 * j + ml;
        if (r < W.rows && t < n) y[t * W.rows + r] = acc[i][j][v];
      }
}

// The legacy kernel's tile for a launch: 64 x 64 while 64 x 64 tiles give at least kLegacyMinWgs workgroups
// (two per CU); else 64 x 32 while those do; else 32 x 32 (more, smaller workgroups: at the QKV shape 16-80 rows
// run 10-20 % faster than with 64 x 32, and 512 rows 3-5 % slower). A wave of a 32 x 32 tile has one MFMA per block, a
// chain of LDS read, MFMA and float term. While a launch leaves a SIMD about one such wave, or two where a block's
// operands take few registers, four blocks go in flight; beyond, the registers cost waves. One block against four, us a
// call at 64-256, 280-512 and 560-768 workgroups (o: 2048 -> 2048 wide, down: 8192 -> 2048):
//   Q8_0  down x 40  41.9 / 34.7   down x 200  49.2 / 46.9   down x 300  59.8 / 62.5
//   Q5_1  down x 40  60.0 / 54.4   down x 200  74.1 / 72.8   down x 300  95.6 / 91.2
//   Q4_0  down x 40  43.7 / 39.8   down x 200  52.3 / 53.3   o x 200  18.0 / 18.0   down x 300  64.5 / 69.2
//   Q5_0  down x 40  53.4 / 51.7   down x 200  68.3 / 72.4   o x 200  22.0 / 23.0   down x 300  88.7 / 97.5
constexpr int64_t legacy_unroll_wgs(int type) { return type == kQ4_0 || type == kQ5_0 ? 256 : 512; }
constexpr int64_t kLegacyMinWgs = 512;
enum LegacyTile { kTile64x64, kTile64x32, kTile32x32 };
template <int T>
hipError_t launch_legacy(LegacyTile tile, unsigned tiles, int64_t n, hipStream_t s, const QGemmBatch& B,
                         const QA& A) {
  if (tile == kTile64x64)
    return nbhs_timing::launch(NBHS_K_QGEMM, qgemm_legacy_kernel<T, 4>, dim3(tiles, unsigned((n + 63) / 64)),
                               dim3(256), s, B, A, n);
  const dim3 grid{tiles, unsigned((n + 31) / 32)};
  if (tile == kTile64x32)
    return nbhs_timing::launch(NBHS_K_QGEMM, qgemm_legacy_kernel<T, 2>, grid, dim3(256), s, B, A, n);
  if (int64_t(grid.x) * grid.y <= legacy_unroll_wgs(T))
    return nbhs_timing::launch(NBHS_K_QGEMM, qgemm_legacy_kernel<T, 2, 32, 4>, grid, dim3(256), s, B, A, n);
  return nbhs_timing::launch(NBHS_K_QGEMM, qgemm_legacy_kernel<T, 2, 32>, grid, dim3(256), s, B, A, n);
}

// The tiled K matmuls, on the fp16 matrix cores (v_mfma_f32_16x16x32_f16).
// The reference's integer lane w of a super-block is aux[w] = sum over the 32 elements e of residue w (four per
// sub-block) of s(e) * q(e) * a(e), with the sub-block scale s varying along it. One MFMA contracts exactly a
// residue. Its A operand is s q / 16, its B operand 16 a (|a| <= 127), both exact in fp16: s q is at most 63 * 31 for
// Q4_K and Q5_K; for Q6_K s (q - 32) is taken as two operands, s n / 16 for the low nibble n and s (h - 2) for the
// two high bits h, whose MFMAs share an accumulator. Every product and every partial sum is an integer below 2^24
// (at most 32 * 4096 * 127), so the fp32 accumulator holds float(aux[w]) exactly, whatever the order: no integer
// slices to combine and no conversion on the VALU, which the float sums bound (per output and residue a product and
// an addition are left; int8 operands take two or more MFMAs and four or more VALU operations).
// The minimum term's sumi = sum_k m_k b_k (b_k: the sub-block's quant sum, |b_k| <= 4064, m_k <= 63) is one
// v_mfma_f32_16x16x16_f16 over b_k = 64 (b_k >> 6) + (b_k & 63) against (m_k, 64 m_k), likewise exact.
// The float arithmetic that follows is the reference's per output and block: d = fp16(d_w) * d_a, sums[w] +=
// d * aux[w], for Q4_K / Q5_K acc -= (fp16(dmin_w) * d_a) * sumi, result acc + sums[0] + ... + sums[7] - the same
// operations in the same order as qgemv_kernel, so the same bits.
// An A operand is built in registers from a row's raw words: and / or place a nibble pair in the mantissa of an fp16
// constant C (C + n ulp(C)), and one packed multiply-add with (s', -C s') leaves s q / 16 exactly.
template <int T>
constexpr int k_slices() { return T == kQ6_K ? 2 : 1; }

// (w & mask) | base as an fp16 pair. The constant base sits in a vector register, so that the pair is one and / or
// instruction (which takes at most one scalar operand).
__device__ __forceinline__ half2_t magic(uint32_t w, uint32_t mask, uint32_t base) {
  asm("" : "+v"(base));
  return __builtin_bit_cast(half2_t, (w & mask) | base);
}
__device__ __forceinline__ half8_t join(half2_t a, half2_t b, half2_t c, half2_t d) {
  return half8_t{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}
__device__ __forceinline__ half2_t pk_fma(half2_t a, half2_t b, half2_t c) { return __builtin_elementwise_fma(a, b, c); }

// The constants of a lane's two sub-blocks (2 kg and 2 kg + 1), from their staged words (k_scale_words).
template <int T>
struct KScales {
  half2_t s[2], c[2];  // Q4_K / Q5_K: s' and -C s', splat. Q6_K: the two 16-element scales and -64 times them
  half2_t c6[2];       // Q6_K: -6 times the scales
  __device__ __forceinline__ void set(uint32_t w0, uint32_t w1) {
    const uint32_t w[2] = {w0, w1};
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const half2_t v = __builtin_bit_cast(half2_t, w[b]);
      if constexpr (T == kQ6_K) {
        s[b] = v;
        c[b] = v * half2_t{-64, -64};
        c6[b] = v * half2_t{-6, -6};
      } else {
        s[b] = half2_t{v[0], v[0]};
        c[b] = half2_t{v[1], v[1]};
      }
    }
  }
};

// The A operand(s) of residue w for a lane's k group kg (sub-blocks 2 kg, 2 kg + 1), as 8 halves in the order
// (sub-block 2 kg: elements 0, 2), (2 kg + 1: 0, 2), (2 kg: 1, 3), (2 kg + 1: 1, 3) - the order of kActQ8_K16.
// Q4_K / Q5_K: q0 the row's quant word 8 kg + w (low nibbles sub-block 2 kg, high nibbles 2 kg + 1), h the high-bit
// word w. Q6_K: q0, q1 the quant words 16 (kg / 2) + w and + 8, of which nibble kg % 2 belongs to sub-blocks 2 kg and
// 2 kg + 1; h the word 8 (kg / 2) + w, their bits from 4 (kg % 2) on.
template <int T>
__device__ __forceinline__ void k_operand(uint32_t q0, uint32_t q1, uint32_t h, int kg, const KScales<T>& k,
                                          half8_t (&a)[k_slices<T>()]) {
  if constexpr (T == kQ6_K) {
    const int sh = 4 * (kg & 1);
    const uint32_t w0 = q0 >> sh, w1 = q1 >> sh, t = h >> sh;
    constexpr uint32_t M = 0x000F000Fu, C = 0x54005400u;  // 64 + n / 16
    a[0] = join(pk_fma(magic(w0, M, C), k.s[0], k.c[0]), pk_fma(magic(w1, M, C), k.s[1], k.c[1]),
                pk_fma(magic(w0 >> 8, M, C), k.s[0], k.c[0]), pk_fma(magic(w1 >> 8, M, C), k.s[1], k.c[1]));
    constexpr uint32_t H = 0x03000300u, D = 0x44004400u;  // 4 + h
    a[1] = join(pk_fma(magic(t << 8, H, D), k.s[0], k.c6[0]), pk_fma(magic(t << 6, H, D), k.s[1], k.c6[1]),
                pk_fma(magic(t, H, D), k.s[0], k.c6[0]), pk_fma(magic(t >> 2, H, D), k.s[1], k.c6[1]));
  } else {
    constexpr uint32_t L = 0x000F000Fu, G = 0x00F000F0u, C = 0x64006400u;  // 1024 + n, 1024 + 16 n
    const uint32_t q8 = q0 >> 8;
    uint32_t h0 = C, h1 = C, h2 = C, h3 = C;
    asm("" : "+v"(h0));
    if constexpr (T == kQ5_K) {  // bits 2 kg, 2 kg + 1 of each byte of h: bit 4 of n
      const uint32_t t = h >> (2 * kg), b = h0;
      h0 = ((t << 4) & 0x00100010u) | b;
      h1 = ((t << 7) & 0x01000100u) | b;
      h2 = ((t >> 4) & 0x00100010u) | b;
      h3 = ((t >> 1) & 0x01000100u) | b;
    } else {
      h1 = h2 = h3 = h0;
    }
    a[0] = join(pk_fma(__builtin_bit_cast(half2_t, (q0 & L) | h0), k.s[0], k.c[0]),
                pk_fma(__builtin_bit_cast(half2_t, (q0 & G) | h1), k.s[1], k.c[1]),
                pk_fma(__builtin_bit_cast(half2_t, (q8 & L) | h2), k.s[0], k.c[0]),
                pk_fma(__builtin_bit_cast(half2_t, (q8 & G) | h3), k.s[1], k.c[1]));
  }
}

// The words KScales takes, of sub-blocks 2 kg and 2 kg + 1, from a row's 16 scale bytes: Q6_K the pairs of 16-element
// scales as fp16; Q4_K / Q5_K (s / 16, -64 s) for the even sub-block, whose nibbles k_operand reads as 1024 + n, and
// (s / 256, -4 s) for the odd one (1024 + 16 n).
template <int T>
__device__ __forceinline__ void k_scale_words(const u32x4_t& sc, int kg, uint32_t (&w)[2]) {
  if constexpr (T == kQ6_K) {
    const uint32_t lo = kg & 1 ? sc[1] : sc[0], hi = kg & 1 ? sc[3] : sc[2], b = kg & 2 ? hi : lo;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      w[i] = __builtin_bit_cast(uint32_t, half2_t{_Float16(int(int8_t((b >> (16 * i)) & 0xFFu))),
                                                  _Float16(int(int8_t((b >> (16 * i + 8)) & 0xFFu)))});
  } else {  // ggml get_scale_min_k4 (quant.cpp:52-61), four sub-blocks to a word
    const uint32_t hi = kg >= 2 ? ~0u : 0u;
    const uint32_t d4 = (((sc[2] & 0x0F0F0F0Fu) | ((sc[0] >> 2) & 0x30303030u)) & hi) | (sc[0] & 0x3F3F3F3Fu & ~hi);
    const int sh = 16 * (kg & 1);
    const float s0 = float((d4 >> sh) & 0xFFu), s1 = float((d4 >> (sh + 8)) & 0xFFu);
    w[0] = __builtin_bit_cast(uint32_t, half2_t{_Float16(s0 * 0.0625f), _Float16(s0 * -64.f)});
    w[1] = __builtin_bit_cast(uint32_t, half2_t{_Float16(s1 * 0.00390625f), _Float16(s1 * -4.f)});
  }
}

// The A operand of a minimum term (Q4_K / Q5_K) for k group kg, in the order of the sum digits (kActQ8_K16): minimums
// 4 (kg % 2) + 0, 2, 1, 3 against the low digits (kg < 2), 64 times them against the high ones.
__device__ __forceinline__ half4_t k_min_operand(const u32x4_t& sc, int kg) {
  const uint32_t hi = kg & 1 ? ~0u : 0u;
  const uint32_t m4 =
      ((((sc[2] >> 4) & 0x0F0F0F0Fu) | ((sc[1] >> 2) & 0x30303030u)) & hi) | (sc[1] & 0x3F3F3F3Fu & ~hi);
  const _Float16 f = kg < 2 ? _Float16(1) : _Float16(64), c = _Float16(1024);
  const half2_t f2 = {f, f}, c2 = {c, c};
  const half2_t a = (magic(m4, 0x00FF00FFu, 0x64006400u) - c2) * f2, b = (magic(m4 >> 8, 0x00FF00FFu, 0x64006400u) - c2) * f2;
  return half4_t{a[0], a[1], b[0], b[1]};
}

__device__ __forceinline__ void buffer_load_lds16(__amdgpu_buffer_rsrc_t rsrc, void* lds_wave_base, uint32_t voff,
                                                  uint32_t soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, lds_wave_base, 16, voff, soff, 0, 0);
#endif
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, int(bytes), 0x00020000);
}
// s_waitcnt with at most n vector loads outstanding and every LDS operation done
constexpr int vm_lds_wait(int n) { return (n & 15) | (7 << 4) | (0 << 8) | ((n >> 4) << 14); }

// qgemm_k_kernel: 64 weight rows x 32 activation rows per workgroup, 16 x 32 per wave. Operands travel global -> LDS
// by direct-to-LDS buffer loads (rows past the ends read as zeros and are never stored; 16-byte chunks XOR-swizzled by
// row, so fragment reads are conflict-free): the activation rows in half super-blocks (four residues, 256 bytes a
// row) through a 3-stage ring, the raw quants and high bits a super-block ahead. The small planes of the next
// super-block (scales, d and dmin; the activation rows' d and sum digits) are loaded into registers, each by one wave
// and each value by one lane, during this super-block and stored to LDS at its end: the L1's rate of lane requests, not
// bytes, bounded the kernel when every lane loaded the values that it uses (Q4_K, 17408 weight rows x 512 activation
// rows, K = 2048: 123 us, 118 without the sums; this form 95). What bounds it is VALU issue (316 operations per wave and
// super-block, 128 of them the sums) with three waves per SIMD between the loads' latencies: by the counters the VALU is
// busy 78 % of the time at 16384 weight rows x 512 and 48 % at 3072, the matrix cores 18 and 11 %. Tiles of 16 x 64 and 32
// x 32 per wave share an operand build among more sums but take two waves per SIMD and spill: 109 us. A layer's QKV (3072
// rows x 512, K = 2048, 16 layers' weights in turn), with int8 slices as operands and with this form: Q4_K 43 and 22 us
// the kernel, 48.7 and 27.9 with the quantization; Q6_K 61.5 and 27.6, 67.3 and 33.3. (Q5_K spills 12 bytes a lane.)
template <int T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void qgemm_k_kernel(QGemmBatch B, QA A,
                                                                                             int64_t n) {
  static_assert(T == kQ4_K || T == kQ5_K || T == kQ6_K, "K types");
  constexpr int NS = k_slices<T>();
  constexpr int WN = 2, AR = 16 * WN;               // activation row groups per wave, activation rows per workgroup
  constexpr int HB = T == kQ6_K ? 64 : T == kQ5_K ? 32 : 0;  // high-bit bytes per row and super-block
  constexpr int kALoads = AR / 16;                  // direct-to-LDS loads per wave of an activation stage,
  constexpr int kQLoads = 2 + (HB > 0 ? 1 : 0);     // and of a super-block's quants and high bits
  // one object per stage: an LDS read then never waits for the loads into another stage
  __shared__ __align__(16) uint8_t ring0[AR * 256], ring1[AR * 256], ring2[AR * 256];
  __shared__ __align__(16) uint8_t quants0[64 * (128 + HB)], quants1[64 * (128 + HB)];  // by super-block parity
  __shared__ __align__(16) u32x4_t scales[2][64];
  __shared__ __align__(16) float wd[2][64], wm[2][64], ad[2][AR];
  __shared__ __align__(16) half4_t digits[2][AR][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ml = lane & 15, kg = lane >> 4;
  int wi = 0;
  for (int i = 1; i < B.n_w; ++i)
    if (int(blockIdx.x) >= B.tile0[i]) wi = i;
  const QW W = B.w[wi];
  float* __restrict__ y = B.y[wi];
  const int64_t row0 = int64_t(int(blockIdx.x) - B.tile0[wi]) * 64, t0 = int64_t(blockIdx.y) * AR;
  const int wrows = int(W.rows - row0 < 64 ? W.rows - row0 : 64), arows = int(n - t0 < AR ? n - t0 : AR);
  const int nb = int(W.nb);
  const __amdgpu_buffer_rsrc_t ra = rsrc_of(A.qs + t0 * nb * 512, int64_t(arows) * nb * 512);
  const __amdgpu_buffer_rsrc_t rq = rsrc_of(W.q + row0 * nb * 128, int64_t(wrows) * nb * 128);
  const __amdgpu_buffer_rsrc_t rh = rsrc_of(HB ? W.h + row0 * nb * HB : W.q, int64_t(wrows) * nb * HB);
  // Load u of the activation rows fills rows 4 (4 u + wave) .. + 3: lane -> (row, position), and the lane loads the
  // chunk that position holds (position p of row r: chunk p ^ (r % 16)).
  uint32_t aoff[kALoads];
#pragma unroll
  for (int u = 0; u < kALoads; ++u) {
    const int r = 4 * (4 * u + wave) + (lane >> 4);
    aoff[u] = uint32_t(r) * uint32_t(nb) * 512 + 16 * ((lane & 15) ^ (r & 15));
  }
  // quants: position p of row r holds chunk p ^ (r / 2 % 8)
  uint32_t qoff[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int r = 8 * (4 * u + wave) + (lane >> 3);
    qoff[u] = uint32_t(r) * uint32_t(nb) * 128 + 16 * ((lane & 7) ^ ((r >> 1) & 7));
  }
  // high bits: Q6_K four chunks per row (position p: chunk p ^ (r / 4 % 4)), Q5_K two (p ^ (r / 8 % 2))
  const int hr = HB == 64 ? 16 * wave + (lane >> 2) : 16 * wave + (lane >> 1);
  const uint32_t hoff = uint32_t(hr) * uint32_t(nb) * HB +
                        16 * (HB == 64 ? (lane & 3) ^ ((hr >> 2) & 3) : (lane & 1) ^ ((hr >> 3) & 1));
  auto ring = [&](auto st_c) __attribute__((always_inline)) {
    constexpr int st = decltype(st_c)::value % 3;
    return st == 0 ? ring0 : st == 1 ? ring1 : ring2;
  };
  auto quants = [&](auto p_c) __attribute__((always_inline)) { return decltype(p_c)::value % 2 == 0 ? quants0 : quants1; };
  auto fetch = [&](int t, auto st_c) __attribute__((always_inline)) {  // stage t: half t % 2 of super-block t / 2
#pragma unroll
    for (int u = 0; u < kALoads; ++u)
      buffer_load_lds16(ra, ring(st_c) + (4 * u + wave) * 1024, aoff[u], uint32_t(t) * 256);
  };
  auto fetch_quants = [&](int sb, auto p_c) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
      buffer_load_lds16(rq, quants(p_c) + (4 * u + wave) * 1024, qoff[u], uint32_t(sb) * 128);
    if constexpr (HB > 0) {
      if (lane < HB) buffer_load_lds16(rh, quants(p_c) + 64 * 128 + wave * (16 * HB), hoff, uint32_t(sb) * HB);
    }
  };
  // This lane's share of a super-block's small planes: wave 0 the scales of weight row `lane`, wave 1 its d and dmin,
  // wave 2 16 bytes of the activation rows' sum digits, wave 3 d of activation row `lane`. Rows past the ends read as
  // zeros.
  const __amdgpu_buffer_rsrc_t rs = rsrc_of(W.s + row0 * nb * 16, int64_t(wrows) * nb * 16),
                               rd = rsrc_of(W.d + row0 * nb, int64_t(wrows) * nb * 2),
                               rm = rsrc_of(T == kQ6_K ? W.d : W.m + row0 * nb, int64_t(wrows) * nb * 2),
                               rad = rsrc_of(A.d + t0 * nb, int64_t(arows) * nb * 4),
                               rbs = rsrc_of(A.bsums + t0 * nb * 16, int64_t(arows) * nb * 32);
  const uint32_t srow = uint32_t(lane) * uint32_t(nb), brow = uint32_t(lane >> 1) * uint32_t(nb) * 32 + 16 * (lane & 1);
  struct Share {
    u32x4_t v;      // waves 0 and 2
    uint16_t d, m;  // wave 1
    uint32_t a;     // wave 3
  };
  auto load_share = [&](int sb, Share& sh) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    if (wave == 0) {
      sh.v = __builtin_amdgcn_raw_buffer_load_b128(rs, srow * 16, sb * 16, 0);
    } else if (wave == 1) {
      sh.d = __builtin_amdgcn_raw_buffer_load_b16(rd, srow * 2, sb * 2, 0);
      if constexpr (T != kQ6_K) sh.m = __builtin_amdgcn_raw_buffer_load_b16(rm, srow * 2, sb * 2, 0);
    } else if (wave == 2) {
      if constexpr (T != kQ6_K) sh.v = __builtin_amdgcn_raw_buffer_load_b128(rbs, brow, sb * 32, 0);
    } else {
      sh.a = __builtin_amdgcn_raw_buffer_load_b32(rad, srow * 4, sb * 4, 0);
    }
#endif
  };
  constexpr int kShareLoads = T == kQ6_K ? 0 : 1;  // at least, of any wave
  auto store_share = [&](int p, Share& sh) __attribute__((always_inline)) {
    // the loads are waited for here, on every path: one left pending on the paths around a branch would make the
    // next reuse of its register wait for all loads in flight
    asm volatile("" : "+v"(sh.v), "+v"(sh.d), "+v"(sh.m), "+v"(sh.a));
    if (wave == 0) {
      scales[p][lane] = sh.v;
    } else if (wave == 1) {
      wd[p][lane] = h2f(sh.d);
      if constexpr (T != kQ6_K) wm[p][lane] = h2f(sh.m);
    } else if (wave == 2) {
      if constexpr (T != kQ6_K) reinterpret_cast<u32x4_t*>(&digits[p][0][0])[lane] = sh.v;
    } else if (lane < AR) {
      ad[p][lane] = __builtin_bit_cast(float, sh.a);
    }
  };
  const int r0 = 16 * wave, ra_ = r0 + ml;  // this wave's weight rows, and the row of this lane's A operand
  // sums[w][j][v]: weight row r0 + 4 kg + v, activation row 16 j + ml (the MFMA's result layout)
  float sums[8][WN][4], acc[WN][4], dv[WN][4];
#pragma unroll
  for (int j = 0; j < WN; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      acc[j][v] = 0.f;
#pragma unroll
      for (int w = 0; w < 8; ++w) sums[w][j][v] = 0.f;
    }
  uint32_t boff[4];  // this lane's activation fragment of residue 4 half + wl, within the first 16 rows
#pragma unroll
  for (int wl = 0; wl < 4; ++wl) boff[wl] = uint32_t(ml * 256 + 16 * ((4 * wl + kg) ^ ml));
  const int nt = 2 * nb;
  Share cur{};
  load_share(0, cur);
  store_share(0, cur);
  fetch_quants(0, std::integral_constant<int, 0>{});
  fetch(0, std::integral_constant<int, 0>{});
  fetch(1, std::integral_constant<int, 1>{});
  uint32_t sw[2];  // k_scale_words of this lane's row
  auto step = [&](int t, auto m_c) __attribute__((always_inline)) {  // m: t % 12
    constexpr int m = decltype(m_c)::value, half = m & 1, p = (m >> 1) & 1;
    const int sb = t >> 1;
    // Every wave's loads of stage t and its LDS stores; the barrier publishes both and certifies that every wave is
    // done with stage t - 1. In flight stay, at half 0, stage t + 1's loads; at half 1 the small planes', the quants'
    // and stage t + 1's, which half 0 issued after stage t's.
    __builtin_amdgcn_s_waitcnt(vm_lds_wait(half == 0 ? kALoads : kShareLoads + kQLoads + kALoads));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if constexpr (half == 0) {  // past the end: the last super-block and stage again
      load_share(sb + 1 < nb ? sb + 1 : sb, cur);
      fetch_quants(sb + 1 < nb ? sb + 1 : sb, std::integral_constant<int, p ^ 1>{});
    }
    fetch(t + 2 < nt ? t + 2 : nt - 1, std::integral_constant<int, m + 2>{});
    const uint8_t* const base = ring(m_c);
    const uint8_t* const qbase = quants(std::integral_constant<int, p>{});
    if constexpr (half == 0) {
      float da[WN];
#pragma unroll
      for (int j = 0; j < WN; ++j) da[j] = ad[p][16 * j + ml];
      const u32x4_t sc = scales[p][ra_];
      k_scale_words<T>(sc, kg, sw);
      const floatx4_t dw = *reinterpret_cast<const floatx4_t*>(&wd[p][r0 + 4 * kg]);
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) dv[j][v] = __fmul_rn(dw[v], da[j]);
      if constexpr (T != kQ6_K) {
        const half4_t am = k_min_operand(sc, kg);
        const floatx4_t dm = *reinterpret_cast<const floatx4_t*>(&wm[p][r0 + 4 * kg]);
#pragma unroll
        for (int j = 0; j < WN; ++j) {
          const floatx4_t sumi =
              __builtin_amdgcn_mfma_f32_16x16x16f16(am, digits[p][16 * j + ml][kg], floatx4_t{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
          for (int v = 0; v < 4; ++v)
            acc[j][v] = opaque(__fsub_rn(acc[j][v], __fmul_rn(__fmul_rn(dm[v], da[j]), sumi[v])));
        }
      }
    }
    // the lane's raw words of the four residues, and its sub-blocks' constants
    u32x4_t q0, q1, h;
    KScales<T> ks;
    ks.set(sw[0], sw[1]);
    auto chunk = [&](int c) {
      return *reinterpret_cast<const u32x4_t*>(qbase + ra_ * 128 + 16 * ((2 * c + half) ^ ((ra_ >> 1) & 7)));
    };
    const uint8_t* const hbase = qbase + 64 * 128 + ra_ * HB;
    if constexpr (T == kQ6_K) {
      q0 = chunk(2 * (kg >> 1));
      q1 = chunk(2 * (kg >> 1) + 1);
      h = *reinterpret_cast<const u32x4_t*>(hbase + 16 * ((2 * (kg >> 1) + half) ^ ((ra_ >> 2) & 3)));
    } else {
      q0 = chunk(kg);
      if constexpr (T == kQ5_K) h = *reinterpret_cast<const u32x4_t*>(hbase + 16 * (half ^ ((ra_ >> 3) & 1)));
    }
    // Residue wl's sums are added while the MFMAs of wl + 1 run and the fragments of wl + 2 are read.
    half8_t b[2][WN];
    floatx4_t c[2][WN];
    auto load_b = [&](int wl) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < WN; ++j) b[wl & 1][j] = *reinterpret_cast<const half8_t*>(base + boff[wl] + j * 4096);
    };
    auto multiply = [&](int wl) __attribute__((always_inline)) {
      half8_t a[NS];
      k_operand<T>(q0[wl], T == kQ6_K ? q1[wl] : 0u, HB ? h[wl] : 0u, kg, ks, a);
#pragma unroll
      for (int j = 0; j < WN; ++j) {
        c[wl & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[0], b[wl & 1][j], floatx4_t{0, 0, 0, 0}, 0, 0, 0);
        if constexpr (NS == 2)
          c[wl & 1][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[NS - 1], b[wl & 1][j], c[wl & 1][j], 0, 0, 0);
      }
    };
    load_b(0);
    load_b(1);
    multiply(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int wl = 0; wl < 4; ++wl) {
      if (wl < 3) multiply(wl + 1);
      if (wl < 2) load_b(wl + 2);
      constexpr int w0 = 4 * half;
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v)  // (opaque: added here, not later)
          sums[w0 + wl][j][v] = opaque(__fadd_rn(sums[w0 + wl][j][v], __fmul_rn(dv[j][v], c[wl & 1][j][v])));
      __builtin_amdgcn_sched_barrier(0);
    }
    // the next super-block's small planes (this parity's last readers passed the barrier before this super-block)
    if constexpr (half == 1) store_share(p ^ 1, cur);
  };
  auto pair = [&](int t, auto m_c) __attribute__((always_inline)) {  // a super-block; false: it was the last
    constexpr int m = decltype(m_c)::value;
    step(t, std::integral_constant<int, m>{});
    step(t + 1, std::integral_constant<int, m + 1>{});
    return t + 2 < nt;
  };
  for (int t = 0;; t += 12) {  // six super-blocks: every stage and parity a compile-time constant
    if (!pair(t, std::integral_constant<int, 0>{}) || !pair(t + 2, std::integral_constant<int, 2>{}) ||
        !pair(t + 4, std::integral_constant<int, 4>{}) || !pair(t + 6, std::integral_constant<int, 6>{}) ||
        !pair(t + 8, std::integral_constant<int, 8>{}) || !pair(t + 10, std::integral_constant<int, 10>{}))
      break;
  }
  __builtin_amdgcn_s_waitcnt(vm_lds_wait(0));  // no load may land in LDS after the workgroup's end
  const bool vec = W.rows % 4 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0;
  const int64_t r = row0 + r0 + 4 * kg;
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int64_t t = t0 + 16 * j + ml;
    floatx4_t o;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      o[v] = acc[j][v];
#pragma unroll
      for (int w = 0; w < 8; ++w) o[v] = __fadd_rn(o[v], sums[w][j][v]);
    }
    if (t < n) {
      if (vec && r < W.rows) {
        *reinterpret_cast<floatx4_t*>(y + t * W.rows + r) = o;
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (r + v < W.rows) y[t * W.rows + r + v] = o[v];
      }
    }
  }
}

// qgemm_k_small_kernel: the K types for calls of few activation rows, where 64-row weight tiles leave most CUs
// idle and each workgroup would walk every super-block alone. A workgroup takes 16 weight rows x 32 activation
// rows and its 4 waves split the super-blocks (wave w: w, w + 4, ...): each computes its super-block's float terms
// - d * aux[l] for the eight lanes and, for Q4_K / Q5_K, the minimum term, with the operands and expressions of
// qgemm_k_kernel, its operands read straight from global memory - and writes them to LDS; per round
// of four super-blocks the 256 threads, two outputs each, add them to their running sums in super-block order:
// the reference's order, so the same bits.
template <int T>
__global__ __launch_bounds__(256) void qgemm_k_small_kernel(QGemmBatch B, QA A, int64_t n) {
  static_assert(T == kQ4_K || T == kQ5_K || T == kQ6_K, "K types");
  constexpr int NS = k_slices<T>();
  constexpr int NTM = T == kQ6_K ? 8 : 9;  // float terms per output and super-block
  __shared__ float terms[4][NTM][16][33];  // [wave][term][weight row][activation row], one column of padding
  __shared__ __align__(16) float rowd[4][16], rowm[4][16];  // per wave: d, dmin of its super-block's 16 rows
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ml = lane & 15, kg = lane >> 4;
  int wi = 0;
  for (int i = 1; i < B.n_w; ++i)
    if (int(blockIdx.x) >= B.tile0[i]) wi = i;
  const QW W = B.w[wi];
  float* __restrict__ y = B.y[wi];
  const int64_t row0 = int64_t(int(blockIdx.x) - B.tile0[wi]) * 16, t0 = int64_t(blockIdx.y) * 32;
  // owner sums: outputs (weight row tid & 15, activation rows (tid >> 4) and (tid >> 4) + 16)
  float sums[2][8], acc[2];
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    acc[o] = 0.f;
#pragma unroll
    for (int l = 0; l < 8; ++l) sums[o][l] = 0.f;
  }
  const int64_t ra = min(row0 + ml, W.rows - 1);  // this lane's operand row
  for (int64_t s0 = 0; s0 < W.nb; s0 += 4) {
    const int64_t sb = s0 + wave;
    const bool has = sb < W.nb;
    const int64_t sbc = has ? sb : W.nb - 1;
    const int64_t wb = ra * W.nb + sbc;
    const u32x4_t sc = *reinterpret_cast<const u32x4_t*>(W.s + wb * 16);
    uint32_t sw[2];
    // the lane's operand words: its row's quant words of its k group (and their high bits), every residue
    u32x4_t qv[T == kQ6_K ? 4 : 2], hv[2];
    if constexpr (T == kQ6_K) {
      const u32x4_t* q = reinterpret_cast<const u32x4_t*>(W.q + wb * 128 + 64 * (kg >> 1));
#pragma unroll
      for (int i = 0; i < 4; ++i) qv[i] = q[i];
      const u32x4_t* h = reinterpret_cast<const u32x4_t*>(W.h + wb * 64 + 32 * (kg >> 1));
      hv[0] = h[0], hv[1] = h[1];
    } else {
      const u32x4_t* q = reinterpret_cast<const u32x4_t*>(W.q + wb * 128 + 32 * kg);
      qv[0] = q[0], qv[1] = q[1];
      if constexpr (T == kQ5_K) {
        const u32x4_t* h = reinterpret_cast<const u32x4_t*>(W.h + wb * 32);
        hv[0] = h[0], hv[1] = h[1];
      }
    }
    half8_t bw[2][8];
    float da[2];
    half4_t bs[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t ab = min(t0 + 16 * j + ml, n - 1) * A.nb + sbc;
      const half8_t* aq = reinterpret_cast<const half8_t*>(A.qs + ab * 512);
#pragma unroll
      for (int w = 0; w < 8; ++w) bw[j][w] = aq[4 * w + kg];
      da[j] = A.d[ab];
      if constexpr (T != kQ6_K) bs[j] = reinterpret_cast<const half4_t*>(A.bsums)[ab * 4 + kg];
    }
    const float d1 = h2f(W.d[wb]), m1 = T == kQ6_K ? 0.f : h2f(W.m[wb]);
    k_scale_words<T>(sc, kg, sw);
    if (kg == 0) rowd[wave][ml] = d1, rowm[wave][ml] = m1;
    __syncthreads();  // this round's row values are in LDS
    if (has) {
      const floatx4_t dw = *reinterpret_cast<const floatx4_t*>(&rowd[wave][4 * kg]);
      float dv[2][4];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) dv[j][v] = __fmul_rn(dw[v], da[j]);
      KScales<T> ks;
      ks.set(sw[0], sw[1]);
#pragma unroll
      for (int w = 0; w < 8; ++w) {
        half8_t a[NS];
        if constexpr (T == kQ6_K)
          k_operand<T>(qv[w >> 2][w & 3], qv[2 + (w >> 2)][w & 3], hv[w >> 2][w & 3], kg, ks, a);
        else
          k_operand<T>(qv[w >> 2][w & 3], 0u, T == kQ5_K ? hv[w >> 2][w & 3] : 0u, kg, ks, a);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          floatx4_t c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[0], bw[j][w], floatx4_t{0, 0, 0, 0}, 0, 0, 0);
          if constexpr (NS == 2) c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[NS - 1], bw[j][w], c, 0, 0, 0);
#pragma unroll
          for (int v = 0; v < 4; ++v) terms[wave][w][4 * kg + v][16 * j + ml] = __fmul_rn(dv[j][v], c[v]);
        }
      }
      if constexpr (T != kQ6_K) {
        const half4_t am = k_min_operand(sc, kg);
        const floatx4_t dm = *reinterpret_cast<const floatx4_t*>(&rowm[wave][4 * kg]);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const floatx4_t sumi = __builtin_amdgcn_mfma_f32_16x16x16f16(am, bs[j], floatx4_t{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
          for (int v = 0; v < 4; ++v)
            terms[wave][NTM - 1][4 * kg + v][16 * j + ml] = __fmul_rn(__fmul_rn(dm[v], da[j]), sumi[v]);
        }
      }
    }
    __syncthreads();  // every wave's terms are in LDS
    const int orow = tid & 15;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (s0 + s < W.nb) {
#pragma unroll
        for (int o = 0; o < 2; ++o) {
          const int ot = (tid >> 4) + 16 * o;
#pragma unroll
          for (int l = 0; l < 8; ++l) sums[o][l] = __fadd_rn(sums[o][l], terms[s][l][orow][ot]);
          if constexpr (T != kQ6_K) acc[o] = __fsub_rn(acc[o], terms[s][NTM - 1][orow][ot]);
        }
      }
    }
    __syncthreads();  // the terms are consumed before the next round overwrites them
  }
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    float r = acc[o];
#pragma unroll
    for (int l = 0; l < 8; ++l) r = __fadd_rn(r, sums[o][l]);
    const int64_t row = row0 + (tid & 15), t = t0 + (tid >> 4) + 16 * o;
    if (row < W.rows && t < n) y[t * W.rows + row] = r;
  }
}

// The small-call K kernel runs while 64 x 32 tiles would give fewer than kKSmallMaxWgs workgroups (QKV shape, 48 such
// row tiles, K = 2048: Q4_K at 32 rows 10.8 us against 12.9, at 64 rows 13.9 against 12.3; 32 row tiles, K = 8192:
// Q6_K at 64 rows 39.7 against 43.9, at 128 rows 62 against 44.7).
constexpr int64_t kKSmallMaxWgs = 80;
template <int T>
hipError_t launch_k(bool small, unsigned tiles, hipStream_t s, const QGemmBatch& B, const QA& A, int64_t n) {
  const dim3 grid{tiles, unsigned((n + 31) / 32)};
  if (small) return nbhs_timing::launch(NBHS_K_QGEMM, qgemm_k_small_kernel<T>, grid, dim3(256), s, B, A, n);
  return nbhs_timing::launch(NBHS_K_QGEMM, qgemm_k_kernel<T>, grid, dim3(256), s, B, A, n);
}

// ---- dequantization (quant.cpp:157-242), four output elements per thread ----

// The ids of a call that fit a kernel argument travel in it: no copy to the device, no wait for the stream.
struct EmbedIds {
  int32_t id[NBHS_EMBED_ARG_IDS];
};

// Elements e .. e + 3 (e % 4 == 0) of block wb of the weight: the reference's expression for each.
template <int T>
__device__ __forceinline__ floatx4_t dequant_four(const QW& W, int64_t wb, int e) {
  const float d = h2f(W.d[wb]);
  floatx4_t v;
  if constexpr (T == kQ8_0 || T == kQ4_0 || T == kQ5_0 || T == kQ5_1) {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(W.q + (T == kQ8_0 ? wb * 32 + e : wb * 16 + (e & 15)));
    uint32_t h = 0;
    if constexpr (T == kQ5_0 || T == kQ5_1) h = reinterpret_cast<const uint32_t*>(W.h)[wb] >> e;
    float m = 0.f;
    if constexpr (T == kQ5_1) m = h2f(W.m[wb]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (T == kQ8_0) {
        v[j] = __fmul_rn(float(int8_t(w >> (8 * j))), d);
      } else {
        int q = (w >> (8 * j + (e < 16 ? 0 : 4))) & 0x0F;
        if constexpr (T != kQ4_0) q |= ((h >> j) & 1u) << 4;
        v[j] = T == kQ5_1 ? __fadd_rn(__fmul_rn(float(q), d), m) : __fmul_rn(float(q - (T == kQ4_0 ? 8 : 16)), d);
      }
    }
  } else {
    // byte i of words w .. w + 3 of sub-block k's residue-ordered group
    const int k = e >> 5, w = e & 7, i = (e >> 3) & 3;
    if constexpr (T == kQ4_K || T == kQ5_K) {
      int sc, mn;
      scale_min_k4(k, W.s + wb * 16, sc, mn);
      const u32x4_t qw = *reinterpret_cast<const u32x4_t*>(W.q + wb * 128 + 32 * (k >> 1) + 4 * w);
      u32x4_t hw;
      if constexpr (T == kQ5_K) hw = *reinterpret_cast<const u32x4_t*>(W.h + wb * 32 + 4 * w);
      const float ds = __fmul_rn(d, float(sc)), ms = __fmul_rn(h2f(W.m[wb]), float(mn));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        int q = (qw[j] >> (8 * i + 4 * (k & 1))) & 0xF;
        if constexpr (T == kQ5_K) q += ((hw[j] >> (8 * i + k)) & 1) ? 16 : 0;
        v[j] = __fsub_rn(__fmul_rn(ds, float(q)), ms);
      }
    } else {  // Q6_K
      const int h = k >> 2, g = k & 3;
      const u32x4_t qw = *reinterpret_cast<const u32x4_t*>(W.q + wb * 128 + 64 * h + 32 * (g & 1) + 4 * w);
      const u32x4_t hw = *reinterpret_cast<const u32x4_t*>(W.h + wb * 64 + 32 * h + 4 * w);
      const float ds = __fmul_rn(d, float(reinterpret_cast<const int8_t*>(W.s)[wb * 16 + (e >> 4)]));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int q = int(((qw[j] >> (8 * i + 4 * (g >> 1))) & 0xF) | (((hw[j] >> (8 * i + 2 * g)) & 3) << 4)) - 32;
        v[j] = __fmul_rn(ds, float(q));
      }
    }
  }
  return v;
}

// Row blockIdx.y's elements, four a thread: word loads and 16-byte stores, a block's scales once. us for one row of Q6_K,
// K = 2048, 5 (with a thread per block, eight threads of 256 dependent loads and stores each, 40); 4096 rows, K = 4096, Q8_0
// 27, Q4_K 31, Q6_K 29 (with a thread per element 44, 58 and 54).
template <int T>
__global__ __launch_bounds__(256) void dequant_rows_kernel(QW W, EmbedIds ids, const int32_t* __restrict__ far_ids,
                                                           int64_t row0, float* __restrict__ out, int vec) {
  constexpr int be = int(block_elems(T));
  const int64_t in = W.nb * be, i = 4 * (int64_t(blockIdx.x) * 256 + threadIdx.x), t = row0 + blockIdx.y;
  if (i >= in) return;
  const int64_t id = far_ids ? far_ids[t] : ids.id[blockIdx.y], wb = id * W.nb + i / be;
  const floatx4_t v = dequant_four<T>(W, wb, int(i % be));
  float* const o = out + t * in + i;
  if (vec) {
    *reinterpret_cast<floatx4_t*>(o) = v;
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = v[j];
  }
}

QW weight_of(int type, const void* w, int64_t rows, int64_t in) {
  const int64_t nb = in / block_elems(type);
  const WeightLayout l = weight_layout(type, rows, nb);
  const uint8_t* base = static_cast<const uint8_t*>(w);
  return QW{base + l.q_off, base + l.h_off, base + l.s_off, reinterpret_cast<const uint16_t*>(base + l.d_off),
            reinterpret_cast<const uint16_t*>(base + l.m_off), rows, nb};
}

// How a call is laid over kgemv_kernel's grid: passes in flight per wave and batches of rows per wave. All workgroups run
// at once, 1 to as many on a CU as its registers and LDS hold, and the fullest CU sets the time: its workgroups times the
// rows a wave of theirs takes (batches x rows of a batch, and half a row for quantizing the activations). Few waves on a
// SIMD and few passes in flight hide less latency; the factors are fitted to 600 calls (2-56 super-blocks, 5120-151936
// rows, 1-4 activation rows) in each of the layouts, which come out 1.2 % from the best one on average. Against a layout by
// a number of waves (4096, with as many batches as fill them), whose grid may end in a second round of a few workgroups, us
// a call: 14336 rows, K = 2048, two activation rows, Q4_K 17.0 -> 13.1; 28672 rows, K = 4096, Q5_K, one 29.6 -> 23.6, two
// 40.3 -> 34.7; Q4_K, four 60.2 -> 51.2; 16384 rows, K = 2048, one, Q6_K 11.7 -> 11.7. Not caught: 131072 rows of 2
// super-blocks, four rows, Q6_K 42.0 -> 44.6, where a second round of short workgroups overlaps the first.
constexpr int64_t kCUs = 256;
struct KGemvPlan {
  int passes = 0;
  int64_t batches = 0;
  double cost = 0;
};

// Workgroups of NT, P on a CU.
template <int T, int NT, int P>
int kgemv_resident() {
  static const int v = [] {
    int b = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, kgemv_kernel<T, NT, P>, 256, 0);
    return e == hipSuccess ? std::clamp(b, 1, 4) : 1;
  }();
  return v;
}

template <int T, int NT, int P>
void plan_kgemv(const int64_t* rows, int n_w, int64_t nb, KGemvPlan& best) {
  const int64_t rp = kGemvChunk / std::min<int64_t>(nb, kGemvChunk), rb = std::min<int64_t>(P * rp, 8);
  if (P > 1 && P * rp > 8) return;
  auto wgs_of = [&](int64_t batches) {
    int64_t wgs = 0;
    for (int i = 0; i < n_w; ++i) wgs += (rows[i] + 4 * rb * batches - 1) / (4 * rb * batches);
    return wgs;
  };
  int64_t total = 0;
  for (int i = 0; i < n_w; ++i) total += rows[i];
  constexpr double kWaves[] = {0, 1.7, 1.15, 1.075, 1}, kPasses = P == 4 ? 1 : P == 2 ? 1.1 : 1.4;
  int64_t last = 0;
  for (int w = kgemv_resident<T, NT, P>(); w >= 1; --w) {
    int64_t batches = std::max<int64_t>(1, (total + rb * 4 * kCUs * w - 1) / (rb * 4 * kCUs * w));
    if (batches == last) continue;  // the same layout
    int64_t wgs = wgs_of(batches);
    while (wgs > kCUs * w) wgs = wgs_of(++batches);  // (a partial last workgroup of each weight)
    last = batches;
    const int64_t per_cu = (wgs + kCUs - 1) / kCUs;
    const double cost = double(per_cu) * (double(batches * rb) + 0.5) * kWaves[per_cu] * kPasses;
    if (best.passes == 0 || cost < best.cost) best = KGemvPlan{P, batches, cost};
  }
}

template <int T, int NT>
int launch_kgemv(const QBatch& B, const int64_t* rows, int n_w, const float* x, int64_t in, int64_t n, hipStream_t s) {
  const int64_t nb = in / 256, rp = kGemvChunk / std::min<int64_t>(nb, kGemvChunk);
  KGemvPlan plan;
  plan_kgemv<T, NT, 4>(rows, n_w, nb, plan);
  plan_kgemv<T, NT, 2>(rows, n_w, nb, plan);
  plan_kgemv<T, NT, 1>(rows, n_w, nb, plan);
  if (plan.batches > INT32_MAX) return NBHS_EINVAL;
  const int64_t wg_rows = 4 * std::min<int64_t>(plan.passes * rp, 8) * plan.batches;
  QBatch b = B;
  int64_t wgs = 0;
  for (int i = 0; i < n_w; ++i) b.wave0[i] = wgs, wgs += (rows[i] + wg_rows - 1) / wg_rows;
  const dim3 grid{unsigned(wgs), 1, 1}, block{256, 1, 1};
  auto go = [&](auto kernel) {
    return nbhs_timing::launch(NBHS_K_QGEMV, kernel, grid, block, s, b, x, in, int(n), int(plan.batches));
  };
  return plan.passes == 4   ? go(kgemv_kernel<T, NT, 4>)
         : plan.passes == 2 ? go(kgemv_kernel<T, NT, 2>)
                            : go(kgemv_kernel<T, NT, 1>);
}

template <int T>
int launch_gemv(const QBatch& B, const int64_t* rows, int n_w, const QA& A, const float* x, int64_t in, int64_t n,
                bool fused, hipStream_t s) {
  int64_t total = 0;
  for (int i = 0; i < n_w; ++i) total += rows[i];
  if constexpr (is_k(T)) {
    if (fused && in / 256 <= kgemv_max_sb(int(n)))
      return n == 1   ? launch_kgemv<T, 1>(B, rows, n_w, x, in, n, s)
             : n == 2 ? launch_kgemv<T, 2>(B, rows, n_w, x, in, n, s)
                      : launch_kgemv<T, 4>(B, rows, n_w, x, in, n, s);
  }
  const bool wide = fused && n == 1 && total >= kWideRows;
  const int rw = rows_per_wave(is_k(T), fused ? (n == 1 ? 1 : 4) : (n <= 4 ? 4 : 16), wide);
  QBatch b = B;
  int64_t waves = 0;
  for (int i = 0; i < n_w; ++i) b.wave0[i] = waves, waves += (rows[i] + rw - 1) / rw;
  if (waves >= (int64_t(1) << 31)) return NBHS_EINVAL;
  const dim3 grid{unsigned(waves), 1, 1}, block{64, 1, 1};
  if (fused) {
    if (wide)
      return nbhs_timing::launch(NBHS_K_QGEMV, qgemv_kernel<T, 1, true, true>, grid, block, s, b, A, x, in, int(n));
    if (n == 1)
      return nbhs_timing::launch(NBHS_K_QGEMV, qgemv_kernel<T, 1, true, false>, grid, block, s, b, A, x, in, int(n));
    return nbhs_timing::launch(NBHS_K_QGEMV, qgemv_kernel<T, 4, true, false>, grid, block, s, b, A, x, in, int(n));
  }
  if (n <= 4)
    return nbhs_timing::launch(NBHS_K_QGEMV, qgemv_kernel<T, 4, false, false>, grid, block, s, b, A, x, in, int(n));
  return nbhs_timing::launch(NBHS_K_QGEMV, qgemv_kernel<T, 16, false, false>, grid, block, s, b, A, x, in, int(n));
}

// ids: host_ids, at most NBHS_EMBED_ARG_IDS, or device memory.
template <int T>
int launch_dequant(const QW& W, const int32_t* host_ids, const int32_t* ids, int64_t n, float* out, hipStream_t s) {
  const int64_t in = W.nb * block_elems(T);
  const int vec = reinterpret_cast<uintptr_t>(out) % 16 == 0 ? 1 : 0;  // (a row is whole blocks: multiples of 32 floats)
  EmbedIds arg{};
  if (host_ids) std::copy(host_ids, host_ids + n, arg.id);
  for (int64_t t0 = 0; t0 < n; t0 += 65535) {
    const dim3 grid{unsigned((in + 1023) / 1024), unsigned(std::min<int64_t>(n - t0, 65535))};
    const hipError_t e = nbhs_timing::launch(NBHS_K_ELEMENTWISE, dequant_rows_kernel<T>, grid, dim3(256), s, W, arg,
                                             host_ids ? nullptr : ids, t0, out, vec);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

int dequant_rows(int type, const void* w, int64_t rows, int64_t in, const int32_t* host_ids, const int32_t* ids, int64_t n,
                 float* out, nbhs_stream stream) {
  if (!is_quant(type) || !w || !out || rows <= 0 || in <= 0 || in % block_elems(type) || n <= 0 ||
      (in + 255) / 256 >= (int64_t(1) << 31))
    return NBHS_EINVAL;
  const QW W = weight_of(type, w, rows, in);
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (type) {
    case kQ4_0: return launch_dequant<kQ4_0>(W, host_ids, ids, n, out, s);
    case kQ5_0: return launch_dequant<kQ5_0>(W, host_ids, ids, n, out, s);
    case kQ5_1: return launch_dequant<kQ5_1>(W, host_ids, ids, n, out, s);
    case kQ8_0: return launch_dequant<kQ8_0>(W, host_ids, ids, n, out, s);
    case kQ4_K: return launch_dequant<kQ4_K>(W, host_ids, ids, n, out, s);
    case kQ5_K: return launch_dequant<kQ5_K>(W, host_ids, ids, n, out, s);
    case kQ6_K: return launch_dequant<kQ6_K>(W, host_ids, ids, n, out, s);
    default: return NBHS_EINVAL;
  }
}

int qgemm_multi(int type, int n_w, const void* const* w, const int64_t* rows, float* const* y, int64_t in, const void* acts,
                int64_t n, nbhs_stream stream) {
  if (!is_quant(type) || n_w <= 0 || n_w > kMaxQWeights || !w || !rows || !y || !acts ||
      in <= 0 || in % block_elems(type) || n <= 0 || (n + 31) / 32 > 65535)
    return NBHS_EINVAL;
  // weight-row tiles of every weight at 64 rows (each weight's tiles start at its tile0 in grid x) and, for the
  // legacy types' smallest launches, at 32
  QGemmBatch B{};
  int64_t tiles64 = 0, tiles32 = 0;
  for (int i = 0; i < n_w; ++i) {
    if (!w[i] || !y[i] || rows[i] <= 0) return NBHS_EINVAL;
    B.w[i] = weight_of(type, w[i], rows[i], in);
    B.y[i] = y[i];
    tiles64 += (rows[i] + 63) / 64;
    tiles32 += (rows[i] + 31) / 32;
    if ((tiles32 + 1) * 2 >= (int64_t(1) << 31)) return NBHS_EINVAL;  // 16-row tiles fit too
  }
  B.n_w = n_w;
  LegacyTile tile = kTile64x64;
  if (!is_k(type)) {
    if (tiles64 * ((n + 63) / 64) >= kLegacyMinWgs && n > 32)
      tile = kTile64x64;
    else if (tiles64 * ((n + 31) / 32) >= kLegacyMinWgs)
      tile = kTile64x32;
    else
      tile = kTile32x32;
  }
  // K types: the small-call kernel (16-row weight tiles, super-blocks split over the waves) when 64-row tiles
  // would give fewer than kKSmallMaxWgs workgroups, or a row is too long for the tiled kernel's 32-bit offsets
  const bool small = is_k(type) && (tiles64 * ((n + 31) / 32) < kKSmallMaxWgs || in >= (int64_t(1) << 24));
  const int64_t tile_rows = small ? 16 : tile == kTile32x32 ? 32 : 64;
  int64_t tiles = 0;
  for (int i = 0; i < n_w; ++i) {
    B.tile0[i] = int(tiles);
    tiles += (rows[i] + tile_rows - 1) / tile_rows;
  }
  const int act = is_k(type) ? int(kActQ8_K16) : act_of(type);
  const ActLayout l = act_layout(act, n, B.w[0].nb);
  const uint8_t* base = static_cast<const uint8_t*>(acts);
  const QA A{reinterpret_cast<const int8_t*>(base + l.qs_off), reinterpret_cast<const float*>(base + l.d_off),
             act == kActQ8_1 ? reinterpret_cast<const float*>(base + l.s_off) : nullptr,
             act == kActQ8_K16 ? reinterpret_cast<const int16_t*>(base + l.bsums_off) : nullptr, B.w[0].nb};
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (type) {
    case kQ4_K: return launch_k<kQ4_K>(small, unsigned(tiles), s, B, A, n);
    case kQ5_K: return launch_k<kQ5_K>(small, unsigned(tiles), s, B, A, n);
    case kQ6_K: return launch_k<kQ6_K>(small, unsigned(tiles), s, B, A, n);
    case kQ4_0: return launch_legacy<kQ4_0>(tile, unsigned(tiles), n, s, B, A);
    case kQ5_0: return launch_legacy<kQ5_0>(tile, unsigned(tiles), n, s, B, A);
    case kQ5_1: return launch_legacy<kQ5_1>(tile, unsigned(tiles), n, s, B, A);
    case kQ8_0: return launch_legacy<kQ8_0>(tile, unsigned(tiles), n, s, B, A);
    default: return NBHS_EINVAL;
  }
}

}  // namespace

extern "C" {

int64_t nbhs_quant_weight_bytes(int type, int64_t rows, int64_t in) {
  if (!is_quant(type) || rows <= 0 || in <= 0 || in % block_elems(type)) return -1;
  return weight_layout(type, rows, in / block_elems(type)).bytes;
}

int64_t nbhs_quant_act_bytes(int type, int64_t n, int64_t in) {
  if (!is_quant(type) || n <= 0 || in <= 0 || in % block_elems(type)) return -1;
  return act_layout(act_of(type), n, in / block_elems(type)).bytes;
}

int64_t nbhs_quant_act_k16_bytes(int type, int64_t n, int64_t in) {
  if (!is_k(type) || n <= 0 || in <= 0 || in % 256) return -1;
  return act_layout(kActQ8_K16, n, in / 256).bytes;
}

int nbhs_quantize_acts(int type, const float* x, int64_t n, int64_t in, void* acts, nbhs_stream stream) {
  if (!is_quant(type) || !x || !acts || n <= 0 || in <= 0 || in % block_elems(type)) return NBHS_EINVAL;
  const int act = act_of(type);
  const int64_t nb = in / block_elems(type), blocks = n * nb;
  const ActLayout l = act_layout(act, n, nb);
  uint8_t* base = static_cast<uint8_t*>(acts);
  int8_t* qs = reinterpret_cast<int8_t*>(base + l.qs_off);
  float* d = reinterpret_cast<float*>(base + l.d_off);
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (act == kActQ8_K) {
    if (blocks >= (int64_t(1) << 31)) return NBHS_EINVAL;
    return nbhs_timing::launch(NBHS_K_QUANTIZE, quantize_q8k_kernel<false>, dim3(unsigned(blocks)), dim3(64), s, x, in,
                               qs, d, reinterpret_cast<int16_t*>(base + l.bsums_off));
  }
  const dim3 grid{unsigned((blocks + 255) / 256), 1, 1};
  if (act == kActQ8_1)
    return nbhs_timing::launch(NBHS_K_QUANTIZE, quantize_q8_kernel<true>, grid, dim3(256), s, x, in, n, qs, d,
                               reinterpret_cast<float*>(base + l.s_off));
  return nbhs_timing::launch(NBHS_K_QUANTIZE, quantize_q8_kernel<false>, grid, dim3(256), s, x, in, n, qs, d,
                             static_cast<float*>(nullptr));
}

int nbhs_quantize_acts_rm(int, const float*, int64_t, int64_t, void*, nbhs_stream) { return NBHS_EINVAL; }

int nbhs_quantize_acts_k16(int type, const float* x, int64_t n, int64_t in, void* acts, int64_t acts_bytes,
                           nbhs_stream stream) {
  const int64_t need = nbhs_quant_act_k16_bytes(type, n, in);
  if (need < 0 || acts_bytes < need || !x || !acts) return NBHS_EINVAL;
  const int64_t nb = in / 256, blocks = n * nb;
  if (blocks >= (int64_t(1) << 31)) return NBHS_EINVAL;
  const ActLayout l = act_layout(kActQ8_K16, n, nb);
  uint8_t* base = static_cast<uint8_t*>(acts);
  return nbhs_timing::launch(NBHS_K_QUANTIZE, quantize_q8k_kernel<true>, dim3(unsigned(blocks)), dim3(64),
                             reinterpret_cast<hipStream_t>(stream), x, in, reinterpret_cast<int8_t*>(base + l.qs_off),
                             reinterpret_cast<float*>(base + l.d_off), reinterpret_cast<int16_t*>(base + l.bsums_off));
}

int nbhs_qgemv_multi(int type, int n_w, const void* const* w, const int64_t* rows, float* const* y, int64_t in,
                     const float* x, const void* acts, int64_t n_acts, int64_t t0, int64_t n, nbhs_stream stream) {
  if (!is_quant(type) || n_w <= 0 || n_w > kMaxQWeights || !w || !rows || !y || in <= 0 ||
      in % block_elems(type) || n <= 0 || n > NBHS_GEMV_MAX_ROWS)
    return NBHS_EINVAL;
  const bool fused = acts == nullptr;
  if (fused ? (!x || n > 4 || t0 != 0 || reinterpret_cast<uintptr_t>(x) % 16 || in % 4) : (t0 < 0 || t0 + n > n_acts))
    return NBHS_EINVAL;
  QBatch B{};
  for (int i = 0; i < n_w; ++i) {
    if (!w[i] || !y[i] || rows[i] <= 0) return NBHS_EINVAL;
    B.w[i] = weight_of(type, w[i], rows[i], in);
    B.y[i] = y[i];
  }
  B.n_w = n_w;
  const int64_t nb = in / block_elems(type);
  QA A{};
  A.nb = nb;
  if (!fused) {
    const int act = act_of(type);
    const ActLayout l = act_layout(act, n_acts, nb);
    const uint8_t* base = static_cast<const uint8_t*>(acts);
    const int64_t b0 = t0 * nb;  // first block of activation row t0
    A.qs = reinterpret_cast<const int8_t*>(base + l.qs_off) + b0 * (act == kActQ8_K ? 256 : 32);
    A.d = reinterpret_cast<const float*>(base + l.d_off) + b0;
    A.s = act == kActQ8_1 ? reinterpret_cast<const float*>(base + l.s_off) + b0 : nullptr;
    A.bsums = reinterpret_cast<const int16_t*>(base + l.bsums_off) + b0 * 16;
  }
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (type) {
    case kQ4_0: return launch_gemv<kQ4_0>(B, rows, n_w, A, x, in, n, fused, s);
    case kQ5_0: return launch_gemv<kQ5_0>(B, rows, n_w, A, x, in, n, fused, s);
    case kQ5_1: return launch_gemv<kQ5_1>(B, rows, n_w, A, x, in, n, fused, s);
    case kQ8_0: return launch_gemv<kQ8_0>(B, rows, n_w, A, x, in, n, fused, s);
    case kQ4_K: return launch_gemv<kQ4_K>(B, rows, n_w, A, x, in, n, fused, s);
    case kQ5_K: return launch_gemv<kQ5_K>(B, rows, n_w, A, x, in, n, fused, s);
    case kQ6_K: return launch_gemv<kQ6_K>(B, rows, n_w, A, x, in, n, fused, s);
    default: return NBHS_EINVAL;
  }
}

int nbhs_qgemm_multi(int type, int n_w, const void* const* w, const int64_t* rows, float* const* y, int64_t in,
                     const void* acts, int64_t n, nbhs_stream stream) {
  return is_k(type) ? NBHS_EINVAL : qgemm_multi(type, n_w, w, rows, y, in, acts, n, stream);
}

int nbhs_qgemm_k16_multi(int type, int n_w, const void* const* w, const int64_t* rows, float* const* y, int64_t in,
                         const void* acts, int64_t acts_bytes, int64_t n, nbhs_stream stream) {
  const int64_t need = nbhs_quant_act_k16_bytes(type, n, in);
  return need < 0 || acts_bytes < need ? NBHS_EINVAL : qgemm_multi(type, n_w, w, rows, y, in, acts, n, stream);
}

int nbhs_dequant_rows(int type, const void* w, int64_t rows, int64_t in, const int32_t* ids, int64_t n, float* out,
                      nbhs_stream stream) {
  return ids ? dequant_rows(type, w, rows, in, nullptr, ids, n, out, stream) : NBHS_EINVAL;
}

int nbhs_dequant_rows_host_ids(int type, const void* w, int64_t rows, int64_t in, const int32_t* ids, int64_t n, float* out,
                               nbhs_stream stream) {
  return ids && n <= NBHS_EMBED_ARG_IDS ? dequant_rows(type, w, rows, in, ids, nullptr, n, out, stream) : NBHS_EINVAL;
}

}  // extern "C"
