// The rest of the Backend's per-token ops on the GPU, so that a whole forward (transformer.cpp:166-230) can stay in
// HBM: embed, rmsnorm, add and silu_mul (backend.h:55-70), with the semantics of ref_ops.cpp.
//  * embed (ref_ops.cpp:80-99): row copy for F32 tables, exact widening for F16; bit-exact.
//  * rmsnorm (ref_ops.cpp:137-148): sum of squares in double (float * float is exact in double, so only the order
//    of the sum differs from the reference), scale = 1 / sqrt(ss / d + eps) in double, y = float(x * scale * w)
//    with the reference's two double products in its order. The file is compiled with -ffp-contract=off, so no
//    multiply-add is fused (the reference's ref_ops.cpp is built the same way).
//  * add (ref_ops.cpp:151-153): one float add per element; bit-exact.
//  * silu_mul (ref_ops.cpp:217-222): gate = g / (1 + exp(-g)) * up in float; exp is the device library's expf,
//    so results match the reference within a few ulp (the reference's own SIMD tier uses its own exp too).
// All four are HBM-bound streams.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "backend/hip/kernel_timing.h"
#include "nibble_hip_shim.h"

namespace {

constexpr int kThreads = 256;

unsigned grid_for(int64_t count) {
  const int64_t blocks = (count + kThreads - 1) / kThreads;
  return unsigned(blocks < 8192 ? (blocks > 0 ? blocks : 1) : 8192);
}

struct EmbedIds {
  int32_t id[NBHS_EMBED_ARG_IDS];
};

// out[t, :] = row ids[t] of the table, widened to float. One workgroup per output row.
template <bool F16>
__global__ __launch_bounds__(kThreads) void embed_kernel(const void* __restrict__ table, EmbedIds ids,
                                                         const int32_t* __restrict__ far_ids, float* __restrict__ out,
                                                         int64_t d) {
  const int64_t t = blockIdx.x;
  const int64_t id = far_ids ? far_ids[t] : ids.id[t];
  float* o = out + t * d;
  if constexpr (F16) {
    const _Float16* r = static_cast<const _Float16*>(table) + id * d;
    for (int64_t k = threadIdx.x; k < d; k += kThreads) o[k] = float(r[k]);
  } else {
    const float* r = static_cast<const float*>(table) + id * d;
    for (int64_t k = threadIdx.x; k < d; k += kThreads) o[k] = r[k];
  }
}

// A value from another lane of the 16-lane row, by DPP (a few cycles; a double __shfl is two trips through LDS).
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, int(uint32_t(b)), CTRL, 0xF, 0xF, true);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, int(uint32_t(b >> 32)), CTRL, 0xF, 0xF, true);
  return __builtin_bit_cast(double, uint64_t(hi) << 32 | lo);
}
__device__ __forceinline__ double lane_f64(double v, int l) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane(int(uint32_t(b)), l), hi = __builtin_amdgcn_readlane(int(uint32_t(b >> 32)), l);
  return __builtin_bit_cast(double, uint64_t(hi) << 32 | lo);
}

__device__ __forceinline__ double wave_sum_f64(double v) {
  v += dpp_f64<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_f64<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_f64<0x141>(v);  // row_half_mirror
  v += dpp_f64<0x140>(v);  // row_mirror
  return (lane_f64(v, 0) + lane_f64(v, 16)) + (lane_f64(v, 32) + lane_f64(v, 48));
}

// One workgroup per row of d elements. A row is a chain of latencies (its loads, the sum over the workgroup, a square
// root and two divisions in double), so its elements stay in registers (up to HELD per thread) and every thread finishes
// the sum by itself: one barrier, no second trip for the scale. One row of 2048: 5.8 -> 4.6 us. Where many short rows keep
// the CUs busy, that arithmetic done by all four waves is the time itself: from kNormMany rows of at most kNormShort elements
// a thread on, one wave does it (ONE) and a second barrier hands the scale on. Every thread against one wave, us: 8192 rows
// of 64 10.0 / 5.2, of 512 11.8 / 7.3, 2048 rows of 512 4.5 / 3.3, 512 rows 3.3 both; rows of 896 are bound by memory (8192
// of them 14.6, 16.4 in the form with a second trip for the scale).
constexpr int kNormHeld = 8, kNormShort = 2, kNormMany = 1024;
template <int HELD, bool ONE>
__global__ __launch_bounds__(kThreads) void rmsnorm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                           float* __restrict__ y, int64_t d, float eps) {
  __shared__ double part[kThreads / 64];
  __shared__ double shared_scale;
  const int64_t t = blockIdx.x;
  const float* xt = x + t * d;
  float held[HELD], wt[HELD];
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int64_t i = threadIdx.x + int64_t(c) * kThreads;
    held[c] = i < d ? xt[i] : 0.f;
    wt[c] = i < d ? w[i] : 0.f;
  }
  double ss = 0.0;
#pragma unroll
  for (int c = 0; c < HELD; ++c) ss = __dadd_rn(ss, __dmul_rn(double(held[c]), double(held[c])));
  for (int64_t i = threadIdx.x + HELD * kThreads; i < d; i += kThreads) {
    const double v = double(xt[i]);
    ss = __dadd_rn(ss, __dmul_rn(v, v));
  }
  ss = wave_sum_f64(ss);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
  __syncthreads();
  double scale;
  if (!ONE || threadIdx.x < 64) {
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < kThreads / 64; ++i) s = __dadd_rn(s, part[i]);
    scale = __ddiv_rn(1.0, __dsqrt_rn(__dadd_rn(__ddiv_rn(s, double(d)), double(eps))));
    if (ONE && threadIdx.x == 0) shared_scale = scale;
  }
  if constexpr (ONE) {
    __syncthreads();
    scale = shared_scale;
  }
  float* yt = y + t * d;
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int64_t i = threadIdx.x + int64_t(c) * kThreads;
    if (i < d) yt[i] = float(__dmul_rn(__dmul_rn(double(held[c]), scale), double(wt[c])));
  }
  for (int64_t i = threadIdx.x + HELD * kThreads; i < d; i += kThreads)
    yt[i] = float(__dmul_rn(__dmul_rn(double(xt[i]), scale), double(w[i])));
}

__global__ __launch_bounds__(kThreads) void add_kernel(float* __restrict__ x, const float* __restrict__ y,
                                                       int64_t count) {
  for (int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x; i < count; i += int64_t(gridDim.x) * kThreads)
    x[i] = __fadd_rn(x[i], y[i]);
}

__global__ __launch_bounds__(kThreads) void silu_mul_kernel(float* __restrict__ gate, const float* __restrict__ up,
                                                            int64_t count) {
  for (int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x; i < count; i += int64_t(gridDim.x) * kThreads) {
    const float g = gate[i];
    gate[i] = __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, expf(-g))), up[i]);
  }
}

// far_ids: device ids, or null with the ids in arg.
int launch_embed(int f16, const void* table, const EmbedIds& arg, const int32_t* far_ids, int64_t n, int64_t d, float* out,
                 nbhs_stream s) {
  const hipStream_t st = reinterpret_cast<hipStream_t>(s);
  if (f16)
    return nbhs_timing::launch(NBHS_K_ELEMENTWISE, embed_kernel<true>, dim3(unsigned(n)), dim3(kThreads), st, table, arg,
                               far_ids, out, d);
  return nbhs_timing::launch(NBHS_K_ELEMENTWISE, embed_kernel<false>, dim3(unsigned(n)), dim3(kThreads), st, table, arg,
                             far_ids, out, d);
}

}  // namespace

extern "C" {

int nbhs_embed(int f16, const void* table, const int32_t* ids, int64_t n, int64_t d, float* out, nbhs_stream s) {
  if (!table || !ids || !out || n <= 0 || d <= 0 || n >= (int64_t(1) << 31)) return NBHS_EINVAL;
  return launch_embed(f16, table, EmbedIds{}, ids, n, d, out, s);
}

int nbhs_embed_host_ids(int f16, const void* table, const int32_t* ids, int64_t n, int64_t d, float* out, nbhs_stream s) {
  if (!table || !ids || !out || n <= 0 || d <= 0 || n > NBHS_EMBED_ARG_IDS) return NBHS_EINVAL;
  EmbedIds arg{};
  std::copy(ids, ids + n, arg.id);
  return launch_embed(f16, table, arg, nullptr, n, d, out, s);
}

int nbhs_rmsnorm_f32(const float* x, const float* w, float* y, int64_t n, int64_t d, float eps, nbhs_stream s) {
  if (!x || !w || !y || n <= 0 || d <= 0 || n >= (int64_t(1) << 31)) return NBHS_EINVAL;
  const hipStream_t st = reinterpret_cast<hipStream_t>(s);
  if (d <= kNormShort * kThreads && n >= kNormMany)
    return nbhs_timing::launch(NBHS_K_RMSNORM, rmsnorm_kernel<kNormShort, true>, dim3(unsigned(n)), dim3(kThreads), st, x, w,
                               y, d, eps);
  return nbhs_timing::launch(NBHS_K_RMSNORM, rmsnorm_kernel<kNormHeld, false>, dim3(unsigned(n)), dim3(kThreads), st, x, w, y,
                             d, eps);
}

int nbhs_add_f32(float* x, const float* y, int64_t count, nbhs_stream s) {
  if (!x || !y || count <= 0) return NBHS_EINVAL;
  return nbhs_timing::launch(NBHS_K_ELEMENTWISE, add_kernel, dim3(grid_for(count)), dim3(kThreads),
                             reinterpret_cast<hipStream_t>(s), x, y, count);
}

int nbhs_silu_mul_f32(float* gate, const float* up, int64_t count, nbhs_stream s) {
  if (!gate || !up || count <= 0) return NBHS_EINVAL;
  return nbhs_timing::launch(NBHS_K_ELEMENTWISE, silu_mul_kernel, dim3(grid_for(count)), dim3(kThreads),
                             reinterpret_cast<hipStream_t>(s), gate, up, count);
}

}  // extern "C"
