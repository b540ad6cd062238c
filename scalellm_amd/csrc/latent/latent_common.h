// latent_common.h -- shared helpers of libslm_latent: element access by dtype, reductions.
#pragma once
#include "common.h"
#include "slm_latent.h"

namespace slm {

typedef __bf16 bf16;
typedef uint32_t u32x4u __attribute__((ext_vector_type(4)));

constexpr float LOG2E_F = 1.4426950408889634f;

template <typename E>
__device__ __forceinline__ float to_f32(E v) { return (float)v; }

// N consecutive elements as fp32 (N * sizeof(E) bytes aligned)
template <typename E, int N>
struct Vec { E v[N]; };
template <int N>
__device__ __forceinline__ void load_f32(const float* p, float (&o)[N]) {
  const Vec<float, N> t = *reinterpret_cast<const Vec<float, N>*>(p);
#pragma unroll
  for (int i = 0; i < N; ++i) o[i] = t.v[i];
}
template <int N>
__device__ __forceinline__ void load_f32(const bf16* p, float (&o)[N]) {
  typedef bf16 vec_t __attribute__((ext_vector_type(N)));
  const vec_t t = *reinterpret_cast<const vec_t*>(p);
#pragma unroll
  for (int i = 0; i < N; ++i) o[i] = (float)t[i];
}
template <>
__device__ __forceinline__ void load_f32<1>(const float* p, float (&o)[1]) { o[0] = *p; }
template <>
__device__ __forceinline__ void load_f32<1>(const bf16* p, float (&o)[1]) { o[0] = (float)*p; }
template <>
__device__ __forceinline__ void load_f32<4>(const float* p, float (&o)[4]) {
  const f32x4 t = *reinterpret_cast<const f32x4*>(p);
  o[0] = t.x; o[1] = t.y; o[2] = t.z; o[3] = t.w;
}
template <>
__device__ __forceinline__ void load_f32<8>(const float* p, float (&o)[8]) {
  const f32x4 t = *reinterpret_cast<const f32x4*>(p), u = *reinterpret_cast<const f32x4*>(p + 4);
  o[0] = t.x; o[1] = t.y; o[2] = t.z; o[3] = t.w;
  o[4] = u.x; o[5] = u.y; o[6] = u.z; o[7] = u.w;
}
template <int N>
__device__ __forceinline__ void store_f32(float* p, const float (&o)[N]) {
  if constexpr (N % 4 == 0) {
#pragma unroll
    for (int i = 0; i < N; i += 4) *reinterpret_cast<f32x4*>(p + i) = f32x4{o[i], o[i + 1], o[i + 2], o[i + 3]};
  } else
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = o[i];
}
template <int N>
__device__ __forceinline__ void store_f32(bf16* p, const float (&o)[N]) {
  if constexpr (N == 4) *reinterpret_cast<u32x2*>(p) = u32x2{pack2<bf16_tag>(o[0], o[1]), pack2<bf16_tag>(o[2], o[3])};
  else if constexpr (N == 8)
    *reinterpret_cast<u32x4*>(p) = u32x4{pack2<bf16_tag>(o[0], o[1]), pack2<bf16_tag>(o[2], o[3]), pack2<bf16_tag>(o[4], o[5]), pack2<bf16_tag>(o[6], o[7])};
  else
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = (bf16)o[i];
}

__device__ __forceinline__ float wave_sum(float v) { return group_sum<64>(v); }
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}
// over a workgroup of 256; `tmp` = 4 floats of LDS, reusable after the call
__device__ __forceinline__ float block_sum256(float v, float* tmp) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) tmp[threadIdx.x >> 6] = v;
  __syncthreads();
  return tmp[0] + tmp[1] + tmp[2] + tmp[3];
}
__device__ __forceinline__ float block_max256(float v, float* tmp) {
  v = wave_max(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) tmp[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmaxf(fmaxf(tmp[0], tmp[1]), fmaxf(tmp[2], tmp[3]));
}

// 4 / (1 + 2^z): the reciprocal corrected once, half the instructions of a division, which are a GLU's length in a product's epilogue
// (5692 x 28672 x 4096 1009 / 993 us).  Of a quarter of the denominator, which is nowhere too small for the instruction; of infinity it is 0,
// whose correction would be of infinity times 0.
__device__ __forceinline__ float sigmoid_quarters(float z) {
  const float d = __builtin_fmaf(fast_exp2(z), 0.25f, 0.25f), r = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(fmaxf(__builtin_fmaf(-d, r, 1.0f), -1.0f), r, r);
}
__device__ __forceinline__ float sigmoid_f32(float x) { return 0.25f * sigmoid_quarters(x * -LOG2E_F); }
__device__ __forceinline__ float clamped_glu_f32(float g, float u, float limit, float alpha, float shift) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return 0.25f * g * sigmoid_quarters(g * (alpha * -LOG2E_F)) * (u + shift);
}

// sequence of a query row: the last s with q_cu[s] <= row (batch >= 1)
__device__ __forceinline__ int seq_of_row(const int32_t* q_cu, int batch, int row) {
  int lo = 0, hi = batch - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (q_cu[mid] <= row) lo = mid; else hi = mid - 1;
  }
  return lo;
}

constexpr float M_INIT_F = -1.0e30f;

// what slm_linear refuses (linear.hip)
int linear_check(const slm_linear_args* a);

// barrier for LDS traffic only: outstanding global loads (register prefetch) stay in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

}  // namespace slm
