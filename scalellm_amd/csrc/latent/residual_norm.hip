// residual_norm.hip -- the fp32 residual stream: what a sub-layer adds (or the embedding), and the norm (RMS, or
// tanh(alpha x), which needs no statistics) in front of the next projection, in one launch.  One workgroup per row; the row stays in
// registers between the sum of squares and the scaling.  Bound: HBM, trivial.
#include <type_traits>

#include "latent_common.h"

namespace slm {

constexpr int RN_THREADS = 256;
constexpr int RN_STEPS = 16;  // register-resident chunks per thread

// over a workgroup of T
template <int T>
__device__ __forceinline__ float row_sum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < T / 64; ++w) s += red[w];
  return s;
}

// V: elements per chunk (4 when every row start is 4-element aligned, else 1).  T: threads of a row.  A row of a batch that fills
// the chip hides its own latency; few rows are as long as a thread's chunks are many, so they get 1024 threads (below 256 rows, from
// 2048 columns; 256 -> 1024 at 4096 columns, 4 slabs: 1 row 4.5 -> 3.0 us, 128 rows 5.1 -> 3.8; 2048 columns 3.3 -> 2.5, 3.7 -> 2.9)
// and more rows 512 (256 / 512 / 1024: 300 x 4096 5.5 / 5.0 / 5.0, 4096 x 2048 18.5 / 17.3 / 19.3, 5692 x 4096 42.4 / 41.4 / 41.5).
template <typename E, int MODE, int V, int T>
__global__ void __launch_bounds__(T) residual_norm_kernel(const slm_residual_norm_args a) {
  constexpr int RN_THREADS = T, RN_STEPS = slm::RN_STEPS * slm::RN_THREADS / T;
  __shared__ float red[T / 64];
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x;
  const int width = (int)a.width;
  auto clear = [&]() {   // (somebody's counters: a launch less.  Last: a store in front of the loads is waited for with them)
    if constexpr (MODE == SLM_RN_EMBED) {
      for (int64_t i = row * T + tid; i < a.n_clear; i += a.rows * T) a.clear[i] = 0;
    }
  };
  const int64_t src_row = (MODE == SLM_RN_PLAIN && a.row_index) ? a.row_index[row] + a.row_shift : row;
  float* r = a.resid + src_row * a.width;
  const E* e0 = nullptr;
  const E* e1 = nullptr;
  if constexpr (MODE == SLM_RN_EMBED) {
    e0 = reinterpret_cast<const E*>(a.embed) + (int64_t)a.tokens[row] * a.ld_embed;
    if (a.pos_table) e1 = reinterpret_cast<const E*>(a.pos_table) + (int64_t)a.positions[row] * a.width;
  }
  if constexpr (MODE == SLM_RN_ADD) e0 = reinterpret_cast<const E*>(a.delta) + row * a.ld_delta;

  float x[RN_STEPS][V];
  float ss = 0.f;
#pragma unroll
  for (int s = 0; s < RN_STEPS; ++s) {
    const int i = (tid + s * RN_THREADS) * V;
    if (i < width) {
      if constexpr (MODE == SLM_RN_EMBED) {
        load_f32<V>(e0 + i, x[s]);
        if (e1) {
          float t[V];
          load_f32<V>(e1 + i, t);
#pragma unroll
          for (int j = 0; j < V; ++j) x[s][j] += t[j];
        }
#pragma unroll
        for (int j = 0; j < V; ++j) x[s][j] *= a.delta_mult;
      } else {
        load_f32<V>(r + i, x[s]);
        if constexpr (MODE == SLM_RN_ADD) {
          float t[V];
          load_f32<V>(e0 + i, t);
#pragma unroll
          for (int j = 0; j < V; ++j) x[s][j] = __builtin_fmaf(t[j], a.delta_mult, x[s][j]);
        }
        if constexpr (MODE == SLM_RN_SLABS) {
          // (all slab loads of a chunk in flight at once)
          const float* sp = a.slabs + row * a.ld_delta + i;
          float d[V];
#pragma unroll
          for (int j = 0; j < V; ++j) d[j] = 0.f;
          for (int k0 = 0; k0 < a.n_slabs; k0 += 8) {
            float t[8][V];
#pragma unroll
            for (int k = 0; k < 8; ++k)
              if (k0 + k < a.n_slabs) load_f32<V>(sp + (k0 + k) * a.slab_stride, t[k]);
#pragma unroll
            for (int k = 0; k < 8; ++k)
              if (k0 + k < a.n_slabs)
#pragma unroll
                for (int j = 0; j < V; ++j) d[j] += t[k][j];
          }
#pragma unroll
          for (int j = 0; j < V; ++j) x[s][j] = __builtin_fmaf(d[j], a.delta_mult, x[s][j]);
        }
      }
      if constexpr (MODE != SLM_RN_PLAIN) store_f32<V>(r + i, x[s]);
#pragma unroll
      for (int j = 0; j < V; ++j) ss = __builtin_fmaf(x[s][j], x[s][j], ss);
    }
  }
  if (!a.weight) return clear();  // (uniform: only the sum was asked for)
  const bool rms = a.norm == SLM_NORM_RMS;
  const float rs = rms ? 1.0f / sqrtf(row_sum<T>(ss, red) / (float)width + a.eps) : 0.f;
  E* o = reinterpret_cast<E*>(a.out) + row * a.ld_out;
#pragma unroll
  for (int s = 0; s < RN_STEPS; ++s) {
    const int i = (tid + s * RN_THREADS) * V;
    if (i < width) {
      float w[V], y[V];
      load_f32<V>(a.weight + i, w);
#pragma unroll
      for (int j = 0; j < V; ++j) y[j] = x[s][j] * rs * w[j];
      if (!rms) {
        float b[V];
        load_f32<V>(a.bias + i, b);
#pragma unroll
        for (int j = 0; j < V; ++j) y[j] = __builtin_fmaf(tanhf(a.norm_alpha * x[s][j]), w[j], b[j]);
      }
      store_f32<V>(o + i, y);
    }
  }
  for (int i = width + tid; i < (int)a.ld_out; i += RN_THREADS) o[i] = (E)0.f;
  clear();
}

// V columns a thread: 8 where every row lies on 16 bytes, else 4.  5692 rows of 14336: 107 us -> 97 (490 MB; a 64-bit division a thread before).
template <typename E, int V>
__global__ void __launch_bounds__(256) clamped_glu_kernel(E* __restrict__ y, const E* __restrict__ gu, uint32_t steps, uint32_t n,
                                                          int64_t ld_gu, int64_t ld_y, float limit, float alpha, float shift) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint32_t row = i / steps, c = (i - row * steps) * V;
  const E* src = gu + row * ld_gu + c;
  float g[V], u[V], o[V];
  load_f32<V>(src, g);
  load_f32<V>(src + (int64_t)steps * V, u);
#pragma unroll
  for (int j = 0; j < V; ++j) o[j] = clamped_glu_f32(g[j], u[j], limit, alpha, shift);
  store_f32<V>(y + row * ld_y + c, o);
}
template <typename E>
static int glu_launch(void* y, const void* gu, int64_t rows, int64_t half, int64_t ld_gu, int64_t ld_y, float limit, float alpha, float shift,
                      hipStream_t st) {
  const bool v8 = half % 8 == 0 && ld_gu % 8 == 0 && ld_y % 8 == 0;
  const int64_t steps = half / (v8 ? 8 : 4), n = rows * steps;
  if (n > 0xffffff00ll) return SLM_ERR_UNSUPPORTED;   // a launch has fewer than 2^32 threads
  const dim3 grid((unsigned)((n + 255) / 256));
  hip_clear_error();
  if (v8) clamped_glu_kernel<E, 8><<<grid, dim3(256), 0, st>>>((E*)y, (const E*)gu, (uint32_t)steps, (uint32_t)n, ld_gu, ld_y, limit, alpha, shift);
  else clamped_glu_kernel<E, 4><<<grid, dim3(256), 0, st>>>((E*)y, (const E*)gu, (uint32_t)steps, (uint32_t)n, ld_gu, ld_y, limit, alpha, shift);
  return hip_check_launch();
}

// The GLU over NS slabs of a streamed product, whose columns come 16 of the gate, the same 16 of the up half in turn: four columns a
// thread, all loads before the sums.  Bound: latency (4096 columns, 64 rows, 4 slabs: 4 MB out of the L2).
template <int NS>
__global__ void __launch_bounds__(256) glu_slabs_kernel(bf16* __restrict__ y, const float* __restrict__ slabs, uint32_t quads, uint32_t n,
                                                        int64_t slab_stride, int64_t ld_y, float limit, float alpha, float shift) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint32_t row = i / quads, c = (i - row * quads) * 4;
  const float* src = slabs + (int64_t)row * (8 * (int64_t)quads) + 2 * (c & ~15u) + (c & 15u);
  f32x4 g[NS], u[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    g[s] = *reinterpret_cast<const f32x4*>(src + s * slab_stride);
    u[s] = *reinterpret_cast<const f32x4*>(src + s * slab_stride + 16);
  }
#pragma unroll
  for (int s = 1; s < NS; ++s) g[0] += g[s], u[0] += u[s];
  bf16* o = y + row * ld_y + c;
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = (bf16)clamped_glu_f32(g[0][j], u[0][j], limit, alpha, shift);
}

template <typename E, int MODE>
static int rn_launch(const slm_residual_norm_args& a, hipStream_t st) {
  const bool v4 = a.width % 4 == 0 && a.ld_delta % 4 == 0 && a.ld_embed % 4 == 0 && a.ld_out % 4 == 0 &&
                  a.slab_stride % 4 == 0 && aligned16(a.resid) && aligned16(a.delta) && aligned16(a.slabs) &&
                  aligned16(a.embed) && aligned16(a.pos_table) && aligned16(a.weight) && aligned16(a.bias) && aligned16(a.out);
  if (a.width > (v4 ? 4 : 1) * RN_THREADS * RN_STEPS) return SLM_ERR_UNSUPPORTED;
  hip_clear_error();
  const dim3 grid((unsigned)a.rows);
  if (v4 && a.rows < 256 && a.width >= 2048) residual_norm_kernel<E, MODE, 4, 1024><<<grid, dim3(1024), 0, st>>>(a);
  else if (v4 && a.width >= 2048) residual_norm_kernel<E, MODE, 4, 512><<<grid, dim3(512), 0, st>>>(a);
  else if (v4) residual_norm_kernel<E, MODE, 4, RN_THREADS><<<grid, dim3(RN_THREADS), 0, st>>>(a);
  else residual_norm_kernel<E, MODE, 1, RN_THREADS><<<grid, dim3(RN_THREADS), 0, st>>>(a);
  return hip_check_launch();
}
template <typename E>
static int rn_mode(const slm_residual_norm_args& a, hipStream_t st) {
  switch (a.mode) {
    case SLM_RN_EMBED: return rn_launch<E, SLM_RN_EMBED>(a, st);
    case SLM_RN_ADD: return rn_launch<E, SLM_RN_ADD>(a, st);
    case SLM_RN_SLABS: return rn_launch<E, SLM_RN_SLABS>(a, st);
    default: return rn_launch<E, SLM_RN_PLAIN>(a, st);
  }
}

}  // namespace slm

using namespace slm;

extern "C" SLM_API const char* slm_latent_version(void) { return "slm_latent 1 (gfx950)"; }
extern "C" SLM_API const char* slm_latent_last_hip_error(void) {
  return hipGetErrorString((hipError_t)hip_last_error_slot());
}
extern "C" SLM_API const char* slm_latent_status_string(int s) {
  switch (s) {
    case SLM_OK: return "ok";
    case SLM_ERR_INVALID_ARG: return "invalid argument";
    case SLM_ERR_UNSUPPORTED: return "unsupported dtype or size";
    case SLM_ERR_WORKSPACE: return "workspace missing or too small";
    case SLM_ERR_LAUNCH: return "kernel launch failed";
    case SLM_ERR_ALIGNMENT: return "pointer or stride not aligned";
    default: return "unknown status";
  }
}

extern "C" SLM_API int slm_residual_norm(const slm_residual_norm_args* a, void* stream) {
  if (!a || a->rows < 0 || a->width <= 0 || !a->resid || a->mode < 0 || a->mode > SLM_RN_PLAIN) return SLM_ERR_INVALID_ARG;
  if (a->rows == 0) return SLM_OK;
  if (a->mode == SLM_RN_EMBED && (!a->tokens || !a->embed || a->ld_embed < a->width || (a->pos_table && !a->positions)))
    return SLM_ERR_INVALID_ARG;
  if (a->mode == SLM_RN_ADD && (!a->delta || a->ld_delta < a->width)) return SLM_ERR_INVALID_ARG;
  if (a->mode == SLM_RN_SLABS && (!a->slabs || a->n_slabs < 1 || a->ld_delta < a->width)) return SLM_ERR_INVALID_ARG;
  if (a->weight ? (!a->out || a->ld_out < a->width) : a->mode == SLM_RN_PLAIN) return SLM_ERR_INVALID_ARG;
  if (a->norm < 0 || a->norm > SLM_NORM_TANH || (a->weight && a->norm == SLM_NORM_TANH && !a->bias)) return SLM_ERR_INVALID_ARG;
  if (a->n_clear < 0 || a->n_clear > 65536 || (a->n_clear && (!a->clear || a->mode != SLM_RN_EMBED))) return SLM_ERR_INVALID_ARG;
  if (a->dtype == SLM_BF16) return rn_mode<bf16>(*a, (hipStream_t)stream);
  if (a->dtype == SLM_F32) return rn_mode<float>(*a, (hipStream_t)stream);
  return SLM_ERR_UNSUPPORTED;
}

extern "C" SLM_API int slm_clamped_glu(void* y, const void* gu, int64_t rows, int64_t half, int64_t ld_gu, int64_t ld_y,
                                       float limit, float glu_alpha, float glu_shift, int32_t dtype, void* stream) {
  if (!y || !gu || rows < 0 || half <= 0 || half % 4 || ld_gu < 2 * half || ld_gu % 4 || ld_y < half || ld_y % 4)
    return SLM_ERR_INVALID_ARG;
  if (!aligned16(y) || !aligned16(gu)) return SLM_ERR_ALIGNMENT;
  if (rows == 0) return SLM_OK;
  if (dtype == SLM_BF16) return glu_launch<bf16>(y, gu, rows, half, ld_gu, ld_y, limit, glu_alpha, glu_shift, (hipStream_t)stream);
  if (dtype == SLM_F32) return glu_launch<float>(y, gu, rows, half, ld_gu, ld_y, limit, glu_alpha, glu_shift, (hipStream_t)stream);
  return SLM_ERR_UNSUPPORTED;
}

extern "C" SLM_API int slm_glu_slabs(void* y, const void* slabs, int64_t rows, int64_t half, int32_t n_slabs, int64_t ld_y, float limit,
                                     float glu_alpha, float glu_shift, void* stream) {
  if (!y || !slabs || rows < 0 || half <= 0 || half % 16 || n_slabs < 1 || n_slabs > 8 || ld_y < half) return SLM_ERR_INVALID_ARG;
  if (!aligned16(slabs)) return SLM_ERR_ALIGNMENT;
  if (rows == 0) return SLM_OK;
  const int64_t quads = half / 4, n = rows * quads;
  if (n > 0xffffff00ll || rows > 0x7fffffff) return SLM_ERR_UNSUPPORTED;   // a launch has fewer than 2^32 threads
  auto launch = [&](auto count) {
    glu_slabs_kernel<decltype(count)::value><<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream>>>(
        (bf16*)y, (const float*)slabs, (uint32_t)quads, (uint32_t)n, rows * 2 * half, ld_y, limit, glu_alpha, glu_shift);
  };
  hip_clear_error();
  switch (n_slabs) {
    case 1: launch(std::integral_constant<int, 1>{}); break;
    case 2: launch(std::integral_constant<int, 2>{}); break;
    case 3: launch(std::integral_constant<int, 3>{}); break;
    case 4: launch(std::integral_constant<int, 4>{}); break;
    case 5: launch(std::integral_constant<int, 5>{}); break;
    case 6: launch(std::integral_constant<int, 6>{}); break;
    case 7: launch(std::integral_constant<int, 7>{}); break;
    default: launch(std::integral_constant<int, 8>{}); break;
  }
  return hip_check_launch();
}
