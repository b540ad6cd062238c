// latent_cache.hip -- the latent cache: append (latent RMS norm + rotation, fused) and gather.
// Cache row of a token: [c_pad] normed latent | [r_pad] rotated key part shared by all heads, zero padded.
// Bound: HBM, trivial.
#include "latent_append.h"

namespace slm {

template <typename E, int V>
__global__ void __launch_bounds__(256) latent_append_kernel(const slm_latent_append_args a) {
  latent_append_row<E, V>(a, blockIdx.x);
}

__global__ void __launch_bounds__(256) latent_gather_kernel(u32x4* __restrict__ out, const u32x4* __restrict__ cache,
                                                            const int32_t* __restrict__ slots, int64_t n_chunks, int chunks) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n_chunks) return;
  const int64_t r = i / chunks;
  out[i] = cache[(int64_t)slots[r] * chunks + i % chunks];
}

}  // namespace slm

using namespace slm;

extern "C" SLM_API int slm_latent_append(const slm_latent_append_args* a, void* stream) {
  if (latent_append_invalid(a)) return SLM_ERR_INVALID_ARG;
  if (a->rows == 0) return SLM_OK;
  hip_clear_error();
  const dim3 grid((unsigned)a->rows);
  hipStream_t st = (hipStream_t)stream;
  const bool v4 = latent_append_by_four(*a);
  if (a->dtype == SLM_BF16) {
    if (v4) latent_append_kernel<bf16, 4><<<grid, dim3(256), 0, st>>>(*a);
    else latent_append_kernel<bf16, 1><<<grid, dim3(256), 0, st>>>(*a);
  } else if (a->dtype == SLM_F32) {
    if (v4) latent_append_kernel<float, 4><<<grid, dim3(256), 0, st>>>(*a);
    else latent_append_kernel<float, 1><<<grid, dim3(256), 0, st>>>(*a);
  } else {
    return SLM_ERR_UNSUPPORTED;
  }
  return hip_check_launch();
}

extern "C" SLM_API int slm_latent_gather(void* out, const void* cache, const int32_t* slots, int64_t n, int64_t row_bytes,
                                         void* stream) {
  if (!out || !cache || !slots || n < 0 || row_bytes <= 0 || row_bytes % 16) return SLM_ERR_INVALID_ARG;
  if (!aligned16(out) || !aligned16(cache)) return SLM_ERR_ALIGNMENT;
  if (n == 0) return SLM_OK;
  const int chunks = (int)(row_bytes / 16);
  const int64_t total = n * chunks;
  hip_clear_error();
  latent_gather_kernel<<<dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream>>>(
      (u32x4*)out, (const u32x4*)cache, slots, total, chunks);
  return hip_check_launch();
}
