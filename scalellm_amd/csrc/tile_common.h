// tile_common.h -- what the kernels of four-wave tiles share (w4_tile.hip, latent/gemm.hip): their place in the grid, the end of their products, and
// tiles that are cut in K.
#pragma once
#include "common.h"

namespace slm {

// A run of `n` items for each of the 8 XCDs, which workgroups go round: item of a workgroup, -1 for none
__device__ __forceinline__ int xcd_run(int wg, int n) {
  const int per = (n + 7) >> 3, i = wg >> 3, t = (wg & 7) * per + i;
  return i < per && t < n ? t : -1;
}

// Behind the last product: the compiler knows nothing of products that inline asm made.  Whoever reads an accumulator takes it from behind the wait.
template <int NT, int MT>
__device__ __forceinline__ void tile_products_settle(f32x4 (&acc)[NT][MT]) {
  asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) asm volatile("" : "+a"(acc[n][m]));
}

// The same where no DMA may outlive the workgroup's LDS
template <int NT, int MT>
__device__ __forceinline__ void tile_settle(f32x4 (&acc)[NT][MT]) {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  tile_products_settle(acc);
}

// The tile's fp32 sums go past the caches to its slabs, [slices][NT MT][256] f32x4; the last slice to arrive (*arrived, zero before) adds them up in
// slice order -- the same bits whoever is last -- and is the one that gets true.  Nobody waits for anybody.  256 threads; lds: 4 bytes of it.
template <int NT, int MT>
__device__ __forceinline__ bool tile_add_slices(f32x4 (&acc)[NT][MT], float* slabs, uint32_t* arrived, int slice, int slices, char* lds) {
  constexpr int FRAGS = NT * MT, C = 8;   // C: fragments in flight
  const int tid = threadIdx.x;
  const __amdgpu_buffer_rsrc_t mine = __builtin_amdgcn_make_buffer_rsrc(slabs, 0, slices * FRAGS * 4096, 0x00020000);
  auto at = [&](int s, int f) { return ((s * FRAGS + f) * 256 + tid) * 16; };
#pragma unroll
  for (int f = 0; f < FRAGS; ++f)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[f / MT][f % MT]), mine, at(slice, f), 0, /*sc1*/ 16);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every wave's sums are out ..
  __syncthreads();
  uint32_t* word = reinterpret_cast<uint32_t*>(lds);
  if (tid == 0) word[0] = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // .. then one announces them
  __syncthreads();
  if (word[0] != (uint32_t)slices - 1) return false;
#pragma unroll
  for (int f0 = 0; f0 < FRAGS; f0 += C) {
    f32x4 sum[C];
#pragma unroll
    for (int f = 0; f < C; ++f) sum[f] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < slices; ++s) {
#pragma unroll
      for (int f = 0; f < C; ++f)
        sum[f] += __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(mine, at(s, f0 + f), 0, /*sc1*/ 16));
    }
#pragma unroll
    for (int f = 0; f < C; ++f) {
      acc[(f0 + f) / MT][(f0 + f) % MT] = sum[f];
      asm volatile("" : "+a"(acc[(f0 + f) / MT][(f0 + f) % MT]));   // (one place for them: else what follows has a copy of all, in front of the branch too)
    }
  }
  return true;
}

// (a kernel: the call may be captured, and memset nodes of a graph have given wrong results on later replays)
static __global__ void __launch_bounds__(256) tile_clear_kernel(uint32_t* p, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0;
}

// More than 64 KiB of dynamic LDS is asked for once per kernel and device
template <typename F>
inline void tile_allow_lds(F* fn, int bytes, bool (&asked)[64]) {
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev >= 0 && dev < 64 && asked[dev]) return;
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (dev >= 0 && dev < 64) asked[dev] = true;
}

}  // namespace slm
