// linear_stream.hip -- y = x W^T in bf16 for up to 128 rows (decode batches, sampled rows), from weights that were
// laid out for it at load.  Bound: the HBM stream of W; above 64 rows what a CU has under way of x and W together.
//
// Layout of W (slm_linear_stream): panels of 64 columns, in a panel steps of 64 k, in a step four blocks of 16 columns,
// each two MFMA operands of 1 KB: lane (r = lane % 16, g = lane / 16) of operand h holds column r, k = 32 h + 8 g .. + 7.
// A workgroup so reads one linear run of memory, 1 KB an instruction.  From [N, K] rows the same bytes come as 16 or 64
// pieces of 64 to 1024 bytes a row stride apart, and that alone costs 1.2 - 2 times the time whatever is in flight
// (reads only, nothing computed: 28672 x 4096 37 us against 51 - 64, 4096 x 14336 20 against 29, 4096 x 4096 6.6 against 9.1).
//
// Two forms:
//   wave-K   (up to 16 rows, and narrow products up to 32) the waves of a workgroup split K and hold NT column blocks; x comes
//            straight from L2 in fragments, each once per workgroup; partial tiles meet in LDS at the end
//   wave-N   (more rows) the waves split the columns, NT blocks each, and share the step's x through two LDS buffers: x is
//            read from L2 once per 64 NT columns, what a fragment load per wave would quadruple.  WK groups of four waves
//            take every WK-th step (twice the waves on a CU where a launch has one workgroup for it)
// Loads of W and x run D steps ahead in a register ring: the loop has no branch in it, so every wait is for the oldest.
//
// What bounds the wave-N form: a CU has some 32 KB of loads under way, which come back in order, so x waits behind W and both
// together come at 50 - 57 GB/s a CU, whatever is asked for how early (rings of 4 or 8 steps, three or six stages of LDS-DMA: level).  A
// step's bytes are 16 KB of x at 128 rows and 8 KB of W for 64 columns; with 64 rows or 128 columns the memory's own rate is near.  So
// row counts have their own tiles (up to 96 rows 96 instead of 128: 28672 x 4096 45.6 / 42.5 us, 14336 -> 4096 27.3 / 26.2).
//
// us at 28672 x 4096 (GLU) / 14336 -> 4096 (slabs) / 16384 x 2048, against the kernel of linear.hip, and above 32 rows the
// vendor product: 1 row 37.7, 20.4, 12.8 (46, 27.6, 16.4); 16 rows 38.6, 20.7, 13.1 (67, 38, 22); 32 rows 36.2, 19.4, 12.6
// (63, 41, 21); 64 rows 38.4, 22.7, 14.6 (57 + 5 for the GLU's launch, 42, 18); 96 rows 42.5, 26.2, 16.5 (55 with the launch, -, 22); 128 rows
// 47.3, 29.8, 19.0 (59 with the launch, 78, 23).
#include <type_traits>

#include "latent_common.h"

namespace slm {

struct StreamK {   // 64 k of a 16-row block: two operands
  bf16x8_t v[2];
};
__device__ __forceinline__ f32x4 stream_mma(const StreamK& a, const StreamK& b, f32x4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v[0], b.v[0], c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v[1], b.v[1], c, 0, 0, 0);
}
// (read once: past the caches' replacement, 10 % at 235 MB)
__device__ __forceinline__ void stream_load_w(StreamK& d, const bf16* p) {
  d.v[0] = __builtin_bit_cast(bf16x8_t, __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p)));
  d.v[1] = __builtin_bit_cast(bf16x8_t, __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + 512)));
}
// this lane's first element of 16-column block nb
__device__ __forceinline__ const bf16* stream_block(const slm_linear_args& a, int64_t nb, int lane) {
  return reinterpret_cast<const bf16*>(a.w) + (nb >> 2) * 64 * a.K + (nb & 3) * 1024 + lane * 8;
}
constexpr int64_t STREAM_STEP = 64 * 64;   // elements from one step of a panel to the next

// Four columns of row m, or one output: y of the epilogue.  n: column of the product, for GLU of its output
template <int EPI>
__device__ __forceinline__ void stream_store(const slm_linear_args& a, int split, int64_t m, int64_t n, f32x4 v, f32x4 up) {
  if constexpr (EPI == SLM_LIN_SLABS) {
    float* y = reinterpret_cast<float*>(a.y) + ((int64_t)split * a.M + m) * a.ldy + n;
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = v[j];
  } else if constexpr (EPI == SLM_LIN_F32) {
    float* y = reinterpret_cast<float*>(a.y) + m * a.ldy + n;
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = a.alpha * v[j];
  } else {
    bf16* y = reinterpret_cast<bf16*>(a.y) + m * a.ldy + n;
    if constexpr (EPI == SLM_LIN_GLU) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = clamped_glu_f32(v[j], up[j], a.limit, a.glu_alpha, a.glu_shift);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = (bf16)v[j];
  }
}

// output column of block nb: GLU panels hold (gate, up, gate, up) blocks
template <int EPI>
__device__ __forceinline__ int64_t stream_column(int64_t nb) { return EPI == SLM_LIN_GLU ? (nb >> 1) * 16 : nb * 16; }

// Products that are cut in K and stored in one launch.  A workgroup's fp32 sums go past the caches to its tile's slabs, the last of the tile's splits to
// arrive adds all of them up in their order -- the same bits whoever is last -- and stores.  It leaves the counter at zero, as it was found.
// For stored products whose columns leave CUs idle: bound by what a CU has under way, a product of 106 workgroups takes as long on 106 CUs as one of
// twice the columns on 212.  Joining costs 2 to 4 us, two thirds of it the sums' way out and back (us, whole / cut in 2: 6752 x 4096 64 rows 22.2 / 17.7,
// 128 rows 28.2 / 22.8; 6464 x 2048 12.3 / 10.7, 16.0 / 13.9).  A step of four layers, 128 rows: 1074 / 1052 us (8b, latent), 887 / 876 (2b, recurrent).
struct StreamJoin {
  float* slabs;          // [tiles][splits][fragments][256] f32x4
  uint32_t* arrived;     // [tiles], zero
};
// F fragments of thread t (of 256; others only take part in the barriers).  word: 4 bytes of LDS that nobody reads past the first barrier
template <int F>
__device__ __forceinline__ bool stream_join(f32x4 (&acc)[F], const StreamJoin& j, int split, int splits, int t, uint32_t* word) {
  const __amdgpu_buffer_rsrc_t slabs =
      __builtin_amdgcn_make_buffer_rsrc(j.slabs + (int64_t)blockIdx.x * splits * (F * 1024), 0, splits * F * 4096, 0x00020000);
  auto at = [&](int s, int f) { return ((s * F + f) * 256 + t) * 16; };
  if (t < 256) {
#pragma unroll
    for (int f = 0; f < F; ++f) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[f]), slabs, at(split, f), 0, /*sc1*/ 16);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every wave's sums are out ..
  __syncthreads();
  if (threadIdx.x == 0) *word = atomicInc(j.arrived + blockIdx.x, (uint32_t)splits - 1);   // .. then one announces them (the last one's turns to zero)
  __syncthreads();
  if (*word != (uint32_t)splits - 1) return false;
  if (t >= 256) return true;
  if (splits == 2) {   // (its own are at hand; the other order has the same sum)
#pragma unroll
    for (int f = 0; f < F; ++f) acc[f] += __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(slabs, at(1 - split, f), 0, /*sc1*/ 16));
    return true;
  }
#pragma unroll
  for (int f = 0; f < F; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < splits; ++s) {
#pragma unroll
    for (int f = 0; f < F; ++f) acc[f] += __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(slabs, at(s, f), 0, /*sc1*/ 16));
  }
  return true;
}

struct NoJoin {};
template <bool JOIN>
using JoinArgs = std::conditional_t<JOIN, StreamJoin, NoJoin>;

// JOIN: by stream_join, one row of tiles
template <int MT, int NT, int D, int EPI, bool JOIN>
__global__ void __launch_bounds__(256) linear_wave_k_kernel(const slm_linear_args a, const JoinArgs<JOIN> j) {
  constexpr bool GLU = EPI == SLM_LIN_GLU;
  static_assert(!JOIN || (EPI == SLM_LIN_STORE && NT * MT == 4), "a tile a wave");
  static_assert(!GLU || NT % 2 == 0, "gate / up pairs");
  __shared__ f32x4 red[4][NT * MT][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int split = blockIdx.z;
  const int64_t nb0 = (int64_t)blockIdx.x * NT, m0 = (int64_t)blockIdx.y * (16 * MT), blocks = a.N >> 4;
  const bf16* wp[NT];
  const bf16* xp[MT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wp[t] = stream_block(a, min(nb0 + t, blocks - 1), lane);
#pragma unroll
  for (int t = 0; t < MT; ++t) xp[t] = reinterpret_cast<const bf16*>(a.x) + min(m0 + 16 * t + r16, a.M - 1) * a.ldx + 8 * g;
  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int v = 0; v < MT; ++v) acc[t][v] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int steps = (int)(a.K >> 6), per = (steps + a.n_splits - 1) / a.n_splits;
  const int s0 = split * per, s1 = min(steps, s0 + per), first = s0 + wave;
  const int cnt = max(0, (s1 - first + 3) >> 2);   // this wave's steps: first, first + 4, ..
  StreamK w[D][NT], x[D][MT];
  auto load = [&](int u, int i) {
    const int64_t s = first + 4 * i;
#pragma unroll
    for (int t = 0; t < NT; ++t) stream_load_w(w[u][t], wp[t] + s * STREAM_STEP);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      x[u][t].v[0] = *reinterpret_cast<const bf16x8_t*>(xp[t] + (s << 6));
      x[u][t].v[1] = *reinterpret_cast<const bf16x8_t*>(xp[t] + (s << 6) + 32);
    }
  };
  auto multiply = [&](int u) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < MT; ++v) acc[t][v] = stream_mma(w[u][t], x[u][v], acc[t][v]);
  };
  if (cnt >= D) {
#pragma unroll
    for (int u = 0; u < D; ++u) load(u, u);
    __builtin_amdgcn_sched_barrier(0);
    int i = 0;
    for (; i + 2 * D <= cnt; i += D) {
#pragma unroll
      for (int u = 0; u < D; ++u) {
        multiply(u);
        __builtin_amdgcn_sched_barrier(0);
        load(u, i + u + D);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int u = 0; u < D; ++u) {
      multiply(u);
      if (i + u + D < cnt) load(u, i + u + D);
    }
#pragma unroll
    for (int u = 0; u < D; ++u)
      if (i + u + D < cnt) multiply(u);
  } else {
#pragma unroll
    for (int u = 0; u < D; ++u)
      if (u < cnt) load(u, u);
#pragma unroll
    for (int u = 0; u < D; ++u)
      if (u < cnt) multiply(u);
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int v = 0; v < MT; ++v) red[wave][t * MT + v][lane] = acc[t][v];
  __syncthreads();
  // a tile per wave: lane = (columns 4 g .. + 3, row r16), the layout of the products
  constexpr int TILES = (GLU ? NT / 2 : NT) * MT;
  auto total = [&](int tile) { return red[0][tile][lane] + red[1][tile][lane] + red[2][tile][lane] + red[3][tile][lane]; };
  if constexpr (JOIN) {
    f32x4 y[1] = {total(wave)};
    if (!stream_join(y, j, split, a.n_splits, tid, reinterpret_cast<uint32_t*>(red))) return;
    const int64_t nb = nb0 + wave / MT, m = m0 + 16 * (wave % MT) + r16;
    if (nb < blocks && m < a.M) stream_store<EPI>(a, 0, m, nb * 16 + 4 * g, y[0], y[0]);
    return;
  }
  for (int i = wave; i < TILES; i += 4) {
    const int t = i / MT * (GLU ? 2 : 1), v = i % MT;
    const int64_t nb = nb0 + t, m = m0 + 16 * v + r16;
    if (nb >= blocks || m >= a.M) continue;
    const f32x4 y = total(t * MT + v);
    stream_store<EPI>(a, split, m, stream_column<EPI>(nb) + 4 * g, y, GLU ? total((t + 1) * MT + v) : y);
  }
}

template <int MT, int NT, int WK, int D, int EPI, bool JOIN>
__global__ void __launch_bounds__(256 * WK) linear_wave_n_kernel(const slm_linear_args a, const JoinArgs<JOIN> j) {
  constexpr bool GLU = EPI == SLM_LIN_GLU;
  static_assert(!JOIN || EPI == SLM_LIN_STORE, "joined products are stored");
  constexpr int GROUP = MT * 16 * 128;    // bytes of a group's step of x in LDS: 16-byte chunk c of row r lies in slot c ^ (r & 7)
  constexpr int AHEAD = MT < 3 ? 1 : NT == 1 ? 3 : 2;
  constexpr int XU = MT * 16 * 8 / 256;   // 16-byte units a thread stages
  constexpr int XB = WK * GROUP, PART = 4 * NT * MT * 1024;
  constexpr int PARTS = (WK - 1) * PART > (GLU && NT == 1 ? PART : 0) ? (WK - 1) * PART : (GLU && NT == 1 ? PART : 0);
  static_assert(MT >= 2 && D % 2 == 0 && (!GLU || NT < 3), "tiles");
  __shared__ __attribute__((aligned(16))) char lds[2 * XB > PARTS ? 2 * XB : PARTS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4, wn = wave & 3, kg = wave >> 2;
  const int split = blockIdx.z;
  const int64_t nb0 = (int64_t)blockIdx.x * (4 * NT) + wn * NT, m0 = (int64_t)blockIdx.y * (16 * MT), blocks = a.N >> 4;
  const bf16* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wp[t] = stream_block(a, min(nb0 + t, blocks - 1), lane);
  const int steps = (int)(a.K >> 6), per = (steps + a.n_splits - 1) / a.n_splits;
  const int s0 = split * per, s1 = min(steps, s0 + per), cnt = s1 - s0;
  const int its = (max(cnt, 0) + WK - 1) / WK;
  const bf16* xp[XU];
  uint32_t xd[XU];
  int xk[XU];
#pragma unroll
  for (int i = 0; i < XU; ++i) {
    const int u = tid + 256 * WK * i, r = u / (8 * WK), c = u % (8 * WK);
    xp[i] = reinterpret_cast<const bf16*>(a.x) + min(m0 + r, a.M - 1) * a.ldx;
    xk[i] = 8 * c;
    xd[i] = c / 8 * GROUP + r * 128 + ((c ^ r) & 7) * 16;
  }
  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int v = 0; v < MT; ++v) acc[t][v] = f32x4{0.f, 0.f, 0.f, 0.f};
  StreamK w[D][NT];
  u32x4 x[D][XU];
  auto load_x = [&](int u, int t, int i) {   // (a group past the last step reads that step again: not multiplied)
    x[u][t] = *reinterpret_cast<const u32x4*>(xp[t] + min(((s0 + i * WK) << 6) + xk[t], (int)a.K - 8));
  };
  auto load_w = [&](int u, int t, int i) {
    stream_load_w(w[u][t], wp[t] + (int64_t)min(s0 + i * WK + kg, steps - 1) * STREAM_STEP);
  };
  auto put = [&](int u, int t, int buf) { *reinterpret_cast<u32x4*>(lds + buf * XB + xd[t]) = x[u][t]; };
  // Fragments are read ahead of their products, loads and the next step's x go between them, one or two at a time: a wave that reads, waits
  // and multiplies in turn, and asks for all its loads at the end, waits for LDS and the address unit most of a step (128 rows, 28672 x 4096 / 14336
  // -> 4096 / 6752 x 4096: 51.2 / 33.9 / 35.3 us; fragments ahead 49.2 / 32.8 / 33.1; rows of LDS without a conflict, where 144-byte ones took 12
  // cycles a read instead of 4, 47.9 / 31.3 / 29.3; loads between the products 47.3 / 29.8 / 28.0).
  StreamK f[AHEAD + 1];
  const int fragment[2] = {kg * GROUP + r16 * 128 + ((g ^ r16) & 7) * 16, kg * GROUP + r16 * 128 + (((4 + g) ^ r16) & 7) * 16};
  auto fetch = [&](int v, int buf) {
#pragma unroll
    for (int h = 0; h < 2; ++h) f[v % (AHEAD + 1)].v[h] = *reinterpret_cast<const bf16x8_t*>(lds + buf * XB + v * 2048 + fragment[h]);
  };
  // step i + u: its products; between them the next step's x is written, x of D steps on and w of D - 1 steps on are asked for
  auto step = [&](int u, int i, bool mine, bool more) {
    constexpr int U = D - 1;
    if (mine) {
#pragma unroll
      for (int v = 0; v < AHEAD; ++v) fetch(v, u & 1);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int v = 0; v < MT; ++v) {
      if (mine && v + AHEAD < MT) fetch(v + AHEAD, u & 1);
#pragma unroll
      for (int t = v * XU / MT; t < (v + 1) * XU / MT; ++t) {
        if (more) load_x(u, t, min(i + u + D, its - 1));
        put((u + 1) % D, t, (u + 1) & 1);
      }
#pragma unroll
      for (int t = v * NT / MT; t < (v + 1) * NT / MT; ++t)
        if (more) load_w((u + U) % D, t, min(i + u + U, its - 1));
      __builtin_amdgcn_sched_barrier(0);
      if (mine) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[t][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][t].v[h], f[v % (AHEAD + 1)].v[h], acc[t][v], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  if (its > 0) {
    // One barrier a step: the next step's x is written while this one's is read; the buffer it goes to was last read
    // in front of the previous barrier.
#pragma unroll
    for (int u = 0; u < D; ++u) {
#pragma unroll
      for (int t = 0; t < XU; ++t) load_x(u, t, min(u, its - 1));
      if (u < D - 1) {
#pragma unroll
        for (int t = 0; t < NT; ++t) load_w(u, t, min(u, its - 1));
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < XU; ++t) put(0, t, 0);
    lds_barrier();
    int i = 0;
    for (; i + D < its; i += D) {
#pragma unroll
      for (int u = 0; u < D; ++u) {
        step(u, i, true, true);
        lds_barrier();
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) load_w(D - 1, t, min(i + D - 1, its - 1));
#pragma unroll
    for (int u = 0; u < D; ++u) {
      if (i + u < its) {
        step(u, i, (i + u) * WK + kg < cnt, false);
        lds_barrier();
      }
    }
  }
  f32x4* part = reinterpret_cast<f32x4*>(lds);
  if constexpr (WK > 1) {
    __syncthreads();
    if (kg > 0) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int v = 0; v < MT; ++v) part[(((kg - 1) * 4 + wn) * NT * MT + t * MT + v) * 64 + lane] = acc[t][v];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int q = 0; q < WK - 1; ++q)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int v = 0; v < MT; ++v) acc[t][v] += part[((q * 4 + wn) * NT * MT + t * MT + v) * 64 + lane];
    }
  }
  if constexpr (GLU && NT == 1) {   // the odd waves hold the up halves of the even ones' gates
    __syncthreads();
    if (kg == 0 && (wn & 1)) {
#pragma unroll
      for (int v = 0; v < MT; ++v) part[(wn * MT + v) * 64 + lane] = acc[0][v];
    }
    __syncthreads();
    if (wn & 1) return;
  }
  if constexpr (JOIN) {
    f32x4 (&flat)[NT * MT] = reinterpret_cast<f32x4 (&)[NT * MT]>(acc);
    if (!stream_join(flat, j, split, a.n_splits, tid, reinterpret_cast<uint32_t*>(lds))) return;
  }
  if (kg > 0) return;
#pragma unroll
  for (int t = 0; t < NT; t += (GLU && NT > 1 ? 2 : 1)) {
    const int64_t nb = nb0 + t;
    if (nb >= blocks) continue;
#pragma unroll
    for (int v = 0; v < MT; ++v) {
      const int64_t m = m0 + 16 * v + r16;
      f32x4 up = acc[t][v];
      if constexpr (GLU && NT == 1) up = part[((wn + 1) * MT + v) * 64 + lane];
      else if constexpr (GLU) up = acc[t + 1][v];
      if (m < a.M) stream_store<EPI>(a, split, m, stream_column<EPI>(nb) + 4 * g, acc[t][v], up);
    }
  }
}

// column tiles of 16 per NT; the grid's x extent
static int64_t stream_tiles(const slm_linear_args& a, int per) { return (a.N / 16 + per - 1) / per; }

// (one row of tiles: M <= 128, joined products)
template <int MT, int NT, int D, int EPI>
static int wave_k_launch(const slm_linear_args& a, hipStream_t st, const StreamJoin* j) {
  const dim3 grid((unsigned)stream_tiles(a, NT), (unsigned)((a.M + 16 * MT - 1) / (16 * MT)), (unsigned)a.n_splits);
  if constexpr (EPI == SLM_LIN_STORE && MT == 2) {
    if (j) {
      linear_wave_k_kernel<MT, NT, D, EPI, true><<<grid, dim3(256), 0, st>>>(a, *j);
      return hip_check_launch();
    }
  }
  linear_wave_k_kernel<MT, NT, D, EPI, false><<<grid, dim3(256), 0, st>>>(a, NoJoin{});
  return hip_check_launch();
}
template <int MT, int NT, int WK, int D, int EPI>
static int wave_n_launch(const slm_linear_args& a, hipStream_t st, const StreamJoin* j) {
  const dim3 grid((unsigned)stream_tiles(a, 4 * NT), (unsigned)((a.M + 16 * MT - 1) / (16 * MT)), (unsigned)a.n_splits);
  if constexpr (EPI == SLM_LIN_STORE) {
    if (j) {
      linear_wave_n_kernel<MT, NT, WK, D, EPI, true><<<grid, dim3(256 * WK), 0, st>>>(a, *j);
      return hip_check_launch();
    }
  }
  linear_wave_n_kernel<MT, NT, WK, D, EPI, false><<<grid, dim3(256 * WK), 0, st>>>(a, NoJoin{});
  return hip_check_launch();
}

// Up to 16 rows the widest tile whose workgroups leave no round of the 256 CUs more than a quarter empty: fewer, longer
// runs (28672 columns, 1 row: NT 4 37.7 us, NT 1 45; 16896 columns, a second round of 8 workgroups: 32 against 29.3).
// With more rows the columns of a wave weigh against the rounds they need, ties to the wider (x is read half as often):
// 64 rows x 28672 x 4096 41 us against 48, 64 rows x 16384 x 2048 20.6 against 15.7.  Up to 32 rows and under 112 panels the chip is
// filled by 32-column tiles (6784 columns: 15.6 us against 18.4).
template <int EPI>
static int stream_shape(const slm_linear_args& a, hipStream_t st, const StreamJoin* j = nullptr) {
  constexpr bool GLU = EPI == SLM_LIN_GLU;
  const int64_t s = a.n_splits;
  auto full = [&](int nt) {
    const int64_t w = stream_tiles(a, nt) * s;
    return 4 * w >= 3 * 256 * ((w + 255) / 256);
  };
  if (a.M <= 16) {
    if (full(4)) return wave_k_launch<1, 4, 3, EPI>(a, st, j);
    if constexpr (!GLU) {
      if (!full(2)) return wave_k_launch<1, 1, 8, EPI>(a, st, j);
    }
    return wave_k_launch<1, 2, 4, EPI>(a, st, j);
  }
  const int64_t rounds1 = (stream_tiles(a, 4) * s + 255) / 256, rounds2 = (stream_tiles(a, 8) * s + 255) / 256;
  const bool wide = 2 * rounds2 <= rounds1;
  if (a.M <= 32) {
    if (stream_tiles(a, 4) * s < 112) return wave_k_launch<2, 2, 4, EPI>(a, st, j);
    return wide ? wave_n_launch<2, 2, 1, 4, EPI>(a, st, j) : wave_n_launch<2, 1, 2, 4, EPI>(a, st, j);
  }
  if (a.M <= 64) return wide ? wave_n_launch<4, 2, 1, 4, EPI>(a, st, j) : wave_n_launch<4, 1, 1, 4, EPI>(a, st, j);
  if (a.M <= 96) return wide ? wave_n_launch<6, 2, 1, 4, EPI>(a, st, j) : wave_n_launch<6, 1, 1, 4, EPI>(a, st, j);
  return wide ? wave_n_launch<8, 2, 2, 2, EPI>(a, st, j) : wave_n_launch<8, 1, 1, 4, EPI>(a, st, j);
}

// A thread moves 16 bytes; a wave writes 1 KB and reads 16 half lines whose other halves the next wave reads (once per
// weight at load: 0.9 GB in 0.6 ms, where a strided copy of the tensor takes 6).
__global__ void __launch_bounds__(256) stream_layout_kernel(u32x4* out, const bf16* w, int64_t N, int64_t K, int64_t units, int glu) {
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (u >= units) return;
  const int lane = (int)(u & 63), h = (int)(u >> 6) & 1, block = (int)(u >> 7) & 3;
  const int64_t rest = u >> 9, steps = K >> 6, step = rest % steps, nb = rest / steps * 4 + block;
  const int64_t row = (glu ? (nb & 1) * (N / 2) + (nb >> 1) * 16 : nb * 16) + (lane & 15);
  out[u] = row < N ? *reinterpret_cast<const u32x4*>(w + row * K + step * 64 + h * 32 + (lane >> 4) * 8) : u32x4{0u, 0u, 0u, 0u};
}

}  // namespace slm

using namespace slm;

extern "C" SLM_API int slm_stream_layout(void* out, const void* w, int64_t N, int64_t K, int32_t glu, void* stream) {
  if (!out || !w || N <= 0 || K <= 0 || N % 16 || K % 64 || (glu && N % 64)) return SLM_ERR_INVALID_ARG;
  if (!aligned16(out) || !aligned16(w)) return SLM_ERR_ALIGNMENT;
  const int64_t units = (N + 63) / 64 * 64 * (K / 8);
  if (units > 256ll * 0x7fffffff) return SLM_ERR_UNSUPPORTED;
  hip_clear_error();
  stream_layout_kernel<<<dim3((unsigned)((units + 255) / 256)), dim3(256), 0, (hipStream_t)stream>>>((u32x4*)out, (const bf16*)w, N, K, units, glu);
  return hip_check_launch();
}

static int stream_check(const slm_linear_args* a, bool join = false) {
  if (!a || !a->x || !a->w || !a->y || a->M < 0 || a->N <= 0 || a->K <= 0 || a->K % 64 || a->N % 16 || a->batch != 1 ||
      a->n_splits < 1 || a->ldx < a->K || a->epilogue < 0 || a->epilogue > SLM_LIN_GLU)
    return SLM_ERR_INVALID_ARG;
  const bool glu = a->epilogue == SLM_LIN_GLU;
  if ((glu && a->N % 64) || (a->n_splits > 1 && a->epilogue != SLM_LIN_SLABS && !join)) return SLM_ERR_INVALID_ARG;
  if (a->ldy < (glu ? a->N / 2 : a->N)) return SLM_ERR_INVALID_ARG;
  if (a->dtype != SLM_BF16 || a->K > (1 << 28) || a->N > (1 << 30) || a->M > (1 << 20) || a->n_splits > 65535) return SLM_ERR_UNSUPPORTED;
  return a->ldx % 8 || !aligned16(a->x) || !aligned16(a->w) ? SLM_ERR_ALIGNMENT : SLM_OK;
}
extern "C" SLM_API int slm_linear_stream(const slm_linear_args* a, void* stream) {
  const int rc = stream_check(a);
  if (rc != SLM_OK || a->M == 0) return rc;
  hip_clear_error();
  hipStream_t st = (hipStream_t)stream;
  switch (a->epilogue) {
    case SLM_LIN_STORE: return stream_shape<SLM_LIN_STORE>(*a, st);
    case SLM_LIN_F32: return stream_shape<SLM_LIN_F32>(*a, st);
    case SLM_LIN_SLABS: return stream_shape<SLM_LIN_SLABS>(*a, st);
    default: return stream_shape<SLM_LIN_GLU>(*a, st);
  }
}

// Joined products: STORE, 17 to 128 rows, at most SLM_STREAM_TICKETS tiles of 32 columns
static bool stream_join_ok(const slm_linear_args* a) {
  return a->epilogue == SLM_LIN_STORE && a->M > 16 && a->M <= 128 && a->n_splits <= 16 && stream_tiles(*a, 2) <= SLM_STREAM_TICKETS;
}
extern "C" SLM_API size_t slm_linear_stream_join_bytes(const slm_linear_args* a) {
  if (stream_check(a, true) != SLM_OK || !stream_join_ok(a)) return 0;
  const int64_t rows = a->M <= 32 ? 32 : a->M <= 64 ? 64 : a->M <= 96 ? 96 : 128;
  return (size_t)(a->n_splits * rows * stream_tiles(*a, 8) * 128 * 4);   // (whole tiles of up to 128 columns)
}
extern "C" SLM_API int slm_linear_stream_join(const slm_linear_args* a, void* workspace, size_t workspace_bytes, uint32_t* tickets, void* stream) {
  const int rc = stream_check(a, true);
  if (rc != SLM_OK) return rc;
  if (!stream_join_ok(a)) return SLM_ERR_UNSUPPORTED;
  if (!tickets || !workspace || workspace_bytes < slm_linear_stream_join_bytes(a)) return SLM_ERR_WORKSPACE;
  if (!aligned16(workspace)) return SLM_ERR_ALIGNMENT;
  const StreamJoin j{(float*)workspace, tickets};
  hip_clear_error();
  return stream_shape<SLM_LIN_STORE>(*a, (hipStream_t)stream, &j);
}
