// linear.hip -- y = x W^T for few rows (decode batches, the vocabulary projection of the sampled rows), and
// for every row count in 32-bit.  Bound: the HBM stream of W.
//
// A workgroup of four waves owns NT blocks of 16 output columns and MT blocks of 16 rows of x and splits K
// over its waves (and over blockIdx for SLABS).  Per step of 64 a lane (r = lane % 16, g = lane / 16) reads
// the 16 consecutive k of row r that start at 16 g -- the four lane groups of a row read one whole 128-byte
// line in bf16 -- and feeds them to the MFMAs in an order of k that is the same for both operands, so no
// shuffle is needed.  The waves' partial tiles meet in LDS; the epilogue runs there.
#include "latent_append.h"

namespace slm {

template <typename E>
struct KStep;  // 64 k of one 16-row block: what a lane holds
template <>
struct KStep<bf16> {
  bf16x8_t v[2];
  __device__ __forceinline__ void load(const bf16* p) {
    v[0] = *reinterpret_cast<const bf16x8_t*>(p);
    v[1] = *reinterpret_cast<const bf16x8_t*>(p + 8);
  }
  __device__ __forceinline__ void zero() {
    v[0] = __builtin_bit_cast(bf16x8_t, u32x4{0u, 0u, 0u, 0u});
    v[1] = v[0];
  }
  static __device__ __forceinline__ f32x4 mma(const KStep& a, const KStep& b, f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v[0], b.v[0], c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v[1], b.v[1], c, 0, 0, 0);
  }
};
template <>
struct KStep<float> {
  f32x4 v[4];
  __device__ __forceinline__ void load(const float* p) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const f32x4*>(p + 4 * i);
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  static __device__ __forceinline__ f32x4 mma(const KStep& a, const KStep& b, f32x4 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[i][j], b.v[i][j], c, 0, 0, 0);
    return c;
  }
};

// GLU: the NT blocks are NT / 2 pairs (gate block, up block half columns further)
template <typename E, int MT, int NT, int U, int EPI>
__device__ __forceinline__ void linear_block(const slm_linear_args& a, const int z) {
  constexpr bool GLU = EPI == SLM_LIN_GLU;
  constexpr int NOUT = GLU ? NT / 2 : NT;  // output column blocks
  static_assert(!GLU || NT % 2 == 0, "gate / up pairs");
  __shared__ f32x4 red[4][NT * MT][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int item = z / a.n_splits, split = z % a.n_splits;
  const int64_t half = a.N / 2;
  const int64_t n_out = GLU ? half : a.N;
  const int64_t n0 = (int64_t)blockIdx.x * (16 * NOUT), m0 = (int64_t)blockIdx.y * (16 * MT);

  const E* wp[NT];
  const E* xp[MT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    int64_t n = GLU ? n0 + 16 * (t >> 1) : n0 + 16 * t;
    n = min(n, n_out - 16) + r16 + (GLU ? (t & 1) * half : 0);  // (a block past the end re-reads the last: not stored)
    wp[t] = reinterpret_cast<const E*>(a.w) + item * a.w_batch + n * a.ldw + 16 * g;
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int64_t m = min(m0 + 16 * t + r16, a.M - 1);
    xp[t] = reinterpret_cast<const E*>(a.x) + item * a.x_batch + m * a.ldx + 16 * g;
  }
  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int u = 0; u < MT; ++u) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int steps = (int)(a.K >> 6);
  const int per = (steps + a.n_splits - 1) / a.n_splits;
  const int s0 = split * per, s1 = min(steps, s0 + per);
  int s = s0 + wave;
  for (; s + 4 * (U - 1) < s1; s += 4 * U) {
    KStep<E> w[U][NT], x[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t k = (int64_t)(s + 4 * u) << 6;
#pragma unroll
      for (int t = 0; t < NT; ++t) w[u][t].load(wp[t] + k);
#pragma unroll
      for (int t = 0; t < MT; ++t) x[u][t].load(xp[t] + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int v = 0; v < MT; ++v) acc[t][v] = KStep<E>::mma(w[u][t], x[u][v], acc[t][v]);
  }
  if constexpr (U > 1) {
    for (; s < s1; s += 4) {
      const int64_t k = (int64_t)s << 6;
      KStep<E> x[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) x[t].load(xp[t] + k);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        KStep<E> w;
        w.load(wp[t] + k);
#pragma unroll
        for (int v = 0; v < MT; ++v) acc[t][v] = KStep<E>::mma(w, x[v], acc[t][v]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int v = 0; v < MT; ++v) red[wave][t * MT + v][lane] = acc[t][v];
  __syncthreads();

  // thread = (column n of 16, row m of 16) of every tile; C layout: row n = 4 (lane / 16) + reg, column m = lane % 16
  const int n = tid & 15, m = tid >> 4;
  const int src = (n >> 2) * 16 + m, reg = n & 3;
  auto total = [&](int t) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) v += reinterpret_cast<const float*>(&red[w][t][src])[reg];
    return v;
  };
#pragma unroll
  for (int t = 0; t < NOUT; ++t) {
    const int64_t nn = n0 + 16 * t + n;
    if (nn >= n_out) continue;
#pragma unroll
    for (int v = 0; v < MT; ++v) {
      const int64_t mm = m0 + 16 * v + m;
      if (mm >= a.M) continue;
      if constexpr (EPI == SLM_LIN_SLABS) {
        reinterpret_cast<float*>(a.y)[((int64_t)split * a.M + mm) * a.ldy + nn] = total(t * MT + v);
      } else if constexpr (EPI == SLM_LIN_F32) {
        reinterpret_cast<float*>(a.y)[item * a.y_batch + mm * a.ldy + nn] = a.alpha * total(t * MT + v);
      } else if constexpr (EPI == SLM_LIN_GLU) {
        reinterpret_cast<E*>(a.y)[mm * a.ldy + nn] =
            (E)clamped_glu_f32(total(2 * t * MT + v), total((2 * t + 1) * MT + v), a.limit, a.glu_alpha, a.glu_shift);
      } else if constexpr (EPI == SLM_LIN_GATE) {
        const float gl = to_f32(reinterpret_cast<const E*>(a.gate)[mm * a.ld_gate + item]);
        reinterpret_cast<E*>(a.y)[item * a.y_batch + mm * a.ldy + nn] = (E)(total(t * MT + v) * sigmoid_f32(gl));
      } else {
        reinterpret_cast<E*>(a.y)[item * a.y_batch + mm * a.ldy + nn] = (E)total(t * MT + v);
      }
    }
  }
}

template <typename E, int MT, int NT, int U, int EPI>
__global__ void __launch_bounds__(256) linear_kernel(const slm_linear_args a) {
  linear_block<E, MT, NT, U, EPI>(a, blockIdx.z);
}
// The first `slices` of the grid write a row of the latent cache per workgroup: neither part reads what the other writes.
template <int MT, int NT, int U>
__global__ void __launch_bounds__(256) linear_append_kernel(const slm_linear_args a, const slm_latent_append_args c, const int slices) {
  if ((int)blockIdx.z >= slices) return linear_block<bf16, MT, NT, U, SLM_LIN_STORE>(a, blockIdx.z - slices);
  const int64_t row = ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
  if (row < c.rows) latent_append_row<bf16, 4>(c, row);
}

// The same where K is one head's queries and more than 32 rows come: a wave takes 64 rows x 32 columns and all of K, so that nothing meets in LDS, and a
// lane ends with eight neighbouring columns, one store of 16 bytes where linear_block has eight of two.  Row i of operand t is column 8 (i / 4) + i % 4 + 4 t;
// the order of k and of the sums is linear_block's: the same bits.
// Bound: the stores (128 rows of 32 heads: 4.7 MB).  us, linear_block / this: 32 heads of 128 -> 512 columns 48 rows 5.0 / 4.0, 128 rows 7.8 / 5.4; 16 heads
// 64 rows 4.0 / 4.1, 128 rows 5.1 / 4.3; 32 heads -> 256 128 rows 5.1 / 4.3; but 16 heads -> 128 128 rows 3.8 / 4.0.
template <int KS>   // K / 64
__global__ void __launch_bounds__(256) linear_append_heads_kernel(const slm_linear_args a, const slm_latent_append_args c, const int slices) {
  if ((int)blockIdx.z < slices) {
    const int64_t row = ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    if (row < c.rows) latent_append_row<bf16, 4>(c, row);
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
  const int64_t item = blockIdx.z - slices, n0 = (int64_t)blockIdx.x * 128 + wave * 32, m0 = (int64_t)blockIdx.y * 64;
  const bf16* w = reinterpret_cast<const bf16*>(a.w) + item * a.w_batch + (n0 + 8 * (r16 >> 2) + (r16 & 3)) * a.ldw + 16 * g;
  const bf16* x = reinterpret_cast<const bf16*>(a.x) + item * a.x_batch + 16 * g;
  KStep<bf16> wf[2][KS], xf[4][KS];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int s = 0; s < KS; ++s) wf[t][s].load(w + 4 * t * a.ldw + 64 * s);
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int s = 0; s < KS; ++s) xf[m][s].load(x + min(m0 + 16 * m + r16, a.M - 1) * a.ldx + 64 * s);
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    f32x4 y[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      y[t] = KStep<bf16>::mma(wf[t][0], xf[m][0], f32x4{0.f, 0.f, 0.f, 0.f});
      if constexpr (KS == 2) y[t] += KStep<bf16>::mma(wf[t][1], xf[m][1], f32x4{0.f, 0.f, 0.f, 0.f});
    }
    const int64_t row = m0 + 16 * m + r16;
    if (row < a.M)
      *reinterpret_cast<u32x4*>(reinterpret_cast<bf16*>(a.y) + item * a.y_batch + row * a.ldy + n0 + 8 * g) =
          u32x4{pack2<bf16_tag>(y[0][0], y[0][1]), pack2<bf16_tag>(y[0][2], y[0][3]), pack2<bf16_tag>(y[1][0], y[1][1]), pack2<bf16_tag>(y[1][2], y[1][3])};
  }
}
static bool append_heads_ok(const slm_linear_args& a) {
  return a.M > 32 && (a.K == 64 || a.K == 128) && a.N % 128 == 0 && a.ldy % 8 == 0 && a.y_batch % 8 == 0 && aligned16(a.y) && a.M <= 256 && a.N * a.batch >= 8192;
}
static int append_heads_launch(const slm_linear_args& a, const slm_latent_append_args& c, hipStream_t st) {
  const int64_t gx = a.N / 128, gy = (a.M + 63) / 64, slices = (c.rows + gx * gy - 1) / (gx * gy);
  if (a.batch + slices > 65535) return SLM_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)(a.batch + slices));
  hip_clear_error();
  if (a.K == 64) linear_append_heads_kernel<1><<<grid, dim3(256), 0, st>>>(a, c, (int)slices);
  else linear_append_heads_kernel<2><<<grid, dim3(256), 0, st>>>(a, c, (int)slices);
  return hip_check_launch();
}

template <typename E, int MT, int NT, int U, int EPI>
static int lin_launch(const slm_linear_args& a, hipStream_t st, const slm_latent_append_args* c) {
  constexpr int NOUT = EPI == SLM_LIN_GLU ? NT / 2 : NT;
  const int64_t n_out = EPI == SLM_LIN_GLU ? a.N / 2 : a.N;
  const int64_t gx = (n_out + 16 * NOUT - 1) / (16 * NOUT), gy = (a.M + 16 * MT - 1) / (16 * MT);
  const int64_t gz = (int64_t)a.batch * a.n_splits;
  if (gx > 0x7fffffff || gy > 65535 || gz > 65535) return SLM_ERR_UNSUPPORTED;
  hip_clear_error();
  if constexpr (sizeof(E) == 2 && EPI == SLM_LIN_STORE) {
    if (c) {
      const int64_t slices = (c->rows + gx * gy - 1) / (gx * gy);
      if (gz + slices > 65535) return SLM_ERR_UNSUPPORTED;
      linear_append_kernel<MT, NT, U><<<dim3((unsigned)gx, (unsigned)gy, (unsigned)(gz + slices)), dim3(256), 0, st>>>(a, *c, (int)slices);
      return hip_check_launch();
    }
  }
  linear_kernel<E, MT, NT, U, EPI><<<dim3((unsigned)gx, (unsigned)gy, (unsigned)gz), dim3(256), 0, st>>>(a);
  return hip_check_launch();
}
// Tiles by row count: one row block streams W with many steps in flight; with more rows the reads of x weigh as much
// as those of W, and wider column blocks (where enough of them are left to fill the chip) read x less often.
template <typename E, int EPI>
static int lin_shape(const slm_linear_args& a, hipStream_t st, const slm_latent_append_args* c = nullptr) {
  constexpr int P = EPI == SLM_LIN_GLU ? 2 : 1;
  if constexpr (sizeof(E) == 4) {
    if (a.M <= 16) return lin_launch<E, 1, P, 1, EPI>(a, st, c);
    return lin_launch<E, 2, 2, 1, EPI>(a, st, c);
  } else {
    if (a.M <= 4) return lin_launch<E, 1, P, 8 / P, EPI>(a, st, c);
    if (a.M <= 16) return lin_launch<E, 1, P, 4 / P, EPI>(a, st, c);
    const bool wide = a.N / 64 * a.batch * a.n_splits >= 256;
    if (a.M <= 32) return wide ? lin_launch<E, 2, 4, 1, EPI>(a, st, c) : lin_launch<E, 2, 2, 2, EPI>(a, st, c);
    return wide ? lin_launch<E, 4, 4, 1, EPI>(a, st, c) : lin_launch<E, 4, 2, 2, EPI>(a, st, c);
  }
}
template <typename E>
static int lin_epi(const slm_linear_args& a, hipStream_t st) {
  switch (a.epilogue) {
    case SLM_LIN_STORE: return lin_shape<E, SLM_LIN_STORE>(a, st);
    case SLM_LIN_F32: return lin_shape<E, SLM_LIN_F32>(a, st);
    case SLM_LIN_SLABS: return lin_shape<E, SLM_LIN_SLABS>(a, st);
    case SLM_LIN_GLU: return lin_shape<E, SLM_LIN_GLU>(a, st);
    default: return lin_shape<E, SLM_LIN_GATE>(a, st);
  }
}

int linear_check(const slm_linear_args* a) {
  if (!a || !a->x || !a->w || !a->y || a->M < 0 || a->N <= 0 || a->K <= 0 || a->K % 64 || a->N % 16 || a->batch < 1 ||
      a->n_splits < 1 || a->ldx < a->K || a->ldw < a->K || a->epilogue < 0 || a->epilogue > SLM_LIN_GATE)
    return SLM_ERR_INVALID_ARG;
  if (a->dtype != SLM_BF16 && a->dtype != SLM_F32) return SLM_ERR_UNSUPPORTED;
  const int64_t al = a->dtype == SLM_BF16 ? 8 : 4;
  if (a->ldx % al || a->ldw % al || a->x_batch % al || a->w_batch % al || !aligned16(a->x) || !aligned16(a->w))
    return SLM_ERR_ALIGNMENT;
  if (a->n_splits > 1 && (a->epilogue != SLM_LIN_SLABS || a->batch != 1)) return SLM_ERR_INVALID_ARG;
  if (a->epilogue == SLM_LIN_GLU && (a->N % 32 || a->batch != 1)) return SLM_ERR_INVALID_ARG;
  if (a->epilogue == SLM_LIN_SLABS && a->batch != 1) return SLM_ERR_INVALID_ARG;
  if (a->epilogue == SLM_LIN_GATE && !a->gate) return SLM_ERR_INVALID_ARG;
  return SLM_OK;
}

}  // namespace slm

using namespace slm;

extern "C" SLM_API int slm_linear(const slm_linear_args* a, void* stream) {
  const int rc = linear_check(a);
  if (rc != SLM_OK) return rc;
  if (a->M == 0) return SLM_OK;
  return a->dtype == SLM_BF16 ? lin_epi<bf16>(*a, (hipStream_t)stream) : lin_epi<float>(*a, (hipStream_t)stream);
}

// One launch where the rows leave the chip idle anyway: a launch that reads what the one in front of it wrote costs 4 us and more
// whatever it does.  (A step of four layers, latent 512, two launches / one: 1 row of 32 heads 493 / 479 us, 32 rows of 16 heads 386 / 369,
// 128 rows of 32 heads 1129 / 1124.)
// And only where the product reads no column that the rotation writes (K is the queries' unrotated width, without padding).
extern "C" SLM_API int slm_latent_append_absorb(const slm_latent_append_args* c, const slm_linear_args* a, void* stream) {
  const int rc = linear_check(a);
  if (rc != SLM_OK) return rc;
  if (latent_append_invalid(c)) return SLM_ERR_INVALID_ARG;
  if (a->epilogue != SLM_LIN_STORE || a->dtype != c->dtype) return SLM_ERR_INVALID_ARG;
  const bool apart = a->x == c->proj && a->ldx == c->ld_proj && a->K <= c->q_dim && a->x_batch == c->q_dim + c->q_rot && a->batch <= c->heads &&
                     c->q_abs && a->y == c->q_abs && a->N <= c->c_pad && a->y_batch == c->c_pad + c->r_pad && a->M <= c->abs_rows;
  if (apart && a->M > 0 && c->rows <= 256 && a->dtype == SLM_BF16 && latent_append_by_four(*c))
    return append_heads_ok(*a) ? append_heads_launch(*a, *c, (hipStream_t)stream) : lin_shape<bf16, SLM_LIN_STORE>(*a, (hipStream_t)stream, c);
  const int rd = slm_latent_append(c, stream);
  return rd != SLM_OK ? rd : slm_linear(a, stream);
}
