// latent_prefill.hip -- attention of prompt portions with latent attention in its expanded form: the latent rows
// a portion can see are gathered and multiplied by W_uk / W_uv once (a plain product), and the portion runs as
// ordinary multi-head attention with unequal query / value widths, causal and windowed, output gate fused.
//
// Work item: one workgroup = (tile of 128 query rows of one sequence, head), prompt_attn.h.  K row = unrotated part (per head) |
// rotated part (shared by the heads, out of the gathered latent rows).
#include "prompt_attn.h"

namespace slm {

struct LatentPrefillK {
  slm_latent_prefill_args a;
  float scale2;
};

template <int DQ, int VP, int GROUPS, int KEYS>
struct LatentWork {
  const LatentPrefillK& p;
  const int lane, group;
  int ctx0, lo, hi, groups, n_turns, q_chunks;
  int qpos, klo, wq0, wq1;          // in context indexes: the lane's row, the first key of its window; the wave's rows
  const bf16 *kv, *ctx;
  int kv_w, ctx_w;                  // bytes of a row

  __device__ __forceinline__ int start_of(int turn) const { return lo + (groups * turn + group) * KEYS; }
  __device__ __forceinline__ int row(int turn, int r) const { return ctx0 + min(start_of(turn) + r, hi - 1); }
  __device__ __forceinline__ const void* key(int at, int c) const {
    const bool own = c < q_chunks;                     // per head, or shared by the heads
    return reinterpret_cast<const char*>((own ? kv : ctx - 8 * q_chunks) + 8 * c) + (int64_t)at * (own ? kv_w : ctx_w);
  }
  __device__ __forceinline__ const void* value(int at, int c) const {
    return reinterpret_cast<const char*>(kv + 8 * (q_chunks + c)) + (int64_t)at * kv_w;
  }
  __device__ __forceinline__ void start() {}
  __device__ __forceinline__ void begin(int) {}
  __device__ __forceinline__ void end(int) {}
  // tiles no row of the wave sees: past its diagonal, before its window
  __device__ __forceinline__ bool seen(int turn) const {
    const int k0 = start_of(turn);
    return k0 <= wq1 && (p.a.window <= 0 || k0 + KEYS > wq0 - p.a.window + 1);
  }
  __device__ __forceinline__ void mask(int turn, f32x16 (&s)[KEYS / 32]) const {
    const int k0 = start_of(turn);
    if (k0 + KEYS - 1 <= wq0 && (p.a.window <= 0 || k0 >= wq1 - p.a.window + 1)) return;
    const int at = k0 + 4 * (lane >> 5), last = qpos - at, from = klo - at;
#pragma unroll
    for (int n = 0; n < KEYS / 32; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int k = 32 * n + 8 * (r >> 2) + (r & 3);
        s[n][r] = (k > last) | (k < from) ? -INFINITY : s[n][r];
      }
  }
  __device__ __forceinline__ float score(float x) const { return x; }
  __device__ __forceinline__ float top(float x) const { return x * p.scale2; }
  __device__ __forceinline__ float below(float x, float m) const { return __builtin_fmaf(x, p.scale2, -m); }
};

// Waves of a SIMD: a third for 64 + 64 columns, whose registers are six too many for it otherwise (32 heads, us, two / three: 4 prompts of 1100 to 2047 68.5 /
// 62.3, 16 x 512 rows by a window of 512 84 / 76)
constexpr int latent_waves(int dq, int vp, int groups) { return groups == 1 && dq + vp <= 128 ? 3 : 2; }

template <int DQ, int VP, int GROUPS>
__global__ void __launch_bounds__(256 * GROUPS) __attribute__((amdgpu_waves_per_eu(latent_waves(DQ, VP, GROUPS))))
latent_prefill_kernel(const LatentPrefillK p) {
  constexpr int QS = DQ / 16, DT = VP / 32;
  // two workgroups on a CU, or two groups of waves: at most 80 KB each (256 + 128 columns: 112 us with 64 keys, 84 with 32)
  constexpr int KEYS = DQ + VP > 320 ? 32 : 64;
  __shared__ __attribute__((aligned(1024))) char lds[prompt_lds_bytes<DQ, VP, GROUPS, KEYS>()];

  const slm_latent_prefill_args& a = p.a;
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = GROUPS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int l31 = lane & 31, hh = lane >> 5;
  // heads fastest: the query tiles of one head stay on one XCD (heads % 8 == 0) and share its keys in L2;
  // tiles come longest first from the host
  const int head = blockIdx.x % a.heads;
  const int32_t* td = a.tiles + 6 * (blockIdx.x / a.heads);
  const int row0 = td[0], n_rows = td[1], ctx0 = td[2], ctx_len = td[3], ctx_pos = td[4], pos0 = td[5];
  const int qi = min(wave * 32 + l31, n_rows - 1);     // this lane's query row

  LatentWork<DQ, VP, GROUPS, KEYS> w{p, lane, group};
  // visible keys of the tile, as indexes into its context
  w.ctx0 = ctx0, w.lo = 0, w.hi = min(ctx_len, pos0 + n_rows - ctx_pos);
  if (a.window > 0) w.lo = max(0, pos0 - a.window + 1 - ctx_pos);
  const int n_tiles = (w.hi - w.lo + KEYS - 1) / KEYS;
  w.groups = prompt_groups<GROUPS>(n_tiles), w.n_turns = (n_tiles + w.groups - 1) / w.groups;
  w.q_chunks = a.q_dim / 8;
  w.qpos = pos0 + qi - ctx_pos;
  w.klo = a.window > 0 ? max(0, w.qpos - a.window + 1) : 0;
  w.wq0 = pos0 - ctx_pos + min(wave * 32, n_rows - 1), w.wq1 = pos0 - ctx_pos + min(wave * 32 + 31, n_rows - 1);
  w.kv = reinterpret_cast<const bf16*>(a.kv) + (int64_t)head * (a.q_dim + a.v_pad);
  w.ctx = reinterpret_cast<const bf16*>(a.ctx) + a.c_pad;
  w.kv_w = a.heads * (a.q_dim + a.v_pad) * 2, w.ctx_w = (a.c_pad + a.r_pad) * 2;

  const bf16* qrow = reinterpret_cast<const bf16*>(a.q) + (int64_t)(row0 + qi) * a.ld_q;
  bf16x8_t qf[QS];
  {
    const bf16* q = qrow + head * DQ + 8 * hh;
#pragma unroll
    for (int s = 0; s < QS; ++s) qf[s] = *reinterpret_cast<const bf16x8_t*>(q + 16 * s);
  }
  f32x16 o[DT];
  float m_run, l_run;
  prompt_attention<DQ, VP, GROUPS, KEYS>(w, lds, qf, o, m_run, l_run);
  if (group || wave * 32 + l31 >= n_rows) return;
  const float f = sigmoid_f32((float)reinterpret_cast<const bf16*>(a.gate)[(int64_t)(row0 + qi) * a.ld_q + a.gate_off + head]) / l_run;
  bf16* out = reinterpret_cast<bf16*>(a.out) + (int64_t)(row0 + qi) * a.ld_out + head * VP + 4 * hh;
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<u32x2*>(out + 32 * d + 2 * r) = u32x2{pack2<bf16_tag>(o[d][r] * f, o[d][r + 1] * f),
                                                              pack2<bf16_tag>(o[d][r + 2] * f, o[d][r + 3] * f)};
}

static bool lp_ok(int dq, int vp) {
  const bool q = dq == 64 || dq == 96 || dq == 128 || dq == 160 || dq == 192 || dq == 256;
  return q && (vp == 32 || vp == 64 || vp == 128) ;
}
template <int DQ, int VP>
static void lp_launch(const LatentPrefillK& p, hipStream_t st) {
  const int64_t workgroups = (int64_t)p.a.n_tiles * p.a.heads;
  if (prompt_two_groups(workgroups, p.a.n_ctx, p.a.n_tiles, p.a.window)) latent_prefill_kernel<DQ, VP, 2><<<dim3((unsigned)workgroups), dim3(512), 0, st>>>(p);
  else latent_prefill_kernel<DQ, VP, 1><<<dim3((unsigned)workgroups), dim3(256), 0, st>>>(p);
}
template <int DQ>
static void lp_v(const LatentPrefillK& p, hipStream_t st) {
  switch (p.a.v_pad) {
    case 32: lp_launch<DQ, 32>(p, st); break;
    case 64: lp_launch<DQ, 64>(p, st); break;
    default: lp_launch<DQ, 128>(p, st);
  }
}

}  // namespace slm

using namespace slm;

extern "C" SLM_API int slm_latent_prefill_supported(int32_t q_dim, int32_t r_pad, int32_t v_pad) {
  return q_dim > 0 && q_dim % 8 == 0 && r_pad % 8 == 0 && lp_ok(q_dim + r_pad, v_pad) ? 1 : 0;
}
extern "C" SLM_API int slm_latent_prefill(const slm_latent_prefill_args* a, void* stream) {
  if (!a || !a->q || !a->ctx || !a->kv || !a->gate || !a->out || !a->tiles || a->n_tiles < 0 || a->heads < 1 ||
      a->n_rows < 0 || a->n_ctx < 0)
    return SLM_ERR_INVALID_ARG;
  if (!slm_latent_prefill_supported(a->q_dim, a->r_pad, a->v_pad)) return SLM_ERR_UNSUPPORTED;
  if (a->ld_q < (int64_t)a->heads * (a->q_dim + a->r_pad) || a->ld_out < (int64_t)a->heads * a->v_pad || a->ld_q % 8 ||
      a->ld_out % 4 || a->c_pad % 8 || !aligned16(a->q) || !aligned16(a->ctx) || !aligned16(a->kv) || !aligned16(a->out))
    return SLM_ERR_ALIGNMENT;
  if (a->n_tiles == 0) return SLM_OK;
  LatentPrefillK p;
  p.a = *a;
  p.scale2 = a->scale * LOG2E_F;
  hip_clear_error();
  switch (a->q_dim + a->r_pad) {
    case 64: lp_v<64>(p, (hipStream_t)stream); break;
    case 96: lp_v<96>(p, (hipStream_t)stream); break;
    case 128: lp_v<128>(p, (hipStream_t)stream); break;
    case 160: lp_v<160>(p, (hipStream_t)stream); break;
    case 192: lp_v<192>(p, (hipStream_t)stream); break;
    default: lp_v<256>(p, (hipStream_t)stream);
  }
  return hip_check_launch();
}
