// window_prefill.hip -- windowed grouped-query attention of prompt portions on MFMA: kept first tokens, capped scores,
// a sink.  The portion's context is a list of cache slots (kept positions, then the window of its first row onwards).
//
// Work item: one workgroup = (tile of 128 query rows of one sequence, head), prompt_attn.h; tiles of 64 or 32 keys, those of the kept
// tokens, then those of the tile's own window.  The slots of a tile reach LDS three turns ahead of its keys.
#include "latent/prompt_attn.h"
#include "window_common.h"

namespace slm {

// Keys of a tile, and waves of a SIMD.  Beside the sums and queries of wide heads the scores of 32 keys leave room for a second wave, and the tiles for a
// second workgroup on the CU; at 256 + 256 there is none either way.  us, 64 keys and one wave / 32 and two, 16 heads, 4096 rows and 32 heads, 8 x 512 rows
// of 2200 to 3584: 192 + 128 173 / 144, 410 / 246; 96 + 192 179 / 140, 428 / 245; 64 + 256 195 / 149, 464 / 265; 192 + 256 228 / 247, 539 / 402.  (256 + 256, one wave:
// 64 keys 234, 556, 32 keys 323, 776.)
constexpr int window_keys(int columns) { return columns > 256 && columns < 512 ? 32 : 64; }
constexpr int window_waves(int columns) { return columns < 512 ? 2 : 1; }

template <int GROUPS, int KEYS, bool CAP>
struct WindowWork {
  const slm_window_prefill_args& a;
  int(*const slots)[KEYS];   // of four turns, the present one and the three to come
  const int wave, lane, group;
  int ctx0, n_keep, lo, hi, n_head, n_tiles, groups, n_turns, next;
  int qidx, klo, wq0, wq1;          // in context indexes: the lane's row, the first key of its window; the wave's rows
  const bf16 *kc, *vc;
  int k_w, v_w;                     // bytes of a cache row
  float factor, cap_k;

  __device__ __forceinline__ int tile_of(int turn) const { return groups * turn + group; }
  __device__ __forceinline__ int tile_start(int t) const { return t < n_head ? t * KEYS : lo + (t - n_head) * KEYS; }
  __device__ __forceinline__ int tile_end(int t) const { return t < n_head ? n_keep : hi; }
  __device__ __forceinline__ int slot_of(int turn) const {
    const int t = min(tile_of(turn), n_tiles - 1);
    return a.slots[ctx0 + min(tile_start(t) + (lane & (KEYS - 1)), tile_end(t) - 1)];
  }
  __device__ __forceinline__ int row(int turn, int r) const { return slots[turn & 3][r]; }
  __device__ __forceinline__ const void* key(int slot, int c) const { return reinterpret_cast<const char*>(kc + 8 * c) + (int64_t)slot * k_w; }
  __device__ __forceinline__ const void* value(int slot, int c) const { return reinterpret_cast<const char*>(vc + 8 * c) + (int64_t)slot * v_w; }
  __device__ __forceinline__ void keep(int turn, int slot) {
    if (KEYS == 64 || lane < KEYS) slots[turn & 3][lane] = slot;
  }
  __device__ __forceinline__ void start() {
    if (wave == 0)
      for (int i = 0; i < 3; ++i) keep(i, slot_of(i));
    __syncthreads();
  }
  __device__ __forceinline__ void begin(int turn) {
    if (wave == 0) next = slot_of(turn + 3);
  }
  __device__ __forceinline__ void end(int turn) {
    if (wave == 0) keep(turn + 3, next);
  }
  // tiles no row of the wave sees: past its diagonal, before its window
  __device__ __forceinline__ bool seen(int turn) const {
    const int t = tile_of(turn), k0 = tile_start(t);
    return t < n_tiles && k0 <= wq1 && (a.window <= 0 || k0 < n_keep || k0 + KEYS > wq0 - a.window + 1);
  }
  __device__ __forceinline__ void mask(int turn, f32x16 (&s)[KEYS / 32]) const {
    const int t = tile_of(turn), k0 = tile_start(t), k_end = tile_end(t);
    if (k0 + KEYS - 1 <= wq0 && k0 + KEYS <= k_end && (a.window <= 0 || k0 >= wq1 - a.window + 1)) return;
    const int at = k0 + 4 * (lane >> 5), last = min(qidx, k_end - 1) - at, from = klo - at, kept = n_keep - at;
#pragma unroll
    for (int n = 0; n < KEYS / 32; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int k = 32 * n + 8 * (r >> 2) + (r & 3);
        s[n][r] = (k > last) | ((k < from) & (k >= kept)) ? -INFINITY : s[n][r];
      }
  }
  // without a cap scale s; with one, cap tanh(s scale / cap) - cap = -2 cap / (1 + exp(2 s scale / cap)): the constant drops
  // out of the differences that the soft-max takes.  Log2 units.
  __device__ __forceinline__ float score(float x) const {
    const float y = x * factor;
    return CAP ? __builtin_amdgcn_rcpf(fmaf(fast_exp2(y), cap_k, cap_k)) : y;
  }
  __device__ __forceinline__ float top(float x) const { return x; }
  __device__ __forceinline__ float below(float x, float m) const { return x - m; }
};

template <int DQ, int VP, int GROUPS, bool CAP>
__global__ void __launch_bounds__(256 * GROUPS) __attribute__((amdgpu_waves_per_eu(window_waves(DQ + VP))))
window_prefill_kernel(const slm_window_prefill_args a) {
  constexpr int QS = DQ / 16, DT = VP / 32, KEYS = window_keys(DQ + VP);
  __shared__ __attribute__((aligned(1024))) char lds[prompt_lds_bytes<DQ, VP, GROUPS, KEYS>()];
  __shared__ int slots[GROUPS][4][KEYS];

  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = GROUPS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int l31 = lane & 31, hh = lane >> 5;
  // heads fastest, neighbours on one XCD (workgroup i goes to XCD i % 8): the heads that share keys run beside each other on
  // one L2, with the same query tile
  const int at = blockIdx.x % a.heads, head = a.heads % 8 ? at : (at & 7) * (a.heads >> 3) + (at >> 3), g = head / (a.heads / a.kv_heads);
  const int32_t* td = a.tiles + 7 * (blockIdx.x / a.heads);
  const int row0 = td[0], n_rows = td[1], ctx0 = td[2], ctx_len = td[3], kept = td[4], first = td[5], pos0 = td[6];
  const int shift = first - kept;                      // position = index + shift behind the kept tokens
  const int qi = min(wave * 32 + l31, n_rows - 1);     // this lane's query row

  WindowWork<GROUPS, KEYS, CAP> w{a, slots[group], wave, lane, group};
  // context indexes the tile needs: [0, n_keep) and [lo, hi)
  w.ctx0 = ctx0, w.hi = min(ctx_len, pos0 + n_rows - shift);
  w.n_keep = a.window > 0 ? min(max(a.keep_first, 0), w.hi) : 0;
  w.lo = a.window > 0 ? max(w.n_keep, pos0 - a.window + 1 - shift) : 0;
  w.n_head = (w.n_keep + KEYS - 1) / KEYS;   // tiles of the kept tokens
  if (w.lo == w.n_keep) w.lo = 0, w.n_head = 0;            // (one range)
  w.n_tiles = w.n_head + (w.hi - w.lo + KEYS - 1) / KEYS;
  w.groups = prompt_groups<GROUPS>(w.n_tiles);
  w.n_turns = (w.n_tiles + w.groups - 1) / w.groups;
  w.qidx = pos0 + qi - shift;
  w.klo = a.window > 0 ? w.qidx - a.window + 1 : 0;
  w.wq0 = pos0 - shift + min(wave * 32, n_rows - 1), w.wq1 = pos0 - shift + min(wave * 32 + 31, n_rows - 1);
  w.kc = reinterpret_cast<const bf16*>(a.key_cache) + (int64_t)g * DQ;
  w.vc = reinterpret_cast<const bf16*>(a.value_cache) + (int64_t)g * VP;
  w.k_w = a.kv_heads * DQ * 2, w.v_w = a.kv_heads * VP * 2;
  const float cap2 = CAP ? a.softcap * LOG2E_F : 0.f;
  w.factor = CAP ? 2.0f * LOG2E_F * a.scale / a.softcap : a.scale * LOG2E_F, w.cap_k = CAP ? -0.5f / cap2 : 0.f;

  bf16x8_t qf[QS];
  {
    const bf16* q = reinterpret_cast<const bf16*>(a.q) + (int64_t)(row0 + qi) * a.ld_q + (int64_t)head * DQ + 8 * hh;
#pragma unroll
    for (int s = 0; s < QS; ++s) qf[s] = *reinterpret_cast<const bf16x8_t*>(q + 16 * s);
  }
  f32x16 o[DT];
  float m_run, l_run;
  prompt_attention<DQ, VP, GROUPS, KEYS>(w, lds, qf, o, m_run, l_run);
  if (group || wave * 32 + l31 >= n_rows) return;
  float f = 1.0f;
  if (a.sink) {
    m_run += cap2;
    const float s2 = a.sink[head] * LOG2E_F, top = fmaxf(m_run, s2);
    f = fast_exp2(m_run - top);
    l_run = l_run * f + fast_exp2(s2 - top);
  }
  const float scale = a.out_scale * f / l_run;
  bf16* out = reinterpret_cast<bf16*>(a.out) + (int64_t)(row0 + qi) * a.ld_out + head * VP + 4 * hh;
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<u32x2*>(out + 32 * d + 2 * r) = u32x2{pack2<bf16_tag>(o[d][r] * scale, o[d][r + 1] * scale),
                                                              pack2<bf16_tag>(o[d][r + 2] * scale, o[d][r + 3] * scale)};
}

static bool wp_width(int w) { return w == 64 || w == 96 || w == 128 || w == 192 || w == 256; }
template <int DQ, int VP>
static void wp_launch(const slm_window_prefill_args& a, hipStream_t st) {
  const int64_t workgroups = (int64_t)a.n_tiles * a.heads;
  auto launch = [&](auto groups, auto cap) {
    window_prefill_kernel<DQ, VP, groups, cap><<<dim3((unsigned)workgroups), dim3(256 * groups), 0, st>>>(a);
  };
  const std::true_type capped;
  const std::false_type plain;
  if constexpr (DQ + VP <= 256) {                      // (as wide as two groups' tiles fit)
    const std::integral_constant<int, 2> two;
    if (prompt_two_groups(workgroups, a.n_ctx, a.n_tiles, a.window)) return a.softcap > 0.f ? launch(two, capped) : launch(two, plain);
  }
  const std::integral_constant<int, 1> one;
  a.softcap > 0.f ? launch(one, capped) : launch(one, plain);
}
template <int DQ>
static void wp_v(const slm_window_prefill_args& a, hipStream_t st) {
  switch (a.v_pad) {
    case 64: wp_launch<DQ, 64>(a, st); break;
    case 96: wp_launch<DQ, 96>(a, st); break;
    case 128: wp_launch<DQ, 128>(a, st); break;
    case 192: wp_launch<DQ, 192>(a, st); break;
    default: wp_launch<DQ, 256>(a, st);
  }
}

}  // namespace slm

using namespace slm;

extern "C" SLM_API int slm_window_prefill_supported(int32_t d_pad, int32_t v_pad) { return wp_width(d_pad) && wp_width(v_pad) ? 1 : 0; }
extern "C" SLM_API int slm_window_prefill(const slm_window_prefill_args* a, void* stream) {
  if (!a || !a->q || !a->key_cache || !a->value_cache || !a->out || !a->slots || !a->tiles || a->n_tiles < 0 || a->heads < 1 ||
      a->kv_heads < 1 || a->heads % a->kv_heads || a->n_rows < 0 || a->n_ctx < 0 || (int64_t)a->n_tiles * a->heads > 0x7fffffff)
    return SLM_ERR_INVALID_ARG;
  if (!slm_window_prefill_supported(a->d_pad, a->v_pad)) return SLM_ERR_UNSUPPORTED;
  if (a->ld_q < (int64_t)a->heads * a->d_pad || a->ld_out < (int64_t)a->heads * a->v_pad || a->ld_q % 8 || a->ld_out % 4 ||
      !aligned16(a->q) || !aligned16(a->key_cache) || !aligned16(a->value_cache) || !aligned16(a->out))
    return SLM_ERR_ALIGNMENT;
  if (a->n_tiles == 0) return SLM_OK;
  hip_clear_error();
  switch (a->d_pad) {
    case 64: wp_v<64>(*a, (hipStream_t)stream); break;
    case 96: wp_v<96>(*a, (hipStream_t)stream); break;
    case 128: wp_v<128>(*a, (hipStream_t)stream); break;
    case 192: wp_v<192>(*a, (hipStream_t)stream); break;
    default: wp_v<256>(*a, (hipStream_t)stream);
  }
  return hip_check_launch();
}
