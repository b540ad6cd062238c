// recurrent.hip -- layers with a matrix state S [dim, vdim] per sequence and head: the gated delta rule with a decay
// per key channel, and decayed linear attention.  Everything here is fp32 besides the projections it reads.
//
//   step     one row per sequence: convolution, activations, unit vectors, gates, the update and (delta) the output norm
//            in one launch.  One workgroup per (row, head); the state is read and written once, past the caches unless it is small.  Bound: HBM
//            (state).  16 heads of 128 x 128: delta 128 rows 71 us with ordinary loads and stores and the inputs one after the
//            other, 52 without (5.2 TB/s), 32 rows 18.4 and 14.1; lightning, the first alone, 128 rows 53 and 46 (5.8 TB/s), 32 rows
//            14.4 and 12.7, 8 rows 6.0 and 5.5, 1 row 4.3 and 4.3.
//   prepare  portions, cut into chunks of 16 tokens, every chunk at once: inputs activated and normed, decays summed, what a chunk's tokens do to
//            each other solved (a 16 x 16 triangular system), and everything that does not wait for the state multiplied out.  Bound: the
//            latency of its inputs, which are loaded before the first is used, its vector instructions (1600 a wave) and the records it writes (2 TB/s).
//            A wave's eight lengths have their root and quotient in a lane each: by all lanes one after the other 92 us (16 heads, 4096 tokens), 83.
//   scan     portions: chunk after chunk.  The columns of S are independent, so a workgroup owns 16 of them and keeps them
//            in registers from the portion's first token to its last; the products are 32-bit MFMAs.  Bound: a chain of two products and an
//            exchange a chunk, 0.6 us (24 products of 32 cycles a wave are 0.35), and the instructions around them.
//   Both, us, 16 heads of 128 x 128 and 4096 tokens: delta 305 with the triangular system and B U in the scan, 64-bit addresses and a wave's
//   read-outs by itself, 212 now; lightning 184 and 133; 8 x 500 tokens, 32 heads: 341 and 285, 209 and 178; 16 heads of 64, 2000 tokens: 120 and 75.
//   gated_norm  the norm and gate behind a scan.
#include "latent/latent_common.h"
#include "slm_mixers.h"

namespace slm {

constexpr bool DELTA_MODE(int m) { return m == SLM_REC_DELTA; }

// n / d for finite n and d in 2^-100 .. 2^100: the reciprocal corrected once, its quotient once (half the instructions of the general division)
__device__ __forceinline__ float quotient(float n, float d) {
  float r = __builtin_amdgcn_rcpf(d);
  r = __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
  const float q = n * r;
  return __builtin_fmaf(__builtin_fmaf(-d, q, n), r, q);
}
__device__ __forceinline__ float silu_f32(float z) { return z / (1.0f + __expf(-z)); }
// z / (1 + exp(-z)) by the same steps; below -69, where 1 + exp(-z) is exp(-z) and past what they take, z exp(z) / 1 (1 + exp(z) is 1); of an
// infinity, whose remainder is not a number, the quotient remains.  No branch: tokens run side by side (16 heads, 4096 tokens: 84 us with two
// branches a token, 76 without).
__device__ __forceinline__ float silu_run(float z) {
  const bool low = z < -69.f;
  const float e = __expf(low ? z : -z), d = 1.0f + e, n = low ? z * e : z;
  float r = __builtin_amdgcn_rcpf(d);
  r = __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
  const float q = n * r;
  return __builtin_fmaf(fmaxf(__builtin_fmaf(-d, q, n), -3.4028235e38f), r, q);
}
// log(1 + x) = log(u) x / (u - 1) with u the rounded 1 + x: what the sum loses of x comes back (Kahan); where u is not 1 both are above 2^-25
__device__ __forceinline__ float softplus_f32(float z) {
  const float x = __expf(-fabsf(z)), u = 1.0f + x;
  const float q = __logf(u) * quotient(x, u - 1.0f), l = u == 1.0f ? x : q;
  return fmaxf(z, 0.f) + l;
}
__device__ __forceinline__ float sigmoid_full(float z) { return 1.0f / (1.0f + expf(-z)); }

// the convolved, activated input of channel c (index into q | k | v) of `row` at position p; rows of the step before
// `row0` come from the ring
template <typename E>
__device__ __forceinline__ float conv_input(const slm_recurrent_args& a, const E* ring, int64_t row, int64_t row0, int p, int c) {
  const int64_t ch = 2 * (int64_t)a.qk_heads * a.dim + (int64_t)a.heads * a.vdim;
  const int qk = a.qk_heads * a.dim;
  const int64_t col = c < qk ? a.off_q + c : c < 2 * qk ? a.off_k + (c - qk) : a.off_v + (c - 2 * qk);
  const E* src = reinterpret_cast<const E*>(a.proj) + col;
  float acc = 0.f;
  for (int j = min(a.taps - 1, p); j >= 0; --j) {
    const float x = row - j >= row0 ? to_f32(src[(row - j) * a.ld_proj]) : to_f32(ring[(int64_t)((p - j) % a.taps) * ch + c]);
    acc = __builtin_fmaf(a.conv_w[(int64_t)(a.taps - 1 - j) * ch + c], x, acc);
  }
  return silu_f32(acc);
}
// The ring entry that the input j > 0 tokens back of position p lies in, of a convolution of at least 2 taps.  Inputs there are not
// (older than the taps, or than the sequence) are left out of the sum; their loads go to an entry that is there, and never to
// that of p itself, which another head of the launch may be writing.
constexpr __host__ __device__ int step_entry(int j, int p, int taps) {
  const int most = taps - 1 < p ? taps - 1 : p, back = j < most ? j : most;
  return (p + taps - (back > 1 ? back : 1)) % taps;
}
constexpr bool step_reads_no_kept_entry() {
  for (int taps = 2; taps <= 4; ++taps)
    for (int p = 0; p < 12; ++p)
      for (int j = 1; j < 4; ++j)
        if (step_entry(j, p, taps) == p % taps || (j <= p && j < taps && step_entry(j, p, taps) != (p - j) % taps)) return false;
  return true;
}
static_assert(step_reads_no_kept_entry(), "the entry of the step's own position is written while the others are read");
// the same for the one row of a step, convolutions of 2 to 4 taps: every load at once
template <typename E>
__device__ __forceinline__ float conv_step4(const slm_recurrent_args& a, const E* ring, int64_t row, int p, int c) {
  const int64_t ch = 2 * (int64_t)a.qk_heads * a.dim + (int64_t)a.heads * a.vdim;
  const int qk = a.qk_heads * a.dim, most = min(a.taps - 1, p);
  const int64_t col = c < qk ? a.off_q + c : c < 2 * qk ? a.off_k + (c - qk) : a.off_v + (c - 2 * qk);
  float w[4], x[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    w[j] = a.conv_w[(int64_t)(a.taps - 1 - min(j, most)) * ch + c];
    x[j] = to_f32(j == 0 ? reinterpret_cast<const E*>(a.proj)[row * a.ld_proj + col] : ring[(int64_t)step_entry(j, p, a.taps) * ch + c]);
  }
  float acc = 0.f;
#pragma unroll
  for (int j = 3; j >= 0; --j)
    if (j <= most) acc = __builtin_fmaf(w[j], x[j], acc);
  return silu_f32(acc);
}
// (raw projection of channel c, what the ring keeps)
template <typename E>
__device__ __forceinline__ E raw_input(const slm_recurrent_args& a, int64_t row, int c) {
  const int qk = a.qk_heads * a.dim;
  const int64_t col = c < qk ? a.off_q + c : c < 2 * qk ? a.off_k + (c - qk) : a.off_v + (c - 2 * qk);
  return reinterpret_cast<const E*>(a.proj)[row * a.ld_proj + col];
}
// the same for the 16 tokens from `row` on (n of them there are), convolutions of at most 4 taps: every input is read once
template <typename E, typename F>
__device__ __forceinline__ void conv_run4(const slm_recurrent_args& a, const E* ring, int64_t row, int64_t row0, int p, int n, int c, F put) {
  const int64_t ch = 2 * (int64_t)a.qk_heads * a.dim + (int64_t)a.heads * a.vdim;
  const int qk = a.qk_heads * a.dim;
  const int64_t col = c < qk ? a.off_q + c : c < 2 * qk ? a.off_k + (c - qk) : a.off_v + (c - 2 * qk);
  const E* src = reinterpret_cast<const E*>(a.proj) + row * a.ld_proj + col;
  float w[4], x[19];   // w[j]: of the input j tokens back; x[3 + t]: the input of token t
#pragma unroll
  for (int j = 0; j < 4; ++j) w[j] = j < a.taps ? a.conv_w[(int64_t)(a.taps - 1 - j) * ch + c] : 0.f;
#pragma unroll
  for (int j = 1; j < 4; ++j) {   // (no branch around a load; where there is no such input, an entry of the ring is read for nothing)
    const bool there = j < a.taps && p >= j;
    const E* before = row - j >= row0 ? src - j * a.ld_proj : ring + (int64_t)(there ? (p - j) % a.taps : 0) * ch + c;
    x[3 - j] = to_f32(*before);
    x[3 - j] = there ? x[3 - j] : 0.f;
  }
#pragma unroll
  for (int t = 0; t < 16; ++t) x[3 + t] = to_f32(src[min(t, n - 1) * a.ld_proj]);
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    float acc = w[3] * x[t];
#pragma unroll
    for (int j = 2; j >= 0; --j) acc = __builtin_fmaf(w[j], x[3 + t - j], acc);
    const float y = silu_run(acc);
    put(t, t < n ? y : 0.f);
  }
}
template <typename E>
__device__ __forceinline__ float decay_exponent(const slm_recurrent_args& a, int64_t row, int head, int c) {
  const float x = to_f32(reinterpret_cast<const E*>(a.low)[row * a.ld_low + (int64_t)head * a.dim + c]);
  return a.neg_a[head] * softplus_f32(x + a.dt_bias[head * a.dim + c]);
}

// four columns of the state; ONCE: past the caches' replacement
template <bool ONCE>
__device__ __forceinline__ f32x4 load_state(const float* p) {
  if constexpr (ONCE) return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
  else return *reinterpret_cast<const f32x4*>(p);
}
template <bool ONCE>
__device__ __forceinline__ void store_state(float* p, f32x4 v) {
  if constexpr (ONCE) __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(p));
  else *reinterpret_cast<f32x4*>(p) = v;
}

// ---------------------------------------------------------------------------------------
// step: threads = 256 per 64 columns; thread = (4 columns, row group of 16), NR rows of its group
// ---------------------------------------------------------------------------------------
template <typename E, int MODE, int NR, bool ONCE>
__global__ void __launch_bounds__(1024) recurrent_step_kernel(const slm_recurrent_args a) {
  constexpr int DK = 16 * NR;
  __shared__ float sq[DK], sk[DK], sg[DK], sv[256], red[16][64], wred[2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nthreads = blockDim.x, n_waves = nthreads >> 6;
  const int head = blockIdx.x % a.heads;
  const int64_t row = blockIdx.x / a.heads;
  const int p = a.positions[row];
  const int slot = a.state_slots[row];
  const int qh = head / (a.heads / a.qk_heads);
  const int colq = (lane & 15) + 16 * (wave >> 2);
  const int rg = (wave & 3) * 4 + (lane >> 4);
  const bool mine = 4 * colq < a.v_pad;
  float* S = a.state + ((int64_t)slot * a.heads + head) * DK * a.v_pad + 4 * colq;

  f32x4 s[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r)
    s[r] = mine && p > 0 ? load_state<ONCE>(S + (int64_t)(rg + 16 * r) * a.v_pad) : f32x4{0.f, 0.f, 0.f, 0.f};

  float beta = 0.f;
  if constexpr (DELTA_MODE(MODE)) {
    const int64_t ch = 2 * (int64_t)a.qk_heads * a.dim + (int64_t)a.heads * a.vdim;
    const int qk = a.qk_heads * a.dim;
    E* ring = reinterpret_cast<E*>(a.conv_ring) + (int64_t)slot * a.taps * ch;
    E* keep = ring + (int64_t)(p % a.taps) * ch;   // (no head reads this entry: the ring holds one more than the history)
    const bool first_of_group = head % (a.heads / a.qk_heads) == 0;
    float nq = 0.f, nk = 0.f;
    // an input each: q, k, the decay, v (one after the other their loads are this kernel's length: 8.2 us for one row of 32 heads)
    for (int i = tid; i < 3 * DK + a.v_pad; i += nthreads) {
      const int kind = min(i / DK, 3), at = i - kind * DK;
      if (kind == 2) {
        sg[at] = at < a.dim ? expf(decay_exponent<E>(a, row, head, at)) : 0.f;
        continue;
      }
      float x = 0.f;
      if (at < (kind == 3 ? a.vdim : a.dim)) {
        const int c = kind == 3 ? 2 * qk + head * a.vdim + at : kind * qk + qh * a.dim + at;
        x = a.taps <= 4 && a.taps > 1 ? conv_step4<E>(a, ring, row, p, c) : conv_input<E>(a, ring, row, row, p, c);
        if (kind == 3 || first_of_group) keep[c] = raw_input<E>(a, row, c);
      }
      if (kind == 0) nq = __builtin_fmaf(x, x, nq);
      if (kind == 1) nk = __builtin_fmaf(x, x, nk);
      (kind == 0 ? sq : kind == 1 ? sk : sv)[at] = x;
    }
    nq = wave_sum(nq), nk = wave_sum(nk);
    if (lane == 0) wred[0][wave] = nq, wred[1][wave] = nk;
    __syncthreads();
    nq = nk = 0.f;
    for (int w = 0; w < n_waves; ++w) nq += wred[0][w], nk += wred[1][w];
    const float fq = a.q_scale / sqrtf(nq + a.unit_eps), fk = 1.0f / sqrtf(nk + a.unit_eps);
    beta = sigmoid_full(to_f32(reinterpret_cast<const E*>(a.proj)[row * a.ld_proj + a.off_b + head]));
    float kv[4] = {0.f, 0.f, 0.f, 0.f}, ks[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const float g = sg[rg + 16 * r];
      ks[r] = sk[rg + 16 * r] * fk;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[r][j] *= g;
        kv[j] = __builtin_fmaf(ks[r], s[r][j], kv[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      kv[j] += __shfl_xor(kv[j], 16, 64);
      kv[j] += __shfl_xor(kv[j], 32, 64);
    }
    if (lane < 16) *reinterpret_cast<f32x4*>(&red[wave][4 * lane]) = f32x4{kv[0], kv[1], kv[2], kv[3]};
    __syncthreads();
    float o[4] = {0.f, 0.f, 0.f, 0.f}, u[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) t += red[(wave & ~3) + w][4 * (lane & 15) + j];
      u[j] = mine ? beta * (sv[4 * colq + j] - t) : 0.f;
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const float q = sq[rg + 16 * r] * fq;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[r][j] = __builtin_fmaf(ks[r], u[j], s[r][j]);
        o[j] = __builtin_fmaf(q, s[r][j], o[j]);
      }
    }
    if (mine)
#pragma unroll
      for (int r = 0; r < NR; ++r) store_state<ONCE>(S + (int64_t)(rg + 16 * r) * a.v_pad, s[r]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o[j] += __shfl_xor(o[j], 16, 64);
      o[j] += __shfl_xor(o[j], 32, 64);
    }
    __syncthreads();
    if (lane < 16) *reinterpret_cast<f32x4*>(&red[wave][4 * lane]) = f32x4{o[0], o[1], o[2], o[3]};
    __syncthreads();
    // read-out: norm over vdim, weight, gate (threads 0 .. v_pad - 1 hold a column each)
    float x = 0.f;
    if (tid < a.v_pad) {
      const int w0 = 4 * (tid >> 6);
#pragma unroll
      for (int w = 0; w < 4; ++w) x += red[w0 + w][tid & 63];
    }
    const float ss = wave_sum(x * x);
    if (lane == 0) wred[0][wave] = ss;
    __syncthreads();
    float total = 0.f;
    for (int w = 0; w < n_waves; ++w) total += wred[0][w];
    const float rs = 1.0f / sqrtf(total / (float)a.vdim + a.eps);
    E* out = reinterpret_cast<E*>(a.out) + row * a.ld_out;
    if (tid < a.vdim) {
      const float gate = to_f32(reinterpret_cast<const E*>(a.low)[row * a.ld_low + a.off_gate + (int64_t)head * a.vdim + tid]);
      out[head * a.vdim + tid] = (E)(x * rs * a.norm_weight[tid] * sigmoid_f32(gate));
    }
    if (head == a.heads - 1)
      for (int64_t i = (int64_t)a.heads * a.vdim + tid; i < a.ld_out; i += nthreads) out[i] = (E)0.f;
  } else {
    const E* pr = reinterpret_cast<const E*>(a.proj) + row * a.ld_proj;
    for (int i = tid; i < DK; i += nthreads) {
      sq[i] = i < a.dim ? silu_f32(to_f32(pr[a.off_q + qh * a.dim + i])) : 0.f;
      sk[i] = i < a.dim ? silu_f32(to_f32(pr[a.off_k + qh * a.dim + i])) : 0.f;
    }
    for (int i = nthreads - 1 - tid; i < a.v_pad; i += nthreads) sv[i] = i < a.vdim ? silu_f32(to_f32(pr[a.off_v + head * a.vdim + i])) : 0.f;
    __syncthreads();
    const float d = a.decay[head];
    float o[4] = {0.f, 0.f, 0.f, 0.f}, v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = mine ? sv[4 * colq + j] : 0.f;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const float k = sk[rg + 16 * r], q = sq[rg + 16 * r];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[r][j] = __builtin_fmaf(k, v[j], s[r][j] * d);
        o[j] = __builtin_fmaf(q, s[r][j], o[j]);
      }
      if (mine) store_state<ONCE>(S + (int64_t)(rg + 16 * r) * a.v_pad, s[r]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o[j] += __shfl_xor(o[j], 16, 64);
      o[j] += __shfl_xor(o[j], 32, 64);
    }
    if (lane < 16) *reinterpret_cast<f32x4*>(&red[wave][4 * lane]) = f32x4{o[0], o[1], o[2], o[3]};
    __syncthreads();
    if (tid < a.v_pad) {
      const int w0 = 4 * (tid >> 6);
      float x = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) x += red[w0 + w][tid & 63];
      a.o[(row * a.heads + head) * a.v_pad + tid] = x;
    }
  }
}

// ---------------------------------------------------------------------------------------
// portions: chunks of 16 tokens
// ---------------------------------------------------------------------------------------
// With L_t the sum of a chunk's log decays up to token t, S0 the state in front of it, x.d = product per key channel:
//   (I + diag(beta) A) U = diag(beta) (V - Kd S0)     A_ts = sum_d k_t k_s exp(L_t - L_s), s < t;  Kd_t = k_t exp(L_t)
//   O  = Qd S0 + B U                                  B_ts = sum_d q_t k_s exp(L_t - L_s), s <= t; Qd_t = q_t exp(L_t)
//   S1 = diag(exp(L_end)) S0 + Kr^T U                 Kr_t = k_t exp(L_end - L_t)
// Every exponent is <= 0: nothing overflows however fast a channel forgets.  Without the delta rule U = V.  With T = (I + diag(beta) A)^-1 diag(beta),
// what does not wait for S0 is worked out chunk by chunk in prepare, and the scan's chain is two products and an exchange long:
//   U = V' - Kd' S0     O = O0 + Qd' S0     V' = T V, Kd' = T Kd, O0 = B T V, Qd' = Qd - B T Kd
// A chunk's record for one head, in floats:
//   Kd' | Qd' (16 x DK each) | Kr^T (DK x 16) | exp(L_end) (DK) | V'^T | O0^T (v_pad x 16 each)
// Matrices are tiles of 16 x 16 in the order the scan's lanes take them, four floats a lane: entry (m, k) at ((k / 4 % 4) 16 + m % 16) 4 + k % 4, so
// that a wave reads a tile as 1 KiB in a row.  Kd', Qd': m token, k channel; Kr^T, V'^T, O0^T: m channel / column, k token.
template <int DK>
struct ChunkRecord {
  static constexpr int KD = 0, QD = 16 * DK, KR = 32 * DK, GE = 48 * DK, V = 49 * DK;
  int v_pad;
  __device__ __forceinline__ int o0() const { return V + 16 * v_pad; }
  __device__ __forceinline__ int64_t size() const { return o0() + 16 * v_pad; }
};
// What 32-bit products have just left in x, before a branch that its first reader lies behind (the compiler counts the wait along one way there only)
__device__ __forceinline__ void settle(f32x4& x) { asm volatile("s_nop 15" : "+v"(x)); }
// c + x y^T over four contraction indexes a lane: lane (l16, g) has x [l16][4 g ..] and y [l16][4 g ..], and gets [4 g ..][l16]
__device__ __forceinline__ f32x4 mma4(const f32x4& x, const f32x4& y, f32x4 c) {
#pragma unroll
  for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[r], y[r], c, 0, 0, 0);
  return c;
}

// one workgroup per (chunk, head); every chunk of the step at once.  With the delta rule A and B are 32-bit MFMAs of k exp(L), q exp(L) and k exp(-L) where
// no channel of the chunk falls below 2^-96 (k is a unit vector: each entry's factors then are in range, their product is below 1); else entry by
// entry, an exponential for each of the 16 x 16 x DK terms.  Without it a token's channels decay alike: B is q k^T, whose entries are scaled, of
// whatever size keys are.
constexpr float DIRECT_BELOW = -96.f;
template <typename E, int MODE, int DK>
__global__ void __launch_bounds__(256) recurrent_prepare_kernel(const slm_recurrent_args a) {
  constexpr bool DELTA = DELTA_MODE(MODE);
  constexpr int LD = DK + 4;                     // (the 16 rows a quarter-wave reads by 16 bytes are in different banks)
  constexpr int TPW = (DK / 16 + 3) / 4;         // channel tiles of a wave: wave, wave + 4 ..
  __shared__ __attribute__((aligned(16))) float sq[16 * LD > 2048 ? 16 * LD : 2048], sk[16 * LD], sL[DELTA ? 16 * LD : 1], sb[16 * 20], sT[16 * 20];
  extern __shared__ __attribute__((aligned(16))) float sv[];   // 16 x v_pad, as in the record
  __shared__ float sa[16][17], sbeta[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int head = blockIdx.x % a.heads;
  const int64_t chunk = blockIdx.x / a.heads;
  const int32_t* cd = a.chunks + 3 * chunk;
  const int seq = cd[0], n = cd[2];
  const int64_t row = cd[1], row0 = a.q_cu[seq];
  const int p = a.positions[row];
  const int qh = head / (a.heads / a.qk_heads), qk = a.qk_heads * a.dim;
  const ChunkRecord<DK> at{a.v_pad};
  float* rec = a.pre + (chunk * a.heads + head) * at.size();
  const E* ring = nullptr;
  if constexpr (DELTA)
    ring = reinterpret_cast<const E*>(a.conv_ring) + (int64_t)a.state_slots[seq] * a.taps * (2 * (int64_t)qk + (int64_t)a.heads * a.vdim);
  const E* in = reinterpret_cast<const E*>(a.proj) + row * a.ld_proj;
  const float step_l = DELTA ? 0.f : fmaxf(log2f(a.decay[head]), -126.f);

  // every input's load before its use: one after the other they were this kernel's length
  constexpr int PER = DK / 16;   // (token, channel) pairs of a thread
  float decay_in[PER], decay_bias[PER];
  if constexpr (DELTA) {
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int t = min((tid + 256 * j) / DK, n - 1), c = min((tid + 256 * j) % DK, a.dim - 1);
      decay_in[j] = to_f32(reinterpret_cast<const E*>(a.low)[(row + t) * a.ld_low + (int64_t)head * a.dim + c]);
      decay_bias[j] = a.dt_bias[head * a.dim + c];
    }
  }
  if (DELTA && a.taps <= 4) {
    for (int i = tid; i < 2 * DK + a.v_pad; i += 256) {
      if (i < 2 * DK) {
        const int c = i < DK ? i : i - DK;
        float* dst = (i < DK ? sq : sk) + c;
        auto put = [&](int t, float x) { dst[t * LD] = x; };
        if (c < a.dim) {
          conv_run4<E>(a, ring, row, row0, p, n, (i < DK ? 0 : qk) + qh * a.dim + c, put);
        } else {
#pragma unroll
          for (int t = 0; t < 16; ++t) put(t, 0.f);
        }
      } else {
        const int c = i - 2 * DK;
        float* dst = sv + (c >> 4) * 256 + (c & 15) * 4;
        f32x4 four;
        auto put = [&](int t, float x) {
          four[t & 3] = x;
          if ((t & 3) == 3) *reinterpret_cast<f32x4*>(dst + (t >> 2) * 64) = four;
        };
        if (c < a.vdim) {
          conv_run4<E>(a, ring, row, row0, p, n, 2 * qk + head * a.vdim + c, put);
        } else {
#pragma unroll
          for (int t = 0; t < 16; ++t) put(t, 0.f);
        }
      }
    }
  } else if constexpr (DELTA) {
    for (int i = tid; i < 16 * DK; i += 256) {
      const int t = i / DK, c = i % DK;
      float q = 0.f, k = 0.f;
      if (t < n && c < a.dim) {
        q = conv_input<E>(a, ring, row + t, row0, p + t, qh * a.dim + c);
        k = conv_input<E>(a, ring, row + t, row0, p + t, qk + qh * a.dim + c);
      }
      sq[t * LD + c] = q, sk[t * LD + c] = k;
    }
    for (int i = tid; i < 16 * a.v_pad; i += 256) {   // (in the record's order)
      const int t = ((i >> 6) & 3) * 4 + (i & 3), c = (i >> 8) * 16 + ((i >> 2) & 15);
      sv[i] = t < n && c < a.vdim ? conv_input<E>(a, ring, row + t, row0, p + t, 2 * qk + head * a.vdim + c) : 0.f;
    }
  } else {
    float q[PER], k[PER], v[4];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int t = min((tid + 256 * j) / DK, n - 1), c = min((tid + 256 * j) % DK, a.dim - 1);
      q[j] = to_f32(in[t * a.ld_proj + a.off_q + qh * a.dim + c]);
      k[j] = to_f32(in[t * a.ld_proj + a.off_k + qh * a.dim + c]);
    }
    for (int i0 = tid; i0 < 16 * a.v_pad; i0 += 1024) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = min((i0 + 256 * j) / a.v_pad, n - 1), c = min((i0 + 256 * j) % a.v_pad, a.vdim - 1);
        v[j] = to_f32(in[(int64_t)t * a.ld_proj + a.off_v + head * a.vdim + c]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = (i0 + 256 * j) / a.v_pad, c = (i0 + 256 * j) % a.v_pad;
        const float y = silu_run(v[j]);
        if (t < 16) sv[(c >> 4) * 256 + (t >> 2) * 64 + (c & 15) * 4 + (t & 3)] = t < n && c < a.vdim ? y : 0.f;
      }
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int t = (tid + 256 * j) / DK, c = (tid + 256 * j) % DK;
      const bool there = t < n && c < a.dim;
      const float y = silu_run(q[j]), z = silu_run(k[j]);
      sq[t * LD + c] = there ? y : 0.f, sk[t * LD + c] = there ? z : 0.f;
    }
  }
  if constexpr (DELTA) {
    const float neg_a = a.neg_a[head];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int t = (tid + 256 * j) / DK, c = (tid + 256 * j) % DK;
      const float l = LOG2E_F * (neg_a * softplus_f32(decay_in[j] + decay_bias[j]));
      sL[t * LD + c] = t < n && c < a.dim ? l : 0.f;
    }
  }
  if (DELTA && tid < 16) sbeta[tid] = tid < n ? sigmoid_full(to_f32(in[tid * a.ld_proj + a.off_b + head])) : 0.f;
  __syncthreads();
  if constexpr (DELTA) {   // unit vectors: four tokens per wave; a lane takes the root and quotient of one of their eight sums
    constexpr int CW = (DK + 63) / 64;
    float q[4][CW], k[4][CW], sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = 4 * wave + j;
      float nq = 0.f, nk = 0.f;
#pragma unroll
      for (int i = 0; i < CW; ++i) {
        const int c = lane + 64 * i;
        const bool there = DK % 64 == 0 || c < DK;
        q[j][i] = there ? sq[t * LD + c] : 0.f, k[j][i] = there ? sk[t * LD + c] : 0.f;
        nq = __builtin_fmaf(q[j][i], q[j][i], nq);
        nk = __builtin_fmaf(k[j][i], k[j][i], nk);
      }
      nq = wave_sum(nq), nk = wave_sum(nk);
      sum = lane == j ? nq : lane == 4 + j ? nk : sum;
    }
    const float f = (lane < 4 ? a.q_scale : 1.0f) / sqrtf(sum + a.unit_eps);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = 4 * wave + j;
      const float fq = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), j));
      const float fk = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), 4 + j));
#pragma unroll
      for (int i = 0; i < CW; ++i) {
        const int c = lane + 64 * i;
        if (DK % 64 == 0 || c < DK) sq[t * LD + c] = q[j][i] * fq, sk[t * LD + c] = k[j][i] * fk;
      }
    }
  }
  float lowest = step_l * n;   // (without the delta rule a token's channels decay alike)
  if (tid < DK) {
    if constexpr (DELTA) {
      float l = 0.f;
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        l += sL[t * LD + tid];
        sL[t * LD + tid] = l;
      }
      lowest = l;
    }
    rec[ChunkRecord<DK>::GE + tid] = fast_exp2(lowest);
  }
  const bool direct = __syncthreads_or(DELTA && (lowest < DIRECT_BELOW || !(lowest <= 0.f)));
  const int l16 = lane & 15, g = lane >> 4;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto lds4 = [](const float* p) { return *reinterpret_cast<const f32x4*>(p); };
  auto summed = [&](int t, int c) { return DELTA ? sL[t * LD + c] : step_l * min(t + 1, n); };
  auto exp4 = [](const f32x4& l) { return f32x4{fast_exp2(l.x), fast_exp2(l.y), fast_exp2(l.z), fast_exp2(l.w)}; };

  f32x4 qd[TPW], pa = zero, pb = zero;   // lane: token l16, channels 4 g .. of a tile
#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    const int tile = wave + 4 * j;
    if (tile >= DK / 16) continue;
    const int at_t = l16 * LD + 16 * tile + 4 * g;
    f32x4 l;
    if constexpr (DELTA) l = lds4(sL + at_t);
    else l = zero + summed(l16, 0);
    const f32x4 e = exp4(l), k = lds4(sk + at_t), q = lds4(sq + at_t);
    qd[j] = q * e;
    if constexpr (!DELTA) {
      pb = mma4(q, k, pb);
    } else if (!direct) {
      const f32x4 ks = k * exp4(-l);
      pa = mma4(k * e, ks, pa);
      pb = mma4(qd[j], ks, pb);
    }
  }
  settle(pa);
  settle(pb);
  if (!DELTA || !direct) {
    f32x4 (*const part)[2][64] = reinterpret_cast<f32x4 (*)[2][64]>(sq);
    __syncthreads();   // (nobody reads q any more)
    if constexpr (DELTA) part[wave][0][lane] = pa;
    part[wave][1][lane] = pb;
    __syncthreads();
    if (wave < 2 && (DELTA || wave == 1)) {   // lane: rows 4 g .., column l16
      f32x4 sum = part[0][wave][lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) sum += part[w][wave][lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 4 * g + r;
        if (wave == 0) sa[t][l16] = l16 < t ? sum[r] : 0.f;
        else sb[t * 20 + l16] = l16 > t ? 0.f : DELTA ? sum[r] : sum[r] * fast_exp2(step_l * (min(t + 1, n) - min(l16 + 1, n)));
      }
    }
  } else {
    const int t = tid >> 4, s = tid & 15;
    float x = 0.f, y = 0.f;
    if (s <= t) {
#pragma unroll 2
      for (int c = 0; c < DK; c += 4) {
        const f32x4 ks = lds4(sk + s * LD + c), kt = lds4(sk + t * LD + c), qt = lds4(sq + t * LD + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float e = ks[j] * fast_exp2(summed(t, c + j) - summed(s, c + j));
          x = __builtin_fmaf(kt[j], e, x);
          y = __builtin_fmaf(qt[j], e, y);
        }
      }
    }
    sb[t * 20 + s] = y;
    sa[t][s] = x;
  }
  __syncthreads();
  f32x4 tv, bt = lds4(sb + l16 * 20 + 4 * g);   // rows l16, columns 4 g .. of T and of B T (without the delta rule: of B)
  if constexpr (DELTA) {
    if (tid < 16) {   // column tid of T by forward substitution
      float x[16];
#pragma unroll
      for (int t = 0; t < 16; ++t) x[t] = t == tid ? 1.0f : 0.f;
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        x[s] *= sbeta[s];
        sT[s * 20 + tid] = x[s];
#pragma unroll
        for (int t = s + 1; t < 16; ++t) x[t] = __builtin_fmaf(-sa[t][s], x[s], x[t]);
      }
    }
    __syncthreads();
    tv = lds4(sT + l16 * 20 + 4 * g);
    f32x4 tt;   // row l16, columns 4 g .. of T^T
#pragma unroll
    for (int r = 0; r < 4; ++r) tt[r] = sT[(4 * g + r) * 20 + l16];
    bt = mma4(tt, bt, zero);
    settle(bt);
  }
#pragma unroll
  for (int j = 0; j < TPW; ++j) {
    const int tile = wave + 4 * j;
    if (tile >= DK / 16) continue;
    const int d = 16 * tile + l16;
    const float end = summed(15, d);
    f32x4 kr, kd;   // channel d, tokens 4 g ..
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float k = sk[(4 * g + r) * LD + d], l = summed(4 * g + r, d);
      kr[r] = k * fast_exp2(end - l);
      kd[r] = k * fast_exp2(l);
    }
    float* at_tile = rec + 256 * tile + 4 * lane;
    *reinterpret_cast<f32x4*>(at_tile + ChunkRecord<DK>::KR) = kr;
    if constexpr (DELTA) {
      *reinterpret_cast<f32x4*>(at_tile + ChunkRecord<DK>::KD) = mma4(kd, tv, zero);
      qd[j] = mma4(-kd, bt, qd[j]);
    }
    *reinterpret_cast<f32x4*>(at_tile + ChunkRecord<DK>::QD) = qd[j];
  }
  for (int tile = wave; tile < a.v_pad / 16; tile += 4) {
    const f32x4 v = lds4(sv + 256 * tile + 4 * lane);   // column l16, tokens 4 g ..
    float* at_tile = rec + ChunkRecord<DK>::V + 256 * tile + 4 * lane;
    *reinterpret_cast<f32x4*>(at_tile) = DELTA ? mma4(tv, v, zero) : v;
    *reinterpret_cast<f32x4*>(at_tile + 16 * a.v_pad) = mma4(bt, v, zero);
  }
}

// One workgroup per (sequence, head, 16 NCT columns of S), chunk after chunk.  Its waves share the key channels: a wave
// keeps TPW tiles [16 x 16] of every column tile of S in registers in the accumulator layout of the 32-bit MFMA (row 4 g + r,
// column l16), which is the layout its right operand takes when the contraction index of product r is 4 g + r.  Partial
// products with S0 meet in LDS, one barrier a chunk, the read-outs' products run under it; read-outs are completed a chunk later.  The operands of the
// next chunks travel meanwhile.  Two column tiles read the records half as often: where enough workgroups are left.
template <int TPW, int NCT>
struct ChunkOperands {
  f32x4 kd[TPW], qd[TPW], kr[TPW], ge[TPW], v[NCT], o0[NCT];
};

template <typename E, int MODE, int DK, int W, int NCT>
__global__ void __launch_bounds__(64 * W, 2) recurrent_scan_kernel(const slm_recurrent_args a) {
  constexpr bool DELTA = DELTA_MODE(MODE);
  constexpr int TPW = DK / 16 / W;
  constexpr int NB = TPW <= 1 || (TPW == 2 && (NCT == 1 || !DELTA)) ? 3 : 2;   // chunks in registers: one in use, the others on their way
  __shared__ f32x4 part_u[2][NCT][W][64], part_o[2][NCT][W][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  // the column blocks of one head on one XCD (workgroups go round the XCDs): they read the same records
  const int n_ct = a.v_pad / 16, n_cb = (n_ct + NCT - 1) / NCT, n_items = (a.batch - a.n_single) * a.heads;
  const int cb = blockIdx.x / 8 % n_cb, item = blockIdx.x / (8 * n_cb) * 8 + blockIdx.x % 8;
  if (item >= n_items) return;
  const int head = item % a.heads, ps = item / a.heads, seq = a.n_single + ps;
  const int64_t row0 = a.q_cu[seq];
  const int n = a.q_cu[seq + 1] - (int)row0;
  const int p0 = a.positions[row0], slot = a.state_slots[seq];
  const int64_t chunk0 = a.seq_chunks[ps];
  const int n_chunks = (n + 15) / 16;
  const ChunkRecord<DK> at{a.v_pad};
  const float* rec0 = a.pre + (chunk0 * a.heads + head) * at.size();
  const int64_t rec_step = a.heads * at.size();
  float* S = a.state + (((int64_t)slot * a.heads + head) * DK + 16 * TPW * wave + 4 * g) * a.v_pad + l16;
  int ct[NCT];   // (an odd last tile is computed twice and stored once)
#pragma unroll
  for (int j = 0; j < NCT; ++j) ct[j] = min(cb * NCT + j, n_ct - 1);

  f32x4 s[NCT][TPW];
#pragma unroll
  for (int j = 0; j < NCT; ++j)
#pragma unroll
    for (int i = 0; i < TPW; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[j][i][r] = p0 > 0 ? S[(int64_t)(16 * i + r) * a.v_pad + 16 * ct[j]] : 0.f;

  // a chunk's record is a buffer: a load is one instruction (of 64-bit addresses half of a chunk's 215 instructions were additions)
  const int rec_bytes = (int)at.size() * 4;
  const uint32_t off = (uint32_t)(lane * 16), koff = off + wave * (TPW * 1024), goff = (uint32_t)(g * 16 + wave * (TPW * 64) + ChunkRecord<DK>::GE * 4);
  static_assert(NCT == 1 || NCT % 2 == 0, "half of the column tiles' read-outs under the writes, half under the reads");
  constexpr int PIECES = TPW * (DELTA ? 4 : 3) + 2 * NCT, SLOTS = 4 * ((DELTA ? 2 : 1) * NCT + 1);
  auto record = [&](int c) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(rec0 + c * rec_step), 0, rec_bytes, 0x00020000); };
  auto load = [&](const __amdgpu_buffer_rsrc_t& rec, ChunkOperands<TPW, NCT>& x, int k) {   // k-th of PIECES
    auto vec = [&](uint32_t at_lane, int from) { return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rec, at_lane, from, 0)); };
    if (k < 2 * NCT) {
      if (k % 2 == 0) x.v[k / 2] = vec(off, ChunkRecord<DK>::V * 4 + 1024 * ct[k / 2]);
      else x.o0[k / 2] = vec(off, at.o0() * 4 + 1024 * ct[k / 2]);
      return;
    }
    const int i = (k - 2 * NCT) % TPW, what = (k - 2 * NCT) / TPW;
    if (what == 0) x.ge[i] = vec(goff + i * 64, 0);
    else if (what == 1) x.qd[i] = vec(koff + i * 1024, ChunkRecord<DK>::QD * 4);
    else if (what == 2) x.kr[i] = vec(koff + i * 1024, ChunkRecord<DK>::KR * 4);
    else x.kd[i] = vec(koff + i * 1024, ChunkRecord<DK>::KD * 4);
  };
  // the read-outs of a chunk, once every wave's part of them is there: of each lane's four rows a wave takes one (of 2 waves: two)
  const int o_row = a.heads * a.v_pad * 4;   // bytes
  float* const o_from = a.o + (row0 - a.n_single) * a.heads * a.v_pad + 16 * ct[0];
  uint32_t o_off[NCT];   // (no scalar offset: that of a lane alone tells what is out of the buffer)
#pragma unroll
  for (int j = 0; j < NCT; ++j) o_off[j] = (uint32_t)((4 * g + wave) * o_row + (head * a.v_pad + 16 * (ct[j] - ct[0]) + l16) * 4);
  struct ReadOuts { float v[4 / W][NCT][W]; };
  auto collect = [&](int c, ReadOuts& y) {
#pragma unroll
    for (int r = 0; r < 4 / W; ++r)
#pragma unroll
      for (int j = 0; j < NCT; ++j)
#pragma unroll
        for (int w = 0; w < W; ++w) y.v[r][j][w] = reinterpret_cast<const float*>(&part_o[c & 1][j][w][lane])[r * W + wave];
  };
  auto finish = [&](int c, const ReadOuts& y) {   // (rows past the portion's last, and chunk -1, are out of the buffer)
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(o_from + (int64_t)16 * c * a.heads * a.v_pad, 0, c < 0 ? 0 : min(n - 16 * c, 16) * o_row - 64 * ct[0], 0x00020000);
#pragma unroll
    for (int r = 0; r < 4 / W; ++r)
#pragma unroll
      for (int j = 0; j < NCT; ++j) {
        float sum = y.v[r][j][0];
#pragma unroll
        for (int w = 1; w < W; ++w) sum += y.v[r][j][w];
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, sum), out, o_off[j] + r * W * o_row, 0, 0);
      }
  };
  // two sums of tiles side by side: the products of one wait for each other
  auto some_products = [&](const f32x4 (&x)[TPW], int j, f32x4& c, f32x4& d, int from, int to, auto between) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r < from || r >= to) continue;
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        f32x4& sum = i & 1 ? d : c;
        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i][r], s[j][i][r], sum, 0, 0, 0);
      }
      between();
    }
  };
  auto products = [&](const f32x4 (&x)[TPW], int j, f32x4 c, auto between) {
    f32x4 d = {0.f, 0.f, 0.f, 0.f};
    some_products(x, j, c, d, 0, 4, between);
    return TPW > 1 ? c + d : c;
  };
  // Chunk c; between its products the loads of chunk `later`, one at a time: the 40 of a workgroup all at once back up in the address unit, and
  // the waves with them (4096 tokens, 16 heads: delta 187 -> 160 us, of 136 without loads, before the read-outs were halved; lightning 124 -> 103; 1000 tokens, 32 heads 51 -> 45, 34 -> 27).
  auto chunk = [&](int c, const ChunkOperands<TPW, NCT>& x, int later, ChunkOperands<TPW, NCT>& xl, bool more) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const int b = c & 1;
    f32x4 o[NCT], u[NCT], pu[NCT][W];
    ReadOuts y;
    const __amdgpu_buffer_rsrc_t rec = record(later);
    int slot = 0;
    auto between = [&]() {
      if (more) {
#pragma unroll
        for (int k = 0; k < PIECES; ++k)
          if (k >= slot * PIECES / SLOTS && k < (slot + 1) * PIECES / SLOTS) load(rec, xl, k);
        __builtin_amdgcn_sched_barrier(0);
      }
      ++slot;
    };
    if constexpr (DELTA) {
#pragma unroll
      for (int j = 0; j < NCT; ++j) part_u[b][j][wave][lane] = products(x.kd, j, zero, between);
      __builtin_amdgcn_sched_barrier(0);
    }
    // (half of the read-outs' products run under the writes of the exchange, half under its reads: 16 heads, 4096 tokens 161 us with all of one
    // column tile's under the writes, 164 under the reads, 153)
    constexpr int UNDER_WRITES = DELTA ? 2 : 4;
    f32x4 od = zero;
    if constexpr (NCT == 1) {
      o[0] = wave == 0 ? x.o0[0] : zero;
      some_products(x.qd, 0, o[0], od, 0, UNDER_WRITES, between);
    }
#pragma unroll
    for (int j = 0; j < NCT / 2; ++j) o[j] = products(x.qd, j, wave == 0 ? x.o0[j] : zero, between);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    if constexpr (DELTA) {
#pragma unroll
      for (int j = 0; j < NCT; ++j)
#pragma unroll
        for (int w = 0; w < W; ++w) pu[j][w] = part_u[b][j][w][lane];
    }
    collect(c - 1, y);   // (in front of the first chunk: of nothing, and not stored)
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (NCT == 1) {
      some_products(x.qd, 0, o[0], od, UNDER_WRITES, 4, between);
      if constexpr (TPW > 1) o[0] += od;
    }
#pragma unroll
    for (int j = (NCT + 1) / 2; j < NCT; ++j) o[j] = products(x.qd, j, wave == 0 ? x.o0[j] : zero, between);
    if constexpr (DELTA) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NCT; ++j) {
      u[j] = x.v[j];
      if constexpr (DELTA) {
#pragma unroll
        for (int w = 0; w < W; ++w) u[j] -= pu[j][w];
      }
    }
#pragma unroll
    for (int j = 0; j < NCT; ++j)
#pragma unroll
      for (int i = 0; i < TPW; ++i) s[j][i] *= x.ge[i];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int i = 0; i < TPW; ++i)
#pragma unroll
        for (int j = 0; j < NCT; ++j) s[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kr[i][r], u[j][r], s[j][i], 0, 0, 0);
      between();
    }
#pragma unroll
    for (int j = 0; j < NCT; ++j) part_o[b][j][wave][lane] = o[j];
    finish(c - 1, y);
  };
  ChunkOperands<TPW, NCT> x[NB];
#pragma unroll
  for (int i = 0; i + 1 < NB; ++i) {
    const __amdgpu_buffer_rsrc_t rec = record(min(i, n_chunks - 1));
#pragma unroll
    for (int k = 0; k < PIECES; ++k) load(rec, x[i], k);
  }
  int c0 = 0;   // (whole rounds without a branch around the loads: a join would make every wait one for the youngest)
  for (; c0 + NB <= n_chunks; c0 += NB) {
#pragma unroll
    for (int i = 0; i < NB; ++i) chunk(c0 + i, x[i], min(c0 + i + NB - 1, n_chunks - 1), x[(i + NB - 1) % NB], true);
  }
#pragma unroll
  for (int i = 0; i + 1 < NB; ++i) {
#pragma unroll
    for (int j = 0; j < NCT; ++j)
#pragma unroll
      for (int t = 0; t < TPW; ++t) settle(s[j][t]);
    if (c0 + i < n_chunks) chunk(c0 + i, x[i], 0, x[i], false);
  }
  lds_barrier();
  ReadOuts y;
  collect(n_chunks - 1, y);
  finish(n_chunks - 1, y);
#pragma unroll
  for (int j = 0; j < NCT; ++j)
    if (cb * NCT + j < n_ct)
#pragma unroll
      for (int i = 0; i < TPW; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[(int64_t)(16 * i + r) * a.v_pad + 16 * ct[j]] = s[j][i][r];

  // the last inputs of the convolutions (their readers ran in the launch before)
  if (DELTA && cb == 0) {
    const int qh = head / (a.heads / a.qk_heads), qk = a.qk_heads * a.dim;
    const int64_t ch = 2 * (int64_t)qk + (int64_t)a.heads * a.vdim;
    E* ring = reinterpret_cast<E*>(a.conv_ring) + (int64_t)slot * a.taps * ch;
    const bool first_of_group = head % (a.heads / a.qk_heads) == 0;
    for (int j = max(0, n - a.taps); j < n; ++j) {
      E* dst = ring + (int64_t)((p0 + j) % a.taps) * ch;
      if (first_of_group)
        for (int i = tid; i < a.dim; i += 64 * W) {
          dst[qh * a.dim + i] = raw_input<E>(a, row0 + j, qh * a.dim + i);
          dst[qk + qh * a.dim + i] = raw_input<E>(a, row0 + j, qk + qh * a.dim + i);
        }
      for (int i = tid; i < a.vdim; i += 64 * W) dst[2 * qk + head * a.vdim + i] = raw_input<E>(a, row0 + j, 2 * qk + head * a.vdim + i);
    }
  }
}

// ---------------------------------------------------------------------------------------
// gated norm: WAVES waves per group
// ---------------------------------------------------------------------------------------
template <typename E, bool PER_HEAD>
__global__ void __launch_bounds__(256) gated_norm_kernel(const slm_gated_norm_args a) {
  __shared__ float red[4];
  const int tid = threadIdx.x, lane = tid & 63;
  if constexpr (PER_HEAD) {
    const int64_t item = (int64_t)blockIdx.x * 4 + (tid >> 6);
    if (item >= a.rows * a.heads) return;
    const int64_t row = item / a.heads;
    const int h = item % a.heads;
    const float* o = a.o + item * a.v_pad;
    const E* gate = reinterpret_cast<const E*>(a.gate) + row * a.ld_gate + (int64_t)h * a.vdim;
    E* out = reinterpret_cast<E*>(a.out) + row * a.ld_out;
    float x[4], gl[4], w[4], ss = 0.f;   // (v_pad <= 256)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = lane + 64 * j;
      const bool in = c < a.vdim;
      x[j] = in ? o[c] : 0.f, gl[j] = in ? to_f32(gate[c]) : 0.f, w[j] = in ? a.weight[c] : 0.f;
      ss = __builtin_fmaf(x[j], x[j], ss);
    }
    const float rs = 1.0f / sqrtf(wave_sum(ss) / (float)a.vdim + a.eps);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (lane + 64 * j < a.vdim) out[h * a.vdim + lane + 64 * j] = (E)(a.scale * x[j] * rs * w[j] * sigmoid_f32(gl[j]));
    if (h == a.heads - 1)
      for (int64_t c = (int64_t)a.heads * a.vdim + lane; c < a.out_width; c += 64) out[c] = (E)0.f;
  } else {
    const int64_t row = blockIdx.x;
    const int n = a.heads * a.vdim;
    const float* o = a.o + row * a.heads * a.v_pad;
    const bool packed = a.vdim == a.v_pad;
    auto at = [&](int i) { return packed ? o[i] : o[i / a.vdim * a.v_pad + i % a.vdim]; };
    float ss = 0.f;
    for (int i = tid; i < n; i += 256) {
      const float x = at(i);
      ss = __builtin_fmaf(x, x, ss);
    }
    const float rs = 1.0f / sqrtf(block_sum256(ss, red) / (float)n + a.eps);
    const E* gate = reinterpret_cast<const E*>(a.gate) + row * a.ld_gate;
    E* out = reinterpret_cast<E*>(a.out) + row * a.ld_out;
    for (int i = tid; i < n; i += 256) out[i] = (E)(a.scale * at(i) * rs * a.weight[i] * sigmoid_f32(to_f32(gate[i])));
    for (int64_t i = n + tid; i < a.out_width; i += 256) out[i] = (E)0.f;
  }
}

// The same where values come in eights and lie on 16 bytes: 16-byte accesses, all loads before the sum.  PER_HEAD: VD / 8
// lanes a head; else 256 threads a row of up to 8192.  4096 rows of 16 heads of 128:
// per head 22.0 us -> 12.9, per row 19.9 -> 14; 32 rows of 32 heads 3.6 -> 3.2, 7.5 -> 4.0.  Rows of fewer than 512 values leave most of its threads
// idle and pay for registers they do not use (4096 rows: 128 values 8.2 us against 4.9 of a value a thread, 384 9.7 / 9.1): the general kernel's.
template <typename E, int VD>
__global__ void __launch_bounds__(256) gated_norm_heads_kernel(const slm_gated_norm_args a) {
  constexpr int L = VD / 8;
  const int tid = threadIdx.x, l = tid % L;
  const int64_t item = (int64_t)blockIdx.x * (256 / L) + tid / L;
  if (item >= a.rows * a.heads) return;
  const int64_t row = item / a.heads;
  const int h = (int)(item - row * a.heads);
  float x[8], gl[8], w[8], ss = 0.f;
  load_f32<8>(a.o + item * VD + 8 * l, x);
  load_f32<8>(reinterpret_cast<const E*>(a.gate) + row * a.ld_gate + (int64_t)h * VD + 8 * l, gl);
  load_f32<8>(a.weight + 8 * l, w);
#pragma unroll
  for (int j = 0; j < 8; ++j) ss = __builtin_fmaf(x[j], x[j], ss);
#pragma unroll
  for (int d = 1; d < L; d <<= 1) ss += __shfl_xor(ss, d, 64);
  const float rs = 1.0f / sqrtf(ss / (float)VD + a.eps);
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = a.scale * x[j] * rs * w[j] * sigmoid_f32(gl[j]);
  E* out = reinterpret_cast<E*>(a.out) + row * a.ld_out;
  store_f32<8>(out + h * VD + 8 * l, x);
  if (h == a.heads - 1)
    for (int64_t c = (int64_t)a.heads * VD + l; c < a.out_width; c += L) out[c] = (E)0.f;
}
template <typename E>
__global__ void __launch_bounds__(256) gated_norm_row_kernel(const slm_gated_norm_args a) {
  constexpr int NV = 4;
  __shared__ float red[4];
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x;
  const int n = a.heads * a.vdim;
  const float* o = a.o + row * n;
  const E* gate = reinterpret_cast<const E*>(a.gate) + row * a.ld_gate;
  E* out = reinterpret_cast<E*>(a.out) + row * a.ld_out;
  float x[NV][8], gl[NV][8], w[NV][8], ss = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = (tid + 256 * v) * 8;
    if (i < n) {
      load_f32<8>(o + i, x[v]);
      load_f32<8>(gate + i, gl[v]);
      load_f32<8>(a.weight + i, w[v]);
    }
  }
#pragma unroll
  for (int v = 0; v < NV; ++v)
    if ((tid + 256 * v) * 8 < n)
#pragma unroll
      for (int j = 0; j < 8; ++j) ss = __builtin_fmaf(x[v][j], x[v][j], ss);
  const float rs = 1.0f / sqrtf(block_sum256(ss, red) / (float)n + a.eps);
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = (tid + 256 * v) * 8;
    if (i < n) {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[v][j] = a.scale * x[v][j] * rs * w[v][j] * sigmoid_f32(gl[v][j]);
      store_f32<8>(out + i, x[v]);
    }
  }
  for (int64_t i = n + tid; i < a.out_width; i += 256) out[i] = (E)0.f;
}
template <typename E>
static bool gated_norm_eights(const slm_gated_norm_args& a, hipStream_t st) {
  if (a.vdim != a.v_pad || a.vdim % 8 || a.ld_gate % 8 || a.ld_out % 8 || !aligned16(a.o) || !aligned16(a.gate) || !aligned16(a.weight) ||
      !aligned16(a.out))
    return false;
  if (!a.per_head) {
    if ((int64_t)a.heads * a.vdim > 8192 || a.heads * a.vdim < 512) return false;
    gated_norm_row_kernel<E><<<dim3((unsigned)a.rows), dim3(256), 0, st>>>(a);
    return true;
  }
  const int64_t items = a.rows * a.heads;
  auto grid = [&](int per) { return dim3((unsigned)((items + per - 1) / per)); };
  if (a.vdim == 64) gated_norm_heads_kernel<E, 64><<<grid(32), dim3(256), 0, st>>>(a);
  else if (a.vdim == 128) gated_norm_heads_kernel<E, 128><<<grid(16), dim3(256), 0, st>>>(a);
  else if (a.vdim == 256) gated_norm_heads_kernel<E, 256><<<grid(8), dim3(256), 0, st>>>(a);
  else return false;
  return true;
}

constexpr int64_t NCT2_MIN = 512;   // column tiles from which a workgroup takes two
static bool rec_sizes_ok(const slm_recurrent_args& a) {
  return a.heads > 0 && a.qk_heads > 0 && a.heads % a.qk_heads == 0 && a.dim > 0 && a.vdim > 0 && a.vdim <= a.v_pad &&
         a.v_pad % 16 == 0 && a.v_pad <= 256 && a.dim_pad >= a.dim && a.dim_pad == slm_recurrent_dim_pad(a.dim) &&
         (a.mode == SLM_REC_DELTA || a.mode == SLM_REC_LIGHTNING) && (a.dtype == SLM_BF16 || a.dtype == SLM_F32) &&
         a.batch >= 1 && a.n_single >= 0 && a.n_single <= a.batch && a.rows >= a.n_single && a.rows <= 0x7fffffff;
}
static bool rec_ptrs_ok(const slm_recurrent_args& a) {
  if (!a.proj || !a.state || !a.positions || !a.q_cu || !a.state_slots || !aligned16(a.state)) return false;
  if (a.mode == SLM_REC_LIGHTNING) return a.decay != nullptr;
  return a.low && a.conv_w && a.conv_ring && a.neg_a && a.dt_bias && a.taps >= 1;
}

// Past the caches' replacement from as many bytes of state on (past / through them, us, layers in turn over 32 MB and more; 128 x 128 heads:
// lightning 64 KB 4.1 / 3.3, 4 MB 4.7 / 4.5, 8 MB 5.1 / 5.9; delta 256 KB 6.5 / 6.3, 1 MB 6.6 / 6.8, 4 MB 6.9 / 7.4; 256 x 256, whose registers hold
// a wave's whole share: lightning 4 MB 9.3 / 7.7, 8 MB 9.7 / 9.0, 16 MB 10.4 / 13.2; delta 4 MB 13.1 / 12.4, 8 MB 13.4 / 15.4).
static bool state_once(const slm_recurrent_args& a) {
  const bool delta = DELTA_MODE(a.mode), wide = a.dim_pad == 256;
  const int64_t least = delta ? (wide ? 8 : 0) : wide ? 16 : 8;
  return (int64_t)a.n_single * a.heads * a.dim_pad * a.v_pad * 4 >= least << 20;
}
template <typename E, int MODE, bool ONCE>
static int rec_step_of(const slm_recurrent_args& a, hipStream_t st) {
  const dim3 grid((unsigned)((int64_t)a.n_single * a.heads)), block(256 * ((a.v_pad + 63) / 64));
  hip_clear_error();
  switch (a.dim_pad / 16) {
    case 2: recurrent_step_kernel<E, MODE, 2, ONCE><<<grid, block, 0, st>>>(a); break;
    case 4: recurrent_step_kernel<E, MODE, 4, ONCE><<<grid, block, 0, st>>>(a); break;
    case 8: recurrent_step_kernel<E, MODE, 8, ONCE><<<grid, block, 0, st>>>(a); break;
    case 12: recurrent_step_kernel<E, MODE, 12, ONCE><<<grid, block, 0, st>>>(a); break;
    default: recurrent_step_kernel<E, MODE, 16, ONCE><<<grid, block, 0, st>>>(a);
  }
  return hip_check_launch();
}
template <typename E, int MODE>
static int rec_step(const slm_recurrent_args& a, hipStream_t st) {
  if (state_once(a)) return rec_step_of<E, MODE, true>(a, st);
  return rec_step_of<E, MODE, false>(a, st);
}
template <typename E, int MODE, int DK, int NCT>
static void rec_scan_nct(const slm_recurrent_args& a, hipStream_t st) {
  constexpr int W = DK / 16 < 4 ? DK / 16 : 4;
  const int64_t items = (int64_t)(a.batch - a.n_single) * a.heads, n_cb = (a.v_pad / 16 + NCT - 1) / NCT;
  recurrent_scan_kernel<E, MODE, DK, W, NCT><<<dim3((unsigned)((items + 7) / 8 * 8 * n_cb)), dim3(64 * W), 0, st>>>(a);
}
template <typename E, int MODE, int DK>
static void rec_scan_dk(const slm_recurrent_args& a, hipStream_t st) {
  if (DK <= 128 && (int64_t)(a.batch - a.n_single) * a.heads * (a.v_pad / 16) >= NCT2_MIN) rec_scan_nct<E, MODE, DK, (DK <= 128 ? 2 : 1)>(a, st);
  else rec_scan_nct<E, MODE, DK, 1>(a, st);
}
template <typename E, int MODE>
static int rec_scan(const slm_recurrent_args& a, hipStream_t st) {
  hip_clear_error();
  switch (a.dim_pad) {
    case 32: rec_scan_dk<E, MODE, 32>(a, st); break;
    case 64: rec_scan_dk<E, MODE, 64>(a, st); break;
    case 128: rec_scan_dk<E, MODE, 128>(a, st); break;
    case 192: rec_scan_dk<E, MODE, 192>(a, st); break;
    default: rec_scan_dk<E, MODE, 256>(a, st);
  }
  return hip_check_launch();
}
template <typename E, int MODE>
static int rec_prepare(const slm_recurrent_args& a, hipStream_t st) {
  const dim3 grid((unsigned)((int64_t)a.n_chunks * a.heads)), block(256);
  const size_t lds = (size_t)a.v_pad * 64;
  hip_clear_error();
  switch (a.dim_pad) {
    case 32: recurrent_prepare_kernel<E, MODE, 32><<<grid, block, lds, st>>>(a); break;
    case 64: recurrent_prepare_kernel<E, MODE, 64><<<grid, block, lds, st>>>(a); break;
    case 128: recurrent_prepare_kernel<E, MODE, 128><<<grid, block, lds, st>>>(a); break;
    case 192: recurrent_prepare_kernel<E, MODE, 192><<<grid, block, lds, st>>>(a); break;
    default: recurrent_prepare_kernel<E, MODE, 256><<<grid, block, lds, st>>>(a);
  }
  return hip_check_launch();
}

}  // namespace slm

using namespace slm;

extern "C" SLM_API int32_t slm_recurrent_dim_pad(int32_t dim) {
  const int32_t w[] = {32, 64, 128, 192, 256};
  for (int32_t x : w)
    if (dim > 0 && dim <= x) return x;
  return 0;
}
#define SLM_REC_DISPATCH(fn)                                                                                               \
  hipStream_t st = (hipStream_t)stream;                                                                                    \
  if (a->mode == SLM_REC_DELTA) return a->dtype == SLM_BF16 ? fn<bf16, SLM_REC_DELTA>(*a, st) : fn<float, SLM_REC_DELTA>(*a, st); \
  return a->dtype == SLM_BF16 ? fn<bf16, SLM_REC_LIGHTNING>(*a, st) : fn<float, SLM_REC_LIGHTNING>(*a, st);

extern "C" SLM_API int slm_recurrent_step(const slm_recurrent_args* a, void* stream) {
  if (!a || !rec_sizes_ok(*a) || !rec_ptrs_ok(*a)) return SLM_ERR_INVALID_ARG;
  if (a->mode == SLM_REC_DELTA ? (!a->out || !a->norm_weight || a->ld_out < (int64_t)a->heads * a->vdim) : !a->o) return SLM_ERR_INVALID_ARG;
  if (a->n_single == 0) return SLM_OK;
  SLM_REC_DISPATCH(rec_step)
}
static bool rec_chunks_ok(const slm_recurrent_args& a) {
  return a.pre && a.chunks && a.seq_chunks && a.n_chunks >= 0 && (int64_t)a.n_chunks * a.heads <= 0x7fffffff;
}
extern "C" SLM_API int64_t slm_recurrent_record_floats(int32_t dim_pad, int32_t v_pad) { return 49 * (int64_t)dim_pad + 32 * (int64_t)v_pad; }
extern "C" SLM_API int slm_recurrent_prepare(const slm_recurrent_args* a, void* stream) {
  if (!a || !rec_sizes_ok(*a) || !rec_ptrs_ok(*a) || !rec_chunks_ok(*a)) return SLM_ERR_INVALID_ARG;
  if (!aligned16(a->pre)) return SLM_ERR_ALIGNMENT;
  if (a->n_chunks == 0) return SLM_OK;
  SLM_REC_DISPATCH(rec_prepare)
}
extern "C" SLM_API int slm_recurrent_scan(const slm_recurrent_args* a, void* stream) {
  if (!a || !rec_sizes_ok(*a) || !rec_ptrs_ok(*a) || !rec_chunks_ok(*a) || !a->o) return SLM_ERR_INVALID_ARG;
  if (!aligned16(a->pre)) return SLM_ERR_ALIGNMENT;
  if (a->batch == a->n_single) return SLM_OK;
  SLM_REC_DISPATCH(rec_scan)
}
extern "C" SLM_API int slm_gated_norm(const slm_gated_norm_args* a, void* stream) {
  if (!a || !a->o || !a->gate || !a->weight || !a->out || a->rows < 0 || a->heads < 1 || a->vdim < 1 || a->v_pad < a->vdim || a->v_pad > 256 ||
      a->out_width < (int64_t)a->heads * a->vdim || a->ld_out < a->out_width || a->rows * a->heads > 0x7fffffff)
    return SLM_ERR_INVALID_ARG;
  if (a->dtype != SLM_BF16 && a->dtype != SLM_F32) return SLM_ERR_UNSUPPORTED;
  if (a->rows == 0) return SLM_OK;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)(a->per_head ? (a->rows * a->heads + 3) / 4 : a->rows)), block(256);
  hip_clear_error();
  if (a->dtype == SLM_BF16 ? gated_norm_eights<bf16>(*a, st) : gated_norm_eights<float>(*a, st)) return hip_check_launch();
  if (a->dtype == SLM_BF16) {
    if (a->per_head) gated_norm_kernel<bf16, true><<<grid, block, 0, st>>>(*a);
    else gated_norm_kernel<bf16, false><<<grid, block, 0, st>>>(*a);
  } else {
    if (a->per_head) gated_norm_kernel<float, true><<<grid, block, 0, st>>>(*a);
    else gated_norm_kernel<float, false><<<grid, block, 0, st>>>(*a);
  }
  return hip_check_launch();
}

extern "C" SLM_API const char* slm_mixers_version(void) { return "slm_mixers 1 (gfx950)"; }
extern "C" SLM_API const char* slm_mixers_last_hip_error(void) { return hipGetErrorString((hipError_t)hip_last_error_slot()); }
extern "C" SLM_API const char* slm_mixers_status_string(int s) {
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
