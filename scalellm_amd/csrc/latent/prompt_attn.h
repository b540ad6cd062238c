// prompt_attn.h -- attention of 128 query rows of a prompt over tiles of KEYS (64, 32) keys, bf16 on v_mfma_f32_32x32x16.
//
//   S^T[KEYS x 32 q]   = K Q^T    A = K rows from LDS, B = Q rows in registers
//   soft-max                       a lane holds KEYS / 2 scores of ONE query row: register reductions + one lane-half exchange
//   O^T[v x 32 q] += V^T P^T       P^T stays in registers: the C-fragment key order {4h + e, 8 + 4h + e} is the
//                                  contraction order; V^T comes out of the row-major tile by the transpose read
// A wave has 32 query rows; four waves (a group) share the tiles in LDS.  With two groups, one takes the even tiles and the
// other the odd ones, and their sums meet in LDS at the end; with few tiles the second group leaves at once.
//
// Bound: the vector ALU, and the rate at which a wave issues.  Per wave and tile at width 128 with capped scores there are 320
// vector operations (4 cycles), 97 exponentials and reciprocals (9.6) and 32 products, which take 32 cycles of the matrix pipe
// and 11 of the vector ALU each; beside another wave of its SIMD a wave needs 2700 cycles for them, alone 3650.  So the products
// run under the vector work of the same wave: the scores of tile t + 1 under the exponentials of tile t, the values of tile t
// under the capping of tile t + 1.  The order is written out slot by slot (one product, the fragment reads of the product four
// slots on, a share of the vector work) and pinned by scheduling barriers.
// Tiles reach LDS without registers (global_load_lds), two K and two V tiles; K is loaded two tiles ahead and V one, one
// barrier a tile.  Such a load writes 1 KB in lane order, so rows have no padding and their 16-byte chunks are permuted
// instead: 16 rows of K, or 4 rows x 64 bytes of V, meet all 64 banks.
// Against products and vector work one after the other, one K and one V tile through registers and two barriers a tile, us, in turn:
// window 128 wide with a cap, 16 heads, 4096 rows 142 -> 103; 32 heads, 8 x 512 rows of 2200 to 3584 264 -> 222; latent
// 192 + 128, 32 heads, 4 prompts of 1100 to 2047 141 -> 123.  There 26 were the loads, of 137 (36 % miss L2;
// 32 KB of a CU are in flight).  Rescaling only after the maximum has grown by 2^8 takes 3 % off, but the largest weight is then no longer a
// 16-bit number and the error grows by 5 %.
#pragma once
#include <algorithm>
#include <utility>
#include "latent/latent_common.h"

namespace slm {

typedef short tr_v4 __attribute__((ext_vector_type(4)));
typedef short tr_v8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) tr_v4 tr_lds_v4;
typedef __attribute__((address_space(3))) const bf16x8_t lds_frag;

template <class F, int... I>
__device__ __forceinline__ void unrolled_(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void unrolled(F&& f) { unrolled_(f, std::make_integer_sequence<int, N>{}); }

constexpr int common_power(int c, int top) { return c % top == 0 ? top : common_power(c, top / 2); }

// Rows of C chunks of 16 bytes in LDS: chunk c of a row lies at position c ^ k_turn(row) (K), c ^ v_turn(row) (V).
template <int C>
struct TileRows {
  static constexpr int K_MASK = common_power(C, 16) - 1, V_MASK = common_power(C / 4, 4) - 1;
  static __device__ __forceinline__ int k_turn(int row) { return row / (16 / (K_MASK + 1)) & K_MASK; }
  static __device__ __forceinline__ int v_turn(int row) { return (row / (4 / (V_MASK + 1)) & V_MASK) * 4; }
};

// Tiles from which the second group has a share (a group takes every prompt_groups-th tile).
constexpr int PROMPT_SHARED = 5;
template <int GROUPS>
__device__ __forceinline__ int prompt_groups(int tiles) { return GROUPS == 2 && tiles >= PROMPT_SHARED ? 2 : 1; }

// Two groups up to 256 workgroups, one on each of the CUs: a workgroup's own chain of tiles then sets the time, and half of it
// is gained; and up to 512 if the prompts are there from their beginnings (no more context rows than rows of the query tiles),
// whose tiles are unequal: a CU with one workgroup of eight waves takes the next when it is through, where two of four waves
// leave the long one alone at the end.  A window makes their tiles alike; below 2048 keys one group is the better one then, too.
// From there on one group, whose workgroups overlap each other's beginnings and ends.
// us, one group / two: window 128 wide, 16 heads, 1 x 1000 rows 33 / 28, 4096 rows (512 workgroups) 131 / 120, 32 heads, 3072
// rows (768) 114 / 126; 4096 rows by the window, 128 keys 26 / 34, 512 40 / 47, 1024 60 / 66, 2048 95 / 103, 3072 106 / 106 (2 x 2048
// rows: 1536 60 / 63, 2048 67 / 63); latent 192 + 128, 32 heads, 4 x 128 rows of 3200 80 / 67, 8 x 256 rows of 2304 (512) 120 / 145, 16
// heads, 4096 rows, window 128 29 / 36, 1024 61 / 68.
inline bool prompt_two_groups(int64_t workgroups, int64_t n_ctx, int64_t n_tiles, int64_t window) {
  return workgroups <= 256 || (workgroups <= 512 && n_ctx <= 128 * n_tiles && (window <= 0 || window >= 2048));
}

template <int DQ, int VP, int GROUPS, int KEYS>
constexpr int prompt_lds_bytes() { return GROUPS * 2 * KEYS * 2 * (DQ + VP); }

// `Work`: n_turns, groups (prompt_groups), and per group
//   row(turn, r)                      handle of the tile's row r (any valid row behind the last key)
//   key(handle, c), value(handle, c)  address of chunk c of that row
//   seen(turn), mask(turn, s)         whether the wave's rows see any key of the tile; -inf where a row does not see a key
//   score(x), top(x), below(x, m)     a product as it is kept; the largest, and the distance to the maximum, in log2 units
//   begin(turn), end(turn)            around a turn, before its barrier
template <int DQ, int VP, int GROUPS, int KEYS, class Work>
__device__ __forceinline__ void prompt_attention(Work& work, char* lds, const bf16x8_t (&qf)[DQ / 16], f32x16 (&o)[VP / 32],
                                                 float& m_run, float& l_run) {
  constexpr int QS = DQ / 16, DT = VP / 32, KC = DQ / 8, VC = VP / 8;
  constexpr int N = KEYS / 32, NA = N * QS, NB = 2 * N * DT;   // products of the two halves of a turn
  constexpr int KL = (KC * KEYS + 255) / 256, VL = (VC * KEYS + 255) / 256;   // loads of a wave per tile
  constexpr int K_TILE = KEYS * DQ * 2, V_TILE = KEYS * VP * 2;
  static_assert((KC * KEYS) % 64 == 0 && (VC * KEYS) % 64 == 0, "whole loads");
  constexpr int LS = NA / 2;                           // slots with loads, from the first
  constexpr int AHEAD = 4, TOP = 3;                    // slots that a fragment is read ahead; first slot with exponentials
  static_assert(NA >= AHEAD && NB >= AHEAD && NA > TOP, "slots");
  typedef TileRows<KC> KR;
  typedef TileRows<VC> VR;
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, hh = lane >> 5, group = GROUPS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const uint32_t base = (uint32_t)(uintptr_t)lds + group * prompt_lds_bytes<DQ, VP, 1, KEYS>();
  if (GROUPS == 2 && group >= work.groups) return;
  const int n_turns = __builtin_amdgcn_readfirstlane(work.n_turns);

  // load i of this wave: chunks 64 (wave + 4 i) + lane of the tile
  // (96 columns of 32 keys: the last load is of two waves only)
  constexpr bool K_PART = KC * KEYS % 256 != 0, V_PART = VC * KEYS % 256 != 0;
  auto k_row = [&](int i) __attribute__((always_inline)) {
    const int r = (int)((64u * (wave + 4 * i) + lane) / KC);
    return K_PART ? min(r, KEYS - 1) : r;
  };
  auto v_row = [&](int i) __attribute__((always_inline)) {
    const int r = (int)((64u * (wave + 4 * i) + lane) / VC);
    return V_PART ? min(r, KEYS - 1) : r;
  };
  // (skipped inside the asm statement: a branch around it would let the compiler move the vector work between the blocks)
  auto to_lds = [&](const void* src, uint32_t dst, int on) __attribute__((always_inline)) {
    asm volatile("s_cmp_eq_u32 %2, 0\n\ts_cbranch_scc1 1f\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off\n1:"
                 : : "v"(src), "s"(dst), "s"(__builtin_amdgcn_readfirstlane(on)) : "memory", "m0", "scc");
  };
  auto load_k = [&](int i, int handle, int buf, int on) __attribute__((always_inline)) {
    const int r = k_row(i), c = (int)((64u * (wave + 4 * i) + lane) % KC);
    if (K_PART) on = on && 64 * (wave + 4 * i) < KC * KEYS;
    to_lds(work.key(handle, c ^ KR::k_turn(r)), base + buf * K_TILE + 1024 * (wave + 4 * i), on);
  };
  auto load_v = [&](int i, int handle, int buf, int on) __attribute__((always_inline)) {
    const int r = v_row(i), c = (int)((64u * (wave + 4 * i) + lane) % VC);
    if (V_PART) on = on && 64 * (wave + 4 * i) < VC * KEYS;
    to_lds(work.value(handle, c ^ VR::v_turn(r)), base + 2 * K_TILE + buf * V_TILE + 1024 * (wave + 4 * i), on);
  };
  auto landed = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  // fragments: K row l31 (+ 32 n), chunk 2 s + hh; V by the transpose read: key 4 hh + (lane % 16) / 4 of every 8,
  // columns 16 (lane / 16 % 2) + 4 (lane % 4)
  uint32_t k_lane = base + l31 * (DQ * 2), k_at = (hh ^ KR::k_turn(l31)) * 16;
  const int v_l = (lane & 15) >> 2;
  uint32_t v_lane = base + 2 * K_TILE + (4 * hh + v_l) * (VP * 2) + (lane & 1) * 8 + (((lane >> 4) & 1) * 2 + ((lane & 3) >> 1)) * 16;
  uint32_t v_x = VR::v_turn(v_l) * 16;
  auto read_k = [&](int buf, int i) __attribute__((always_inline)) {   // product i: keys 32 (i % N), step i / N
    const int c = 2 * (i / N);
    const uint32_t ad = (k_at ^ ((c & KR::K_MASK) * 16)) + (k_lane + buf * K_TILE) + (i % N * 32 * DQ * 2 + (c & ~KR::K_MASK) * 16);
    return *(lds_frag*)(uintptr_t)ad;
  };
  auto read_v = [&](int buf, int i) __attribute__((always_inline)) {   // product i: keys 16 (i / DT), columns 32 (i % DT)
    const int f = i / DT, d = i % DT;
    const uint32_t ad = (v_x ^ ((d & VR::V_MASK) * 64)) + (v_lane + buf * V_TILE) + (16 * f * VP * 2 + (d & ~VR::V_MASK) * 64);
    const tr_v4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_lds_v4*)(uintptr_t)ad);
    const tr_v4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_lds_v4*)(uintptr_t)(ad + 16 * VP));
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  constexpr f32x16 zero = {};
  // (the sums stay in one place over the branches: without it they are copied, which spills at width 128)
  auto whole = [](f32x16(&x)[DT]) __attribute__((always_inline)) {
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      if constexpr (DQ + VP >= 512) asm volatile("" : "+a"(x[d]));
      else asm volatile("" : "+v"(x[d]));
    }
  };

#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = zero;
  m_run = M_INIT_F, l_run = 0.f;

  f32x16 s[N], sn[N];                                  // scores of the present tile, products of the next
  bf16x8_t fr[AHEAD];
  auto score_slot = [&](auto slot, auto slots) __attribute__((always_inline)) {
    constexpr int e0 = slot * 16 * N / slots, e1 = (slot + 1) * 16 * N / slots;
#pragma unroll
    for (int e = e0; e < e1; ++e) {
      float x = work.score(sn[e >> 4][e & 15]);
      asm volatile("" : "+v"(x));                      // (stays in its slot)
      s[e >> 4][e & 15] = x;
    }
  };
  auto product_a = [&](auto i, int buf) __attribute__((always_inline)) {
    sn[i % N] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[i % AHEAD], qf[i / N], i < N ? zero : sn[i % N], 0, 0, 0);
    if constexpr (i + AHEAD < NA) fr[i % AHEAD] = read_k(buf, i + AHEAD);
  };

  work.start();
#pragma unroll
  for (int i = 0; i < KL; ++i) load_k(i, work.row(0, k_row(i)), 0, 1);
#pragma unroll
  for (int i = 0; i < KL; ++i) load_k(i, work.row(1, k_row(i)), 1, n_turns > 1);
#pragma unroll
  for (int i = 0; i < VL; ++i) load_v(i, work.row(0, v_row(i)), 0, 1);
  // (the first tile's keys are waited for alone, which is 3 to 8 % of chains of three tiles; a wave has at least these loads behind them)
  constexpr int K_BEHIND = KC * KEYS / 256, V_BEHIND = VC * KEYS / 256;
  if (n_turns > 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(K_BEHIND + V_BEHIND) : "memory");
  else asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(V_BEHIND) : "memory");
  unrolled<AHEAD>([&](auto i) __attribute__((always_inline)) { fr[i] = read_k(0, i); });
  unrolled<NA>([&](auto i) __attribute__((always_inline)) { product_a(i, 0); });
  score_slot(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
  landed();   // (the first tile of K is read before the third is loaded over it)

  // The last turn is code of its own: there is no tile behind it whose scores to multiply and cap, a quarter of a chain of three tiles' (us: latent 64 + 32 / 64
  // columns, 32 heads, 16 x 512 rows by a window of 64 47 / 44; window 128 wide with a cap, 16 heads, 4096 rows 108 / 103, 32 heads, 8 x 512 rows of 2200 to 3584
  // 229 / 222).
  auto one_turn = [&](int turn, auto is_last) __attribute__((always_inline)) {
    constexpr bool LAST = decltype(is_last)::value;
    const int b = turn & 1, more_k = turn + 2 < n_turns;
    if (!LAST) work.begin(turn);
    asm volatile("" : "+v"(k_at), "+v"(v_x), "+v"(k_lane), "+v"(v_lane));   // (their combinations are not kept over the turns)
    int rows[KL + VL];
    auto row = [&](auto l) __attribute__((always_inline)) {
      if constexpr (l < KL) rows[l] = work.row(turn + 2, k_row(l));
      else if constexpr (l < KL + VL) rows[l] = work.row(turn + 1, v_row(l - KL));
    };
    if constexpr (!LAST) {
      unrolled<2>(row);
      unrolled<AHEAD>([&](auto i) __attribute__((always_inline)) { fr[i] = read_k(1 - b, i); });
    }
    work.mask(turn, s);
    whole(o);
    __builtin_amdgcn_sched_barrier(0);
    float mx = s[0][0], m_new = 0.f, alpha = 0.f, sum = 0.f;
    u32x4 pw[2 * N];
    unrolled<NA>([&](auto i) __attribute__((always_inline)) {
      constexpr int slot = i;
      if constexpr (!LAST) product_a(i, 1 - b);
      if constexpr (slot + AHEAD >= NA) fr[slot % AHEAD] = read_v(b, slot + AHEAD - NA);
      constexpr int l0 = std::min(slot * (KL + VL) / LS, KL + VL), l1 = std::min((slot + 1) * (KL + VL) / LS, KL + VL);
      unrolled<LAST ? 0 : l1 - l0>([&](auto e) __attribute__((always_inline)) {
        constexpr int l = l0 + e;
        if constexpr (l < KL) load_k(l, rows[l], b, more_k);
        else load_v(l - KL, rows[l], 1 - b, 1);
        row(std::integral_constant<int, l + 2>{});
      });
      if constexpr (slot < 2) {
#pragma unroll
        for (int r = 0; r < 8 * N; ++r) mx = fmaxf(mx, s[slot * N / 2][N == 1 ? 8 * slot + r : r]);
      } else if constexpr (slot < TOP) {
        const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1]));
        m_new = fmaxf(m_run, work.top(mx));
        alpha = fast_exp2(m_run - m_new);
        m_run = m_new;
      } else {
        constexpr int p0 = (slot - TOP) * 8 * N / (NA - TOP), p1 = (slot + 1 - TOP) * 8 * N / (NA - TOP);
        unrolled<p1 - p0>([&](auto e) __attribute__((always_inline)) {
          constexpr int p = p0 + e, n = p / 8, r = 2 * (p % 8);
          const float e0 = fast_exp2(work.below(s[n][r], m_new)), e1 = fast_exp2(work.below(s[n][r + 1], m_new));
          sum += e0 + e1;
          uint32_t w = pack2<bf16_tag>(e0, e1);
          asm volatile("" : "+v"(w), "+v"(sum));       // (stays in its slot)
          pw[p / 4][p % 4] = w;
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    l_run = l_run * alpha + sum;
    if (__any(alpha != 1.0f)) {
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
    }
    whole(o);
    __builtin_amdgcn_sched_barrier(0);
    if (work.seen(turn)) {
      unrolled<NB>([&](auto i) __attribute__((always_inline)) {
        constexpr int slot = i, d = slot % DT;
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[(slot + NA) % AHEAD], __builtin_bit_cast(bf16x8_t, pw[slot / DT]), o[d], 0, 0, 0);
        if constexpr (slot + AHEAD < NB) fr[(slot + NA) % AHEAD] = read_v(b, slot + AHEAD);
        if constexpr (!LAST) score_slot(i, std::integral_constant<int, NB>{});
        __builtin_amdgcn_sched_barrier(0);
      });
    } else if constexpr (!LAST) {                      // (no row of the wave sees a key of this tile: p is 0, V is not touched)
      unrolled<1>([&](auto i) __attribute__((always_inline)) { score_slot(i, std::integral_constant<int, 1>{}); });
    }
    if constexpr (!LAST) {
      work.end(turn);
      landed();
    }
  };
  for (int turn = 0; turn + 1 < n_turns; ++turn) one_turn(turn, std::false_type{});
  one_turn(n_turns - 1, std::true_type{});

  whole(o);
  l_run += __shfl_xor(l_run, 32, 64);
  if constexpr (GROUPS == 2) {
    if (work.groups == 1) return;
    lds_barrier();                                     // (the last tiles are read)
    static_assert(DT * 4 * 256 * 16 + 2048 <= prompt_lds_bytes<DQ, VP, 2, KEYS>(), "the sums of the second group");
    float* const ml = reinterpret_cast<float*>(lds) + tid;
    f32x4* const part = reinterpret_cast<f32x4*>(lds + 2048) + tid;
    if (group) {
      ml[0] = m_run, ml[256] = l_run;
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int r = 0; r < 16; r += 4) part[(4 * d + r / 4) * 256] = f32x4{o[d][r], o[d][r + 1], o[d][r + 2], o[d][r + 3]};
    }
    lds_barrier();
    if (group) return;
    const float m1 = ml[0], top = fmaxf(m_run, m1), f0 = fast_exp2(m_run - top), f1 = fast_exp2(m1 - top);
    m_run = top, l_run = l_run * f0 + ml[256] * f1;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int r = 0; r < 16; r += 4) {
        const f32x4 p = part[(4 * d + r / 4) * 256];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[d][r + j] = o[d][r + j] * f0 + p[j] * f1;
      }
  }
}

}  // namespace slm
