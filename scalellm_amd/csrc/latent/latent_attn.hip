// latent_attn.hip -- attention of single query rows over the paged latent cache ("absorbed" form: the
// unrotated query is already multiplied by W_uk, so every head scores against the cached row itself and
// accumulates the cached latent; W_uv is applied to the result).  All heads share every cache byte.
//
// Work item: (query row, block of 16 MH heads, split of its visible range).  Visible = positions
// [max(0, p - window + 1), p] of the row's sequence; a portion of several tokens is several rows.
//
// latent_attn_kernel (bf16, MFMA 16x16x32), eight waves, 32 cache rows per tile, a ring of four to eight tiles in LDS:
//   staging   global -> LDS by LDS-DMA (a wave instruction writes 1 KiB linearly), all but one tile of the ring in flight
//             behind counted waits; block-table entries of the range are staged in LDS first (LA_TBL at a time), so
//             no other load sits in the vmcnt queue.  The image is swizzled on the source side: 16-byte unit u of row r holds chunk
//             u ^ (r / 2 % 8), which keeps both fragment reads below off each other's banks
//   S = C Q^T 16 x 16 blocks, one a wave (16 heads: half a contraction each), A = cache rows, B = the wave's head
//             block, held in registers; S to LDS.  One tile AHEAD of the rest, so that a tile costs one barrier and a
//             wave's soft-max has another tile's products to hide behind
//   softmax   every wave reads the scores back in the B layout of the second product (column = head = lane % 16,
//             8 consecutive keys) and does the row statistics itself: no second exchange, one scalar per lane
//   O^T += C^T P^T   a wave owns an eighth of the latent columns (several head blocks: a quarter of them for half of the blocks); A = C^T out of the row-major tile by the transpose
//             read (ds_read_b64_tr_b16: 4 keys of one column per lane)
// Bound: HBM (the cache stream) for 16 heads, 128 rows of 4096 keys 5.5 TB/s; with 32 the soft-max every wave repeats, between two
// barriers, is as long as the stream (the same with every tile out of the L2: 104 us).  32 heads, 128 rows of 4096 keys: 126 us with
// the soft-max of both head blocks in every wave and a 64-bit address per lane and row, 110 with half of it and one address a tile;
// 64 rows of 500 - 1000 keys 32.5 -> 30.6.  Ranges that are split leave fp32 partials for latent_attn_combine_kernel.
//
// latent_attn_any_kernel: any size, any dtype, VALU: the 32-bit path and sizes without an MFMA form.
#include <algorithm>

#include "latent_common.h"
#include "tile_common.h"

namespace slm {

constexpr int LA_MAX_SPLITS = 128;
constexpr int LA_VALUES_WEIGHTS = 512;   // rows and splits of a workgroup of latent_values_kernel

struct LatentAttnK {
  slm_latent_attn_args a;
  int n_splits;
  float* o_part;   // [rows][heads][n_splits][c_pad]
  float* ml_part;  // [rows][heads][n_splits][2]
  float scale2;    // scale * log2(e)
  int block_shift, block_mask;
  int mh;          // head blocks of 16 per workgroup
  bool stream;     // the cache is read past the caches' replacement
};

typedef short tr_v4 __attribute__((ext_vector_type(4)));
typedef short tr_v8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) tr_v4 tr_lds_v4;

// maximum over the four lanes that share lane % 16
__device__ __forceinline__ float max_over_groups(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// waits until at most `tiles` tiles of PER DMA instructions each are in flight (0 <= tiles <= MAX)
template <int MAX, int PER>
__device__ __forceinline__ void wait_tiles(int tiles) {
  if constexpr (MAX > 0) {
    if (tiles < MAX) return wait_tiles<MAX - 1, PER>(tiles);
  }
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(MAX * PER) : "memory");
}

constexpr int LA_KT = 32;     // cache rows per tile
constexpr int LA_TBL = 1024;  // block-table entries staged in LDS at a time

template <int KP, int RP, int MH>
__global__ void __launch_bounds__(512) latent_attn_kernel(const LatentAttnK p) {
  constexpr int R = KP + RP;
  constexpr int KT = LA_KT;
  constexpr int CH = R / 8;                  // 16-byte chunks of a cache row
  constexpr int CHP = (CH + 7) / 8 * 8;      // 16-byte units of a row in LDS
  constexpr int ROWB = CHP * 16, TILE = KT * ROWB;
  constexpr int NTOT = KT * CHP / 64;        // DMA instructions of a tile: NHI in the first NTOT % 8 waves, NLO in the others
  constexpr int NHI = (NTOT + 7) / 8, NLO = NTOT / 8;
  constexpr int QS = R / 32;                 // MFMA k-steps of the scores
  constexpr int KH = MH == 1 ? 2 : 1;        // waves that share a score block's contraction
  constexpr int QW = (QS + KH - 1) / KH;     // k-steps per wave
  constexpr int HS = MH == 1 ? 1 : 2;        // groups of head blocks: a wave takes one, MG blocks,
  constexpr int MG = MH / HS, CG = 8 / HS;   // and one of CG groups of the latent's columns,
  constexpr int NT = KP >= 16 * CG ? KP / (16 * CG) : 1;  // NT blocks of 16
  constexpr int SS = KT + 4;                 // score row stride (floats)
  constexpr int SC = KH * 16 * MH * SS;      // floats of one tile's scores
  constexpr int FIT = (163840 - 8 * SC - 4 * LA_TBL) / TILE, NBUF = FIT > 8 ? 8 : FIT;  // tiles in the ring
  static_assert(NBUF >= 4 && (NBUF - 3) * NHI < 63, "ring and counted waits");
  __shared__ __attribute__((aligned(16))) char ring[NBUF * TILE];
  __shared__ __attribute__((aligned(16))) float sc[2][SC];
  __shared__ int tbl[LA_TBL];

  const slm_latent_attn_args& a = p.a;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int hblocks = (a.heads + 16 * MH - 1) / (16 * MH);
  // head blocks of one (row, split) sit 8 blocks apart in the grid: they share a cache range and, dispatched
  // round-robin over the 8 XCDs, an L2
  const int64_t items = a.rows * p.n_splits;
  const int64_t group = blockIdx.x / (8 * hblocks), in_group = blockIdx.x % (8 * hblocks);
  const int64_t item = group * 8 + in_group % 8;
  const int hb = (int)(in_group / 8);
  if (item >= items) return;
  const int64_t row = item / p.n_splits;
  const int split = (int)(item % p.n_splits);
  const int h0 = hb * 16 * MH;

  // score block of this wave: head block hw, key block kb, k-steps from kh * QW
  const int kb = wave & 1, hw = (wave >> 1) & (MH - 1), kh = KH == 2 ? (wave >> 1) & 1 : 0;
  const bool scorer = wave < 2 * MH * KH;
  bf16x8_t qf[QW];
  {
    const int h = h0 + 16 * hw + l16;
    const bf16* q = reinterpret_cast<const bf16*>(a.q_abs) + (row * a.heads + min(h, a.heads - 1)) * R + 8 * g;
#pragma unroll
    for (int s = 0; s < QW; ++s) {
      const int step = kh * QW + s;
      qf[s] = *reinterpret_cast<const bf16x8_t*>(q + 32 * min(step, QS - 1));
      if (KH * QW != QS && step >= QS) qf[s] = __builtin_bit_cast(bf16x8_t, u32x4{0u, 0u, 0u, 0u});
    }
  }

  // decode batches: row r is sequence r.  Looked up as if, all loads at once; otherwise the search
  const int guess = min((int)row, a.batch - 1);
  const int g0 = a.q_cu[guess], g1 = a.q_cu[guess + 1], pos = a.positions[row];
  int bcu = a.block_cu[guess];
  if (g0 != (int)row || g1 != (int)row + 1) bcu = a.block_cu[seq_of_row(a.q_cu, a.batch, (int)row)];
  int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  int hi = pos + 1;
  if (p.n_splits > 1) {
    const int first = lo & -KT, tiles = (hi - first + KT - 1) / KT;
    const int per = (tiles + p.n_splits - 1) / p.n_splits * KT;
    lo = min(hi, max(lo, first + split * per));
    hi = min(hi, first + (split + 1) * per);
  }
  // (the queries have arrived before the first DMA is issued: a wait for them later would drain the ring)
#pragma unroll
  for (int s = 0; s < QW; ++s) asm volatile("" : "+v"(qf[s]));

  // the segment of the range whose block-table entries are staged: keys [lo, hi), in tiles from the multiple of KT at or before lo
  const int range_hi = hi;
  int blk0 = 0, n_tiles = 0, base = 0;
  const uint32_t ring0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring;
  const char* cache = reinterpret_cast<const char*>(a.cache);
  uint32_t from[NHI];   // where this lane's pieces lie in a tile of consecutive rows
#pragma unroll
  for (int i = 0; i < NHI; ++i) {
    const int u = min(wave + 8 * i, NTOT - 1) * 64 + lane, r = u / CHP;
    from[i] = (uint32_t)(r * (R * 2) + 16 * min((u % CHP) ^ ((r >> 1) & 7), CH - 1));
  }
  auto entry = [&](int t) { return tbl[(min(max(base + t * KT, lo), hi - 1) >> p.block_shift) - blk0]; };
  // A whole tile within a block of the cache: one uniform address.  Else a row at a time (rows there are not re-read the first or the last
  // there is; masked below).  (16 heads, every tile out of the L2: 95 us -> 82.)
  // (inline asm: through the builtin the compiler makes every read of the ring wait for the DMA into its other tiles)
  auto issue = [&](int t, int first_slot) {
    const uint32_t dst0 = ring0 + (uint32_t)(t % NBUF) * TILE;
    const int k0 = base + t * KT;
    if (p.block_shift >= 5 && k0 >= lo && k0 + KT <= hi) {
      const char* src = cache + (int64_t)(__builtin_amdgcn_readfirstlane(first_slot) + (k0 & p.block_mask)) * (R * 2);
      if (p.stream) {
#pragma unroll
        for (int i = 0; i < NHI; ++i)
          if (i < NLO || wave < NTOT % 8)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt"
                         :
                         : "v"(from[i]), "s"(src), "s"(dst0 + (uint32_t)(wave + 8 * i) * 1024u)
                         : "memory", "m0");
      } else {
#pragma unroll
        for (int i = 0; i < NHI; ++i)
          if (i < NLO || wave < NTOT % 8)
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                         :
                         : "v"(from[i]), "s"(src), "s"(dst0 + (uint32_t)(wave + 8 * i) * 1024u)
                         : "memory", "m0");
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < NHI; ++i) {
      const uint32_t r = from[i] / (R * 2), c = from[i] % (R * 2);
      const int key = max(lo, min(k0 + (int)r, hi - 1));
      const int slot = tbl[(key >> p.block_shift) - blk0];
      const char* src = cache + (int64_t)(slot + (key & p.block_mask)) * (R * 2) + c;
      if (i < NLO || wave < NTOT % 8)
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                     :
                     : "v"(src), "s"(dst0 + (uint32_t)(wave + 8 * i) * 1024u)
                     : "memory", "m0");
    }
  };

  f32x4 o[MG][NT];
  float m_run[MG], l_run[MG];
#pragma unroll
  for (int m = 0; m < MG; ++m) {
    m_run[m] = M_INIT_F;
    l_run[m] = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) o[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // fragment reads: A of the scores (row l16 of a 16-key block, chunk 4 i + g), and the transpose read (keys
  // 8 g + l16 / 4 and + 4, 8-byte piece l16 % 4 of a 16-column block)
  const uint32_t k_row = (uint32_t)l16 * ROWB, k_x = (uint32_t)((l16 >> 1) & 7) ^ (uint32_t)g;
  const uint32_t tr_row = (uint32_t)(8 * g + (l16 >> 2)) * ROWB + (uint32_t)(l16 & 1) * 8u;
  const uint32_t tr_x0 = (uint32_t)((4 * g + (l16 >> 3)) & 7) ^ (uint32_t)((l16 >> 1) & 1);
  const uint32_t tr_x1 = (uint32_t)((4 * g + 2 + (l16 >> 3)) & 7) ^ (uint32_t)((l16 >> 1) & 1);
  const int hg = wave / CG, cg = wave % CG;
  const uint32_t tr_c = (uint32_t)cg * (2 * NT);
  const bool columns = cg < KP / (16 * NT);

  constexpr int QC = QW > 10 ? (QW + 2) / 3 : QW;   // k-steps read ahead of the products (register budget)
  bf16x8_t kf[QC];
  auto read_rows = [&](int t, int first) {   // A fragments of tile t, k-steps from `first` of this wave's
    const uint32_t base = ring0 + (uint32_t)(t % NBUF) * TILE + (uint32_t)(16 * kb) * ROWB + k_row;
#pragma unroll
    for (int i = 0; i < QC; ++i) {
      const uint32_t step = (uint32_t)(kh * QW + first + i);
      kf[i] = *(__attribute__((address_space(3))) const bf16x8_t*)(uintptr_t)(base + (((4u * min(step, (uint32_t)QS - 1)) ^ k_x) << 4));
    }
  };
  auto score = [&](int t) {
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < QW; c += QC) {
      if (c > 0) read_rows(t, c);
#pragma unroll
      for (int i = 0; i < QC; i += 2) {
        if (c + i < QW) s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[i], qf[c + i], s0, 0, 0, 0);
        if (i + 1 < QC && c + i + 1 < QW) s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[i + 1], qf[c + i + 1], s1, 0, 0, 0);
      }
    }
    // lane: head l16, keys 16 kb + 4 g .. + 3
    *reinterpret_cast<f32x4*>(&sc[t & 1][(16 * (MH * kh + hw) + l16) * SS + 16 * kb + 4 * g]) = s0 + s1;
  };
  auto arrived = [&](int younger) {   // the wave's part of a tile, with the younger tiles of the ring still in flight
    if (NTOT % 8 == 0 || wave < NTOT % 8) wait_tiles<NBUF - 2, NHI>(younger);
    else wait_tiles<NBUF - 2, NLO>(younger);
  };
  for (; lo < range_hi; lo = hi) {
    blk0 = lo >> p.block_shift;
    hi = min(range_hi, (blk0 + LA_TBL) << p.block_shift);
    base = lo & -KT;
    n_tiles = (hi - base + KT - 1) / KT;
    for (int i = tid; i <= ((hi - 1) >> p.block_shift) - blk0; i += 512) tbl[i] = a.block_table[bcu + blk0 + i];
    __syncthreads();
#pragma unroll 1
    for (int t = 0; t < min(NBUF - 1, n_tiles); ++t) issue(t, entry(t));
    int slot = entry(NBUF - 1);   // (of the tile issued next: read a tile ahead)
    arrived(min(NBUF - 2, n_tiles - 1));
    lds_barrier();
    if (scorer) {
      read_rows(0, 0);
      score(0);
    }
    for (int t = 0; t < n_tiles; ++t) {
      const int k0 = base + t * KT;
      if (t + 1 < n_tiles) arrived(min(NBUF - 3, n_tiles - 2 - t));
      lds_barrier();   // tile t + 1 and the scores of tile t are there, tile t - 1 is done with
      if (t + NBUF - 1 < n_tiles) issue(t + NBUF - 1, slot);
      slot = entry(t + NBUF);
      const uint32_t tile = ring0 + (uint32_t)(t % NBUF) * TILE;
      const bool next = scorer && t + 1 < n_tiles;
      if (next) read_rows(t + 1, 0);
      if (!columns) {   // (a latent of 64: four waves hold all of it)
        if (next) score(t + 1);
        continue;
      }
      // ---- scores back in the B layout of the second product, C^T fragments behind them (read under the soft-max)
      f32x4 raw[MG][KH][2];
#pragma unroll
      for (int m = 0; m < MG; ++m)
#pragma unroll
        for (int k = 0; k < KH; ++k) {
          const float* sp = &sc[t & 1][(16 * (MH * k + MG * hg + m) + l16) * SS + 8 * g];
          raw[m][k][0] = *reinterpret_cast<const f32x4*>(sp);
          raw[m][k][1] = *reinterpret_cast<const f32x4*>(sp + 4);
        }
      __builtin_amdgcn_sched_barrier(0);
      tr_v8 ct[NT];
#pragma unroll
      for (int t2 = 0; t2 < NT; ++t2) {
        const uint32_t cc = tr_c + 2u * t2, ad = tile + tr_row;
        const tr_v4 c0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_lds_v4*)(uintptr_t)(ad + ((cc ^ tr_x0) << 4)));
        const tr_v4 c1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_lds_v4*)(uintptr_t)(ad + 4 * ROWB + ((cc ^ tr_x1) << 4)));
        ct[t2] = __builtin_shufflevector(c0, c1, 0, 1, 2, 3, 4, 5, 6, 7);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (next) score(t + 1);
      // ---- soft-max
      const bool cut = k0 < lo || k0 + KT > hi;
      bf16x8_t pf[MG];
#pragma unroll
      for (int m = 0; m < MG; ++m) {
        float v[8];
        float mx = M_INIT_F;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float x = raw[m][0][j >> 2][j & 3];
#pragma unroll
          for (int k = 1; k < KH; ++k) x += raw[m][k][j >> 2][j & 3];
          v[j] = x * p.scale2;
        }
        if (cut)
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (k0 + 8 * g + j < lo || k0 + 8 * g + j >= hi) v[j] = -INFINITY;
#pragma unroll
        for (int j = 0; j < 8; ++j) mx = fmaxf(mx, v[j]);
        mx = max_over_groups(mx);
        const float m_new = fmaxf(m_run[m], mx);
        const float alpha = fast_exp2(m_run[m] - m_new);
        m_run[m] = m_new;
        float sum = 0.f;
        u32x4 w;
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          const float e0 = fast_exp2(v[j] - m_new), e1 = fast_exp2(v[j + 1] - m_new);
          sum += e0 + e1;
          w[j >> 1] = pack2<bf16_tag>(e0, e1);
        }
        pf[m] = __builtin_bit_cast(bf16x8_t, w);
        l_run[m] = l_run[m] * alpha + sum;
        if (__any(alpha != 1.0f)) {
#pragma unroll
          for (int t2 = 0; t2 < NT; ++t2) o[m][t2] *= alpha;
        }
      }
      // ---- O^T += C^T P^T
#pragma unroll
      for (int t2 = 0; t2 < NT; ++t2)
#pragma unroll
        for (int m = 0; m < MG; ++m)
          o[m][t2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ct[t2]), pf[m], o[m][t2], 0, 0, 0);
    }
    lds_barrier();   // ring and table are free for the next segment
  }

  // The accumulators (lane: head l16 of a block, latent columns 16 NT cg + 16 t + 4 g .. + 3) go through the ring, so
  // that whole lines leave the chip: straight from the registers a store touches 64 bytes of 16 rows.
  constexpr int OS = KP + 4;   // row stride (floats)
  static_assert(16 * MH * OS * 4 <= NBUF * TILE, "the output tile fits the ring");
  float* ot = reinterpret_cast<float*>(ring);
#pragma unroll
  for (int m = 0; m < MG; ++m) {
    const int hr = 16 * (MG * hg + m) + l16;
    if (columns) {
#pragma unroll
      for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(ot + hr * OS + cg * (16 * NT) + 16 * t + 4 * g) = o[m][t];
    }
    float l = l_run[m];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (cg == 0 && g == 0) {
      sc[0][hr] = m_run[m];
      sc[1][hr] = l;
    }
  }
  __syncthreads();
  const int n_heads = min(16 * MH, a.heads - h0);
  for (int i = tid; i < n_heads * (KP / 4); i += 512) {
    const int hr = i / (KP / 4), c = i % (KP / 4) * 4;
    const int64_t rh = row * a.heads + h0 + hr;
    f32x4 v = *reinterpret_cast<const f32x4*>(ot + hr * OS + c);
    if (p.n_splits == 1) {
      v *= 1.0f / sc[1][hr];  // (every row sees itself: the sum is positive)
      *reinterpret_cast<u32x2*>(reinterpret_cast<bf16*>(a.out) + rh * KP + c) =
          u32x2{pack2<bf16_tag>(v.x, v.y), pack2<bf16_tag>(v.z, v.w)};
    } else {
      *reinterpret_cast<f32x4*>(p.o_part + (rh * p.n_splits + split) * KP + c) = v;
    }
  }
  if (p.n_splits > 1 && tid < n_heads) {
    const int64_t pi = (row * a.heads + h0 + tid) * p.n_splits + split;
    p.ml_part[2 * pi] = sc[0][tid];
    p.ml_part[2 * pi + 1] = sc[1][tid];
  }
}

// Merges the splits.  A workgroup takes 256 / G groups of four columns, G threads share a group's splits.
template <int G>
__global__ void __launch_bounds__(256) latent_attn_combine_kernel(const LatentAttnK p) {
  constexpr int Q = 256 / G;
  __shared__ f32x4 part[G > 1 ? G : 1][Q];
  const int n = p.n_splits, c4 = p.a.c_pad / 4, tid = threadIdx.x;
  const int64_t quad = (int64_t)blockIdx.x * Q + tid % Q;
  if (G == 1 && quad >= p.a.rows * p.a.heads * c4) return;   // (G > 1: whole workgroups, c4 % Q == 0)
  const int64_t rh = quad / c4;
  const int c = (int)(quad % c4) * 4, sg = tid / Q;
  const float* ml = p.ml_part + 2 * rh * n;
  const float* src = p.o_part + rh * n * p.a.c_pad + c;
  float m, inv;
  if constexpr (G == 1) {
    m = M_INIT_F;
    for (int s = 0; s < n; ++s) m = fmaxf(m, ml[2 * s]);
    float l = 0.f;
    for (int s = 0; s < n; ++s) l += ml[2 * s + 1] * fast_exp2(ml[2 * s] - m);
    inv = 1.0f / l;
  } else {
    // every wave the same statistics: two splits per lane
    const int lane = tid & 63;
    const float m0 = lane < n ? ml[2 * lane] : M_INIT_F, m1 = lane + 64 < n ? ml[2 * lane + 128] : M_INIT_F;
    const float l0 = lane < n ? ml[2 * lane + 1] : 0.f, l1 = lane + 64 < n ? ml[2 * lane + 129] : 0.f;
    m = wave_max(fmaxf(m0, m1));
    inv = 1.0f / wave_sum(l0 * fast_exp2(m0 - m) + l1 * fast_exp2(m1 - m));
  }
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = sg; s < n; s += G) o += *reinterpret_cast<const f32x4*>(src + (int64_t)s * p.a.c_pad) * fast_exp2(ml[2 * s] - m);
  if constexpr (G > 1) {
    part[sg][tid % Q] = o;
    __syncthreads();
    if (sg) return;
#pragma unroll
    for (int s = 1; s < G; ++s) o += part[s][tid % Q];
  }
  o *= inv;
  *reinterpret_cast<u32x2*>(reinterpret_cast<bf16*>(p.a.out) + rh * p.a.c_pad + c) =
      u32x2{pack2<bf16_tag>(o.x, o.y), pack2<bf16_tag>(o.z, o.w)};
}

// The splits' merge and what is multiplied out behind it (W_uv and the output gate, v) in one launch.  A workgroup has rows_per rows of a
// head, all their columns and up to 128 of the product's: the merged rows lie in LDS in 16-bit, W comes there by LDS-DMA while the splits are read, a
// wave owns 16 columns.  16-byte chunk c of row r lies in slot c ^ (r & SW).
// Bound: latency, and 130 - 190 KB a CU of splits and W.  With the attention in front of it, us, two launches / this, latent 512 -> 128, 4000 keys:
// 16 heads 8 rows 21.7 / 20.2, 32 rows 40.0 / 36.7, 128 rows 111.6 / 104.0; 32 heads 4 rows 20.1 / 19.4, 32 rows 45.8 / 42.1, 128 rows 114.5 / 109.1.
template <int KP>
__global__ void __launch_bounds__(512) latent_values_kernel(const LatentAttnK p, const slm_linear_args v, const int rows_per) {
  constexpr int C4 = KP / 4, PH = 512 / C4, SW = KP >= 128 ? 15 : 7, U = 8;
  __shared__ __attribute__((aligned(16))) char merged[16 * KP * 2];
  __shared__ float weight[LA_VALUES_WEIGHTS], total[16];
  __shared__ f32x4 part[PH][C4];
  extern __shared__ __attribute__((aligned(16))) char w_lds[];   // [8 waves][16 columns][KP]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
  const int head = blockIdx.x, n = p.n_splits;   // (heads go round the XCDs: a head's workgroups share W in an L2)
  const int64_t row0 = (int64_t)blockIdx.y * rows_per;
  const int rows = (int)min((int64_t)rows_per, p.a.rows - row0);
  auto pair = [&](int r) { return (row0 + r) * p.a.heads + head; };

  // threads: column quad, and a row or (fewer rows than phases) a share of a row's splits
  const int c4 = tid % C4, phase = tid / C4;
  int row_phases = PH;
  while (row_phases > 1 && row_phases / 2 >= rows) row_phases /= 2;
  const int shares = PH / row_phases, sg = phase / row_phases, r_first = phase % row_phases;
  const int per_row = (n + shares - 1) / shares, items = (rows + row_phases - 1) / row_phases * per_row;
  auto split = [&](int i) { return sg + i % per_row * shares; };
  auto load = [&](int i) {
    const int r = min(r_first + i / per_row * row_phases, rows - 1), s = min(split(i), n - 1);
    return *reinterpret_cast<const f32x4*>(p.o_part + (pair(r) * n + s) * KP + 4 * c4);
  };
  f32x4 x[U];
#pragma unroll
  for (int u = 0; u < U; ++u) x[u] = load(min(u, items - 1));

  // rows wave, wave + 8: two splits a lane
  for (int r = wave; r < rows; r += 8) {
    const float* ml = p.ml_part + 2 * pair(r) * n;
    const float m0 = lane < n ? ml[2 * lane] : M_INIT_F, m1 = lane + 64 < n ? ml[2 * lane + 128] : M_INIT_F;
    const float l0 = lane < n ? ml[2 * lane + 1] : 0.f, l1 = lane + 64 < n ? ml[2 * lane + 129] : 0.f;
    const float m = wave_max(fmaxf(m0, m1)), e0 = fast_exp2(m0 - m), e1 = fast_exp2(m1 - m), l = wave_sum(l0 * e0 + l1 * e1);
    if (lane < n) weight[r * n + lane] = e0;
    if (lane + 64 < n) weight[r * n + lane + 64] = e1;
    if (lane == 0) total[r] = 1.0f / l;
  }
  const int64_t n0 = ((int64_t)blockIdx.z * 8 + wave) * 16;
  const bool columns = n0 < v.N;
  char* const mine = w_lds + wave * (16 * KP * 2);
  if (columns) {
    const char* const w = reinterpret_cast<const char*>(v.w) + (head * v.w_batch + n0 * KP) * 2;
    const uint32_t dst0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)mine;
#pragma unroll
    for (int i = 0; i < KP / 32; ++i) {
      const int r = (i * 1024 + lane * 16) / (KP * 2), c = (lane * 16) % (KP * 2) / 16;
      const uint32_t off = (uint32_t)(r * (KP * 2) + ((c ^ (r & SW)) << 4)), dst = dst0 + i * 1024;
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" : : "v"(off), "s"(dst), "s"(w) : "memory", "m0");
    }
  }
  __syncthreads();
  auto keep = [&](int r, f32x4 o) {
    o *= total[r];
    *reinterpret_cast<u32x2*>(merged + r * (KP * 2) + (((c4 >> 1) ^ (r & SW)) << 4) + (c4 & 1) * 8) = u32x2{pack2<bf16_tag>(o.x, o.y), pack2<bf16_tag>(o.z, o.w)};
  };
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; i0 < items; i0 += U) {
    if (i0 > 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = load(min(i0 + u, items - 1));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + u, r = r_first + i / per_row * row_phases, s = split(i);
      if (i < items && r < rows) {
        if (s < n) o += x[u] * weight[r * n + s];
        if (shares == 1 && i % per_row == per_row - 1) {
          keep(r, o);
          o = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
  }
  if (shares > 1) {
    part[phase][c4] = o;
    __syncthreads();
    if (sg == 0 && r_first < rows) {
      for (int s = 1; s < shares; ++s) o += part[s * row_phases + r_first][c4];
      keep(r_first, o);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (a wave's own columns)
  __syncthreads();
  if (!columns) return;
  f32x4 y[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int s = 0; s < KP / 32; ++s) {
    const int at = r16 * (KP * 2) + (((4 * s + g) ^ (r16 & SW)) << 4);
    y[s & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t*>(mine + at), *reinterpret_cast<const bf16x8_t*>(merged + at), y[s & 1], 0, 0, 0);
  }
  if (r16 >= rows) return;
  const int64_t row = row0 + r16;
  f32x4 out = y[0] + y[1];
  if (v.epilogue == SLM_LIN_GATE) out *= sigmoid_f32(to_f32(reinterpret_cast<const bf16*>(v.gate)[row * v.ld_gate + head]));
  *reinterpret_cast<u32x2*>(reinterpret_cast<bf16*>(v.y) + head * v.y_batch + row * v.ldy + n0 + 4 * g) =
      u32x2{pack2<bf16_tag>(out.x, out.y), pack2<bf16_tag>(out.z, out.w)};
}

static void la_combine(const LatentAttnK& p, hipStream_t st) {
  const int64_t quads = p.a.rows * p.a.heads * (p.a.c_pad / 4);
  if (p.n_splits <= 8) latent_attn_combine_kernel<1><<<dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st>>>(p);
  else latent_attn_combine_kernel<16><<<dim3((unsigned)(quads / 16)), dim3(256), 0, st>>>(p);
}

constexpr int ANY_COLS = 8;  // latent columns per thread (c_pad <= 2048)

template <typename E>
__global__ void __launch_bounds__(256) latent_attn_any_kernel(const LatentAttnK p) {
  extern __shared__ float q_lds[];  // the absorbed query
  __shared__ float pr[256];
  __shared__ int slots[256];
  __shared__ float red[4];
  const slm_latent_attn_args& a = p.a;
  const int tid = threadIdx.x, R = a.c_pad + a.r_pad;
  const int64_t row = blockIdx.x / a.heads, rh = blockIdx.x;
  const int seq = seq_of_row(a.q_cu, a.batch, (int)row);
  const int pos = a.positions[row], bcu = a.block_cu[seq];
  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0, hi = pos + 1;
  const E* cache = reinterpret_cast<const E*>(a.cache);
  for (int i = tid; i < R; i += 256) q_lds[i] = to_f32(reinterpret_cast<const E*>(a.q_abs)[rh * R + i]);
  float acc[ANY_COLS];
#pragma unroll
  for (int c = 0; c < ANY_COLS; ++c) acc[c] = 0.f;
  float m = M_INIT_F, l = 0.f;
  for (int k0 = lo; k0 < hi; k0 += 256) {
    __syncthreads();
    const int key = k0 + tid;
    float s = -INFINITY;
    if (key < hi) {
      const int slot = a.block_table[bcu + (key >> p.block_shift)] + (key & p.block_mask);
      slots[tid] = slot;
      const E* r = cache + (int64_t)slot * R;
      float d = 0.f;
      for (int i = 0; i < R; i += 4) {
        float v[4];
        load_f32<4>(r + i, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) d = __builtin_fmaf(v[j], q_lds[i + j], d);
      }
      s = d * a.scale;
    }
    const float m_new = fmaxf(m, block_max256(s, red));
    const float e = key < hi ? expf(s - m_new) : 0.f;
    const float alpha = expf(m - m_new);
    pr[tid] = e;
    l = l * alpha + block_sum256(e, red);
    m = m_new;
    __syncthreads();
    const int n = min(256, hi - k0);
#pragma unroll
    for (int c = 0; c < ANY_COLS; ++c) {
      const int col = tid + 256 * c;
      if (col < a.c_pad) {
        float v = acc[c] * alpha;
        for (int j = 0; j < n; ++j) v = __builtin_fmaf(pr[j], to_f32(cache[(int64_t)slots[j] * R + col]), v);
        acc[c] = v;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < ANY_COLS; ++c) {
    const int col = tid + 256 * c;
    if (col < a.c_pad) reinterpret_cast<E*>(a.out)[rh * a.c_pad + col] = (E)(acc[c] / l);
  }
}

static int64_t la_keys(const slm_latent_attn_args& a) {
  const int64_t len = a.max_kv_len > 0 ? a.max_kv_len : 1;
  return a.window > 0 && a.window < len ? a.window : len;
}
// Head blocks of 16 per workgroup (the scores of four do not fit beside the tiles of the widest latent).  Few rows leave fewer
// splits, and fewer partials behind them, with a block to a workgroup: the blocks of a split share an L2.  It reads the keys once a
// block, though, which shows from a number of keys on that the width sets (one block / two, us; latent 512, 32 heads: 1 row x 4096 16.2 /
// 18.8, 8 x 4096 22.4 / 25.8, 20 x 4096 36.7 / 36.7, 16 x 12000 61 / 53, 23 x 32000 212 / 145; 256: 8 x 4096 19.3 / 19.7, 12 x 4096 23.4 / 22.2; 128,
// 24 heads: 8 x 1500 11.0 / 12.1, 16 x 1500 14.1 / 12.9, 16 x 12000 47 / 31; 64: 12 x 4096 15.6 / 15.8, 16 x 12000 29.6 / 26; 32 rows, 2000 -
// 4001 keys, latent 512: 50 / 42).
static int la_mh(const slm_latent_attn_args& a) {
  const int64_t few = a.c_pad >= 512 ? 90000 : a.c_pad == 256 ? 40000 : a.c_pad == 128 ? 18000 : 48000;
  if (a.rows < 24 && a.heads <= 32 && a.rows * la_keys(a) <= few) return 1;
  return a.heads > 32 && a.c_pad < 512 ? 4 : a.heads > 16 ? 2 : 1;
}
static bool la_mfma(int c_pad, int r_pad, int dtype) {
  return dtype == SLM_BF16 && (c_pad == 64 || c_pad == 128 || c_pad == 256 || c_pad == 512) && (r_pad == 32 || r_pad == 64);
}
static int la_splits(const slm_latent_attn_args& a) {
  if (!la_mfma(a.c_pad, a.r_pad, a.dtype) || a.generic) return 1;
  if (a.n_splits > 0) return a.n_splits < LA_MAX_SPLITS ? a.n_splits : LA_MAX_SPLITS;
  const int mh = la_mh(a);
  const int64_t wgs = a.rows * ((a.heads + 16 * mh - 1) / (16 * mh));
  const int64_t tiles = (la_keys(a) + LA_KT - 1) / LA_KT;
  // one round of workgroups: a ring of a wide latent fills a CU's LDS, narrow ones sit on a CU together
  const int per_cu = a.c_pad > 64 ? 1 : 2;
  int64_t n = 256 * per_cu / (wgs > 0 ? wgs : 1);
  if (n > tiles) n = tiles;
  // Four tiles a split at least, above 32 (64 for one workgroup a split and for narrow latents): the key count is a bound, of a captured graph that of its
  // longest context, and what merges the splits reads those without a key too.  Bound 4096, as many as go / this, us, 300, 1000, 2500, 4096 keys: latent 512, 16
  // heads 1 row 14.5 / 13.2, 15.3 / 13.6, 15.9 / 15.2, 16.1 / 15.4; 2 rows 17.8 / 13.6, 17.8 / 13.7, 18.3 / 16.0, 18.9 / 17.2; 32 heads 1 row 17.9 / 14.0, 17.9 / 14.0, 18.0 /
  // 16.1, 18.3 / 17.1; 256, 16 heads 2 rows 12.8 / 11.8, 12.8 / 11.8, -, 14.4 / 13.7.
  const int64_t enough = std::max<int64_t>(a.c_pad >= 512 && wgs > 1 ? 32 : 64, tiles / 4);
  if (n > enough) n = enough;
  if (n > LA_MAX_SPLITS) n = LA_MAX_SPLITS;
  return n < 1 ? 1 : (int)n;
}

template <int KP>
static void la_values_launch(const LatentAttnK& p, const slm_linear_args& v, int rows_per, hipStream_t st) {
  constexpr int bytes = 8 * 16 * KP * 2;
  auto fn = latent_values_kernel<KP>;
  static bool asked[64] = {};
  tile_allow_lds(fn, bytes, asked);
  fn<<<dim3((unsigned)p.a.heads, (unsigned)((p.a.rows + rows_per - 1) / rows_per), (unsigned)((v.N + 127) / 128)), dim3(512), bytes, st>>>(p, v, rows_per);
}
// Rows of a head per workgroup, as many as leave one round of workgroups; 0: two launches.  Those where there are fewer than 128 pairs of row and head: one
// row's 64 or 128 splits are then up to a quarter of a megabyte for each of few workgroups, where the merge by itself spreads them over the chip -- but for the
// widest latent's 32 splits and 32 pairs and more (with the attention, us, two launches / one: 32 heads 1 row of 300 keys 14.5 / 14.0, of 4096 17.6 / 17.1; 16 heads 4
// rows 15.4 / 14.7, 19.3 / 18.5).  Of values wider than a workgroup's 128 columns several workgroups merge the same splits, which pays only where all of them are one
// round (256 wide, us, two launches / one: 16 heads 8 rows of 1500 keys 17.9 / 16.5, 16 rows of 300 16.2 / 19.5; 32 heads 8 rows of 1500 20.7 / 23.8).
static int la_values_rows(const LatentAttnK& p, const slm_linear_args& v) {
  const slm_latent_attn_args& a = p.a;
  if (v.x != a.out || v.M != a.rows || v.K != a.c_pad || v.ldw != v.K || v.x_batch != a.c_pad || v.ldx != (int64_t)a.heads * a.c_pad || v.batch != a.heads ||
      v.dtype != SLM_BF16 || v.y_batch % 4 || v.ldy % 4 || (uintptr_t)v.y % 8 || v.w_batch % 8)
    return 0;
  const int64_t pairs = a.rows * a.heads;
  const int64_t r = std::min<int64_t>(16, (pairs + 255) / 256);
  const int64_t row_blocks = (a.rows + r - 1) / r;
  if (v.N > 128 && a.heads * row_blocks * ((v.N + 127) / 128) > 256) return 0;
  const bool fill = pairs >= 128 * r || (a.c_pad >= 512 && pairs >= 32 && p.n_splits <= 32);
  return fill && r * p.n_splits <= LA_VALUES_WEIGHTS && row_blocks <= 65535 ? (int)r : 0;
}

template <int KP, int RP, int MH>
static void la_launch(const LatentAttnK& p, hipStream_t st) {
  const int hblocks = (p.a.heads + 16 * MH - 1) / (16 * MH);
  const int64_t groups = (p.a.rows * p.n_splits + 7) / 8;
  latent_attn_kernel<KP, RP, MH><<<dim3((unsigned)(groups * 8 * hblocks)), dim3(512), 0, st>>>(p);
}
template <int KP, int RP>
static void la_heads(const LatentAttnK& p, hipStream_t st) {
  if (p.mh == 1) la_launch<KP, RP, 1>(p, st);
  else if (p.mh == 2) la_launch<KP, RP, 2>(p, st);
  if constexpr (KP < 512) {
    if (p.mh == 4) la_launch<KP, RP, 4>(p, st);
  }
}
template <int KP>
static void la_rot(const LatentAttnK& p, hipStream_t st) {
  if (p.a.r_pad == 32) la_heads<KP, 32>(p, st);
  else la_heads<KP, 64>(p, st);
}

static int la_check(const slm_latent_attn_args* a) {
  if (!a || a->rows < 0 || a->batch < 1 || a->heads < 1 || a->c_pad < 64 || a->c_pad % 64 || a->r_pad < 32 || a->r_pad % 32 ||
      !is_pow2(a->block_size))
    return SLM_ERR_INVALID_ARG;
  if (a->dtype != SLM_BF16 && a->dtype != SLM_F32) return SLM_ERR_UNSUPPORTED;
  if (a->c_pad > 256 * ANY_COLS || a->r_pad > 1024) return SLM_ERR_UNSUPPORTED;
  return SLM_OK;
}

}  // namespace slm

using namespace slm;

extern "C" SLM_API int slm_latent_attn_is_mfma(int32_t c_pad, int32_t r_pad, int32_t dtype) {
  return la_mfma(c_pad, r_pad, dtype) ? 1 : 0;
}
extern "C" SLM_API size_t slm_latent_attn_workspace_bytes(const slm_latent_attn_args* a) {
  if (la_check(a) != SLM_OK) return 0;
  const int n = la_splits(*a);
  return n <= 1 ? 0 : (size_t)a->rows * a->heads * n * (a->c_pad + 2) * 4;
}
static int la_run(const slm_latent_attn_args* a, const slm_linear_args* v, void* stream) {
  const int rc = la_check(a);
  if (rc != SLM_OK) return rc;
  if (!a->q_abs || !a->cache || !a->out || !a->positions || !a->q_cu || !a->block_table || !a->block_cu) return SLM_ERR_INVALID_ARG;
  if (!aligned16(a->q_abs) || !aligned16(a->cache) || !aligned16(a->out)) return SLM_ERR_ALIGNMENT;
  if (a->rows == 0) return SLM_OK;
  LatentAttnK p;
  p.a = *a;
  p.n_splits = la_splits(*a);
  p.scale2 = a->scale * LOG2E_F;
  p.block_shift = ilog2(a->block_size);
  p.block_mask = a->block_size - 1;
  p.mh = la_mh(*a);
  // a stream far beyond the caches, each row of it read by one workgroup (128 rows x 4096: 16 heads 124 -> 111 us, 32 heads 134 -> 126;
  // 8 rows, 38 MB: 26.9 -> 30)
  p.stream = a->heads <= 16 * p.mh && a->rows * la_keys(*a) * (a->c_pad + a->r_pad) * 2 >= (100ll << 20);
  p.o_part = p.ml_part = nullptr;
  if (p.n_splits > 1) {
    if (!a->workspace || !aligned16(a->workspace) || a->workspace_bytes < slm_latent_attn_workspace_bytes(a)) return SLM_ERR_WORKSPACE;
    p.o_part = (float*)a->workspace;
    p.ml_part = p.o_part + (size_t)a->rows * a->heads * p.n_splits * a->c_pad;
  }
  hipStream_t st = (hipStream_t)stream;
  hip_clear_error();
  if (!a->generic && la_mfma(a->c_pad, a->r_pad, a->dtype)) {
    switch (a->c_pad) {
      case 64: la_rot<64>(p, st); break;
      case 128: la_rot<128>(p, st); break;
      case 256: la_rot<256>(p, st); break;
      default: la_rot<512>(p, st);
    }
    if (p.n_splits > 1) {
      const int rows = v ? la_values_rows(p, *v) : 0;
      if (rows) {
        switch (a->c_pad) {
          case 64: la_values_launch<64>(p, *v, rows, st); break;
          case 128: la_values_launch<128>(p, *v, rows, st); break;
          case 256: la_values_launch<256>(p, *v, rows, st); break;
          default: la_values_launch<512>(p, *v, rows, st);
        }
        return hip_check_launch();
      }
      la_combine(p, st);
    }
  } else {
    const dim3 grid((unsigned)(a->rows * a->heads));
    const size_t lds = (size_t)(a->c_pad + a->r_pad) * 4;
    if (a->dtype == SLM_BF16) latent_attn_any_kernel<bf16><<<grid, dim3(256), lds, st>>>(p);
    else latent_attn_any_kernel<float><<<grid, dim3(256), lds, st>>>(p);
  }
  const int rl = hip_check_launch();
  return rl != SLM_OK || !v ? rl : slm_linear(v, stream);
}
extern "C" SLM_API int slm_latent_attn(const slm_latent_attn_args* a, void* stream) { return la_run(a, nullptr, stream); }
extern "C" SLM_API int slm_latent_attn_values(const slm_latent_attn_args* a, const slm_linear_args* v, void* stream) {
  if (!v || !v->w || !v->y || v->M < 0 || v->N <= 0 || v->N % 16 || v->n_splits != 1 || (v->epilogue != SLM_LIN_STORE && v->epilogue != SLM_LIN_GATE) ||
      (v->epilogue == SLM_LIN_GATE && !v->gate))
    return SLM_ERR_INVALID_ARG;
  if (!aligned16(v->w)) return SLM_ERR_ALIGNMENT;
  const int rc = linear_check(v);   // (whichever way it goes, and in front of the attention)
  if (rc != SLM_OK) return rc;
  return la_run(a, v, stream);
}
