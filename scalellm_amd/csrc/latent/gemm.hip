// gemm.hip -- y = x W^T in bf16 or half precision for many rows (prompts, mixed steps), from row-major x and W, with the GLU as an epilogue.
//
// Four waves, one to a SIMD, hold a quarter of the tile each: 128 x 128 products of 16 x 16 x 32 in 256 accumulators read 0.5 KB
// of LDS per 1024 matrix-pipe cycles and SIMD, where eight waves of 128 x 64 read 0.75 -- and what bounds a large product here is power
// (8192^3: 576 us on zeros, 718 on normal numbers), which operand traffic is part of (with 32 x 32 x 16 products 6 % more).  The
// accumulators are pinned to the second half of the register file by inline asm: left to itself the compiler spreads them over
// both and copies 1000 registers a step.
//
// A step is 64 of k, 128 bytes a row, so that LDS-DMA moves whole lines; 16-byte chunk c of row r lies in slot c ^ (r & 7), which
// the DMA does on its global side.  Each step's products come in two halves of 32 k: the first runs over the LDS reads of the
// second, the second over those of the next step's first.  One barrier a step, between the halves: there this stage has been read
// by all waves and the next one has landed.  x has three stages and its DMA runs half a step apart from that of w: all 16
// instructions of a step at once back up in the address unit, and a wave alone on its SIMD stalls with them (on zeros 14 %
// more).  256 x 256: 160 KB of LDS.
//
// A workgroup goes from tile to tile: the DMA of a tile's last steps brings the first stages of the next one, which so are there when the
// epilogue ends.  That is 5 us of a tile's 97 (256 x 256, K 4096), but power takes most of it back (us, both timed in turn): 3226 x 16896 x 4096
// 358 -> 350, 4096 x 8512 x 2048 119 -> 115, 4096 x 16384 x 4096 395 -> 388, 5692 x 4096 x 14336 492 -> 490, 8192^3 level.  (Where it goes in the loop matters: sources chosen by
// the step cost 3 % of every product; the steps come in parts instead.)
//
// Tiles that do not fill the last round of the chip are cut in K (slices > 1): every slice leaves fp32 sums past the caches, the last one
// to arrive (a counter per tile) adds them up in slice order and stores.  Nobody waits for anybody.
//
// us by the device, vendor product (and the GLU's launch) / this, normal numbers: 5692 x 28672 x 4096 GLU 1069 / 975 (1.37 PFLOP/s),
// 5692 x 4096 x 14336 737 / 490, 5692 x 4096 x 4096 148 / 145, 3226 x 28672 x 4096 GLU 703 / 559, 3226 x 16896 x 4096 441 / 350, 4096 x 16384 x 2048 GLU
// 226 / 206, 4096 x 8512 x 2048 152 / 115, 1000 x 4096 x 14336 131 / 108, 600 x 28672 x 4096 GLU 147 / 132, 300 x 4096 x 14336 72 / 64,
// 207 x 16384 x 2048 GLU 30 / 22.  Behind the vendor product where its tiles fill whole rounds (8192^3 678 / 718, 4096^3 89 / 94), with one row of tiles
// over large weights (129 x 28672 x 4096 GLU 59 / 74), and on short and narrow products (weights out of memory: 197 x 2048 x 2048 11.8 / 13.7, 284 x 3664 x
// 2048 15.3 / 16.0; but 197 x 4096 x 4096 22.2 / 20.3, 197 x 4096 x 14336 56 / 45), which its callers take here for the sake of the host.
#include <type_traits>

#include "latent_common.h"
#include "tile_common.h"

namespace slm {

struct GemmK {
  const char* x;
  const char* w;
  uint16_t* y;
  float* slabs;            // [tiles cut][slices][fragments][256] f32x4
  uint32_t* arrived;       // [tiles cut], zero
  int64_t M, N, K, ldy;
  uint32_t ldx2, ldw2;     // bytes
  int mb, nb, whole, cut, slices, group;   // tiles: `whole` by one workgroup each, `cut` by `slices` each
  float limit, alpha, shift;
};

// T: bf16_tag or f16_tag
template <typename T>
__device__ __forceinline__ void gemm_product(f32x4& c, const u32x4& w, const u32x4& x) {
  if constexpr (std::is_same<T, bf16_tag>::value) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
  else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
}

template <typename T, int BM, int BN, int WS, bool GLU>
__global__ void __launch_bounds__(256, 1) gemm_kernel(const GemmK a) {
  constexpr int XS = 3;                              // stages of x; WS: of w
  constexpr int XB = BM * 128, WB = BN * 128;        // bytes of a stage
  constexpr int MT = BM / 32, NT = BN / 32;          // 16-row / 16-column tiles of a wave
  constexpr int XD = BM / 32, WD = BN / 32, ND = XD + WD;   // DMA instructions of a wave and step (8 rows each)
  constexpr int R = MT + NT, MM = MT * NT;           // LDS reads and products of a half step
  constexpr int LATE = XD + (WS == 3 ? WD : 0);      // DMA under way that the next step does not need
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4, wm = wave & 1, wn = wave >> 1;

  // What a workgroup does one after the other: items blockIdx.x, + gridDim.x, ..  (whole tiles: a multiple of 8 of them)
  struct Item {
    int m0, n0, slice, own, s0, steps;
  };
  const int whole_items = (a.whole + 7) & ~7, all = (int)(a.K >> 6);
  auto item = [&](int v, Item& it) -> bool {
    int t;
    it.slice = 0;
    it.own = -1;
    it.s0 = 0;
    it.steps = all;
    if (v < whole_items) {
      t = xcd_run(v, a.whole);
      if (t < 0) return false;
    } else {
      const int u = xcd_run(v - whole_items, a.cut * a.slices);
      if (u < 0) return false;
      it.own = u / a.slices;
      it.slice = u - it.own * a.slices;
      t = a.whole + it.own;
      const int per = (all + a.slices - 1) / a.slices;
      it.s0 = it.slice * per;
      it.steps = min(per, all - it.s0);   // (the plan leaves no slice empty)
    }
    // `group` row blocks by columns: neighbours in a run share rows of x and of w in their L2
    const int gsz = a.group * a.nb, gi = t / gsz, in = t - gi * gsz;
    const int rows_in = min(a.group, a.mb - gi * a.group);
    it.m0 = (gi * a.group + in % rows_in) * BM;
    it.n0 = in / rows_in * (GLU ? BN / 2 : BN);
    return true;
  };
  Item cur, nxt;
  if (!item(blockIdx.x, cur)) return;
  const int half = (int)(a.N / 2);

  // instruction i of this wave brings 8 rows of 128 bytes (rows past the end: the last one, not stored)
  uint32_t off[ND];
  auto offset = [&](int i, const Item& it, int l) {
    const int r = (i < XD ? (wave * XD + i) : (wave * WD + i - XD)) * 8 + (l >> 3);
    const uint32_t k = (uint32_t)(((l & 7) ^ (i < XD ? r & 7 : (r & 3) | ((r >> 1) & 4))) << 4);
    if (i < XD) {
      off[i] = (uint32_t)min(it.m0 + r, (int)a.M - 1) * a.ldx2 + k;
    } else if constexpr (GLU) {   // of a wave's BN / 2 columns half are of the gate, then the same of the up half
      const int q = r / (BN / 2), c = r % (BN / 2);
      const int n = min(it.n0 + q * (BN / 4) + c % (BN / 4), half - 1) + (c >= BN / 4 ? half : 0);
      off[i] = (uint32_t)n * a.ldw2 + k;
    } else {
      off[i] = (uint32_t)min(it.n0 + r, (int)a.N - 1) * a.ldw2 + k;
    }
  };
#pragma unroll
  for (int i = 0; i < ND; ++i) offset(i, cur, lane);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const uint32_t xdst = lds0 + wave * (XD * 1024), wdst = lds0 + XS * XB + wave * (WD * 1024);
  auto dma = [&](int i, uint32_t kb, uint32_t at) {   // kb: byte offset in the rows, at: of the stage
    const uint32_t dst = (i < XD ? xdst + i * 1024 : wdst + (i - XD) * 1024) + at;
    const char* base = (i < XD ? a.x : a.w) + kb;
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" : : "v"(off[i]), "s"(dst), "s"(base) : "memory", "m0");
  };
  // (what is made of it is made where it stands: kept through the products it spills)
  auto here = [](int l) {
    asm volatile("" : "+v"(l));
    return l;
  };

  // Columns of a pair of tiles go to them by fours, so that a lane ends with eight neighbours.  Chunk c of a row of w lies in slot
  // c ^ (row % 4 + 4 (row / 8 % 2)): eight lanes read eight slots of either matrix.
  const int xrow = wm * (BM / 2) + r16, wrow = wn * (BN / 2) + 8 * (r16 >> 2) + (r16 & 3);
  u32x4 fx[2][MT], fw[2][NT];                   // operands of the two halves
  auto read = [&](int j, int h, uint32_t xa, uint32_t wa) {   // j-th of R
    const int slot = ((h * 4 + g) ^ (r16 & 7)) << 4;   // (of w: row % 4 = r16 % 4, row / 8 % 2 = r16 / 4 % 2: the same)
    if (j < MT) fx[h][j] = *reinterpret_cast<const u32x4*>(lds + xa + (xrow + 16 * j) * 128 + slot);
    else fw[h][j - MT] = *reinterpret_cast<const u32x4*>(lds + XS * XB + wa + (wrow + 32 * ((j - MT) >> 1) + 4 * ((j - MT) & 1)) * 128 + slot);
  };
  // (rows there and back: a product takes one operand of the one before it, which is 0.5 % of a large product's time)
  auto turn = [](int q) { return q / MT % 2 ? MT - 1 - q % MT : q % MT; };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  int v = blockIdx.x;
  bool more = item(v + (int)gridDim.x, nxt);   // (then every item has more than WS steps)
  // byte offsets in the rows of the step that x and w are loaded for; steps past the end of the last item load its last one again
  uint32_t kx = (uint32_t)cur.s0 << 7, kw = kx, last = kx + ((uint32_t)(cur.steps - 1) << 7);
#pragma unroll
  for (int p = 0; p < WS; ++p) {
#pragma unroll
    for (int i = 0; i < ND; ++i)
      if (i >= XD || p < 2) dma(i, i < XD ? kx : kw, p * (i < XD ? XB : WB));
    if (p < 2) kx = min(kx + 128, last);
    kw = min(kw + 128, last);
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(ND + (WS - 2) * WD) : "memory");   // the first stages are there
#pragma unroll
  for (int j = 0; j < R; ++j) {
    read(j, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
  uint32_t xa = 0, wa = 0, xl = 2 * XB;   // this step's stages, and the one that x is loaded to
  for (;;) {
    // The last steps' DMA is the next item's first: it runs under the epilogue.  So the steps come in parts, w's sources change WS of them before
    // the end, x's two.
    int left = more ? cur.steps - WS : cur.steps, part = more ? WS : 1;
    for (;;) {
      do {
        const uint32_t xn = xa == (XS - 1) * XB ? 0 : xa + XB, wnext = wa == (WS - 1) * WB ? 0 : wa + WB;
#pragma unroll
        for (int b = 0; b < R; ++b) {
#pragma unroll
          for (int i = b * XD / R; i < (b + 1) * XD / R; ++i) dma(i, kx, xl);
          read(b, 1, xa, wa);
#pragma unroll
          for (int q = b * MM / R; q < (b + 1) * MM / R; ++q) gemm_product<T>(acc[q / MT][turn(q)], fw[0][q / MT], fx[0][turn(q)]);
          __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(LATE) : "memory");
        kx = min(kx + 128, last);
#pragma unroll
        for (int b = 0; b < R; ++b) {
          if (b < WD) dma(XD + b, kw, wa);
          read(b, 0, xn, wnext);
#pragma unroll
          for (int q = b * MM / R; q < (b + 1) * MM / R; ++q) gemm_product<T>(acc[q / MT][turn(q)], fw[1][q / MT], fx[1][turn(q)]);
          __builtin_amdgcn_sched_barrier(0);
        }
        kw = min(kw + 128, last);
        xl = xa;
        xa = xn;
        wa = wnext;
      } while (--left > 0);
      if (part == 1) break;
      const int l = here(lane);
      if (part == WS) {
        last = (uint32_t)(nxt.s0 + nxt.steps - 1) << 7;
        kw = (uint32_t)nxt.s0 << 7;
#pragma unroll
        for (int i = XD; i < ND; ++i) offset(i, nxt, l);
      }
      if (part == 2) {
        kx = (uint32_t)nxt.s0 << 7;
#pragma unroll
        for (int i = 0; i < XD; ++i) offset(i, nxt, l);
      }
      left = part == 2 ? 2 : 1;
      --part;
    }
    if (!more) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    tile_products_settle(acc);
    if (cur.own >= 0 && !tile_add_slices(acc, a.slabs + (int64_t)cur.own * a.slices * (MM * 1024), a.arrived + cur.own, cur.slice, a.slices, lds)) return;

    // lane: columns 8 g .. + 7 of a pair of tiles, row r16
    const int el = here(lane), e16 = el & 15, eg = el >> 4;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int row = cur.m0 + wm * (BM / 2) + 16 * m + e16;
      uint16_t* y = a.y + row * a.ldy;
#pragma unroll
      for (int n = 0; n < (GLU ? NT / 2 : NT); n += 2) {
        const int col = cur.n0 + wn * (GLU ? BN / 4 : BN / 2) + 16 * n + 8 * eg;
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          o[j] = acc[n + (j >> 2)][m][j & 3];
          if constexpr (GLU) o[j] = clamped_glu_f32(o[j], acc[n + (j >> 2) + NT / 2][m][j & 3], a.limit, a.alpha, a.shift);
        }
        if (row < a.M && col < (GLU ? half : (int)a.N))
          *reinterpret_cast<u32x4*>(y + col) = u32x4{pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]), pack2<T>(o[4], o[5]), pack2<T>(o[6], o[7])};
      }
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+a"(acc[n][m]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!more) return;
    cur = nxt;
    v += gridDim.x;
    more = item(v + (int)gridDim.x, nxt);
  }
}

// Tiles, and what they take: us of a step of 64 k alone on the chip and with every CU busy (power), and of a tile beside its steps.
// Fitted to 900 timings of 90 products of 65 - 5700 rows, with a workgroup for each tile.  Since workgroups go from tile to tile the tile taken is 0.8 %
// behind the best one on average (154 products of 161 - 8400 rows); constants fitted to these were 0.9 % behind.
struct GemmTile {
  int bm, bn;
  float step, busy, rest;
};
constexpr GemmTile GEMM_TILES[] = {{256, 256, 0.914f, 1.386f, 8.6f}, {256, 128, 0.521f, 0.778f, 5.0f}, {128, 128, 0.311f, 0.488f, 3.4f}, {128, 256, 0.542f, 0.800f, 5.3f},
                                   {256, 192, 0.725f, 1.037f, 6.6f}, {192, 256, 0.743f, 1.071f, 6.6f}, {160, 256, 0.647f, 0.909f, 6.1f}};
constexpr int GEMM_N_TILES = sizeof(GEMM_TILES) / sizeof(GEMM_TILES[0]), GEMM_128_128 = 2, GEMM_256_192 = 4;   // (the last has no GLU)
constexpr int GEMM_CUS = 256;
static_assert(SLM_GEMM_COUNTERS >= GEMM_CUS, "a counter for each tile of a round");
constexpr float GEMM_CUT = 6.f, GEMM_SLABS = 3.5e6f;   // us of cutting tiles, bytes of their slabs that take one more

struct GemmPlan {
  int tile, mb, nb, whole, cut, slices;
  float us;
  size_t bytes;   // workspace: counters, then slabs
};

static GemmPlan gemm_plan_of(const slm_linear_args& a, int tile, int slices) {
  const GemmTile& t = GEMM_TILES[tile];
  const bool glu = a.epilogue == SLM_LIN_GLU;
  const int64_t cols = glu ? a.N / 2 : a.N, wide = glu ? t.bn / 2 : t.bn;
  GemmPlan p{};
  p.tile = tile;
  p.mb = (int)((a.M + t.bm - 1) / t.bm);
  p.nb = (int)((cols + wide - 1) / wide);
  const int tiles = p.mb * p.nb, left = tiles % GEMM_CUS, steps = (int)(a.K >> 6);
  // the last round's tiles are cut by as many as leave it one round, at least four steps each
  int s = slices;
  if (s <= 0) {
    const int most = t.bm * t.bn == 128 * 128 ? 8 : 4;
    s = left ? GEMM_CUS / left : 1;
    s = s < most ? s : most;
    while (s > 1 && steps / s < 4) --s;
  }
  if (!left) s = 1;
  s = s < steps ? s : steps;
  while (s > 1 && (steps + s - 1) / s * (s - 1) >= steps) --s;   // no slice is empty
  p.slices = s;
  p.cut = s > 1 ? left : 0;
  p.whole = tiles - p.cut;
  const size_t slabs = (size_t)p.cut * s * t.bm * t.bn * 4;
  p.bytes = p.cut ? 1024 + slabs : 0;
  auto round = [&](int wgs, int n) { return t.rest + n * (t.step + (t.busy - t.step) * (float)wgs / GEMM_CUS); };
  p.us = (float)(tiles / GEMM_CUS) * round(GEMM_CUS, steps);
  if (p.cut) p.us += round(left * s, (steps + s - 1) / s) + GEMM_CUT + (float)slabs / GEMM_SLABS;
  else if (left) p.us += round(left, steps);
  return p;
}
// Slices of a product whose tiles of 128 x 128 leave the chip's one round partly empty.  Its weights come from memory, for which a step is 0.42 to 0.52 us
// whatever the tile does (the constants above are of products that wait for their operands less); joining s slices is 2.4 + 1.15 s: the last one
// reads s tiles of 64 KB one after the other.  us, 197 rows, slices 1 / 2 / 3 / 4 / 6 / 8: 2048 x 2048 18.7 / 15.2 / 13.9 / 13.7 / 14.9 / 16.5, 2048 x 8192 60.0 /
// 39.0 / 30.2 / 26.5 / 23.7 / 25.2, 4096 x 14336 (1 to 4) 114 / 68 / 53 / 45, 3664 x 2048 18.9 / 15.7 / 14.9 / 15.2, 6752 x 4096 35.3 / 27.2; 512 rows, 4096 x
// 4096 37.4 / 27.6; 4096 x 512 6.9 / 9.9.
static int gemm_few_tiles(int tiles, int steps) {
  int best = 1;
  float least = 0.f;
  for (int s = 1; s <= 8 && (s == 1 || (tiles * s <= GEMM_CUS && steps / s >= 4)); ++s) {
    const float us = (float)((steps + s - 1) / s) * (0.42f + 0.1f * (float)(tiles * s) / GEMM_CUS) + (s > 1 ? 2.4f + 1.15f * (float)s : 0.f);
    if (s == 1 || us < least) best = s, least = us;
  }
  return best;
}
// tile -1: the one that takes least; slices 0: as many as pay, 1: none
static GemmPlan gemm_plan(const slm_linear_args& a, int tile, int slices) {
  if (tile >= 0) return gemm_plan_of(a, tile, slices);
  GemmPlan best{};
  for (int t = 0; t < GEMM_N_TILES; ++t) {
    if (t == GEMM_256_192 && a.epilogue == SLM_LIN_GLU) continue;
    for (int s = slices > 0 ? slices : 0; s <= (slices > 0 ? slices : 1); ++s) {
      const GemmPlan p = gemm_plan_of(a, t, s);
      if (best.us == 0.f || p.us < best.us) best = p;
    }
  }
  if (slices <= 0 && best.tile == GEMM_128_128 && best.mb * best.nb < GEMM_CUS)
    best = gemm_plan_of(a, GEMM_128_128, gemm_few_tiles(best.mb * best.nb, (int)(a.K >> 6)));
  return best;
}

template <typename T, int BM, int BN, int WS, bool GLU>
static int gemm_launch(const GemmK& k, hipStream_t st) {
  constexpr int bytes = (3 * BM + WS * BN) * 128;
  auto fn = gemm_kernel<T, BM, BN, WS, GLU>;
  static bool asked[64] = {};
  tile_allow_lds(fn, bytes, asked);
  // A workgroup goes from one to the next only where the shortest, the last slice, is long enough to load the next one's first stages, and a slice
  // is the last of a workgroup's items (the plan's slices fill one round at most, behind whole ones).
  const int parts = (k.cut * k.slices + 7) / 8 * 8, items = (k.whole + 7) / 8 * 8 + parts, all = (int)(k.K >> 6);
  const int shortest = k.cut ? all - (all + k.slices - 1) / k.slices * (k.slices - 1) : all;
  const unsigned wgs = (unsigned)(shortest > WS && items > GEMM_CUS && parts <= GEMM_CUS ? GEMM_CUS : items);
  fn<<<dim3(wgs), dim3(256), bytes, st>>>(k);
  return hip_check_launch();
}
template <typename T, bool GLU>
static int gemm_tile(const GemmPlan& p, const GemmK& k, hipStream_t st) {
  switch (p.tile) {
    case 0: return gemm_launch<T, 256, 256, 2, GLU>(k, st);
    case 1: return gemm_launch<T, 256, 128, 3, GLU>(k, st);
    case 2: return gemm_launch<T, 128, 128, 3, GLU>(k, st);
    case 3: return gemm_launch<T, 128, 256, 3, GLU>(k, st);
    case 5: return gemm_launch<T, 192, 256, 2, GLU>(k, st);
    case 6: return gemm_launch<T, 160, 256, 3, GLU>(k, st);
    default:
      if constexpr (!GLU) return gemm_launch<T, 256, 192, 2, GLU>(k, st);
      return SLM_ERR_UNSUPPORTED;
  }
}

// What the kernel takes: 16-byte rows, byte offsets of 32 bits
static int gemm_check(const slm_linear_args* a, int tile, int slices, int dtype) {
  if (!a || !a->x || !a->w || !a->y || a->M < 0 || a->N <= 0 || a->K <= 0 || a->K % 64 || a->N % 16 || a->batch != 1 || a->n_splits != 1 ||
      a->ldx < a->K || a->ldw < a->K || (a->epilogue != SLM_LIN_STORE && a->epilogue != SLM_LIN_GLU) || tile < -1 || tile >= GEMM_N_TILES || slices < 0)
    return SLM_ERR_INVALID_ARG;
  const bool glu = a->epilogue == SLM_LIN_GLU;
  if (a->ldy < (glu ? a->N / 2 : a->N)) return SLM_ERR_INVALID_ARG;
  if (a->dtype != dtype || (glu && (a->N % 32 || tile == GEMM_256_192))) return SLM_ERR_UNSUPPORTED;
  if (a->ldx % 8 || a->ldw % 8 || a->ldy % 8 || !aligned16(a->x) || !aligned16(a->w) || !aligned16(a->y)) return SLM_ERR_ALIGNMENT;
  const int64_t most = 1ll << 31;
  if (a->M > most / 2 / a->ldx || a->N > most / 2 / a->ldw || a->M > (1 << 24) || a->N > (1 << 24)) return SLM_ERR_UNSUPPORTED;
  return SLM_OK;
}

}  // namespace slm

using namespace slm;

extern "C" SLM_API size_t slm_gemm_workspace_bytes(const slm_linear_args* a, int32_t tile, int32_t slices) {
  return gemm_check(a, tile, slices, a && a->dtype == SLM_F16 ? SLM_F16 : SLM_BF16) == SLM_OK && a->M ? gemm_plan(*a, tile, slices).bytes : 0;
}

template <typename T>
static int gemm_run(const slm_linear_args* a, void* workspace, size_t workspace_bytes, uint32_t* counters, int32_t tile, int32_t slices, void* stream) {
  const int rc = gemm_check(a, tile, slices, std::is_same<T, bf16_tag>::value ? SLM_BF16 : SLM_F16);
  if (rc != SLM_OK || a->M == 0) return rc;
  GemmPlan p = gemm_plan(*a, tile, slices);
  if (p.cut && (!workspace || workspace_bytes < p.bytes)) p = gemm_plan(*a, tile, 1);   // (no scratch: no cut)
  if (p.cut && !aligned16(workspace)) return SLM_ERR_ALIGNMENT;
  GemmK k{};
  k.x = (const char*)a->x; k.w = (const char*)a->w; k.y = (uint16_t*)a->y;
  k.M = a->M; k.N = a->N; k.K = a->K; k.ldy = a->ldy; k.ldx2 = (uint32_t)(a->ldx * 2); k.ldw2 = (uint32_t)(a->ldw * 2);
  k.limit = a->limit; k.alpha = a->glu_alpha; k.shift = a->glu_shift;
  k.mb = p.mb; k.nb = p.nb; k.whole = p.whole; k.cut = p.cut; k.slices = p.slices; k.group = 8;
  k.arrived = counters ? counters : (uint32_t*)workspace; k.slabs = (float*)((char*)workspace + 1024);
  hipStream_t st = (hipStream_t)stream;
  hip_clear_error();
  if (p.cut && !counters) tile_clear_kernel<<<dim3(1), dim3(256), 0, st>>>(k.arrived, p.cut);
  return a->epilogue == SLM_LIN_GLU ? gemm_tile<T, true>(p, k, st) : gemm_tile<T, false>(p, k, st);
}
extern "C" SLM_API int slm_gemm(const slm_linear_args* a, void* workspace, size_t workspace_bytes, int32_t tile, int32_t slices, void* stream) {
  return gemm_run<bf16_tag>(a, workspace, workspace_bytes, nullptr, tile, slices, stream);
}
extern "C" SLM_API int slm_gemm_half(const slm_linear_args* a, void* workspace, size_t workspace_bytes, int32_t tile, int32_t slices, void* stream) {
  return gemm_run<f16_tag>(a, workspace, workspace_bytes, nullptr, tile, slices, stream);
}
extern "C" SLM_API int slm_gemm_counted(const slm_linear_args* a, void* workspace, size_t workspace_bytes, uint32_t* counters, int32_t tile, int32_t slices, void* stream) {
  if (!a || !counters) return SLM_ERR_INVALID_ARG;
  return a->dtype == SLM_F16 ? gemm_run<f16_tag>(a, workspace, workspace_bytes, counters, tile, slices, stream)
                             : gemm_run<bf16_tag>(a, workspace, workspace_bytes, counters, tile, slices, stream);
}
