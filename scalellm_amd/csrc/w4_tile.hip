// w4_tile.hip -- int4-weight x bf16-activation GEMM for many rows (prompts, mixed steps), four waves a tile.
//
// Same operator as w4.hip (replaces marlin::gptq_gemm, reference gptq_gemm.cu:585-710), same packed layout (w4.hip header), same
// bit-faithful dequant (W4Dq<bf16_tag>, marlin/numeric_conversion.h:19-62).
//
// Four waves, one to a SIMD, take all rows and a quarter of the columns each: 256 x 64 products of 16 x 16 x 32 at most, in accumulators that
// inline asm pins to the second half of the register file.  A step is 64 of k.  Activations come by LDS-DMA, 128 bytes a row, and are
// read by every wave; 16-byte chunk c of row r lies in slot c ^ (r & 7).  No two waves share a column, so weights never are in LDS as 16-bit rows:
// their words come by LDS-DMA as well (8 KB a step instead of the 32 a 16-bit weight takes; loads into registers would have waits of the
// compiler's, which knows nothing of the DMA beside them), and a lane makes operands of the ones it needs itself, half a step ahead of their products:
// 1.2 vector instructions beside each product, which holds the matrix pipe for four.  (As rows that two waves share, written to LDS
// and read back, the same tile took 97 us on an idle chip and 463 on a full one where this takes 88 and 448.)
//
// Step s: first half, products of k 0 - 31 over the LDS reads of k 32 - 63; the words of step s + RS are fetched; barrier: this stage
// has been read by all, step s + 1 is there; second half, products of k 32 - 63 over the reads of step s + 1, and the activations of
// step s + XS are fetched into the freed stage.
//
// Tiles that do not fill the chip once are cut in K: every slice leaves fp32 sums past the caches, the last one to arrive adds them up in slice
// order and stores.  Nobody waits for anybody.  All tiles are cut or none: a column's sum then has one order wherever it lies, which the SiLU of
// a paired weight owes to that of the plain one (the last of several rounds alone would gain 2 % on some sizes).
#include <type_traits>

#include "tile_common.h"
#include "w4_common.h"

namespace slm {

struct W4TileK {
  const char* x;
  const uint32_t* wq;
  const uint32_t* sz;
  const uint16_t* bias;
  uint16_t* c;
  float* slabs;            // [tiles][slices][fragments][256] f32x4, where there are slices
  uint32_t* arrived;       // [tiles], zero
  int64_t M, N, K, ldc;
  uint32_t lda2;           // bytes
  int cpg_shift;           // log2(steps of a scale group)
  int mb, nb, tiles, slices, group;
  int silu, wide;          // wide: 16-byte stores
};

__device__ __forceinline__ void tile_product(f32x4& c, const u32x4& w, const u32x4& x) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
}

// W4Dq<bf16_tag>::word() in eight pieces of one to three vector instructions
struct W4Pieces {
  W4Dq<bf16_tag> dq{0u};
  W4Dq<bf16_tag>::Nib n;
  f32x2 a, b;
  uint32_t out[4];
  __device__ __forceinline__ void run(int piece, uint32_t w) {
    switch (piece) {
      case 0: n = dq.split(w); break;
      case 1: a = __builtin_amdgcn_cvt_pk_f32_fp8((int)n.lo, false); b = __builtin_amdgcn_cvt_pk_f32_fp8((int)n.lo, true); break;
      case 2: a = __builtin_elementwise_fma(a, dq.s512, dq.c2); b = __builtin_elementwise_fma(b, dq.s512, dq.c2); break;
      case 3: out[0] = pack2<bf16_tag>(a[0], b[0]); out[2] = pack2<bf16_tag>(a[1], b[1]); break;
      case 4: a = __builtin_amdgcn_cvt_pk_f32_fp8((int)n.hi, false); break;
      case 5: b = __builtin_amdgcn_cvt_pk_f32_fp8((int)n.hi, true); a = __builtin_elementwise_fma(a, dq.s512, dq.c2); break;
      case 6: b = __builtin_elementwise_fma(b, dq.s512, dq.c2); break;
      default: out[1] = pack2<bf16_tag>(a[0], b[0]); out[3] = pack2<bf16_tag>(a[1], b[1]);
    }
  }
};

// f(0) .. f(N - 1), each with its index as a constant (the loops over blocks are past what the compiler unrolls)
template <int N, int I = 0, typename F>
__device__ __forceinline__ void in_turn(const F& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    in_turn<N, I + 1>(f);
  }
}

// Half a step's work on words lies so in its blocks: unit u of 2 nt (column tile u / 2) in the last block b with b * 2 nt / mt == u, and the DMA that
// overwrites a stage in the last tw + ngc blocks, in front of their units: the first scales, words, second scales.  In the first half step the
// stage that it overwrites is the one whose words (and second scales) for k 32 .. 63 are still on their way to registers; the DMA waits for
// those it overwrites, and the order sees to it that their first unit, which waits for them anyway, is not in a later block.
constexpr int w4_tile_unit_block(int u, int mt, int nt) {
  int b = 0;
  while ((b + 1) * 2 * nt / mt <= u) ++b;
  return b;
}
constexpr bool w4_tile_words_in_order(int mt, int nt, int tw, int ngc) {
  const int first = mt - tw - ngc;   // block of the first scales
  for (int n = 0; n < nt; ++n) {
    const int taken = w4_tile_unit_block(2 * n, mt, nt);
    if (first + 1 + n / 2 < taken || (ngc == 2 && first + 1 + tw < taken)) return false;
  }
  return true;
}

constexpr int W4_TILE_LDS(int bm, int bn, int ngc) { return 3 * bm * 128 + 4 * 4 * (bn / 128 * 1024 + ngc * 256); }

// NGC: scale groups of a step (2 of 32 rows; else 1)
template <int BM, int BN, int NGC>
__global__ void __launch_bounds__(256, 1) w4_tile_kernel(const W4TileK a) {
  constexpr int XS = 3, RS = 4;                      // stages of activations, of words
  constexpr int TW = BN / 128;                       // packed 32-column tiles of a wave
  constexpr int XB = BM * 128;                       // bytes of a stage
  constexpr int OWN = TW * 1024 + NGC * 256, RB = 4 * OWN;   // of words and scales: a wave's, all
  constexpr int R0 = XS * XB;
  constexpr int MT = BM / 16, NT = 2 * TW;           // 16-row / 16-column tiles of a wave
  constexpr int XD = BM / 32, NR = TW + NGC;         // DMA instructions of a wave and step: activations; words and scales
  constexpr int MM = MT * NT;                        // products of a half step, in MT blocks with an LDS read each
  constexpr int U = 2 * NT;                          // half words that become operands in a half step
  constexpr int LATE = 2 * NR + XD;                  // DMA under way that the next step does not need
  static_assert(NT < MT && NR <= MT && XD <= MT && U <= MT, "blocks");
  static_assert(w4_tile_words_in_order(MT, NT, TW, NGC), "a stage's words are taken before they are overwritten");
  static_assert(R0 + RS * RB == W4_TILE_LDS(BM, BN, NGC) && R0 + RS * RB <= 160 * 1024, "LDS");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;

  const int item = xcd_run(blockIdx.x, a.tiles * a.slices);
  if (item < 0) return;
  const int t = item / a.slices, slice = item - t * a.slices;
  // `group` row blocks by columns: neighbours in a run share rows of x and of w in their L2
  const int gsz = a.group * a.nb, gi = t / gsz, in = t - gi * gsz;
  const int rows_in = min(a.group, a.mb - gi * a.group);
  const int mb = gi * a.group + in % rows_in, nb = in / rows_in;
  const int64_t m0 = (int64_t)mb * BM, n0 = (int64_t)nb * BN;
  const int n_tiles = (int)(a.N >> 5);

  // DMA: an instruction brings 8 rows of 128 bytes of x (rows past the end: the last one, not stored), a packed tile, or the scales
  uint32_t xoff[XD], woff[TW], zoff;
#pragma unroll
  for (int i = 0; i < XD; ++i) {
    const int r = (wave * XD + i) * 8 + (lane >> 3);
    xoff[i] = (uint32_t)min(m0 + r, a.M - 1) * a.lda2 + (uint32_t)(((lane & 7) ^ (r & 7)) << 4);
  }
  const int tile0 = (int)(n0 >> 5) + wave * TW;
#pragma unroll
  for (int i = 0; i < TW; ++i) woff[i] = (uint32_t)min(tile0 + i, n_tiles - 1) * 1024 + lane * 16;
  zoff = (uint32_t)(min(tile0 + (TW == 2 ? lane >> 5 : 0), n_tiles - 1) * 32 + (lane & 31)) * 4;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const uint32_t xdst = lds0 + wave * (XD * 1024), rdst = lds0 + R0 + wave * OWN;
  const int all = (int)(a.K >> 6), per = (all + a.slices - 1) / a.slices;
  const int s0 = slice * per, steps = min(per, all - s0);   // (the plan leaves no slice empty)
  auto at_step = [&](int s) { return s0 + min(s, steps - 1); };   // (steps past the end load the last one again)
  auto dma_x = [&](int i, int s, uint32_t at) {
    const char* base = a.x + ((int64_t)at_step(s) << 7);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" : : "v"(xoff[i]), "s"(xdst + at + i * 1024), "s"(base) : "memory", "m0");
  };
  auto dma_w = [&](int i, int s, uint32_t at) {   // i-th of NR: scales, words, second scales
    const int c = at_step(s), w = i - 1;
    if (w >= 0 && w < TW) {
      const char* base = reinterpret_cast<const char*>(a.wq) + (int64_t)c * n_tiles * 1024;
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2" : : "v"(woff[w >= 0 && w < TW ? w : 0]), "s"(rdst + at + w * 1024), "s"(base) : "memory", "m0");
    } else {
      const int h = i > TW;
      const int64_t grp = NGC == 2 ? 2 * c + h : c >> a.cpg_shift;
      const char* base = reinterpret_cast<const char*>(a.sz) + grp * a.N * 4;
      asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, %2" : : "v"(zoff), "s"(rdst + at + TW * 1024 + h * 256), "s"(base) : "memory", "m0");
    }
  };

  u32x4 fx[2][MT], fw[2][NT];                   // operands of the two halves
  const uint32_t xrow = (uint32_t)r16 * 128;
  auto read = [&](int j, int h, uint32_t xa) {   // j-th of MT
    fx[h][j] = *reinterpret_cast<const u32x4*>(lds + xa + xrow + 2048 * j + (((h * 4 + g) ^ (r16 & 7)) << 4));
  };
  // Columns of a pair of tiles go to them by fours, so that a lane ends with eight neighbours: lane r16 of tile n has this one of packed tile n / 2.
  // Its eight weights of k 32 h + 8 g are word 2 h + g / 2 of the packed tile's lane `column` + 32 (g % 2).
  const int column = 8 * (r16 >> 2) + (r16 & 3);   // (+ 4 for odd n)
  uint32_t words[2][NT], scales[NGC][NT];
  const uint32_t wfrom = R0 + wave * OWN + (column + 32 * (g & 1)) * 16 + (g >> 1) * 4, zfrom = R0 + wave * OWN + TW * 1024 + column * 4;
  auto fetch = [&](int n, int h, uint32_t at) {   // (this wave's own DMA: no barrier)
    words[h][n] = *reinterpret_cast<const uint32_t*>(lds + wfrom + at + (n >> 1) * 1024 + (n & 1) * 64 + h * 8);
    if (h == 0 || NGC == 2) scales[NGC == 2 ? h : 0][n] = *reinterpret_cast<const uint32_t*>(lds + zfrom + at + (NGC == 2 ? h * 256 : 0) + (n >> 1) * 128 + (n & 1) * 16);
  };
  auto taken = [&](uint32_t& v) { asm volatile("" : : "v"(v)); };
  W4Pieces dq[NT];
  auto piece = [&](int u, int q, int h) {   // q-th of four of unit u: words of half h
    const int n = u >> 1;
    if (!(u & 1) && q == 0 && (h == 0 || NGC == 2)) dq[n].dq = W4Dq<bf16_tag>(scales[NGC == 2 ? h : 0][n]);
    dq[n].run(4 * (u & 1) + q, words[h][n]);
    if ((u & 1) && q == 3) fw[h][n] = u32x4{dq[n].out[0], dq[n].out[1], dq[n].out[2], dq[n].out[3]};
  };

  f32x4 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  // a block of products of half h, and between them the operands of the next half
  auto block = [&](auto block_index, auto half) {
    constexpr int b = block_index, h = half, q0 = b * NT, u = b * U / MT;
    in_turn<NT>([&](auto q) {
      constexpr int n = (q0 + q) / MT, m = (q0 + q) % MT;
      tile_product(acc[n][m], fw[h][n], fx[h][m]);
      if constexpr ((b + 1) * U / MT > u) {
#pragma unroll
        for (int k = 0; k < 4 / NT; ++k) piece(u, q * (4 / NT) + k, 1 - h);
        __builtin_amdgcn_sched_barrier(0);
      }
    });
  };
  constexpr std::integral_constant<int, 0> FIRST{};
  constexpr std::integral_constant<int, 1> SECOND{};

  // (in the order of the loop: x(1), words(3), x(2))
#pragma unroll
  for (int p = 0; p < RS - 1; ++p)
#pragma unroll
    for (int i = 0; i < NR; ++i) dma_w(i, p, p * RB);
#pragma unroll
  for (int p = 0; p < XS; ++p) {
    if (p == XS - 1)
#pragma unroll
      for (int i = 0; i < NR; ++i) dma_w(i, RS - 1, (RS - 1) * RB);
#pragma unroll
    for (int i = 0; i < XD; ++i) dma_x(i, p, p * XB);
  }
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(XS * XD + NR) : "memory");
#pragma unroll
  for (int n = 0; n < NT; ++n) fetch(n, 0, 0);
#pragma unroll
  for (int k = 0; k < 4 * U; ++k) piece(k >> 2, k & 3, 0);
#pragma unroll
  for (int n = 0; n < NT; ++n) fetch(n, 1, 0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((XS - 1) * XD + NR) : "memory");   // the first stage is there
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    read(j, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
  uint32_t xa = 0, ra = 0;   // this step's stages
  // 24 bytes behind a multiple of 32, by which instructions are fetched: 192 x 256 tiles, groups of 32, take 80.5 us for 2183 x 4096 x 4096 from there, 82.3 from 0, 8 and 16
  asm volatile(".p2align 5\n\t.rept 6\n\ts_nop 0\n\t.endr");
  int s = 0;   // (a loop of no steps would have the accumulators set up once more)
  do {
    const uint32_t xn = xa == (XS - 1) * XB ? 0 : xa + XB, rn = ra == (RS - 1) * RB ? 0 : ra + RB;
    in_turn<MT>([&](auto b) {
      if constexpr (b >= MT - NR) {
        constexpr int i = b - (MT - NR);
        // (what is fetched from there is waited for here at the latest)
        if constexpr (i >= 1 && i <= TW) taken(words[1][2 * i - 2]), taken(words[1][2 * i - 1]);
        if constexpr (i > TW) in_turn<NT>([&](auto n) { taken(scales[NGC - 1][n]); });
        dma_w(i, s + RS, ra);
      }
      read(b, 1, xa);
      if constexpr (b >= 1 && b <= NT) fetch(b - 1, 0, rn);
      block(b, FIRST);
      __builtin_amdgcn_sched_barrier(0);
    });
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(LATE) : "memory");
    in_turn<MT>([&](auto b) {
      if constexpr (b < XD) dma_x(b, s + XS, xa);
      read(b, 0, xn);
      if constexpr (b >= MT - NT) fetch(b - (MT - NT), 1, rn);
      block(b, SECOND);
      __builtin_amdgcn_sched_barrier(0);
    });
    xa = xn;
    ra = rn;
  } while (++s < steps);
  tile_settle(acc);
  if (a.slices > 1 && !tile_add_slices(acc, a.slabs + (int64_t)t * a.slices * (MM * 1024), a.arrived + t, slice, a.slices, lds)) return;

  // Out through LDS, 64 (32) rows at a time, and from there in whole lines.  A wave has its own columns' rows to itself, so that their order alone is enough;
  // of one packed tile a wave a pair's gate is in one wave, its up in the next, and they take half of the rows each.  Rows are read four at a
  // time: one after the other, and with a bias added where there is none, 2183 x 4096 x 28672 with the SiLU took 430 us, 422 now, 2183 x 4096 x 4096 77
  // and 75.4.  (Most of what is left, 6 us a tile, is the stores of all CUs at the same time.)
  // (The code for these rows is there once, apart from the accumulators: written out per accumulator it was 10000 instructions, and 13 us more.)
  constexpr int CW = BN / 4, LR = CW * 4 + 16;       // columns of a wave, bytes of a row of them
  constexpr int OR = BM % 64 ? 32 : 64;              // rows at a time
  static_assert(4 * OR * LR <= R0 + RS * RB, "LDS of the rows");
  char* const mine = lds + wave * (OR * LR) + r16 * LR + g * 32;
  auto out = [&](auto with_silu, auto with_bias) __attribute__((always_inline)) {
    constexpr bool SILU = decltype(with_silu)::value, BIAS = decltype(with_bias)::value, PAIRS = TW == 1 && SILU;
    constexpr int PER_ROW = SILU ? 4 : CW / 8, BY = 64 / PER_ROW;   // lanes of a row, eight columns each; rows at a time
    constexpr int TURNS = (PAIRS ? OR / 2 : OR) / BY, AT_ONCE = TURNS < 4 ? TURNS : 4;
    const int from = PAIRS ? wave & 2 : wave, lcol = lane % PER_ROW * 8, row0 = lane / PER_ROW + (PAIRS ? (wave & 1) * (OR / 2) : 0);
    const int64_t col = n0 + from * CW + lcol;
    const char* const gate = lds + from * (OR * LR) + lcol * 4 + row0 * LR;
    const char* const up = gate + (TW == 2 ? 128 : OR * LR);
    const bool inside = col < a.N;
    float bias[2][8];
    if constexpr (BIAS) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        bias[0][j] = inside ? lo_f32<bf16_tag>((uint32_t)a.bias[col + j]) : 0.f;
        bias[1][j] = inside && SILU ? lo_f32<bf16_tag>((uint32_t)a.bias[col + 32 + j]) : 0.f;
      }
    }
    uint16_t* const c = a.c + (SILU ? (col >> 6) * 32 + lcol : col);
    __syncthreads();
#pragma unroll 1
    for (int q = 0; q < BM / OR; ++q) {
      if (PAIRS && q > 0) __syncthreads();
      in_turn<BM / OR>([&](auto which) __attribute__((always_inline)) {
        constexpr int Q = which;
        if (q == Q) {   // (different code to the compiler: one code for all of them would index the accumulators, in memory)
          asm volatile("; rows from %0" : : "n"(OR * Q));
#pragma unroll
          for (int m = 0; m < OR / 16; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) *reinterpret_cast<f32x4*>(mine + 16 * m * LR + (n >> 1) * 128 + (n & 1) * 16) = acc[n][OR / 16 * Q + m];
          asm volatile("; rows from %0" : : "n"(OR * Q));
        }
      });
      if constexpr (PAIRS) __syncthreads();
      else wave_lds_order();
#pragma unroll 1
      for (int i0 = 0; i0 < TURNS; i0 += AT_ONCE) {
        f32x4 v[AT_ONCE][2], u[AT_ONCE][2];
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            v[i][h] = *reinterpret_cast<const f32x4*>(gate + (i0 + i) * (BY * LR) + 16 * h);
            if constexpr (SILU) u[i][h] = *reinterpret_cast<const f32x4*>(up + (i0 + i) * (BY * LR) + 16 * h);
          }
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i) {
          const int64_t row = m0 + OR * q + row0 + (i0 + i) * BY;
          float y[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            y[j] = v[i][j >> 2][j & 3];
            if constexpr (BIAS) y[j] += bias[0][j];
            if constexpr (SILU) {
              float z = u[i][j >> 2][j & 3];
              if constexpr (BIAS) z += bias[1][j];
              y[j] = silu_mul_acc<bf16_tag>(y[j], z);
            }
          }
          const u32x4 o = {pack2<bf16_tag>(y[0], y[1]), pack2<bf16_tag>(y[2], y[3]), pack2<bf16_tag>(y[4], y[5]), pack2<bf16_tag>(y[6], y[7])};
          if (row < a.M && inside) {
            uint16_t* const dst = c + row * a.ldc;
            if (a.wide) *reinterpret_cast<u32x4*>(dst) = o;
            else
#pragma unroll
              for (int j = 0; j < 8; ++j) dst[j] = (uint16_t)(o[j >> 1] >> (16 * (j & 1)));
          }
        }
      }
      if constexpr (!PAIRS) wave_lds_order();
    }
  };
  if (a.silu) a.bias ? out(std::true_type{}, std::true_type{}) : out(std::true_type{}, std::false_type{});
  else a.bias ? out(std::false_type{}, std::true_type{}) : out(std::false_type{}, std::false_type{});
}

// Tiles, and what they take: us of a step of 64 k alone on the chip and with every CU busy (power), and of a tile beside its steps.
// A CU holds two of 128 x 128; from the second on a step of both takes 0.8 of `busy` and more.  Fitted to 2000 timings of 170 products of
// 129 - 5120 rows; by them the tile taken is 0.5 % behind the best one on average, 5 % at worst (without 160 x 256, and with 128 x 128 as one
// that fills a CU: 3.7 % and 19 %).  160 x 256: 2183 x 14336 x 4096 are 224 tiles, 228 us, where 192 x 256 leaves 64 CUs idle and takes 241;
// 2183 x 4096 x 4096 69.4 and 75.6; 160 x 4096 x 28672 with the SiLU 51 and 61.
struct W4Tile {
  int bm, bn, on_cu;
  float step, busy, rest;
};
constexpr W4Tile W4_TILES[] = {{256, 256, 1, 1.174f, 1.389f, 9.9f}, {256, 128, 1, 0.711f, 0.854f, 6.7f}, {128, 128, 2, 0.575f, 0.980f, 3.7f},
                               {128, 256, 1, 0.871f, 0.887f, 6.3f}, {192, 256, 1, 0.966f, 1.106f, 8.5f}, {160, 256, 1, 0.862f, 0.975f, 7.9f}};
constexpr int W4_N_TILES = sizeof(W4_TILES) / sizeof(W4_TILES[0]);
constexpr int W4_TILE_CUS = 256;
constexpr float W4_TILE_CUT = 4.6f, W4_TILE_SLABS = 4.1e6f;   // us of cutting tiles, bytes of their slabs that take one more

static W4TilePlan w4_tile_plan_of(int64_t M, int64_t N, int64_t K, int tile, int slices) {
  const W4Tile& t = W4_TILES[tile];
  W4TilePlan p{};
  p.tile = tile;
  p.mb = (int)((M + t.bm - 1) / t.bm);
  p.nb = (int)((N + t.bn - 1) / t.bn);
  const int steps = (int)(K >> 6);
  p.tiles = p.mb * p.nb;
  // few tiles are cut by as many as leave them one round, at least eight steps each
  int s = slices;
  if (s <= 0) {
    s = W4_TILE_CUS / p.tiles;
    s = s < 8 ? s : 8;
    while (s > 1 && steps / s < 8) --s;
  }
  s = s < steps ? s : steps;
  while (s > 1 && p.tiles * s > W4_TILE_CUS) --s;                // (the scratch's bound)
  while (s > 1 && (steps + s - 1) / s * (s - 1) >= steps) --s;   // no slice is empty
  p.slices = s > 1 ? s : 1;
  const size_t slabs = (size_t)p.tiles * s * t.bm * t.bn * 4;
  auto round = [&](int wgs, int n) {
    const float load = (float)wgs / W4_TILE_CUS;
    if (t.on_cu == 2) return t.rest + n * (load <= 1.f ? t.step : t.busy * (0.6f + 0.2f * load));
    return t.rest + n * (t.step + (t.busy - t.step) * load);
  };
  const int full = W4_TILE_CUS * t.on_cu, left = p.tiles % full;
  p.us = (float)(p.tiles / full) * round(full, steps);
  if (p.slices > 1) p.us = round(p.tiles * s, (steps + s - 1) / s) + W4_TILE_CUT + (float)slabs / W4_TILE_SLABS;
  else if (left) p.us += round(left, steps);
  return p;
}
W4TilePlan w4_tile_plan(int64_t M, int64_t N, int64_t K, int tile, int slices) {
  if (tile >= 0 && tile < W4_N_TILES) return w4_tile_plan_of(M, N, K, tile, slices);
  W4TilePlan best{};
  for (int t = 0; t < W4_N_TILES; ++t)
    for (int s = slices > 0 ? slices : 0; s <= (slices > 0 ? slices : 1); ++s) {
      const W4TilePlan p = w4_tile_plan_of(M, N, K, t, s);
      if (best.us == 0.f || p.us < best.us) best = p;
    }
  return best;
}

template <int BM, int BN, int NGC>
static void w4_tile_launch(const W4TileK& k, hipStream_t st) {
  constexpr int bytes = W4_TILE_LDS(BM, BN, NGC);
  auto fn = w4_tile_kernel<BM, BN, NGC>;
  static bool asked[64] = {};
  tile_allow_lds(fn, bytes, asked);
  const unsigned wgs = (unsigned)((k.tiles * k.slices + 7) / 8 * 8);
  fn<<<dim3(wgs), dim3(256), bytes, st>>>(k);
}
template <int NGC>
static void w4_tile_shape(int tile, const W4TileK& k, hipStream_t st) {
  switch (tile) {
    case 0: return w4_tile_launch<256, 256, NGC>(k, st);
    case 1: return w4_tile_launch<256, 128, NGC>(k, st);
    case 2: return w4_tile_launch<128, 128, NGC>(k, st);
    case 3: return w4_tile_launch<128, 256, NGC>(k, st);
    case 4: return w4_tile_launch<192, 256, NGC>(k, st);
    default: return w4_tile_launch<160, 256, NGC>(k, st);
  }
}

void launch_w4_tile(const GemmKParams& kp, const W4TilePlan& p, void* workspace, int ng, hipStream_t st) {
  W4TileK k{};
  k.x = (const char*)kp.a; k.wq = kp.wq; k.sz = kp.sz; k.bias = (const uint16_t*)kp.bias; k.c = (uint16_t*)kp.c;
  k.M = kp.M; k.N = kp.N; k.K = kp.K; k.ldc = kp.ldc; k.lda2 = (uint32_t)(kp.lda * 2);
  k.cpg_shift = kp.gs_shift >= 6 ? kp.gs_shift - 6 : 0;
  k.mb = p.mb; k.nb = p.nb; k.tiles = p.tiles; k.slices = p.slices; k.group = 8;
  k.silu = kp.silu;
  k.wide = kp.ldc % 8 == 0 && aligned16(kp.c);
  k.arrived = (uint32_t*)workspace; k.slabs = (float*)((char*)workspace + W4_TILE_SYNC_BYTES);
  if (p.slices > 1) tile_clear_kernel<<<dim3(1), dim3(256), 0, st>>>(k.arrived, p.tiles);
  ng == 4 ? w4_tile_shape<2>(p.tile, k, st) : w4_tile_shape<1>(p.tile, k, st);
}

}  // namespace slm
