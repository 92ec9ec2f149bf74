// bf16 products of many rows on the matrix cores, one weight for all rows or one per group of rows (the experts of a routed
// feed-forward): out[m][n] = sum_k X[m][k] W[n][k], fp32 sums in order of k, K in steps of 64.
//
// A workgroup of four wavefronts, one a SIMD, makes tiles of BM x BN outputs, a wavefront a quarter (BM/2 x BN/2, in AGPRs; the
// products are inline asm, since the compiler moves accumulators of 256 registers about). It runs on the whole unit (one workgroup a
// unit, its LDS) and goes from tile to tile; the stages of 64 k of all its tiles are one stream, so that the first stages of a
// tile are on their way while the tile before it is finished and written.
// What bounds it, at 2048 x 37888 x 3584 (256 x 256, 422 us, 1.32 PFLOP/s; the kernel before, with eight wavefronts in two groups that read
// and multiplied in turn, 467): the card's power first (the matrix cores are busy 0.65 to 0.77 of the cycles at 1.9 to 2.0 GHz, of 2.4), so what
// moves operands costs clock. Wavefronts of 128 x 128 outputs read 16 KiB of LDS for 64 instructions, eight of 128 x 64 24 KiB
// (435 us with this schedule). An operand read takes the matrix cores four cycles of issue whatever the order. The
// texture units come next: a load into LDS of 1 KiB takes them 20 to 25 cycles where its rows are whole lines of 128
// bytes and 47 where they are half lines (stages of 32 k: 490 us). So a stage is 64 k, and the depth is in separate rings
// of stages for x and w (NX, NW), as many as the unit's 160 KiB hold. Loads are asked for at the start of a half stage, every
// second operand read, not spread over it: a late one is waited for (453 us spread, 435 so).
// A stage has two halves of 32 k. In the first the products of its first 32 k run, beside them the operand reads of its second 32 k
// and the loads of x's stage NX - 1 ahead; then a wait for the loads of the next stage, and the barrier. Behind it the products
// of the second 32 k, the operand reads of the next stage's first 32 k, and the loads of w's stage NW ahead, into the place that
// the barrier has freed.
// A row's eight 16-byte pieces lie at their index xor three bits of the row, so that the rows of an operand read hit
// different banks. The product is formed as W X^T, and which row of w stands at which row of an operand tile is chosen so that a lane
// ends up with 8 neighbouring outputs (16 where they become 8 gated ones): stores of 16 bytes, lines of 64 bytes a row.
// Groups: a row of tiles belongs to one group (`tile_begin`: the first tile row of each), its rows are the slots of a list
// (group_rows_kernel), their sources named by `rows_of`.
// Tiles go to an XCD in stretches, eight row tiles by column after column: the 32 workgroups of an XCD read about 8 + 4
// tiles of operands at once.
#pragma once
#include <type_traits>
#include "common.h"
#include "hector_kernels.h"

typedef __bf16 gt_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gt_f32x4 __attribute__((ext_vector_type(4)));
#define GT_BK 64
#define GT_THREADS 256
#define GT_BAND 8       // row tiles that take a column of tiles together

enum { GT_BF16 = 0, GT_GATED = 1, GT_F32 = 2 };

struct GtCase {
  const uint16_t* x;          // [rows][ldx]
  const uint16_t* w;          // group e's weight at w + e * w_group, rows of ldw
  void* out;
  const void* bias;           // [N] or null (GT_BF16)
  int bias_dtype;
  int M, N, K;                // M: rows, or with groups the slots there may be
  int64_t ldx, ldw, ldo, w_group;
  const int32_t* tile_begin;  // [groups + 1] or null: one group of all rows
  const int32_t* rows_of;     // a slot's row of x, -1: none; null: the slot itself
  const float* scale;         // a slot's factor (GT_GATED) or null
  const int32_t* out_of;      // GT_F32: a slot's row of out, -1: none; null: the slot itself
  int groups;
  int spread;                 // GT_GATED: the result goes to row rows_of[slot], columns from group * N / 2 on
  GatedAct act;
  int slices;                 // GT_F32: K slices, each K long: of x and w from slice * K on, sums to out + slice * M * ldo
  int unary;                  // GT_BF16: HE_ACT_RELU2 or HE_ACT_RELU of the result rounded to bf16; -1: none
  bool wide;                  // every row of out begins at a 16-byte boundary
};

// one KiB: eight rows of a stage into LDS; ONCE: past the caches (nothing else of the launch reads it)
template <bool ONCE = false>
__device__ __forceinline__ void gt_load(uint32_t to, uint32_t offset, const void* base) {
  if constexpr (ONCE) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(to), "v"(offset), "s"(base) : "memory", "m0");
    return;
  }
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(offset), "s"(base) : "memory", "m0");
}
// all but the last N vector memory operations of this wavefront are done, and its LDS reads
template <int N>
__device__ __forceinline__ void gt_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N > 63 ? 63 : N) : "memory");
}
// c += w x^T, or (FIRST) c = w x^T
template <bool FIRST>
__device__ __forceinline__ void gt_mfma(gt_f32x4& c, gt_bf16x8 w, gt_bf16x8 x) {
  if constexpr (FIRST) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(w), "v"(x));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(w), "v"(x));
}
// nothing is moved across
__device__ __forceinline__ void gt_fixed() { __builtin_amdgcn_sched_barrier(0); }

// a list that this launch does not write, read through the scalar cache
__device__ __forceinline__ int gt_at(const int32_t* list, int i) {
  return ((const __attribute__((address_space(4))) int32_t*)(uintptr_t)list)[i];
}

struct GtTile {
  int m0, n0, group, slice;
};

// ONE: a single row of tiles, whose weights each workgroup reads alone.
template <int BM, int BN, int NX, int NW, int EPI, bool CLAMPED, bool ONE>
__global__ __launch_bounds__(GT_THREADS, 1) void gemm_tall_kernel(GtCase c) {
  constexpr int TM = BM / 2, TN = BN / 2, XI = TM / 16, WI = TN / 16;      // a wavefront's outputs, its 16-row operand tiles
  constexpr int XL = BM / 32, WL = BN / 32;                                // its loads of a stage
  constexpr int W16 = EPI == GT_GATED ? WI / 4 * 4 : 0, W8 = WI / 2 * 2;   // operand tiles of w by fours (16 outputs a lane), by pairs (8)
  constexpr uint32_t XSTAGE = BM * GT_BK * 2, WSTAGE = BN * GT_BK * 2, WRING = NX * XSTAGE;
  static_assert(WRING + NW * WSTAGE <= 160 * 1024 && NX >= 3 && NW >= 2, "the rings");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[WRING + NW * WSTAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntiles = (c.N + BN - 1) / BN;
  const int mtiles = c.tile_begin ? gt_at(c.tile_begin, c.groups) : (c.M + BM - 1) / BM;
  const int of_slice = mtiles * ntiles, total = of_slice * (EPI == GT_F32 ? c.slices : 1), per_xcd = (total + HE_XCDS - 1) / HE_XCDS;
  // this XCD's tiles: `count` of them from `begin` on; this workgroup's: every `stride`th of these
  const int begin = blockIdx.x % HE_XCDS * per_xcd, count = min(per_xcd, total - begin), stride = gridDim.x / HE_XCDS;
  const int mine = blockIdx.x / HE_XCDS;
  if (mine >= count) return;                               // (the whole workgroup)
  const int stages = c.K / GT_BK;

  auto tile_at = [&](int i) {
    int tile = begin + i;
    GtTile t = {0, 0, 0, 0};
    if (EPI == GT_F32 && c.slices > 1) t.slice = tile / of_slice, tile -= t.slice * of_slice;
    int first = 0, deep = mtiles;
    if (c.tile_begin) {
      int lo = 0, hi = c.groups;                           // the last group that begins at or before this tile
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (gt_at(c.tile_begin, mid) * ntiles <= tile) lo = mid;
        else hi = mid;
      }
      t.group = lo;
      first = gt_at(c.tile_begin, lo);
      deep = gt_at(c.tile_begin, lo + 1) - first;
    }
    const int local = tile - first * ntiles;
    const int band = local / (GT_BAND * ntiles), in_band = local - band * (GT_BAND * ntiles);
    deep = min(GT_BAND, deep - GT_BAND * band);
    t.m0 = (first + GT_BAND * band + in_band % deep) * BM;
    t.n0 = in_band / deep * BN;
    return t;
  };

  // ---- the stream of stages: where x's and w's next loads come from
  const uint8_t *xbase, *wbase;
  uint32_t xoff[XL], woff[WL];                             // a lane's 16 bytes of each of its wavefront's chunks of eight rows
  int xi = mine, wi = mine, xs = 0, ws = 0;                // tile and stage
  auto aim_x = [&]() {
    const GtTile t = tile_at(xi);
    xbase = (const uint8_t*)(c.x + (c.rows_of ? 0 : (int64_t)t.m0 * c.ldx) + (int64_t)t.slice * c.K);
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int r = 8 * (wave * XL + i) + (lane >> 3);
      const int64_t row = c.rows_of ? max(c.rows_of[t.m0 + r], 0) : min(r, c.M - 1 - t.m0);
      xoff[i] = (uint32_t)(row * c.ldx * 2) + ((lane & 7) ^ (r & 7)) * 16;
    }
  };
  auto aim_w = [&]() {
    const GtTile t = tile_at(wi);
    wbase = (const uint8_t*)(c.w + t.group * c.w_group + (int64_t)t.n0 * c.ldw + (int64_t)t.slice * c.K);
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      const int r = 8 * (wave * WL + i) + (lane >> 3), in_wave = r % TN;
      const int turn = (in_wave & 3) + ((in_wave >> (in_wave < 16 * W16 ? 4 : 3)) & 1) * 4;
      woff[i] = (uint32_t)(min(r, c.N - 1 - t.n0) * c.ldw * 2) + ((lane & 7) ^ turn) * 16;
    }
  };
  // (behind the last tile its own stages again, which nobody reads)
  auto next_x = [&]() {
    xbase += GT_BK * 2;
    if (++xs == stages) {
      xs = 0;
      if (xi + stride < count) xi += stride;
      aim_x();
    }
  };
  auto next_w = [&]() {
    wbase += GT_BK * 2;
    if (++ws == stages) {
      ws = 0;
      if (wi + stride < count) wi += stride;
      aim_w();
    }
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  const uint32_t xto = lds0 + wave * XL * 1024, wto = lds0 + WRING + wave * WL * 1024;
  auto load_x = [&](int i, uint32_t at) { gt_load(xto + at + i * 1024, xoff[i], xbase); };
  auto load_w = [&](int i, uint32_t at) { gt_load<ONE>(wto + at + i * 1024, woff[i], wbase); };

  // ---- operand reads: row r16 of a 16-row tile, 8 k from 8 g on
  const int r16 = lane & 15, g = lane >> 4, wm = wave >> 1, wn = wave & 1;
  const uint32_t piece[2] = {(uint32_t)((g ^ (r16 & 7)) * 16), (uint32_t)(((4 + g) ^ (r16 & 7)) * 16)};
  const uint32_t xrow = (wm * TM + r16) * 128;
  // w's rows: a result's row 4 g + e of tile j is column 16 g + 4 (j & 3) + e of its four tiles, 8 g + 4 (j & 1) + e of its
  // pair, or (a single last one) 8 (g & 1) + 4 (g >> 1) + e of itself
  const uint32_t wrow16 = WRING + (wn * TN + 16 * (r16 >> 2) + (r16 & 3)) * 128, wrow8 = WRING + (wn * TN + 8 * (r16 >> 2) + (r16 & 3)) * 128;
  const uint32_t wrow4 = WRING + (wn * TN + 8 * ((r16 >> 2) & 1) + 4 * (r16 >> 3) + (r16 & 3)) * 128;
  gt_bf16x8 xv[2][XI], wv[2][WI];
  gt_f32x4 acc[XI][WI];
  auto read_x = [&](int kk, int i, uint32_t at) { xv[kk][i] = *reinterpret_cast<const gt_bf16x8*>(lds + at + xrow + piece[kk] + i * 2048); };
  auto read_w = [&](int kk, int j, uint32_t at) {
    const uint32_t row = j < W16 ? wrow16 + (64 * (j >> 2) + 4 * (j & 3)) * 128
                                 : j < W8 ? wrow8 + (32 * (j >> 1) + 4 * (j & 1)) * 128 : wrow4 + 16 * j * 128;
    wv[kk][j] = *reinterpret_cast<const gt_bf16x8*>(lds + at + row + piece[kk]);
  };

  // x's stages 0 .. NX - 2 and w's 0 .. NW - 1, in the order in which they are waited for
  aim_x();
  aim_w();
#pragma unroll
  for (int q = 0; q < (NX - 1 > NW ? NX - 1 : NW); ++q) {
    if (q < NX - 1) {
#pragma unroll
      for (int i = 0; i < XL; ++i) load_x(i, q * XSTAGE);
      next_x();
    }
    if (q < NW) {
#pragma unroll
      for (int i = 0; i < WL; ++i) load_w(i, q * WSTAGE);
      next_w();
    }
  }
  gt_wait<(NX - 2) * XL + (NW - 1) * WL>();
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int j = 0; j < WI; ++j) read_w(0, j, 0);
#pragma unroll
  for (int i = 0; i < XI; ++i) read_x(0, i, 0);
  gt_wait<63>();

  // Loads that may be on their way where the next stage must have arrived: those asked for behind it, x's and w's in turn.
  constexpr int LATER = XL + (NW >= 3 ? WL + (NX >= 4 ? XL + (NW >= 4 ? WL : 0) : 0) : 0);
  constexpr int STORES = EPI == GT_F32 ? XI * WI : XI * (W16 / 4 + (W8 - W16) / 2 + WI - W8);      // of a whole tile
  uint32_t xat = 0, wat = 0;                               // the current stage in the rings
  bool stored = false;                                     // STORES stores stand between the two
  for (int i0 = mine; i0 < count; i0 += stride) {
    auto first_half = [&](auto first) {
      constexpr int OPS = XI + WI + XL;
      const uint32_t to = xat == 0 ? (NX - 1) * XSTAGE : xat - XSTAGE;
      int m = 0, r = 0, l = 0;
#pragma unroll
      for (int o = 0; o < OPS; ++o) {
        if ((o % 2 == 0 && l < XL) || r == XI + WI) load_x(l++, to);
        else if (r < WI) read_w(1, r++, wat);
        else read_x(1, r++ - WI, xat);
        gt_fixed();
#pragma unroll
        for (; m < (o + 1) * XI * WI / OPS; ++m) gt_mfma<decltype(first)::value>(acc[m / WI][m % WI], wv[0][m % WI], xv[0][m / WI]);
        gt_fixed();
      }
      next_x();
    };
    auto second_half = [&]() {
      constexpr int OPS = XI + WI + WL;
      const uint32_t nx = xat == (NX - 1) * XSTAGE ? 0 : xat + XSTAGE, nw = wat == (NW - 1) * WSTAGE ? 0 : wat + WSTAGE;
      gt_fixed();
      __builtin_amdgcn_s_barrier();
      gt_fixed();
      int m = 0, r = 0, l = 0;
#pragma unroll
      for (int o = 0; o < OPS; ++o) {
        if ((o % 2 == 0 && l < WL) || r == XI + WI) load_w(l++, wat);
        else if (r < WI) read_w(0, r++, nw);
        else read_x(0, r++ - WI, nx);
        gt_fixed();
#pragma unroll
        for (; m < (o + 1) * XI * WI / OPS; ++m) gt_mfma<false>(acc[m / WI][m % WI], wv[1][m % WI], xv[1][m / WI]);
        gt_fixed();
      }
      next_w();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      gt_fixed();
      xat = nx;
      wat = nw;
    };
    first_half(std::true_type());
    if (stored) gt_wait<LATER + STORES>();
    else gt_wait<LATER>();
    second_half();
    for (int s = 1; s < stages; ++s) {
      first_half(std::false_type());
      gt_wait<LATER>();
      second_half();
    }
    // the last products' results are there 18 cycles after them: no accumulator is read before this (the empty asm below
    // keeps its place behind it, and every read its place behind that)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    gt_fixed();
    const GtTile t = tile_at(i0);
    const bool wide = c.wide && t.n0 + BN <= c.N;          // all columns are real: stores of 16 bytes (8 and 4 of a last pair, single)
    const bool whole = wide && !c.tile_begin && t.m0 + BM <= c.M;
    stored = whole;
#pragma unroll
    for (int i = 0; i < XI; ++i) {
#pragma unroll
      for (int j = 0; j < WI; ++j) asm volatile("" : "+a"(acc[i][j]));
      const int m = t.m0 + wm * TM + 16 * i + r16;
      if (!whole && !c.tile_begin && m >= c.M) continue;
      const float f = EPI == GT_GATED && c.scale ? c.scale[m] : 1.f;
      const int to = EPI == GT_GATED && c.spread ? c.rows_of[m] : EPI == GT_F32 && c.out_of ? c.out_of[m] : m;
      if (to < 0) continue;
      const int64_t row = to * c.ldo + (EPI == GT_GATED && c.spread ? (int64_t)t.group * (c.N / 2) : 0);
      // gate and up are rounded to bf16 first, as where a kernel of its own reads them from memory: the two ways then
      // differ by the order of fp32 sums alone (a choice of weight zero gives exact zeros, whatever its row holds). The activation is the one
      // those kernels have, bit for bit: beside a router over rows that no norm has evened out a last bit turns near ties into other
      // choices (with an exponential and a reciprocal of fewer corrections, 12001 x 37888 x 3584 2364 us instead of 2484, one such
      // design's logits moved by 7 % of their size)
      auto gated = [&](gt_f32x4 v) {
        const uint32_t p = pack2_bf16(v[0], v[1]), q = pack2_bf16(v[2], v[3]);
        const float a = f == 0.f ? 0.f : he_gated_act<CLAMPED>(__uint_as_float(p << 16), __uint_as_float(p & 0xffff0000u), c.act) * f;
        const float b = f == 0.f ? 0.f : he_gated_act<CLAMPED>(__uint_as_float(q << 16), __uint_as_float(q & 0xffff0000u), c.act) * f;
        return pack2_bf16(a, b);
      };
      auto plain = [&](gt_f32x4 v, int n) {
        if (c.bias)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += load_param(c.bias, n + e, c.bias_dtype);
        uint2 p = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
        if (c.unary >= 0) {
          auto relu = [&](uint32_t bits) {
            const float r = fmaxf(__uint_as_float(bits), 0.f);
            return c.unary == HE_ACT_RELU2 ? r * r : r;
          };
          p.x = pack2_bf16(relu(p.x << 16), relu(p.x & 0xffff0000u));
          p.y = pack2_bf16(relu(p.y << 16), relu(p.y & 0xffff0000u));
        }
        return p;
      };
#pragma unroll
      for (int j = 0; j < WI; j += j < W16 ? 4 : j < W8 ? 2 : 1) {
        // a lane's 16, 8 or 4 columns from n on (N is a multiple of 4: of 8 columns the first four or all are real)
        const int n = t.n0 + wn * TN + 16 * j + (j < W16 ? 16 * g : j < W8 ? 8 * g : 8 * (g & 1) + 4 * (g >> 1));
        if (!wide && n >= c.N) continue;
        if (EPI == GT_GATED) {
          uint16_t* p = (uint16_t*)c.out + row + n / 2;
          if (j < W16) {
            const uint4 v = make_uint4(gated(acc[i][j]), gated(acc[i][(j + 1) % WI]), gated(acc[i][(j + 2) % WI]), gated(acc[i][(j + 3) % WI]));
            if (wide) {
              *reinterpret_cast<uint4*>(p) = v;
            } else {
              const uint32_t words[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (n + 4 * q < c.N) reinterpret_cast<uint32_t*>(p)[q] = words[q];
            }
          } else if (j < W8) {
            const uint2 v = make_uint2(gated(acc[i][j]), gated(acc[i][(j + 1) % WI]));
            if (wide) {
              *reinterpret_cast<uint2*>(p) = v;
            } else {
              reinterpret_cast<uint32_t*>(p)[0] = v.x;
              if (n + 4 < c.N) reinterpret_cast<uint32_t*>(p)[1] = v.y;
            }
          } else {
            *reinterpret_cast<uint32_t*>(p) = gated(acc[i][j]);
          }
        } else if (EPI == GT_F32) {
          float* p = (float*)c.out + (int64_t)t.slice * c.M * c.ldo + row + n;
          *reinterpret_cast<gt_f32x4*>(p) = acc[i][j];
          if (j < W8 && (wide || n + 4 < c.N)) *reinterpret_cast<gt_f32x4*>(p + 4) = acc[i][(j + 1) % WI];
        } else {
          uint16_t* p = (uint16_t*)c.out + row + n;
          const uint2 a = plain(acc[i][j], n);
          if (j >= W8) {
            *reinterpret_cast<uint2*>(p) = a;
          } else if (wide) {
            const uint2 b = plain(acc[i][(j + 1) % WI], n + 4);
            *reinterpret_cast<uint4*>(p) = make_uint4(a.x, a.y, b.x, b.y);
          } else {
            *reinterpret_cast<uint2*>(p) = a;
            if (n + 4 < c.N) *reinterpret_cast<uint2*>(p + 4) = plain(acc[i][(j + 1) % WI], n + 4);
          }
        }
      }
      gt_fixed();
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // nothing may be on its way into LDS that is no longer this workgroup's
}

// The tiles there are: F(BM, BN, NX, NW).
#define GT_TILES(F) \
  F(256, 256, 3, 2) F(256, 224, 3, 2) F(256, 192, 3, 2) F(256, 160, 3, 3) F(128, 288, 3, 3) F(128, 256, 4, 3) F(128, 224, 4, 3) F(128, 160, 4, 4)

// A product with a single row of tiles runs in one no taller than it needs, its weights read past the caches: F(tile's BM, BN, BM, NX, NW), the
// lowest first. (Gate||up of 37888 x 3584 alone, weights from memory: 256 rows 76.7 -> 72.8 us, 203 in a tile of 224 75.3 -> 66, 150 in one of 160 71.6 -> 59,
// 100 of 128 59.1 -> 54.4; two rows of tiles past the caches 1.01 to 1.08 of the time without.) The heights between 128 and 256 are for steps that run as
// they are and for what is left of a long step behind turns of 8192 rows: steps of up to 512 rows that run as graphs are padded to powers of two.
#define GT_ONE_TILES(F)                                                                                                      \
  F(256, 160, 160, 4, 4) F(256, 160, 192, 4, 3) F(256, 160, 224, 3, 3) F(256, 160, 256, 3, 3)                                \
  F(256, 224, 160, 3, 3) F(256, 224, 192, 3, 3) F(256, 224, 224, 3, 2) F(256, 224, 256, 3, 2)                                \
  F(256, 256, 256, 3, 2) F(256, 192, 256, 3, 2) F(128, 288, 128, 3, 3) F(128, 256, 128, 4, 3) F(128, 224, 128, 4, 3) F(128, 160, 128, 4, 4)

template <int BM, int BN, int NX, int NW, int EPI, bool CLAMPED, bool ONE = false>
int gt_run(const GtCase& c, int mtiles, hipStream_t s) {
  const int64_t tiles = (int64_t)mtiles * ((c.N + BN - 1) / BN) * c.slices;
  HE_REQUIRE(tiles < (1 << 28), "he_gemm_tall: %d x %d outputs are too many for one launch", c.M, c.N);
  const int units = he_cus() / HE_XCDS * HE_XCDS, grid = (int)(tiles < units ? (tiles + HE_XCDS - 1) / HE_XCDS * HE_XCDS : units);
  gemm_tall_kernel<BM, BN, NX, NW, EPI, CLAMPED, ONE><<<grid, GT_THREADS, 0, s>>>(c);
  return he_check_launch("he_gemm_tall");
}
template <int EPI, bool CLAMPED>
int gt_run_tile(const GtCase& c, int tile, int mtiles, hipStream_t s) {
#define GT_ONE_CASE(TBM, BN, BM, NX, NW) \
  if (mtiles == 1 && !c.tile_begin && tile == ((TBM) << 16 | (BN)) && c.M <= BM) return gt_run<BM, BN, NX, NW, EPI, CLAMPED, true>(c, 1, s);
  GT_ONE_TILES(GT_ONE_CASE)
#undef GT_ONE_CASE
#define GT_CASE(BM, BN, NX, NW) if (tile == ((BM) << 16 | (BN))) return gt_run<BM, BN, NX, NW, EPI, CLAMPED>(c, mtiles, s);
  GT_TILES(GT_CASE)
#undef GT_CASE
  return -1;
}
// tile: BM << 16 | BN; -1: no such tile
int gt_run_bf16(const GtCase& c, int tile, int mtiles, hipStream_t s);
int gt_run_gated(const GtCase& c, int tile, int mtiles, hipStream_t s);
int gt_run_clamped(const GtCase& c, int tile, int mtiles, hipStream_t s);
int gt_run_f32(const GtCase& c, int tile, int mtiles, hipStream_t s);
