// The 32-bit product of many rows in gemm_plain.hip's order (segments of 128 k, each a chain of multiply-adds in ascending k, added one
// after the other), on the fp32 matrix cores, for rows that begin at 16-byte boundaries and K in 32s.
//
// What bounds it is the matrix cores alone (a loop of products without memory 137 to 147 TFLOP/s, 35 cycles a product at 2.4 GHz; operands come
// at a tenth of what a unit takes in), so it is written for what kept them idle: a workgroup of eight wavefronts that owns a unit and
// goes from tile to tile; stages of 32 k of all its tiles as one stream, loaded straight into LDS (1 KiB, eight rows, a
// wavefront and instruction) three stages ahead; operands read a step of 4 k ahead, two reads an instruction; the sums of a
// segment added to the totals beside the next segment's first products, which begin at zero by themselves; and tiles of 128 rows
// and any sixteens of columns up to 144, so that a product's tiles are whole rounds of the chip. Two wavefronts a SIMD: with one (32 rows
// each) a product took 42 cycles, reads and waits in full view; so it takes 37 to 39. 1003 rows of 3584 x 18944 (256 tiles of 128 x 112) 1375
// us with 128 x 128 tiles through registers and a barrier a stage, 1054 so (129 TFLOP/s); 37888 x 3584 2411 and 2194; 4608 x 3584
// 334 and 260; 2048 rows of 3584 x 18944 2450 and 2103.
// A wavefront has sixteen rows and all columns. v_mfma_f32_16x16x4_f32, formed as W X^T: a lane's operand is a float, row lane % 16,
// k = lane / 16; its results four neighbouring columns of one row. A row's eight 16-byte pieces lie at their index xor bits 1 to
// 3 of the row: the 64 floats of an operand read stand in 64 banks.
#pragma clang fp contract(off)
#include <type_traits>
#include "common.h"
#include "hector_kernels.h"

typedef float gr_f32x4 __attribute__((ext_vector_type(4)));
#define GR_BM 128
#define GR_BK 32
#define GR_SEG 128
#define GR_BUFS 4
#define GR_BAND 8
#define GR_WAVES 8

struct GrCase {
  float* c;
  const float *a, *w;
  const void* bias;
  int bias_dtype, M, N, K;
  int64_t lda, ldw, ldc;
  bool wide;                  // four outputs of a row can be stored at once, and N is a multiple of 4
};

__device__ __forceinline__ void gr_load(uint32_t to, uint32_t offset, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(offset), "s"(base) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void gr_wait() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void gr_fixed() { __builtin_amdgcn_sched_barrier(0); }

template <int BN>
__global__ __launch_bounds__(64 * GR_WAVES, GR_WAVES / 4) void gemm_plain_rounds_kernel(GrCase c) {
  constexpr int XI = GR_BM / 16 / GR_WAVES, WI = BN / 16, NM = XI * WI;          // 16-row operand tiles of a wavefront, products of a step
  constexpr int CHUNKS = (GR_BM + BN) / 8, EACH = (CHUNKS + GR_WAVES - 1) / GR_WAVES;      // (the last wavefronts may load the last chunk again)
  constexpr uint32_t STAGE = (GR_BM + BN) * GR_BK * 4;
  static_assert(GR_BUFS * STAGE <= 160 * 1024, "a unit's LDS");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[GR_BUFS * STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntiles = (c.N + BN - 1) / BN, mtiles = (c.M + GR_BM - 1) / GR_BM;
  const int total = mtiles * ntiles, per_xcd = (total + HE_XCDS - 1) / HE_XCDS;
  // this XCD's tiles: `count` of them from `begin` on; this workgroup's: every `stride`th of these
  const int begin = blockIdx.x % HE_XCDS * per_xcd, count = min(per_xcd, total - begin), stride = gridDim.x / HE_XCDS;
  const int mine = blockIdx.x / HE_XCDS;
  if (mine >= count) return;                                 // (the whole workgroup)
  const int stages = c.K / GR_BK;
  auto tile_at = [&](int i, int& m0, int& n0) {
    const int tile = begin + i, band = tile / (GR_BAND * ntiles), in_band = tile - band * (GR_BAND * ntiles);
    const int deep = min(GR_BAND, mtiles - GR_BAND * band);
    m0 = (GR_BAND * band + in_band % deep) * GR_BM;
    n0 = in_band / deep * BN;
  };

  // ---- the stream of stages
  const uint8_t *xbase, *wbase;
  uint32_t off[EACH];
  int next = mine, ns = 0;
  auto aim = [&]() {
    int m0, n0;
    tile_at(next, m0, n0);
    xbase = (const uint8_t*)(c.a + (int64_t)m0 * c.lda);
    wbase = (const uint8_t*)(c.w + (int64_t)n0 * c.ldw);
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int chunk = min(wave * EACH + i, CHUNKS - 1), r = 8 * chunk + (lane >> 3);
      const int row = chunk < GR_BM / 8 ? min(r, c.M - 1 - m0) : min(r - GR_BM, c.N - 1 - n0);
      off[i] = (uint32_t)(row * (chunk < GR_BM / 8 ? c.lda : c.ldw) * 4) + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    }
  };
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  auto load = [&](int i, uint32_t at) {
    const int chunk = min(wave * EACH + i, CHUNKS - 1);
    gr_load(lds0 + at + chunk * 1024, off[i], chunk < GR_BM / 8 ? xbase : wbase);
  };
  auto step_on = [&]() {                                     // (behind the last tile its own stages again, which nobody reads)
    xbase += GR_BK * 4;
    wbase += GR_BK * 4;
    if (++ns == stages) {
      ns = 0;
      if (next + stride < count) next += stride;
      aim();
    }
  };

  // ---- operand reads: this lane's float of step j (4 k) of a 16-row tile
  const int r16 = lane & 15, g = lane >> 4;
  const uint32_t xrow = (wave * 16 * XI + r16) * 128 + g * 4, wrow = (GR_BM + r16) * 128 + g * 4, turn = (r16 >> 1) * 16;
  float xv[2][XI], wv[2][WI];
  gr_f32x4 acc[XI][WI], sum[XI][WI];
  auto read_x = [&](int set, int j, int i, uint32_t at) { xv[set][i] = *reinterpret_cast<const float*>(lds + at + xrow + ((16 * j) ^ turn) + i * 2048); };
  auto read_w = [&](int set, int j, int i, uint32_t at) { wv[set][i] = *reinterpret_cast<const float*>(lds + at + wrow + ((16 * j) ^ turn) + i * 2048); };

  aim();
#pragma unroll
  for (int q = 0; q < GR_BUFS; ++q) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) load(i, q * STAGE);
    step_on();
  }
  gr_wait<EACH * (GR_BUFS - 1)>();
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < WI; ++i) read_w(0, 0, i, 0);
#pragma unroll
  for (int i = 0; i < XI; ++i) read_x(0, 0, i, 0);
  uint32_t at = 0;
  // a stage: eight steps; SEGMENT: its first step begins a segment
  auto stage = [&](auto segment) {
    const uint32_t behind = at == (GR_BUFS - 1) * STAGE ? 0 : at + STAGE;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      // the next step's operands, two reads an instruction, beside the first half of this step's products: the second half covers their way
      constexpr int OPS = 1 + (WI + 1) / 2;
      if (j == 7) {
        // the next stage has arrived (the two behind it may be on their way), and everyone has read this one
        gr_fixed();
        gr_wait<EACH * (GR_BUFS - 2)>();
        __builtin_amdgcn_s_barrier();
        gr_fixed();
      }
      int m = 0;
#pragma unroll
      for (int o = 0; o < OPS; ++o) {
        const uint32_t from = j == 7 ? behind : at;
        if (o == 0) {
#pragma unroll
          for (int i = 0; i < XI; ++i) read_x((j + 1) & 1, (j + 1) & 7, i, from);
        } else {
          read_w((j + 1) & 1, (j + 1) & 7, 2 * o - 2, from);
          if (2 * o - 1 < WI) read_w((j + 1) & 1, (j + 1) & 7, 2 * o - 1, from);
        }
        if (j == 7)                                          // into the stage's own place
#pragma unroll
          for (int i = o * EACH / OPS; i < (o + 1) * EACH / OPS; ++i) load(i, at);
        gr_fixed();
#pragma unroll
        for (; m < (o == OPS - 1 ? NM : (o + 1) * NM / (2 * OPS)); ++m) {
          gr_f32x4& s = acc[m / WI][m % WI];
          if (decltype(segment)::value && j == 0) {
            sum[m / WI][m % WI] += s;
            s = gr_f32x4{0.f, 0.f, 0.f, 0.f};
          }
          s = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j & 1][m % WI], xv[j & 1][m / WI], s, 0, 0, 0);
        }
        gr_fixed();
      }
    }
    step_on();
    at = behind;
  };
  for (int i0 = mine; i0 < count; i0 += stride) {
#pragma unroll
    for (int i = 0; i < XI; ++i)
#pragma unroll
      for (int j = 0; j < WI; ++j) acc[i][j] = sum[i][j] = gr_f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < stages; ++s) {
      if (s % (GR_SEG / GR_BK) == 0) stage(std::true_type());
      else stage(std::false_type());
    }
    int m0, n0;
    tile_at(i0, m0, n0);
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int m = m0 + 16 * (wave * XI + i) + r16;
#pragma unroll
      for (int j = 0; j < WI; ++j) {
        const int n = n0 + 16 * j + 4 * g;
        gr_f32x4 v = sum[i][j] + acc[i][j];
        if (m >= c.M || n >= c.N) continue;
        if (c.bias)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += load_param(c.bias, min(n + e, c.N - 1), c.bias_dtype);
        float* p = c.c + m * c.ldc + n;
        if (c.wide) {
          *reinterpret_cast<gr_f32x4*>(p) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < c.N) p[e] = v[e];
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // nothing may be on its way into LDS that is no longer this workgroup's
}

// The columns of the tile: the least rounds of the chip, each as long as a stage takes: 0.27 us and 0.0133 for every column (16
// columns 0.45, 64 1.06, 112 1.80, 144 2.29 us).
static float gr_time(int M, int N, int bn) {
  const int64_t tiles = (int64_t)((M + GR_BM - 1) / GR_BM) * ((N + bn - 1) / bn);
  return (float)((tiles + he_cus() - 1) / he_cus()) * (bn + 20);
}
static int gr_columns(int M, int N) {
  int best = 144;
  for (int bn = 128; bn >= 16; bn -= 16)
    if (gr_time(M, N, bn) < gr_time(M, N, best)) best = bn;
  return best;
}

// Microseconds a k of K takes.
float he_gemm_plain_rounds_estimate(int M, int N) { return gr_time(M, N, gr_columns(M, N)) * (0.0133f / GR_BK); }

int he_gemm_plain_rounds(float* C, const float* A, const float* W, const void* bias, int bias_dtype, int M, int N, int K,
                         int64_t lda, int64_t ldw, int64_t ldc, hipStream_t s) {
  const int bn = gr_columns(M, N);
  const int64_t tiles = (int64_t)((M + GR_BM - 1) / GR_BM) * ((N + bn - 1) / bn);
  HE_REQUIRE(tiles < (1 << 30), "he_gemm_plain: M=%d N=%d too large for one launch", M, N);
  const int units = he_cus() / HE_XCDS * HE_XCDS, grid = (int)(tiles < units ? (tiles + HE_XCDS - 1) / HE_XCDS * HE_XCDS : units);
  const GrCase c = {C, A, W, bias, bias_dtype, M, N, K, lda, ldw, ldc, (ldc & 3) == 0 && (N & 3) == 0 && ((uintptr_t)C & 15) == 0};
  switch (bn) {
#define GR_CASE(BN_) case BN_: gemm_plain_rounds_kernel<BN_><<<grid, 64 * GR_WAVES, 0, s>>>(c); break;
    GR_CASE(16) GR_CASE(32) GR_CASE(48) GR_CASE(64) GR_CASE(80) GR_CASE(96) GR_CASE(112) GR_CASE(128) GR_CASE(144)
  }
  return he_check_launch("he_gemm_plain");
}
