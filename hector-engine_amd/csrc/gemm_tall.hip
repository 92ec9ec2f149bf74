// bf16 products of many rows on the matrix cores, one weight for all rows or one per group of rows (the experts of a routed
// feed-forward): out[m][n] = sum_k X[m][k] W[n][k], fp32 sums, K in steps of 64.
//
// A workgroup of eight wavefronts makes BM x 256 outputs (BM 256 or 128), a wavefront BM/2 x 64 of them: what its operand
// reads cost LDS, 12 KiB for 32 instructions of 16 cycles at BM 256, stays below what the unit's LDS gives. A
// stage of 64 k of both operands goes from memory straight into LDS (global_load_lds, 16 bytes a lane), one stage ahead of
// the one that is multiplied (two at BM 128, whose stages are half as long and fit three times: 2048 x 3584 x 18944 with
// weights from memory 357 us with one, 265 with two; the library's product 354). A row's eight 16-byte pieces lie at their index xor the row, so that the
// sixteen rows of an operand read hit different banks. The product is formed as W X^T: a lane then holds four
// neighbouring outputs of one row, two (gate, up) pairs where the weight's rows alternate.
// Groups: a row of tiles belongs to one group (`tile_begin`: the first tile row of each), its rows are the slots of a list
// (group_rows_kernel), their sources named by `rows_of`. The grid is sized by what the host knows; workgroups beyond the tiles
// there are leave at once. Tiles go to an XCD in stretches, eight row tiles by column after column: the 32 workgroups an XCD
// has at once read about 8 + 4 tiles of operands (12001 x 3584 x 18944: 1087 TFLOP/s without, 1176 with).
// The wavefronts work in two groups, one phase apart: while the four of one group (one a SIMD) multiply, the other four
// read their operands of the next 32 k. A stage is two such pairs of phases; each phase ends in a barrier, the second group
// begins one barrier later. A group waits for its loads of the next stage in the phase whose barrier stands before the
// first group reads that stage; a stage's buffer is filled again after the barrier behind the second group's last read of
// it. (2048 x 37888 x 3584: 1010 TFLOP/s with one barrier a stage and the groups together, 1150 so.)
#include "common.h"
#include "hector_kernels.h"

typedef __bf16 gt_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gt_f32x4 __attribute__((ext_vector_type(4)));
#define GT_BN 256
#define GT_BK 64
#define GT_WAVES 8
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
};

// one KiB: eight rows of a stage into LDS
__device__ __forceinline__ void gt_load(uint32_t to, uint32_t offset, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(offset), "s"(base) : "memory", "m0");
}

// this wavefront's loads of the next stage have arrived (those of the one after it may be on their way)
template <int LATER>
__device__ __forceinline__ void gt_wait(bool more) {
  if (LATER > 0 && more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATER) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int BM, int EPI, bool CLAMPED>
__global__ __launch_bounds__(GT_WAVES * 64, 2) void gemm_tall_kernel(GtCase c) {
  constexpr int XI = BM / 32, WI = 4;                    // 16-row operand tiles of a wavefront
  constexpr int XC = BM / 8 / GT_WAVES, WC = GT_BN / 8 / GT_WAVES;
  constexpr int NBUF = BM == 128 ? 3 : 2;
  constexpr uint32_t STAGE = (BM + GT_BN) * GT_BK * 2;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[NBUF * STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntiles = (c.N + GT_BN - 1) / GT_BN;
  const int mtiles = c.tile_begin ? c.tile_begin[c.groups] : (c.M + BM - 1) / BM;
  const int total = mtiles * ntiles;
  const int per_xcd = (total + HE_XCDS - 1) / HE_XCDS;
  const int in_xcd = blockIdx.x / HE_XCDS;
  const int tile = (blockIdx.x % HE_XCDS) * per_xcd + in_xcd;
  if (in_xcd >= per_xcd || tile >= total) return;        // (the whole workgroup)
  int group = 0, first = 0, count = mtiles;
  if (c.tile_begin) {
    int lo = 0, hi = c.groups;                           // the last group that begins at or before this tile
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (c.tile_begin[mid] * ntiles <= tile) lo = mid;
      else hi = mid;
    }
    group = lo;
    first = c.tile_begin[group];
    count = c.tile_begin[group + 1] - first;
  }
  const int local = tile - first * ntiles;
  const int band = local / (GT_BAND * ntiles), in_band = local - band * (GT_BAND * ntiles), deep = min(GT_BAND, count - GT_BAND * band);
  const int m0 = (first + GT_BAND * band + in_band % deep) * BM, n0 = in_band / deep * GT_BN;
  // sources: a lane's 16 bytes of each of its wavefront's chunks of eight rows
  const uint8_t* xbase = (const uint8_t*)(c.x + (c.rows_of ? 0 : (int64_t)m0 * c.ldx));
  const uint8_t* wbase = (const uint8_t*)(c.w + group * c.w_group + (int64_t)n0 * c.ldw);
  const uint32_t piece = (uint32_t)((lane & 7) ^ (lane >> 3)) * 16;
  uint32_t xoff[XC], woff[WC];
#pragma unroll
  for (int i = 0; i < XC; ++i) {
    const int r = 8 * (wave * XC + i) + (lane >> 3);
    int64_t row = c.rows_of ? max(c.rows_of[m0 + r], 0) : min(r, c.M - 1 - m0);
    xoff[i] = (uint32_t)(row * c.ldx * 2) + piece;
  }
#pragma unroll
  for (int i = 0; i < WC; ++i) {
    const int r = 8 * (wave * WC + i) + (lane >> 3);
    woff[i] = (uint32_t)(min(r, c.N - 1 - n0) * c.ldw * 2) + piece;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  const uint32_t xto = lds0 + wave * XC * 1024, wto = lds0 + BM * GT_BK * 2 + wave * WC * 1024;
  auto fetch = [&](uint32_t buf) {
#pragma unroll
    for (int i = 0; i < XC; ++i) gt_load(xto + buf + i * 1024, xoff[i], xbase);
#pragma unroll
    for (int i = 0; i < WC; ++i) gt_load(wto + buf + i * 1024, woff[i], wbase);
    xbase += GT_BK * 2;
    wbase += GT_BK * 2;
  };
  gt_f32x4 acc[XI][WI];
#pragma unroll
  for (int i = 0; i < XI; ++i)
#pragma unroll
    for (int j = 0; j < WI; ++j) acc[i][j] = gt_f32x4{0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, g = lane >> 4;
  const int wm = wave >> 2, wn = wave & 3;
  const uint32_t xrow = (wm * (BM / 2) + r16) * 128, wrow = BM * 128 + (wn * 64 + r16) * 128;
  const uint32_t at[2] = {(uint32_t)((g ^ (r16 & 7)) * 16), (uint32_t)(((4 + g) ^ (r16 & 7)) * 16)};
  const int stages = c.K / GT_BK;
  fetch(0);
  if (NBUF == 3 && stages > 1) {
    fetch(STAGE);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(XC + WC) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __builtin_amdgcn_s_barrier();
  if (wave >= 4) __builtin_amdgcn_s_barrier();           // the second group works one phase behind
  gt_bf16x8 xv[XI], wv[WI];
  uint32_t buf = 0;
  for (int s = 0; s < stages; ++s, buf = buf == (NBUF - 1) * STAGE ? 0 : buf + STAGE) {
    const bool more = s + NBUF - 1 < stages;             // a stage is asked for in this one
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      if (kk == 0 && more) fetch(buf >= STAGE ? buf - STAGE : (NBUF - 1) * STAGE);
#pragma unroll
      for (int j = 0; j < WI; ++j) wv[j] = *reinterpret_cast<const gt_bf16x8*>(lds + buf + wrow + at[kk] + j * 2048);
#pragma unroll
      for (int i = 0; i < XI; ++i) xv[i] = *reinterpret_cast<const gt_bf16x8*>(lds + buf + xrow + at[kk] + i * 2048);
      if (kk == 1 && wave >= 4) gt_wait<NBUF == 3 ? XC + WC : 0>(more);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < XI; ++i)
#pragma unroll
        for (int j = 0; j < WI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[j], xv[i], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
      if (kk == 1 && wave < 4) gt_wait<NBUF == 3 ? XC + WC : 0>(more);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (wave < 4) __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int m = m0 + wm * (BM / 2) + 16 * i + r16;
    if (!c.tile_begin && m >= c.M) continue;
    const float f = EPI == GT_GATED && c.scale ? c.scale[m] : 1.f;
    const int to = EPI == GT_GATED && c.spread ? c.rows_of[m] : EPI == GT_F32 && c.out_of ? c.out_of[m] : m;
    if (to < 0) continue;
    const int64_t at0 = to * c.ldo + (EPI == GT_GATED && c.spread ? (int64_t)group * (c.N / 2) : 0);
#pragma unroll
    for (int j = 0; j < WI; ++j) {
      const int n = n0 + wn * 64 + 16 * j + 4 * g;       // (N is a multiple of 4)
      if (n >= c.N) continue;
      gt_f32x4 v = acc[i][j];
      if (EPI == GT_GATED) {
        // gate and up are rounded to bf16 first, as where a kernel of its own reads them from memory: the two ways then
        // differ by the order of fp32 sums alone (a choice of weight zero gives exact zeros, whatever its row holds)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = bf16_bits_to_float(float_to_bf16_bits(v[e]));
        const float a = f == 0.f ? 0.f : he_gated_act<CLAMPED>(v[0], v[1], c.act) * f;
        const float b = f == 0.f ? 0.f : he_gated_act<CLAMPED>(v[2], v[3], c.act) * f;
        *reinterpret_cast<uint32_t*>((uint16_t*)c.out + at0 + n / 2) = pack2_bf16(a, b);
      } else if (EPI == GT_F32) {
        *reinterpret_cast<gt_f32x4*>((float*)c.out + at0 + n) = v;
      } else {
        if (c.bias)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += load_param(c.bias, n + e, c.bias_dtype);
        *reinterpret_cast<uint2*>((uint16_t*)c.out + at0 + n) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
      }
    }
  }
}

template <int BM>
static int gt_launch(const GtCase& c, int mtiles, int epi, hipStream_t s) {
  const int64_t tiles = (int64_t)mtiles * ((c.N + GT_BN - 1) / GT_BN);
  HE_REQUIRE(tiles < (1 << 28), "he_gemm_tall: %d x %d outputs are too many for one launch", c.M, c.N);
  const int grid = (int)((tiles + HE_XCDS - 1) / HE_XCDS * HE_XCDS);
  const bool clamped = !(c.act.alpha == 1.f && !(c.act.limit < INFINITY) && c.act.shift == 0.f && c.act.cubic == 0.f);
  if (epi == GT_GATED && clamped) gemm_tall_kernel<BM, GT_GATED, true><<<grid, GT_WAVES * 64, 0, s>>>(c);
  else if (epi == GT_GATED) gemm_tall_kernel<BM, GT_GATED, false><<<grid, GT_WAVES * 64, 0, s>>>(c);
  else if (epi == GT_F32) gemm_tall_kernel<BM, GT_F32, false><<<grid, GT_WAVES * 64, 0, s>>>(c);
  else gemm_tall_kernel<BM, GT_BF16, false><<<grid, GT_WAVES * 64, 0, s>>>(c);
  return he_check_launch("he_gemm_tall");
}

extern "C" int he_gemm_tall_bf16(void* out, const void* x, const void* w, const void* bias, int bias_dtype, int M, int N, int K,
                                 int64_t ldx, int64_t ldw, int64_t ldo, int epilogue, int bm, float alpha, float limit,
                                 float up_shift, float cubic, void* stream) {
  HE_REQUIRE(M >= 0 && N > 0 && K > 0 && N % 4 == 0 && K % GT_BK == 0, "he_gemm_tall: bad sizes M=%d N=%d K=%d", M, N, K);
  HE_REQUIRE(ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0 && ldo % (epilogue == GT_GATED ? 2 : 4) == 0 &&
                 ldo >= (epilogue == GT_GATED ? N / 2 : N),
             "he_gemm_tall: bad leading dimensions");
  HE_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0, "he_gemm_tall: pointers must be 16-byte aligned");
  HE_REQUIRE(epilogue >= GT_BF16 && epilogue <= GT_F32 && (bm == 128 || bm == 256), "he_gemm_tall: unknown form");
  HE_REQUIRE(bias == nullptr || epilogue == GT_BF16, "he_gemm_tall: a bias goes with plain bf16 results");
  HE_REQUIRE((int64_t)GT_BN * ldx * 2 < (1ll << 32) && (int64_t)GT_BN * ldw * 2 < (1ll << 32), "he_gemm_tall: rows too long");
  if (M == 0) return 0;
  GtCase c = {(const uint16_t*)x, (const uint16_t*)w, out, bias, bias_dtype, M, N, K, ldx, ldw, ldo, 0, nullptr, nullptr,
              nullptr, nullptr, 1, 0, {alpha, limit > 0.f ? limit : INFINITY, up_shift, cubic}};
  return bm == 256 ? gt_launch<256>(c, (M + 255) / 256, epilogue, (hipStream_t)stream)
                   : gt_launch<128>(c, (M + 127) / 128, epilogue, (hipStream_t)stream);
}

// ---- rows in groups: a token's choice of experts -----------------------------------------------
// ids [rows][top] (an expert, or what has none: below 0 or from `groups` on). Every expert gets whole tiles of BM slots;
// its tokens take them in the order of the rows. tile_begin [groups + 1]: an expert's first tile; rows_of / scale: a
// slot's row (-1: none) and the weight of that choice; choice_of: its place in ids (-1: none); slot_of [rows][top]: where a
// choice went (-1: nowhere).
// grid: an expert a workgroup, each counts all of them (a few thousand ids from L2) and writes its own.
#define GR_THREADS 1024
#define GR_MAX_GROUPS 1024
__global__ __launch_bounds__(GR_THREADS) void group_rows_kernel(int32_t* __restrict__ tile_begin, int32_t* __restrict__ rows_of,
                                                                float* __restrict__ scale, int32_t* __restrict__ slot_of,
                                                                int32_t* __restrict__ choice_of, const int32_t* __restrict__ ids,
                                                                const float* __restrict__ weights, int n, int top, int groups, int bm) {
  __shared__ int hist[GR_MAX_GROUPS];
  __shared__ int wave_sums[GR_THREADS / 64];
  __shared__ int begin_sh;
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int i = tid; i < groups; i += GR_THREADS) hist[i] = 0;
  if (tid == 0) begin_sh = 0;
  __syncthreads();
  const int each = (n + GR_THREADS - 1) / GR_THREADS;      // a thread's own stretch of the choices, in order
  const int lo = min(n, tid * each), hi = min(n, lo + each);
  int own = 0;
  for (int i = lo; i < hi; ++i) {
    const int id = ids[i];
    if (id >= 0 && id < groups) atomicAdd(&hist[id], 1);
    else if (e == 0) slot_of[i] = -1;
    own += id == e;
  }
  __syncthreads();
  int before = 0;
  for (int i = tid; i < e; i += GR_THREADS) before += (hist[i] + bm - 1) / bm;
  if (before) atomicAdd(&begin_sh, before);
  int upto = own;                                          // sums over the threads so far, this one included
  for (int m = 1; m < 64; m <<= 1) {
    const int v = __shfl_up(upto, m);
    if (lane >= m) upto += v;
  }
  if (lane == 63) wave_sums[wave] = upto;
  __syncthreads();
  int slot = upto - own;
  for (int w = 0; w < wave; ++w) slot += wave_sums[w];
  const int begin = begin_sh, tiles = (hist[e] + bm - 1) / bm;
  slot += begin * bm;
  for (int i = lo; i < hi; ++i) {
    if (ids[i] != e) continue;
    rows_of[slot] = i / top;
    scale[slot] = weights[i];
    choice_of[slot] = i;
    slot_of[i] = slot++;
  }
  for (int s = begin * bm + hist[e] + tid; s < (begin + tiles) * bm; s += GR_THREADS) rows_of[s] = choice_of[s] = -1, scale[s] = 0.f;
  if (tid == 0) tile_begin[e] = begin;
  if (tid == 0 && e == groups - 1) tile_begin[groups] = begin + tiles;
}

// tiles of bm slots that `choices` choices among `groups` experts can take
static int gr_most_tiles(int64_t choices, int groups, int bm) {
  return (int)(choices / bm + (choices < groups ? choices : groups));
}
extern "C" int he_group_rows_most_tiles(int rows, int top, int groups, int bm) {
  return rows <= 0 || top <= 0 || groups <= 0 || bm <= 0 ? 0 : gr_most_tiles((int64_t)rows * top, groups, bm);
}

// out[row][d] = the sum over the row's choices that an expert took (slot_of) of partial[row][choice][d], in their order, + dense[row][groups] * x[row][d]
// (x null: without).
__global__ __launch_bounds__(256) void combine_groups_kernel(uint16_t* __restrict__ out, const float* __restrict__ partial,
                                                             const int32_t* __restrict__ slot_of, const float* __restrict__ dense,
                                                             const uint16_t* __restrict__ x, int top, int groups, int D) {
  const int64_t row = blockIdx.y;
  const int d = 4 * (blockIdx.x * 256 + threadIdx.x);
  if (d >= D) return;
  gt_f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < top; ++k) {
    const int64_t choice = row * top + k;
    if (slot_of[choice] >= 0) sum += *reinterpret_cast<const gt_f32x4*>(partial + choice * D + d);
  }
  if (x != nullptr) {
    const float w = dense[row * (groups + 1) + groups];
    const uint2 v = *reinterpret_cast<const uint2*>(x + row * D + d);
    const uint32_t words[2] = {v.x, v.y};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (w == 0.f) break;                                 // (a row without such a choice takes nothing of x, whatever it holds)
      sum[2 * i] = fmaf(w, __uint_as_float(words[i] << 16), sum[2 * i]);
      sum[2 * i + 1] = fmaf(w, __uint_as_float(words[i] & 0xffff0000u), sum[2 * i + 1]);
    }
  }
  *reinterpret_cast<uint2*>(out + row * D + d) = make_uint2(pack2_bf16(sum[0], sum[1]), pack2_bf16(sum[2], sum[3]));
}

// The experts of a routed feed-forward, each over the rows that chose it: out[row] = the sum over the row's choices e of
// weight * down_e (act(gate_e x, up_e x)) + dense[row][real] * x (identity). Fused matrices as he_chosen_experts takes them
// (without shared columns). Scratch: lists int32 (he_routed_groups_ints), h bf16 [slots][I], slots
// = bm * he_group_rows_most_tiles(rows, top, real, bm), partial fp32 [rows][top][D]: by choice, since with few rows and many experts
// nearly all slots are padding (65 rows, 8 of 256 experts, D 7168: 33,280 slots for 520 choices, 954 MB against 15).
// down null: the activations alone, h_bf16 [rows][real I] with expert e's columns from e I on, the chosen ones written (the
// caller has cleared it); out, partial and dense are not used.
extern "C" int64_t he_routed_groups_ints(int rows, int top, int real, int bm) {
  return (real + 1 + 3) / 4 * 4 + 3ll * bm * he_group_rows_most_tiles(rows, top, real, bm) + (int64_t)rows * top;
}
extern "C" int he_routed_groups(void* out, void* lists_i32, void* h_bf16, void* partial_f32, const void* x, const void* gate_up,
                                const void* down, int64_t ldw, const void* ids_i32, const void* weights_f32,
                                const void* dense_f32, int rows, int top, int real, int I, int D, int identity, int bm,
                                float alpha, float limit, float up_shift, float cubic, void* stream) {
  HE_REQUIRE(rows >= 0 && top > 0 && real > 0 && real <= GR_MAX_GROUPS && I > 0 && D > 0, "he_routed_groups: bad sizes");
  const int spread = down == nullptr;
  HE_REQUIRE(I % GT_BK == 0 && D % GT_BK == 0 && (spread || (ldw % 8 == 0 && ldw >= (int64_t)real * I)),
             "he_routed_groups: I=%d and D=%d must be multiples of %d", I, D, GT_BK);
  HE_REQUIRE(bm == 128 || bm == 256, "he_routed_groups: tiles of 128 or 256 rows");
  HE_REQUIRE((((uintptr_t)out | (uintptr_t)lists_i32 | (uintptr_t)h_bf16 | (uintptr_t)partial_f32 | (uintptr_t)x |
               (uintptr_t)gate_up | (uintptr_t)down) & 15) == 0, "he_routed_groups: pointers must be 16-byte aligned");
  HE_REQUIRE((int64_t)rows * D * 2 < (1ll << 32) && (int64_t)GT_BN * ldw * 2 < (1ll << 32) && (int64_t)rows * top < (1 << 26) && rows <= 65535,
             "he_routed_groups: %d rows are too many", rows);
  if (rows == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const int mtiles = gr_most_tiles((int64_t)rows * top, real, bm), slots = bm * mtiles;
  int32_t* tile_begin = (int32_t*)lists_i32;
  int32_t* rows_of = tile_begin + (real + 1 + 3) / 4 * 4;
  float* scale = (float*)(rows_of + slots);
  int32_t* choice_of = (int32_t*)(scale + slots);
  int32_t* slot_of = choice_of + slots;
  group_rows_kernel<<<real, GR_THREADS, 0, s>>>(tile_begin, rows_of, scale, slot_of, choice_of, (const int32_t*)ids_i32,
                                                (const float*)weights_f32, rows * top, top, real, bm);
  int rc = he_check_launch("he_routed_groups (lists)");
  if (rc) return rc;
  const GatedAct act = {alpha, limit > 0.f ? limit : INFINITY, up_shift, cubic};
  GtCase up = {(const uint16_t*)x, (const uint16_t*)gate_up, h_bf16, nullptr, 0, slots, 2 * I, D, D, D, spread ? (int64_t)real * I : I, (int64_t)2 * I * D,
               tile_begin, rows_of, scale, nullptr, real, spread, act};
  GtCase dn = {(const uint16_t*)h_bf16, (const uint16_t*)down, partial_f32, nullptr, 0, slots, D, I, I, ldw, D, I, tile_begin,
               nullptr, nullptr, choice_of, real, 0, act};
  rc = bm == 256 ? gt_launch<256>(up, mtiles, GT_GATED, s) : gt_launch<128>(up, mtiles, GT_GATED, s);
  if (rc || spread) return rc;
  rc = bm == 256 ? gt_launch<256>(dn, mtiles, GT_F32, s) : gt_launch<128>(dn, mtiles, GT_F32, s);
  if (rc) return rc;
  combine_groups_kernel<<<dim3((D + 1023) / 1024, rows), 256, 0, s>>>((uint16_t*)out, (const float*)partial_f32, slot_of,
                                                                      (const float*)dense_f32, identity ? (const uint16_t*)x : nullptr,
                                                                      top, real, D);
  return he_check_launch("he_routed_groups (sum)");
}
