// bf16 products of many rows (the kernel: gemm_tall_tiles.h), and the experts of a routed feed-forward over the rows that chose them.
#include "gemm_tall_tiles.h"

static int gt_launch(GtCase c, int tile, int mtiles, int epi, hipStream_t s) {
  c.wide = ((uintptr_t)c.out & 15) == 0 && c.ldo * (epi == GT_F32 ? 4 : 2) % 16 == 0;
  const bool clamped = !(c.act.alpha == 1.f && !(c.act.limit < INFINITY) && c.act.shift == 0.f && c.act.cubic == 0.f);
  if (epi == GT_F32) return gt_run_f32(c, tile, mtiles, s);
  if (epi == GT_GATED) return clamped ? gt_run_clamped(c, tile, mtiles, s) : gt_run_gated(c, tile, mtiles, s);
  return gt_run_bf16(c, tile, mtiles, s);
}

extern "C" int he_gemm_tall_bf16(void* out, const void* x, const void* w, const void* bias, int bias_dtype, int M, int N, int K,
                                 int64_t ldx, int64_t ldw, int64_t ldo, int epilogue, int tile, float alpha, float limit,
                                 float up_shift, float cubic, int unary, int slices, void* stream) {
  HE_REQUIRE(M >= 0 && N > 0 && K > 0 && N % 4 == 0 && K % GT_BK == 0, "he_gemm_tall: bad sizes M=%d N=%d K=%d", M, N, K);
  HE_REQUIRE(ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0 && ldo % (epilogue == GT_GATED ? 2 : 4) == 0 &&
                 ldo >= (epilogue == GT_GATED ? N / 2 : N),
             "he_gemm_tall: bad leading dimensions");
  HE_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0, "he_gemm_tall: pointers must be 16-byte aligned");
  const int bm = tile >> 16, bn = tile & 0xffff;
  bool known = false;
#define GT_KNOWN(BM, BN, NX, NW) known = known || (bm == BM && bn == BN);
  GT_TILES(GT_KNOWN)
  HE_REQUIRE(epilogue >= GT_BF16 && epilogue <= GT_F32 && known, "he_gemm_tall: unknown form");
  HE_REQUIRE(slices >= 1 && (slices == 1 || epilogue == GT_F32) && K % slices == 0 && K / slices % GT_BK == 0,
             "he_gemm_tall: %d K slices: of fp32 results, each in whole stages", slices);
  HE_REQUIRE(bias == nullptr || epilogue == GT_BF16, "he_gemm_tall: a bias goes with plain bf16 results");
  HE_REQUIRE(unary < 0 || (epilogue == GT_BF16 && (unary == HE_ACT_RELU2 || unary == HE_ACT_RELU)),
             "he_gemm_tall: no such activation of one input, or not of plain bf16 results");
  HE_REQUIRE((int64_t)288 * ldx * 2 < (1ll << 32) && (int64_t)288 * ldw * 2 < (1ll << 32), "he_gemm_tall: rows too long");
  if (M == 0) return 0;
  const GtCase c = {(const uint16_t*)x, (const uint16_t*)w, out, bias, bias_dtype, M, N, K / slices, ldx, ldw, ldo, 0, nullptr, nullptr,
                    nullptr, nullptr, 1, 0, {alpha, limit > 0.f ? limit : INFINITY, up_shift, cubic}, slices, unary, false};
  return gt_launch(c, tile, (M + bm - 1) / bm, epilogue, (hipStream_t)stream);
}

// The tile of a product: the least estimate of its time, in rounds of the chip. A round costs a start and the write of its results (5 us)
// and its stages: microseconds a stage with all units at work, from products of 8192 cubed, 2048 x 37888 x 3584 and 2048 x 3584 x
// 18944 in every tile. Over 509 random products (65 to 12001 rows, 256 to 56000 columns, K 1088 to 27648) the choice takes 1.001 of the
// time of the fastest of the eight in the geometric mean, 1.09 at most, two above 1.05: 2048 x 3584 x 18944 225 us in 256 tiles of 128 x 224 (one round), 235 in 128 x 256, 339 in 256 x 256; 12001 x 3584 x 18944 1144 us
// in 256 x 224, 1216 in 256 x 256.
struct GtCost {
  int bm, bn;
  float stage;
};
static const GtCost gt_costs[] = {{256, 256, 1.40f}, {256, 224, 1.27f}, {256, 192, 1.13f}, {256, 160, 0.97f},
                                  {128, 288, 0.94f}, {128, 256, 0.83f}, {128, 224, 0.76f}, {128, 160, 0.65f}};
// slices: K slices, each a product of K / slices.
extern "C" int he_gemm_tall_tile(int M, int N, int K, int slices) {
  int best = 0;
  float least = INFINITY;
  for (const GtCost& t : gt_costs) {
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * slices;
    const int64_t rounds = (tiles + he_cus() - 1) / he_cus();
    const float us = rounds * (5.f + K / slices / GT_BK * t.stage);
    if (us < least) least = us, best = t.bm << 16 | t.bn;
  }
  return best;
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
  HE_REQUIRE((int64_t)rows * D * 2 < (1ll << 32) && (int64_t)256 * ldw * 2 < (1ll << 32) && (int64_t)rows * top < (1 << 26) && rows <= 65535,
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
  const GtCase up = {(const uint16_t*)x, (const uint16_t*)gate_up, h_bf16, nullptr, 0, slots, 2 * I, D, D, D, spread ? (int64_t)real * I : I, (int64_t)2 * I * D,
               tile_begin, rows_of, scale, nullptr, real, spread, act, 1, -1, false};
  const GtCase dn = {(const uint16_t*)h_bf16, (const uint16_t*)down, partial_f32, nullptr, 0, slots, D, I, I, ldw, D, I, tile_begin,
               nullptr, nullptr, choice_of, real, 0, act, 1, -1, false};
  rc = gt_launch(up, bm << 16 | 256, mtiles, GT_GATED, s);
  if (rc || spread) return rc;
  rc = gt_launch(dn, bm << 16 | 256, mtiles, GT_F32, s);
  if (rc) return rc;
  combine_groups_kernel<<<dim3((D + 1023) / 1024, rows), 256, 0, s>>>((uint16_t*)out, (const float*)partial_f32, slot_of,
                                                                      (const float*)dense_f32, identity ? (const uint16_t*)x : nullptr,
                                                                      top, real, D);
  return he_check_launch("he_routed_groups (sum)");
}
