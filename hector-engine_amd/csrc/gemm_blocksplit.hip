// bf16 matrix product for few rows (M <= 32) with K cut inside the workgroup:
// C[M,N] = X[M,K] * W[N,K]^T (+ bias), or the gated activation of a gate||up
// weight. One workgroup owns up to 32 weight rows (blocksplit_plan; 64 in ordered_plan); its NW wavefronts take one K slice
// each (operands straight from global memory into the MFMA registers, laid out so that the weight is read in whole lines, see
// BsLanes), leave their fp32 sums in LDS, and the workgroup adds the slices in wavefront order and writes
// the result. The sum is complete inside one launch: no partial sums in global
// memory, no second kernel, no atomics, and the order of the additions is fixed.
// What bounds it: the weight's way from memory (6.3 to 6.6 TB/s at 37888 x 3584 up to 8 rows), and for small products the launch and one
// trip to memory: nothing is read ahead of the first weights, and what the epilogue reads is asked for behind them.
//
// Gated epilogue: the weight alternates gate and up rows (gate i at row 2i, its up at
// 2i + 1), so the four neighbouring weight rows whose sums a thread holds are two
// (gate, up) pairs, and the output is silu(gate) * up, [M, N/2] (reference:
// kernels/activations.cu:183-198 as a kernel of its own).
//
// Two more epilogues carry an RMS norm across a pair of products without a kernel of
// its own (reference: kernels/fused_add_rmsnorm.cu:47-81 as a separate kernel):
//   residual: r[m][n] += acc (+ bias), stored fp32 in place; xg[m][n] = bf16(r * g[n]) with
//     the gain g of the norm that follows; and the sum of r^2 over the workgroup's columns
//     per row, one partial per workgroup: sq[m][block].
//   row scale: the consumer of xg adds the partials of a row in a fixed order,
//     s[m] = 1 / sqrt(sum / dim + eps), and multiplies its sums by s[m] before bias or
//     gate: W (r g s) = s W (r g). The norm's statistics stay fp32.
//
// Activations between two such products may lie piece-major instead of row-major: a [M, D]
// bf16 tensor as 16-byte pieces [D / 8][M][8], element (m, d) at ((d / 8) M + m) 8 + d % 8.
// The lanes of an activation operand load then read neighbouring pieces (whole lines)
// instead of one piece of a line in each row. The
// producing epilogue writes the layout, the consuming product reads it (x_pieces / out_pieces).
#include "common.h"
//
// The kernel is in gemm_blocksplit_tiles.h, its tilings are compiled in
// gemm_blocksplit_tiles_*.hip; this file has the rule that picks a tiling and the entry points.
#include "gemm_blocksplit_tiles.h"


// The tiling of a product, from its sizes only, so that it always runs the same way. Swept on MI355X over NA, S, NW and the rows of a
// workgroup at 20 shapes (896 x 896 to 152064 x 3584 and 5120 x 27648) with 1, 4, 8 and 16 rows, weights from memory: this choice is within 4 % of the best of
// some 60 tilings at all but the smallest.
// Weight rows of a workgroup: the multiple of four (outputs are stored in fours; 3584 x 3584 in rows of 14 8.5 us, of 16 7.2) up to 16 or
// 32 that costs least as rounds of the chip times rows and a start worth four rows, of equal ones the largest (each workgroup reads all of
// X). 5120 x 27648 at 8 rows in rows of 20 52 us, of 8 or 10 55 to 58; 8512 x 2048 at 1 row in twelves 9.1, in sixteens
// 9.8; 37888 x 3584 at 16 rows in thirty-twos 49, in eights 86.
// NW = 8 wavefronts take a K slice each; 4 where that leaves a slice one instruction and the chip has other workgroups to run
// (151936 x 896 at 4 rows 43 us, with eight 52). A wavefront with a single accumulator asks for two units a step (896 x 4864 at 8 rows 6.0 us, 6.8).
// plan arguments NA, S, NW <= 0: this choice; NA: instructions' weight rows a wavefront holds (1, 2 or 4; 1 or 2 above 16 rows), S: units a step.
// (More than 16 rows come here with plan arguments alone: see ordered_plan.)
static BlockSplitPlan blocksplit_plan(int M, int N, int K, int NA, int S, int NW) {
  BlockSplitPlan p;
  const int cus = he_cus();
  p.SP = M <= 4 ? 2 : M <= 16 ? 1 : 0;
  p.MT = M <= 8 ? 1 : 2;
  const int rt = 16 >> p.SP, km = p.SP == 0 ? 64 : 32 << p.SP, units = (K + km - 1) / km;
  int rows = 0, best = 0;
  for (int r = p.SP == 2 ? 16 : 32; r >= 4; r -= 4) {
    const int blocks = (N + r - 1) / r, cost = (blocks + cus - 1) / cus * (r + 4);
    if (rows == 0 || cost < best) best = cost, rows = r;
  }
  p.NA = rows <= rt ? 1 : rows <= 2 * rt ? 2 : 4;
  if (NA > 0) p.NA = NA, rows = rt * NA;
  p.S = S > 0 ? (S > 1 ? 2 : 1) : p.NA == 1 ? 2 : 1;
  p.rows_per_block = rows;
  if (NW <= 0) {
    NW = units < 16 && N >= 2 * cus * rows ? 4 : 8;
    while (NW > 1 && 2 * units <= NW) NW >>= 1;
  }
  if (NW > bs_max_waves(p.MT, p.NA, p.S)) NW = bs_max_waves(p.MT, p.NA, p.S);
  p.NW = NW;
  p.units = (units + NW - 1) / NW;
  p.turn = p.S;
  return p;
}

// The tiling of the ordered sums: tiles, K slices and turns of 128 u k as this product had them before its lanes were spread. For weights of up
// to 16 rows whose results reach a router over rows that no norm has evened out (there another order of sums turns near ties over), and for
// 17 to 32 rows.
static BlockSplitPlan ordered_plan(int M, int N, int K) {
  BlockSplitPlan p;
  const int cus = he_cus();
  p.SP = 0, p.MT = M <= 16 ? 1 : 2;
  int r, u, nw;
  if (N >= 256 * cus) {             // 256 rows or more a unit
    if (M <= 8) r = 2, u = 1, nw = 8;
    else r = p.MT == 1 ? 4 : 2, u = 2, nw = 4;
  } else if (K >= 8192) {           // long K
    const int groups = (N + 31) / 32, last_round = groups % cus;   // with two tiles a workgroup
    if (N < 16 * cus) r = 1, u = 1, nw = p.MT == 1 ? 8 : 4;
    else if (p.MT == 2) r = 2, u = 2, nw = 4;
    else if (M > 8 && N >= 40 * cus) r = 4, u = 2, nw = 4;
    else if (groups < cus) r = 2, u = 1, nw = 8;
    else if (groups < 4 * cus && last_round > 0 && last_round <= cus / 2) r = 1, u = 1, nw = 8;
    else if (K >= 16384) r = 2, u = 2, nw = 8;
    else r = 2, u = 4, nw = 4;
  } else if (N >= 64 * cus) {       // wide N
    r = M > 8 && p.MT == 1 ? 4 : 2, u = 1, nw = 8;
    if (K < 5120) r = 2;
    if (p.MT == 2 || K < 5120) u = 2, nw = 4;
  } else {                          // small products
    r = N >= 16 * cus ? 2 : 1, u = p.MT == 1 && K < 5120 ? 4 : 1, nw = 8;
  }
  int rows = 0;
  if (r <= 2 && N >= 2 * cus && N < 256 * cus) {      // dealt out evenly over the compute units, an even number each
    const int rounds = (N + cus * 32 - 1) / (cus * 32);
    rows = ((N + cus * rounds - 1) / (cus * rounds) + 1) & ~1;
    r = rows > 16 ? 2 : 1;
  }
  while (nw > 1 && K / nw < 128) nw >>= 1;      // (at most 8: bs_max_waves for any of these)
  // (Two units of a turn a step also where a wavefront has one accumulator and turns of two: 2048 x 32768 in sixteen groups, 4 rows, 31.7 -> 28.5 us;
  // with two accumulators 65536 x 2048 so 36.7 -> 41.9; above 16 rows 3584 x 18944 39.5 -> 38.0, but 3584 x 3584 11.3 -> 12.1.)
  p.NA = r, p.S = u > 1 || (r == 1 && (p.MT == 1 || K >= 8192)) ? 2 : 1, p.NW = nw;
  p.units = ((K + nw - 1) / nw + 63) / 64;
  p.turn = 2 * u;
  p.rows_per_block = rows > 0 ? rows : 16 * r;
  return p;
}

// Workgroups (= partial sums of squares per row) the residual epilogue of this product gives.
extern "C" int he_gemm_blocksplit_blocks(int M, int N, int K) {
  if (M <= 0 || M > HE_BLOCKSPLIT_MAX_M || N <= 0 || K <= 0) return 0;
  const BlockSplitPlan p = M > 16 ? ordered_plan(M, N, K) : blocksplit_plan(M, N, K, 0, 0, 0);
  return (N + p.rows_per_block - 1) / p.rows_per_block;
}

// NA, S, NW: the tiling asked for, <= 0 the one blocksplit_plan chooses (NW wavefronts = K slices per workgroup). S = 4 asks for two units, as 2 does
// (not beside NA = 4).
// scale_partials: sums of squares of the input rows (the rows are then scaled before
// bias or gate); resid: the residual epilogue (C is not written; gain, xg, sq_out needed). unary: an activation of one input
// (he_unary's kinds) of the bf16 results, -1: none: a feed-forward without a gate writes its activations at once (a launch of its
// own for 18944 of them took 4.7 us beside the product's 26). used: groups of the weight that no row uses are not read (BsFusion):
// the experts of a routed step that nobody chose. ordered: see ordered_plan.
extern "C" int he_gemm_blocksplit_fused_bf16(void* C, const void* A, const void* W,
                                             const void* bias, int M, int N, int K, int out_dtype,
                                             int bias_dtype, int gated, int NA, int S, int NW,
                                             const void* scale_partials, int scale_count,
                                             float scale_eps, void* resid, const void* gain,
                                             int gain_dtype, void* xg, void* sq_out,
                                             int sq_count, int x_pieces, int out_pieces,
                                             float act_alpha, float act_limit, float act_shift, float act_cubic,
                                             float resid_scale, const void* dyt_bias,
                                             const void* dyt_alpha, int unary, const void* used, int used_ld,
                                             int used_count, int used_rows, int used_k, int ordered, void* stream) {
  HE_REQUIRE((dyt_alpha == nullptr) == (dyt_bias == nullptr), "he_gemm_blocksplit_bf16: Dynamic Tanh needs alpha and bias");
  HE_REQUIRE(M > 0 && M <= HE_BLOCKSPLIT_MAX_M, "he_gemm_blocksplit_bf16: M=%d outside [1, %d]", M,
             HE_BLOCKSPLIT_MAX_M);
  HE_REQUIRE(N > 0 && K > 0, "he_gemm_blocksplit_bf16: bad sizes N=%d K=%d", N, K);
  HE_REQUIRE((K & 7) == 0, "he_gemm_blocksplit_bf16: K=%d must be a multiple of 8", K);
  HE_REQUIRE(out_dtype == HE_BF16 || out_dtype == HE_F32, "he_gemm_blocksplit_bf16: bad out dtype");
  HE_REQUIRE((((uintptr_t)A | (uintptr_t)W) & 15) == 0,
             "he_gemm_blocksplit_bf16: operands must be 16-byte aligned");
  HE_REQUIRE(!gated || ((N & 1) == 0 && bias == nullptr),
             "he_gemm_blocksplit_bf16: the gated epilogue needs an even N=%d and no bias", N);
  HE_REQUIRE(scale_partials == nullptr || scale_count > 0,
             "he_gemm_blocksplit_bf16: row scale without partial sums");
  HE_REQUIRE(!(x_pieces || out_pieces) || M <= 16,
             "he_gemm_blocksplit_bf16: piece-major activations are for up to 16 rows, not %d", M);
  HE_REQUIRE(!out_pieces || ((resid != nullptr || out_dtype == HE_BF16) && ((gated ? N / 2 : N) & 7) == 0),
             "he_gemm_blocksplit_bf16: a piece-major output is bf16 and a multiple of 8 wide");
  HE_REQUIRE(unary < 0 || (unary <= HE_ACT_RELU && !gated && resid == nullptr && out_dtype == HE_BF16),
             "he_gemm_blocksplit_bf16: an activation of one input goes with plain bf16 results");
  HE_REQUIRE(used == nullptr || (M <= 16 && !gated && used_count >= 0 && used_ld >= used_count && used_rows >= 0 && used_k >= 0 &&
                                 (used_rows > 0) != (used_k > 0) && (used_k == 0 || used_k >= 512) &&
                                 (resid == nullptr || used_rows == 0) && (resid != nullptr || out_dtype == HE_BF16)),
             "he_gemm_blocksplit_bf16: groups that are used: up to 16 rows, bf16 results, along the rows or in stretches of 512 k and more");
  HE_REQUIRE(!ordered || (M <= 16 && resid == nullptr && NA <= 0 && S <= 0 && NW <= 0),
             "he_gemm_blocksplit_bf16: ordered sums are for up to 16 rows, plan themselves and leave no residual");
  HE_REQUIRE(NA <= (M <= 16 ? 4 : 2) && NA != 3 && S <= (M <= 16 && NA != 4 ? 4 : 2) && S != 3,
             "he_gemm_blocksplit_bf16: no tiling NA=%d S=%d at M=%d", NA, S, M);
  const bool planned = NA <= 0 && S <= 0 && NW <= 0;
  const BlockSplitPlan p = ordered || (planned && M > 16) ? ordered_plan(M, N, K) : blocksplit_plan(M, N, K, NA, S, NW);
  // (a lane's offsets into X and into its workgroup's weight rows are 32 bits of bytes)
  const int most_rows = N < p.rows_per_block ? N : p.rows_per_block;
  HE_REQUIRE((int64_t)(M > most_rows ? M : most_rows) * K < (1ll << 31), "he_gemm_blocksplit_bf16: K=%d: rows too long", K);
  HE_REQUIRE(p.NW >= 1 && p.NW <= 16, "he_gemm_blocksplit_bf16: %d wavefronts outside [1, 16]",
             p.NW);
  const int blocks = (N + p.rows_per_block - 1) / p.rows_per_block;
  if (resid != nullptr) {
    HE_REQUIRE(!gated && gain != nullptr && xg != nullptr && sq_out != nullptr,
               "he_gemm_blocksplit_bf16: the residual epilogue needs gain, xg and sq_out, and no gate");
    HE_REQUIRE(sq_count == blocks,
               "he_gemm_blocksplit_bf16: %d partial sums per row given, the product has %d workgroups",
               sq_count, blocks);
    HE_REQUIRE(gain_dtype == HE_F32 || gain_dtype == HE_BF16, "he_gemm_blocksplit_bf16: bad gain dtype");
  } else {
    HE_REQUIRE(C != nullptr, "he_gemm_blocksplit_bf16: no output");
  }
  BsFusion fu;
  fu.scale_partials = (const float*)scale_partials;
  fu.scale_count = scale_count;
  fu.scale_eps = scale_eps;
  fu.scale_dim = K;
  fu.resid = (float*)resid;
  fu.gain = gain;
  fu.gain_dtype = gain_dtype;
  fu.xg = (uint16_t*)xg;
  fu.sq_out = (float*)sq_out;
  fu.out_pieces = out_pieces;
  fu.act_clamped = gated && !he_gated_act_is_silu(act_alpha, act_limit, act_shift, act_cubic);
  fu.act.alpha = act_alpha;
  fu.act.limit = act_limit > 0.f ? act_limit : INFINITY;
  fu.act.shift = act_shift;
  fu.act.cubic = act_cubic;
  fu.unary = unary;
  fu.used = (const float*)used;
  fu.used_ld = used_ld, fu.used_count = used_count, fu.used_rows = used_rows, fu.used_k = used_k;
  fu.resid_scale = resid_scale;
  fu.dyt_bias = dyt_bias;
  fu.dyt_alpha = dyt_alpha;
  hipStream_t s = (hipStream_t)stream;
  const bool f32 = out_dtype != HE_BF16;
  const int rc = (resid != nullptr ? (used ? he_blocksplit_tiles_used_resid : he_blocksplit_tiles_resid)
                  : used           ? he_blocksplit_tiles_used_bf16
                  : gated          ? (f32 ? he_blocksplit_tiles_gated_f32 : he_blocksplit_tiles_gated_bf16)
                                   : (f32 ? he_blocksplit_tiles_f32 : he_blocksplit_tiles_bf16))(p, C, A, W, bias, bias_dtype, M, N, K, fu,
                                                                                                  x_pieces != 0, s);
  if (rc) return rc;
  return he_check_launch("he_gemm_blocksplit_bf16");
}

extern "C" int he_gemm_blocksplit_bf16(void* C, const void* A, const void* W, const void* bias,
                                       int M, int N, int K, int out_dtype, int bias_dtype,
                                       int gated, int NA, int S, int NW, void* stream) {
  return he_gemm_blocksplit_fused_bf16(C, A, W, bias, M, N, K, out_dtype, bias_dtype, gated, NA, S,
                                       NW, nullptr, 0, 0.f, nullptr, nullptr, HE_F32, nullptr,
                                       nullptr, 0, 0, 0, 1.f, 0.f, 0.f, 0.f, 1.f, nullptr, nullptr, -1, nullptr, 0, 0, 0, 0, 0, stream);
}
