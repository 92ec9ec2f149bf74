// A token's choice among experts, the experts' gated activation weighted by that choice, and the
// combination of the two score maps of a differential attention head.
#include "common.h"
#include "hector_kernels.h"
#include <type_traits>

#define ROUTE_MAX_EXPERTS 1024

// One workgroup a row, or two rows. logits [rows][E] fp32, or, with x and router given, the router's product itself:
// logits[e] = sum_i x[row][i] * router[e][i] in fp32 (router fp32 [E][D]; a lane adds its elements i = lane,
// lane + 64, ... in that order, the lanes' sums meet in the wavefront's butterfly: one fixed order a row,
// whatever else the step holds). bias (or null): a stored number an output, added to its logit first. x_pieces: the bf16
// rows lie piece-major for the grid's rows. s = softmax(logits) over all E outputs; the choice is made
// on c = s + correction: the E outputs are cut into `groups` equal runs of neighbours, each run ranked by the
// largest c it holds; outside the `keep` best runs every c is replaced by -inf, and the `top` largest c that
// are left are chosen. The weight of a chosen output is s * scale (s, not c; the weights are not made to sum
// to one). The last E - real outputs are experts without weights whose result is the input
// itself: their weights are added up in column `real` of dense. dense [rows][real + 1] holds the
// weight of every expert (0 where not chosen); ids / weights [rows][top] list the chosen ones.
//
// A step of many rows is bound by the reads of the router's matrix from L2, D * E * 4 bytes a workgroup: two rows share them.
// What bounds a step of few rows is the chain: the router's rows come from memory, so a wavefront asks for those of up to four
// outputs, with the row, its scale's parts, the biases and corrections, all at the start; the choice is made by the first wavefront alone, PL
// outputs a lane in registers, without a barrier or a walk through LDS a choice, while the others write the scaled row. (2 rows of 2048, 18
// outputs in 3 groups, 4 chosen: 14.5 us with eight wavefronts that meet at two barriers a choice and ask for one output at a time, 9 so; 2048 rows 41 us and 31; one
// row of 300 outputs in 5 groups, 8 chosen, 89 and 36. The loads in two turns, the scale, the corrections and the scaled row one after the other in front of
// the choice: the same 2 rows within a step 10.4 us, so 7.3.)
#define ROUTE_WAVES 8

// Rows x whose norm's scale is still owed (partials null: none is): the rows are bf16(x * inv) with inv as scale_rows_kernel forms it, and
// the workgroup leaves them, row-major, in `out`: a launch less (2 rows of 2048, 18 outputs: 8.0 us in two launches, 7.1 in one, warm; with
// 128 outputs, whose rows' scaling is done again for every four outputs of a wavefront, 20.0 and 20.5: up to 64 outputs only).
struct RouteOwed {
  const float* partials;      // [rows][count]: the row's sum of squares in parts
  int count;
  float eps;
  uint16_t* out;
};

__device__ __forceinline__ float4 route_four(const uint2 b) {
  return make_float4(__uint_as_float(b.x << 16), __uint_as_float(b.x & 0xffff0000u), __uint_as_float(b.y << 16),
                     __uint_as_float(b.y & 0xffff0000u));
}

__device__ __forceinline__ uint2 route_scaled(const uint2 b, float inv) {
  const float4 v = route_four(b);
  return make_uint2(float_to_bf16_bits(v.x * inv) | (uint32_t)float_to_bf16_bits(v.y * inv) << 16,
                    float_to_bf16_bits(v.z * inv) | (uint32_t)float_to_bf16_bits(v.w * inv) << 16);
}

// The scale a row still owes, from its parts in the order lane, lane + 64, ...: the first ROUTE_PARTS of a lane are asked for ahead.
#define ROUTE_PARTS 4
struct RouteParts {
  float v[ROUTE_PARTS];
};
__device__ __forceinline__ RouteParts route_parts(const RouteOwed& owed, int64_t row) {
  RouteParts p;
#pragma unroll
  for (int j = 0; j < ROUTE_PARTS; ++j) p.v[j] = owed.partials[row * owed.count + min((int)(threadIdx.x & 63) + 64 * j, owed.count - 1)];
  return p;
}
__device__ __forceinline__ float route_inv(const RouteParts& p, const RouteOwed& owed, int64_t row, int D) {
  const int lane = threadIdx.x & 63;
  float part = 0.f;
#pragma unroll
  for (int j = 0; j < ROUTE_PARTS; ++j)
    if (lane + 64 * j < owed.count) part += p.v[j];
  for (int i = lane + 64 * ROUTE_PARTS; i < owed.count; i += 64) part += owed.partials[row * owed.count + i];
  return 1.0f / sqrtf(wave_sum(part) / (float)D + owed.eps);
}

// The dot products of row x with the router's rows e0, e0 + ROUTE_WAVES, ... (OUT of them, those beyond E repeat the last): four elements
// a lane and turn, four sums a lane that meet in index order. The loads of up to eight turns (rows of 2048 elements) are
// asked for together, ahead of what the row's scale is made of: one trip to memory.
template <int OUT, bool OWED>
__device__ __forceinline__ void route_dots(float (&z)[OUT], const void* x, int x_dtype, const float* router, int64_t row, int rows, int D, int E,
                                           int e0, int x_pieces, const RouteParts& parts, const RouteOwed& owed) {
  const int lane = threadIdx.x & 63;
  const bool vec = (D & 3) == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)router & 15) == 0;
  const float* w[OUT];
  float a[OUT][4];
#pragma unroll
  for (int o = 0; o < OUT; ++o) {
    w[o] = router + (int64_t)min(e0 + o * ROUTE_WAVES, E - 1) * D;
#pragma unroll
    for (int j = 0; j < 4; ++j) a[o][j] = 0.f;
  }
  if (vec) {
    constexpr int TURNS = OUT > 2 ? 4 : 8;
    // row-major: four elements i at 4 i; piece-major [D / 8][rows][8]: half i & 1 of the row's piece i / 2
    const uint2* xh = reinterpret_cast<const uint2*>((const uint16_t*)x) + (x_pieces ? 2 * row : row * (D >> 2));
    const float4* xf = reinterpret_cast<const float4*>((const float*)x + row * D);
    const int64_t piece = 2 * (int64_t)rows;
    const int n = D >> 2;
    float inv = 1.f;
    const auto walk = [&](auto bf) {         // one loop a type, without a branch around its loads
      for (int i0 = 0; i0 < n; i0 += 64 * TURNS) {
        uint2 xb[TURNS];
        float4 xv[TURNS], wv[TURNS][OUT];
#pragma unroll
        for (int t = 0; t < TURNS; ++t) {
          const int i = min(i0 + 64 * t + lane, n - 1);
          if constexpr (decltype(bf)::value) xb[t] = xh[x_pieces ? (i >> 1) * piece + (i & 1) : i];
          else xv[t] = xf[i];
#pragma unroll
          for (int o = 0; o < OUT; ++o) wv[t][o] = reinterpret_cast<const float4*>(w[o])[i];
        }
        __builtin_amdgcn_sched_barrier(0);
        if (OWED && i0 == 0) inv = route_inv(parts, owed, row, D);
#pragma unroll
        for (int t = 0; t < TURNS; ++t) {
          if (i0 + 64 * t + lane >= n) continue;
          if constexpr (decltype(bf)::value) xv[t] = route_four(OWED ? route_scaled(xb[t], inv) : xb[t]);
#pragma unroll
          for (int o = 0; o < OUT; ++o) {
            a[o][0] = fmaf(xv[t].x, wv[t][o].x, a[o][0]);
            a[o][1] = fmaf(xv[t].y, wv[t][o].y, a[o][1]);
            a[o][2] = fmaf(xv[t].z, wv[t][o].z, a[o][2]);
            a[o][3] = fmaf(xv[t].w, wv[t][o].w, a[o][3]);
          }
        }
      }
    };
    if (OWED || x_dtype == HE_BF16) walk(std::true_type{});
    else walk(std::false_type{});
  } else {
    for (int i = lane; i < D; i += 64) {
      const float xv = x_dtype == HE_BF16 ? bf16_bits_to_float(((const uint16_t*)x)[row * D + i])
                                          : ((const float*)x)[row * D + i];
#pragma unroll
      for (int o = 0; o < OUT; ++o) a[o][0] = fmaf(xv, w[o][i], a[o][0]);
    }
  }
#pragma unroll
  for (int o = 0; o < OUT; ++o) z[o] = wave_sum((a[o][0] + a[o][1]) + (a[o][2] + a[o][3]));
}

// The same for RW rows from row0 on (those beyond the last repeat it), row-major, so that a load of the router's rows serves RW of them: every
// product and sum as above.
template <int OUT, int RW>
__device__ __forceinline__ void route_dots_rows(float (&z)[RW][OUT], const void* x, int x_dtype, const float* router, int row0, int rows,
                                                int D, int E, int e0) {
  const int lane = threadIdx.x & 63;
  const float* w[OUT];
  int64_t at[RW];
  float a[RW][OUT][4];
#pragma unroll
  for (int r = 0; r < RW; ++r) at[r] = (int64_t)min(row0 + r, rows - 1) * (D >> 2);
#pragma unroll
  for (int o = 0; o < OUT; ++o) {
    w[o] = router + (int64_t)min(e0 + o * ROUTE_WAVES, E - 1) * D;
#pragma unroll
    for (int r = 0; r < RW; ++r)
#pragma unroll
      for (int j = 0; j < 4; ++j) a[r][o][j] = 0.f;
  }
  const auto turns = [&](auto bf) {         // one loop a type, without a branch in it: a turn's loads are in flight together
#pragma unroll 2
    for (int i = lane; i < (D >> 2); i += 64) {
      float4 xv[RW];
#pragma unroll
      for (int r = 0; r < RW; ++r) {
        if constexpr (decltype(bf)::value) xv[r] = route_four(((const uint2*)x)[at[r] + i]);
        else xv[r] = ((const float4*)x)[at[r] + i];
      }
#pragma unroll
      for (int o = 0; o < OUT; ++o) {
        const float4 wv = reinterpret_cast<const float4*>(w[o])[i];
#pragma unroll
        for (int r = 0; r < RW; ++r) {
          a[r][o][0] = fmaf(xv[r].x, wv.x, a[r][o][0]);
          a[r][o][1] = fmaf(xv[r].y, wv.y, a[r][o][1]);
          a[r][o][2] = fmaf(xv[r].z, wv.z, a[r][o][2]);
          a[r][o][3] = fmaf(xv[r].w, wv.w, a[r][o][3]);
        }
      }
    }
  };
  if (x_dtype == HE_BF16) turns(std::true_type{});
  else turns(std::false_type{});
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int o = 0; o < OUT; ++o) z[r][o] = wave_sum((a[r][o][0] + a[r][o][1]) + (a[r][o][2] + a[r][o][3]));
}

// The lowest index among the largest of the lanes' values (lane, lane + 64, ...), NaN never; `none` if all are NaN.
template <int PL>
__device__ __forceinline__ int route_argmax(const float (&c)[PL], int none) {
  float v = -INFINITY;
#pragma unroll
  for (int j = 0; j < PL; ++j) v = fmaxf(v, c[j]);
  v = wave_max(v);
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    const unsigned long long hit = __builtin_amdgcn_ballot_w64(c[j] == v);
    if (hit != 0) return 64 * j + __ffsll((long long)hit) - 1;       // (the same in all lanes)
  }
  return none;
}

template <int PL, int RW, bool OWED>
__global__ __launch_bounds__(64 * ROUTE_WAVES) void route_kernel(
    float* __restrict__ dense, int32_t* __restrict__ ids, float* __restrict__ weights, const float* __restrict__ logits,
    const void* __restrict__ x, int x_dtype, const float* __restrict__ router, int D,
    const void* __restrict__ correction, int c_dtype, int rows, int E, int real, int groups, int keep, int top, float scale,
    int normalize, const void* __restrict__ bias, int bias_dtype, int x_pieces, RouteOwed owed) {
  static_assert(RW <= ROUTE_WAVES && (RW == 1 || !OWED), "a wavefront chooses for a row");
  __shared__ float z_all[RW][64 * PL], c_all[RW][64 * PL];
  const int row0 = blockIdx.x * RW;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  // what the choosing wavefronts need at the end, asked for at the start (each lane its first output's)
  const bool chooses = wave < RW && row0 + wave < rows;
  float bias0 = 0.f, correction0 = 0.f;
  if (chooses && lane < E) {
    if (bias) bias0 = load_param(bias, lane, bias_dtype);
    if (correction) correction0 = load_param(correction, lane, c_dtype);
  }
  RouteParts parts = {};
  if (OWED) parts = route_parts(owed, row0);
  if (x != nullptr) {
    for (int e0 = wave; e0 < E; e0 += 4 * ROUTE_WAVES) {
      if (e0 + 2 * ROUTE_WAVES < E) {
        float z[RW][4];
        if constexpr (RW == 1) route_dots<4, OWED>(z[0], x, x_dtype, router, row0, rows, D, E, e0, x_pieces, parts, owed);
        else route_dots_rows<4, RW>(z, x, x_dtype, router, row0, rows, D, E, e0);
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
          for (int o = 0; o < 4; ++o)
            if (lane == 0 && e0 + o * ROUTE_WAVES < E) z_all[r][e0 + o * ROUTE_WAVES] = z[r][o];
      } else {
        float z[RW][2];
        if constexpr (RW == 1) route_dots<2, OWED>(z[0], x, x_dtype, router, row0, rows, D, E, e0, x_pieces, parts, owed);
        else route_dots_rows<2, RW>(z, x, x_dtype, router, row0, rows, D, E, e0);
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
          for (int o = 0; o < 2; ++o)
            if (lane == 0 && e0 + o * ROUTE_WAVES < E) z_all[r][e0 + o * ROUTE_WAVES] = z[r][o];
      }
    }
    __syncthreads();
  }
  if (OWED && wave >= RW) {      // the scaled row, by the wavefronts that don't choose
    const float inv = route_inv(parts, owed, row0, D);
    const uint2* xh = reinterpret_cast<const uint2*>((const uint16_t*)x) + (x_pieces ? 2 * (int64_t)row0 : (int64_t)row0 * (D >> 2));
    uint2* to = reinterpret_cast<uint2*>(owed.out) + (int64_t)row0 * (D >> 2);
    for (int i = threadIdx.x - 64 * RW; i < (D >> 2); i += 64 * (ROUTE_WAVES - RW))
      to[i] = route_scaled(x_pieces ? xh[(i >> 1) * (2 * (int64_t)rows) + (i & 1)] : xh[i], inv);
  }
  const int64_t row = row0 + wave;
  if (wave >= RW || row >= rows) return;
  float* z_sh = z_all[wave];
  float* c_sh = c_all[wave];
  // element j of a lane's arrays is output lane + 64 j; those beyond E are NaN to the choice
  float z[PL], s[PL], c[PL], d[PL];
  float mx = -INFINITY;
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    const int e = lane + 64 * j;
    z[j] = s[j] = d[j] = 0.f;
    if (e >= E) continue;
    z[j] = (x != nullptr ? z_sh[e] : logits[row * E + e]) + (bias ? j == 0 ? bias0 : load_param(bias, e, bias_dtype) : 0.f);
    mx = fmaxf(mx, z[j]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    if (lane + 64 * j >= E) continue;
    s[j] = expf(z[j] - mx);
    sum += s[j];
  }
  sum = wave_sum(sum);
  const float inv = 1.f / sum;
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    // a score is rounded, then its sum with the correction: as one multiply-add, for the outputs whose correction is at hand, two outputs of equal
    // scores and corrections on both sides of 64 would no longer tie
#pragma clang fp contract(off)
    const int e = lane + 64 * j;
    s[j] *= inv;
    // (without a correction the choice is made on the logits themselves: the same order, and no two meet at zero)
    c[j] = e >= E ? NAN : correction ? s[j] + (j == 0 ? correction0 : load_param(correction, e, c_dtype)) : z[j];
  }
  if (keep < groups) {
    // a lane ranks whole groups; the kept ones are marked by NaN, then the others' outputs are masked
    const int size = E / groups;
#pragma unroll
    for (int j = 0; j < PL; ++j) c_sh[lane + 64 * j] = c[j];
    __builtin_amdgcn_wave_barrier();
    float g[PL];
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      const int group = lane + 64 * j;
      g[j] = NAN;
      if (group >= groups) continue;
      float best = -INFINITY;
#pragma unroll 4
      for (int i = 0; i < size; ++i) best = fmaxf(best, c_sh[group * size + i]);
      g[j] = best == INFINITY ? NAN : best;      // (such a group is kept beside the `keep` best)
    }
    for (int k = 0; k < keep; ++k) {
      const int best = route_argmax<PL>(g, E);
#pragma unroll
      for (int j = 0; j < PL; ++j)
        if (best == lane + 64 * j) g[j] = NAN;
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < PL; ++j) c_sh[lane + 64 * j] = g[j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < PL; ++j) {
      const int e = lane + 64 * j;
      if (e < E && !isnan(c_sh[e / size])) c[j] = -INFINITY;
    }
  }
  float chosen_sum = 0.f, rest = 0.f;      // the chosen outputs' scores; the weights of those from `real` on: both in the order of the choice
  for (int k = 0; k < top; ++k) {
    const int e = route_argmax<PL>(c, E);
    const bool found = e < E;
    float score = 0.f;
#pragma unroll
    for (int j = 0; j < PL; ++j)
      if (e >> 6 == j) score = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s[j]), e & 63));
    const float w = found ? score * scale : 0.f;
    if (found) {
      chosen_sum += score;
      if (e >= real) rest += w;
#pragma unroll
      for (int j = 0; j < PL; ++j)
        if (e == lane + 64 * j) c[j] = NAN, d[j] = w;
    }
    if (lane == 0) {
      ids[row * top + k] = found ? e : -1;
      // normalize: the chosen outputs' weights are made to sum to `scale` (the softmax over the chosen logits alone), below
      weights[row * top + k] = w;
    }
  }
  const float norm = normalize ? 1.f / chosen_sum : 1.f;
#pragma unroll
  for (int j = 0; j < PL; ++j) {
    const int e = lane + 64 * j;
    if (e < real) dense[row * (real + 1) + e] = normalize ? d[j] * norm : d[j];
  }
  if (lane == 0) {
    dense[row * (real + 1) + real] = normalize ? rest * norm : rest;
    if (normalize)
      for (int k = 0; k < top; ++k) weights[row * top + k] *= norm;
  }
}

extern "C" int he_route_tokens(void* dense_f32, void* ids_i32, void* weights_f32, const void* logits_f32,
                               const void* x, int x_dtype, const void* router_f32, int D,
                               const void* correction, int c_dtype, int rows, int E, int real, int groups, int keep,
                               int top, float scale, int normalize, const void* bias, int bias_dtype, int x_pieces,
                               const void* partials_f32, int count, float eps, void* scaled_out, void* stream) {
  HE_REQUIRE((logits_f32 != nullptr) != (x != nullptr), "he_route_tokens: give the logits, or the rows and the router");
  HE_REQUIRE(x == nullptr || (router_f32 != nullptr && D > 0 && (x_dtype == HE_BF16 || x_dtype == HE_F32)),
             "he_route_tokens: the router's matrix is missing");
  HE_REQUIRE(rows >= 0 && E > 0 && E <= ROUTE_MAX_EXPERTS && real >= 0 && real <= E,
             "he_route_tokens: bad sizes E=%d real=%d (at most %d outputs)", E, real, ROUTE_MAX_EXPERTS);
  HE_REQUIRE(groups > 0 && E % groups == 0 && keep > 0 && keep <= groups,
             "he_route_tokens: %d outputs do not form %d equal groups of which %d are kept", E, groups, keep);
  HE_REQUIRE(top > 0 && top <= keep * (E / groups), "he_route_tokens: %d chosen of %d kept outputs", top,
             keep * (E / groups));
  HE_REQUIRE(!x_pieces || (x != nullptr && x_dtype == HE_BF16 && (D & 7) == 0 && (((uintptr_t)x | (uintptr_t)router_f32) & 15) == 0),
             "he_route_tokens: piece-major rows are bf16, 16-byte aligned and a multiple of 8 wide");
  HE_REQUIRE(partials_f32 == nullptr ||
                 (x != nullptr && x_dtype == HE_BF16 && E <= 64 && scaled_out != nullptr && count > 0 && (D & 7) == 0 &&
                  (((uintptr_t)x | (uintptr_t)router_f32 | (uintptr_t)scaled_out) & 15) == 0),
             "he_route_tokens: rows whose scale is owed are bf16, 16-byte aligned and a multiple of 8 wide, for at most 64 outputs");
  if (rows == 0) return 0;
  const RouteOwed owed = {(const float*)partials_f32, count, eps, (uint16_t*)scaled_out};
#define ROUTE_LAUNCH(PL, RW, OWED)                                                                                             \
  route_kernel<PL, RW, OWED><<<(rows + (RW) - 1) / (RW), 64 * ROUTE_WAVES, 0, (hipStream_t)stream>>>(                               \
      (float*)dense_f32, (int32_t*)ids_i32, (float*)weights_f32, (const float*)logits_f32, x, x_dtype, (const float*)router_f32, D, \
      correction, c_dtype, rows, E, real, groups, keep, top, scale, normalize, bias, bias_dtype, x_pieces, owed)
  // Two rows a workgroup where that leaves no compute unit idle: one load of the router's rows serves both, and two wavefronts choose at once.
  // (us with one row a workgroup and two, bf16 rows of 2048: 18 outputs, 256 rows 6.3 and 5.8, 512 rows 9.7 and 6.0, 4096 rows
  // 53.6 and 23.7; 128 outputs 20.1 and 18.2, 33.8 and 19.2, 222 and 96.5; 64 rows the same within 0.3. Four rows a workgroup: 7.2, 7.3 and
  // 21.8 with 18 outputs, 27, 27 and 98 with 128.)
  const bool shared = x != nullptr && !x_pieces && rows > 256 && (D & 3) == 0 && (((uintptr_t)x | (uintptr_t)router_f32) & 15) == 0;
#define ROUTE_OUTPUTS(PL)                       \
  if (shared) ROUTE_LAUNCH(PL, 2, false);       \
  else ROUTE_LAUNCH(PL, 1, false)
  if (partials_f32 != nullptr) ROUTE_LAUNCH(1, 1, true);
  else if (E <= 64) { ROUTE_OUTPUTS(1); }
  else if (E <= 256) { ROUTE_OUTPUTS(4); }
  else { ROUTE_OUTPUTS(16); }
#undef ROUTE_OUTPUTS
#undef ROUTE_LAUNCH
  return he_check_launch("he_route_tokens");
}

// out [rows][real * I + shared + extra]: column e * I + i = act(gate, up) * dense[row][e] with gate and up the
// columns 2 (e I + i) and 2 (e I + i) + 1 of gate_up (a fused weight whose rows alternate gate and up),
// act as he_gated_act; the `shared` columns behind them likewise with weight 1 (an expert every row uses); the last `extra` columns = dense[row][real] * h[row][:] (the share of the
// experts whose result is their input). A product over these columns with the experts' down
// matrices side by side (and an identity block for the extra columns) is the weighted sum of the
// chosen experts' results.
template <typename T, bool CLAMPED>
__global__ void routed_act_kernel(T* __restrict__ out, const T* __restrict__ gate_up, const float* __restrict__ dense,
                                  const T* __restrict__ h, int real, int I, int shared, int extra, GatedAct act) {
  const int64_t row = blockIdx.y;
  const int gated = real * I + shared;
  const int cols = gated + extra;
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= cols) return;
  const float* d = dense + row * (real + 1);
  float v;
  if (j < gated) {
    const float w = j < real * I ? d[j / I] : 1.f;
    const T* gu = gate_up + row * (int64_t)(2 * gated) + 2 * j;
    // an expert that was not chosen gives exact zeros, whatever its rows hold
    v = w == 0.f ? 0.f : he_gated_act<CLAMPED>(to_float(gu[0]), to_float(gu[1]), act) * w;
  } else {
    const float w = d[real];
    v = w == 0.f ? 0.f : w * to_float(h[row * (int64_t)extra + (j - gated)]);
  }
  out[row * (int64_t)cols + j] = from_float<T>(v);
}

// The same for bf16 rows, eight columns a thread (16-byte loads and stores): needs I and extra in multiples of 8.
template <bool CLAMPED>
__global__ void routed_act_vec_kernel(uint16_t* __restrict__ out, const uint16_t* __restrict__ gate_up,
                                      const float* __restrict__ dense, const uint16_t* __restrict__ h, int real, int I,
                                      int shared, int extra, GatedAct act) {
  const int64_t row = blockIdx.y;
  const int gated = real * I + shared;
  const int cols = gated + extra;
  const int j = 8 * (blockIdx.x * blockDim.x + threadIdx.x);
  if (j >= cols) return;
  const float* d = dense + row * (real + 1);
  float v[8];
  if (j < gated) {
    const float w = j < real * I ? d[j / I] : 1.f;
    const uint4* gu = reinterpret_cast<const uint4*>(gate_up + row * (int64_t)(2 * gated) + 2 * j);
    const uint4 lo = gu[0], hi = gu[1];
    const uint32_t pairs[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};      // (gate, up) a word
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[i] = w == 0.f ? 0.f
                      : he_gated_act<CLAMPED>(__uint_as_float(pairs[i] << 16), __uint_as_float(pairs[i] & 0xffff0000u), act) * w;
  } else {
    const float w = d[real];
    const uint4 raw = *reinterpret_cast<const uint4*>(h + row * (int64_t)extra + (j - gated));
    const uint32_t words[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = w == 0.f ? 0.f : w * __uint_as_float(words[i] << 16);
      v[2 * i + 1] = w == 0.f ? 0.f : w * __uint_as_float(words[i] & 0xffff0000u);
    }
  }
  *reinterpret_cast<uint4*>(out + row * (int64_t)cols + j) =
      make_uint4(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]), pack2_bf16(v[4], v[5]), pack2_bf16(v[6], v[7]));
}

extern "C" int he_routed_act(void* out, const void* gate_up, const void* dense_f32, const void* h, int rows, int real,
                             int I, int shared, int extra, int dtype, float alpha, float limit, float up_shift, float cubic,
                             void* stream) {
  HE_REQUIRE(rows >= 0 && real >= 0 && I > 0 && shared >= 0 && extra >= 0 && (int64_t)real * I + shared + extra > 0, "he_routed_act: bad sizes");
  HE_REQUIRE(extra == 0 || h != nullptr, "he_routed_act: the input rows are missing");
  HE_REQUIRE(dtype == HE_BF16 || dtype == HE_F32, "he_routed_act: unknown dtype %d", dtype);
  if (rows == 0) return 0;
  const int cols = real * I + shared + extra;
  const dim3 grid((cols + 255) / 256, rows);
  hipStream_t s = (hipStream_t)stream;
  const bool clamped = !he_gated_act_is_silu(alpha, limit, up_shift, cubic);
  const GatedAct act = {alpha, limit > 0.f ? limit : INFINITY, up_shift, cubic};
  if (dtype == HE_BF16 && I % 8 == 0 && shared % 8 == 0 && extra % 8 == 0 &&
      ((((uintptr_t)out) | ((uintptr_t)gate_up) | ((uintptr_t)h)) & 15) == 0) {
    const dim3 vgrid((cols / 8 + 255) / 256, rows);
    if (clamped)
      routed_act_vec_kernel<true><<<vgrid, 256, 0, s>>>((uint16_t*)out, (const uint16_t*)gate_up, (const float*)dense_f32,
                                                        (const uint16_t*)h, real, I, shared, extra, act);
    else
      routed_act_vec_kernel<false><<<vgrid, 256, 0, s>>>((uint16_t*)out, (const uint16_t*)gate_up, (const float*)dense_f32,
                                                         (const uint16_t*)h, real, I, shared, extra, act);
    return he_check_launch("he_routed_act");
  }
#define ACT_LAUNCH(T, CL)                                                                                      \
  routed_act_kernel<T, CL><<<grid, 256, 0, s>>>((T*)out, (const T*)gate_up, (const float*)dense_f32, (const T*)h, real, \
                                                I, shared, extra, act)
  if (dtype == HE_BF16) {
    if (clamped) ACT_LAUNCH(bf16_t, true); else ACT_LAUNCH(bf16_t, false);
  } else {
    if (clamped) ACT_LAUNCH(float, true); else ACT_LAUNCH(float, false);
  }
#undef ACT_LAUNCH
  return he_check_launch("he_routed_act");
}

// ---- the chosen experts alone, for steps of very few rows ---------------------------------------
// Where a step's rows choose fewer experts than there are, the two products over all experts read weights
// nobody asked for. These two kernels walk only the chosen experts' rows of the same fused matrices (bf16):
// a wavefront an output, the lanes along K with 16-byte loads, sums in fp32. Weights that one row of the step alone reads come past the caches, those
// of an expert that several rows chose, and of the shared columns, by way of them: 8 rows of 4 choices among 64 experts of 1024 over 2048 and 2048 shared
// columns, weights from memory, 80 us all by way of the caches, 86 all past them, 75 so; where all rows choose the same experts 47, 70 and 49. (One row of 4 choices
// among 16 experts of 2048 over 2048 28.2 and 25.5.) Two rows' experts come past the caches whoever chose them: by way of them where both did, 2 rows of 4
// among those 16 take 37.3 us instead of 39.6 when alone, but within a step the small kernels behind them find their code and arguments gone, 0.2 to 0.4 us
// each, and a request of eight such steps takes 0.6 % longer (5284 and 5255 us). (Read past the caches by two rows, those of 3 rows and more are slower by more than that: 4 rows
// of 2 among 16 of 1024 over 2048 20.6 us instead of 19.4.)
__device__ __forceinline__ float dot8_bf16(const uint4& a, const uint4& b, float acc) {
  const uint32_t x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    acc = fmaf(__uint_as_float(x[i] << 16), __uint_as_float(y[i] << 16), acc);
    acc = fmaf(__uint_as_float(x[i] & 0xffff0000u), __uint_as_float(y[i] & 0xffff0000u), acc);
  }
  return acc;
}

// ONCE: past the caches (he_load16_once).
template <bool ONCE>
__device__ __forceinline__ uint4 chosen_load(const uint16_t* p) {
  return ONCE ? he_load16_once<uint4>(p) : *reinterpret_cast<const uint4*>(p);
}

// The ids of a step of several rows, a lane each (up to 64: one trip to memory for all that a wavefront asks of them).
struct ChosenIds {
  int rows, n, mine;
  bool held;
  __device__ __forceinline__ ChosenIds(const int32_t* __restrict__ ids, int rows, int top)
      : rows(rows), n(rows * top), mine(0), held(rows > 2 && n <= 64) {
    if (held) mine = ids[min((int)(threadIdx.x & 63), n - 1)];
  }
  __device__ __forceinline__ int at(const int32_t* __restrict__ ids, int i) const { return held ? __builtin_amdgcn_readlane(mine, i) : ids[i]; }
  // whether one row alone chose expert e (of more than 64 ids: not said; of one or two rows: taken so)
  __device__ __forceinline__ bool alone(int e) const {
    return rows <= 2 || (held && __popcll(__ballot((int)(threadIdx.x & 63) < n && mine == e)) == 1);
  }
};

// Grid y: the rows * top (row, choice) pairs, then, with shared columns, the rows once more: those write h_shared[row][i].
// h[(row, k), i] = weight[row, k] * act(gate . x[row], up . x[row]) with gate and up the rows 2 (e I + i) and
// 2 (e I + i) + 1 of gate_up [2 real I][D], e = ids[row, k]; zeros where e is no expert with weights.
template <bool CLAMPED>
__global__ __launch_bounds__(256) void chosen_gate_up_kernel(uint16_t* __restrict__ h, const uint16_t* __restrict__ x,
                                                             const uint16_t* __restrict__ gate_up,
                                                             const int32_t* __restrict__ ids,
                                                             const float* __restrict__ weights, int top, int real, int I,
                                                             int shared, int rows, int x_pieces, int D, GatedAct act) {
  const int lane = threadIdx.x & 63;
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
  const bool common = (int)blockIdx.y >= rows * top;   // the columns every row uses
  const int64_t rk = blockIdx.y;                 // row * top + k
  if (i >= (common ? shared : I)) return;
  const ChosenIds chosen(ids, rows, top);
  const int e = common ? real : chosen.at(ids, (int)rk);
  const int64_t row = common ? rk - (int64_t)rows * top : rk / top;
  float g = 0.f, u = 0.f;
  if (common || (e >= 0 && e < real)) {
    const uint16_t* wg = gate_up + ((int64_t)e * I + i) * 2 * D;
    // row-major rows, or piece-major [D / 8][rows][8]
    const uint16_t* xr = x + (x_pieces ? 8 * row : row * D);
    const int64_t x_step = x_pieces ? rows : 1;
    const auto walk = [&](auto once) {
      constexpr bool ONCE = decltype(once)::value;
#pragma unroll 4
      for (int c = lane * 8; c < D; c += 512) {
        const uint4 xv = *reinterpret_cast<const uint4*>(xr + c * x_step);
        g = dot8_bf16(chosen_load<ONCE>(wg + c), xv, g);
        u = dot8_bf16(chosen_load<ONCE>(wg + D + c), xv, u);
      }
    };
    if (common ? rows == 1 : chosen.alone(e)) walk(std::true_type{});
    else walk(std::false_type{});
  }
  g = wave_sum(g);
  u = wave_sum(u);
  if (lane == 0) {
    const float v = common ? he_gated_act<CLAMPED>(g, u, act)
                    : (e >= 0 && e < real) ? he_gated_act<CLAMPED>(g, u, act) * weights[rk] : 0.f;
    h[common ? (int64_t)rows * top * I + row * shared + i : rk * I + i] = float_to_bf16_bits(v);
  }
}

// out[row, d] = sum over the row's chosen experts e of down[d][e I ..] . h[(row, k)] (+ down[d][real I ..] . h_shared[row]) + dense[row][real] * x[row, d]
// (down [D][ldw]: the experts' matrices side by side; the last term is the identity experts' share).
__global__ __launch_bounds__(256) void chosen_down_kernel(uint16_t* __restrict__ out, const uint16_t* __restrict__ h,
                                                          const uint16_t* __restrict__ x, const uint16_t* __restrict__ down,
                                                          int64_t ldw, const int32_t* __restrict__ ids,
                                                          const float* __restrict__ dense, int top, int real, int I,
                                                          int shared, int identity, int D) {
  const int lane = threadIdx.x & 63;
  const int d = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t row = blockIdx.y;
  if (d >= D) return;
  const int rows = gridDim.y;
  float acc = 0.f;
  const auto walk = [&](const uint16_t* w, const uint16_t* hr, int n, auto once) {
    constexpr bool ONCE = decltype(once)::value;
#pragma unroll 4
    for (int c = lane * 8; c < n; c += 512) acc = dot8_bf16(chosen_load<ONCE>(w + c), *reinterpret_cast<const uint4*>(hr + c), acc);
  };
  const ChosenIds chosen(ids, rows, top);
  for (int k = 0; k < top; ++k) {
    const int e = chosen.at(ids, (int)row * top + k);
    if (e < 0 || e >= real) continue;
    const uint16_t* w = down + (int64_t)d * ldw + (int64_t)e * I;
    const uint16_t* hr = h + (row * top + k) * I;
    if (chosen.alone(e)) walk(w, hr, I, std::true_type{});
    else walk(w, hr, I, std::false_type{});
  }
  const uint16_t* ws = down + (int64_t)d * ldw + (int64_t)real * I;
  const uint16_t* hs = h + (int64_t)rows * top * I + row * shared;
  if (rows == 1) walk(ws, hs, shared, std::true_type{});
  else walk(ws, hs, shared, std::false_type{});
  acc = wave_sum(acc);
  if (lane == 0)
    out[row * D + d] = float_to_bf16_bits(
        identity ? fmaf(dense[row * (real + 1) + real], bf16_bits_to_float(x[row * D + d]), acc) : acc);
}

extern "C" int he_chosen_experts(void* out, void* h_scratch, const void* x, const void* gate_up, const void* down,
                                 int64_t ldw, const void* ids_i32, const void* weights_f32, const void* dense_f32,
                                 int rows, int top, int real, int I, int shared, int D, float alpha, float limit,
                                 float up_shift, float cubic, int x_pieces, void* stream) {
  HE_REQUIRE(rows >= 0 && top > 0 && real > 0 && I > 0 && D > 0, "he_chosen_experts: bad sizes");
  HE_REQUIRE(I % 8 == 0 && shared >= 0 && shared % 8 == 0 && D % 8 == 0 && ldw % 8 == 0 && ldw >= (int64_t)real * I + shared,
             "he_chosen_experts: I=%d, shared=%d, D=%d and the down matrix's row stride must be multiples of 8", I, shared, D);
  const int identity = ldw > (int64_t)real * I + shared;
  HE_REQUIRE(!(x_pieces && identity), "he_chosen_experts: the identity experts' share reads row-major rows");
  HE_REQUIRE(((((uintptr_t)out) | ((uintptr_t)h_scratch) | ((uintptr_t)x) | ((uintptr_t)gate_up) | ((uintptr_t)down)) & 15) == 0,
             "he_chosen_experts: pointers must be 16-byte aligned");
  HE_REQUIRE((int64_t)rows * (top + 1) <= 65535, "he_chosen_experts: too many rows");
  if (rows == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const bool clamped = !he_gated_act_is_silu(alpha, limit, up_shift, cubic);
  const GatedAct act = {alpha, limit > 0.f ? limit : INFINITY, up_shift, cubic};
  const dim3 grid_up((max(I, shared) + 3) / 4, rows * (top + (shared > 0 ? 1 : 0)));
  if (clamped)
    chosen_gate_up_kernel<true><<<grid_up, 256, 0, s>>>((uint16_t*)h_scratch, (const uint16_t*)x, (const uint16_t*)gate_up,
                                                        (const int32_t*)ids_i32, (const float*)weights_f32, top, real, I,
                                                        shared, rows, x_pieces, D, act);
  else
    chosen_gate_up_kernel<false><<<grid_up, 256, 0, s>>>((uint16_t*)h_scratch, (const uint16_t*)x, (const uint16_t*)gate_up,
                                                         (const int32_t*)ids_i32, (const float*)weights_f32, top, real, I,
                                                         shared, rows, x_pieces, D, act);
  int st = he_check_launch("he_chosen_experts (gate, up)");
  if (st) return st;
  chosen_down_kernel<<<dim3((D + 3) / 4, rows), 256, 0, s>>>((uint16_t*)out, (const uint16_t*)h_scratch, (const uint16_t*)x,
                                                             (const uint16_t*)down, ldw, (const int32_t*)ids_i32,
                                                             (const float*)dense_f32, top, real, I, shared, identity, D);
  return he_check_launch("he_chosen_experts (down)");
}

// Differential attention's last step. attn [rows][2 H][hd] holds, for kv head g and its R = H / G
// query heads, first the R outputs of score map 1 and then the R outputs of map 2 (head order
// [g][map][r]); out [rows][H][vd], head h = g R + r:
//   o = a1 - lambda a2;  out = o / sqrt(mean(o^2) + eps) * post
// over the vd values of a head (no learned gain). One wavefront a (row, head).
template <typename T>
__global__ __launch_bounds__(64) void diff_heads_kernel(T* __restrict__ out, const T* __restrict__ attn, int H, int G,
                                                        int hd, int vd, float lambda, float post, float eps) {
  const int64_t row = blockIdx.y;
  const int h = blockIdx.x;
  const int R = H / G;
  const int g = h / R, r = h - g * R;
  const T* a1 = attn + (row * 2 * H + (int64_t)(2 * g) * R + r) * hd;
  const T* a2 = a1 + (int64_t)R * hd;
  float sq = 0.f;
  for (int i = threadIdx.x; i < vd; i += 64) {
    const float o = fmaf(-lambda, to_float(a2[i]), to_float(a1[i]));
    sq = fmaf(o, o, sq);
  }
  sq = wave_sum(sq);
  const float mul = post / sqrtf(sq / (float)vd + eps);
  T* dst = out + (row * H + h) * vd;
  for (int i = threadIdx.x; i < vd; i += 64) {
    const float o = fmaf(-lambda, to_float(a2[i]), to_float(a1[i]));
    dst[i] = from_float<T>(o * mul);
  }
}

extern "C" int he_diff_heads(void* out, const void* attn, int rows, int H, int G, int hd, int vd, float lambda,
                             float post, float eps, int dtype, void* stream) {
  HE_REQUIRE(rows >= 0 && H > 0 && G > 0 && H % G == 0 && vd > 0 && vd <= hd, "he_diff_heads: bad sizes H=%d G=%d hd=%d vd=%d",
             H, G, hd, vd);
  HE_REQUIRE(dtype == HE_BF16 || dtype == HE_F32, "he_diff_heads: unknown dtype %d", dtype);
  if (rows == 0) return 0;
  const dim3 grid(H, rows);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == HE_BF16)
    diff_heads_kernel<bf16_t><<<grid, 64, 0, s>>>((bf16_t*)out, (const bf16_t*)attn, H, G, hd, vd, lambda, post, eps);
  else
    diff_heads_kernel<float><<<grid, 64, 0, s>>>((float*)out, (const float*)attn, H, G, hd, vd, lambda, post, eps);
  return he_check_launch("he_diff_heads");
}
