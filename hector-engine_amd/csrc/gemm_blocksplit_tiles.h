// The kernel of gemm_blocksplit.hip and its launch, shared by the files that each compile its
// tilings for one epilogue and output type (gemm_blocksplit_tiles_*.hip): compiled in one file
// they would set the time of the whole build.
#pragma once
#include "common.h"
#include "hector_kernels.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

__device__ __forceinline__ bf16x8 bs_load8(const char* p) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}

// Four neighbouring outputs. align: how many elements the address is a multiple of (4, 2 or 1).
template <typename TC>
__device__ __forceinline__ void bs_store4(TC* p, const float v[4], int align, int valid);
template <>
__device__ __forceinline__ void bs_store4<float>(float* p, const float v[4], int align, int valid) {
  if (align >= 4 && valid == 4) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  } else if (align >= 2 && valid == 4) {
    *reinterpret_cast<float2*>(p) = make_float2(v[0], v[1]);
    *reinterpret_cast<float2*>(p + 2) = make_float2(v[2], v[3]);
  } else {
    for (int i = 0; i < valid; ++i) p[i] = v[i];
  }
}
template <>
__device__ __forceinline__ void bs_store4<bf16_t>(bf16_t* p, const float v[4], int align,
                                                  int valid) {
  const uint32_t lo = (uint32_t)float_to_bf16_bits(v[0]) | ((uint32_t)float_to_bf16_bits(v[1]) << 16);
  const uint32_t hi = (uint32_t)float_to_bf16_bits(v[2]) | ((uint32_t)float_to_bf16_bits(v[3]) << 16);
  if (align >= 4 && valid == 4) {
    *reinterpret_cast<uint2*>(p) = make_uint2(lo, hi);
  } else if (align >= 2 && valid == 4) {
    *reinterpret_cast<uint32_t*>(p) = lo;
    *reinterpret_cast<uint32_t*>(p + 2) = hi;
  } else {
    for (int i = 0; i < valid; ++i) p[i].v = float_to_bf16_bits(v[i]);
  }
}

template <typename TC>
__device__ __forceinline__ void bs_store2(TC* p, const float v[2], bool vec, int valid);
template <>
__device__ __forceinline__ void bs_store2<float>(float* p, const float v[2], bool vec, int valid) {
  if (vec && valid == 2) {
    *reinterpret_cast<float2*>(p) = make_float2(v[0], v[1]);
  } else {
    for (int i = 0; i < valid; ++i) p[i] = v[i];
  }
}
template <>
__device__ __forceinline__ void bs_store2<bf16_t>(bf16_t* p, const float v[2], bool vec,
                                                  int valid) {
  if (vec && valid == 2) {
    *reinterpret_cast<uint32_t*>(p) =
        (uint32_t)float_to_bf16_bits(v[0]) | ((uint32_t)float_to_bf16_bits(v[1]) << 16);
  } else {
    for (int i = 0; i < valid; ++i) p[i].v = float_to_bf16_bits(v[i]);
  }
}

// `count` (2 or 4) neighbouring columns of row m from column `col` on, into a piece-major
// [M, D] bf16 tensor; `valid` of them exist.
__device__ __forceinline__ void bs_store_pieces(uint16_t* base, int M, int m, int col, const float* v,
                                                int count, int valid) {
  auto at = [&](int c) { return base + ((int64_t)(c >> 3) * M + m) * 8 + (c & 7); };
  if (valid == count && (col & 1) == 0) {        // pairs never straddle a piece
    const uint32_t lo = (uint32_t)float_to_bf16_bits(v[0]) | ((uint32_t)float_to_bf16_bits(v[1]) << 16);
    if (count == 2) {
      *reinterpret_cast<uint32_t*>(at(col)) = lo;
      return;
    }
    const uint32_t hi = (uint32_t)float_to_bf16_bits(v[2]) | ((uint32_t)float_to_bf16_bits(v[3]) << 16);
    if ((col & 3) == 0) {
      *reinterpret_cast<uint2*>(at(col)) = make_uint2(lo, hi);
    } else {
      *reinterpret_cast<uint32_t*>(at(col)) = lo;
      *reinterpret_cast<uint32_t*>(at(col + 2)) = hi;
    }
    return;
  }
  for (int i = 0; i < valid; ++i) *at(col + i) = float_to_bf16_bits(v[i]);
}

// How a wavefront lays its lanes over the weight. An instruction of 16 x 16 outputs over 32 k has 16 columns for rows of X, of which
// a step of few rows would leave most empty. SP spreads the columns: column c is row c >> SP of X at the k chunk c & (2^SP - 1), and
// likewise tile row r is weight row r >> SP at chunk r & (2^SP - 1). Only outputs whose two chunks agree are sums of matching k; they
// lie in neighbouring lanes and are added at the end (bs_spread_sum). What it buys is the loads: an instruction's operand is
// 16 >> SP weight rows of 64 << SP bytes each, whole lines from SP = 1 on with neighbouring lanes side by side, where 16 rows are half a
// line each. Whole lines can be asked for past the caches (he_load16_once), which half lines cannot: the other half would be
// fetched twice. Alone, weights from memory: 37888 x 3584 at 1 row 49.0 -> 42.9 us (6.3 TB/s), at 8 rows 51.2 -> 41.4, 3584 x 3584 at 1 row 7.7 -> 6.7.
// SP = 0 keeps each sum in the order this product had before: a unit of 64 k is two instructions, whose lanes take the halves of 16
// neighbouring k (loaded as whole lines all the same, see he_halves_to_rows), and the K slices and, by workgroup, the turn each
// wavefront begins at are those it had. For 17 to 32 rows, whose rows of X are loaded in whole lines too (37888 x 3584 at 17, 24 and 32 rows 60.8, 67.3
// and 72.4 us with half lines of both, so 54.6, 60.5 and 67.0; half lines of X alone 56.7, 65.6 and 75.0), and where a caller asks for that order (`ordered`).
template <int SP>
struct BsLanes {
  static constexpr int RT = 16 >> SP;              // weight rows, and rows of X, of an instruction
  static constexpr int PARTS = 1 << SP;
  static constexpr int H = SP == 0 ? 2 : 1;        // instructions of a unit
  static constexpr int KM = SP == 0 ? 64 : 32 << SP;   // k of a unit
};

template <int SP>
__device__ __forceinline__ float bs_spread_sum(float v) {      // over the 2^SP neighbouring lanes, the same in each
  if (SP >= 1) v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0xB1, 0xf, 0xf, true));      // lanes 1 0 3 2
  if (SP >= 2) v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x4E, 0xf, 0xf, true));      // lanes 2 3 0 1
  return v;
}

// Registers hold the operands of two steps (the loads of the next step are issued before
// the products of this one), 8 S (NA + MT) of them (16 with SP = 0); above 4 operands a step the workgroup is
// limited to 8 wavefronts so that each may use 256 registers.
constexpr int bs_max_waves(int MT, int NA, int S) { return S * (NA + MT) <= 4 ? 16 : 8; }

template <int MT, int NA, int S, int H>
struct BsFrags {
  bf16x8 a[S][H][NA], b[S][H][MT];
};

struct BsFusion {
  const float* scale_partials;   // [M][scale_count] or null: sums of squares of the input rows
  int scale_count;
  float scale_eps;
  int scale_dim;
  float* resid;                  // [M][N] fp32 or null: residual rows, updated in place
  const void* gain;              // [N] gain of the following norm
  int gain_dtype;
  uint16_t* xg;                  // [M][N] bf16 out: resid * gain
  float* sq_out;                 // [M][gridDim.x] out: sum of resid^2 over this workgroup's columns
  int out_pieces;                // the bf16 output (C, or xg) is written piece-major
  int act_clamped;               // the gated epilogue runs he_gated_act with `act`, not SiLU(gate) * up
  GatedAct act;
  // USED: the weight's rows (used_rows a group) or k (used_k a group) come in groups, and group e < used_count is multiplied where
  // some row m has used[m used_ld + e] != 0; the others' weights are not read. Outputs of unused rows' workgroups are not written
  // (their reader takes none of them); x is zero along unused k, whose products would add zeros.
  const float* used;
  int used_ld, used_count, used_rows, used_k;
  int unary;                     // >= 0: the bf16 output is he_unary of the result rounded to bf16
  float resid_scale;             // the residual epilogue adds resid_scale * result
  const void* dyt_bias;          // with dyt_alpha: xg = tanh(alpha * resid) * gain + dyt_bias (Dynamic Tanh; both of
  const void* dyt_alpha;         // gain's dtype; alpha one stored number), and sq_out = 0: nothing is owed
};

// The residual values, gains and bias of an output item: row m, columns n .. n + valid.
__device__ __forceinline__ void bs_load_resid(const BsFusion& fu, int m, int n, int valid, int N, int align, float res[4], float gain[4]) {
  const float* p = fu.resid + (int64_t)m * N + n;
  if (valid == 4 && align >= 4) {
    const float4 r4 = *reinterpret_cast<const float4*>(p);
    res[0] = r4.x, res[1] = r4.y, res[2] = r4.z, res[3] = r4.w;
  } else if (valid == 4 && align >= 2) {
    const float2 a = *reinterpret_cast<const float2*>(p), b = *reinterpret_cast<const float2*>(p + 2);
    res[0] = a.x, res[1] = a.y, res[2] = b.x, res[3] = b.y;
  } else {
    for (int i = 0; i < 4; ++i) res[i] = i < valid ? p[i] : 0.f;
  }
  if (valid == 4 && fu.gain_dtype == HE_BF16 && (n & 1) == 0 && (((uintptr_t)fu.gain) & 3) == 0) {
    const uint32_t* g = reinterpret_cast<const uint32_t*>((const uint16_t*)fu.gain + n);
    const uint32_t a = g[0], b = g[1];
    gain[0] = __uint_as_float(a << 16), gain[1] = __uint_as_float(a & 0xffff0000u);
    gain[2] = __uint_as_float(b << 16), gain[3] = __uint_as_float(b & 0xffff0000u);
  } else {
    for (int i = 0; i < 4; ++i) gain[i] = i < valid ? load_param(fu.gain, n + i, fu.gain_dtype) : 0.f;
  }
}

// Whether some row of the step uses group e (any lane's question; M <= 16).
__device__ __forceinline__ bool bs_used(const BsFusion& fu, int M, int e) {
  if (e >= fu.used_count) return true;
  bool any = false;
#pragma unroll
  for (int m = 0; m < 16; ++m)
    if (m < M) any |= fu.used[(int64_t)m * fu.used_ld + e] != 0.f;
  return any;
}

enum BsOut { BS_PLAIN, BS_GATED, BS_RESID };

// grid: one workgroup per rows_per_block weight rows, at most RT NA; block: 64 * NW threads, each wavefront `units_per_wave`
// units' k; turn: units that are walked together (ORDERED: the turns of a wavefront begin at one that depends on its workgroup). The
// arguments that the first loads need come first.
// USED (of a routed feed-forward in a step of a few rows: the experts that nobody chose, a third of 16 at 4 rows of 4 choices): a
// workgroup of rows nobody uses leaves before it asks for weights; along K a wavefront walks the steps of the groups that are
// used in the order it walks all of them, so its sums are the same bits.
template <int SP, int MT, int NA, int S, BsOut OUT, bool PIECES, bool USED, typename TC>
__global__ __launch_bounds__(64 * bs_max_waves(MT, NA, S)) void gemm_blocksplit_kernel(
    const uint16_t* __restrict__ W, const uint16_t* __restrict__ X, int M, int N, int K, int rows_per_block, int units_per_wave,
    int turn, int bias_dtype, TC* __restrict__ C, const void* __restrict__ bias, BsFusion fu) {
  using L = BsLanes<SP>;
  constexpr bool ORDERED = SP == 0;
  constexpr bool X_LINES = ORDERED && MT == 2;  // rows of X in whole lines too, where there are enough of them
  constexpr int ROWS = L::RT * NA;              // weight rows a workgroup can hold
  constexpr int MX = L::RT * MT;                // rows of X
  extern __shared__ float4 tiles[];             // [NW][MX][ROWS] floats
  __shared__ float row_scale[MX];
  float* const red = reinterpret_cast<float*>(tiles);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nw = blockDim.x >> 6;
  const int n0 = blockIdx.x * rows_per_block;
  const int n_end = min(N, n0 + rows_per_block);
  const int lr = lane & 15, lg = lane >> 4;
  const int row = lr >> SP;                                       // of an instruction's weight rows
  // columns that a row of X takes (with SP = 0 and few rows they repeat it, so that neighbouring lanes read few rows)
  const int spread = ORDERED ? (M <= 4 ? 2 : M <= 8 ? 1 : 0) : SP;
  const int xrow = lr >> spread;
  const int units = (K + L::KM - 1) / L::KM;
  const int u0 = min(wave * units_per_wave, units), u1 = min(units, u0 + units_per_wave);
  if (USED && fu.used_rows > 0) {
    const int e0 = n0 / fu.used_rows, e1 = (n_end - 1) / fu.used_rows;
    if (e1 - e0 < 64 && __ballot(lane <= e1 - e0 && bs_used(fu, M, e0 + lane)) == 0) return;      // (the whole workgroup)
  }

  // a lane's weight rows are neighbours (row NA + a), so that the sums it ends with are neighbouring columns
  const char* const wb = reinterpret_cast<const char*>(W + (int64_t)n0 * K);
  const char* const xb = reinterpret_cast<const char*>(X);
  const int k_lane = SP == 0 ? 16 * lg : 8 * ((lg << SP) | (lr & (L::PARTS - 1)));    // this lane's first k of a unit
  uint32_t wo[L::H][NA], xo[L::H][MT];
  const bool upper = (lr & 8) != 0;
#pragma unroll
  for (int h = 0; h < L::H; ++h)
#pragma unroll
    for (int a = 0; a < NA; ++a) wo[h][a] = 2u * (uint32_t)(min((SP == 0 ? (lr & 7) + 8 * h : row) * NA + a, n_end - n0 - 1) * K);
#pragma unroll
  for (int h = 0; h < L::H; ++h)
#pragma unroll
    for (int t = 0; t < MT; ++t) xo[h][t] = 2u * (uint32_t)(min(t * L::RT + (X_LINES ? (lr & 7) + 8 * h : xrow), M - 1) * (PIECES ? 8 : K));
  const uint32_t xk = PIECES ? 2 * M : 2;                         // piece-major X: the piece of 8 k from k on lies at k M (+ 8 row)

  floatx4 acc[NA][MT];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[a][t] = floatx4{0.f, 0.f, 0.f, 0.f};

  // Steps of S units, the operands of two steps in registers: the loads of one go out together, ahead of the products of
  // the other. Of a last step that is not whole the last k are loaded again in place of what lies beyond (no branch, no second
  // trip to memory), and those products are left out, or of zeros where only some lanes lie beyond K.
  BsFrags<MT, NA, S, L::H> f0, f1;
  auto load = [&](BsFrags<MT, NA, S, L::H>& f, int u) {
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int h = 0; h < L::H; ++h) {
        const uint32_t k = min(min(u + s, u1 - 1) * L::KM + k_lane + 8 * h, K - 8);
        const uint32_t kw = SP == 0 ? min(min(u + s, u1 - 1) * L::KM + k_lane + (lr & 8), K - 8) : k;      // (see he_halves_to_rows)
#pragma unroll
        for (int a = 0; a < NA; ++a) f.a[s][h][a] = he_load16_once<bf16x8>(wb + (wo[h][a] + 2 * kw));
#pragma unroll
        for (int t = 0; t < MT; ++t) f.b[s][h][t] = bs_load8(xb + (xo[h][t] + (X_LINES ? kw : k) * xk));
      }
  };
  auto in_place = [&](BsFrags<MT, NA, S, L::H>& f, int s) {
    if constexpr (SP == 0)
#pragma unroll
      for (int a = 0; a < NA; ++a) he_halves_to_rows(f.a[s][0][a], f.a[s][1][a], upper);
    if constexpr (X_LINES)
#pragma unroll
      for (int t = 0; t < MT; ++t) he_halves_to_rows(f.b[s][0][t], f.b[s][1][t], upper);
  };
  auto multiply_unit = [&](const BsFrags<MT, NA, S, L::H>& f, int s) {
#pragma unroll
    for (int h = 0; h < L::H; ++h)
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[a][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.a[s][h][a], f.b[s][h][t], acc[a][t], 0, 0, 0);
  };
  auto multiply = [&](BsFrags<MT, NA, S, L::H>& f) {
#pragma unroll
    for (int s = 0; s < S; ++s) in_place(f, s), multiply_unit(f, s);
  };
  auto multiply_last = [&](BsFrags<MT, NA, S, L::H>& f, int u) {
    const bf16x8 zero = __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (u + s < u1) {
        in_place(f, s);
        if ((u + s + 1) * L::KM > K) {
#pragma unroll
          for (int h = 0; h < L::H; ++h) {
            const bool beyond = (u + s) * L::KM + k_lane + 8 * h >= K;
#pragma unroll
            for (int a = 0; a < NA; ++a) f.a[s][h][a] = beyond ? zero : f.a[s][h][a];
#pragma unroll
            for (int t = 0; t < MT; ++t) f.b[s][h][t] = beyond ? zero : f.b[s][h][t];
          }
        }
        multiply_unit(f, s);
      }
  };

  // The order of the units: whole turns from turn `first` on, around, then what is left. USED along K: bit t of `turns` says that
  // turn t meets a group that is used (of more than 64 turns: all do).
  const int n = u1 - u0, whole = max(min(u1, K / L::KM) - u0, 0) / turn * turn;
  const int first = ORDERED && whole > 0 ? (int)((blockIdx.x * 3u) % (unsigned)(whole / turn)) * turn : 0;
  int left = (n + S - 1) / S, j = 0;
  uint64_t turns = ~0ull;
  auto unit = [&](int j) { return u0 + (!ORDERED || j >= whole ? j : j + first < whole ? j + first : j + first - whole); };
  auto skip = [&]() {
    if (USED)
      while (j < whole && ((turns >> (((unit(j) - u0) / turn) & 63)) & 1) == 0) j += turn;
  };
  if (USED && fu.used_k > 0 && whole > 0 && whole <= 64 * turn) {
    const int at = (u0 + min(lane * turn, whole - turn)) * L::KM, e0 = at / fu.used_k, e1 = min(at + turn * L::KM - 1, K - 1) / fu.used_k;
    bool any = bs_used(fu, M, e0);
    if (e1 != e0) any = any || bs_used(fu, M, e1);      // (groups are no shorter than a turn)
    turns = __ballot(any && lane * turn < whole);
    left = __popcll(turns) * (turn / S) + (n - whole + S - 1) / S;
    skip();
  }
  int u = unit(j);
  auto next = [&]() {
    j += S;
    if (USED && turns != ~0ull && j < whole && j % turn == 0) skip();
    return u = unit(j);
  };
  if (left > 0) load(f0, u);
  __builtin_amdgcn_sched_barrier(0);

  // Loads the epilogue needs go out behind the first weights, so that their latency is not added at the end: the partial sums of
  // squares of the input rows (wavefront w takes the rows w, w + nw, ...; lanes hold strided partials), and the residual
  // values, gains and bias of this thread's first outputs.
  const bool scaled = fu.scale_partials != nullptr;
  constexpr int SCALE_ROWS = (MX + 3) / 4;      // rows a wavefront takes: all of them with 4 wavefronts
  constexpr int SCALE_LOADS = SCALE_ROWS <= 2 ? 8 : 4;
  const bool scale_early = scaled && fu.scale_count <= 64 * SCALE_LOADS && M <= SCALE_ROWS * nw;
  float pv[SCALE_ROWS][SCALE_LOADS];
  if (scale_early) {
#pragma unroll
    for (int j = 0; j < SCALE_ROWS; ++j) {
      const float* p = fu.scale_partials + (int64_t)min(wave + j * nw, M - 1) * fu.scale_count;
#pragma unroll
      for (int q = 0; q < SCALE_LOADS; ++q) pv[j][q] = p[min(lane + 64 * q, fu.scale_count - 1)];
    }
  }
  constexpr int G = ROWS / 4;                   // items of four columns a row
  const int items = M * G;
  const int out_align = ((N | n0) & 3) == 0 ? 4 : (((N | n0) & 1) == 0 ? 2 : 1);
  float res0[4] = {0.f, 0.f, 0.f, 0.f}, gain0[4] = {0.f, 0.f, 0.f, 0.f}, bias0[4] = {0.f, 0.f, 0.f, 0.f};
  auto ahead = [&](int item) {
    const int m = item / G, at = n0 + 4 * (item % G), valid = max(0, min(4, n_end - at));
    if (OUT == BS_RESID) bs_load_resid(fu, m, at, valid, N, out_align, res0, gain0);
    if (OUT != BS_GATED && bias != nullptr)
#pragma unroll
      for (int i = 0; i < 4; ++i) bias0[i] = load_param(bias, min(at + i, N - 1), bias_dtype);
  };
  if (OUT != BS_GATED && (int)threadIdx.x < items) ahead(threadIdx.x);
  __builtin_amdgcn_sched_barrier(0);

  if (left > 0) {
    for (; left > 2; left -= 2) {
      load(f1, next());
      __builtin_amdgcn_sched_barrier(0);   // the loads of a step go out together, ahead of the products
      multiply(f0);
      __builtin_amdgcn_sched_barrier(0);
      load(f0, next());
      __builtin_amdgcn_sched_barrier(0);
      multiply(f1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (left == 2) {
      load(f1, next());
      __builtin_amdgcn_sched_barrier(0);
      multiply(f0);
      multiply_last(f1, u);
    } else {
      multiply_last(f0, u);
    }
  }

  if (scaled) {
    if (scale_early) {
#pragma unroll
      for (int j = 0; j < SCALE_ROWS; ++j) {
        float part = 0.f;
#pragma unroll
        for (int q = 0; q < SCALE_LOADS; ++q) part += lane + 64 * q < fu.scale_count ? pv[j][q] : 0.f;
        const float total = wave_sum(part);
        if (lane == 0 && wave + j * nw < M) row_scale[wave + j * nw] = 1.0f / sqrtf(total / (float)fu.scale_dim + fu.scale_eps);
      }
    } else {
      for (int m = wave; m < M; m += nw) {
        float part = 0.f;
        for (int i = lane; i < fu.scale_count; i += 64) part += fu.scale_partials[(int64_t)m * fu.scale_count + i];
        const float total = wave_sum(part);
        if (lane == 0) row_scale[m] = 1.0f / sqrtf(total / (float)fu.scale_dim + fu.scale_eps);
      }
    }
  }

  // every wavefront leaves its sums: tile row 4 lg + i of an instruction is weight row (4 lg + i) >> SP at chunk (4 lg + i) % 2^SP
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = t * L::RT + xrow, part = lr & ((1 << spread) - 1);
    constexpr int J = 4 >> SP;
    float v[J * NA];
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        float x = acc[a][t][j * L::PARTS];
#pragma unroll
        for (int i = 1; i < L::PARTS; ++i) x = part == i ? acc[a][t][j * L::PARTS + i] : x;
        v[j * NA + a] = bs_spread_sum<SP>(x);
      }
    if (part == 0 && m < M) {
      float* at = red + (wave * MX + m) * ROWS + lg * J * NA;
      if constexpr (J * NA % 4 == 0) {
#pragma unroll
        for (int i = 0; i < J * NA; i += 4) *reinterpret_cast<float4*>(at + i) = make_float4(v[i], v[i + 1], v[i + 2], v[i + 3]);
      } else {
#pragma unroll
        for (int i = 0; i < J * NA; ++i) at[i] = v[i];
      }
    }
  }
  __syncthreads();

  // a thread adds four neighbouring columns of a row over the wavefronts in their order and writes them
  for (int item = threadIdx.x; item < items; item += blockDim.x) {
    const int m = item / G, n = n0 + 4 * (item % G);
    const int valid = max(0, min(4, n_end - n));
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int w = 0; w < nw; ++w) {
      const float4 v = *reinterpret_cast<const float4*>(red + (w * MX + m) * ROWS + 4 * (item % G));
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    float v[4] = {s.x, s.y, s.z, s.w};
    const float rs = scaled ? row_scale[m] : 1.f;
    if (OUT == BS_GATED) {
      // the thread's four weight rows are two (gate, up) pairs: two outputs
      const int NO = N >> 1, pairs = valid >> 1;
      if (pairs <= 0) continue;
      float y[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float g = v[2 * i] * rs;
        y[i] = fu.act_clamped ? he_gated_act<true>(g, v[2 * i + 1] * rs, fu.act)
                              : g / (1.f + expf(-g)) * (v[2 * i + 1] * rs);
      }
      if (fu.out_pieces)
        bs_store_pieces(reinterpret_cast<uint16_t*>(C), M, m, n >> 1, y, 2, pairs);
      else
        bs_store2<TC>(C + (int64_t)m * NO + (n >> 1), y, ((NO | (n0 >> 1)) & 1) == 0, pairs);
    } else {
      if (item != (int)threadIdx.x) ahead(item);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = v[i] * rs + bias0[i];
      if (OUT == BS_PLAIN) {
        if (fu.unary >= 0)
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = he_unary(bf16_bits_to_float(float_to_bf16_bits(v[i])), fu.unary);
        if (valid > 0) {
          if (fu.out_pieces)
            bs_store_pieces(reinterpret_cast<uint16_t*>(C), M, m, n, v, 4, valid);
          else
            bs_store4<TC>(C + (int64_t)m * N + n, v, out_align, valid);
        }
        continue;
      }
      const bool dyt = fu.dyt_alpha != nullptr;
      const float dyt_a = dyt ? load_param(fu.dyt_alpha, 0, fu.gain_dtype) : 0.f;
      float sq = 0.f, x[4], xgv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = res0[i] + fu.resid_scale * v[i];
        xgv[i] = he_carried_norm(x[i], gain0[i], fu.dyt_bias, min(n + i, N - 1), fu.gain_dtype, dyt, dyt_a);
        if (i < valid && !dyt) sq += x[i] * x[i];
      }
      if (valid > 0) {
        const int64_t at = (int64_t)m * N + n;
        bs_store4<float>(fu.resid + at, x, out_align, valid);
        if (fu.out_pieces)
          bs_store_pieces(fu.xg, M, m, n, xgv, 4, valid);
        else
          bs_store4<bf16_t>(reinterpret_cast<bf16_t*>(fu.xg) + at, xgv, out_align, valid);
      }
      // a row's items are neighbouring lanes (G of them, a power of two)
#pragma unroll
      for (int step = 1; step < G; step <<= 1) sq += __shfl_xor(sq, step, HE_WAVE);
      if (item % G == 0) fu.sq_out[(int64_t)m * gridDim.x + blockIdx.x] = sq;
    }
  }
}

struct BlockSplitPlan {
  int SP, MT, NA, S, NW, units;      // units: of a wavefront
  int turn;                          // units walked together, a multiple of S
  int rows_per_block;                // weight rows of a workgroup, at most (16 >> SP) NA
};

template <int SP, int MT, int NA, int S, BsOut OUT, bool USED, typename TC>
static inline void launch_blocksplit(const BlockSplitPlan& p, void* C, const void* X, const void* W,
                              const void* bias, int bias_dtype, int M, int N, int K,
                              const BsFusion& fu, bool x_pieces, hipStream_t s) {
  const int blocks = (N + p.rows_per_block - 1) / p.rows_per_block;
  const size_t lds = (size_t)p.NW * BsLanes<SP>::RT * MT * BsLanes<SP>::RT * NA * sizeof(float);
  if constexpr (SP > 0 || MT == 1) {   // piece-major activations are for up to 16 rows
    if (x_pieces) {
      gemm_blocksplit_kernel<SP, MT, NA, S, OUT, true, USED, TC><<<blocks, 64 * p.NW, lds, s>>>(
          (const uint16_t*)W, (const uint16_t*)X, M, N, K, p.rows_per_block, p.units, p.turn, bias_dtype, (TC*)C, bias, fu);
      return;
    }
  }
  gemm_blocksplit_kernel<SP, MT, NA, S, OUT, false, USED, TC><<<blocks, 64 * p.NW, lds, s>>>(
      (const uint16_t*)W, (const uint16_t*)X, M, N, K, p.rows_per_block, p.units, p.turn, bias_dtype, (TC*)C, bias, fu);
}

// Every tiling with one epilogue and output type: a function per file of
// gemm_blocksplit_tiles_*.hip. Returns 0 after a launch, -1 with the error set when the plan
// names no tiling.
#define HE_BS_DISPATCH_ARGS                                                                         \
  const BlockSplitPlan &p, void *C, const void *X, const void *W, const void *bias, int bias_dtype, \
      int M, int N, int K, const BsFusion &fu, bool x_pieces, hipStream_t s
int he_blocksplit_tiles_bf16(HE_BS_DISPATCH_ARGS);
int he_blocksplit_tiles_resid(HE_BS_DISPATCH_ARGS);
int he_blocksplit_tiles_f32(HE_BS_DISPATCH_ARGS);
int he_blocksplit_tiles_gated_bf16(HE_BS_DISPATCH_ARGS);
int he_blocksplit_tiles_gated_f32(HE_BS_DISPATCH_ARGS);
int he_blocksplit_tiles_used_bf16(HE_BS_DISPATCH_ARGS);
int he_blocksplit_tiles_used_resid(HE_BS_DISPATCH_ARGS);      // (up to 16 rows)

#define HE_BS_TILING(SP_, MT_, NA_, S_, OUT_, USED_, TC_)                                         \
  if (p.SP == SP_ && p.MT == MT_ && p.NA == NA_ && p.S == S_) {                                     \
    launch_blocksplit<SP_, MT_, NA_, S_, OUT_, USED_, TC_>(p, C, X, W, bias, bias_dtype, M, N, K, fu, x_pieces, s); \
    return 0;                                                                                       \
  }
#define HE_BS_SIXTEEN_ROWS(OUT_, USED_, TC_)                                                      \
  HE_BS_TILING(2, 1, 1, 1, OUT_, USED_, TC_) HE_BS_TILING(2, 1, 1, 2, OUT_, USED_, TC_)         \
  HE_BS_TILING(2, 1, 2, 1, OUT_, USED_, TC_) HE_BS_TILING(2, 1, 2, 2, OUT_, USED_, TC_)         \
  HE_BS_TILING(2, 1, 4, 1, OUT_, USED_, TC_) HE_BS_TILING(2, 1, 4, 2, OUT_, USED_, TC_)         \
  HE_BS_TILING(1, 1, 1, 1, OUT_, USED_, TC_) HE_BS_TILING(1, 1, 1, 2, OUT_, USED_, TC_)         \
  HE_BS_TILING(1, 1, 2, 1, OUT_, USED_, TC_) HE_BS_TILING(1, 1, 2, 2, OUT_, USED_, TC_)         \
  HE_BS_TILING(1, 1, 4, 1, OUT_, USED_, TC_) HE_BS_TILING(1, 1, 4, 2, OUT_, USED_, TC_)         \
  HE_BS_TILING(1, 2, 1, 1, OUT_, USED_, TC_) HE_BS_TILING(1, 2, 1, 2, OUT_, USED_, TC_)         \
  HE_BS_TILING(1, 2, 2, 1, OUT_, USED_, TC_) HE_BS_TILING(1, 2, 2, 2, OUT_, USED_, TC_)         \
  HE_BS_TILING(1, 2, 4, 1, OUT_, USED_, TC_) HE_BS_TILING(1, 2, 4, 2, OUT_, USED_, TC_)
// (what ordered_plan gives; no residual epilogue goes with it)
#define HE_BS_ORDERED(OUT_, USED_, TC_)                                                           \
  HE_BS_TILING(0, 1, 1, 2, OUT_, USED_, TC_)                                                      \
  HE_BS_TILING(0, 1, 2, 1, OUT_, USED_, TC_) HE_BS_TILING(0, 1, 2, 2, OUT_, USED_, TC_)         \
  HE_BS_TILING(0, 1, 4, 1, OUT_, USED_, TC_) HE_BS_TILING(0, 1, 4, 2, OUT_, USED_, TC_)
#define HE_BS_THIRTY_TWO_ROWS(OUT_, TC_)                                                          \
  HE_BS_TILING(0, 2, 1, 1, OUT_, false, TC_) HE_BS_TILING(0, 2, 1, 2, OUT_, false, TC_)         \
  HE_BS_TILING(0, 2, 2, 1, OUT_, false, TC_) HE_BS_TILING(0, 2, 2, 2, OUT_, false, TC_)
#define HE_BS_NO_TILING                                                                           \
  he_set_error("he_gemm_blocksplit_bf16: no kernel for SP=%d MT=%d NA=%d S=%d", p.SP, p.MT, p.NA, p.S); \
  return -1
