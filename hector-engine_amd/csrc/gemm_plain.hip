// Plain matrix product  C[M,N] = A[M,K] * W[N,K]^T (+ bias[N])  with fp32 FMA accumulation
// in one fixed order per output element, whatever M and whichever rows share the launch, so
// a row's result never depends on the batch it is in or on how the step was cut. It is the
// true 32-bit path of every linear layer and the reference beside the MFMA kernels.
// Weight layout [N, K] row-major as in the reference (kernels/register_kernels.cpp:373-386).
//
// The order: K is cut into segments of GP_SEG (128) consecutive k. The sum of a segment is one
// chain of FMAs over its k in ascending order, begun at zero; the element is the segment
// sums added one after the other in segment order, begun at zero; then the bias.
// These kernels keep this order and give the same bits:
//   mfma    fp32 operands, many rows: tiles of up to 128 x 128 outputs on the matrix cores;
//   rounds  the same for aligned rows and K in 32s (gemm_plain_rounds.hip): tiles that are whole rounds of the chip;
//   stream  fp32 operands, up to 64 rows, K in whole segments: matrix cores, a workgroup per 16 weight rows;
//   tiles   bf16 operands: 64 x 64 outputs a workgroup, staged through LDS, every thread 4 x 4 outputs;
//   rows    up to GP_ROWS_MAX_M rows that stream does not take (gp_streams), with a workspace: a thread owns one weight
//           row and one segment and walks it with all M activation rows at once, so a product
//           has N * ceil(K / GP_SEG) threads however few its rows are; the segment sums go
//           to a workspace and a second kernel adds them in order.
// No multiply and add of this file is fused unless it is written as an fma: the same lines are
// compiled into several kernels that must give the same bits.
#pragma clang fp contract(off)
#include "common.h"
#include "hector_kernels.h"

#define GP_BM 64
#define GP_BN 64
#define GP_BK 16
#define GP_SEG 128          // a multiple of GP_BK
#define GP_ROWS_MAX_M 8

template <typename TA, typename TW, typename TC>
// (six wavefronts a SIMD, as without the segment totals: left alone the compiler takes registers for four)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6, 8))) void gemm_plain_kernel(
    TC* __restrict__ C, const TA* __restrict__ A, const TW* __restrict__ W,
    const void* __restrict__ bias, int bias_dtype, int M, int N, int K, int64_t lda, int64_t ldw,
    int64_t ldc) {
  __shared__ float As[GP_BK][GP_BM + 1];
  __shared__ float Ws[GP_BK][GP_BN + 1];
  const int tid = threadIdx.x;
  const int tx = tid & 15;  // along N
  const int ty = tid >> 4;  // along M
  const int m0 = blockIdx.y * GP_BM;
  const int n0 = blockIdx.x * GP_BN;
  const int lrow = tid >> 2;       // 0..63
  const int lk = (tid & 3) * 4;    // 0,4,8,12
  float acc[4][4], total[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f, total[i][j] = 0.f;

  for (int k0 = 0; k0 < K; k0 += GP_BK) {
    const int am = m0 + lrow, wn = n0 + lrow;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + lk + j;
      As[lk + j][lrow] = (am < M && k < K) ? to_float(A[am * lda + k]) : 0.f;
      Ws[lk + j][lrow] = (wn < N && k < K) ? to_float(W[wn * ldw + k]) : 0.f;
    }
    __syncthreads();
    // the chain of a segment holds its own k only: the last tile of K may be short
#define GP_TILE_STEP(kk)                                                     \
  {                                                                          \
    float a[4], b[4];                                                        \
    _Pragma("unroll") for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i]; \
    _Pragma("unroll") for (int j = 0; j < 4; ++j) b[j] = Ws[kk][tx * 4 + j]; \
    _Pragma("unroll") for (int i = 0; i < 4; ++i)                            \
        _Pragma("unroll") for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]); \
  }
    if (k0 + GP_BK <= K) {
#pragma unroll
      for (int kk = 0; kk < GP_BK; ++kk) GP_TILE_STEP(kk)
    } else {
      for (int kk = 0; kk < K - k0; ++kk) GP_TILE_STEP(kk)
    }
#undef GP_TILE_STEP
    __syncthreads();
    if ((k0 + GP_BK) % GP_SEG == 0 || k0 + GP_BK >= K) {   // the segment ends here
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) total[i][j] += acc[i][j], acc[i][j] = 0.f;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      float v = total[i][j];
      if (bias != nullptr) v += load_param(bias, n, bias_dtype);
      C[m * ldc + n] = from_float<TC>(v);
    }
  }
}

// The 32-bit product of more than GP_MROWS_MAX_M rows on the matrix cores, in the same order: a chain of
// v_mfma_f32_32x32x2_f32 on one accumulator gives bit for bit the chain of FMAs over ascending k (measured
// over normal, tiny, denormal, huge and non-finite operands), so a segment is 64 instructions begun at zero and
// the segment sums are added as everywhere. A lane's operand for four instructions is one 16-byte LDS read: a row's
// even k of a stage lie before its odd k (lanes 0..31 feed the even k of an instruction, lanes 32..63 the odd
// one). Four wavefronts, two by two, each with BM/2 x BN/2 outputs; a stage of 32 k in LDS while the next one is on
// its way in registers, one barrier a stage. Bound by the matrix cores (the loop reaches 139 TFLOP/s without
// memory): the gate||up of the 7B shape (37888 x 3584) at 1003 rows takes 2.42 ms (112 TFLOP/s), its down projection
// 1.38 ms; tiles on the vector ALU, which has half as many products a clock, took 4.80 and 5.20 ms. Columns of tiles go to an XCD in stretches: the row tiles that read one stretch of
// weights run behind one L2.
typedef float gp_f32x16 __attribute__((ext_vector_type(16)));
typedef float gp_f32x4 __attribute__((ext_vector_type(4)));
#define GPM_BK 32
#define GPM_LD 36           // floats a row of a stage: 16 even k, 16 odd k, 4 of padding (reads without bank conflicts)
template <int BM, int BN>
__global__ __launch_bounds__(256, 2) void gemm_plain_mfma_kernel(
    float* __restrict__ C, const float* __restrict__ A, const float* __restrict__ W,
    const void* __restrict__ bias, int bias_dtype, int M, int N, int K, int64_t lda, int64_t ldw,
    int64_t ldc, int mtiles, int ntiles, int vec) {
  constexpr int TM = BM / 64, TN = BN / 64;      // 32 x 32 tiles of a wavefront
  constexpr int LA = BM / 32, LW = BN / 32;      // 16-byte loads of a thread and stage
  __shared__ __attribute__((aligned(16))) float stage[2][(BM + BN) * GPM_LD];
  const int per_xcd = (mtiles * ntiles + HE_XCDS - 1) / HE_XCDS;
  const int tile = (blockIdx.x % HE_XCDS) * per_xcd + blockIdx.x / HE_XCDS;
  if (tile >= mtiles * ntiles) return;           // (the whole workgroup)
  const int m0 = (tile % mtiles) * BM, n0 = (tile / mtiles) * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r32 = lane & 31, half = lane >> 5;
  const int lrow = tid >> 3, lk = (tid & 7) * 4;
  // rows beyond the matrices are the last row again: their outputs are not stored
  const float* asrc[LA];
  const float* wsrc[LW];
#pragma unroll
  for (int i = 0; i < LA; ++i) asrc[i] = A + (int64_t)min(m0 + lrow + 32 * i, M - 1) * lda;
#pragma unroll
  for (int i = 0; i < LW; ++i) wsrc[i] = W + (int64_t)min(n0 + lrow + 32 * i, N - 1) * ldw;
  gp_f32x4 av[LA], wv[LW];
  auto fetch = [&](int k0) {
    if (vec && k0 + GPM_BK <= K) {
#pragma unroll
      for (int i = 0; i < LA; ++i) av[i] = *reinterpret_cast<const gp_f32x4*>(asrc[i] + k0 + lk);
#pragma unroll
      for (int i = 0; i < LW; ++i) wv[i] = *reinterpret_cast<const gp_f32x4*>(wsrc[i] + k0 + lk);
    } else {      // K's end, or rows that are not 16-byte aligned: zeros beyond K leave a chain as it is
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = k0 + lk + e;
#pragma unroll
        for (int i = 0; i < LA; ++i) av[i][e] = k < K ? asrc[i][k] : 0.f;
#pragma unroll
        for (int i = 0; i < LW; ++i) wv[i][e] = k < K ? wsrc[i][k] : 0.f;
      }
    }
  };
  auto put = [&](float* to) {
#pragma unroll
    for (int i = 0; i < LA + LW; ++i) {
      const gp_f32x4 v = i < LA ? av[i < LA ? i : 0] : wv[i < LA ? 0 : i - LA];
      float* row = to + (lrow + 32 * i) * GPM_LD + lk / 2;
      *reinterpret_cast<float2*>(row) = make_float2(v[0], v[2]);
      *reinterpret_cast<float2*>(row + 16) = make_float2(v[1], v[3]);
    }
  };
  gp_f32x16 acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f, total[i][j][e] = 0.f;
  const int arow = ((wave >> 1) * (BM / 2) + r32) * GPM_LD + half * 16;
  const int wrow = (BM + (wave & 1) * (BN / 2) + r32) * GPM_LD + half * 16;
  fetch(0);
  put(stage[0]);
  __syncthreads();
  int cur = 0;
  for (int k0 = 0; k0 < K; k0 += GPM_BK, cur ^= 1) {
    const bool more = k0 + GPM_BK < K;
    if (more) fetch(k0 + GPM_BK);
    const float* at = stage[cur];
#pragma unroll
    for (int j = 0; j < 4; ++j) {                // eight k
      gp_f32x4 a[TM], b[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) a[i] = *reinterpret_cast<const gp_f32x4*>(at + arow + i * 32 * GPM_LD + 4 * j);
#pragma unroll
      for (int i = 0; i < TN; ++i) b[i] = *reinterpret_cast<const gp_f32x4*>(at + wrow + i * 32 * GPM_LD + 4 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int x = 0; x < TM; ++x)
#pragma unroll
          for (int y = 0; y < TN; ++y)
            acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[x][e], b[y][e], acc[x][y], 0, 0, 0);
    }
    if ((k0 + GPM_BK) % GP_SEG == 0 || !more) {  // the segment ends here
#pragma unroll
      for (int x = 0; x < TM; ++x)
#pragma unroll
        for (int y = 0; y < TN; ++y)
#pragma unroll
          for (int e = 0; e < 16; ++e) total[x][y][e] += acc[x][y][e], acc[x][y][e] = 0.f;
    }
    if (more) put(stage[cur ^ 1]);
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < TM; ++x)
#pragma unroll
    for (int y = 0; y < TN; ++y) {
      const int n = n0 + (wave & 1) * (BN / 2) + 32 * y + r32;
      const float b = bias != nullptr && n < N ? load_param(bias, n, bias_dtype) : 0.f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + (wave >> 1) * (BM / 2) + 32 * x + (e >> 2) * 8 + half * 4 + (e & 3);
        if (m < M && n < N) C[m * ldc + n] = bias != nullptr ? total[x][y][e] + b : total[x][y][e];
      }
    }
}

// The 32-bit product of up to GP_MROWS_MAX_M rows in the same order, bound by the weights' way from memory. A
// workgroup owns 16 weight rows and all activation rows (MT tiles of 16) and walks K with NW wavefronts, each
// a segment of its own at a time: v_mfma_f32_16x16x4_f32 chains, whose sums go to LDS; after FLUSH rounds of
// segments the workgroup adds them to its totals in segment order. So a weight of 3,584 rows still has 224 workgroups
// with 16 wavefronts' loads in flight, and nothing goes through a workspace. (7B gate||up, 543 MB: 1 row 88 us, 4 rows 86,
// 16 rows 101, 64 rows 288; a lane a weight row on the vector ALU and a second kernel for the segment sums, up to 8
// rows, 104 and 114; 64 x 64 tiles, which more rows went through, 657 at 16 rows and, for the down projection's 3,584
// weight rows of 18,944, 2479 where this takes 53.) A wavefront fetches a stage of KS k
// of its 16 weight rows (and activation rows) whole lines at a time, two stages ahead, into its own LDS region, the
// 16-byte pieces of row r at their index xor r, from which the operand of lane (row, k mod 4) is read a float at a
// time without bank conflicts; up to 64 rows the weights past the caches (ONCE: he_load16_once; at 4 rows the 543 MB 95 -> 86 us; more rows are two
// workgroups' of the same weights, 2048 x 8192 at 65 rows 61.9 and 62.6 so). For weights of whole segments in aligned rows.
#define GP_MROWS_MAX_M 64
template <int MT, int NW, int KS, bool ONCE>
__global__ __launch_bounds__(NW * 64) void gemm_plain_stream_kernel(
    float* __restrict__ C, const float* __restrict__ A, const float* __restrict__ W, const void* __restrict__ bias,
    int bias_dtype, int M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc) {
  constexpr int FLUSH = NW * MT < 16 ? 16 / (NW * MT) : 1;   // rounds whose segment sums LDS holds
  constexpr int P = KS / 4;                      // 16-byte pieces of a row and stage
  constexpr int LD = KS / 16;                    // loads of a lane for 16 rows of a stage
  constexpr int SPS = GP_SEG / KS;               // stages of a segment
  __shared__ gp_f32x4 tiles[NW][(1 + MT) * 16 * P];
  __shared__ float sums[FLUSH * NW][MT * 256];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * 16;
  const int segments = K / GP_SEG;
  A += (int64_t)blockIdx.y * (16 * MT) * lda;    // (more activation rows than a workgroup takes: the next ones along y)
  C += (int64_t)blockIdx.y * (16 * MT) * ldc;
  M -= blockIdx.y * (16 * MT);
  // load t of a stage: row t * (64 / P) + lane / P of the 16, piece lane % P
  const int lrow = lane / P, piece = lane % P;
  const float* wsrc[LD];
  const float* asrc[MT][LD];
  bool real[MT][LD];
#pragma unroll
  for (int t = 0; t < LD; ++t) {
    const int r = t * (64 / P) + lrow;
    wsrc[t] = W + (int64_t)min(n0 + r, N - 1) * ldw + 4 * piece;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      real[i][t] = 16 * i + r < M;               // (rows beyond M stay zero: nothing is fetched for them)
      asrc[i][t] = A + (int64_t)min(16 * i + r, M - 1) * lda + 4 * piece;
    }
  }
  gp_f32x4* mine = tiles[wave];
  const int rounds = (segments + NW - 1) / NW;
  const int stages = rounds * SPS;               // of every wavefront; a stage of no segment does nothing
  gp_f32x4 wv[2][LD], av[2][MT][LD];
  const gp_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < LD; ++t) av[b][i][t] = zero;
#define GPS_FETCH(B_, ST_)                                                                           \
  {                                                                                                  \
    const int seg_ = wave + NW * ((ST_) / SPS);                                                      \
    if (seg_ < segments) {                                                                           \
      const int64_t k_ = (int64_t)seg_ * GP_SEG + ((ST_) % SPS) * KS;                                \
      _Pragma("unroll") for (int t = 0; t < LD; ++t) wv[B_][t] =                          \
          ONCE ? he_load16_once<gp_f32x4>(wsrc[t] + k_) : *reinterpret_cast<const gp_f32x4*>(wsrc[t] + k_); \
      _Pragma("unroll") for (int i = 0; i < MT; ++i)                                                 \
        _Pragma("unroll") for (int t = 0; t < LD; ++t)                                               \
          if (real[i][t]) av[B_][i][t] = *reinterpret_cast<const gp_f32x4*>(asrc[i][t] + k_);        \
    }                                                                                                \
  }
  gp_f32x4 acc[MT];
  float total[MT * 256 / (NW * 64) > 0 ? MT * 256 / (NW * 64) : 1];
  constexpr int OWN = sizeof(total) / sizeof(float);   // outputs a thread adds up (threads beyond MT * 256: none)
#pragma unroll
  for (int i = 0; i < OWN; ++i) total[i] = 0.f;
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = zero;
  const int r16 = lane & 15, h = lane >> 4;
#define GPS_STAGE(B_, ST_)                                                                           \
  {                                                                                                  \
    const int seg_ = wave + NW * ((ST_) / SPS);                                                      \
    if (seg_ < segments) {                                                                           \
      _Pragma("unroll") for (int t = 0; t < LD; ++t) {                                               \
        const int r = t * (64 / P) + lrow;                                                           \
        mine[r * P + (piece ^ (r % P))] = wv[B_][t];                                                 \
        _Pragma("unroll") for (int i = 0; i < MT; ++i)                                               \
          mine[(16 * (1 + i) + r) * P + (piece ^ (r % P))] = av[B_][i][t];                           \
      }                                                                                              \
      __builtin_amdgcn_wave_barrier();                                                               \
    }                                                                                                \
    GPS_FETCH(B_, (ST_) + 2)                                                                         \
    if (seg_ < segments) {                                                                           \
      const float* f = reinterpret_cast<const float*>(mine) + r16 * KS + h;                          \
      _Pragma("unroll") for (int j = 0; j < P; ++j) {                                                \
        const int o = 4 * (j ^ (r16 % P));                                                           \
        const float w = f[o];                                                                        \
        _Pragma("unroll") for (int i = 0; i < MT; ++i)                                               \
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[16 * (1 + i) * KS + o], w, acc[i], 0, 0, 0); \
      }                                                                                              \
      __builtin_amdgcn_wave_barrier();                                                               \
      if ((ST_) % SPS == SPS - 1) {                                                                  \
        float* to = sums[((ST_) / SPS % FLUSH) * NW + wave];                                         \
        _Pragma("unroll") for (int i = 0; i < MT; ++i) {                                             \
          _Pragma("unroll") for (int e = 0; e < 4; ++e) to[i * 256 + (4 * h + e) * 16 + r16] = acc[i][e]; \
          acc[i] = zero;                                                                             \
        }                                                                                            \
      }                                                                                              \
    }                                                                                                \
  }
  GPS_FETCH(0, 0)
  GPS_FETCH(1, 1)
  for (int st = 0; st < stages; st += 2) {       // (SPS is even)
    GPS_STAGE(0, st)
    GPS_STAGE(1, st + 1)
    const int round = (st + 2) / SPS;            // rounds done, where a round ends here
    if ((st + 2) % SPS == 0 && (round % FLUSH == 0 || round == rounds)) {
      __syncthreads();
      const int first = (round - 1) / FLUSH * FLUSH * NW, count = min(segments - first, FLUSH * NW);
#pragma unroll
      for (int i = 0; i < OWN; ++i) {
        const int o = tid + i * NW * 64;
        if (o < MT * 256)
          for (int s = 0; s < count; ++s) total[i] += sums[s][o];
      }
      __syncthreads();
    }
  }
#undef GPS_FETCH
#undef GPS_STAGE
#pragma unroll
  for (int i = 0; i < OWN; ++i) {
    const int o = tid + i * NW * 64, m = o >> 4, n = n0 + (o & 15);
    if (o >= MT * 256 || m >= M || n >= N) continue;
    C[m * ldc + n] = bias != nullptr ? total[i] + load_param(bias, n, bias_dtype) : total[i];
  }
}

// The sums of one segment for one weight row and MT activation rows. grid (ceil(N / 64),
// ceil(segments / 4)), block (64, 4): the lanes of a wavefront hold 64 neighbouring weight rows,
// its four wavefronts four segments. The activation values are the same for all lanes.
template <int MT, typename TA, typename TW>
__global__ __launch_bounds__(256) void gemm_plain_rows_kernel(
    float* __restrict__ partial, const TA* __restrict__ A, const TW* __restrict__ W, int M, int N, int K,
    int64_t lda, int64_t ldw, int segments) {
  const int n = blockIdx.x * 64 + threadIdx.x;
  const int seg = __builtin_amdgcn_readfirstlane(blockIdx.y * 4 + threadIdx.y);
  if (seg >= segments) return;
  const int k_begin = seg * GP_SEG, k_end = min(K, k_begin + GP_SEG);
  const TW* wrow = W + (int64_t)min(n, N - 1) * ldw;
  float acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = 0.f;
  const TA* arow[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) arow[m] = A + (int64_t)min(m, M - 1) * lda;
  int k = k_begin;
  const bool vec = sizeof(TW) == 4 && (ldw & 3) == 0 && (((uintptr_t)W) & 15) == 0;
  if (vec) {
    // 64 k of the row at a time: sixteen loads of 16 bytes on their way before the first product
    constexpr int UN = 16;
    for (; k + 4 * UN <= k_end; k += 4 * UN) {
      float4 wv[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) wv[u] = *reinterpret_cast<const float4*>(wrow + k + 4 * u);
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const float w[4] = {wv[u].x, wv[u].y, wv[u].z, wv[u].w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m] = fmaf(to_float(arow[m][k + 4 * u + e]), w[e], acc[m]);
      }
    }
    for (; k + 4 <= k_end; k += 4) {
      const float4 w4 = *reinterpret_cast<const float4*>(wrow + k);
      const float w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m] = fmaf(to_float(arow[m][k + e]), w[e], acc[m]);
    }
  }
  for (; k < k_end; ++k) {
    const float w = to_float(wrow[k]);
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = fmaf(to_float(arow[m][k]), w, acc[m]);
  }
  if (n < N) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m < M) partial[((int64_t)seg * M + m) * N + n] = acc[m];
  }
}

// The same sums for 32-bit weights whose K is whole segments, with the weights fetched line by
// line: in the kernel above the 64 lanes of a load touch 64 cache lines (each lane its own row), and
// the rate at which a compute unit looks lines up bounds it (3.6 TB/s at the Qwen2.5-7B shape). Here
// eight neighbouring lanes fetch the 128 bytes of one row, a load touches eight lines, and the
// wavefront turns the tile round in LDS: 32 k of its 64 rows at a time (two such chunks on their
// way while one is multiplied), the values go into the wavefront's own LDS region as
// [16-byte piece][row, 65 to a piece][4], from which lane n reads the pieces of row n one after the
// other (a read of 64 lanes is one KiB on end) and extends its chain of FMAs in ascending k. The
// region is the wavefront's own: LDS runs a wavefront's writes and reads in program order, so no
// barrier is needed, and the compiler keeps stores and loads that may name the same address in
// order. (A wavefront-scope fence here kept the staging registers in scratch memory.) grid and
// block as above.
#define GP_TURN_ROWS 65
template <int MT>
__global__ __launch_bounds__(256) void gemm_plain_rows_turned_kernel(
    float* __restrict__ partial, const float* __restrict__ A, const float* __restrict__ W, int M, int N, int K,
    int64_t lda, int64_t ldw, int segments) {
  __shared__ float4 turned[4][8 * GP_TURN_ROWS];
  const int lane = threadIdx.x;
  const int n0 = blockIdx.x * 64;
  const int seg = __builtin_amdgcn_readfirstlane(blockIdx.y * 4 + threadIdx.y);
  if (seg >= segments) return;
  const int k_begin = seg * GP_SEG;
  // load i of a chunk of 32 k: row 8 i + lane / 8 of the tile, piece lane % 8 of its 128 bytes
  const int lrow = lane >> 3, piece = lane & 7;
  const float* src[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) src[i] = W + (int64_t)min(n0 + 8 * i + lrow, N - 1) * ldw + k_begin + 4 * piece;
  float4 w0[8], w1[8];   // two chunks of 32 k on their way while a third is multiplied
#pragma unroll
  for (int i = 0; i < 8; ++i) w0[i] = he_load16_once<float4>(src[i]);
#pragma unroll
  for (int i = 0; i < 8; ++i) w1[i] = he_load16_once<float4>(src[i] + 32);
  float acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = 0.f;
  const float* arow[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) arow[m] = A + (int64_t)min(m, M - 1) * lda + k_begin;
  float4* mine = turned[threadIdx.y];
#define GP_TURN(WV_, C_)                                                                          \
  {                                                                                               \
    _Pragma("unroll") for (int i = 0; i < 8; ++i) mine[piece * GP_TURN_ROWS + 8 * i + lrow] = WV_[i]; \
    __builtin_amdgcn_wave_barrier();                                                              \
    _Pragma("unroll") for (int p = 0; p < 8; ++p) {                                               \
      const float4 w4 = mine[p * GP_TURN_ROWS + lane];                                            \
      const float w[4] = {w4.x, w4.y, w4.z, w4.w};                                                \
      _Pragma("unroll") for (int e = 0; e < 4; ++e)                                               \
        _Pragma("unroll") for (int m = 0; m < MT; ++m)                                            \
          acc[m] = fmaf(arow[m][32 * (C_) + 4 * p + e], w[e], acc[m]);                            \
    }                                                                                             \
    __builtin_amdgcn_wave_barrier();                                                              \
  }
  // (the scheduler would ask for all four chunks at once and then spill two of them: each
  // sched_barrier keeps a group of loads where it is written)
  __builtin_amdgcn_sched_barrier(0);
  GP_TURN(w0, 0)
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) w0[i] = he_load16_once<float4>(src[i] + 64);
  __builtin_amdgcn_sched_barrier(0);
  GP_TURN(w1, 1)
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) w1[i] = he_load16_once<float4>(src[i] + 96);
  __builtin_amdgcn_sched_barrier(0);
  GP_TURN(w0, 2)
  GP_TURN(w1, 3)
#undef GP_TURN
  const int n = n0 + lane;
  if (n < N) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (m < M) partial[((int64_t)seg * M + m) * N + n] = acc[m];
  }
}

template <typename TC>
__global__ __launch_bounds__(256) void gemm_plain_rows_sum_kernel(
    TC* __restrict__ C, const float* __restrict__ partial, const void* __restrict__ bias, int bias_dtype,
    int M, int N, int64_t ldc, int segments) {
  const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
  if (n >= N) return;
  float total = 0.f;
  int s = 0;
  for (; s + 8 <= segments; s += 8) {   // eight sums on their way at a time; added in segment order
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = partial[((int64_t)(s + u) * M + m) * N + n];
#pragma unroll
    for (int u = 0; u < 8; ++u) total += v[u];
  }
  for (; s < segments; ++s) total += partial[((int64_t)s * M + m) * N + n];
  if (bias != nullptr) total += load_param(bias, n, bias_dtype);
  C[(int64_t)m * ldc + n] = from_float<TC>(total);
}

// Whether a 32-bit product runs through the streaming kernel: up to GP_MROWS_MAX_M rows, and up to twice as many where tiles of 64 x 64
// would leave half of the units idle (3584 x 18944 at 128 rows: 458 us in tiles, 4608 x 3584, whose tiles fill the chip, 86);
// weights of whole segments in aligned rows. Its workgroups are 16 weight rows and its wavefronts a segment each, so it is
// left where these do not fill the chip. K in few segments against many weight rows, whose wavefronts mostly idle: up to 8
// rows the rows kernel (32000 x 256 at 1 row 10.4 us, streamed 14.0; 65536 x 128 at 8 rows 19.8, 22.1), above that tiles
// (151936 x 128 at 64 rows 44, 182; 16384 x 512 at 64 rows 20, 28; but 16384 x 256 at 16 rows 11.6, 8.6, and 8192 x 256
// at 64 even). Long K against few weight rows, a unit's own rate of about 30 bytes a ns: the rows kernel (512 x 12288
// at 1 row 13.6, 26.6, at 8 rows 20, 29; 1024 x 4864 at 4 rows 13.5, 14.1; 2048 x 8192 at 1 row 20.1, 22.7, at 4 rows 23.8, 22.2).
// Workgroups that fill part of their last round (a unit with one more than the others takes that much longer), the less of it
// the more rows: 4608 x 3584 at 1 row 17.0, 20.1, at 4 rows 20.8, 20.6; 4160 x 8192 at 4 rows 37.4, 43.8; 5120 x 5120 at 1 row
// 24.7, 27.8 (weights from memory; over 7758 random sizes of 1 to 8 rows the choice takes 0.69 of the rows kernel's time in the
// geometric mean, 24 of them 1.1 to 1.17 of it).
static bool gp_streams(int M, int N, int K, bool aligned) {
  const int segments = K / GP_SEG, cus = he_cus();
  if (!aligned || K % GP_SEG != 0) return false;
  if (M > GP_MROWS_MAX_M) return M <= 2 * GP_MROWS_MAX_M && 4 * ((N + 63) / 64) <= cus;
  if (segments <= (M + 15) / 16 && N >= (M <= 16 ? 96 : 64) * cus) return false;
  if (M > GP_ROWS_MAX_M) return true;
  if (segments <= 4 && N >= 96 * cus) return M > 4 && M * segments > (N >= 192 * cus ? 16 : 8);
  if (segments <= 4 && N >= 66 * cus) return M * segments > (N >= 82 * cus ? 4 : 2);
  if (segments >= 24 && N <= 4 * cus) return 4 * M > segments - 16;
  if (segments >= 24 && 2 * N <= 13 * cus) return M > 2 && 8 * M > segments - 8;
  if (segments >= 24 && N <= 8 * cus) return M > 2;
  const int workgroups = (N + 15) / 16, held = (workgroups + cus - 1) / cus * cus;       // held: what whole rounds have room for
  const bool idle = workgroups > cus && N <= 40 * cus && 10ll * M * held <= 108ll * held - 120ll * workgroups;
  return !idle || segments < 16 || (segments < 24 && M > 1);
}

// Floats of workspace with which a product of M rows runs through the kernels for few rows (0: another kernel takes it, which
// needs none). in_dtype, out_dtype below 0: the most that any operands of these sizes take.
extern "C" int64_t he_gemm_plain_workspace_floats(int M, int N, int K, int in_dtype, int out_dtype, int aligned) {
  if (M <= 0 || M > GP_ROWS_MAX_M || N <= 0 || K <= 0) return 0;
  if (in_dtype == HE_F32 && out_dtype == HE_F32 && gp_streams(M, N, K, aligned != 0)) return 0;
  return (int64_t)((K + GP_SEG - 1) / GP_SEG) * M * N;
}

template <typename TA, typename TW, typename TC>
static int launch_rows(void* C, const void* A, const void* W, const void* bias, int bias_dtype, int M,
                       int N, int K, int64_t lda, int64_t ldw, int64_t ldc, float* ws, hipStream_t s) {
  const int segments = (K + GP_SEG - 1) / GP_SEG;
  dim3 grid((N + 63) / 64, (segments + 3) / 4), block(64, 4);
  HE_REQUIRE(grid.y <= 65535, "he_gemm_plain: K=%d too long for one launch", K);
  // 32-bit weights in whole segments, rows 16-byte aligned: fetched line by line and turned round in LDS
  constexpr bool f32 = sizeof(TA) == 4 && sizeof(TW) == 4;
  const bool turned = f32 && K % GP_SEG == 0 && (ldw & 3) == 0 && (((uintptr_t)W) & 15) == 0;
#define GP_ROWS(MT_)                                                                                  \
  if (turned)                                                                                         \
    gemm_plain_rows_turned_kernel<MT_><<<grid, block, 0, s>>>(ws, (const float*)A, (const float*)W, M, N, K, \
                                                              lda, ldw, segments);                    \
  else                                                                                                \
    gemm_plain_rows_kernel<MT_, TA, TW><<<grid, block, 0, s>>>(ws, (const TA*)A, (const TW*)W, M, N, K, \
                                                               lda, ldw, segments)
  if (M == 1) GP_ROWS(1);
  else if (M == 2) GP_ROWS(2);
  else if (M <= 4) GP_ROWS(4);
  else GP_ROWS(8);
#undef GP_ROWS
  int rc = he_check_launch("he_gemm_plain");
  if (rc) return rc;
  gemm_plain_rows_sum_kernel<TC><<<dim3((N + 255) / 256, M), 256, 0, s>>>((TC*)C, ws, bias, bias_dtype, M, N,
                                                                          ldc, segments);
  return he_check_launch("he_gemm_plain");
}

// The kernel that streams the weights. 16 wavefronts a workgroup where the weight's rows
// give a compute unit one workgroup or less, else 8 (two workgroups share a unit).
static int launch_stream(float* C, const float* A, const float* W, const void* bias, int bias_dtype, int M, int N, int K,
                         int64_t lda, int64_t ldw, int64_t ldc, hipStream_t s) {
  const dim3 grid((N + 15) / 16, (M + GP_MROWS_MAX_M - 1) / GP_MROWS_MAX_M);
#define GP_STREAM(MT_, NW_, KS_, ONCE_) \
  gemm_plain_stream_kernel<MT_, NW_, KS_, ONCE_><<<grid, NW_ * 64, 0, s>>>(C, A, W, bias, bias_dtype, M, N, K, lda, ldw, ldc)
  if (M <= 16) {
    if ((int)grid.x <= he_cus()) GP_STREAM(1, 16, 64, true);
    else GP_STREAM(1, 8, 64, true);
  } else if (M <= 32) {
    GP_STREAM(2, 8, 32, true);
  } else if (M <= GP_MROWS_MAX_M) {
    GP_STREAM(4, 8, 32, true);
  } else {
    GP_STREAM(4, 8, 32, false);
  }
#undef GP_STREAM
  return he_check_launch("he_gemm_plain");
}

// gemm_plain_rounds.hip
int he_gemm_plain_rounds(float* C, const float* A, const float* W, const void* bias, int bias_dtype, int M, int N, int K, int64_t lda,
                         int64_t ldw, int64_t ldc, hipStream_t s);
float he_gemm_plain_rounds_estimate(int M, int N);

// The tile of this file's kernel: of its sizes the one whose fullest compute unit has the least to do (a unit's workgroups share its
// matrix cores, so its time is the outputs dealt to it); the larger tile where they tie, as it reads fewer operands an output.
struct GpTile {
  int bm, bn;
  int64_t tiles, most;        // outputs of the fullest unit
};
static GpTile gp_tile(int M, int N) {
  GpTile best = {};
  const int sizes[3][2] = {{128, 128}, {128, 64}, {64, 64}};
  for (auto& size : sizes) {
    const int64_t tiles = (int64_t)((M + size[0] - 1) / size[0]) * ((N + size[1] - 1) / size[1]);
    const int64_t most = (tiles + he_cus() - 1) / he_cus() * size[0] * size[1];
    if (best.bm == 0 || most < best.most) best = {size[0], size[1], tiles, most};
  }
  return best;
}

// Whether the product of rows that begin at 16-byte boundaries goes to gemm_plain_rounds.hip: K in 32s and more than one of its stages (with
// one 700 x 288 x 32 takes 5.4 us there, 4.5 here), unless so many rows of its tiles of 128 are padding that its estimate is above this file's
// kernel's time, 4.5 ps an output and k of the fullest unit (130 rows of 37888 x 3584 602 us there, 470 here). wide: four outputs of a row are
// stored at once; where they are not, single stores outlast the products of a K below 512 (532 x 14083 x 64 31.3 us and 20.5, 946 x 4567 x 160
// 27.9 and 24.2, 559 x 3297 x 512 27.1 and 26.4). Over 227 products of 33 to 4000 rows, 16 to 30000 columns and K 32 to 20000 the 206 that are
// not refused by these two lines take 0.62 to 1.04 of the time with this file's kernel alone.
extern "C" int he_gemm_plain_in_rounds(int M, int N, int K, int wide) {
  return K % 32 == 0 && K >= 64 && (wide || K >= 512) && he_gemm_plain_rounds_estimate(M, N) <= 4.5e-6f * gp_tile(M, N).most;
}

// More rows: tiles on the matrix cores.
static int launch_mfma(float* C, const float* A, const float* W, const void* bias, int bias_dtype, int M, int N, int K,
                       int64_t lda, int64_t ldw, int64_t ldc, hipStream_t s) {
  const int vec = (lda & 3) == 0 && (ldw & 3) == 0 && (((uintptr_t)A) & 15) == 0 && (((uintptr_t)W) & 15) == 0;
  // (lda, ldw: a lane's offsets into a tile's rows are 32-bit)
  if (vec && lda < (1 << 22) && ldw < (1 << 22) &&
      he_gemm_plain_in_rounds(M, N, K, (ldc & 3) == 0 && (N & 3) == 0 && ((uintptr_t)C & 15) == 0))
    return he_gemm_plain_rounds(C, A, W, bias, bias_dtype, M, N, K, lda, ldw, ldc, s);
  const GpTile tile = gp_tile(M, N);
  const int bm = tile.bm, bn = tile.bn;
  HE_REQUIRE(tile.tiles < (1 << 30), "he_gemm_plain: M=%d N=%d too large for one launch", M, N);
  const int mt = (M + bm - 1) / bm, nt = (N + bn - 1) / bn;
  const int grid = (int)((tile.tiles + HE_XCDS - 1) / HE_XCDS * HE_XCDS);
#define GP_MFMA(BM_, BN_) \
  gemm_plain_mfma_kernel<BM_, BN_><<<grid, 256, 0, s>>>(C, A, W, bias, bias_dtype, M, N, K, lda, ldw, ldc, mt, nt, vec)
  if (bn == 128) GP_MFMA(128, 128);
  else if (bm == 128) GP_MFMA(128, 64);
  else GP_MFMA(64, 64);
#undef GP_MFMA
  return he_check_launch("he_gemm_plain");
}

// workspace_f32 (may be null) of workspace_floats floats: with as many as he_gemm_plain_workspace_floats names for
// these operands, or more, a product of few rows that is not streamed runs through the
// kernels made for it. The result is the same bit for bit either way.
extern "C" int he_gemm_plain(void* C, const void* A, const void* W, const void* bias, int M, int N,
                             int K, int64_t lda, int64_t ldw, int64_t ldc, int in_dtype,
                             int out_dtype, int bias_dtype, void* workspace_f32,
                             int64_t workspace_floats, void* stream) {
  HE_REQUIRE(M >= 0 && N > 0 && K > 0, "he_gemm_plain: bad sizes M=%d N=%d K=%d", M, N, K);
  HE_REQUIRE(lda >= K && ldw >= K && ldc >= N, "he_gemm_plain: bad leading dimensions");
  if (M == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const bool f32 = in_dtype == HE_F32 && out_dtype == HE_F32;
  const bool aligned = (lda & 3) == 0 && (ldw & 3) == 0 && (((uintptr_t)A) & 15) == 0 && (((uintptr_t)W) & 15) == 0;
  if (f32 && gp_streams(M, N, K, aligned))
    return launch_stream((float*)C, (const float*)A, (const float*)W, bias, bias_dtype, M, N, K, lda, ldw, ldc, s);
  const int64_t need = he_gemm_plain_workspace_floats(M, N, K, in_dtype, out_dtype, aligned);
  if (need > 0 && workspace_f32 != nullptr && workspace_floats >= need) {
    float* ws = (float*)workspace_f32;
    if (in_dtype == HE_F32 && out_dtype == HE_F32)
      return launch_rows<float, float, float>(C, A, W, bias, bias_dtype, M, N, K, lda, ldw, ldc, ws, s);
    if (in_dtype == HE_BF16 && out_dtype == HE_BF16)
      return launch_rows<bf16_t, bf16_t, bf16_t>(C, A, W, bias, bias_dtype, M, N, K, lda, ldw, ldc, ws, s);
    if (in_dtype == HE_BF16 && out_dtype == HE_F32)
      return launch_rows<bf16_t, bf16_t, float>(C, A, W, bias, bias_dtype, M, N, K, lda, ldw, ldc, ws, s);
    HE_REQUIRE(false, "he_gemm_plain: unsupported dtypes in=%d out=%d", in_dtype, out_dtype);
  }
  if (f32)
    return launch_mfma((float*)C, (const float*)A, (const float*)W, bias, bias_dtype, M, N, K, lda, ldw, ldc, s);
  dim3 grid((N + GP_BN - 1) / GP_BN, (M + GP_BM - 1) / GP_BM);
  HE_REQUIRE(grid.y <= 65535, "he_gemm_plain: M=%d too large for one launch", M);
  if (in_dtype == HE_BF16 && out_dtype == HE_BF16)
    gemm_plain_kernel<bf16_t, bf16_t, bf16_t><<<grid, 256, 0, s>>>(
        (bf16_t*)C, (const bf16_t*)A, (const bf16_t*)W, bias, bias_dtype, M, N, K, lda, ldw, ldc);
  else if (in_dtype == HE_BF16 && out_dtype == HE_F32)
    gemm_plain_kernel<bf16_t, bf16_t, float><<<grid, 256, 0, s>>>(
        (float*)C, (const bf16_t*)A, (const bf16_t*)W, bias, bias_dtype, M, N, K, lda, ldw, ldc);
  else
    HE_REQUIRE(false, "he_gemm_plain: unsupported dtypes in=%d out=%d", in_dtype, out_dtype);
  return he_check_launch("he_gemm_plain");
}
