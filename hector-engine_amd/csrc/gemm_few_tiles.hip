// bf16 products of some hundred rows and few columns, whose tiles are fewer than the chip has units: out[m][n] = sum_k X[m][k]
// W[n][k] (+ bias), fp32 sums in order of k, K in steps of 64.
//
// What bounds such a product is not the matrix cores but what one unit takes in: its weights come from memory, and a unit's loads
// into LDS run at some 54 GB/s whatever the tile, the wavefronts or the stages asked for ahead (64 x 64 tiles of a K of 3584: 16 KiB a stage in
// 0.30 us, 64 x 96 20 KiB in 0.37, 128 x 128 32 KiB in 0.6). So the time is (BM + BN) K, and the tile is the one of least
// BM + BN whose tiles are one round of the chip; tiles come in 64 or 128 rows and any sixteens of columns from 32 to 128 for that. (256 rows: 4608 x
// 3584 36.7 us by the library's choice, 22.1 here; 5120 x 5120 48.8 and 30.6; 1152 x 896 7.6 and 5.5.)
//
// A workgroup of four wavefronts, each a quarter of the rows and all columns. A stage of 64 k of both operands goes from
// memory straight into LDS, 1 KiB (eight rows) a wavefront and instruction, four stages in flight; a row's eight 16-byte
// pieces lie at their index xor the row, so that the sixteen rows of an operand read hit different banks. One barrier a stage.
#include "common.h"
#include "hector_kernels.h"

typedef __bf16 ft_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ft_f32x4 __attribute__((ext_vector_type(4)));
#define FT_BK 64
#define FT_WAVES 4
#define FT_BUFS 4

struct FtCase {
  const uint16_t* x;          // [M][ldx]
  const uint16_t* w;          // [N][ldw]
  uint16_t* out;              // [M][ldo]
  const void* bias;           // [N] or null
  int bias_dtype;
  int M, N, K;
  int64_t ldx, ldw, ldo;
};

__device__ __forceinline__ void ft_load(uint32_t to, uint32_t offset, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(offset), "s"(base) : "memory", "m0");
}
// this wavefront's loads but the last N have arrived, and its LDS reads
template <int N>
__device__ __forceinline__ void ft_wait() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory"); }

template <int BM, int BN>
__global__ __launch_bounds__(64 * FT_WAVES, 1) void gemm_few_tiles_kernel(FtCase c) {
  constexpr int XI = BM / 64, WI = BN / 16;                       // 16-row operand tiles of a wavefront
  constexpr int CHUNKS = (BM + BN) / 8, EACH = CHUNKS / FT_WAVES, MORE = CHUNKS % FT_WAVES;   // (the first MORE wavefronts load one more)
  constexpr uint32_t STAGE = (BM + BN) * FT_BK * 2;
  static_assert(FT_BUFS * STAGE <= 160 * 1024, "a unit's LDS");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[FT_BUFS * STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int mtiles = (c.M + BM - 1) / BM;
  // the row tiles that read one stretch of weights run behind one L2
  const int total = mtiles * ((c.N + BN - 1) / BN), per_xcd = (total + HE_XCDS - 1) / HE_XCDS;
  const int tile = (blockIdx.x % HE_XCDS) * per_xcd + blockIdx.x / HE_XCDS;
  if ((int)blockIdx.x / HE_XCDS >= per_xcd || tile >= total) return;       // (the whole workgroup)
  const int m0 = tile % mtiles * BM, n0 = tile / mtiles * BN;
  const uint32_t piece = (uint32_t)((lane & 7) ^ (lane >> 3)) * 16;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  // a chunk: eight rows of x or of w; rows beyond the matrices are their last row again, whose outputs are not stored
  const uint8_t* xbase = (const uint8_t*)(c.x + (int64_t)m0 * c.ldx);
  const uint8_t* wbase = (const uint8_t*)(c.w + (int64_t)n0 * c.ldw);
  uint32_t off[EACH + 1];
#pragma unroll
  for (int i = 0; i <= EACH; ++i) {
    const int row = 8 * (i * FT_WAVES + wave) + (lane >> 3);
    off[i] = (uint32_t)(row < BM ? min(row, c.M - 1 - m0) * c.ldx * 2 : min(row - BM, c.N - 1 - n0) * c.ldw * 2) + piece;
  }
  const bool more = MORE > 0 && wave < MORE;                      // (the same in the wavefront)
  const int stages = c.K / FT_BK;
  int left = stages - 1;
  auto fetch = [&](uint32_t buf) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int chunk = i * FT_WAVES + wave;
      ft_load(lds0 + buf + chunk * 1024, off[i], chunk < BM / 8 ? xbase : wbase);
    }
    if (more) ft_load(lds0 + buf + (EACH * FT_WAVES + wave) * 1024, off[EACH], wbase);
    const int on = left > 0 ? FT_BK * 2 : 0;                      // (behind the last stage it is fetched again, and not read)
    xbase += on;
    wbase += on;
    --left;
  };
  ft_f32x4 acc[XI][WI];
#pragma unroll
  for (int i = 0; i < XI; ++i)
#pragma unroll
    for (int j = 0; j < WI; ++j) acc[i][j] = ft_f32x4{0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, g = lane >> 4;
  const uint32_t xrow = (wave * (BM / FT_WAVES) + r16) * 128, wrow = (BM + r16) * 128;
  const uint32_t at[2] = {(uint32_t)((g ^ (r16 & 7)) * 16), (uint32_t)(((4 + g) ^ (r16 & 7)) * 16)};
#pragma unroll
  for (int s = 0; s < FT_BUFS - 1; ++s) fetch(s * STAGE);
  uint32_t buf = 0, fill = (FT_BUFS - 1) * STAGE;
  for (int s = 0; s < stages; ++s) {
    if (more) ft_wait<(FT_BUFS - 2) * (EACH + 1)>();
    else ft_wait<(FT_BUFS - 2) * EACH>();
    __builtin_amdgcn_s_barrier();                                 // this stage is there, and everyone has read the one before it
    __builtin_amdgcn_sched_barrier(0);
    fetch(fill);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      ft_bf16x8 wv[WI], xv[XI];
#pragma unroll
      for (int j = 0; j < WI; ++j) wv[j] = *reinterpret_cast<const ft_bf16x8*>(lds + buf + wrow + at[kk] + j * 2048);
#pragma unroll
      for (int i = 0; i < XI; ++i) xv[i] = *reinterpret_cast<const ft_bf16x8*>(lds + buf + xrow + at[kk] + i * 2048);
#pragma unroll
      for (int i = 0; i < XI; ++i)
#pragma unroll
        for (int j = 0; j < WI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[j], xv[i], acc[i][j], 0, 0, 0);
    }
    buf = buf == (FT_BUFS - 1) * STAGE ? 0 : buf + STAGE;
    fill = fill == (FT_BUFS - 1) * STAGE ? 0 : fill + STAGE;
  }
  ft_wait<0>();                                                   // (nothing is on its way into LDS that is given back)
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int m = m0 + wave * (BM / FT_WAVES) + 16 * i + r16;
    if (m >= c.M) continue;
#pragma unroll
    for (int j = 0; j < WI; ++j) {
      const int n = n0 + 16 * j + 4 * g;                          // (N is a multiple of 4)
      if (n >= c.N) continue;
      ft_f32x4 v = acc[i][j];
      if (c.bias)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += load_param(c.bias, n + e, c.bias_dtype);
      *reinterpret_cast<uint2*>(c.out + m * c.ldo + n) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
    }
  }
}

// The tile of a product: BM << 16 | BN, or 0 where no tile makes it one round of the chip. The least BM + BN; of equal ones the
// taller, which reads the weights less often.
extern "C" int he_gemm_few_tiles_tile(int M, int N) {
  if (M <= 0 || N <= 0) return 0;
  const int cus = he_cus();
  int best = 0, cost = 1 << 30;
  for (int bm = 128; bm >= 64; bm /= 2)
    for (int bn = 32; bn <= 128; bn += 16)
      if ((int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn) <= cus && bm + bn < cost) best = bm << 16 | bn, cost = bm + bn;
  return best;
}

template <int BM, int BN>
static int ft_launch(const FtCase& c, hipStream_t s) {
  const int64_t total = (int64_t)((c.M + BM - 1) / BM) * ((c.N + BN - 1) / BN);
  gemm_few_tiles_kernel<BM, BN><<<(unsigned)((total + HE_XCDS - 1) / HE_XCDS * HE_XCDS), 64 * FT_WAVES, 0, s>>>(c);
  return he_check_launch("he_gemm_few_tiles");
}

// tile: as he_gemm_few_tiles_tile gives it (any of its tiles is taken, also where they are more than a round).
extern "C" int he_gemm_few_tiles_bf16(void* out, const void* x, const void* w, const void* bias, int bias_dtype, int M, int N, int K,
                                      int64_t ldx, int64_t ldw, int64_t ldo, int tile, void* stream) {
  HE_REQUIRE(M >= 0 && N > 0 && K > 0 && N % 4 == 0 && K % FT_BK == 0, "he_gemm_few_tiles: bad sizes M=%d N=%d K=%d", M, N, K);
  HE_REQUIRE(ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0 && ldo >= N && ldo % 4 == 0, "he_gemm_few_tiles: bad leading dimensions");
  HE_REQUIRE((((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) == 0, "he_gemm_few_tiles: pointers must be 16-byte aligned");
  HE_REQUIRE(128 * ldx * 2 < (1ll << 32) && 128 * ldw * 2 < (1ll << 32), "he_gemm_few_tiles: rows too long");
  if (M == 0) return 0;
  const FtCase c = {(const uint16_t*)x, (const uint16_t*)w, (uint16_t*)out, bias, bias_dtype, M, N, K, ldx, ldw, ldo};
  hipStream_t s = (hipStream_t)stream;
#define FT_TILES(BM)                                                                                                      \
  switch (tile & 0xffff) {                                                                                                \
    case 32: return ft_launch<BM, 32>(c, s);                                                                              \
    case 48: return ft_launch<BM, 48>(c, s);                                                                              \
    case 64: return ft_launch<BM, 64>(c, s);                                                                              \
    case 80: return ft_launch<BM, 80>(c, s);                                                                              \
    case 96: return ft_launch<BM, 96>(c, s);                                                                              \
    case 112: return ft_launch<BM, 112>(c, s);                                                                            \
    case 128: return ft_launch<BM, 128>(c, s);                                                                            \
  }
  if (tile >> 16 == 64) { FT_TILES(64) }
  if (tile >> 16 == 128) { FT_TILES(128) }
#undef FT_TILES
  HE_REQUIRE(false, "he_gemm_few_tiles: no tiles of %d x %d", tile >> 16, tile & 0xffff);
}
