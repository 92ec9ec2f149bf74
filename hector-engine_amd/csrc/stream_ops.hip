// Small operations around the layers. On whole rows of the residual stream's width:
//   he_depth_mix   the stream that goes on after a layer as a weighted sum of the embedding's output and
//                  of every layer's result so far
//   he_gated_add   out = a + sigmoid(x . g) * b, one number a row in front of b
// and on the page tables:
//   he_scatter_i32 table[index] = value
#include "common.h"
#include "hector_kernels.h"

// entries: n indexes, then n values. Bound by its launch: a step's new and given-back pages are some tens of entries.
__global__ __launch_bounds__(256) void scatter_i32_kernel(int32_t* __restrict__ table, const int32_t* __restrict__ entries, int n,
                                                          int64_t size) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int at = entries[i];
  if (at >= 0 && at < size) table[at] = entries[n + i];
}

extern "C" int he_scatter_i32(void* table_i32, const void* entries_i32, int n, int64_t size, void* stream) {
  HE_REQUIRE(n >= 0 && size >= 0 && n <= (1 << 30), "he_scatter_i32: bad sizes n=%d", n);
  if (n == 0) return 0;
  scatter_i32_kernel<<<(n + 255) / 256, 256, 0, (hipStream_t)stream>>>((int32_t*)table_i32, (const int32_t*)entries_i32, n, size);
  return he_check_launch("he_scatter_i32");
}

// kept: fp32 [n or more][count] (plane j at j * plane elements): planes 0 .. n - 2 hold the earlier results.
// resid (fp32 [count]) holds the newest result: it is stored as plane n - 1, and resid becomes
// sum_j coeffs[j] * plane_j, added in ascending j.
__global__ __launch_bounds__(256) void depth_mix_kernel(float* __restrict__ resid, float* __restrict__ kept,
                                                        int64_t plane, const void* __restrict__ coeffs, int c_dtype,
                                                        int n, int64_t count) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const float newest = resid[i];
  kept[(int64_t)(n - 1) * plane + i] = newest;
  float acc = 0.f;
  for (int j = 0; j + 1 < n; ++j) acc = fmaf(load_param(coeffs, j, c_dtype), kept[(int64_t)j * plane + i], acc);
  resid[i] = fmaf(load_param(coeffs, n - 1, c_dtype), newest, acc);
}

extern "C" int he_depth_mix(void* resid_f32, void* kept_f32, int64_t plane, const void* coeffs, int c_dtype, int n,
                            int64_t count, void* stream) {
  HE_REQUIRE(n >= 1 && count >= 0 && plane >= count, "he_depth_mix: bad sizes n=%d", n);
  HE_REQUIRE(c_dtype == HE_BF16 || c_dtype == HE_F32, "he_depth_mix: unknown dtype %d", c_dtype);
  if (count == 0) return 0;
  const int64_t blocks = (count + 255) / 256;
  depth_mix_kernel<<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>((float*)resid_f32, (float*)kept_f32, plane, coeffs,
                                                                      c_dtype, n, count);
  return he_check_launch("he_depth_mix");
}

// out[r, :] = a[r, :] + sigmoid(sum_i x[r, i] * g[i]) * b[r, :]; x [rows, Dx], a, b, out [rows, D]; the sum in fp32.
// KEPT: a thread's first elements, asked for together, a and b beside the sum they wait for (4 rows of 2048: 4.9 us with a load at a time, 4.1).
template <typename T, int KEPT>
__global__ __launch_bounds__(256) void gated_add_kernel(T* __restrict__ out, const T* __restrict__ a,
                                                        const T* __restrict__ b, const T* __restrict__ x,
                                                        const void* __restrict__ g, int g_dtype, int D, int Dx) {
  __shared__ float scratch[16];
  const int64_t row = blockIdx.x;
  float xv[KEPT], gv[KEPT], av[KEPT], bv[KEPT];
#pragma unroll
  for (int k = 0; k < KEPT; ++k) {
    const int i = min((int)(threadIdx.x + k * blockDim.x), Dx - 1), j = min((int)(threadIdx.x + k * blockDim.x), D - 1);
    xv[k] = to_float(x[row * Dx + i]);
    gv[k] = load_param(g, i, g_dtype);
    av[k] = to_float(a[row * D + j]);
    bv[k] = to_float(b[row * D + j]);
  }
  float dot = 0.f;
#pragma unroll
  for (int k = 0; k < KEPT; ++k)
    if ((int)(threadIdx.x + k * blockDim.x) < Dx) dot = fmaf(xv[k], gv[k], dot);
  for (int i = threadIdx.x + KEPT * blockDim.x; i < Dx; i += blockDim.x) dot = fmaf(to_float(x[row * Dx + i]), load_param(g, i, g_dtype), dot);
  dot = block_sum(dot, scratch);
  const float w = 1.f / (1.f + expf(-dot));
#pragma unroll
  for (int k = 0; k < KEPT; ++k) {
    const int i = threadIdx.x + k * blockDim.x;
    if (i < D) out[row * D + i] = from_float<T>(fmaf(w, bv[k], av[k]));
  }
  for (int i = threadIdx.x + KEPT * blockDim.x; i < D; i += blockDim.x)
    out[row * D + i] = from_float<T>(fmaf(w, to_float(b[row * D + i]), to_float(a[row * D + i])));
}

extern "C" int he_gated_add(void* out, const void* a, const void* b, const void* x, const void* g, int g_dtype,
                            int rows, int D, int Dx, int dtype, void* stream) {
  HE_REQUIRE(rows >= 0 && D > 0 && Dx > 0, "he_gated_add: bad sizes");
  HE_REQUIRE((dtype == HE_BF16 || dtype == HE_F32) && (g_dtype == HE_BF16 || g_dtype == HE_F32), "he_gated_add: unknown dtype");
  if (rows == 0) return 0;
  const int threads = D >= 1024 ? 256 : (D >= 256 ? 128 : 64);
  hipStream_t s = (hipStream_t)stream;
#define GA_LAUNCH(T, KEPT) \
  gated_add_kernel<T, KEPT><<<rows, threads, 0, s>>>((T*)out, (const T*)a, (const T*)b, (const T*)x, g, g_dtype, D, Dx)
  const bool few = D <= 2 * threads && Dx <= 2 * threads;
  if (dtype == HE_BF16 && few) GA_LAUNCH(bf16_t, 2);
  else if (dtype == HE_BF16) GA_LAUNCH(bf16_t, 8);
  else if (few) GA_LAUNCH(float, 2);
  else GA_LAUNCH(float, 8);
#undef GA_LAUNCH
  return he_check_launch("he_gated_add");
}
