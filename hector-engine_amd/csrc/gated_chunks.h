// A memory per head whose rows have gates of their own, by chunks of CK_ROWS rows on the fp32 matrix cores:
//   S_t = exp(f_t) S_(t-1) + w_t v_t k_t^T  (dv x dk),  y_t = S_t q_t
// with a logarithm f_t <= 0 of what is kept and a weight w_t >= 0 of what is written a row. One after the other the
// rows are a chain of multiply-adds that leaves the chip waiting (the matrix memory of 14 heads of 128 x 256: 0.52 us a
// row, a prompt of 2,048 rows 1,003 us; the state space of 64 heads of 128 x 64: 665 us). In a chunk, with F_i the sum of f over its first i rows and S
// the memory before it,
//   y_i = exp(F_i) S q_i + sum over j <= i of exp(F_i - F_j) w_j (k_j . q_i) v_j
//   S'  = exp(F_n) S + sum over j of exp(F_n - F_j) w_j v_j k_j^T
// are matrix products, in three launches: every chunk's own share of S' (all chunks at once), the memory before every
// chunk (one walk over the chunks of a sequence, element by element), every chunk's rows (all at once). (The same two prompts of
// 2,048 rows: 141 and 138 us alone.)
// F is summed in 64 bits and no exponent is positive, so the powers are as exact as the
// walk's; everything else is fp32 arithmetic as there. What bounds the three: the share and the rows kernel the fp32
// products, the walk over chunks the memories it reads and writes (two passes over 4 (dv + 1) dk bytes a head and chunk).
//
// NORMED (the matrix memory): w_t = exp(i_t), S carries a factor exp(-m_t), m_t = max(f_t + m_(t-1), i_t), and
// y is divided by max(|n_t . q_t|, exp(-m_t)) + 1e-6 with n the same recurrence over k alone: n is one more column of S. In a chunk
// m_i = F_i + max(m before it, the largest i_j - F_j up to j = i); a chunk's own share is kept relative to its own G = the
// largest F_n - F_j + i_j until the walk knows m.
//
// The policy P gives what differs: static NORMED; gate(row, h, f, in): f, and in = i_t (NORMED) or w_t; place(st, h, c, d): where
// four neighbouring key dims from d on of column c (dv: n) of S lie in a sequence's state; keep(...) puts them back (n into every copy of it);
// m(st, h) and keep_m(...): NORMED's m and its copies; result(y, x, h): what follows the products.
#pragma once
#include <algorithm>
#include <climits>

#include "chunks.h"

#define GC_LD 68      // floats between rows of 64 in LDS (four banks on from row to row)
#define GC_KB 32      // key dims of a block of the rows kernel
#define GC_KLD 36
#define GC_WINDOW_FLOATS (64 << 20)   // memories held between the launches at once (256 MiB)
// No step goes by chunks whose longest sequence has no more rows than this; from there on gc_pays says.
#define GC_FROM 64
// Of several sequences in such a step, those of up to GC_SHORT rows are walked, in launches of their own: a chunk costs what a whole one does (one of
// 14 heads of 128 x 256 3.7 us in a step of many; a walk of one row 0.8, of 2 to 8 3.0 to 3.9, of 40 12; of 64 heads of 128 x 64 4.0 and 1.2, 1.4
// to 2.5, 6.7) and moves the memory three times. Up to GC_FEW rows a walk stages nothing, or little.
#define GC_SHORT 16
#define GC_FEW 4
static inline int gc_from(int num_seqs) { return num_seqs > 1 ? GC_SHORT : 0; }

// Where chunks pay: the rows of one sequence alone, of the longest beside shorter ones, and the rows the others have on average where they pay
// from GC_FROM on.
struct GcLines {
  int alone, beside, others;
};

#define GC_FORGETS -1e7f
typedef float gc_acc __attribute__((ext_vector_type(16)));

template <typename T>
struct GcArgs {
  const T* q;              // head h's at (h / per) dk
  const T* k;
  const T* v;              // at h dv
  int64_t stride;          // elements between rows
  int per;                 // heads that share q and k
  float q_scale;
  const int32_t* cu;
  const int32_t* slot;
  int num_seqs, H, dk, dv, dkp;      // dkp: key dims with the state's padding, a multiple of 4
  int from;                // sequences of up to so many rows are the walk's (gc_from)
  uint8_t* state;
  int64_t state_stride, state_offset;
  float* ws;               // [chunk of the window][H][cols][dkp]: first the chunks' shares, then the memories before them
  double* ends;            // [chunk of the window][H][2]: F_n and G of a chunk
};
template <typename T, class P>
__host__ __device__ constexpr int gc_cols(int dv) { return dv + (P::NORMED ? 1 : 0); }

__device__ __forceinline__ float4 gc_load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 gc_load4(const bf16_t* p) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                     __uint_as_float(v.y & 0xffff0000u));
}
// Four numbers at dim d of a row of a chunk of n rows from `first` on; zeros beyond the chunk or the head. The load itself
// stands behind no condition, so that a tile's loads go out together.
template <typename T>
__device__ __forceinline__ float4 gc_tile4(const T* first, int64_t stride, int row, int n, int d, int width) {
  const float4 v = gc_load4(first + min(row, n - 1) * stride + (d < width ? d : 0));
  return row < n && d < width ? v : make_float4(0.f, 0.f, 0.f, 0.f);
}

// exp(x) of an x <= 0 that is a difference of sums in 64 bits: what x loses as a 32-bit number would show in the power times |x|
__device__ __forceinline__ float gc_exp(double x) {
  const float hi = (float)x;
  if (hi < -104.f) return 0.f;      // (below half of the smallest number; -inf among them)
  const float e = expf(hi);
  return fmaf(e, (float)(x - (double)hi), e);
}

// Sums of many products are formed sixteen at a time, as two chains of eight, and then added: a chain of all of them would lose more in
// rounding than the walk's sums, which are spread over the lanes of a value dim. KEEP: what an addition loses is carried along to the next (NORMED,
// whose results are quotients of two such sums: keys of 512 dims and one sign were 1.15 times as far from 64 bits as the walk without it, and are 0.91 so;
// 2,048 rows of 14 heads of 128 x 256 take 141 us for it, 130 before).
template <bool KEEP>
__device__ __forceinline__ void gc_add(gc_acc& a, gc_acc& lost, const gc_acc& b, const gc_acc& c) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    if (KEEP) {
      const float more = b[r] + c[r] - lost[r], sum = a[r] + more;
      lost[r] = (sum - a[r]) - more;
      a[r] = sum;
    } else {
      a[r] += b[r] + c[r];
    }
  }
}
__device__ __forceinline__ gc_acc gc_mfma4(const float4& a, const float4& b) {
  gc_acc s = {0.f};
  s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, s, 0, 0, 0);
  s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, s, 0, 0, 0);
  s = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, s, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, s, 0, 0, 0);
}

// F of the lane's row (lane < 64: the rows of the chunk, summed up to and with it) and in; rows beyond the chunk keep everything and
// write nothing. NORMED: peak = the largest in - F up to and with the lane's row.
template <class P>
__device__ __forceinline__ void gc_gates(const P& p, int64_t r0, int n, int h, int lane, double& F, float& in, double& peak) {
  float f;
  p.gate(r0 + min(lane, n - 1), h, f, in);
  if (lane >= n) f = 0.f, in = P::NORMED ? -INFINITY : 0.f;
  // (a row that forgets everything has f = -inf, and differences of sums with it would be no numbers: exp of what stands in its place is 0 too, and
  // 64 of them are known to 1e-7 in 64 bits; NaN stays)
  if (f < GC_FORGETS) f = GC_FORGETS;
  F = (double)f;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double u = __shfl_up(F, o);
    if (lane >= o) F += u;
  }
  peak = 0.;
  if (P::NORMED) {
    peak = (double)in - F;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double u = __shfl_up(peak, o);
      if (lane >= o) peak = fmax(peak, u);
    }
  }
}

// The m behind a chunk of those ends.
__device__ __forceinline__ float gc_next_m(const double2& e, float m) { return (float)fmax(e.x + (double)m, e.y); }

// ---- every chunk's own share of the memory behind it -----------------------------------------------------
// One workgroup of four wavefronts a (64 key dims x 64 columns, head, chunk), a wavefront 32 x 32 of it, two rows of the
// chunk an instruction (v_mfma_f32_32x32x2_f32: A lane l holds A[l % 32][l / 32], B likewise, D register r of lane l is
// D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32]).
template <typename T, class P>
__global__ __launch_bounds__(256) void gc_share_kernel(GcArgs<T> a, P p, int t0) {
  __shared__ __attribute__((aligned(16))) float ks[CK_ROWS * GC_LD], vs[CK_ROWS * GC_LD];
  __shared__ float weight[CK_ROWS], part[4][64];
  const int h = blockIdx.y;
  int seq, chunk;
  if (!ck_find(t0 + (int)blockIdx.z, a.cu, a.num_seqs, a.from, seq, chunk)) return;
  if (a.slot[seq] < 0) return;
  const int vb = (a.dv + 63) / 64;
  const int d0 = ((int)blockIdx.x / vb) * 64, c0 = ((int)blockIdx.x % vb) * 64;
  const int64_t r0 = a.cu[seq] + (int64_t)chunk * CK_ROWS;
  const int n = min(CK_ROWS, (int)(a.cu[seq + 1] - r0));
  const int t = threadIdx.x, d = 4 * (t & 15);
  const T* kr = a.k + r0 * a.stride + (int64_t)(h / a.per) * a.dk;
  const T* vr = a.v + r0 * a.stride + (int64_t)h * a.dv;
  float4 kx[4], vx[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    kx[i] = gc_tile4(kr, a.stride, (t >> 4) + 16 * i, n, d0 + d, a.dk);
    vx[i] = gc_tile4(vr, a.stride, (t >> 4) + 16 * i, n, c0 + d, a.dv);
  }
  if (t < 64) {
    double F, peak;
    float in;
    gc_gates(p, r0, n, h, t, F, in, peak);
    // (G as a 32-bit number: where it becomes the m behind the chunk, the share is taken as it is)
    const double Fn = __shfl(F, 63), G = P::NORMED ? (float)(Fn + __shfl(peak, 63)) : 0.;
    // (in = -inf writes nothing, also where all of a chunk's rows have it and G is -inf)
    weight[t] = !P::NORMED ? in * gc_exp(Fn - F) : in == -INFINITY ? 0.f : gc_exp(Fn - F + (double)in - G);
    if (t == 0 && blockIdx.x == 0) *reinterpret_cast<double2*>(a.ends + 2 * ((int64_t)blockIdx.z * a.H + h)) = make_double2(Fn, G);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = (t >> 4) + 16 * i;
    const float w = weight[row];
    *reinterpret_cast<float4*>(ks + row * GC_LD + d) = make_float4(kx[i].x * w, kx[i].y * w, kx[i].z * w, kx[i].w * w);
    *reinterpret_cast<float4*>(vs + row * GC_LD + d) = vx[i];
  }
  __syncthreads();
  const int cols = gc_cols<T, P>(a.dv);
  float* out = a.ws + ((int64_t)blockIdx.z * a.H + h) * cols * a.dkp;
  const int wave = t >> 6, l32 = t & 31, hl = (t >> 5) & 1;
  const int i0 = (wave >> 1) * 32, j0 = (wave & 1) * 32;       // columns of S, key dims
  gc_acc acc = {0.f};
  for (int g0 = 0; g0 < n; g0 += 16) {
    gc_acc some[2] = {{0.f}, {0.f}};
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int row = g0 + 8 * hl + m;
      some[m & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vs[row * GC_LD + i0 + l32], ks[row * GC_LD + j0 + l32], some[m & 1], 0, 0, 0);
    }
    gc_add<false>(acc, acc, some[0], some[1]);
  }
  const int od = d0 + j0 + l32;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int c = c0 + i0 + 8 * (r >> 2) + 4 * hl + (r & 3);
    if (c < a.dv && od < a.dkp) out[(int64_t)c * a.dkp + od] = acc[r];
  }
  if (P::NORMED && c0 == 0) {      // n's share: the weighted rows of k alone
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) sum += ks[(16 * wave + e) * GC_LD + (t & 63)];
    part[wave][t & 63] = sum;
    __syncthreads();
    if (t < 64 && d0 + t < a.dkp) out[(int64_t)a.dv * a.dkp + d0 + t] = (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
  }
}

// ---- the memory before every chunk ---------------------------------------------------------------------
// A thread holds four neighbouring key dims of a column of a sequence's S and walks its chunks in the window
// [t0, t0 + nt): the chunk's share is taken out, the memory before the chunk put in its place. Behind them S goes back to the state: the
// next window's walk takes it from there.
template <typename T, class P>
__global__ __launch_bounds__(256) void gc_carry_kernel(GcArgs<T> a, P p, int t0, int nt, float* __restrict__ before_m) {
  const int seq = blockIdx.z, h = blockIdx.y;
  const int slot = a.slot[seq];
  if (slot < 0 || a.cu[seq + 1] - a.cu[seq] <= a.from) return;
  int before = 0;
  for (int s0 = 0; s0 < seq; s0 += 64) {
    const int s = s0 + (int)(threadIdx.x & 63);
    int n = s < seq ? ck_chunks(a.cu, s, a.from) : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
    before += n;
  }
  const int first = max(0, t0 - before), end = min(ck_chunks(a.cu, seq, a.from), t0 + nt - before);
  if (first >= end) return;
  const int cols = gc_cols<T, P>(a.dv);
  const int64_t memory = (int64_t)cols * a.dkp, step = (int64_t)a.H * memory;
  const int64_t id = blockIdx.x * 256ll + threadIdx.x, at = 4 * id;
  const bool own = at < memory;
  const int c = own ? (int)(at / a.dkp) : 0, d = own ? (int)(at % a.dkp) : 0;
  float* st = reinterpret_cast<float*>(a.state + (int64_t)slot * a.state_stride + a.state_offset);
  float* place = p.place(st, h, c, d);
  const int64_t base = (int64_t)(before + first - t0) * a.H + h;
  float* w = a.ws + base * memory + (own ? at : 0);
  const double2* ends = reinterpret_cast<const double2*>(a.ends) + base;
  float m = p.m(st, h);
  float4 S = *reinterpret_cast<const float4*>(place);
  constexpr int AHEAD = 8;
  for (int i = first; i < end; i += AHEAD) {
    float4 mine[AHEAD];
    double2 e[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int k = min(u, end - 1 - i);
      mine[u] = *reinterpret_cast<const float4*>(w + k * step);
      e[u] = ends[(int64_t)k * a.H];
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (i + u < end) {
        if (own) *reinterpret_cast<float4*>(w + u * step) = S;
        if (P::NORMED && id == 0) before_m[base + (int64_t)(i + u - first) * a.H] = m;
        const float next = P::NORMED ? gc_next_m(e[u], m) : 0.f;
        const float keep = gc_exp(e[u].x + (double)m - (double)next), take = P::NORMED ? gc_exp(e[u].y - (double)next) : 1.f;
        S.x = fmaf(keep, S.x, take * mine[u].x);
        S.y = fmaf(keep, S.y, take * mine[u].y);
        S.z = fmaf(keep, S.z, take * mine[u].z);
        S.w = fmaf(keep, S.w, take * mine[u].w);
        m = next;
      }
    }
    w += AHEAD * step;
    ends += (int64_t)AHEAD * a.H;
  }
  if (own) p.keep(st, h, c, d, S);            // (m is kept by the rows kernel: every workgroup here reads it)
}

// ---- every chunk's rows --------------------------------------------------------------------------------
// One workgroup of four wavefronts a (64 columns, head, chunk), a wavefront 32 rows x 32 columns: the rows' products with the
// keys of the chunk (a square of which the part behind the diagonal is left out) and with the memory before it, block
// by block of 32 key dims; then the square, weighted, on the values.
template <typename T, class P>
__global__ __launch_bounds__(256, P::NORMED ? 3 : 4) void gc_rows_kernel(float* __restrict__ y, GcArgs<T> a, P p, int t0, int nt, const float* __restrict__ before_m) {
  // rows of q, rows of k, columns of the memory; later the square and the values
  __shared__ __attribute__((aligned(16))) float lds[2 * CK_ROWS * GC_LD];
  static_assert(3 * CK_ROWS * GC_KLD <= 2 * CK_ROWS * GC_LD, "the blocks fit where the square and the values will be");
  float* qs = lds;
  float* ks = qs + CK_ROWS * GC_KLD;
  float* ss = ks + CK_ROWS * GC_KLD;
  float* square_s = lds;
  float* vs = lds + CK_ROWS * GC_LD;
  __shared__ double Fs[CK_ROWS];
  __shared__ float ins[CK_ROWS], ms[CK_ROWS], olds[CK_ROWS], dens[CK_ROWS];
  __shared__ __attribute__((aligned(16))) float ns[GC_KB];
  const int h = blockIdx.y, c0 = (int)blockIdx.x * 64;
  const int t = threadIdx.x, wave = t >> 6, l32 = t & 31, hl = (t >> 5) & 1;
  int seq, chunk;
  if (!ck_find(t0 + (int)blockIdx.z, a.cu, a.num_seqs, a.from, seq, chunk)) return;
  if (a.slot[seq] < 0) return;
  const int64_t r0 = a.cu[seq] + (int64_t)chunk * CK_ROWS;
  const int n = min(CK_ROWS, (int)(a.cu[seq + 1] - r0));
  const int i0 = (wave >> 1) * 32, j0 = (wave & 1) * 32;
  const int cols = gc_cols<T, P>(a.dv);
  const int64_t item = (int64_t)blockIdx.z * a.H + h;
  const float* S = a.ws + item * cols * a.dkp;
  const T* qr = a.q + r0 * a.stride + (int64_t)(h / a.per) * a.dk;
  const T* kr = a.k + r0 * a.stride + (int64_t)(h / a.per) * a.dk;
  const T* vr = a.v + r0 * a.stride + (int64_t)h * a.dv;
  if (t < 64) {
    double F, peak;
    float in;
    gc_gates(p, r0, n, h, t, F, in, peak);
    const double m0 = P::NORMED ? (double)before_m[item] : 0.;
    const float m = P::NORMED ? (float)(F + fmax(m0, peak)) : 0.f;
    Fs[t] = F;
    ins[t] = in;
    ms[t] = m;
    olds[t] = gc_exp(F + m0 - (double)m);
  }
  // the sequence's last chunk in the window: its m goes with the S and n that the walk over the chunks has kept, also where the sequence goes
  // on in the next window, whose walk begins with all three
  if (P::NORMED && blockIdx.x == 0 && ((int)blockIdx.z == nt - 1 || (chunk + 1) * CK_ROWS >= a.cu[seq + 1] - a.cu[seq])) {
    const double2 e = *reinterpret_cast<const double2*>(a.ends + 2 * item);
    p.keep_m(reinterpret_cast<float*>(a.state + (int64_t)a.slot[seq] * a.state_stride + a.state_offset), h, gc_next_m(e, before_m[item]), t);
  }
  gc_acc square = {0.f}, out = {0.f}, lost_s = {0.f}, lost_o = {0.f};
  float den = 0.f, lost_d = 0.f;              // NORMED: n . q of row t / 4, this thread's share
  for (int d0 = 0; d0 < a.dkp; d0 += GC_KB) {
    const int d = 4 * (t & 7);
    float4 qx[2], kx[2], sx[2], nx = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = (t >> 3) + 32 * i;
      qx[i] = gc_tile4(qr, a.stride, row, n, d0 + d, a.dk);
      kx[i] = gc_tile4(kr, a.stride, row, n, d0 + d, a.dk);
      sx[i] = gc_tile4(S + (int64_t)c0 * a.dkp, a.dkp, row, a.dv - c0, d0 + d, a.dkp);
    }
    if (P::NORMED) nx = gc_tile4(S + (int64_t)a.dv * a.dkp, 0, 0, 1, d0 + d, a.dkp);
    __syncthreads();                          // (the block before has been read)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int at = ((t >> 3) + 32 * i) * GC_KLD + d;
      *reinterpret_cast<float4*>(qs + at) = make_float4(qx[i].x * a.q_scale, qx[i].y * a.q_scale, qx[i].z * a.q_scale, qx[i].w * a.q_scale);
      *reinterpret_cast<float4*>(ks + at) = kx[i];
      *reinterpret_cast<float4*>(ss + at) = sx[i];
    }
    if (P::NORMED && t < 8) *reinterpret_cast<float4*>(ns + d) = nx;
    __syncthreads();
#pragma unroll 1
    for (int g0 = 0; g0 < GC_KB; g0 += 16) {
      float4 qv[2], kv[2], sv[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int g = g0 + 8 * u + 4 * hl;
        qv[u] = *reinterpret_cast<const float4*>(qs + (i0 + l32) * GC_KLD + g);
        kv[u] = *reinterpret_cast<const float4*>(ks + (j0 + l32) * GC_KLD + g);
        sv[u] = *reinterpret_cast<const float4*>(ss + (j0 + l32) * GC_KLD + g);
      }
      gc_add<P::NORMED>(out, lost_o, gc_mfma4(qv[0], sv[0]), gc_mfma4(qv[1], sv[1]));
      __builtin_amdgcn_sched_barrier(0);
      if (j0 <= i0) gc_add<P::NORMED>(square, lost_s, gc_mfma4(qv[0], kv[0]), gc_mfma4(qv[1], kv[1]));      // (the same in the wavefront)
    }
    if (P::NORMED) {
      float some = 0.f;
#pragma unroll
      for (int e = 0; e < GC_KB / 4; e += 4) {
        const float4 qv = *reinterpret_cast<const float4*>(qs + (t >> 2) * GC_KLD + 8 * (t & 3) + e);
        const float4 nv = *reinterpret_cast<const float4*>(ns + 8 * (t & 3) + e);
        some = fmaf(qv.x, nv.x, fmaf(qv.y, nv.y, fmaf(qv.z, nv.z, fmaf(qv.w, nv.w, some))));
      }
      const float more = some - lost_d, sum = den + more;
      lost_d = (sum - den) - more;
      den = sum;
    }
  }
  float4 vx[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) vx[i] = gc_tile4(vr, a.stride, (t >> 4) + 16 * i, n, c0 + 4 * (t & 15), a.dv);
  float zero = 0.f;                           // (what is not finite shows as NaN)
#pragma unroll
  for (int i = 0; i < 4; ++i) zero = fmaf(vx[i].x, 0.f, fmaf(vx[i].y, 0.f, fmaf(vx[i].z, 0.f, fmaf(vx[i].w, 0.f, zero))));
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) *reinterpret_cast<float4*>(vs + ((t >> 4) + 16 * i) * GC_LD + 4 * (t & 15)) = vx[i];
  {
    const int j = j0 + l32;
    const double Fj = Fs[j];
    const float inj = ins[j];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = i0 + 8 * (r >> 2) + 4 * hl + (r & 3);
      const float e = P::NORMED ? gc_exp(Fs[i] - Fj + (double)inj - (double)ms[i]) : inj * gc_exp(Fs[i] - Fj);
      square_s[i * GC_LD + j] = j <= i && j < n ? e * square[r] : 0.f;
    }
  }
  const bool finite = !__syncthreads_or(!(zero == 0.f));
  if (P::NORMED) {
    float some = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      const float4 s = *reinterpret_cast<const float4*>(square_s + (t >> 2) * GC_LD + 16 * (t & 3) + e);
      some += (s.x + s.y) + (s.z + s.w);
    }
    den = fmaf(den, olds[t >> 2], some);
    den += __shfl_xor(den, 1);
    den += __shfl_xor(den, 2);
    if ((t & 3) == 0) dens[t >> 2] = fmaxf(fabsf(den), expf(-ms[t >> 2])) + 1e-6f;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) square[r] = lost_s[r] = 0.f;      // (from here on the square's share of the result)
#pragma unroll
  for (int g0 = 0; g0 < CK_ROWS; g0 += 16) {
    if (g0 >= i0 + 32 || g0 >= n || !finite) break;      // (the same in the wavefront)
    gc_acc some[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int g = g0 + 8 * u + 4 * hl;
      const float* v = vs + g * GC_LD + j0 + l32;
      some[u] = gc_mfma4(*reinterpret_cast<const float4*>(square_s + (i0 + l32) * GC_LD + g), make_float4(v[0], v[GC_LD], v[2 * GC_LD], v[3 * GC_LD]));
    }
    gc_add<P::NORMED>(square, lost_s, some[0], some[1]);
  }
  if (!finite) {      // a row sees the values up to its own: an infinity behind it, times the square's zero, would be NaN
    for (int j = 0; j < n; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = i0 + 8 * (r >> 2) + 4 * hl + (r & 3);
        if (j <= i) square[r] = fmaf(square_s[i * GC_LD + j], vs[j * GC_LD + j0 + l32], square[r]);
      }
    }
  }
  if (P::NORMED) __syncthreads();
  const int c = c0 + j0 + l32;
  if (c < a.dv) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = i0 + 8 * (r >> 2) + 4 * hl + (r & 3);
      const float sum = fmaf(out[r], olds[i], square[r]);
      if (i < n) y[(r0 + i) * a.H * a.dv + (int64_t)h * a.dv + c] = P::NORMED ? sum / dens[i] : p.result(sum, vs[i * GC_LD + j0 + l32], h);
    }
  }
}

// Whether a step is faster by chunks. The walk of the longest sequence hides those of the others; behind the chunks these stand alone, and
// sequences of GC_FEW to GC_SHORT rows cost there what memory / 65536 rows of the longest one's walk do. (us walked and by chunks, 14 heads of 128 x 256; 64 heads
// of 128 x 64: 70 rows 42 and 34; 29 and 34. 140 rows 73 and 36; 51 and 36. 70 rows beside 7 of one row 46 and 45; 30 and 50. Beside 63 201 and 93; 140 and 144.
// 200 beside 31 of one row 145 and 69; 93 and 92. 70 beside 15 of 40 195 and 106; 109 and 105. 70 beside 31 of 8 143 and 161; 91 and 122.)
static inline bool gc_pays(int rows, int num_seqs, int max_q_len, int64_t memory, const GcLines& lines) {
  const int longest = std::min(rows, max_q_len);
  if (num_seqs == 1) return longest > lines.alone;
  const int others = (rows - longest) / (num_seqs - 1);
  if (others >= lines.others) return longest > GC_FROM;
  return longest > lines.beside + (others > GC_FEW ? (num_seqs - 1) * memory / 65536 : 0);
}

// No fewer than the chunks of a step's sequences: whole ones, and one more of every sequence that has chunks.
static inline int64_t gc_chunks(int rows, int num_seqs) {
  return rows / CK_ROWS + std::min(num_seqs, rows / (gc_from(num_seqs) + 1));
}

// Chunks whose memories are held at once, and the floats of workspace for them: memories, ends and the m before them.
static inline int64_t gc_window(int rows, int num_seqs, int64_t memory) {
  const int64_t chunks = gc_chunks(rows, num_seqs);
  int64_t most = GC_WINDOW_FLOATS / memory;
  if (most > 32768) most = 32768;
  return chunks < most ? chunks : (most < 1 ? 1 : most);
}
static inline int64_t gc_floats(int rows, int num_seqs, int max_q_len, int H, int cols, int dkp, const GcLines& lines) {
  const int64_t memory = (int64_t)H * cols * dkp;
  if (num_seqs <= 0 || !gc_pays(rows, num_seqs, max_q_len, memory, lines)) return 0;
  return gc_window(rows, num_seqs, memory) * (memory + 6ll * H);
}

template <typename T, class P>
static int gc_run(float* y, const GcArgs<T>& args, const P& p, int rows, float* workspace, const char* name, hipStream_t s) {
  GcArgs<T> a = args;
  const int cols = gc_cols<T, P>(a.dv);
  const int64_t memory = (int64_t)a.H * cols * a.dkp;
  const int window = (int)gc_window(rows, a.num_seqs, memory), chunks = (int)gc_chunks(rows, a.num_seqs);
  a.ws = workspace;
  a.ends = reinterpret_cast<double*>(a.ws + window * memory);      // (a memory is whole fours)
  float* before_m = reinterpret_cast<float*>(a.ends + 2ll * window * a.H);
  const int kb = (a.dkp + 63) / 64, vb = (a.dv + 63) / 64;
  for (int t0 = 0; t0 < chunks; t0 += window) {
    const int nt = chunks - t0 < window ? chunks - t0 : window;
    gc_share_kernel<T, P><<<dim3(kb * vb, a.H, nt), 256, 0, s>>>(a, p, t0);
    gc_carry_kernel<T, P><<<dim3((unsigned)((memory / a.H / 4 + 255) / 256), a.H, a.num_seqs), 256, 0, s>>>(a, p, t0, nt, before_m);
    gc_rows_kernel<T, P><<<dim3(vb, a.H, nt), 256, 0, s>>>(y, a, p, t0, nt, before_m);
  }
  return he_check_launch(name);
}

// Whole fours of every row and head, which the kernels above load at once. (Head sizes that are none are not given a workspace either.)
static inline bool gc_heads(int dk, int dv) { return dk % 4 == 0 && dv % 4 == 0; }
template <typename T>
static inline bool gc_takes(const GcArgs<T>& a) {
  return gc_heads(a.dk, a.dv) && a.stride % 4 == 0 && a.H <= 65535 && a.num_seqs <= 65535 &&
         (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v) & (4 * sizeof(T) - 1)) == 0;
}
