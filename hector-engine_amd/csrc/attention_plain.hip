// Plain attention over the paged cache in fp32, in one fixed order per (query, head): the keys
// are taken page by page (64 positions, by absolute position), inside a page one by one in
// ascending position with an online softmax begun afresh, and the pages' results (m, l, sums)
// are joined one after the other in ascending position. The result for a query depends only on
// its own position and the cache rows [first, p], never on how the step was cut or batched, so
// prompt steps and one-token steps give identical bits. It is the 32-bit path's attention and
// the reference beside the MFMA kernels.
//
// For the query at absolute position p: first = window > 0 ? max(0, p+1-window) : 0, and with
// chunk > 0 no earlier than the start of p's chunk, p - p % chunk (chunks are counted from position 0);
// s_j = (q . k_j) * scale for j in [first, p], out = sum_j softmax(s)_j v_j,
// kv head = h / (H / KVH)   (reference: kernels/attention.cu:155-316, :664-773, :60).
// sinks (one number a head, or null): the softmax's denominator also holds exp(sink_h), which has no
// key and no value; it joins last, after the pages. A score may fall with the distance by a slope a head, or be
// capped and then shifted by a table a head over the distance (ap_shape). gate (one number a row and head, or null): the
// head's output is multiplied by sigmoid(gate) before it is stored.
//
// (32-bit caches with head sizes of 32, 64, 96 or 128 have an order of their own, on the matrix cores: further down.)
//
// Three launches keep that order and give the same bits: one wavefront per (query, head) that walks
// the pages itself (or, in a step of many queries, per four neighbouring queries, which share what
// they fetch); or, for steps of few queries over many keys (one-token steps), a wavefront
// per (query, head, page) that leaves its page's result in a workspace, and a second kernel that
// joins them in order (one wavefront alone would walk thousands of keys while the chip idles:
// a one-token step of 28 heads over 2,048 keys took 2.4 ms so).
// No multiply and add of this file is fused unless it is written as an fma: the same lines are
// compiled into several kernels that must give the same bits.
#pragma clang fp contract(off)
#include "cache_layout.h"
#include "hector_kernels.h"

#define AP_MAX_PER_LANE 16

// the first key the query at position p sees
__device__ __forceinline__ int ap_first(int p, int window, int chunk) {
  int first = window > 0 ? max(0, p + 1 - window) : 0;
  if (chunk > 0) first = max(first, p - p % chunk);
  return first;
}

// NPL: head elements a lane holds (head_dim / 64 rounded up to 1, 2, 4, 8 or 16)
template <int NPL>
struct ApState {
  float m, l;
  float acc[NPL];
};

// The score of one key: k holds this lane's elements of the key. It does not depend on the keys
// before it, so the scores of a group of keys are computed side by side ahead of the chain below.
template <int NPL>
__device__ __forceinline__ float ap_score(const float (&qv)[NPL], const float (&k)[NPL], float scale, int lane,
                                          int npl, int hd) {
  float part = 0.f;
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const int d = lane + i * HE_WAVE;
    if (i < npl && d < hd) part = fmaf(qv[i], k[i], part);
  }
  return wave_sum(part) * scale;
}

// One key joins the running softmax of a page: s is its score, v this lane's elements of its value.
// Of the two weights exp(m - m_new) and exp(s - m_new) one is exp(0) = 1: one exponential a key.
template <int NPL>
__device__ __forceinline__ void ap_update(ApState<NPL>& st, float s, const float (&v)[NPL], int lane, int npl,
                                          int hd) {
  const bool up = s > st.m;                 // the reference point moves to s
  const float m_new = up ? s : st.m;
  const float e = expf(up ? st.m - s : s - st.m);
  const float alpha = up ? e : 1.f;
  const float w = up ? 1.f : s == -INFINITY ? 0.f : e;      // (also where no key had weight yet: there e is exp(-inf + inf))
  st.l = fmaf(st.l, alpha, w);
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const int d = lane + i * HE_WAVE;
    if (i < npl && d < hd) st.acc[i] = fmaf(st.acc[i], alpha, w * v[i]);
  }
  st.m = m_new;
}

// What shapes a score beyond q . k * scale: a slope over the distance, or a cap and a table over the distance (of this head).
struct ApShape {
  float slope, cap;
  const float* table;    // the head's entries, or null
  int last;              // the table's last index
};
// the score of a key `back` positions before the query (negative: a key the caller leaves out)
__device__ __forceinline__ float ap_shape(const ApShape& sh, float s, int back) {
  if (sh.cap > 0.f) s = sh.cap * tanhf(s / sh.cap);
  if (sh.table != nullptr) return s + sh.table[min(max(back, 0), sh.last)];
  return fmaf(sh.slope, (float)-back, s);
}

#define AP_GROUP 4
// The key and value elements of this lane for the AP_GROUP keys from j0 on (positions beyond j_hi
// read key j_hi again: no load stands behind a condition, so the compiler counts what is in flight).
template <typename T, int NPL>
__device__ __forceinline__ void ap_fetch(float (&kv)[AP_GROUP][NPL], float (&vv)[AP_GROUP][NPL], const T* kpage,
                                         const T* vpage, int j0, int j_hi, int KS, int NT, int lane, int npl,
                                         int hd) {
#pragma unroll
  for (int g = 0; g < AP_GROUP; ++g) {
    const int off = min(j0 + g, j_hi) & (HE_PAGE_TOKENS - 1);
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      const int d = lane + i * HE_WAVE;
      const bool has = i < npl && d < hd;
      kv[g][i] = has ? to_float(kpage[he_k_index(off, d, KS)]) : 0.f;
      vv[g][i] = has ? to_float(vpage[he_v_index(off, d, NT)]) : 0.f;
    }
  }
}

// The online softmax of the keys [j_lo, j_hi] of one page (they lie in the same page), begun afresh.
// Every multiply-add is written out as an fma: these lines are compiled into several kernels,
// and the compiler would otherwise be free to fuse each copy its own way.
template <typename T, int NPL>
__device__ __forceinline__ void ap_page(ApState<NPL>& st, const float (&qv)[NPL], const T* kpool,
                                        const T* vpool, int page, int num_pages, int KVH, int kvh, int hd,
                                        int j_lo, int j_hi, float scale, int lane, int npl, const ApShape& sh,
                                        int p) {
  st.m = -INFINITY;
  st.l = 0.f;
#pragma unroll
  for (int i = 0; i < NPL; ++i) st.acc[i] = 0.f;
  if (page < 0 || page >= num_pages) return;  // never for an admitted batch
  // the pages are stored in the MFMA kernels' operand order (cache_layout.h)
  const T* kpage = kpool + ((int64_t)page * KVH + kvh) * he_k_page_elems(hd);
  const T* vpage = vpool + ((int64_t)page * KVH + kvh) * he_v_page_elems(hd);
  const int KS = he_k_steps(hd), NT = he_v_tiles(hd);
  // Four keys at a time, in two sets of registers: while the chain of the softmax takes the keys of
  // one set one by one in ascending position, the elements of the next four are on their way (a key
  // at a time, each load was waited for before the next was asked for: 1 us a key; four at a time
  // without the second set, a wait of its own for every four: a page of 64 keys 39 us).
  float ka[AP_GROUP][NPL], va[AP_GROUP][NPL], kb[AP_GROUP][NPL], vb[AP_GROUP][NPL];
  ap_fetch<T, NPL>(ka, va, kpage, vpage, j_lo, j_hi, KS, NT, lane, npl, hd);
  for (int j0 = j_lo; j0 <= j_hi; j0 += 2 * AP_GROUP) {
    ap_fetch<T, NPL>(kb, vb, kpage, vpage, j0 + AP_GROUP, j_hi, KS, NT, lane, npl, hd);
    float sc[AP_GROUP];
#pragma unroll
    for (int g = 0; g < AP_GROUP; ++g)
      sc[g] = ap_shape(sh, ap_score<NPL>(qv, ka[g], scale, lane, npl, hd), p - (j0 + g));
#pragma unroll
    for (int g = 0; g < AP_GROUP; ++g)
      if (j0 + g <= j_hi) ap_update<NPL>(st, sc[g], va[g], lane, npl, hd);
    ap_fetch<T, NPL>(ka, va, kpage, vpage, j0 + 2 * AP_GROUP, j_hi, KS, NT, lane, npl, hd);
#pragma unroll
    for (int g = 0; g < AP_GROUP; ++g)
      sc[g] = ap_shape(sh, ap_score<NPL>(qv, kb[g], scale, lane, npl, hd), p - (j0 + AP_GROUP + g));
#pragma unroll
    for (int g = 0; g < AP_GROUP; ++g)
      if (j0 + AP_GROUP + g <= j_hi) ap_update<NPL>(st, sc[g], vb[g], lane, npl, hd);
  }
}

// total <- total joined with the result of the next page (one that had keys). A page whose scores are all -inf has a sum of 0 and
// is passed over; scores that are no numbers leave a sum that is none, which joins and stays visible.
template <int NPL>
__device__ __forceinline__ void ap_join(ApState<NPL>& total, const ApState<NPL>& st) {
  if (!(st.m > -INFINITY) && st.l == 0.f) return;
  const float m_new = fmaxf(total.m, st.m);
  const float a = total.m > -INFINITY ? expf(total.m - m_new) : 0.f;
  const float b = expf(st.m - m_new);
  total.l = fmaf(total.l, a, st.l * b);
#pragma unroll
  for (int i = 0; i < NPL; ++i) total.acc[i] = fmaf(total.acc[i], a, st.acc[i] * b);
  total.m = m_new;
}

// What a (row, head) is finished with: the sink joins the softmax, the gate scales the output.
struct ApExtras {
  const void* sinks;     // [H] or null
  int sinks_dtype;
  const void* gate;      // gate[row * gate_stride + h] in the activation dtype, or null
  int64_t gate_stride;
  const float* slopes;   // [H] or null: the score of key j for the query at p loses slopes[h] * (p - j)
  const float* table;    // [H][table_len] or null: the score gains table[h][min(p - j, table_len - 1)]
  int table_len;
  float cap;             // > 0: a score s becomes cap * tanh(s / cap) first
};
__device__ __forceinline__ ApShape ap_shape_of(const ApExtras& ex, int h) {
  return ApShape{ex.slopes ? ex.slopes[h] : 0.f, ex.cap, ex.table ? ex.table + (int64_t)h * ex.table_len : nullptr,
                 ex.table_len - 1};
}
template <typename T, int NPL>
__device__ __forceinline__ float ap_finish(ApState<NPL>& total, const ApExtras& ex, int64_t row, int h) {
  if (ex.sinks != nullptr) {
    ApState<NPL> sk;
    sk.m = load_param(ex.sinks, h, ex.sinks_dtype);
    sk.l = sk.m > -INFINITY ? 1.f : 0.f;         // a sink of -inf (or none that is a number) is passed over
#pragma unroll
    for (int i = 0; i < NPL; ++i) sk.acc[i] = 0.f;
    ap_join(total, sk);
  }
  if (ex.gate == nullptr) return 1.f;
  const float g = to_float(((const T*)ex.gate)[row * ex.gate_stride + h]);
  return 1.f / (1.f + expf(-g));
}

// ---- 32-bit caches with head sizes of 32, 64, 96 or 128: both products on the matrix cores -------------------------
//
// A chain of v_mfma_f32_16x16x4_f32 on one accumulator is, bit for bit, a chain of FMAs over its k, so a fixed order
// of the products costs nothing there. The order of a (query, head), the same in every launch: a score is the sum,
// over ks, of (c0 + c1) + (c2 + c3), c the chain of the 8 dims 32 ks + 8 g + 2 c + e in the order of (e, g) (one chain of 128
// would round more often than sums across a wavefront's lanes do: against 64 bits it is off by 3.1e-7 of the output's norm instead of
// 2.8e-7, as such sums gave, at 1003 keys); a page's scores are taken off their maximum together, the sum of
// the exponentials is, for each g, that of the keys 32 h + 8 g + 4 t + i in the order of (h, t, i), then (0 + 1) + (2 + 3)
// over g; a value dim is one chain over the keys 32 h + 8 g + e in the order of (h, e, g); the pages are joined one
// after the other as above. These orders are the pages' own layout (cache_layout.h): a lane's operands are the eight
// consecutive elements it fetches, and the scores a lane holds (S^T = K Q^T: its column is a query, its rows are keys)
// are the operand of O^T = V^T P^T as they are. Nothing goes through LDS.
//
// A key a query does not see has weight zero; where some value of the page is not finite and some query of the tile
// does not see all of the page (or the page is not held, never for an admitted batch), the page's values are added key by key without the keys a query does not see (0 times
// infinity would reach it). Values of keys beyond the tile's last position are taken as zero (nothing was written there).
typedef float ap_f4 __attribute__((ext_vector_type(4)));
template <int KS>
struct ApPage32 {      // one page's operands as fetched: [half][key tile][k step][two pieces], [half][dim tile][two pieces]
  ap_f4 k[2][2][KS][2];
  ap_f4 v[2][2 * KS][2];
};
// A page is fetched through a buffer descriptor of its own: the address is one register, a scalar offset and an immediate
// (as 64-bit pointers the addresses of a page's 64 loads took registers that its elements need).
__device__ __forceinline__ ap_f4 ap32_load(__amdgpu_buffer_rsrc_t page, int lane, int piece) {
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
  const u4 r = __builtin_amdgcn_raw_buffer_load_b128(page, lane * 32, piece * 16, 0);
  return __builtin_bit_cast(ap_f4, r);
}
template <int KS>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ap32_rsrc(const float* page) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)page, 0, HE_PAGE_TOKENS * 32 * KS * 4, 0x00027000);
}
template <int KS>
__device__ __forceinline__ void ap32_fetch_k(ApPage32<KS>& pg, __amdgpu_buffer_rsrc_t kpage, int h, int lane) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int b = 0; b < 2; ++b) pg.k[h][t][ks][b] = ap32_load(kpage, lane, ((h * 2 + t) * KS + ks) * 128 + b);
}
template <int KS>
__device__ __forceinline__ void ap32_fetch_v(ApPage32<KS>& pg, __amdgpu_buffer_rsrc_t vpage, int h, int lane) {
#pragma unroll
  for (int dt = 0; dt < 2 * KS; ++dt)
#pragma unroll
    for (int b = 0; b < 2; ++b) pg.v[h][dt][b] = ap32_load(vpage, lane, (h * 2 * KS + dt) * 128 + b);
}
// 16 queries: the lane's column is query lane % 16
template <int KS>
struct ApTile32 {
  ap_f4* q;              // LDS: the lane's dims 32 ks + 8 g + 4 b .. + 3 of its query at (2 ks + b) 64
  ap_f4* total;          // LDS: dims 16 dt + 4 g .. + 3 of the sums so far at 64 dt
  float m, l;
  int p, first;          // the keys the column sees: [first, p] (p < first: no query)
  ApShape sh;
};
// The page whose first key is j0 joins the tile; pg holds its keys on entry and, with NEXT, those of next_k on return (not
// under a condition: registers that may keep their old keys would be held through the page). last: no key beyond it has been
// written. whole: every column sees all of it. With NEXT a page's halves of 32 keys take turns in the registers, so that
// two wavefronts fit a SIMD (one's products beside the other's softmax and waits): a half's values are asked for
// behind its scores, a half of the next page's keys behind its value products. Without it all values come before the scores.
template <int KS, bool NEXT, bool SHAPED>
__device__ __forceinline__ void ap32_page(ApTile32<KS>& t, ApPage32<KS>& pg, const float* vpage_at, const float* next_k_at,
                                          bool held, int j0, int last, bool whole, float scale, int lane) {
  const int g = lane >> 4;
  const __amdgpu_buffer_rsrc_t vpage = ap32_rsrc<KS>(vpage_at), next_k = ap32_rsrc<KS>(next_k_at);
  ap_f4 s[2][2];
  if (!NEXT) ap32_fetch_v<KS>(pg, vpage, 0, lane), ap32_fetch_v<KS>(pg, vpage, 1, lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      ap_f4 part[4][2];
      const ap_f4 qv[2] = {t.q[2 * ks * HE_WAVE], t.q[(2 * ks + 1) * HE_WAVE]};
#pragma unroll
      for (int e = 0; e < 2; ++e)      // (the eight chains in turn: an instruction does not wait for the one before it)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const int d = 2 * (c & 1) + e;
            part[c][x] = __builtin_amdgcn_mfma_f32_16x16x4f32(pg.k[h][x][ks][c >> 1][d], qv[c >> 1][d],
                                                              e == 0 ? ap_f4{0.f, 0.f, 0.f, 0.f} : part[c][x], 0, 0, 0);
          }
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float all = (part[0][x][i] + part[1][x][i]) + (part[2][x][i] + part[3][x][i]);
          s[h][x][i] = ks == 0 ? all : s[h][x][i] + all;
        }
      __builtin_amdgcn_sched_barrier(0);      // (the parts of several k steps at once would not fit the registers)
    }
    __builtin_amdgcn_sched_barrier(0);
    if (NEXT) ap32_fetch_v<KS>(pg, vpage, h, lane);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (SHAPED) {      // (as ap_shape, a kind at a time and a score at a time: what all of them would need at once does not fit the registers)
#define AP32_EACH(V_, ...)                                               \
  _Pragma("unroll") for (int h = 0; h < 2; ++h)                          \
      _Pragma("unroll") for (int x = 0; x < 2; ++x)                      \
          _Pragma("unroll") for (int i = 0; i < 4; ++i) {                \
    const int back = t.p - (j0 + 32 * h + 8 * g + 4 * x + i);            \
    (void)back;                                                          \
    float V_ = s[h][x][i];                                               \
    __VA_ARGS__;                                                         \
    s[h][x][i] = V_;                                                     \
    __builtin_amdgcn_sched_barrier(0);                                   \
  }
    AP32_EACH(v, v = v * scale)
    if (t.sh.cap > 0.f) AP32_EACH(v, v = t.sh.cap * tanhf(v / t.sh.cap))
    if (t.sh.table != nullptr) AP32_EACH(v, v = v + t.sh.table[min(max(back, 0), t.sh.last)])
    else AP32_EACH(v, v = fmaf(t.sh.slope, (float)-back, v))
#undef AP32_EACH
  }
  float top = -INFINITY;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = j0 + 32 * h + 8 * g + 4 * x + i;
        const float v = SHAPED ? s[h][x][i] : s[h][x][i] * scale;
        s[h][x][i] = held && j >= t.first && j <= t.p ? v : -INFINITY;
        top = fmaxf(top, s[h][x][i]);
      }
  top = fmaxf(top, __shfl_xor(top, 16));
  top = fmaxf(top, __shfl_xor(top, 32));
  const float off = top > -INFINITY ? top : 0.f;
  float sum = 0.f;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v = s[h][x][i];
        const float w = v == top && top > -INFINITY ? 1.f : expf(v - off);
        s[h][x][i] = w;
        sum += w;
      }
  const float l = xor32_sum(xor16_sum(sum));
  ap_f4 acc[2 * KS];
#pragma unroll
  for (int dt = 0; dt < 2 * KS; ++dt) acc[dt] = ap_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    bool by_key = false;
    if (!whole) {
      float none = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int dt = 0; dt < 2 * KS; ++dt) {
          const float v = j0 + 32 * h + 8 * g + e > last ? 0.f : pg.v[h][dt][e >> 2][e & 3];
          pg.v[h][dt][e >> 2][e & 3] = v;
          none = fmaf(v, 0.f, none);
        }
      by_key = __any(none != 0.f);
    }
    if (!by_key) {
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int dt = 0; dt < 2 * KS; ++dt)
          acc[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(pg.v[h][dt][e >> 2][e & 3], s[h][e >> 2][e & 3], acc[dt], 0, 0, 0);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma nounroll
        for (int gg = 0; gg < 4; ++gg) {
          int own = g;
          asm volatile("" : "+v"(own));      // (the addresses of this rare path are not kept in registers all along)
          const int key = 32 * h + 8 * gg + e;
          const float w = __shfl(s[h][e >> 2][e & 3], (lane & 15) + 16 * gg);
          if (held && j0 + key >= t.first && j0 + key <= t.p) {
#pragma unroll
            for (int dt = 0; dt < 2 * KS; ++dt)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                acc[dt][i] = fmaf(vpage_at[he_v_index(key, 16 * dt + 4 * own + i, 2 * KS)], w, acc[dt][i]);
          }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (NEXT) ap32_fetch_k<KS>(pg, next_k, h, lane);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (top > -INFINITY || l != 0.f) {                // as ap_join
    const float m_new = fmaxf(t.m, top);
    const float a = t.m > -INFINITY ? expf(t.m - m_new) : 0.f;
    const float b = expf(top - m_new);
    t.l = fmaf(t.l, a, l * b);
#pragma unroll
    for (int dt = 0; dt < 2 * KS; ++dt) {
      ap_f4 v = t.total[dt * HE_WAVE];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = fmaf(v[i], a, acc[dt][i] * b);
      t.total[dt * HE_WAVE] = v;
    }
    t.m = m_new;
  }
}
template <int KS>
__device__ __forceinline__ void ap32_begin(ApTile32<KS>& t, const float* qrow, bool has, int lane) {
  const int g = lane >> 4;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int b = 0; b < 2; ++b)
      t.q[(2 * ks + b) * HE_WAVE] = has ? *reinterpret_cast<const ap_f4*>(qrow + 32 * ks + 8 * g + 4 * b) : ap_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int dt = 0; dt < 2 * KS; ++dt) t.total[dt * HE_WAVE] = ap_f4{0.f, 0.f, 0.f, 0.f};
  t.m = -INFINITY;
  t.l = 0.f;
}
template <int KS>
__device__ __forceinline__ void ap32_store(ApTile32<KS>& t, float* o, const ApExtras& ex, int64_t row, int h, int lane) {
  // the sink joins last; the gate scales what is stored
  float gf = 1.f, a = 1.f;
  const float sink = ex.sinks != nullptr ? load_param(ex.sinks, h, ex.sinks_dtype) : -INFINITY;
  const bool sinks = sink > -INFINITY;            // (as ap_finish)
  if (sinks) {
    const float m_new = fmaxf(t.m, sink);
    a = t.m > -INFINITY ? expf(t.m - m_new) : 0.f;
    t.l = fmaf(t.l, a, expf(sink - m_new));
  }
  if (ex.gate != nullptr) gf = 1.f / (1.f + expf(-((const float*)ex.gate)[row * ex.gate_stride + h]));
  const float inv = t.l > 0.f ? 1.f / t.l : 0.f;
#pragma unroll
  for (int dt = 0; dt < 2 * KS; ++dt) {
    ap_f4 v = t.total[dt * HE_WAVE];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (sinks) v[i] = fmaf(v[i], a, 0.f);
      v[i] = ex.gate ? v[i] * inv * gf : v[i] * inv;
    }
    *reinterpret_cast<ap_f4*>(o + 16 * dt + 4 * (lane >> 4)) = v;
  }
}

// Rows of an aligned group of 16 that are neighbours in one sequence are a run; runs of at least AP32_RUN rows go through
// the kernel for many queries, the others through the kernel for one.
#define AP32_TILE 16
#define AP32_RUN 8
// bit i: row r0 + i begins a run (r0 the group's first row; rows beyond the step begin one each)
__device__ __forceinline__ uint32_t ap32_runs(const int32_t* row_seq, const int32_t* positions, int r0, int rows, int lane) {
  const int r = r0 + (lane & 15);
  const int seq = r < rows ? row_seq[r] : -1, p = r < rows ? positions[r] : 0;
  const int seq_before = __shfl_up(seq, 1), p_before = __shfl_up(p, 1);
  const bool begins = (lane & 15) == 0 || seq < 0 || seq != seq_before || p != p_before + 1;
  return (uint32_t)__ballot(begins) & 0xffffu;
}
__device__ __forceinline__ int ap32_run_end(uint32_t begins, int i) {      // the first row behind the run that row i is in
  const uint32_t later = begins & ~((2u << i) - 1u);
  return later ? __ffs(later) - 1 : AP32_TILE;
}
__device__ __forceinline__ int ap32_run_begin(uint32_t begins, int i) { return 31 - __clz(begins & ((2u << i) - 1u)); }

// Many queries: a wavefront takes 16 rows of one head, run by run. grid (ceil(rows / 16), ceil(H / 4)), the last rows (the most
// keys) first; a workgroup's wavefronts walk the same pages for neighbouring heads. Per page 256 instructions of 32 cycles
// on the matrix cores (head size 128) beside the softmax of the other wavefront of the SIMD. 1003 tokens, 28 heads of 128:
// 202 us a layer; 1850 with a wavefront's lanes along the dims and a sum across the wavefront for every score.
template <int KS, bool SHAPED>
__global__ __launch_bounds__(256, 2) void attention_f32_rows_kernel(
    float* __restrict__ out, const float* __restrict__ q, const float* __restrict__ kpool, const float* __restrict__ vpool,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ row_seq, const int32_t* __restrict__ seq_slot,
    const int32_t* __restrict__ page_table, int max_blocks, int num_pages, int rows, int H, int KVH, int window, int chunk,
    float scale, ApExtras ex) {
  constexpr int hd = 32 * KS;
  const int lane = threadIdx.x & (HE_WAVE - 1);
  const int h = blockIdx.y * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (h >= H) return;
  const int r0 = (gridDim.x - 1 - blockIdx.x) * AP32_TILE;
  const int kvh = h / (H / KVH);
  __shared__ ap_f4 own[4][KS * 4 * HE_WAVE];    // queries and sums (each wavefront's own, each lane its own places of it)
  const uint32_t begins = ap32_runs(row_seq, positions, r0, rows, lane);
  for (int i0 = 0; i0 < AP32_TILE && r0 + i0 < rows;) {
    const int i1 = ap32_run_end(begins, i0);
    const int seq = row_seq[r0 + i0];
    const int begin = i0;
    i0 = i1;
    if (seq < 0 || i1 - begin < AP32_RUN) continue;
    const int p0 = positions[r0 + begin], p_last = p0 + (i1 - begin) - 1;
    ApTile32<KS> t;
    t.q = own[threadIdx.x >> 6] + lane;
    t.total = t.q + 2 * KS * HE_WAVE;
    const int c = lane & 15;
    const bool has = c >= begin && c < i1;
    t.p = has ? p0 + c - begin : -1;
    t.first = has ? ap_first(t.p, window, chunk) : 0;
    t.sh = ap_shape_of(ex, h);
    ap32_begin<KS>(t, q + ((int64_t)(r0 + (has ? c : begin)) * H + h) * hd, has, lane);
    const int32_t* pt = page_table + (int64_t)seq_slot[seq] * max_blocks;
    const int first = ap_first(p0, window, chunk);      // (first never falls along a run)
    const int first_last = ap_first(p_last, window, chunk);
    const int c0 = first >> HE_PAGE_SHIFT, c1 = p_last >> HE_PAGE_SHIFT;
    ApPage32<KS> pg;
    int page = __builtin_amdgcn_readfirstlane(pt[c0]);
    bool held = page >= 0 && page < num_pages;          // always, for an admitted batch
    const int64_t elems = 32 * KS * HE_PAGE_TOKENS;
    for (int half = 0; half < 2; ++half)
      ap32_fetch_k<KS>(pg, ap32_rsrc<KS>(kpool + ((held ? page : 0) * (int64_t)KVH + kvh) * elems), half, lane);
    for (int b = c0; b <= c1; ++b) {
      const float* vpage = vpool + ((held ? page : 0) * (int64_t)KVH + kvh) * elems;
      const int next = __builtin_amdgcn_readfirstlane(pt[min(b + 1, c1)]);
      const bool next_held = next >= 0 && next < num_pages;
      const float* next_k = kpool + ((next_held ? next : 0) * (int64_t)KVH + kvh) * elems;
      const int j0 = b << HE_PAGE_SHIFT;
      // (a column without a query sees nothing of any page: the sums it takes part in are not stored)
      const bool whole = held && j0 >= first_last && j0 + HE_PAGE_TOKENS - 1 <= p0;
      ap32_page<KS, true, SHAPED>(t, pg, vpage, next_k, held, j0, p_last, whole, scale, lane);
      page = next;
      held = next_held;
    }
    if (has) ap32_store<KS>(t, out + ((int64_t)(r0 + c) * H + h) * hd, ex, r0 + c, h, lane);
  }
}

// One query: a wavefront takes one row and up to 16 heads of one kv head (its columns), and all pages or (SPLIT: a page's result
// goes to ws as attention_plain_kernel's does) every parts-th of them. Rows of long runs are left out where the kernel above takes
// them (runs_elsewhere). A unit is a wavefront: rows x kv heads x tiles of 16 heads x parts, the parts in the outermost order, so that the units with pages
// come first and lie on all L2 domains (parts innermost, 64 of them: four of eight domains had work). Units without
// a page of their own leave at once, but each holds its registers and LDS through three dependent loads: a step that
// replays a graph is launched for the most keys it may have, and a unit a page of those took 58 us where 32 sequences of 8
// keys, 16 heads on 16, may have 4200; parts that fill the chip take 18, and at 1000 keys
// 130 where those took 188.
// 4 sequences of about 700 keys, 28 heads of 128 on 4: 14.1 us, 38 with a wavefront a head.
template <int KS, bool SPLIT, bool SHAPED>
__global__ __launch_bounds__(256, SPLIT && KS >= 3 ? 1 : 2) void attention_f32_one_kernel(
    float* __restrict__ out, float* __restrict__ ws, const float* __restrict__ q, const float* __restrict__ kpool,
    const float* __restrict__ vpool, const int32_t* __restrict__ positions, const int32_t* __restrict__ row_seq,
    const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ page_table, int max_blocks, int num_pages, int rows,
    int H, int KVH, int window, int chunk, float scale, int pages, int parts, int runs_elsewhere, ApExtras ex) {
  constexpr int hd = 32 * KS;
  const int lane = threadIdx.x & (HE_WAVE - 1);
  const int group = H / KVH, tiles = (group + 15) / 16;
  int64_t unit = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = (int)(unit % tiles);
  unit /= tiles;
  const int kvh = (int)(unit % KVH);
  unit /= KVH;
  const int row = (int)(unit % rows), z = (int)(unit / rows);
  if (z >= parts) return;
  const int col = 16 * tile + (lane & 15);
  const bool has = col < group;
  const int h = kvh * group + min(col, group - 1);
  float* o = out + ((int64_t)row * H + h) * hd;
  const int seq = row_seq[row];
  if (seq < 0) {
    if (!SPLIT && has)
#pragma unroll
      for (int dt = 0; dt < 2 * KS; ++dt) *reinterpret_cast<ap_f4*>(o + 16 * dt + 4 * (lane >> 4)) = ap_f4{0.f, 0.f, 0.f, 0.f};
    return;
  }
  if (runs_elsewhere) {
    const int r0 = row & ~(AP32_TILE - 1);
    const uint32_t begins = ap32_runs(row_seq, positions, r0, rows, lane);
    if (ap32_run_end(begins, row - r0) - ap32_run_begin(begins, row - r0) >= AP32_RUN) return;
  }
  const int p = positions[row];
  const int first = ap_first(p, window, chunk);
  const int c0 = first >> HE_PAGE_SHIFT, c1 = min(p >> HE_PAGE_SHIFT, SPLIT ? c0 + pages - 1 : 0x7fffffff);
  if (SPLIT && c0 + z > c1) return;
  const int32_t* pt = page_table + (int64_t)seq_slot[seq] * max_blocks;
  extern __shared__ ap_f4 own_of_each[];         // [wavefronts][KS * 4 * HE_WAVE]
  ApTile32<KS> t;
  t.q = own_of_each + (threadIdx.x >> 6) * (KS * 4 * HE_WAVE) + lane;
  t.total = t.q + 2 * KS * HE_WAVE;
  t.p = has ? p : -1;
  t.first = has ? first : 0;
  t.sh = ap_shape_of(ex, h);
  ApPage32<KS> pg;
  const int64_t elems = 32 * KS * HE_PAGE_TOKENS;
  const int step = SPLIT ? parts : 1;
  int page = __builtin_amdgcn_readfirstlane(pt[c0 + z]);
  bool held = page >= 0 && page < num_pages;
  auto fetch_k = [&] {
    for (int half = 0; half < 2; ++half)
      ap32_fetch_k<KS>(pg, ap32_rsrc<KS>(kpool + ((held ? page : 0) * (int64_t)KVH + kvh) * elems), half, lane);
  };
  fetch_k();
  ap32_begin<KS>(t, q + ((int64_t)row * H + h) * hd, has, lane);
  for (int c = c0 + z;;) {
    const float* vpage = vpool + ((held ? page : 0) * (int64_t)KVH + kvh) * elems;
    const int next = __builtin_amdgcn_readfirstlane(pt[min(c + step, c1)]);
    const bool next_held = next >= 0 && next < num_pages;
    const float* next_k = kpool + ((next_held ? next : 0) * (int64_t)KVH + kvh) * elems;
    const int j0 = c << HE_PAGE_SHIFT;
    const bool whole = held && j0 >= first && j0 + HE_PAGE_TOKENS - 1 <= p;
    ap32_page<KS, !SPLIT, SHAPED>(t, pg, vpage, next_k, held, j0, p, whole, scale, lane);
    page = next;
    held = next_held;
    if (SPLIT) {
      float* w = ws + (((int64_t)row * H + h) * pages + (c - c0)) * (hd + 2);
#pragma unroll
      for (int dt = 0; dt < 2 * KS; ++dt) {
        if (has)
#pragma unroll
          for (int i = 0; i < 4; ++i) w[16 * dt + 4 * (lane >> 4) + i] = t.total[dt * HE_WAVE][i];
        t.total[dt * HE_WAVE] = ap_f4{0.f, 0.f, 0.f, 0.f};
      }
      if (has && lane < 16) w[hd] = t.m, w[hd + 1] = t.l;
      t.m = -INFINITY;
      t.l = 0.f;
    }
    c += step;
    if (c > c1) break;
    if (SPLIT) fetch_k();
  }
  if (SPLIT || !has) return;
  ap32_store<KS>(t, o, ex, row, h, lane);
}

// grid (rows, ceil(H / 4), pages): pages == 1: the wavefront walks all pages of its query and stores
// the result; pages > 1: it takes the page (first >> 6) + blockIdx.z alone and stores (m, l, sums)
// into ws [row][head][pages][hd + 2], if the query has such a page.
template <typename T, int NPL>
__global__ __launch_bounds__(256) void attention_plain_kernel(
    T* __restrict__ out, float* __restrict__ ws, const T* __restrict__ q, const T* __restrict__ kpool,
    const T* __restrict__ vpool, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ row_seq, const int32_t* __restrict__ seq_slot,
    const int32_t* __restrict__ page_table, int max_blocks, int num_pages, int H, int KVH, int hd,
    int window, int chunk, float scale, ApExtras ex) {
  const int lane = threadIdx.x & (HE_WAVE - 1);
  const int h = blockIdx.y * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int64_t row = blockIdx.x;
  if (h >= H) return;
  const bool split = gridDim.z > 1;
  T* o = out + (row * H + h) * (int64_t)hd;
  const int seq = row_seq[row];
  const int npl = (hd + HE_WAVE - 1) / HE_WAVE;
  if (seq < 0) {
    if (!split)
      for (int i = 0; i < npl; ++i) {
        const int d = lane + i * HE_WAVE;
        if (d < hd) o[d] = from_float<T>(0.f);
      }
    return;
  }
  const int p = positions[row];
  const int slot = seq_slot[seq];
  const int kvh = h / (H / KVH);
  const ApShape sh = ap_shape_of(ex, h);
  const int first = ap_first(p, window, chunk);
  const int32_t* pt = page_table + (int64_t)slot * max_blocks;
  const int c_first = first >> HE_PAGE_SHIFT, c_last = p >> HE_PAGE_SHIFT;
  if (split && c_first + (int)blockIdx.z > c_last) return;

  float qv[NPL];
  const T* qrow = q + (row * H + h) * (int64_t)hd;
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const int d = lane + i * HE_WAVE;
    qv[i] = (i < npl && d < hd) ? to_float(qrow[d]) : 0.f;
  }
  ApState<NPL> st;
  if (split) {
    const int c = c_first + blockIdx.z;
    ap_page<T, NPL>(st, qv, kpool, vpool, pt[c], num_pages, KVH, kvh, hd, max(first, c << HE_PAGE_SHIFT),
               min(p, (c << HE_PAGE_SHIFT) + HE_PAGE_TOKENS - 1), scale, lane, npl, sh, p);
    float* w = ws + ((row * H + h) * (int64_t)gridDim.z + blockIdx.z) * (hd + 2);
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      const int d = lane + i * HE_WAVE;
      if (i < npl && d < hd) w[d] = st.acc[i];
    }
    if (lane == 0) w[hd] = st.m, w[hd + 1] = st.l;
    return;
  }
  ApState<NPL> total;
  total.m = -INFINITY;
  total.l = 0.f;
#pragma unroll
  for (int i = 0; i < NPL; ++i) total.acc[i] = 0.f;
  for (int c = c_first; c <= c_last; ++c) {
    ap_page<T, NPL>(st, qv, kpool, vpool, pt[c], num_pages, KVH, kvh, hd, max(first, c << HE_PAGE_SHIFT),
               min(p, (c << HE_PAGE_SHIFT) + HE_PAGE_TOKENS - 1), scale, lane, npl, sh, p);
    ap_join(total, st);
  }
  const float gf = ap_finish<T, NPL>(total, ex, row, h);
  const float inv = total.l > 0.f ? 1.f / total.l : 0.f;
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const int d = lane + i * HE_WAVE;
    if (i < npl && d < hd) o[d] = from_float<T>(ex.gate ? total.acc[i] * inv * gf : total.acc[i] * inv);
  }
}

// Four neighbouring queries of one sequence and head in one wavefront (whole prompts): every key
// and value is fetched once for the four, and each query still takes its own keys [first, p] page by
// page in the order above, so the bits are those of the kernel that takes a query at a time. A
// group of four rows that is not four consecutive positions of one sequence (the end of a
// sequence, padding) is taken query by query. grid (ceil(rows / 4), ceil(H / 4)).
#define AP_ROWS 4
template <typename T, int NPL>
__global__ __launch_bounds__(256) void attention_plain_rows_kernel(
    T* __restrict__ out, const T* __restrict__ q, const T* __restrict__ kpool, const T* __restrict__ vpool,
    const int32_t* __restrict__ positions, const int32_t* __restrict__ row_seq,
    const int32_t* __restrict__ seq_slot, const int32_t* __restrict__ page_table, int max_blocks,
    int num_pages, int rows, int H, int KVH, int hd, int window, int chunk, float scale, ApExtras ex) {
  const int lane = threadIdx.x & (HE_WAVE - 1);
  const int h = blockIdx.y * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (h >= H) return;
  const int64_t row0 = (int64_t)blockIdx.x * AP_ROWS;
  const int npl = (hd + HE_WAVE - 1) / HE_WAVE;
  const int kvh = h / (H / KVH);
  const int n_rows = (int)min((int64_t)AP_ROWS, rows - row0);
  const ApShape sh = ap_shape_of(ex, h);
  const int seq0 = row_seq[row0], p0 = positions[row0];
  bool together = n_rows == AP_ROWS && seq0 >= 0;
  for (int r = 1; r < n_rows; ++r) together = together && row_seq[row0 + r] == seq0 && positions[row0 + r] == p0 + r;
  auto store = [&](int64_t row, ApState<NPL>& total) {
    T* o = out + (row * H + h) * (int64_t)hd;
    const float gf = row_seq[row] >= 0 ? ap_finish<T, NPL>(total, ex, row, h) : 1.f;
    const float inv = total.l > 0.f ? 1.f / total.l : 0.f;
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      const int d = lane + i * HE_WAVE;
      if (i < npl && d < hd) o[d] = from_float<T>(ex.gate ? total.acc[i] * inv * gf : total.acc[i] * inv);
    }
  };
  auto load_q = [&](float (&qv)[NPL], int64_t row) {
    const T* qrow = q + (row * H + h) * (int64_t)hd;
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      const int d = lane + i * HE_WAVE;
      qv[i] = (i < npl && d < hd) ? to_float(qrow[d]) : 0.f;
    }
  };
  if (!together) {
    for (int r = 0; r < n_rows; ++r) {
      const int64_t row = row0 + r;
      ApState<NPL> total, st;
      total.m = -INFINITY;
      total.l = 0.f;
#pragma unroll
      for (int i = 0; i < NPL; ++i) total.acc[i] = 0.f;
      const int seq = row_seq[row];
      if (seq >= 0) {
        const int p = positions[row];
        const int first = ap_first(p, window, chunk);
        const int32_t* pt = page_table + (int64_t)seq_slot[seq] * max_blocks;
        float qv[NPL];
        load_q(qv, row);
        for (int c = first >> HE_PAGE_SHIFT; c <= (p >> HE_PAGE_SHIFT); ++c) {
          ap_page<T, NPL>(st, qv, kpool, vpool, pt[c], num_pages, KVH, kvh, hd, max(first, c << HE_PAGE_SHIFT),
                          min(p, (c << HE_PAGE_SHIFT) + HE_PAGE_TOKENS - 1), scale, lane, npl, sh, p);
          ap_join(total, st);
        }
      }
      store(row, total);
    }
    return;
  }
  const int32_t* pt = page_table + (int64_t)seq_slot[seq0] * max_blocks;
  float qv[AP_ROWS][NPL];
  ApState<NPL> total[AP_ROWS], st[AP_ROWS];
  int first[AP_ROWS];
#pragma unroll
  for (int r = 0; r < AP_ROWS; ++r) {
    load_q(qv[r], row0 + r);
    first[r] = ap_first(p0 + r, window, chunk);
    total[r].m = -INFINITY;
    total[r].l = 0.f;
#pragma unroll
    for (int i = 0; i < NPL; ++i) total[r].acc[i] = 0.f;
  }
  const int KS = he_k_steps(hd), NT = he_v_tiles(hd);
  const int p_last = p0 + AP_ROWS - 1;
  for (int c = first[0] >> HE_PAGE_SHIFT; c <= (p_last >> HE_PAGE_SHIFT); ++c) {
#pragma unroll
    for (int r = 0; r < AP_ROWS; ++r) {
      st[r].m = -INFINITY;
      st[r].l = 0.f;
#pragma unroll
      for (int i = 0; i < NPL; ++i) st[r].acc[i] = 0.f;
    }
    const int page = pt[c];
    if (page >= 0 && page < num_pages) {
      const int64_t base = ((int64_t)page * KVH + kvh) * he_k_page_elems(hd);
      const int64_t vbase = ((int64_t)page * KVH + kvh) * he_v_page_elems(hd);
      const int j_lo = max(first[0], c << HE_PAGE_SHIFT), j_hi = min(p_last, (c << HE_PAGE_SHIFT) + HE_PAGE_TOKENS - 1);
      const T* kpage = kpool + base;
      const T* vpage = vpool + vbase;
      // two sets of registers, as in ap_page: the next four keys are on their way while these are taken
      float ka[AP_GROUP][NPL], va[AP_GROUP][NPL], kb[AP_GROUP][NPL], vb[AP_GROUP][NPL];
      ap_fetch<T, NPL>(ka, va, kpage, vpage, j_lo, j_hi, KS, NT, lane, npl, hd);
      for (int j0 = j_lo; j0 <= j_hi; j0 += 2 * AP_GROUP) {
        ap_fetch<T, NPL>(kb, vb, kpage, vpage, j0 + AP_GROUP, j_hi, KS, NT, lane, npl, hd);
        float sc[AP_GROUP][AP_ROWS];
#pragma unroll
        for (int g = 0; g < AP_GROUP; ++g)
#pragma unroll
          for (int r = 0; r < AP_ROWS; ++r)
            sc[g][r] = ap_shape(sh, ap_score<NPL>(qv[r], ka[g], scale, lane, npl, hd), p0 + r - (j0 + g));
#pragma unroll
        for (int g = 0; g < AP_GROUP; ++g) {
          const int j = j0 + g;
#pragma unroll
          for (int r = 0; r < AP_ROWS; ++r)
            if (j <= j_hi && j >= first[r] && j <= p0 + r) ap_update<NPL>(st[r], sc[g][r], va[g], lane, npl, hd);
        }
        ap_fetch<T, NPL>(ka, va, kpage, vpage, j0 + 2 * AP_GROUP, j_hi, KS, NT, lane, npl, hd);
#pragma unroll
        for (int g = 0; g < AP_GROUP; ++g)
#pragma unroll
          for (int r = 0; r < AP_ROWS; ++r)
            sc[g][r] = ap_shape(sh, ap_score<NPL>(qv[r], kb[g], scale, lane, npl, hd), p0 + r - (j0 + AP_GROUP + g));
#pragma unroll
        for (int g = 0; g < AP_GROUP; ++g) {
          const int j = j0 + AP_GROUP + g;
#pragma unroll
          for (int r = 0; r < AP_ROWS; ++r)
            if (j <= j_hi && j >= first[r] && j <= p0 + r) ap_update<NPL>(st[r], sc[g][r], vb[g], lane, npl, hd);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < AP_ROWS; ++r) ap_join(total[r], st[r]);
  }
#pragma unroll
  for (int r = 0; r < AP_ROWS; ++r) store(row0 + r, total[r]);
}

// Joins the pages' results of a split launch in ascending position. grid (rows, ceil(H / 4)).
template <typename T, int NPL>
__global__ __launch_bounds__(256) void attention_plain_join_kernel(
    T* __restrict__ out, const float* __restrict__ ws, const int32_t* __restrict__ positions,
    const int32_t* __restrict__ row_seq, int H, int hd, int window, int chunk, int pages, ApExtras ex) {
  const int lane = threadIdx.x & (HE_WAVE - 1);
  const int h = blockIdx.y * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int64_t row = blockIdx.x;
  if (h >= H) return;
  T* o = out + (row * H + h) * (int64_t)hd;
  const int npl = (hd + HE_WAVE - 1) / HE_WAVE;
  ApState<NPL> total;
  total.m = -INFINITY;
  total.l = 0.f;
#pragma unroll
  for (int i = 0; i < NPL; ++i) total.acc[i] = 0.f;
  float gf = 1.f;
  if (row_seq[row] >= 0) {
    const int p = positions[row];
    const int first = ap_first(p, window, chunk);
    const int count = (p >> HE_PAGE_SHIFT) - (first >> HE_PAGE_SHIFT) + 1;
    if (count > pages) {
      // the caller's bound on the keys was too low: no part of the result may pass for one
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        const int d = lane + i * HE_WAVE;
        if (i < npl && d < hd) o[d] = from_float<T>(NAN);
      }
      return;
    }
    // eight pages' results are asked for together and then joined one after the other in order
    // (one at a time, every page waited for its own loads: 17 us for 33 pages)
    constexpr int AHEAD = 8;
    for (int z0 = 0; z0 < count; z0 += AHEAD) {
      ApState<NPL> part[AHEAD];
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const float* w = ws + ((row * H + h) * (int64_t)pages + min(z0 + u, count - 1)) * (hd + 2);
#pragma unroll
        for (int i = 0; i < NPL; ++i) {
          const int d = lane + i * HE_WAVE;
          part[u].acc[i] = (i < npl && d < hd) ? w[d] : 0.f;
        }
        part[u].m = w[hd];
        part[u].l = w[hd + 1];
      }
#pragma unroll
      for (int u = 0; u < AHEAD; ++u)
        if (z0 + u < count) ap_join(total, part[u]);
    }
    gf = ap_finish<T, NPL>(total, ex, row, h);
  }
  const float inv = total.l > 0.f ? 1.f / total.l : 0.f;
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const int d = lane + i * HE_WAVE;
    if (i < npl && d < hd) o[d] = from_float<T>(ex.gate ? total.acc[i] * inv * gf : total.acc[i] * inv);
  }
}

// Pages a query of this step has at most (what a split launch needs room for), given the most keys
// a sequence holds after the step.
// reach: the most keys a query sees (its window, or its chunk; 0: all before it)
static int ap_pages(int most_keys, int reach) {
  int pages = (most_keys + HE_PAGE_TOKENS - 1) / HE_PAGE_TOKENS;
  if (reach > 0) pages = min(pages, (reach + HE_PAGE_TOKENS - 2) / HE_PAGE_TOKENS + 1);
  return max(pages, 1);
}
static int ap_reach(int window, int chunk) {
  if (window > 0 && chunk > 0) return min(window, chunk);
  return window > 0 ? window : max(chunk, 0);
}

// Floats of workspace with which the step's attention runs page by page in parallel (0: one
// wavefront per query and head walks the pages itself; that is the better launch for a step with
// many queries).
extern "C" int64_t he_attention_plain_workspace_floats(int rows, int H, int hd, int most_keys, int window,
                                                       int chunk) {
  if (rows <= 0 || H <= 0 || hd <= 0 || most_keys <= 0) return 0;
  const int pages = ap_pages(most_keys, ap_reach(window, chunk));
  if (pages < 2 || (int64_t)rows * H > 8 * he_cus()) return 0;
  return (int64_t)rows * H * pages * (hd + 2);
}

extern "C" int he_attention_plain(void* out, const void* q, const void* kpool, const void* vpool,
                                  const void* positions, const void* row_seq, const void* seq_slot,
                                  const void* page_table, int max_blocks, int num_pages, int rows,
                                  int H, int KVH, int hd, int window, int chunk, float scale,
                                  const void* sinks, int sinks_dtype, const void* gate,
                                  int64_t gate_stride, int dtype, int most_keys, void* workspace_f32,
                                  int64_t workspace_floats, const void* slopes_f32, const void* table_f32,
                                  int table_len, float cap, void* stream) {
  HE_REQUIRE(rows >= 0 && H > 0 && KVH > 0 && hd > 0, "he_attention_plain: bad sizes");
  HE_REQUIRE(H % KVH == 0, "he_attention_plain: heads %d not a multiple of kv heads %d", H, KVH);
  HE_REQUIRE(hd <= AP_MAX_PER_LANE * HE_WAVE, "he_attention_plain: head_dim %d above %d", hd,
             AP_MAX_PER_LANE * HE_WAVE);
  HE_REQUIRE(dtype == HE_BF16 || dtype == HE_F32, "he_attention_plain: unknown dtype %d", dtype);
  HE_REQUIRE(sinks == nullptr || sinks_dtype == HE_BF16 || sinks_dtype == HE_F32,
             "he_attention_plain: unknown dtype %d of the sinks", sinks_dtype);
  HE_REQUIRE(slopes_f32 == nullptr || table_f32 == nullptr, "he_attention_plain: slopes and a distance table exclude each other");
  HE_REQUIRE(table_f32 == nullptr || table_len > 0, "he_attention_plain: an empty distance table");
  if (rows == 0) return 0;
  const ApExtras ex = {sinks, sinks_dtype, gate, gate_stride, (const float*)slopes_f32, (const float*)table_f32, table_len, cap};
  // page by page in parallel when the caller brought room for it (the same bits either way)
  const int64_t need = he_attention_plain_workspace_floats(rows, H, hd, most_keys, window, chunk);
  const bool split = need > 0 && workspace_f32 != nullptr && workspace_floats >= need;
  const int pages = split ? ap_pages(most_keys, ap_reach(window, chunk)) : 1;
  HE_REQUIRE(pages <= 65535, "he_attention_plain: %d pages of keys are too many for one launch", pages);
  dim3 grid(rows, (H + 3) / 4, pages);
  float* ws = (float*)workspace_f32;
  hipStream_t s = (hipStream_t)stream;
  // 32-bit caches whose head size is whole steps of the matrix cores' operands
  const bool mfma = dtype == HE_F32 && hd % 32 == 0 && hd <= 128 && (((uintptr_t)q | (uintptr_t)kpool | (uintptr_t)vpool | (uintptr_t)out) & 15) == 0;
  const bool by_runs = mfma && !split && rows >= AP32_TILE;
  const int64_t columns = (int64_t)rows * KVH * ((H / KVH + 15) / 16);
  // (parts a query: as many wavefronts as the chip holds of this kernel, one a SIMD at head sizes of 96 and 128, two below)
  const int parts = (int)max((int64_t)1, min((int64_t)pages, (hd > 64 ? 4 : 8) * he_cus() / columns));
  const int64_t units = columns * parts;
  // The launch of single queries: four units a workgroup, or one where compute units would stay without any (16 sequences of 16
  // keys, 28 heads on 4: 17.5 us by fours, 16.8 by one).
  const int ones_waves = units <= 2 * he_cus() ? 1 : 4;
  const int64_t ones = (units + ones_waves - 1) / ones_waves;
  const dim3 ones_grid((unsigned)(ones < (1 << 22) ? ones : 1 << 22), (unsigned)((ones + (1 << 22) - 1) >> 22));
  const bool shaped = slopes_f32 != nullptr || table_f32 != nullptr || cap > 0.f;
#define AP32_ONE(KS_, SPLIT_, SHAPED_)                                                                               \
  attention_f32_one_kernel<KS_, SPLIT_, SHAPED_><<<ones_grid, ones_waves * HE_WAVE, ones_waves * KS_ * 4096, s>>>(  \
      (float*)out, ws, (const float*)q, (const float*)kpool, (const float*)vpool, (const int32_t*)positions,         \
      (const int32_t*)row_seq, (const int32_t*)seq_slot, (const int32_t*)page_table, max_blocks, num_pages, rows, H, KVH, \
      window, chunk, scale, pages, parts, by_runs ? 1 : 0, ex)
#define AP32_SHAPED(KS_, SHAPED_)                                                                                    \
  {                                                                                                                  \
    if (by_runs)                                                                                                     \
      attention_f32_rows_kernel<KS_, SHAPED_><<<dim3((rows + AP32_TILE - 1) / AP32_TILE, (H + 3) / 4), 256, 0, s>>>( \
          (float*)out, (const float*)q, (const float*)kpool, (const float*)vpool, (const int32_t*)positions,         \
          (const int32_t*)row_seq, (const int32_t*)seq_slot, (const int32_t*)page_table, max_blocks, num_pages, rows, H, \
          KVH, window, chunk, scale, ex);                                                                            \
    if (split) AP32_ONE(KS_, true, SHAPED_);                                                                         \
    else AP32_ONE(KS_, false, SHAPED_);                                                                              \
  }
#define AP32_LAUNCH(KS_)                                                                                             \
  {                                                                                                                  \
    if (shaped) AP32_SHAPED(KS_, true)                                                                               \
    else AP32_SHAPED(KS_, false)                                                                                     \
  }
#define AP_LAUNCH(T, NPL)                                                                      \
  attention_plain_kernel<T, NPL><<<grid, 256, 0, s>>>(                                         \
      (T*)out, ws, (const T*)q, (const T*)kpool, (const T*)vpool, (const int32_t*)positions,   \
      (const int32_t*)row_seq, (const int32_t*)seq_slot, (const int32_t*)page_table,           \
      max_blocks, num_pages, H, KVH, hd, window, chunk, scale, ex)
#define AP_JOIN(T, NPL)                                                                        \
  attention_plain_join_kernel<T, NPL><<<dim3(rows, (H + 3) / 4), 256, 0, s>>>(                 \
      (T*)out, ws, (const int32_t*)positions, (const int32_t*)row_seq, H, hd, window, chunk, pages, ex)
  const int npl = (hd + HE_WAVE - 1) / HE_WAVE;   // elements a lane holds: 1, 2, up to 4, up to 8, up to 16
#define AP_BY_SIZE(WHAT)                                  \
  if (dtype == HE_BF16) {                                 \
    if (npl <= 1) WHAT(bf16_t, 1);                        \
    else if (npl <= 2) WHAT(bf16_t, 2);                   \
    else if (npl <= 4) WHAT(bf16_t, 4);                   \
    else if (npl <= 8) WHAT(bf16_t, 8);                   \
    else WHAT(bf16_t, 16);                                \
  } else {                                                \
    if (npl <= 1) WHAT(float, 1);                         \
    else if (npl <= 2) WHAT(float, 2);                    \
    else if (npl <= 4) WHAT(float, 4);                    \
    else if (npl <= 8) WHAT(float, 8);                    \
    else WHAT(float, 16);                                 \
  }
#define AP_ROWS_LAUNCH(T, NPL)                                                                          \
  attention_plain_rows_kernel<T, NPL><<<dim3((rows + AP_ROWS - 1) / AP_ROWS, (H + 3) / 4), 256, 0, s>>>(   \
      (T*)out, (const T*)q, (const T*)kpool, (const T*)vpool, (const int32_t*)positions,               \
      (const int32_t*)row_seq, (const int32_t*)seq_slot, (const int32_t*)page_table, max_blocks,       \
      num_pages, rows, H, KVH, hd, window, chunk, scale, ex)
  if (mfma) {
    if (hd == 32) AP32_LAUNCH(1)
    else if (hd == 64) AP32_LAUNCH(2)
    else if (hd == 96) AP32_LAUNCH(3)
    else AP32_LAUNCH(4)
    int rc = he_check_launch("he_attention_plain");
    if (rc || !split) return rc;
    AP_BY_SIZE(AP_JOIN)
    return he_check_launch("he_attention_plain");
  }
  if (!split && rows >= 64) {      // a step of many queries: four neighbours a wavefront share their keys
    AP_BY_SIZE(AP_ROWS_LAUNCH)
    return he_check_launch("he_attention_plain");
  }
  AP_BY_SIZE(AP_LAUNCH)
  int rc = he_check_launch("he_attention_plain");
  if (rc || !split) return rc;
  AP_BY_SIZE(AP_JOIN)
#undef AP_BY_SIZE
#undef AP_ROWS_LAUNCH
#undef AP_LAUNCH
#undef AP32_LAUNCH
#undef AP32_SHAPED
#undef AP32_ONE
#undef AP_JOIN
  return he_check_launch("he_attention_plain");
}
