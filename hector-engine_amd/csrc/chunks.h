// The rows of a step's sequences in chunks of CK_ROWS, counted through the sequences: what the scans that go by chunks share.
#pragma once
#include "common.h"

#define CK_ROWS 64

// ---- which chunk is whose ------------------------------------------------------------------------------
// Sequences of up to `from` rows have none (they are walked).
__device__ __forceinline__ int ck_chunks(const int32_t* cu, int s, int from) {
  const int n = cu[s + 1] - cu[s];
  return n > from ? (n + CK_ROWS - 1) / CK_ROWS : 0;
}

// Chunk t of the step, counted through its sequences: the sequence and the chunk inside it. Every wavefront finds it
// for itself (64 sequences a turn). False: the step has no chunk t.
__device__ __forceinline__ bool ck_find(int t, const int32_t* __restrict__ cu, int num_seqs, int from, int& seq, int& chunk) {
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int s0 = 0; s0 < num_seqs; s0 += 64) {
    const int s = s0 + lane;
    const int n = s < num_seqs ? ck_chunks(cu, s, from) : 0;
    int upto = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(upto, o);
      if (lane >= o) upto += u;
    }
    const unsigned long long hit = __ballot(t < base + upto);
    if (hit != 0) {
      const int f = __ffsll((long long)hit) - 1;
      seq = s0 + f;
      chunk = t - base - __shfl(upto - n, f);
      return true;
    }
    base += __shfl(upto, 63);
  }
  return false;
}
