// argmax_impl.h -- candidate merge of the parallel greedy argmax, shared by
// misc.hip and the LM-head GEMV (gemv_impl.h).
//
// sample_argmax (reference src/tokenizer.rs:179-189) returns the first index
// of the maximum under a strict `>` scan from logits[0]: NaN never wins, and a
// NaN logits[0] yields 0.  In parallel: every non-NaN element is a candidate,
// candidates combine by (larger value, then lower index) -- a total order, so
// the tree shape cannot change the answer -- and the NaN-logits[0] case is
// applied at the end.  +0 and -0 compare equal, as in the scan.
#pragma once

#include "device_common.h"

#define ARGMAX_NONE 0xffffffffu

AMMON_DEV void cand_merge(float &v, uint32_t &i, float v2, uint32_t i2) {
  if (i2 == ARGMAX_NONE) return;
  if (i == ARGMAX_NONE || v2 > v || (!(v > v2) && i2 < i)) {
    v = v2;
    i = i2;
  }
}

// Workgroup reduction of the candidates; sv / si hold AMMON_WAVES entries of
// LDS.  Within a wave by lane exchange, the waves' through LDS: one barrier (a
// tree over LDS takes nine).  The order of merging does not matter.  Call
// uniformly.
AMMON_DEV void block_cand_reduce(float &v, uint32_t &i, float *sv, uint32_t *si) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float v2 = __shfl_xor(v, off, 64);
    const uint32_t i2 = __shfl_xor(i, off, 64);
    cand_merge(v, i, v2, i2);
  }
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    sv[wave] = v;
    si[wave] = i;
  }
  __syncthreads();
  v = sv[0];
  i = si[0];
#pragma unroll
  for (int w = 1; w < AMMON_WAVES; ++w) cand_merge(v, i, sv[w], si[w]);
}

