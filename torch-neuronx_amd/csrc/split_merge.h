// Merge of the partial rows that a call with split keys leaves in its workspace (fwd_mfma_w32.hip,
// f32_mfma.hip, decode_fp8kv.hip): out = sum_c w_c O_c / sum_c w_c l_c with w_c = 2^(m_c - max m), or e^ of it.
//
// One workgroup per output row.  What bounds it is not the bytes (a few MB, in L2) but the trips to
// them: it is a launch between two others whose work is one chain of dependent loads.  So the parts are
// dealt to SLICES groups of threads, a thread owning four columns of its slice's parts, and a slice asks
// for the statistics and the rows of eight parts at once, before it knows any weight: one trip to
// memory for up to 8 * SLICES parts.  The slices' results meet in LDS.  (A thread per column walking the
// parts eight at a time with the weights worked out in two passes before took 10.2 us for the 128 parts
// of a sequence of 32768 keys at head dim 128, decode_fp8kv.hip; in slices 4.0, and the decode call 25.6 -> 19.9.)
#pragma once

#include "mfma_common.h"

namespace mi355 {

// SLICES: 16 where a row may have more than 16 parts, 4 otherwise (a batch: many rows, few parts each;
// more threads per row would only be more idle ones).  TPR: threads per part row, four columns each.
constexpr int kMergeFew = 4, kMergeMany = 16;
static inline int merge_slices_for(int64_t parts) { return parts > 16 ? kMergeMany : kMergeFew; }

// What a part of a forward call leaves as its row's log-sum-exp, l being the sum behind it.  A row whose sum is NaN has
// lse = -inf like one without a live key, but must not pass for one here, or the parts without the NaN would be the result:
// it leaves the NaN, and the merged row is NaN too (with lse = -inf), as it is where the keys are not split.
__device__ __forceinline__ float part_lse_of(float l, float lse) { return l == l ? lse : l; }

template <int SLICES, int TPR>
struct MergeLds {
  float o[SLICES][TPR * 4];
  float m[SLICES], l[SLICES];
};

// ml(c, m, l): statistics of part c, m in the log2 domain or (LN) the natural one (m = -inf: a part without
// keys, its row is never used whatever it holds; m = NaN: the merged row is NaN).  (The domain is the caller's: a
// log-sum-exp turned into the other one and back takes two roundings of its own size, lse 4.1e-7 -> 4.4e-7 off at
// float32, 8 heads, S=2048; here only differences are converted.)  row(c): this thread's four columns of part c.
// Workgroup of SLICES * TPR threads; on return thread d < 4 * TPR holds column d of the weighted sum (O), and M and L are
// those of the row.
template <bool LN, int SLICES, int TPR, typename ML, typename ROW>
__device__ __forceinline__ void merge_parts(MergeLds<SLICES, TPR>& lds, int np, ML ml, ROW row, float& O, float& M, float& L) {
  static_assert(SLICES >= 4, "one thread per column at the end");
  constexpr int BATCH = 8;
  const int slice = threadIdx.x / TPR, quad = threadIdx.x % TPR;
  auto weight = [](float d) { return __builtin_amdgcn_exp2f(LN ? d * kLog2eF : d); };
  float ms = -INFINITY, ls = 0.f;
  f32x4 os = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = slice; c0 < np; c0 += SLICES * BATCH) {
    float m[BATCH], l[BATCH];
    f32x4 o[BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const int c = c0 + SLICES * i;
      m[i] = -INFINITY, l[i] = 0.f, o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (c < np) {
        ml(c, m[i], l[i]);
        o[i] = row(c);
      }
    }
    float mn = ms;
#pragma unroll
    for (int i = 0; i < BATCH; ++i) mn = fmaxf(mn, m[i]);
    // (no part with a score so far: the reference is 0, the weights are too, and a NaN among the sums - a part whose
    // scores are all NaN has no maximum - still makes the row's sum one)
    const float ref = mn == -INFINITY ? 0.f : mn;
    const float f = weight(ms - ref);
    ls *= f, os *= f;
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      const float w = weight(m[i] - ref);
      ls = fmaf(l[i], w, ls);
#pragma unroll
      for (int e = 0; e < 4; ++e) os[e] = m[i] == -INFINITY ? os[e] : fmaf(o[i][e], w, os[e]);
    }
    ms = mn;
  }
  *(f32x4*)(&lds.o[slice][quad * 4]) = os;
  if (quad == 0) lds.m[slice] = ms, lds.l[slice] = ls;
  __syncthreads();
  M = -INFINITY, L = 0.f, O = 0.f;
#pragma unroll
  for (int s = 0; s < SLICES; ++s) M = fmaxf(M, lds.m[s]);
  const float ref = M == -INFINITY ? 0.f : M;  // (as above: no part with a score, or none but those with a NaN)
  const int d = min((int)threadIdx.x, 4 * TPR - 1);
#pragma unroll
  for (int s = 0; s < SLICES; ++s) {
    const float w = weight(lds.m[s] - ref);
    L = fmaf(lds.l[s], w, L);
    O = fmaf(lds.o[s][d], w, O);
  }
}

}  // namespace mi355
