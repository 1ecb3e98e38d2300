// The keys a position sees under the masks of masked_attn.hip, as one virtual range.
#pragma once
#include <hip/hip_runtime.h>

namespace k8s {

// The visible keys of position `pos`: [a0, a1) and [lo, pos], walked as x in [0, nA + nB).
struct KeyRuns {
  int a0, nA, lo, total;
  __device__ __forceinline__ int key(int x) const { return x < nA ? a0 + x : lo + (x - nA); }
};

__device__ __forceinline__ KeyRuns key_runs(int pos, int chunk, int window, int keep_first) {
  KeyRuns k;
  k.a0 = chunk > 0 ? (pos / chunk) * chunk : 0;
  k.lo = k.a0;
  k.nA = 0;
  if (window > 0) {
    k.lo = max(k.a0, pos - window + 1);
    k.nA = max(0, min(keep_first, k.lo) - k.a0);
  }
  k.total = k.nA + pos - k.lo + 1;
  return k;
}

// A value mixed with another layer's of the same token, the same bits in every kernel that does it.
__device__ __forceinline__ float mix_value(float lam, float v, float other) { return fmaf(lam, other, (1.f - lam) * v); }

}  // namespace k8s
