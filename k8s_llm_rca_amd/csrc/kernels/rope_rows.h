// cos | sin of a step's positions, for the kernel that makes them alone (masked_attn.hip) and for those that make them beside
// a step's first rows (hyper_conn.hip, dyt_ops.hip), where they were one or two launches of 2 to 4 us in every step.
#pragma once
#include <hip/hip_runtime.h>

namespace k8s {

// cs [T][2 half]: cos | sin of positions[t] * freq[j], times amp (the product in double); entry i = t half + j
__device__ __forceinline__ void rope_entry(const int* __restrict__ positions, const double* __restrict__ freq, float amp,
                                           float* __restrict__ cs, int half, size_t i) {
  const size_t t = i / half;
  const int j = (int)(i - t * half);
  double si, co;
  sincos((double)positions[t] * freq[j], &si, &co);
  cs[t * 2 * half + j] = (float)co * amp;
  cs[t * 2 * half + half + j] = (float)si * amp;
}

constexpr int kRopeTables = 2;
struct RopeTables {
  const int* pos;
  const double* freq[kRopeTables];
  float* cs[kRopeTables];
  float amp[kRopeTables];
  int half[kRopeTables];               // 0: no such table
};

// Workgroups behind a launch's own `rows` ones, one entry a thread
inline unsigned rope_blocks(const RopeTables& r, int rows, int threads) {
  size_t n = 0;
  for (int k = 0; k < kRopeTables; ++k) n += (size_t)rows * r.half[k];
  return (unsigned)((n + threads - 1) / threads);
}
inline bool rope_tables_ok(const RopeTables& r) {
  for (int k = 0; k < kRopeTables; ++k)
    if (r.half[k] < 0 || (r.half[k] && (!r.pos || !r.freq[k] || !r.cs[k]))) return false;
  return true;
}
__device__ __forceinline__ void rope_block(const RopeTables& r, int rows) {
  size_t i = (size_t)(blockIdx.x - rows) * blockDim.x + threadIdx.x;
#pragma unroll
  for (int k = 0; k < kRopeTables; ++k) {
    const size_t n = (size_t)rows * r.half[k];
    if (i < n) return rope_entry(r.pos, r.freq[k], r.amp[k], r.cs[k], r.half[k], i);
    i -= n;
  }
}

}  // namespace k8s
