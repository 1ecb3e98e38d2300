// Between the two passes of a recurrence over ranges of a prompt (linear_attn.hip, mixer_ops.hip): every range's end-from-zero state
// becomes its START state, S <- p_k S + end_k, and the last S goes to the sequence's slot.  A thread has VEC entries of a (sequence,
// head).  What bounds it is the states' bytes, read and written once; asked for one behind the other's store they came a range at a
// time, and with one entry a thread as 4 bytes a lane.
// us of the kernel before / now, 16 heads of 128 x 128 in engine steps:  7 sequences in 27 to 30 ranges 20.9 / 13.5 (5.3 TB/s), 8 in 32
// 24.0 / 13.4;  2 in 11 chunks of the fp32 scan, whose factors were a chain of multiplications each, 19.0 / 6.6.
#pragma once
#include "common.h"

namespace k8s {

template <int VEC>
struct CarryVec {
  typedef float type __attribute__((ext_vector_type(VEC)));
};

// n ranges, `step` numbers apart from `ck` on; p(k): the factor of range k
template <int VEC, typename F>
__device__ __forceinline__ void carry_states(float* st, bool fresh, float* ck, size_t step, int n, F&& p) {
  using T = typename CarryVec<VEC>::type;
  constexpr int U = 8;                 // ranges asked for at once
  T S = T(0.f);
  if (!fresh) S = *reinterpret_cast<const T*>(st);
  for (int k0 = 0; k0 < n; k0 += U) {
    T end[U];
#pragma unroll
    for (int u = 0; u < U; ++u) end[u] = *reinterpret_cast<const T*>(ck + (size_t)min(k0 + u, n - 1) * step);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k0 + u >= n) break;
      *reinterpret_cast<T*>(ck + (size_t)(k0 + u) * step) = S;
      const float f = p(k0 + u);
#pragma unroll
      for (int i = 0; i < VEC; ++i) S[i] = fmaf(f, S[i], end[u][i]);
    }
  }
  *reinterpret_cast<T*>(st) = S;
}

// four entries a thread where the states lie on 16 bytes
__host__ inline bool carry_by_four(const void* state, const void* cs, int DV) {
  return DV % 4 == 0 && !(((uintptr_t)state | (uintptr_t)cs) & 15);
}

}  // namespace k8s
