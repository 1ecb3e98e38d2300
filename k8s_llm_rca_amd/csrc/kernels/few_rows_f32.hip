// y [M][N] = x [M][K] . w [N][K]^T in fp32 for up to eight rows: the products of reply steps in float32.
//
// Each weight is used M times, so the rate is that of reading w.  A workgroup of four waves takes four rows of w, its threads
// neighbouring quadruples of K in turn: every load is 4 KB of consecutive weights, none is read twice, all of a step are in
// flight together, and even 2048 columns are 512 workgroups.  x comes from the caches.  Which sums a thread makes depends
// on K alone: a row's bits are the same among one and among eight.  The sums over the wave halve the values with the
// distance: one after the other they cost 1 us a row (2048 x 2048, 4 rows: 8.5 -> 5.8 us).
// What bounds it: the weights up to four rows (2048 x 8192: 12.5 to 13.5 us, 5.0 TB/s; hipBLASLt's sums 23), then the rows
// of x, which each workgroup reads from its caches.  Error against 64 bits 9.4e-8 at K 2048 (hipBLASLt 4.1e-7).
//
// GLU: w = [N gate rows; N up rows], y = g sigmoid(g) u of both (glu_clamp_kernel's arithmetic without its limits): a workgroup
// takes two rows of each, so that the two rows of sums are not written, read and launched for again (8192 x 2048 at two
// rows: 20.4 + 4.7 us -> 20.8 in a traced step).
#include "common.h"

namespace k8s {

constexpr int kFewN = 4;       // rows of w per workgroup

template <int M, bool GLU>
__global__ void __launch_bounds__(256) few_rows_f32_kernel(const float* __restrict__ x, int ldx, const float* __restrict__ w,
                                                           float* __restrict__ y, int N, int K) {
  __shared__ float red[4][kFewN * M];
  constexpr int R = GLU ? kFewN / 2 : kFewN;       // outputs of a workgroup
  const int tid = threadIdx.x, n0 = blockIdx.x * R;
  const float* wp[kFewN];
#pragma unroll
  for (int r = 0; r < kFewN; ++r) wp[r] = w + ((size_t)min(n0 + r % R, N - 1) + (r < R ? 0 : N)) * K;
  float acc[kFewN][M] = {};
#pragma unroll 2
  for (int k = 4 * tid; k < K; k += 1024) {
    f32x4 wv[kFewN];
#pragma unroll
    for (int r = 0; r < kFewN; ++r) wv[r] = ldw_nt<f32x4>(wp[r] + k);
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const f32x4 xv = *reinterpret_cast<const f32x4*>(x + (size_t)m * ldx + k);
#pragma unroll
      for (int r = 0; r < kFewN; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[r][m] = fmaf(xv[i], wv[r][i], acc[r][m]);
    }
  }
  constexpr int V = kFewN * (M > 4 ? 8 : M > 2 ? 4 : M);
  float v[V];
#pragma unroll
  for (int i = 0; i < V; ++i) v[i] = i < kFewN * M ? acc[i % kFewN][i / kFewN] : 0.f;
  const float sum = wave_sums<V>(v);
  const int at = (tid & 63) / (64 / V);
  if (tid % (64 / V) == 0 && at < kFewN * M) red[tid >> 6][at] = sum;
  __syncthreads();
  if (tid < R * M && n0 + tid % R < N) {
    auto sum = [&](int i) { return (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]); };
    const int m = tid / R, r = tid % R;
    float t = sum(m * kFewN + r);
    if constexpr (GLU) {
      const float g = fminf(t, INFINITY), u = fminf(fmaxf(sum(m * kFewN + R + r), -INFINITY), INFINITY);
      t = g / (1.f + expf(-1.f * g)) * (u + 0.f);
    }
    y[(size_t)m * N + n0 + r] = t;
  }
}

}  // namespace k8s

using namespace k8s;

template <bool GLU>
static int few_rows(const float* x, int ldx, const float* w, float* y, int M, int N, int K, hipStream_t s) {
  if (M < 1 || M > 8 || N < 1 || K < 4 || K % 4 || ldx % 4 || (M > 1 && ldx < K) || (((uintptr_t)x | (uintptr_t)w) & 15))
    return (int)hipErrorInvalidValue;
  constexpr int R = GLU ? kFewN / 2 : kFewN;
  const dim3 g((N + R - 1) / R);
#define K8S_FR(MM) \
  case MM: hipLaunchKernelGGL((few_rows_f32_kernel<MM, GLU>), g, dim3(256), 0, s, x, ldx, w, y, N, K); break
  switch (M) {
    K8S_FR(1);
    K8S_FR(2);
    K8S_FR(3);
    K8S_FR(4);
    K8S_FR(5);
    K8S_FR(6);
    K8S_FR(7);
    K8S_FR(8);
  }
#undef K8S_FR
  return (int)hipGetLastError();
}

// M <= 8, K % 4 == 0, rows of x and w 16-byte aligned.
K8S_API int k8s_few_rows_f32(const float* x, int ldx, const float* w, float* y, int M, int N, int K, hipStream_t s) {
  return few_rows<false>(x, ldx, w, y, M, N, K, s);
}

// The gated unit of w = [gate rows; up rows], N of each.
K8S_API int k8s_few_rows_glu_f32(const float* x, int ldx, const float* w, float* y, int M, int N, int K, hipStream_t s) {
  return few_rows<true>(x, ldx, w, y, M, N, K, s);
}
