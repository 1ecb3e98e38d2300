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
//
// ADD: what stands between a sublayer's last product and the next sublayer's input, as gemm_step.hip has it for bf16 (x += s(m)
// product [+ es emb[id]], h = x nw and the row's sum of squares in parts, one a workgroup).  SCALED: the product behind it, whose
// sums are divided by the root mean square that the parts give; a wave reads a row's parts in front of the weights and adds
// them behind (up to four rows, a wave each; _into_f32, row_step.py).  The pass in between was a launch of 4.6 us in which two
// workgroups read 50 KB:  2048 x 8192, the pass and 8192 x 2048 at 1, 2, 4 rows 27.7 -> 25.3, 28.9 -> 25.5, 31.7 -> 29.9 us.
#include "common.h"

namespace k8s {

constexpr int kFewN = 4;       // rows of w per workgroup

constexpr int kFewSums = 64;   // ADD: sums of squares of the operand's own norm, at most
constexpr int kFewMaxK = 4096; // SCALED

struct FewAdd {
  float* x;              // [M][N], in place
  const float* rs;       // [M][rn] or null: the product is divided by sqrt(sum / rw + reps)
  const int* eid;        // [M]: rows of emb, times es, are added too; or null
  const float* emb;
  const float* nw;       // [N]
  float* part;           // [M][N / 4]
  float rw, reps, es;
  int rn;
};
struct FewScale {
  const float* part;     // [M][K / 4]
  float eps;
};

template <int M, bool GLU, bool ADD, bool SCALED>
__global__ void __launch_bounds__(256) few_rows_f32_kernel(const float* __restrict__ x, int ldx, const float* __restrict__ w,
                                                           float* __restrict__ y, int N, int K, FewAdd ad, FewScale sc) {
  __shared__ float red[4][kFewN * M];
  constexpr int R = GLU ? kFewN / 2 : kFewN;       // outputs of a workgroup
  const int tid = threadIdx.x, n0 = blockIdx.x * R;
  const float* wp[kFewN];
#pragma unroll
  for (int r = 0; r < kFewN; ++r) wp[r] = w + ((size_t)min(n0 + r % R, N - 1) + (r < R ? 0 : N)) * K;
  // SCALED: row wv, a lane the quads of parts lane, lane + 64, ..
  static_assert(!(ADD || SCALED) || M <= 4, "a wave a row");
  constexpr int SQ = SCALED ? kFewMaxK / 1024 : 1;
  const int lane = tid & 63, wv = tid >> 6;
  f32x4 pq[SQ];
  if constexpr (SCALED) {
#pragma unroll
    for (int j = 0; j < SQ; ++j) {
      pq[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (wv < M && 16 * (lane + 64 * j) < K)
        pq[j] = *reinterpret_cast<const f32x4*>(sc.part + (size_t)wv * (K / 4) + 4 * (lane + 64 * j));
    }
  }
  const int om = tid / R, on = n0 + tid % R;
  float xv = 0.f, nw = 0.f, ev = 0.f, rv = 0.f;
  if (ADD && ad.rs && wv < M && lane < ad.rn) rv = ad.rs[(size_t)wv * ad.rn + lane];
  if (ADD && tid < R * M) {
    xv = ad.x[(size_t)om * N + on];
    nw = ad.nw[on];
    if (ad.eid) ev = ad.emb[(size_t)ad.eid[om] * N + on];
  }
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
  __shared__ float factor[SCALED || ADD ? M : 1];
  if constexpr (SCALED) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < SQ; ++j) s += (pq[j][0] + pq[j][1]) + (pq[j][2] + pq[j][3]);
    s = wave_sum_dpp(s);
    if (lane == 63 && wv < M) factor[wv] = 1.f / sqrtf(s / (float)K + sc.eps);
  }
  if constexpr (ADD) {
    if (wv < M) {
      const float s = wave_sum_dpp(rv);
      if (lane == 63) factor[wv] = ad.rs ? 1.f / sqrtf(s / ad.rw + ad.reps) : 1.f;
    }
  }
  __syncthreads();
  if (tid < R * M && n0 + tid % R < N) {
    const int m = tid / R, r = tid % R;
    auto sum = [&](int i) {
      float t = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
      if constexpr (SCALED) t *= factor[m];
      return t;
    };
    float t = sum(m * kFewN + r);
    if constexpr (GLU) {
      const float g = fminf(t, INFINITY), u = fminf(fmaxf(sum(m * kFewN + R + r), -INFINITY), INFINITY);
      t = g / (1.f + expf(-1.f * g)) * (u + 0.f);
    }
    if constexpr (ADD) {                                   // y: h
      xv = fmaf(factor[m], t, xv);
      if (ad.eid) xv = fmaf(ad.es, ev, xv);
      ad.x[(size_t)m * N + on] = xv;
      t = xv * nw;
      float q = xv * xv;                                   // (N % 4 == 0: all four lanes are here)
      q += __shfl_xor(q, 1, 4);
      q += __shfl_xor(q, 2, 4);
      if (r == 0) ad.part[(size_t)m * (N / 4) + blockIdx.x] = q;
    }
    y[(size_t)m * N + n0 + r] = t;
  }
}

}  // namespace k8s

using namespace k8s;

template <bool GLU, bool ADD = false, bool SCALED = false>
static int few_rows(const float* x, int ldx, const float* w, float* y, int M, int N, int K, hipStream_t s,
                    const FewAdd& ad = FewAdd{}, const FewScale& sc = FewScale{}) {
  if (M < 1 || M > 8 || N < 1 || K < 4 || K % 4 || ldx % 4 || (M > 1 && ldx < K) || (((uintptr_t)x | (uintptr_t)w) & 15))
    return (int)hipErrorInvalidValue;
  constexpr int R = GLU ? kFewN / 2 : kFewN;
  const dim3 g((N + R - 1) / R);
#define K8S_FR(MM) \
  case MM: hipLaunchKernelGGL((few_rows_f32_kernel<MM, GLU, ADD, SCALED>), g, dim3(256), 0, s, x, ldx, w, y, N, K, ad, sc); break
  if constexpr (ADD || SCALED) {
    switch (M) {
      K8S_FR(1);
      K8S_FR(2);
      K8S_FR(3);
      K8S_FR(4);
      default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
  } else {
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

// x += s(m) a . w^T [+ es emb[id]];  h = x nw, part[m][N / 4] the sums of x^2 over 4 columns each (s(m): 1, or 1 / sqrt(sum of
// rs[m][0 .. rn) / rw + reps)).  M <= 4, N % 4 == 0.
K8S_API int k8s_few_rows_f32_add(const float* a, int lda, const float* w, float* x, const float* rs, int rn, float rw, float reps,
                                 const int* eid, const float* emb, float es, const float* nw, float* h, float* part, int M, int N,
                                 int K, hipStream_t s) {
  if (N % 4 || !x || !nw || !h || !part || (eid && !emb) || (rs && (rn < 1 || rn > kFewSums || !(rw > 0.f))))
    return (int)hipErrorInvalidValue;
  return few_rows<false, true>(a, lda, w, h, M, N, K, s, FewAdd{x, rs, eid, emb, nw, part, rw, reps, es, rn});
}

// k8s_few_rows_f32 (glu: k8s_few_rows_glu_f32) of rows that are still to be divided by sqrt(sum of part[m] / K + eps).
// M <= 4, K % 16 == 0, up to 4096; part on 16 bytes.
K8S_API int k8s_few_rows_f32_scaled(const float* x, int ldx, const float* w, float* y, int M, int N, int K, int glu,
                                    const float* part, float eps, hipStream_t s) {
  if (K % 16 || K > kFewMaxK || !part || ((uintptr_t)part & 15)) return (int)hipErrorInvalidValue;
  const FewScale sc{part, eps};
  return glu ? few_rows<true, false, true>(x, ldx, w, y, M, N, K, s, FewAdd{}, sc)
             : few_rows<false, false, true>(x, ldx, w, y, M, N, K, s, FewAdd{}, sc);
}
