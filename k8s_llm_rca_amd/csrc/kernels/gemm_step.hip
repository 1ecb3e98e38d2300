// A sublayer's last product for up to 16 rows, together with all that stands between it and the next sublayer's input:
//   x += sy s(m) (A . W^T) [+ sy2 (A2 . W2^T)] [+ es emb[id]]          (x [M][N] fp32, in place)
//   h  = tanh(alpha x) nw + nb  in bf16,      or      h = x nw in bf16 and the row's sum of squares in parts,
// which the product behind divides its sums by (gemm_rows.hip, RowScale): the root mean square is one factor a row, so that it
// may follow the sums, and no launch has to wait for whole rows.  s(m) is the same for the operand itself (rs: its sums of
// squares, one of them a head).
//
// A reply step is a chain of launches, in which the residual's pass between two products (sums of the K ranges, addition,
// norm) was one of 4.6 us that moves some 100 KB.  For the epilogue to own its columns a workgroup takes 8 rows of W over all
// of K: 256 workgroups at 2048 columns, every wave with an eighth of K and its whole share of W and A asked for up front, in
// turn.  A load covers 8 rows x 128 bytes, whole lines, neighbouring lanes neighbouring pieces of a row, and is turned into
// fragments in the wave's own LDS (piece p of row r at p ^ r: no bank conflicts).  The matrix instruction takes what 8 rows of
// 128 bytes hold as it is: columns 0 - 7 are the rows' first 64 bytes, 8 - 15 the second, and where A is laid out the same way
// (up to 8 rows), the two diagonal blocks of its result are the two halves of K; the blocks beside them are of no use.  (9 to 16
// rows: one instruction with each half of K of A, of which the result keeps the matching columns.)
//
// What bounds it is the weights' way from memory; of A every workgroup reads all rows.  Loaded in fragment order (neighbouring
// lanes in different rows), W and A came at 36 KB a us and compute unit out of the second-level cache, where rows of 128 bytes
// come at 84, and A's share took as long as W's: us at 1, 4, 7, 8, 12, 16 rows so / turned in LDS:  2048 x 8192 8.2 / 8.0, 9.2 / 8.3,
// 9.9 / 8.4, 10.3 / 8.8, 12.1 / 9.9, 13.4 / 10.5;  2048 x 2048 4.1 / 4.0, 4.4 / 4.1, 4.6 / 4.2, 4.7 / 4.2, 5.1 / 4.6, 5.6 / 4.8;  4096 x
// 4096 8.0 / 7.9, 9.1 / 7.9, 10.2 / 8.5, 10.4 / 8.9, 12.6 / 9.9, 13.6 / 10.6;  6144 x 8192 20.4 / 19.4, 23.2 / 19.9, 26.2 / 21.0, 27.6 /
// 21.5, 33.2 / 27.1, 37.0 / 28.6.  (4 slots of LDS a wave, with 9 rows and more 2, so that two workgroups fit a compute unit: 4096 x
// 4096 at 16 rows 12.9 with four.)
#include "common.h"

namespace k8s {

constexpr int kSpWaves = 8, kSpCols = 8, kSpStep = 64;    // K entries of a load instruction
constexpr int kSpMaxLoads = 16, kSpMaxRows = 16, kSpSums = 64;

struct StepProduct {
  const uint16_t* a;     // [M][lda]
  const uint16_t* w;     // [N][K]
  const uint16_t* a2;    // [M][lda2], [N][K]: a second product, taken by the upper half of the waves; or null
  const uint16_t* w2;
  float* x;              // [M][N], in place
  const float* rs;       // [M][rn] or null: the first product is divided by sqrt(sum / rw + reps)
  const int* eid;        // [M]: rows of emb, times es, are added too; or null
  const uint16_t* emb;
  const float* nw;       // [N]
  const float* nb;       // [N]: the tanh form; null: the sums of squares go to part
  uint16_t* h;           // [M][N]
  float* part;           // [M][N / 8]
  float sy, sy2, rw, reps, es, alpha;
  int lda, lda2, rn;
};

// grid: strips of 8 rows of W.  MF: 8-row halves of the matrix instruction that A fills.
template <int NB, int MF>
__global__ void __launch_bounds__(64 * kSpWaves, 2) gemm_step_kernel(StepProduct p, int M, int N, int K) {
  constexpr int SLOTS = MF == 1 ? 4 : 2, RING = NB < SLOTS ? NB : SLOTS;
  __shared__ __attribute__((aligned(16))) uint16_t turn[kSpWaves][RING][8 * (MF + 1) * kSpStep];    // A's rows, then W's
  __shared__ float red[kSpWaves][2][8 * MF][kSpCols];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * kSpCols;
  // ---- what the epilogue needs: one entry of x a thread
  const int m = tid >> 3, n = n0 + (tid & 7);
  const bool mine = m < M;
  float xv = 0.f, nw = 0.f, nb = 0.f, rv[kSpSums / 8];
  int id = 0;
  if (mine) {
    if (p.eid) id = p.eid[m];
    xv = p.x[(size_t)m * N + n];
    nw = p.nw[n];
    if (p.nb) nb = p.nb[n];
    if (p.rs) {
#pragma unroll
      for (int j = 0; j < kSpSums / 8; ++j) {
        const int i = 8 * j + (tid & 7);
        rv[j] = i < p.rn ? p.rs[(size_t)m * p.rn + i] : 0.f;
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- this wave's K range, of the first or the second product
  const bool two = p.w2 != nullptr, second = two && wv >= kSpWaves / 2;
  const int kbeg = (second ? wv - kSpWaves / 2 : wv) * NB * kSpStep;
  const uint16_t* wp = (second ? p.w2 : p.w) + (size_t)(n0 + (lane >> 3)) * K + kbeg + 8 * (lane & 7);
  const uint16_t* a = second ? p.a2 : p.a;
  const int lda = second ? p.lda2 : p.lda;
  // A: lane -> row lane / 8 (of each 8), piece lane % 8 of 128 bytes, which lies at piece ^ row in LDS
  const int ar = lane >> 3, apc = lane & 7;
  const uint16_t* ap[MF];
#pragma unroll
  for (int f = 0; f < MF; ++f) ap[f] = a + (size_t)min(8 * f + ar, M - 1) * lda + kbeg + 8 * apc;
  u16x8 wq[NB];
  u16x8 aq[NB][MF];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    wq[i] = ldw_nt<u16x8>(wp + i * kSpStep);
#pragma unroll
    for (int f = 0; f < MF; ++f) {
      if constexpr (MF == 1) aq[i][f] = u16x8{};
      if (MF == 2 || ar < M) aq[i][f] = *reinterpret_cast<const u16x8*>(ap[f] + i * kSpStep);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  float ev = 0.f;
  if (mine && p.eid) ev = bf2f(p.emb[(size_t)id * N + n]);
  __builtin_amdgcn_sched_barrier(0);
  f32x4 acc[MF];
#pragma unroll
  for (int f = 0; f < MF; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  // fragments: MF 1: row r % 8, a piece of the half r / 8;  MF 2: row r, a piece of each half
  const int fr = MF == 1 ? r & 7 : r, fp = MF == 1 ? (r >> 3) * 4 + g : g;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    uint16_t* at = turn[wv][i % RING];
#pragma unroll
    for (int f = 0; f < MF; ++f) *reinterpret_cast<u16x8*>(at + (8 * f + ar) * kSpStep + 8 * (apc ^ ar)) = aq[i][f];
    uint16_t* wt = at + 8 * MF * kSpStep;
    *reinterpret_cast<u16x8*>(wt + ar * kSpStep + 8 * (apc ^ ar)) = wq[i];
    wave_lds_fence();
    const bf16x8 wf = *reinterpret_cast<const bf16x8*>(wt + (r & 7) * kSpStep + 8 * (((r >> 3) * 4 + g) ^ (r & 7)));
#pragma unroll
    for (int f = 0; f < MF; ++f) {
      const bf16x8 af = *reinterpret_cast<const bf16x8*>(at + fr * kSpStep + 8 * ((fp + 4 * f) ^ (fr & 7)));
      acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, wf, acc[f], 0, 0, 0);
    }
  }
  // acc[f][v]: row 4 g + v, column r (8 - 15: the second 64 bytes of the rows)
  if constexpr (MF == 1) {
    if ((g >> 1) == (r >> 3)) {
#pragma unroll
      for (int v = 0; v < 4; ++v) red[wv][r >> 3][(4 * g + v) & 7][r & 7] = acc[0][v];
    }
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wv][r >> 3][4 * g + v][r & 7] = r < 8 ? acc[0][v] : acc[MF - 1][v];
  }
  __syncthreads();
  if (!mine) return;
  float t[2] = {0.f, 0.f};
#pragma unroll
  for (int q = 0; q < kSpWaves; ++q) {
    const float v = red[q][0][m][tid & 7] + red[q][1][m][tid & 7];
    t[two ? q / (kSpWaves / 2) : 0] += v;
  }
  if (p.rs) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < kSpSums / 8; ++j) s += rv[j];
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) s += __shfl_xor(s, o, 8);
    t[0] *= 1.f / sqrtf(s / p.rw + p.reps);
  }
  xv = fmaf(p.sy, t[0], xv);
  if (two) xv = fmaf(p.sy2, t[1], xv);
  if (p.eid) xv = fmaf(p.es, ev, xv);
  p.x[(size_t)m * N + n] = xv;
  if (p.nb) {
    p.h[(size_t)m * N + n] = f2bf(fmaf(tanhf(p.alpha * xv), nw, nb));
  } else {
    p.h[(size_t)m * N + n] = f2bf(xv * nw);
    float s = xv * xv;
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) s += __shfl_xor(s, o, 8);
    if ((tid & 7) == 0) p.part[(size_t)m * (N / kSpCols) + blockIdx.x] = s;
  }
}

static int step_product(const StepProduct& p, int M, int N, int K, hipStream_t s) {
  auto off = [](const void* q, int n) { return ((uintptr_t)q % n) != 0; };
  const int waves = p.w2 ? kSpWaves / 2 : kSpWaves, nb = K / (kSpStep * waves);
  if (M <= 0 || M > kSpMaxRows || N <= 0 || N % kSpCols || K <= 0 || K % (kSpStep * waves) || nb > kSpMaxLoads || !p.a ||
      !p.w || !p.x || !p.nw || !p.h || (!p.nb && !p.part) || (p.eid && !p.emb) || off(p.a, 16) || off(p.w, 16) ||
      p.lda % 8 || (M > 1 && p.lda < K) || (p.rs && (p.rn < 1 || p.rn > kSpSums || !(p.rw > 0.f))))
    return (int)hipErrorInvalidValue;
  if (p.w2 && (!p.a2 || off(p.a2, 16) || off(p.w2, 16) || p.lda2 % 8 || (M > 1 && p.lda2 < K)))
    return (int)hipErrorInvalidValue;
  const dim3 g(N / kSpCols), b(64 * kSpWaves);
#define K8S_SP(NB)                                                                                     \
  case NB:                                                                                             \
    if (M <= 8)                                                                                        \
      hipLaunchKernelGGL((gemm_step_kernel<NB, 1>), g, b, 0, s, p, M, N, K);                           \
    else                                                                                               \
      hipLaunchKernelGGL((gemm_step_kernel<NB, 2>), g, b, 0, s, p, M, N, K);                           \
    break
  switch (nb) {
    K8S_SP(1);
    K8S_SP(2);
    K8S_SP(3);
    K8S_SP(4);
    K8S_SP(5);
    K8S_SP(6);
    K8S_SP(7);
    K8S_SP(8);
    K8S_SP(10);
    K8S_SP(12);
    K8S_SP(14);
    K8S_SP(16);
    default: return (int)hipErrorInvalidValue;
  }
#undef K8S_SP
  return (int)hipGetLastError();
}

}  // namespace k8s

using namespace k8s;

// x += s(m) a . w^T [+ es emb[id]];  h = bf16(x nw), part[m][N / 8] the sums of x^2 over 8 columns each.
K8S_API int k8s_gemm_step_rms(const void* a, int lda, const void* w, float* x, const float* rs, int rn, float rw, float reps,
                              const int* eid, const void* emb, float es, const float* nw, void* h, float* part, int M, int N,
                              int K, hipStream_t s) {
  StepProduct p{};
  p.a = (const uint16_t*)a, p.lda = lda, p.w = (const uint16_t*)w, p.x = x, p.sy = 1.f;
  p.rs = rs, p.rn = rn, p.rw = rw, p.reps = reps, p.eid = eid, p.emb = (const uint16_t*)emb, p.es = es;
  p.nw = nw, p.h = (uint16_t*)h, p.part = part;
  return step_product(p, M, N, K, s);
}

// x += sy a . w^T [+ sy2 a2 . w2^T];  h = bf16(tanh(alpha x) nw + nb).
K8S_API int k8s_gemm_step_dyt(const void* a, int lda, const void* w, float sy, const void* a2, int lda2, const void* w2,
                              float sy2, float* x, float alpha, const float* nw, const float* nb, void* h, int M, int N, int K,
                              hipStream_t s) {
  if (!nb) return (int)hipErrorInvalidValue;
  StepProduct p{};
  p.a = (const uint16_t*)a, p.lda = lda, p.w = (const uint16_t*)w, p.sy = sy;
  p.a2 = (const uint16_t*)a2, p.lda2 = lda2, p.w2 = (const uint16_t*)w2, p.sy2 = sy2;
  p.x = x, p.alpha = alpha, p.nw = nw, p.nb = nb, p.h = (uint16_t*)h;
  return step_product(p, M, N, K, s);
}
