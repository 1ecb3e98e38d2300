// The product of ONE row behind the residual's pass that makes its input, in one launch:
//   x' = x + (what the sublayer before gave),  h = norm(x') in bf16,  y = W . h   (W [N][K] bf16, fp32 sums, K <= 2048).
//
// A reply step of one sequence is a chain of launches in which every second one is that pass: 3 to 4 us in which one to
// eight workgroups read some 40 KB while the weights of the product behind it wait.  Here every workgroup makes the row for
// itself, from the caches, while all of its weights are already on their way: a wave takes RW rows of W whole (or the
// workgroup's range of K), a load instruction is 1 KB of one row, and a wave's whole share (up to 64 registers a lane) is
// asked for right behind the row's own loads -- loads are waited for in the order they were asked in, so that the pass
// does not wait for a weight and its chain of latencies runs under the stream.  With one row there is nothing for a matrix
// instruction to share, so the sums are fp32 multiply-adds on the registers that the loads filled.
// Workgroups of eight waves: each reads those 40 KB, and with four waves the caches' rate showed (SwiGLU 13.7 against 12.8).
// What bounds it is the weights' way from memory, below some 16 MB the chain of latencies.
//
// us in a replayed chain with cold weights, K 2048, four planes: pass and product (gemm_rows.hip) apart / the product alone /
// this:  8192 SwiGLU 15.3 / 12.3 / 12.8;  8192 bf16 10.4 / 7.3 / 7.4;  2560 fp32 6.9 / 4.0 / 4.5;  1088 fp32 5.9 / 2.9 / 3.7;
// 32768 fp32 26.1 / 23.0 / 23.3;  behind the dyt pass 8192 squared relu 9.6 / 7.3 / 7.6, 8736 fp32 10.9 / 8.5 / 9.6, 2576
// fp32 6.7 / 4.3 / 4.4, 2304 bf16 6.6 / 4.2 / 4.4, 32768 fp32 25.5 / 22.8 / 23.6.
//
// The residual goes to a second buffer, written by one workgroup: the others are still reading the first.  The pass's
// arithmetic is that of hyper_step_kernel with one stream (hyper_conn.hip) and add_dyt4_kernel (dyt_ops.hip), so that x' and
// h have their bits.
#include "common.h"

namespace k8s {

enum StepNorm { kStepRms = 0, kStepDyt = 1 };
enum StepOut { kStepBf16 = 0, kStepF32 = 1, kStepSilu = 2, kStepRelu2 = 3 };   // as in gemm_rows.hip

constexpr int kStepCols = 512;       // entries of K that a wave's load instruction covers
constexpr int kStepPlanes = 4;       // planes of y, at most
constexpr int kStepSums = 64;        // of rs, at most: one a lane
constexpr int kStepWaves = 8;
constexpr int kStepMaxK = 2048;     // four entries a thread

struct RowStep {
  const float* x;        // [K]
  float* x_out;          // [K], another buffer
  const float* y;        // [yp][K] planes, times sy
  const float* y2;       // [yp2][K], times sy2; or null (dyt)
  const float* rs;       // [rn] or null (rms): y is divided by sqrt(sum / rw + reps)
  const int* eid;        // rows of emb, times es, are added too; or null (rms)
  const uint16_t* emb;
  const float* w;        // the norm's weight
  const float* b;        // dyt: tanh(alpha x') w + b
  uint16_t* h_out;       // [K] or null: h for further readers
  float sy, sy2, rw, reps, es, alpha, eps;
  int yp, yp2, rn;
};

// four entries of a sum of n <= kStepPlanes planes, asked for at once and not waited for (past the last plane: it again)
struct PlaneLoads {
  f32x4 p[kStepPlanes];
  __device__ __forceinline__ void ask(const float* q, size_t step, int n) {
#pragma unroll
    for (int k = 0; k < kStepPlanes; ++k) p[k] = *reinterpret_cast<const f32x4*>(q + (size_t)min(k, n - 1) * step);
  }
  __device__ __forceinline__ f32x4 sum(int n) const {     // p0 + p1 + ... as in sum_planes4
    f32x4 v = p[0];
#pragma unroll
    for (int k = 1; k < kStepPlanes; ++k)
      if (k < n) v += p[k];
    return v;
  }
};

// LDS written before is there for the whole workgroup; leaves loads from memory in flight
__device__ __forceinline__ void step_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// grid (strips of 8 RW rows of W, ranges of K); SwiGLU: half a strip's rows are gate rows, half the up rows of the same columns.
template <int NORM, int OUT, int RW, int NCH>
__global__ void __launch_bounds__(64 * kStepWaves, 2)
    gemm_row_step_kernel(RowStep a, const uint16_t* __restrict__ w, void* __restrict__ y, int N, int K) {
  constexpr int KS = kStepCols * NCH;                            // this workgroup's range of K
  __shared__ __attribute__((aligned(16))) uint16_t xs[NORM == kStepDyt ? KS : kStepMaxK];
  __shared__ float red[kStepWaves];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int kbeg = blockIdx.y * KS;
  const int from = NORM == kStepDyt ? kbeg : 0, len = NORM == kStepDyt ? KS : K;   // the entries this workgroup makes
  // ---- the row: four neighbouring entries a thread (past the end: the last ones again, not used)
  const int at = from + min(4 * tid, len - 4);
  const bool on = 4 * tid < len;
  f32x4 nb;
  u16x4 ev;
  PlaneLoads yl, y2l;
  float rv = 0.f;
  f32x4 xv = *reinterpret_cast<const f32x4*>(a.x + at);
  yl.ask(a.y + at, K, a.yp);
  const f32x4 nw = *reinterpret_cast<const f32x4*>(a.w + at);
  if (NORM == kStepDyt) nb = *reinterpret_cast<const f32x4*>(a.b + at);
  if (NORM == kStepDyt && a.y2) y2l.ask(a.y2 + at, K, a.yp2);
  if (NORM == kStepRms && a.rs) rv = a.rs[min(lane, a.rn - 1)];
  const bool embeds = NORM == kStepRms && a.eid;
  if (embeds) ev = *reinterpret_cast<const u16x4*>(a.emb + (size_t)a.eid[0] * K + at);
  __builtin_amdgcn_sched_barrier(0);
  // ---- the weights
  constexpr int HR = OUT == kStepSilu ? RW / 2 : RW;             // rows of a half (of all)
  const int n0 = (blockIdx.x * kStepWaves + wv) * HR;
  u16x8 wq[RW][NCH];
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const size_t row = n0 + i % HR + (i < HR ? 0 : (size_t)N);
#pragma unroll
    for (int j = 0; j < NCH; ++j) wq[i][j] = ldw_nt<u16x8>(w + row * K + kbeg + j * kStepCols + 8 * lane);
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- the pass
  const bool store = blockIdx.x == 0 && (NORM == kStepDyt || blockIdx.y == 0);
  f32x4 yv = yl.sum(a.yp);
  float r = 1.f;
  if (NORM == kStepDyt) {
#pragma unroll
    for (int k = 0; k < 4; ++k) xv[k] = fmaf(a.sy, yv[k], xv[k]);
    if (a.y2) {
      yv = y2l.sum(a.yp2);
#pragma unroll
      for (int k = 0; k < 4; ++k) xv[k] = fmaf(a.sy2, yv[k], xv[k]);
    }
  } else {
    if (a.rs) yv *= 1.f / sqrtf(wave_sum(lane < a.rn ? rv : 0.f) / a.rw + a.reps);
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      xv[k] = yv[k] + xv[k];
      if (embeds) xv[k] = fmaf(a.es, bf2f(ev[k]), xv[k]);
      ss = fmaf(xv[k], xv[k], ss);
    }
    ss = wave_sum(on ? ss : 0.f);
    if (lane == 0) red[wv] = ss;
    step_barrier();
    float all = 0.f;
#pragma unroll
    for (int k = 0; k < kStepWaves; ++k) all += red[k];
    r = 1.f / sqrtf(all / (float)K + a.eps);
  }
  if (on) {
    u16x4 h;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      h[k] = f2bf(NORM == kStepDyt ? fmaf(tanhf(a.alpha * xv[k]), nw[k], nb[k]) : xv[k] * r * nw[k]);
    *reinterpret_cast<u16x4*>(xs + 4 * tid) = h;
    if (store) {
      *reinterpret_cast<f32x4*>(a.x_out + at) = xv;
      if (a.h_out) *reinterpret_cast<u16x4*>(a.h_out + at) = h;
    }
  }
  step_barrier();
  // ---- the product
  float hf[NCH][8], acc[RW] = {};
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const u16x8 hv = *reinterpret_cast<const u16x8*>(xs + (kbeg - from) + j * kStepCols + 8 * lane);
#pragma unroll
    for (int e = 0; e < 8; ++e) hf[j][e] = bf2f(hv[e]);
  }
#pragma unroll
  for (int i = 0; i < RW; ++i)                                   // in the order in which they were asked for
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[i] = fmaf(hf[j][e], bf2f(wq[i][j][e]), acc[i]);
  const float t = wave_sums<RW>(acc);
  constexpr int G = 64 / RW;                                     // lanes that end with the same sum
  const int i = lane / G;
  if constexpr (OUT == kStepSilu) {
    const float fa = bf2f(f2bf(t)), fb = bf2f(f2bf(__shfl_xor(t, 32, 64)));   // rounded as the separate pass reads them
    if (lane < 32 && lane % G == 0) reinterpret_cast<uint16_t*>(y)[n0 + i] = f2bf(silu_gate(fa) * fb);
  } else if (lane % G == 0) {
    if constexpr (OUT == kStepF32)
      reinterpret_cast<float*>(y)[(size_t)blockIdx.y * N + n0 + i] = t;
    else
      reinterpret_cast<uint16_t*>(y)[n0 + i] = f2bf(OUT == kStepRelu2 ? relu_sq_f(t) : t);
  }
}

template <int NORM, int OUT, int RW>
static int row_step_launch(const RowStep& a, const void* w, void* y, int N, int K, int ranges, hipStream_t s) {
  const int strip = kStepWaves * (OUT == kStepSilu ? RW / 2 : RW), nch = K / kStepCols / ranges;
  if (N % strip) return (int)hipErrorInvalidValue;
  const dim3 g(N / strip, ranges), b(64 * kStepWaves);
#define K8S_STEP(C) \
  case C: hipLaunchKernelGGL((gemm_row_step_kernel<NORM, OUT, RW, C>), g, b, 0, s, a, (const uint16_t*)w, y, N, K); break
  switch (nch) {
    K8S_STEP(1);
    K8S_STEP(2);
    K8S_STEP(3);
    K8S_STEP(4);
    default: return (int)hipErrorInvalidValue;
  }
#undef K8S_STEP
  return (int)hipGetLastError();
}

template <int RW>
static int row_step_any(int norm, int out, const RowStep& a, const void* w, void* y, int N, int K, int ranges, hipStream_t s) {
  if (norm == kStepRms) {
    switch (out) {
      case kStepBf16: return row_step_launch<kStepRms, kStepBf16, RW>(a, w, y, N, K, ranges, s);
      case kStepF32: return row_step_launch<kStepRms, kStepF32, RW>(a, w, y, N, K, ranges, s);
      case kStepSilu: return row_step_launch<kStepRms, kStepSilu, RW>(a, w, y, N, K, ranges, s);
    }
  } else {
    switch (out) {
      case kStepBf16: return row_step_launch<kStepDyt, kStepBf16, RW>(a, w, y, N, K, ranges, s);
      case kStepF32: return row_step_launch<kStepDyt, kStepF32, RW>(a, w, y, N, K, ranges, s);
      case kStepRelu2: return row_step_launch<kStepDyt, kStepRelu2, RW>(a, w, y, N, K, ranges, s);
    }
  }
  return (int)hipErrorInvalidValue;
}

static bool row_step_ok(const RowStep& a, const void* w, const void* y, int N, int K, int nf, int ranges, int out) {
  auto off = [](const void* p, int n) { return ((uintptr_t)p % n) != 0; };
  return a.x && a.x_out && a.x_out != a.x && a.y && a.yp >= 1 && a.yp <= kStepPlanes && a.w && w && y && N > 0 &&
         K >= kStepCols && K <= kStepMaxK &&
         ranges >= 1 && K % (kStepCols * ranges) == 0 && (nf == 1 || nf == 2) && (ranges == 1 || out == kStepF32) &&
         !off(a.x, 16) && !off(a.x_out, 16) && !off(a.y, 16) && !off(a.y2, 16) && !off(a.w, 16) && !off(a.b, 16) &&
         !off(a.h_out, 8) && !off(a.emb, 8) && !off(w, 16);
}

}  // namespace k8s

using namespace k8s;

// nf: 1 or 2, 16 nf rows of w a workgroup; ranges > 1: fp32 planes [ranges][N].  out: 0 bf16, 1 fp32, 2 SwiGLU (w [2N][K]).
K8S_API int k8s_gemm_row_step_rms(const float* x, float* x_out, const float* y, int yp, const float* rs, int rn, float rw,
                                  float reps, const int* eid, const void* emb, float es, const float* nw, float eps, void* h_out,
                                  const void* w, void* out, int N, int K, int nf, int ranges, int kind, hipStream_t s) {
  RowStep a{};
  a.x = x, a.x_out = x_out, a.y = y, a.yp = yp, a.rs = rs, a.rn = rn, a.rw = rw, a.reps = reps, a.eid = eid;
  a.emb = (const uint16_t*)emb, a.es = es, a.w = nw, a.eps = eps, a.h_out = (uint16_t*)h_out;
  if (!row_step_ok(a, w, out, N, K, nf, ranges, kind) || (eid && !emb) || (rs && (rn < 1 || rn > kStepSums || !(rw > 0.f))))
    return (int)hipErrorInvalidValue;
  return nf == 1 ? row_step_any<2>(kStepRms, kind, a, w, out, N, K, ranges, s)
                 : row_step_any<4>(kStepRms, kind, a, w, out, N, K, ranges, s);
}

// The same behind x' = x + sy y (+ sy2 y2), h = tanh(alpha x') nw + nb.  kind: 0 bf16, 1 fp32, 3 max(., 0)^2.
K8S_API int k8s_gemm_row_step_dyt(const float* x, float* x_out, const float* y, int yp, float sy, const float* y2, int yp2,
                                  float sy2, float alpha, const float* nw, const float* nb, void* h_out, const void* w,
                                  void* out, int N, int K, int nf, int ranges, int kind, hipStream_t s) {
  RowStep a{};
  a.x = x, a.x_out = x_out, a.y = y, a.yp = yp, a.sy = sy, a.y2 = y2, a.yp2 = yp2, a.sy2 = sy2, a.alpha = alpha;
  a.w = nw, a.b = nb, a.h_out = (uint16_t*)h_out;
  if (!row_step_ok(a, w, out, N, K, nf, ranges, kind) || !nb || (y2 && (yp2 < 1 || yp2 > kStepPlanes)))
    return (int)hipErrorInvalidValue;
  return nf == 1 ? row_step_any<2>(kStepDyt, kind, a, w, out, N, K, ranges, s)
                 : row_step_any<4>(kStepDyt, kind, a, w, out, N, K, ranges, s);
}
