// Products of 17 to 64 rows, Y[M][N] = X[M][K] . W[N][K]^T, bf16 operands, fp32 accumulation (steps of a batch of single tokens).
//
// The weights' stream is laid out as in gemm_rows.hip: four waves take a quarter of a workgroup's K each and never wait for each
// other before the end.  Here the rows are as many bytes as a workgroup's weights, so they come the same way, eight lanes to a row of
// 128 bytes, two chunks of 64 entries of both in flight in registers, and are turned into fragments in the wave's own LDS (16-byte
// piece j of row n at piece j ^ (n & 7): no bank conflicts).  Every byte of X and W passes a compute unit once, where the strips of
// gemm_stream.hip have a barrier a chunk and read the strip of W once for every 16 rows out of LDS.
//
// What bounds it: what a compute unit has in flight.  The time grows with X's bytes as if they took a third of the time of W's
// (16384 x 2048 SwiGLU 12.9, 13.2, 14.6, 16.1 us at 17, 32, 48, 64 rows, its weights alone 10.9), and neither eight waves (16.6,
// 16.8, 17.5, 29), three or four chunks in flight (13.2 - 18.8) nor starting the strips at different chunks (13.4, 13.6, 15.6, 16.2)
// takes it away.  us, before (gemm_stream.hip, gemm_rows.hip, hipBLASLt by shape) / this:
//   rows                        24            32            48            64
//   16384 x 2048 SwiGLU     13.8 / 13.2   14.0 / 13.3   18.2 / 14.6   17.5 / 16.1
//   16384 x 4096 SwiGLU     25.5 / 23.7   24.3 / 23.4   38.4 / 24.9   31.5 / 27.3
//   8192 x 2048 relu^2       8.9 / 7.9     9.5 / 8.2    11.2 / 9.4    11.4 / 10.4
//   2560 x 2048              9.3 / 6.6     9.4 / 7.0     9.9 / 8.1    10.1 / 9.3
//   2576 x 2048, fp32 out    7.3 / 6.7     8.1 / 7.2     9.9 / 8.2    10.1 / 9.3
//   16384 x 2048, fp32 out  13.6 / 13.1   14.2 / 13.4   17.8 / 14.7   18.0 / 16.3
//   2048 x 8192, K ranges    9.2 / 8.0     9.1 / 8.4     9.5 / 9.7     9.7 / 10.7    (and the norm's pass, which has four planes to
//                           13.2 / 12.1   13.3 / 11.8   13.6 / 13.2   14.1 / 14.4     read for eight)
// The rule of what it takes: ops/linear.py, batch_plan.
#include "common.h"
#include "gates.h"

namespace k8s {
namespace batch {

enum Out { kBf16 = 0, kF32 = 1, kSilu = 2, kRelu2 = 3 };
constexpr int NW = 4;                    // waves
constexpr int CH = 64;                   // K entries of a chunk: rows of 128 bytes

// a wave's LDS: a chunk of W and of X, at the end its share of the sums (fp32)
constexpr int wave_lds(int MT, int NF) {
  const int staged = 2 * CH * 16 * (MT + NF), sums = 4 * 16 * MT * 16 * NF;
  return staged > sums ? staged : sums;
}

// grid (strips, K ranges); K range of kslice = NW waves x whole chunks.  MT, NF: 16-row fragments of X and of W.  SwiGLU: 8 NF gate rows,
// then their up rows.  The last strip may begin within the one before it, which writes the columns that both have.
template <int MT, int NF, int OUT>
__global__ void __launch_bounds__(64 * NW, MT + NF < 7 ? 2 : 1)
    gemm_batch_kernel(const uint16_t* __restrict__ x, int ldx, const uint16_t* __restrict__ w, void* __restrict__ y, int ldy, int M,
                      int N, int K, int kslice) {
  constexpr int HR = 8 * NF, NWL = 2 * NF, NXL = 2 * MT;    // load instructions of a chunk: 8 rows each
  constexpr int WL = wave_lds(MT, NF);
  constexpr int STRIP = (OUT == kSilu ? 8 : 16) * NF;
  __shared__ __attribute__((aligned(16))) unsigned char sm[NW * WL];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int kw = kslice / NW, kbeg = blockIdx.y * kslice + wv * kw, nch = kw / CH;
  const int n0 = min((int)blockIdx.x * STRIP, N - STRIP);
  uint16_t* const ws = reinterpret_cast<uint16_t*>(sm + wv * WL);
  uint16_t* const xs = ws + 16 * NF * CH;

  // a lane: row lane / 8 of a load's 8, its piece lane % 8 of 16 bytes, which lies at piece ^ row in LDS
  const int hi = lane >> 3, pc = lane & 7;
  const uint32_t woff = 2u * ((uint32_t)hi * K + 8 * pc);
  uint32_t xoff[NXL];
#pragma unroll
  for (int i = 0; i < NXL; ++i) xoff[i] = 2u * ((uint32_t)min(8 * i + hi, M - 1) * ldx + 8 * pc);
  const int dst = hi * CH + 8 * (pc ^ hi);
  u16x8 wq[2][NWL], xq[2][NXL];
  auto load = [&](int st, int c) {
#pragma unroll
    for (int i = 0; i < NWL; ++i) {
      const size_t row = OUT == kSilu ? (size_t)n0 + (8 * i >= HR ? N : 0) + 8 * i % HR : (size_t)n0 + 8 * i;
      wq[st][i] = ldw_nt<u16x8>(reinterpret_cast<const char*>(w + row * K + kbeg + c * CH) + woff);
    }
#pragma unroll
    for (int i = 0; i < NXL; ++i)
      xq[st][i] = *reinterpret_cast<const u16x8*>(reinterpret_cast<const char*>(x + kbeg + c * CH) + xoff[i]);
  };
  f32x4 acc[MT][NF];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[mt][f] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int st, int c, bool more) {
#pragma unroll
    for (int i = 0; i < NWL; ++i) *reinterpret_cast<u16x8*>(ws + 8 * i * CH + dst) = wq[st][i];
#pragma unroll
    for (int i = 0; i < NXL; ++i) *reinterpret_cast<u16x8*>(xs + 8 * i * CH + dst) = xq[st][i];
    wave_lds_fence();
    __builtin_amdgcn_sched_barrier(0);
    if (more) load(st, c + 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < CH / 32; ++s) {
      const int at = r * CH + 8 * ((4 * s + g) ^ (r & 7));
      bf16x8 wf[NF], xf[MT];
#pragma unroll
      for (int f = 0; f < NF; ++f) wf[f] = *reinterpret_cast<const bf16x8*>(ws + 16 * f * CH + at);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xf[mt] = *reinterpret_cast<const bf16x8*>(xs + 16 * mt * CH + at);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[mt][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[f], xf[mt], acc[mt][f], 0, 0, 0);
    }
    wave_lds_fence();
    __builtin_amdgcn_sched_barrier(0);
  };
  load(0, 0);
  __builtin_amdgcn_sched_barrier(0);
  if (nch > 1) {
    load(1, 1);
    __builtin_amdgcn_sched_barrier(0);
    int c = 0;
    for (; c + 3 < nch; c += 2) {
      step(0, c, true);
      step(1, c + 1, true);
    }
    if (c + 2 < nch) {
      step(0, c, true);
      step(1, c + 1, false);
      step(0, c + 2, false);
    } else {
      step(0, c, false);
      step(1, c + 1, false);
    }
  } else {
    step(0, 0, false);
  }

  // acc[mt][f][v]: this wave's share of row 16 mt + r, strip column 16 f + 4 g + v; summed over the waves in their order.  Four columns
  // p of row m lie at piece p ^ m.
  constexpr int PP = 4 * NF;
  float* const red = reinterpret_cast<float*>(ws);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int f = 0; f < NF; ++f)
      *reinterpret_cast<f32x4*>(red + ((16 * mt + r) * PP + ((4 * f + g) ^ (r & (PP - 1)))) * 4) = acc[mt][f];
  __syncthreads();
  auto total = [&](int m, int p) {
    const unsigned char* at = sm + 16 * (m * PP + (p ^ (m & (PP - 1))));
    f32x4 t = *reinterpret_cast<const f32x4*>(at);
#pragma unroll
    for (int q = 1; q < NW; ++q) t += *reinterpret_cast<const f32x4*>(at + q * WL);
    return t;
  };
  constexpr int OP = STRIP / 4;          // pieces of four results of a row
  for (int e = threadIdx.x; e < M * OP; e += 64 * NW) {
    const int m = e / OP, p = e % OP;
    if (n0 + 4 * p < (int)blockIdx.x * STRIP) continue;     // (the strip before has it)
    const f32x4 t = total(m, p);
    const size_t o = (size_t)m * ldy + n0 + 4 * p;
    if constexpr (OUT == kF32) {
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(y) + (size_t)blockIdx.y * M * N + o) = t;
    } else {
      u16x4 h;
      if constexpr (OUT == kSilu) {      // gate and up rounded as the separate pass reads them
        const f32x4 u = total(m, OP + p);
#pragma unroll
        for (int v = 0; v < 4; ++v) h[v] = f2bf(silu_gate(bf2f(f2bf(t[v]))) * bf2f(f2bf(u[v])));
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) h[v] = f2bf(OUT == kRelu2 ? relu_sq_f(t[v]) : t[v]);
      }
      *reinterpret_cast<u16x4*>(reinterpret_cast<uint16_t*>(y) + o) = h;
    }
  }
}

template <int MT, int NF>
static int launch(const void* x, int ldx, const void* w, void* y, int ldy, int M, int N, int K, int ranges, int out, hipStream_t s) {
  const int strip = (out == kSilu ? 8 : 16) * NF;
  if (N < strip || (out == kSilu && N % strip) || K % (ranges * NW * CH)) return (int)hipErrorInvalidValue;
  const dim3 g((N + strip - 1) / strip, ranges), b(64 * NW);
#define K8S_BATCH(OUT)                                                                                                       \
  hipLaunchKernelGGL((gemm_batch_kernel<MT, NF, OUT>), g, b, 0, s, (const uint16_t*)x, ldx, (const uint16_t*)w, y, ldy, M, N, K, \
                     K / ranges)
  switch (out) {
    case kBf16: K8S_BATCH(kBf16); break;
    case kF32: K8S_BATCH(kF32); break;
    case kSilu: K8S_BATCH(kSilu); break;
    default: K8S_BATCH(kRelu2); break;
  }
#undef K8S_BATCH
  return (int)hipGetLastError();
}
template <int MT>
static int launch_as(const void* x, int ldx, const void* w, void* y, int ldy, int M, int N, int K, int nf, int ranges, int out,
                     hipStream_t s) {
  switch (nf) {
    case 2: return launch<MT, 2>(x, ldx, w, y, ldy, M, N, K, ranges, out, s);
    case 4: return launch<MT, 4>(x, ldx, w, y, ldy, M, N, K, ranges, out, s);
  }
  return (int)hipErrorInvalidValue;
}

}  // namespace batch
}  // namespace k8s

using namespace k8s;

// nf: 16-row fragments of W of a workgroup, 2 or 4; K in whole chunks of 64 for each of its four waves; ranges > 1: fp32
// planes [ranges][M][N].  out: 0 bf16, 1 fp32, 2 silu(x . w[0:N]^T) * (x . w[N:2N]^T), 3 max(., 0)^2.  N a multiple of 16, no smaller
// than a strip, of SwiGLU a multiple of 8 nf; x (its rows too), w and y lie on 16 bytes.
K8S_API int k8s_gemm_batch(const void* x, int ldx, const void* w, void* y, int ldy, int M, int N, int K, int nf, int ranges,
                           int out, hipStream_t s) {
  using namespace k8s::batch;
  auto off = [](const void* p) { return !p || ((uintptr_t)p & 15); };
  if (M < 1 || M > 64 || N < 1 || N % 16 || K < 1 || ranges < 1 || (ranges > 1 && (out != kF32 || ldy != N)) || out < kBf16 || out > kRelu2 ||
      ldx % 8 || ldx < K || ldx > (1 << 24) || K > (1 << 24) || ldy < N || ldy % 8 || off(x) || off(w) || off(y))
    return (int)hipErrorInvalidValue;
  if (M <= 32) return launch_as<2>(x, ldx, w, y, ldy, M, N, K, nf, ranges, out, s);
  if (M <= 48) return launch_as<3>(x, ldx, w, y, ldy, M, N, K, nf, ranges, out, s);
  return launch_as<4>(x, ldx, w, y, ldy, M, N, K, nf, ranges, out, s);
}
