// Products of up to 32 rows, Y[M][N] = X[M][K] . W[N][K]^T, bf16 operands, fp32 accumulation (steps of single tokens); of 17 to 32 rows
// those that gemm_batch.hip leaves.
//
// What bounds them is the weights' way from memory, so the kernel is laid out for that stream: every load instruction of W
// covers 256 bytes (CH = 128) or 128 bytes (CH = 64) of a row, not the 64 of a matrix fragment read straight from memory;
// the four waves of a workgroup take a quarter of its K each and never wait for each other before the end.  A wave holds two
// chunks of 16 NF rows x CH in flight in registers, turns one through its own LDS into fragments (16-byte piece j of row n
// at piece j ^ (n & 7): no bank conflicts) and asks for the next.  X goes from L2 into registers, behind the W that it
// belongs to, so that a step waits for its own loads and leaves the next W in flight.
//
// NF: 16-row fragments of W a workgroup takes.  More of them read X less often (X of 16 rows is as many bytes as one
// fragment of W) and leave fewer workgroups; the caller takes the one that leaves the fullest waves of 256.
//
// Read alone, 16384 x 2048 takes 10.9 us on this card, 28672 x 4096 35.0 and 128256 x 4096 152 (6.2, 6.7 and 6.9 TB/s).
// us, before (gemm_stream.hip, gemm_skinny.hip, hipBLASLt by shape) / this:
//   rows                          1            8            16           32
//   16384 x 2048 SwiGLU       16.2 / 12.0  16.7 / 12.2  16.4 / 12.5  16.6 / 14.6
//   28672 x 4096 SwiGLU       43.4 / 35.3  42.9 / 36.7  42.6 / 37.2  46.7 / 40.8
//   8192 x 2048                8.8 / 7.1    9.7 / 7.4   10.9 / 7.9   10.3 / 9.0
//   6144 x 4096               13.4 / 9.5   15.7 / 10.1  18.2 / 11.1  15.2 / 14.2
//   2048 x 8192, K ranges      8.3 / 7.4    9.0 / 7.6    9.1 / 8.1    9.1 / 8.5
//   32768 x 2048, fp32 out    32.0 / 21.4  32.1 / 21.5  32.1 / 22.5  34.3 / 24.5
//   128256 x 4096, fp32 out    184 / 160    194 / 165    199 / 171    210 / 194
#include "common.h"
#include "gates.h"
#include "norm_prologue.h"

namespace k8s {

enum RowsOut { kRowsBf16 = 0, kRowsF32 = 1, kRowsSilu = 2, kRowsRelu2 = 3, kRowsRope = 4, kRowsConv = 5 };

constexpr int kRowsWaves = 4;

// rotation and paged KV write behind the qkv projection (the layout of rope_kv_kernel, norm_act.hip)
struct RowsRope {
  const int* pos;
  const float* cos_sin;  // [max_pos][128]: cos[0..63] | sin[0..63]
  const int* slots;      // [M], -1: no write; or null
  uint16_t* kc;          // [blocks][nkv][BS][128]
  uint16_t* vc;          // [blocks][nkv][128][BS]
  int nq, nkv, BS;
};

// The first `cols` columns rounded to bf16 and convolved with their sequence's last inputs (short_conv_tile_kernel, mixer_ops.hip:
// every row the only one of its sequence), the rest as they are, in fp32
struct RowsConv {
  int cols, taps, ldr, act;
  const float* w;        // [cols][taps], the last is the row's own
  float* tail;           // [slots][taps - 1][cols]
  const int* pos0;
  const int* slot;
  float* rest;           // [M][ldr]
};
constexpr int kConvTaps = 4;

// How x comes: as it is; normed by every workgroup (NormIn); or the product's rows are divided by the root mean square of what
// x was made from (RowScale), whose sums of squares a gemm_step (gemm_step.hip) left in parts.
enum RowsIn { kRowsPlain = 0, kRowsNorm = 1, kRowsScaled = 2 };
constexpr int kRowsParts = 256;          // parts of a row's sum of squares, at most: four a lane

struct RowScale {
  const float* part;     // [M][parts]
  int parts;             // a multiple of 4
  float width, eps;
};

// a wave's LDS: one chunk of W, at the end its share of the sums (fp32)
constexpr int rows_lds(int MT, int NF, int CH) { return 16 * NF * (CH > 32 * MT ? CH : 32 * MT); }

// grid (strips, K ranges); K range of kslice = 4 waves x whole chunks.  Forms of two halves (SwiGLU: gate and up rows, rope:
// entries d and d + 64 of a head) take 8 NF rows of each.  NORM: x is the normed row block that the workgroup makes itself
// (norm_prologue.h) while its first weights are on their way; the row's own loads are asked for in front of them (6144 x 4096
// rotated 13.5 -> 11.6 us, 28672 x 4096 SwiGLU 39.4 -> 37.6, on four fragments instead of one 36.3).  Scaled: a wave sums the
// parts of up to four rows, asked for in front of the weights, and every sum is multiplied before it is rounded or stored.
// Convolved: a thread's first entry has its earlier inputs and taps asked for behind the first weights
// (2304 columns and 144 others, K 2048, 1 and 16 rows: three launches of 10.6 and 12.4 us -> 5.3 and 6.2).
template <int MT, int NF, int CH, int OUT, int IN>
__global__ void __launch_bounds__(kRowsWaves * 64, 2)
    gemm_rows_kernel(const uint16_t* __restrict__ x, int ldx, const uint16_t* __restrict__ w, void* __restrict__ y, int ldy,
                     int M, int N, int K, int kslice, RowsRope rp, NormIn nin, RowScale rsc, RowsConv cv) {
  constexpr bool NORM = IN == kRowsNorm, SCALED = IN == kRowsScaled;
  static_assert(!SCALED || MT == 1);
  constexpr bool kHalves = OUT == kRowsSilu || OUT == kRowsRope;
  constexpr int HR = 8 * NF;            // rows of a half
  constexpr int PP = CH / 8;            // 16-byte pieces of a row's chunk
  constexpr int RI = 64 / PP;           // rows of a load instruction
  constexpr int ND = 16 * NF / RI;      // load instructions a chunk
  constexpr int NS = CH / 32;           // matrix steps a chunk
  constexpr int WL = rows_lds(MT, NF, CH);
  __shared__ __attribute__((aligned(16))) uint16_t sm[kRowsWaves * WL];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int kw = kslice / kRowsWaves;   // K of a wave
  const int kbeg = blockIdx.y * kslice + wv * kw;
  const int nch = kw / CH;
  const int n0 = blockIdx.x * (kHalves ? HR : 16 * NF);     // first column (of a pair: its first half)
  size_t first = n0, gap = 0;           // W row of the strip's first row; from there to the second half's first
  if constexpr (OUT == kRowsSilu) gap = N;
  if constexpr (OUT == kRowsRope) first = (size_t)(n0 >> 6) * 128 + (n0 & 63), gap = 64;
  uint16_t* const mine = sm + wv * WL;

  // load i of a chunk: rows RI i .. + RI; a lane: row lane / PP of them, piece lane % PP
  const int hi = lane / PP, pc = lane % PP;
  const uint32_t voff = 2u * ((uint32_t)hi * K + 8 * pc);
  auto wsrc = [&](int i, int c) {
    const int row = RI * i;
    const size_t wr = kHalves ? first + (row >= HR ? gap : 0) + row % HR : first + row;
    return reinterpret_cast<const char*>(w) + 2 * (wr * K + kbeg + c * CH) + voff;
  };
  auto wdst = [&](int i) { return mine + (RI * i + hi) * CH + 8 * (pc ^ ((RI * i + hi) & 7)); };
  if constexpr (NORM) {
    x = k8s_norm_lds;
    ldx = K;
  }
  const uint16_t* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) xrow[mt] = x + (size_t)min(mt * 16 + r, M - 1) * ldx + kbeg + 8 * g;

  f32x4 acc[MT][NF];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[mt][f] = f32x4{0.f, 0.f, 0.f, 0.f};
  u16x8 wq[2][ND];
  bf16x8 xq[NS][MT];
  auto load_w = [&](int st, int c) {
#pragma unroll
    for (int i = 0; i < ND; ++i) wq[st][i] = ldw_nt<u16x8>(wsrc(i, c));
  };
  auto load_x = [&](int c) {
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) xq[s][mt] = *reinterpret_cast<const bf16x8*>(xrow[mt] + c * CH + 32 * s);
  };
  // asked for in this order: W0 X0 W1 | X1 W2 | X2 W3 ...  The scheduler must not change it: loads are waited for in order.
  auto step = [&](int st, int c, int left) {
#pragma unroll
    for (int i = 0; i < ND; ++i) *reinterpret_cast<u16x8*>(wdst(i)) = wq[st][i];
    wave_lds_fence();
    if constexpr (NORM) load_x(c);
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const bf16x8 wf = *reinterpret_cast<const bf16x8*>(mine + (16 * f + r) * CH + 8 * ((4 * s + g) ^ (r & 7)));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[mt][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xq[s][mt], wf, acc[mt][f], 0, 0, 0);
      }
    wave_lds_fence();
    __builtin_amdgcn_sched_barrier(0);
    if (!NORM && left > 0) load_x(c + 1);
    __builtin_amdgcn_sched_barrier(0);
    if (left > 1) load_w(st, c + 2);
    __builtin_amdgcn_sched_barrier(0);
  };
  NormRow nrow;
  u16x8 nwv[kNormMaxChunks];
  if constexpr (NORM) norm_ask(nrow, nwv, 0, M, nin);
  f32x4 pv[SCALED ? 4 : 1];
  if constexpr (SCALED) {
#pragma unroll
    for (int q = 0; q < 4; ++q)                                   // (past the last row or part: the last ones again, not used)
      pv[q] = *reinterpret_cast<const f32x4*>(rsc.part + (size_t)min(wv + kRowsWaves * q, M - 1) * rsc.parts +
                                              min(4 * lane, rsc.parts - 4));
  }
  // (rows and channels past the last: the last ones, not used)
  struct ConvAt {
    int p0;
    float* tl;
    const float* w;
  };
  auto conv_row = [&](int e) {
    const int m = min(e / (16 * NF), M - 1), c = min(n0 + e % (16 * NF), cv.cols - 1);
    return ConvAt{cv.pos0[m], cv.tail + (size_t)cv.slot[m] * (cv.taps - 1) * cv.cols + c, cv.w + (size_t)c * cv.taps};
  };
  float hist[kConvTaps], taps[kConvTaps];
  auto conv_ask = [&](const ConvAt& at) {
#pragma unroll
    for (int j = 0; j < kConvTaps; ++j) {
      taps[j] = at.w[min(j, cv.taps - 1)];
      hist[j] = j < cv.taps - 1 && at.p0 - (cv.taps - 1 - j) >= 0 ? at.tl[(size_t)j * cv.cols] : 0.f;
    }
  };
  ConvAt cat;
  if constexpr (OUT == kRowsConv) cat = conv_row(threadIdx.x);
  __builtin_amdgcn_sched_barrier(0);
  load_w(0, 0);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (!NORM) load_x(0);
  __builtin_amdgcn_sched_barrier(0);
  if (NORM || nch > 1) load_w(1, nch > 1 ? 1 : 0);   // (no branch between the row and its use: the waits count what is in flight)
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (OUT == kRowsConv) {
    conv_ask(cat);
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (NORM) {
    __shared__ float nscr[16];
    norm_rows_to_lds<true>(k8s_norm_lds, M, nin, blockIdx.x == 0 && blockIdx.y == 0, nscr, nrow, nwv);
  }
  __shared__ float factor[SCALED ? 16 : 1];
  if constexpr (SCALED) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float ss = wave_sum_dpp(4 * lane < rsc.parts ? pv[q][0] + pv[q][1] + pv[q][2] + pv[q][3] : 0.f);
      if (lane == 63) factor[wv + kRowsWaves * q] = 1.f / sqrtf(ss / rsc.width + rsc.eps);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if (nch > 1) {
    int c = 0;
    for (; c + 3 < nch; c += 2) {
      step(0, c, 2);
      step(1, c + 1, 2);
    }
    if (c + 2 < nch) {
      step(0, c, 2);
      step(1, c + 1, 1);
      step(0, c + 2, 0);
    } else {
      step(0, c, 1);
      step(1, c + 1, 0);
    }
  } else {
    step(0, 0, 0);
  }

  // acc[mt][f][v]: this wave's share of row 16 mt + 4 g + v, strip row 16 f + r; summed over the waves in their order
  float* red = reinterpret_cast<float*>(mine);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[(16 * mt + 4 * g + v) * 16 * NF + 16 * f + r] = acc[mt][f][v];
  __syncthreads();
  const float* all = reinterpret_cast<const float*>(sm);
  auto total = [&](int m, int n) {
    const float* p = all + m * 16 * NF + n;
    float t = p[0];
#pragma unroll
    for (int q = 1; q < kRowsWaves; ++q) t += p[q * WL / 2];
    if constexpr (SCALED) t *= factor[m];
    return t;
  };
  uint16_t* yb = reinterpret_cast<uint16_t*>(y);
  if constexpr (kHalves) {
    for (int e = threadIdx.x; e < HR * M; e += kRowsWaves * 64) {
      const int m = e / HR, n = e % HR;
      uint16_t a = f2bf(total(m, n)), b = f2bf(total(m, HR + n));
      const float fa = bf2f(a), fb = bf2f(b);
      if constexpr (OUT == kRowsSilu) {       // gate and up rounded as the separate pass reads them
        yb[(size_t)m * ldy + n0 + n] = f2bf(silu_gate(fa) * fb);
      } else {
        const int hd = (n0 + n) >> 6, d = (n0 + n) & 63;
        if (hd < rp.nq + rp.nkv) {
          const float* cs = rp.cos_sin + (size_t)rp.pos[m] * 128;
          float ra, rb;
          rope_pair(fa, fb, cs[d], cs[64 + d], ra, rb);
          a = f2bf(ra);
          b = f2bf(rb);
        }
        uint16_t* yr = yb + (size_t)m * ldy + hd * 128;
        yr[d] = a;
        yr[d + 64] = b;
        const int slot = rp.slots ? rp.slots[m] : -1;
        if (slot < 0 || hd < rp.nq) continue;
        const int blk = slot / rp.BS, off = slot % rp.BS;
        if (hd < rp.nq + rp.nkv) {
          uint16_t* kp = rp.kc + (((size_t)blk * rp.nkv + (hd - rp.nq)) * rp.BS + off) * 128;
          kp[d] = a;
          kp[d + 64] = b;
        } else {
          uint16_t* vp = rp.vc + ((size_t)blk * rp.nkv + (hd - rp.nq - rp.nkv)) * 128 * rp.BS + off;
          vp[(size_t)d * rp.BS] = a;
          vp[(size_t)(d + 64) * rp.BS] = b;
        }
      }
    }
  } else {
    for (int e = threadIdx.x; e < 16 * NF * M; e += kRowsWaves * 64) {
      const int m = e / (16 * NF), n = e % (16 * NF);
      const float t = total(m, n);
      if constexpr (OUT == kRowsConv) {
        if (n0 >= cv.cols) {
          cv.rest[(size_t)m * cv.ldr + n0 - cv.cols + n] = t;
          continue;
        }
        if (e != (int)threadIdx.x) conv_ask(cat = conv_row(e));
        const float own = bf2f(f2bf(t));
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < kConvTaps; ++j)
          if (j < cv.taps) sum = fmaf(taps[j], j < cv.taps - 1 ? hist[j] : own, sum);
        yb[(size_t)m * ldy + n0 + n] = f2bf(cv.act ? silu_f(sum) : sum);
#pragma unroll
        for (int j = 0; j < kConvTaps - 1; ++j)
          if (j < cv.taps - 1) cat.tl[(size_t)j * cv.cols] = j < cv.taps - 2 ? hist[j + 1] : own;
      } else if constexpr (OUT == kRowsF32)
        reinterpret_cast<float*>(y)[(size_t)blockIdx.y * M * N + (size_t)m * ldy + n0 + n] = t;
      else
        yb[(size_t)m * ldy + n0 + n] = f2bf(OUT == kRowsRelu2 ? relu_sq_f(t) : t);
    }
  }
}

template <int MT, int NF, int CH, int IN>
static int rows_launch(const void* x, int ldx, const void* w, void* y, int ldy, int M, int N, int K, int ranges, int out,
                       const RowsRope& rp, const NormIn& nin, const RowScale& rsc, const RowsConv& cv, hipStream_t s) {
  constexpr bool NORM = IN == kRowsNorm;
  const bool halves = out == kRowsSilu || out == kRowsRope;
  const int strip = (halves ? 8 : 16) * NF, cols = out == kRowsRope ? N / 2 : N;   // rope: columns counted as pairs
  if (M <= 0 || M > 16 * MT || (NORM && M > kNormMaxRows) || N <= 0 || N % (out == kRowsRope ? 128 : 1) || cols % strip ||
      ranges < 1 || K <= 0 || K % (ranges * kRowsWaves * CH) || (ranges > 1 && out != kRowsF32) ||
      ldy < (out == kRowsConv ? cv.cols : N) || (out == kRowsConv && (cv.cols % strip || cv.ldr < N - cv.cols)) || (ranges > 1 && ldy != N) || !w || !y || ((uintptr_t)w & 15))
    return (int)hipErrorInvalidValue;
  if (!NORM && (!x || ((uintptr_t)x & 15) || ldx % 8 || (M > 1 && ldx < K))) return (int)hipErrorInvalidValue;
  if (out == kRowsRope && rp.slots && (!rp.kc || !rp.vc)) return (int)hipErrorInvalidValue;
  const dim3 g(cols / strip, ranges), b(kRowsWaves * 64);
  const size_t lds = NORM ? (size_t)M * K * 2 : 0;
#define K8S_ROWS(OUT)                                                                                                   \
  hipLaunchKernelGGL((gemm_rows_kernel<MT, NF, CH, OUT, IN>), g, b, lds, s, (const uint16_t*)x, ldx, (const uint16_t*)w, y, \
                     ldy, M, N, K, K / ranges, rp, nin, rsc, cv)
  if constexpr (NORM) {
    switch (out) {
      case kRowsSilu: K8S_ROWS(kRowsSilu); break;
      case kRowsRope: K8S_ROWS(kRowsRope); break;
      default: return (int)hipErrorInvalidValue;
    }
  } else if constexpr (IN == kRowsScaled) {
    switch (out) {
      case kRowsBf16: K8S_ROWS(kRowsBf16); break;
      case kRowsF32: K8S_ROWS(kRowsF32); break;
      case kRowsSilu: K8S_ROWS(kRowsSilu); break;
      default: return (int)hipErrorInvalidValue;
    }
  } else {
    switch (out) {
      case kRowsBf16: K8S_ROWS(kRowsBf16); break;
      case kRowsF32: K8S_ROWS(kRowsF32); break;
      case kRowsSilu: K8S_ROWS(kRowsSilu); break;
      case kRowsRelu2: K8S_ROWS(kRowsRelu2); break;
      case kRowsRope: K8S_ROWS(kRowsRope); break;
      case kRowsConv:
        if constexpr (MT == 1) {
          K8S_ROWS(kRowsConv);
          break;
        }
      default: return (int)hipErrorInvalidValue;
    }
  }
#undef K8S_ROWS
  return (int)hipGetLastError();
}

template <int IN>
static int rows_any(const void* x, int ldx, const void* w, void* y, int ldy, int M, int N, int K, int nf, int ranges, int out,
                    const RowsRope& rp, const NormIn& nin, const RowScale& rsc, const RowsConv& cv, hipStream_t s) {
#define K8S_ROWS_AS(MT, NF, CH) \
  return rows_launch<MT, NF, CH, IN>(x, ldx, w, y, ldy, M, N, K, ranges, out, rp, nin, rsc, cv, s)
  if (M <= 16) {
    switch (nf) {
      case 1: K8S_ROWS_AS(1, 1, 128);
      case 2: K8S_ROWS_AS(1, 2, 128);
      case 4: K8S_ROWS_AS(1, 4, 64);
    }
  } else if constexpr (IN == kRowsPlain) {
    switch (nf) {
      case 2: K8S_ROWS_AS(2, 2, 64);
      case 4: K8S_ROWS_AS(2, 4, 64);
    }
  }
#undef K8S_ROWS_AS
  return (int)hipErrorInvalidValue;
}

}  // namespace k8s

using namespace k8s;

// nf: 16-row fragments of a workgroup, 1 (up to 16 rows), 2 or 4; ranges > 1: fp32 planes [ranges][M][N].
// out: 0 bf16, 1 fp32, 2 silu(x . w[0:N]^T) * (x . w[N:2N]^T), 3 max(., 0)^2.  K: whole chunks for each of four waves
// (128 entries, 64 where nf is 4 or there are more than 16 rows).  x (its rows too) and w lie on 16 bytes.
K8S_API int k8s_gemm_rows(const void* x, int ldx, const void* w, void* y, int ldy, int M, int N, int K, int nf, int ranges,
                          int out, hipStream_t s) {
  if (out < kRowsBf16 || out > kRowsRelu2) return (int)hipErrorInvalidValue;
  return rows_any<kRowsPlain>(x, ldx, w, y, ldy, M, N, K, nf, ranges, out, RowsRope{}, NormIn{}, RowScale{}, RowsConv{}, s);
}

// The same for up to 16 rows, row m divided by sqrt(sum(part[m]) / width + eps).  out: 0 bf16, 1 fp32, 2 SwiGLU.
K8S_API int k8s_gemm_rows_scaled(const void* x, int ldx, const void* w, void* y, int ldy, int M, int N, int K, int nf, int ranges,
                                 int out, const float* part, int parts, float width, float eps, hipStream_t s) {
  if (!part || ((uintptr_t)part & 15) || parts < 4 || parts % 4 || parts > kRowsParts || M > 16 || !(width > 0.f))
    return (int)hipErrorInvalidValue;
  return rows_any<kRowsScaled>(x, ldx, w, y, ldy, M, N, K, nf, ranges, out, RowsRope{}, NormIn{},
                               RowScale{part, parts, width, eps}, RowsConv{}, s);
}

// Up to 16 rows, each the only one of its sequence: y [M][cols] <- the first `cols` columns (a multiple of 16 nf) as
// k8s_gemm_rows and k8s_short_conv (no bias, 1 to 4 taps) leave them, tail too; rest [M][N - cols] <- the others in fp32.
K8S_API int k8s_gemm_rows_conv(const void* x, int ldx, const void* w, void* y, int cols, float* rest, int M, int N, int K, int nf,
                               const float* conv_w, int taps, float* tail, const int* pos0, const int* slot, int act,
                               hipStream_t s) {
  if (M > 16 || cols <= 0 || cols > N || (cols < N && !rest) || !conv_w || taps < 1 || taps > kConvTaps || (taps > 1 && !tail) ||
      !pos0 || !slot)
    return (int)hipErrorInvalidValue;
  return rows_any<kRowsPlain>(x, ldx, w, y, cols, M, N, K, nf, 1, kRowsConv, RowsRope{}, NormIn{}, RowScale{},
                              RowsConv{cols, taps, N - cols, act, conv_w, tail, pos0, slot, rest}, s);
}

// qkv = x . w^T (w = [q heads; k heads; v heads] x 128 rows) with q and k rotated and k, v written to their pages: what
// k8s_gemm_rows and k8s_rope_kv give, to the bit.
K8S_API int k8s_gemm_rows_rope(const void* x, int ldx, const void* w, void* qkv, int ldq, int M, int N, int K, int nf,
                               const int* pos, const float* cos_sin, const int* slots, void* kc, void* vc, int nq, int nkv,
                               int BS, hipStream_t s) {
  if (N != (nq + 2 * nkv) * 128 || !pos || !cos_sin || BS <= 0) return (int)hipErrorInvalidValue;
  const RowsRope rp{pos, cos_sin, slots, (uint16_t*)kc, (uint16_t*)vc, nq, nkv, BS};
  return rows_any<kRowsPlain>(x, ldx, w, qkv, ldq, M, N, K, nf, 1, kRowsRope, rp, NormIn{}, RowScale{}, RowsConv{}, s);
}

// The SwiGLU (pos null) or rotating form on X = rmsnorm(x [or the planes `part`] + res_in) * norm_w, made by every workgroup
// (norm_prologue.h; up to 4 rows): to the bit what the separate norm and the product give.  res_out (!= res_in) <- x + res_in.
K8S_API int k8s_gemm_rows_norm(const void* x, int x_stride, const float* part, int splits, const void* res_in, void* res_out,
                               const void* norm_w, float eps, const void* w, void* y, int ldy, int M, int N, int K, int nf,
                               const int* pos, const float* cos_sin, const int* slots, void* kc, void* vc, int nq, int nkv,
                               int BS, hipStream_t s) {
  auto off = [](const void* p) { return ((uintptr_t)p & 15) != 0; };
  if (M <= 0 || M > kNormMaxRows || K % 8 || K / 8 > 256 * kNormMaxChunks || !norm_w || (!x && !part) ||
      off(x) || off(part) || off(res_in) || off(res_out) || off(norm_w) || (!part && (x_stride % 8 || (M > 1 && x_stride < K))) ||
      (part && (splits < 1 || !res_in)) || (res_in && (!res_out || res_out == res_in)) ||
      (pos && (N != (nq + 2 * nkv) * 128 || !cos_sin || BS <= 0)))
    return (int)hipErrorInvalidValue;
  const NormIn nin{(const uint16_t*)x, part, (const uint16_t*)res_in, (uint16_t*)res_out, (const uint16_t*)norm_w,
                   x_stride, splits, K, eps};
  const RowsRope rp{pos, cos_sin, slots, (uint16_t*)kc, (uint16_t*)vc, nq, nkv, BS};
  return rows_any<kRowsNorm>(nullptr, 0, w, y, ldy, M, N, K, nf, 1, pos ? kRowsRope : kRowsSilu, rp, nin, RowScale{}, RowsConv{}, s);
}
