// Products of some tens to some thousands of fp32 rows, Y[M][N] = X[M][K] . W[N][K]^T, on the bf16 matrix instructions.
//
// The fp32 matrix instruction does a sixteenth of the bf16 one's work, and the library's fp32 products reach 120 to 140 TFLOP/s
// at 600 rows.  An fp32 number is the exact sum of three bf16 numbers (8 significant bits each, rounded to nearest: a1 =
// bf16(a), a2 = bf16(a - a1), a3 = a - a1 - a2), and of the nine products of two such sums six are kept: a1 b1, a1 b2, a2 b1,
// a2 b2, a1 b3, a3 b1.  What is left out is below 2^-26 of the product, a quarter of fp32's own rounding; sums stay in fp32.
// Relative error (2-norm, against 64 bits) of 622 rows of unit normals, the library / this:  K 2048 8.1e-7 / 7.0e-7 (in four
// ranges 3.4e-7);  K 8192 1.6e-6 / 1.4e-6 (7.2e-7).
//
// X is split once, by a pass of its own, into three planes of bf16 (every column tile reads it).  A workgroup of four waves makes
// 16 MT x 128 outputs, each wave 32 columns of all rows, K in steps of 32: X's planes go straight into LDS (16 rows x 64 bytes
// an instruction, as the fragments are read: no bank conflict), two buffers of them, a step ahead; no wave shares its columns, so
// that W is read in fragment order and split in registers: asked for between the halves of a step's matrix instructions,
// waited for in front of the next step's loads into LDS (so that no wait is for those: us without / so at 622 rows, ten
// fragments, 16384 x 2048 203 / 196, 8192 x 2048 136 / 116, 2048 x 8192 in four ranges 136 / 117), split between that step's
// halves.  Two to four workgroups share a compute unit.  The tiles of one panel of the larger operand follow each other on one XCD.
// Few tiles: K in ranges, whose sums (planes) the consumer adds.
//
// What bounds it: the power (1.8 GHz at a bf16 rate of 1.1 PFLOP/s) and, where there are few workgroups, a step's chain (1.2 us
// with four fragments, 1.65 with ten).  us, the library / the pass and this, out of memory:  16384 x 2048 at 333, 622, 1024 rows
// 210 / 150, 380 / 231, 515 / 341;  8192 x 2048 at 622, 1024 183 / 131, 257 / 182;  2048 x 8192 in eight ranges 176 / 124, 246 / 207
// and their sums.  In a first form, whose loads did not overlap: with X split by every workgroup 330 instead of 236, with
// W in LDS as well 361; the splits placed between the matrix instructions one by one 357.
#include "common.h"

namespace k8s {

constexpr int kSfN = 128, kSfK = 32;
constexpr float kSfWild = 3.39e38f;                               // rounds to an infinity in bf16, or a little less

enum SplitOut { kSplitPlain = 0, kSplitGlu = 1 };

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct Split3 {
  u32x2 p[3];            // four bf16 each
};

__device__ __forceinline__ uint32_t pair_bf(float a, float b) {                  // one instruction
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
}
__device__ __forceinline__ float low_bf(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float high_bf(uint32_t v) { return __uint_as_float(v & 0xffff0000u); }

// Four numbers as sums of three.  wild: some lane has a number that bf16 rounds to an infinity, or one that is: its first part is
// cut instead of rounded, and the others are zero where that is all of it (an infinity stays one, a NaN stays NaN).
__device__ __forceinline__ void split3(const f32x4& a, Split3& s, bool wild) {
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float u = a[2 * k], v = a[2 * k + 1];
    uint32_t h = pair_bf(u, v);
    if (wild) {
      if (fabsf(u) >= kSfWild) h = (h & 0xffff0000u) | (__float_as_uint(u) >> 16);
      if (fabsf(v) >= kSfWild) h = (h & 0xffffu) | (__float_as_uint(v) & 0xffff0000u);
    }
    s.p[0][k] = h;
    float ru = u - low_bf(h), rv = v - high_bf(h);
    if (wild) {
      if (u == low_bf(h)) ru = 0.f;
      if (v == high_bf(h)) rv = 0.f;
    }
    h = pair_bf(ru, rv);
    s.p[1][k] = h;
    s.p[2][k] = pair_bf(ru - low_bf(h), rv - high_bf(h));
  }
}

// A row (of X) or a row's K range (of W) whose largest number is below kSfLow, or kSfTiny, is multiplied by kSfUp, and its sums by
// the inverse: the third part of a number below 2^-110 would fall out of bf16's range.  The largest is below 2^-26 then, so that
// no sum overflows that did not.
constexpr float kSfLow = 0x1p-90f, kSfTiny = 0x1p-100f, kSfUp = 0x1p64f;

// x [M][K] (rows ldx apart) -> p [3][M][K], f [M]: what the row's sums are to be multiplied by (NaN: a number of the row is NaN).
// A workgroup a row.
__global__ void __launch_bounds__(256) split_rows_kernel(const float* __restrict__ x, int ldx, uint16_t* __restrict__ p,
                                                         float* __restrict__ f, int M, int K) {
  __shared__ float red[4];
  const int m = blockIdx.x, tid = threadIdx.x;
  const size_t plane = (size_t)M * K;
  x += (size_t)m * ldx;
  p += (size_t)m * K;
  float most = 0.f;
  bool nan = false;
  auto pass = [&](float up) {
#pragma unroll 2
    for (int c = 4 * tid; c < K; c += 1024) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(x + c) * up;
      Split3 s;
      split3(v, s, true);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        most = fmaxf(most, fabsf(v[k]));
        nan |= v[k] != v[k];
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x2*>(p + q * plane + c) = s.p[q];
    }
  };
  pass(1.f);
  most = wave_max(most);
  if ((tid & 63) == 0) red[tid >> 6] = most;
  nan = __syncthreads_or(nan);
  most = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const bool low = most > 0.f && most < kSfLow;
  if (low) pass(kSfUp);
  if (tid == 0) f[m] = nan ? __builtin_nanf("") : low ? 1.f / kSfUp : 1.f;
}

typedef __attribute__((address_space(3))) void sf_lds_t;
__device__ __forceinline__ void sf_to_lds(const uint16_t* src, uint16_t* dst) {  // 16 bytes a lane, the wave's 1 KB in a row
  __builtin_amdgcn_global_load_lds(src, (sf_lds_t*)dst, 16, 0, 0);
}

// One sum in fp32, by the whole wave (m, wrow alike in all lanes)
__device__ __forceinline__ float fp32_dot(const uint16_t* xpl, const float* w, int m, size_t wrow, int M, int K, int k0,
                                                    int n) {
  const uint16_t* a = xpl + (size_t)m * K + k0;
  const float* b = w + wrow * K + k0;
  const size_t plane = (size_t)M * K;
  float t = 0.f;
  for (int k = 4 * (threadIdx.x & 63); k < n; k += 256) {
    const u16x4 p0 = *reinterpret_cast<const u16x4*>(a + k), p1 = *reinterpret_cast<const u16x4*>(a + plane + k),
                p2 = *reinterpret_cast<const u16x4*>(a + 2 * plane + k);
    const f32x4 v = *reinterpret_cast<const f32x4*>(b + k);
#pragma unroll
    for (int j = 0; j < 4; ++j) t = fmaf(bf2f(p0[j]) + bf2f(p1[j]) + bf2f(p2[j]), v[j], t);
  }
  return wave_sum(t);
}

// grid: (row tiles x column tiles, K ranges).  The end of a step counts the loads behind its own into LDS, so their order is
// fixed: no pointer here is __restrict__, since loads through such a one may pass any clobber (tests/test_split_f32_waits.py
// reads the assembly).
template <int MT, int OUT>
__global__ void __launch_bounds__(256, MT <= 4 ? 4 : MT <= 8 ? 3 : 2)      // (what LDS lets onto a compute unit)
    gemm_split_f32_kernel(const uint16_t* xpl, const float* xfac, const float* w, float* y, int M, int N, int K, int n_mt, int n_nt) {
  constexpr int BM = 16 * MT, ND = 3 * MT, PER = (ND + 3) / 4;    // LDS-DMA instructions of a step, of a wave
  // (one variable: beside another one the compiler waits for the loads into LDS in front of every read of it)
  __shared__ struct {
    __attribute__((aligned(1024))) uint16_t xs[2][3][BM * kSfK];
    float fac[BM];                                                // of X's rows
    float up[kSfN];                                               // of the panel's rows of W, made for a second walk
    int low[4];
  } lds;
  auto& xs = lds.xs;
  auto& fac = lds.fac;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the tiles that share the larger operand's panel on one XCD, one after the other
  int tm, tn;
  {
    const bool by_w = 4 * (size_t)N * (OUT == kSplitGlu ? 2 : 1) >= 6 * (size_t)M;
    const int outer = by_w ? n_nt : n_mt, inner = by_w ? n_mt : n_nt;
    const int b = blockIdx.x, q = outer >> 3, whole = 8 * q * inner;
    const int o = b < whole ? (b & 7) + 8 * ((b >> 3) / inner) : 8 * q + (b - whole) / inner;
    const int i = b < whole ? (b >> 3) % inner : (b - whole) % inner;
    tn = by_w ? o : i, tm = by_w ? i : o;
  }
  const int m0 = tm * BM, n0 = tn * (OUT == kSplitGlu ? kSfN / 2 : kSfN);
  const int kr = K / gridDim.y, k0 = blockIdx.y * kr, steps = kr / kSfK;
  const uint16_t* xp[PER];                                        // instruction wv + 4 i: plane / MT, fragment % MT
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int d = min(wv + 4 * i, ND - 1);                        // (past the last one: it again)
    xp[i] = xpl + ((size_t)(d / MT) * M + min(m0 + 16 * (d % MT) + (lane >> 2), M - 1)) * K + k0 + 8 * (lane & 3);
  }
  const float* wp[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {                                   // SwiGLU: 16 gate rows and their up rows
    const size_t row = OUT == kSplitGlu ? min(n0 + 16 * wv + r, N - 1) + (size_t)j * N : min(n0 + 32 * wv + 16 * j + r, N - 1);
    wp[j] = w + row * K + k0 + 8 * g;
  }
  if (tid < BM) fac[tid] = xfac[min(m0 + tid, M - 1)];            // (up to 192 rows; there when the first step ends)
  f32x4 wq[2][2];
  bf16x8 wf[2][3];
  float top[2] = {0.f, 0.f};                                      // the largest numbers of this lane's rows of W
  auto load_x = [&](int s, int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int d = min(wv + 4 * i, ND - 1);
      sf_to_lds(xp[i] + s * kSfK, &xs[buf][0][d * 16 * kSfK]);
    }
  };
  auto load_w = [&](int s) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) wq[j][h] = *reinterpret_cast<const f32x4*>(wp[j] + s * kSfK + 4 * h);
  };
  auto wild = [&] {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) top[j] = fmaxf(top[j], fmaxf(fabsf(wq[j][0][k]), fabsf(wq[j][1][k])));
    return (bool)__any(fmaxf(top[0], top[1]) >= kSfWild);
  };
  bool again = false;
  auto take = [&](bf16x8 (&f)[2][3], bool wi) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      Split3 a, b;
      const float up = wi && again ? lds.up[32 * wv + 16 * j + r] : 1.f;
      split3(wi ? wq[j][0] * up : wq[j][0], a, wi);
      split3(wi ? wq[j][1] * up : wq[j][1], b, wi);
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        f[j][p] = __builtin_bit_cast(bf16x8, (u32x4{a.p[p][0], a.p[p][1], b.p[p][0], b.p[p][1]}));
      }
    }
  };
  auto take_any = [&](bf16x8 (&f)[2][3]) {
    if (__builtin_expect(wild() || again, 0))
      take(f, true);
    else
      take(f, false);
  };
  auto bar = [] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 acc[MT][2];
  auto fence = [] {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // two rows of fragments: 24 matrix instructions
  auto multiply = [&](int buf, int i) {
    bf16x8 xf[2][3];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        xf[h][p] = *reinterpret_cast<const bf16x8*>(&xs[buf][p][(16 * (i + h) + r) * kSfK + 8 * g]);
    constexpr int PX[6] = {2, 0, 1, 1, 0, 0}, PW[6] = {0, 2, 1, 0, 1, 0};        // small ones first
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i + h][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j][PW[q]], xf[h][PX[q]], acc[i + h][j], 0, 0, 0);
  };
  for (;;) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    load_w(0);
    load_x(0, 0);
    take_any(wf);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                // X of step 0
    bar();
    load_w(min(1, steps - 1));
    for (int s = 0; s < steps; ++s) {                               // (the last step loads and splits what it has once more, unread)
      const int buf = s & 1;
      constexpr int H = MT / 4 * 2;
      // W of the next step has come before the loads into LDS are asked for: with these on their way the compiler waits for all
      // loads where it needs one
      asm volatile("" : "+v"(wq[0][0]), "+v"(wq[0][1]), "+v"(wq[1][0]), "+v"(wq[1][1])::"memory");
      fence();
      load_x(min(s + 1, steps - 1), buf ^ 1);
      fence();
#pragma unroll
      for (int i = 0; i < H; i += 2) multiply(buf, i);
      bf16x8 nf[2][3];
      take_any(nf);
      fence();
      load_w(min(s + 2, steps - 1));                                // four loads: what the wait below leaves on its way
      fence();
#pragma unroll
      for (int i = H; i < MT; i += 2) multiply(buf, i);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int p = 0; p < 3; ++p) wf[j][p] = nf[j][p];
      fence();
      asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");   // the next step's X; this step's fragments are read
      bar();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // no load into LDS outlives the walk
    // W's rows of tiny numbers (lanes 0 to 15 of a wave have two each): once more, with factors
    bool any = false;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float t = fmaxf(top[j], __shfl_xor(top[j], 16, 64));
      t = fmaxf(t, __shfl_xor(t, 32, 64));
      const bool tiny = t > 0.f && t < kSfTiny;
      if (!again) lds.up[32 * wv + 16 * j + r] = tiny ? kSfUp : 1.f;
      any |= tiny;
    }
    any = __any(any);
    if (lane == 0) lds.low[wv] = any;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    bar();
    if (__builtin_expect(again || !(lds.low[0] | lds.low[1] | lds.low[2] | lds.low[3]), 1)) break;
    again = true;
  }
  if (__builtin_expect(again, 0)) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float down = 1.f / lds.up[32 * wv + 16 * j + 4 * g + v];
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i][j][v] *= down;
      }
  }
  // acc[i][j][v]: row m0 + 16 i + r, panel row 32 wv + 16 j + 4 g + v
  //
  // An infinity meets the other operand's parts of both signs, or none, and gives NaN where it should stay one: sums that are
  // NaN though no number of their rows is are made again in fp32.
  bool lost = false;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const float f = fac[16 * i + r];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) lost |= acc[i][j][v] != acc[i][j][v] && f == f;
  }
  if (__builtin_expect(__any(lost), 0)) {
    bool nan[2] = {false, false};                                 // of this lane's rows of W
#pragma unroll 1
    for (int s = 0; s < steps; ++s) {
      load_w(s);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) nan[j >> 1] |= wq[j >> 1][j & 1][k] != wq[j >> 1][j & 1][k];
    }
    float* const st = reinterpret_cast<float*>(&xs[0][0][0]) + wv * BM * 16;     // the wave's sums of 16 columns (X is done with)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint64_t bits = __ballot(nan[j]), bad = bits | bits >> 16 | bits >> 32 | bits >> 48;
#pragma unroll
      for (int i = 0; i < MT; ++i) *reinterpret_cast<f32x4*>(st + (16 * i + r) * 16 + 4 * g) = acc[i][j];
      fence();
#pragma unroll 1
      for (int e = lane; e < BM * 16; e += 64) {
        const float t = st[e], f = fac[e >> 4];
        for (uint64_t b = __ballot(t != t && f == f && !(bad >> (e & 15) & 1)); b; b &= b - 1) {
          const int q = __ffsll((unsigned long long)b) - 1, at = e - lane + q, c = at & 15;
          const size_t wr = OUT == kSplitGlu ? min(n0 + 16 * wv + c, N - 1) + (size_t)j * N : min(n0 + 32 * wv + 16 * j + c, N - 1);
          const float sum = fp32_dot(xpl, w, min(m0 + (at >> 4), M - 1), wr, M, K, k0, kr);
          if (lane == q) st[e] = sum;
        }
      }
      fence();
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i][j] = *reinterpret_cast<const f32x4*>(st + (16 * i + r) * 16 + 4 * g);
      fence();
    }
  }
  float* const o = y + (size_t)blockIdx.y * M * N;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + 16 * i + r;
    if (m >= M) continue;
    const float f = fac[16 * i + r];
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] *= f;
    if constexpr (OUT == kSplitGlu) {
      const int n = n0 + 16 * wv + 4 * g;
      if (n >= N) continue;
      f32x4 t;
#pragma unroll
      for (int v = 0; v < 4; ++v) t[v] = acc[i][0][v] / (1.f + expf(-acc[i][0][v])) * acc[i][1][v];
      *reinterpret_cast<f32x4*>(o + (size_t)m * N + n) = t;
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n0 + 32 * wv + 16 * j + 4 * g;
        if (n < N) *reinterpret_cast<f32x4*>(o + (size_t)m * N + n) = acc[i][j];
      }
    }
  }
}

template <int OUT>
static int split_f32(const uint16_t* xp, const float* f, const float* w, float* y, int M, int N, int K, int mt, int ranges, hipStream_t s) {
  if (M <= 0 || N <= 0 || N % 4 || K <= 0 || ranges < 1 || K % (kSfK * ranges) || !xp || !f || !w || !y || ((uintptr_t)xp & 15) ||
      ((uintptr_t)w & 15) || ((uintptr_t)y & 15) || (OUT == kSplitGlu && (ranges > 1 || N % 64)))
    return (int)hipErrorInvalidValue;
  const int bn = OUT == kSplitGlu ? kSfN / 2 : kSfN, n_nt = (N + bn - 1) / bn, n_mt = (M + 16 * mt - 1) / (16 * mt);
#define K8S_SF(MT)                                                                                                        \
  case MT:                                                                                                                \
    hipLaunchKernelGGL((gemm_split_f32_kernel<MT, OUT>), dim3(n_mt * n_nt, ranges), dim3(256), 0, s, xp, f, w, y, M, N, K,   \
                       n_mt, n_nt);                                                                                             \
    break
  switch (mt) {
    K8S_SF(4);
    K8S_SF(6);
    K8S_SF(8);
    K8S_SF(10);
    K8S_SF(12);
    default: return (int)hipErrorInvalidValue;
  }
#undef K8S_SF
  return (int)hipGetLastError();
}

}  // namespace k8s

using namespace k8s;

// x [M][K] fp32 (rows ldx apart, on 16 bytes) -> three bf16 planes p [3][M][K] and f [M]: a row is f times the planes' sum (NaN
// where a number of it is).
K8S_API int k8s_split_rows_f32(const float* x, int ldx, void* p, float* f, int M, int K, hipStream_t s) {
  if (M <= 0 || K <= 0 || K % 4 || ldx % 4 || (M > 1 && ldx < K) || !x || !p || !f || ((uintptr_t)x & 15) || ((uintptr_t)p & 7))
    return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(split_rows_kernel, dim3(M), dim3(256), 0, s, x, ldx, (uint16_t*)p, f, M, K);
  return (int)hipGetLastError();
}

// y [ranges][M][N] fp32: the products of xp's rows (three planes and their factors) and w [N][K] over K ranges.  mt: 16-row
// fragments of a tile, 4, 6, 8, 10 or 12.  N a multiple of 4, K of 32 ranges; xp, w, y on 16 bytes.
K8S_API int k8s_gemm_split_f32(const void* xp, const float* f, const float* w, float* y, int M, int N, int K, int mt, int ranges,
                               hipStream_t s) {
  return split_f32<kSplitPlain>((const uint16_t*)xp, f, w, y, M, N, K, mt, ranges, s);
}

// y [M][N] = silu(x . w[0:N]^T) * (x . w[N:2N]^T), N a multiple of 64.
K8S_API int k8s_gemm_split_glu_f32(const void* xp, const float* f, const float* w, float* y, int M, int N, int K, int mt,
                                   hipStream_t s) {
  return split_f32<kSplitGlu>((const uint16_t*)xp, f, w, y, M, N, K, mt, 1, s);
}
