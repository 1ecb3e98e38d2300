// Small products of a few rows (reply steps), on the vector pipes: a matrix of a quarter megabyte a head or less, whose
// time is the launch and one trip to memory.
//
// head_proj:  out[t][h][n] = sum_k a[t][h][k] w[h][k][n], bf16 or fp32 with fp32 sums (a latent layer's query into latent space,
//   its output out of it), and, in the same launch, the rotated key part's queries: the RD entries behind a[t][h][0 .. K)
//   turned in neighbouring pairs by cs [t][RD] (cos | sin), filled up with zeros to RP.
// low_rank_pair:  out_i[t][n] = sum_k bf16(x[t][c_i + k]) w_i[n][k] for two column ranges of the same fp32 rows.
//
// A workgroup has 64 columns and TR rows, its threads split K: every weight load of a thread is on its way before the
// first sum, a weight is unpacked once for TR rows, the rows are broadcast from LDS, the K ranges are added in order.
#include "common.h"

namespace k8s {

template <typename TX>
struct HeadProjArgs {
  const TX* a;            // element (t, h, k) at t * ast + h * ash + k
  long ast, ash;
  const TX* w;            // [H][K][N]
  TX* out;                // element (t, h, n) at t * ost + h * osh + n
  long ost, osh;
  int T, H, K, N;
  const float* cs;
  TX* qr;                 // [T][H][RP] or null
  int RD, RP;
};

__device__ __forceinline__ float ldx(const uint16_t* p) { return bf2f(*p); }
__device__ __forceinline__ float ldx(const float* p) { return *p; }
__device__ __forceinline__ void stx(uint16_t* p, float v) { *p = f2bf(v); }
__device__ __forceinline__ void stx(float* p, float v) { *p = v; }
// two neighbouring weights as they lie in memory
template <typename TX>
struct Pair;
template <>
struct Pair<uint16_t> {
  uint32_t v;
  __device__ __forceinline__ float lo() const { return bf2f((uint16_t)v); }
  __device__ __forceinline__ float hi() const { return bf2f((uint16_t)(v >> 16)); }
};
template <>
struct alignas(8) Pair<float> {
  float a, b;
  __device__ __forceinline__ float lo() const { return a; }
  __device__ __forceinline__ float hi() const { return b; }
};

// U: weight rows in flight per thread
template <int TR, int U, typename TX>
__global__ void __launch_bounds__(256) head_proj_kernel(HeadProjArgs<TX> a) {
  extern __shared__ float smem[];                          // [K][TR], then [8][TR][64]
  const int tid = threadIdx.x, c = 2 * (tid & 31), kg = tid >> 5, n0 = blockIdx.x * 64, h = blockIdx.y;
  const int t0 = blockIdx.z * TR, nt = min(TR, a.T - t0), KG = a.K / 8;
  const TX* wp = a.w + ((size_t)h * a.K + (size_t)kg * KG) * a.N + n0 + c;
  Pair<TX> wv[U];
#pragma unroll
  for (int u = 0; u < U; ++u) wv[u] = *reinterpret_cast<const Pair<TX>*>(wp + (size_t)min(u, KG - 1) * a.N);
  for (int e = tid; e < a.K * TR; e += 256) {
    const int k = e % a.K, t = e / a.K;
    smem[k * TR + t] = t < nt ? ldx(a.a + (size_t)(t0 + t) * a.ast + (size_t)h * a.ash + k) : 0.f;
  }
  if (a.qr && blockIdx.x == 0) {
    const int hp = a.RP >> 1, half = a.RD >> 1;
    for (int e = tid; e < nt * hp; e += 256) {
      const int t = t0 + e / hp, i = e % hp;
      float x = 0.f, y = 0.f;
      if (i < half) {
        const TX* p = a.a + (size_t)t * a.ast + (size_t)h * a.ash + a.K + 2 * i;
        const float u = ldx(p), v = ldx(p + 1), co = a.cs[(size_t)t * a.RD + i], si = a.cs[(size_t)t * a.RD + half + i];
        x = u * co - v * si;
        y = v * co + u * si;
      }
      TX* q = a.qr + ((size_t)t * a.H + h) * a.RP + 2 * i;
      stx(q, x);
      stx(q + 1, y);
    }
  }
  __syncthreads();
  float acc[TR][2] = {};
  for (int k0 = 0; k0 < KG; k0 += U) {
    if (k0 > 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) wv[u] = *reinterpret_cast<const Pair<TX>*>(wp + (size_t)min(k0 + u, KG - 1) * a.N);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k0 + u < KG) {
        const float w0 = wv[u].lo(), w1 = wv[u].hi();
        const float* xs = smem + (kg * KG + k0 + u) * TR;
#pragma unroll
        for (int t = 0; t < TR; ++t) {
          acc[t][0] = fmaf(xs[t], w0, acc[t][0]);
          acc[t][1] = fmaf(xs[t], w1, acc[t][1]);
        }
      }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < TR; ++t) {
    smem[(kg * TR + t) * 64 + c] = acc[t][0];
    smem[(kg * TR + t) * 64 + c + 1] = acc[t][1];
  }
  __syncthreads();
  for (int e = tid; e < nt * 64; e += 256) {
    float v = 0.f;
#pragma unroll
    for (int g = 0; g < 8; ++g) v += smem[g * TR * 64 + e];
    stx(a.out + (size_t)(t0 + e / 64) * a.ost + (size_t)h * a.osh + n0 + e % 64, v);
  }
}

struct LowRankArgs {
  const float* x;
  int xs, T;
  int col[2], K[2], N[2];
  const uint16_t* w[2];   // [N][K]
  float* out[2];          // [T][N]
};

template <int TR>
__global__ void __launch_bounds__(256) low_rank_pair_kernel(LowRankArgs a) {
  extern __shared__ float smem[];                          // [K][TR], then [4][TR][64]
  const int s0 = (a.N[0] + 63) / 64, i = (int)blockIdx.x >= s0, n0 = 64 * (blockIdx.x - (i ? s0 : 0));
  const int K = a.K[i], N = a.N[i], KG = K / 4, tid = threadIdx.x, c = tid & 63, kg = tid >> 6;
  const int t0 = blockIdx.y * TR, nt = min(TR, a.T - t0);
  const uint16_t* wp = a.w[i] + (size_t)min(n0 + c, N - 1) * K + kg * KG;
  u16x8 wv = *reinterpret_cast<const u16x8*>(wp);
  for (int e = tid; e < K * TR; e += 256) {
    const int k = e % K, t = e / K;
    smem[k * TR + t] = t < nt ? bf2f(f2bf(a.x[(size_t)(t0 + t) * a.xs + a.col[i] + k])) : 0.f;
  }
  __syncthreads();
  float acc[TR] = {};
  for (int k0 = 0; k0 < KG; k0 += 8) {
    const u16x8 w = wv;
    if (k0 + 8 < KG) wv = *reinterpret_cast<const u16x8*>(wp + k0 + 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float* xs = smem + (kg * KG + k0 + j) * TR;
#pragma unroll
      for (int t = 0; t < TR; ++t) acc[t] = fmaf(xs[t], bf2f(w[j]), acc[t]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < TR; ++t) smem[(kg * TR + t) * 64 + c] = acc[t];
  __syncthreads();
  for (int e = tid; e < nt * 64; e += 256) {
    float v = 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) v += smem[g * TR * 64 + e];
    if (n0 + e % 64 < N) a.out[i][(size_t)(t0 + e / 64) * N + n0 + e % 64] = v;
  }
}

}  // namespace k8s

using namespace k8s;

// rows per workgroup: one, four or eight (of head_proj with more than 128 entries a head: one or four)
#define K8S_TR(T, ...)            \
  if ((T) == 1) {                 \
    constexpr int TR = 1;         \
    __VA_ARGS__;                  \
  } else if ((T) <= 4) {          \
    constexpr int TR = 4;         \
    __VA_ARGS__;                  \
  } else {                        \
    constexpr int TR = 8;         \
    __VA_ARGS__;                  \
  }

template <typename TX>
static int head_proj_launch(const void* x, long ast, long ash, const void* w, void* out, long ost, long osh, int T, int H,
                            int K, int N, const float* cs, void* qr, int RD, int RP, hipStream_t s) {
  HeadProjArgs<TX> a{(const TX*)x, ast, ash, (const TX*)w, (TX*)out, ost, osh, T, H, K, N, cs, (TX*)qr, RD, RP};
  K8S_TR(K > 128 && T > 4 ? 4 : T, {
    const size_t lds = sizeof(float) * TR * (K > 512 ? K : 512);
    const dim3 grid(N / 64, H, (T + TR - 1) / TR);
    if (K <= 128)
      hipLaunchKernelGGL((head_proj_kernel<TR, 16, TX>), grid, dim3(256), lds, s, a);
    else
      hipLaunchKernelGGL((head_proj_kernel<TR, 32, TX>), grid, dim3(256), lds, s, a);
  });
  return (int)hipGetLastError();
}

// K % 8 == 0 up to 1024, N % 64 == 0; qr null: no rotated part.  dt: 0 bf16, 1 fp32.
K8S_API int k8s_head_proj(const void* x, long ast, long ash, const void* w, void* out, long ost, long osh, int T, int H,
                          int K, int N, const float* cs, void* qr, int RD, int RP, int dt, hipStream_t s) {
  if (T <= 0) return 0;
  if (H < 1 || K < 8 || K % 8 || K > 1024 || N < 64 || N % 64 || dt < 0 || dt > 1 || (uintptr_t)w % (dt ? 8 : 4) ||
      (qr && (RD < 0 || RD % 2 || RP % 2 || RP < RD || (RD && !cs))))
    return (int)hipErrorInvalidValue;
  return (dt ? head_proj_launch<float> : head_proj_launch<uint16_t>)(x, ast, ash, w, out, ost, osh, T, H, K, N, cs, qr, RD,
                                                                     RP, s);
}

// K0, K1 % 32 == 0 up to 1024; weights 16-byte aligned.
K8S_API int k8s_low_rank_pair(const float* x, int xs, int T, int col0, int K0, const void* w0, int N0, float* out0, int col1,
                              int K1, const void* w1, int N1, float* out1, hipStream_t s) {
  if (T <= 0) return 0;
  if (K0 < 32 || K1 < 32 || K0 % 32 || K1 % 32 || K0 > 1024 || K1 > 1024 || N0 < 1 || N1 < 1 || (uintptr_t)w0 % 16 ||
      (uintptr_t)w1 % 16)
    return (int)hipErrorInvalidValue;
  LowRankArgs a{x, xs, T, {col0, col1}, {K0, K1}, {N0, N1}, {(const uint16_t*)w0, (const uint16_t*)w1}, {out0, out1}};
  const int K = K0 > K1 ? K0 : K1;
  K8S_TR(T, {
    const size_t lds = sizeof(float) * TR * (K > 256 ? K : 256);
    hipLaunchKernelGGL((low_rank_pair_kernel<TR>), dim3((N0 + 63) / 64 + (N1 + 63) / 64, (T + TR - 1) / TR), dim3(256), lds, s,
                       a);
  });
  return (int)hipGetLastError();
}
