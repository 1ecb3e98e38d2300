// Single tokens of a latent attention layer, from the joint down projection to the heads' queries, in one launch: the rows'
// planes added, the query latent divided by its root mean square and multiplied by W_uq, the key-value latent normed and
// written to its pages with the rotated key part behind it (latent_norm, seq_ops.hip, and a product).
//
// What bounds the two launches is that they are two: 3.8 to 5.1 us with one workgroup a row, then 3.4 to 5 us for 4.7 MB of
// weights.  Here every strip of 16 columns of W_uq norms all rows itself, a wave a row (or two), with its weights on their
// way; the rows come from L2, 6 KB each (two planes of 768), and the pages are written by M workgroups beside the strips.
// us of both launches / of this, 768 + 256 + 64 numbers of two planes, 3072 x 768, in a replayed chain with cold weights, at
// 1, 7, 16 rows 7.5 / 3.6, 7.9 / 4.1, 8.1 / 4.8 (where the line lies: latent_up, seq_ops.py).
#include "common.h"

namespace k8s {

constexpr int kLsWaves = 8, kLsRows = 16, kLsTail = 2048;

struct LatentStep {
  const float* dn;        // [planes][M][ld], pstep apart: query latent [QR] | latent [KR] | rotated part [RD]
  size_t pstep;
  const uint16_t* wq;     // [QR]
  const uint16_t* wkv;    // [KR]
  const uint16_t* w;      // [N][QR]
  uint16_t* q;            // [M][N]
  const int* slots;
  uint16_t* cache;        // rows of KR + RP
  uint16_t* cache_t;      // [pages][KR][BS] or null
  const float* cs;        // [M][RD]: cos | sin
  int ld, planes, BS, KR, RD, RP, strips;
  float eps;
};

// A row's latent to its pages: what latent_norm_kernel writes, in its order
__device__ __forceinline__ void latent_to_pages(const LatentStep& a, int t, int QR, float* row, float* scratch) {
  constexpr int NT = 64 * kLsWaves;
  const float* mrow = a.dn + (size_t)t * a.ld + QR;
  const int slot = a.slots[t], all = a.KR + a.RD;
  for (int c = 4 * threadIdx.x; c < all; c += 4 * NT)
    *reinterpret_cast<f32x4*>(row + c) = sum_planes4(mrow + c, a.pstep, a.planes);
  __syncthreads();
  float ss = 0.f;
  for (int c = threadIdx.x; c < a.KR; c += NT) ss = fmaf(row[c], row[c], ss);
  ss = block_sum(ss, scratch);
  const float inv = 1.f / sqrtf(ss / (float)a.KR + a.eps);
  if (slot < 0) return;
  const size_t page = slot / a.BS, off = slot - page * a.BS;
  uint16_t* out = a.cache + (size_t)slot * (a.KR + a.RP);
  for (int c = threadIdx.x; c < a.KR; c += NT) {
    const uint16_t v = f2bf(row[c] * inv * bf2f(a.wkv[c]));
    out[c] = v;
    if (a.cache_t) a.cache_t[(page * a.KR + c) * a.BS + off] = v;
  }
  const int half = a.RD >> 1;
  for (int i = threadIdx.x; i < a.RP; i += NT) {
    float v = 0.f;
    if (i < a.RD) {
      const float* p = row + a.KR + (i & ~1);
      const float co = a.cs[(size_t)t * a.RD + (i >> 1)], si = a.cs[(size_t)t * a.RD + half + (i >> 1)];
      v = (i & 1) ? p[1] * co + p[0] * si : p[0] * co - p[1] * si;
    }
    out[a.KR + i] = f2bf(v);
  }
}

// QR = 256 NB; PL planes.  grid: strips of 16 columns, then the rows.
template <int NB, int PL>
__global__ void __launch_bounds__(64 * kLsWaves) latent_step_kernel(LatentStep a, int M, int N) {
  constexpr int QR = 256 * NB, LD = QR + 8;
  __shared__ __attribute__((aligned(16))) uint16_t xs[kLsRows * LD];
  __shared__ float red[kLsWaves][16][16];
  if ((int)blockIdx.x >= a.strips) {
    __shared__ __attribute__((aligned(16))) float row[kLsTail];
    latent_to_pages(a, blockIdx.x - a.strips, QR, row, &red[0][0][0]);
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r = lane & 15, g = lane >> 4, n0 = blockIdx.x * 16;
  constexpr int RW = kLsRows / kLsWaves;
  f32x4 raw[RW][NB][PL];
  u16x4 wn[NB];
#pragma unroll
  for (int i = 0; i < RW; ++i)
    if (wv + kLsWaves * i < M) {
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int p = 0; p < PL; ++p)
          raw[i][j][p] = *reinterpret_cast<const f32x4*>(a.dn + p * a.pstep + (size_t)(wv + kLsWaves * i) * a.ld + 256 * j + 4 * lane);
    }
#pragma unroll
  for (int j = 0; j < NB; ++j) wn[j] = *reinterpret_cast<const u16x4*>(a.wq + 256 * j + 4 * lane);
  __builtin_amdgcn_sched_barrier(0);
  const uint16_t* wp = a.w + (size_t)(n0 + r) * QR + wv * 32 * NB + 8 * g;
  bf16x8 wf[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) wf[j] = ldw_nt<bf16x8>(wp + 32 * j);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int m = wv + kLsWaves * i;
    if (m >= M) break;
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
#pragma unroll
      for (int p = 1; p < PL; ++p) raw[i][j][0] += raw[i][j][p];
#pragma unroll
      for (int k = 0; k < 4; ++k) ss = fmaf(raw[i][j][0][k], raw[i][j][0][k], ss);
    }
    const float inv = 1.f / sqrtf(wave_sum(ss) / (float)QR + a.eps);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      u16x4 o;
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] = f2bf(raw[i][j][0][k] * inv * bf2f(wn[j][k]));
      *reinterpret_cast<u16x4*>(xs + m * LD + 256 * j + 4 * lane) = o;
    }
  }
  __syncthreads();
  const uint16_t* xp = xs + min(r, M - 1) * LD + wv * 32 * NB + 8 * g;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < NB; ++j)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(xp + 32 * j), wf[j], acc, 0, 0, 0);
#pragma unroll
  for (int v = 0; v < 4; ++v) red[wv][4 * g + v][r] = acc[v];          // row 4 g + v, column r
  __syncthreads();
  const int m = tid >> 4, n = tid & 15;
  if (m >= M) return;
  float t = red[0][m][n];
#pragma unroll
  for (int k = 1; k < kLsWaves; ++k) t += red[k][m][n];
  a.q[(size_t)m * N + n0 + n] = f2bf(t);
}

}  // namespace k8s

using namespace k8s;

// Up to 16 rows; QR 256, 512, 768, 1024, 1536 or 2048, planes 1, 2 or 4, of QR x planes at most 4096; N % 16 == 0, KR + RD <= 2048.
// dn, w on 16 bytes, wq on 8; ld, pstep and KR + RD multiples of 4.
K8S_API int k8s_latent_step(const float* dn, int ld, int planes, long pstep, const void* wq, const void* wkv, const void* w,
                            void* q, const int* slots, void* cache, void* cache_t, int BS, int M, int N, int QR, int KR,
                            float eps, int RD, int RP, const float* cs, hipStream_t s) {
  if (M <= 0) return 0;
  if (M > kLsRows || N <= 0 || N % 16 || KR <= 0 || RD < 0 || (RD & 1) || RP < RD || (RP & 1) || (RD && !cs) || (KR + RD) % 4 ||
      KR + RD > kLsTail || BS < 1 || ld % 4 || ld < QR + KR + RD || (planes > 1 && pstep % 4) || !dn || !wq || !wkv || !w || !q ||
      !slots || !cache || (((uintptr_t)dn | (uintptr_t)w) & 15) || ((uintptr_t)wq & 7))
    return (int)hipErrorInvalidValue;
  const LatentStep a{dn, (size_t)pstep, (const uint16_t*)wq, (const uint16_t*)wkv, (const uint16_t*)w, (uint16_t*)q, slots,
                     (uint16_t*)cache, (uint16_t*)cache_t, cs, ld, planes, BS, KR, RD, RP, N / 16, eps};
#define K8S_LS(NB, PL)                                                                                                \
  if (QR == 256 * NB && planes == PL) {                                                                               \
    hipLaunchKernelGGL((latent_step_kernel<NB, PL>), dim3(N / 16 + M), dim3(64 * kLsWaves), 0, s, a, M, N);           \
    return (int)hipGetLastError();                                                                                    \
  }
#define K8S_LSP(NB) K8S_LS(NB, 1) K8S_LS(NB, 2) K8S_LS(NB, 4)
  K8S_LSP(1)
  K8S_LSP(2)
  K8S_LSP(3)
  K8S_LSP(4)
  K8S_LS(6, 1)
  K8S_LS(6, 2)
  K8S_LS(8, 1)
  K8S_LS(8, 2)
#undef K8S_LSP
#undef K8S_LS
  return (int)hipErrorInvalidValue;
}
