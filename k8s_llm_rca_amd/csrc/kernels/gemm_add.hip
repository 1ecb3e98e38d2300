// A prompt's products into the fp32 residual, together with what reads it next (gemm_step.hip is the same for up to 16 rows):
//   x += sy s(m) (A . W^T) [+ es emb[id]]          (x [M][N] fp32, in place)
//   then nothing;   or h = tanh(alpha x) nw + nb in bf16;   or h = x nw in bf16 and the row's sum of squares in parts of 256
//   columns, which SwiGLU's product behind divides its sums by (k8s_gemm_big_silu_scaled).
// s(m) divides the operand's rows by the root mean square of what they were made from (rs: its sums of squares).
//
// The pass between two products reads the residual and the product (with fewer than some 6000 rows, where the product was no
// whole wave of 256-row tiles and did not add itself) and writes residual and activations: 19 to 25 us at 4096 rows of 2048,
// 41 at 16384, all of it the memory's.  Here the residual is read and written once and the activations leave with it.
//
// The tiles: row_tiles.h.
//
// What bounds it: with 256-row tiles the power limit (1.4 PFLOP/s); with 128 and 160 rows the fragments' way out of LDS, a
// phase's 12 to 14 reads a wave in front of 16 to 20 matrix instructions (1.15 - 1.2 PFLOP/s, what the library's tiles of that size
// do).  us of product and pass / of this with tanh, 2048 x 2048 and 2048 x 8192 at 2600, 4096, 4850, 6144, 10000, 16384 rows:
//   45 / 42, 60 / 48, 70 / 55, 71 / 64, 112 / 105, 170 / 159;   107 / 99, 136 / 120, 160 / 138, 174 / 169, 344 / 284, 424 / 419;
// with the norm left to the product behind 44 / 39, 57 / 44, 69 / 51, 71 / 58, 112 / 98, 169 / 146;   101 / 94, 134 / 117, 159 / 136, 168 / 163,
// 341 / 274, 429 / 405.  tanh is 5 to 11 us of it a wave of tiles: vector instructions while the matrix units wait.
// The residual asked for in front of the last tile's products, with that tile's code of its own, changed nothing (registers).
#include "row_tiles.h"

namespace k8s {
namespace padd {

enum Then { kNothing = 0, kDyt = 1, kScaled = 2 };

struct AddArgs {
  const uint16_t* a;     // [M][lda]
  const uint16_t* w;     // [N][K]
  float* x;              // [M][N], in place
  const float* nw;       // [N]
  const float* nb;       // [N]
  uint16_t* h;           // [M][N]
  float* part;           // [M][N / 256]
  const float* rs;       // [M][rn] or null: the product's rows are divided by sqrt(sum / rw + reps)
  const int* eid;        // [M]: rows of emb, times es, are added too; or null
  const uint16_t* emb;   // [.][N]
  float sy, alpha, rw, reps, es;
  int lda, rn, M, N, K, n_mt, n_nt;
};

// What follows the residual's entries t (four columns from c0, at o of the row): the activations; kScaled: the sum of squares of
// the wave's columns, in its last lane.
template <int THEN>
__device__ __forceinline__ float then_row(const AddArgs& p, size_t o, const f32x4& nw, const f32x4& nb, const f32x4& t) {
  u16x4 h;
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if constexpr (THEN == kDyt) {
      h[c] = f2bf(fmaf(tanhf(p.alpha * t[c]), nw[c], nb[c]));
    } else {
      s = fmaf(t[c], t[c], s);
      h[c] = f2bf(t[c] * nw[c]);
    }
  }
  *reinterpret_cast<u16x4*>(p.h + o) = h;
  return THEN == kScaled ? wave_sum_dpp(s) : 0.f;
}
template <int THEN>
__device__ __forceinline__ void then_ask(const AddArgs& p, int c0, f32x4& nw, f32x4& nb) {
  nw = nb = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (THEN != kNothing) nw = *reinterpret_cast<const f32x4*>(p.nw + c0);
  if constexpr (THEN == kDyt) nb = *reinterpret_cast<const f32x4*>(p.nb + c0);
}

// F: 16-row fragments of a wave.  EXTRA: rs and eid may be set.
template <int F, int THEN, bool EXTRA>
__global__ void __launch_bounds__(512, 1) gemm_add_kernel(AddArgs p) {
  using Tile = RowTile<F>;
  constexpr int HM = Tile::HM;
  __shared__ __attribute__((aligned(1024))) unsigned char sm[Tile::LDS];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wv >> 2;
  int tm, tn;
  tile_of(p.n_mt, p.n_nt, tm, tn);
  const int M = p.M, N = p.N, m0 = tm * Tile::BM;
  f32x4 acc[2][F][2];
  Tile::product(p.a, p.lda, p.w, M, p.K, m0, sm, acc, [&](int h, int R) { return tn * BN + eight_columns(h, R); });

  // ---- epilogue
  constexpr int RW = HM / 8;                                // rows of a half that a wave takes
  const int c0 = tn * BN + 4 * lane;
  f32x4 t[RW], nw, nb;
  float rv[EXTRA ? RW : 1];
  then_ask<THEN>(p, c0, nw, nb);
  auto row = [&](int half, int i) { return m0 + HM * half + 8 * i + wv; };
  auto ask = [&](int half) {
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const size_t m = min(row(half, i), M - 1);
      t[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.x + m * N + c0));
      if constexpr (EXTRA) rv[i] = p.rs && lane < p.rn ? p.rs[m * p.rn + lane] : 0.f;
    }
  };
  auto put = [&](int half) {
    if (wr == half) Tile::put(sm, acc);
  };
  auto finish = [&](int half) {
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int r = 8 * i + wv, m = row(half, i);
      f32x4 v = Tile::get(sm, r);
      if (m >= M) continue;
      if (EXTRA && p.rs) v *= 1.f / sqrtf(last_lane(wave_sum_dpp(rv[i])) / p.rw + p.reps);
#pragma unroll
      for (int c = 0; c < 4; ++c) t[i][c] = fmaf(p.sy, v[c], t[i][c]);
      if (EXTRA && p.eid) {
        const u16x4 e = *reinterpret_cast<const u16x4*>(p.emb + (size_t)p.eid[m] * N + c0);
#pragma unroll
        for (int c = 0; c < 4; ++c) t[i][c] = fmaf(p.es, bf2f(e[c]), t[i][c]);
      }
      *reinterpret_cast<f32x4*>(p.x + (size_t)m * N + c0) = t[i];
      if constexpr (THEN != kNothing) {
        const float ss = then_row<THEN>(p, (size_t)m * N + c0, nw, nb, t[i]);
        if (THEN == kScaled && lane == 63) p.part[(size_t)m * p.n_nt + tn] = ss;
      }
    }
  };
  ask(0);
  lds_bar();                                                // (the last fragments are read, no DMA is in flight)
  put(0);
  lds_bar();
  finish(0);
  ask(1);
  lds_bar();
  put(1);
  lds_bar();
  finish(1);
}

template <int F, int THEN, bool EXTRA>
static int launch(AddArgs p, hipStream_t s) {
  p.n_mt = (p.M + 32 * F - 1) / (32 * F);
  p.n_nt = p.N / BN;
  hipLaunchKernelGGL((gemm_add_kernel<F, THEN, EXTRA>), dim3(p.n_mt * p.n_nt), dim3(512), 0, s, p);
  return (int)hipGetLastError();
}
template <int F>
static int launch_then(const AddArgs& p, int then, hipStream_t s) {
  const bool extra = p.rs || p.eid;
  switch (then) {
    case kNothing: return extra ? launch<F, kNothing, true>(p, s) : launch<F, kNothing, false>(p, s);
    case kDyt: return extra ? (int)hipErrorInvalidValue : launch<F, kDyt, false>(p, s);
    case kScaled: return extra ? launch<F, kScaled, true>(p, s) : launch<F, kScaled, false>(p, s);
  }
  return (int)hipErrorInvalidValue;
}

// The same behind a product that left planes y [planes][M][N]: the few rows past whole waves of tiles.
template <int THEN>
__global__ void __launch_bounds__(256) add_rows_kernel(AddArgs p, const float* __restrict__ y, int planes) {
  const int lane = threadIdx.x & 63, m = blockIdx.x, N = p.N;
  float f = 1.f;
  if (p.rs) {
    const float s = wave_sum(lane < p.rn ? p.rs[(size_t)m * p.rn + lane] : 0.f);
    f = 1.f / sqrtf(s / p.rw + p.reps);
  }
  for (int j = threadIdx.x >> 6; j < p.n_nt; j += 4) {
    const int c0 = j * BN + 4 * lane;
    const size_t o = (size_t)m * N + c0;
    const f32x4 v = sum_planes4(y + o, (size_t)p.M * N, planes);
    f32x4 t = *reinterpret_cast<const f32x4*>(p.x + o);
#pragma unroll
    for (int c = 0; c < 4; ++c) t[c] = fmaf(p.sy, v[c] * f, t[c]);
    if (p.eid) {
      const u16x4 e = *reinterpret_cast<const u16x4*>(p.emb + (size_t)p.eid[m] * N + c0);
#pragma unroll
      for (int c = 0; c < 4; ++c) t[c] = fmaf(p.es, bf2f(e[c]), t[c]);
    }
    *reinterpret_cast<f32x4*>(p.x + o) = t;
    if constexpr (THEN != kNothing) {
      f32x4 nw, nb;
      then_ask<THEN>(p, c0, nw, nb);
      const float s = then_row<THEN>(p, o, nw, nb, t);
      if (THEN == kScaled && lane == 63) p.part[(size_t)m * p.n_nt + j] = s;
    }
  }
}

static bool args_ok(const AddArgs& p, int then) {
  auto off = [](const void* q, int n) { return ((uintptr_t)q % n) != 0; };
  if (p.M <= 0 || p.N <= 0 || p.N % BN || !p.x || off(p.x, 16) || then < kNothing || then > kScaled) return false;
  if (then != kNothing && (!p.nw || !p.h || off(p.nw, 16) || off(p.h, 8))) return false;
  if (then == kDyt && (!p.nb || off(p.nb, 16) || p.rs || p.eid)) return false;
  if (then == kScaled && !p.part) return false;
  if (p.rs && (p.rn < 1 || p.rn > 64 || !(p.rw > 0.f))) return false;
  return !p.eid || (p.emb && !off(p.emb, 8));
}

}  // namespace padd
}  // namespace k8s

using namespace k8s;

#define K8S_ADD_PARAMS                                                                                                     \
  float *x, float sy, const float *rs, int rn, float rw, float reps, const int *eid, const void *emb, float es, int then,    \
      float alpha, const float *nw, const float *nb, void *h, float *part, int M, int N
static padd::AddArgs add_args(K8S_ADD_PARAMS) {
  (void)then;
  padd::AddArgs p{};
  p.x = x, p.sy = sy, p.rs = rs, p.rn = rn, p.rw = rw, p.reps = reps, p.eid = eid, p.emb = (const uint16_t*)emb, p.es = es;
  p.alpha = alpha, p.nw = nw, p.nb = nb, p.h = (uint16_t*)h, p.part = part, p.M = M, p.N = N, p.n_nt = N / padd::BN;
  return p;
}
#define K8S_ADD_NAMES x, sy, rs, rn, rw, reps, eid, emb, es, then, alpha, nw, nb, h, part, M, N

// then: 0 nothing, 1 h = bf16(tanh(alpha x) nw + nb) (without rs and eid), 2 h = bf16(x nw) and part [M][N / 256].  f: rows of a tile
// / 32 (4, 5, 6, 8).  N a multiple of 256, K of 64; x, nw, nb, a (its rows too) and w lie on 16 bytes, h and emb on 8.
K8S_API int k8s_gemm_add(const void* a, int lda, const void* w, K8S_ADD_PARAMS, int K, int f, hipStream_t s) {
  using namespace k8s::padd;
  AddArgs p = add_args(K8S_ADD_NAMES);
  p.a = (const uint16_t*)a, p.lda = lda, p.w = (const uint16_t*)w, p.K = K;
  if (!args_ok(p, then) || K <= 0 || K % BK || !a || !w || ((uintptr_t)a & 15) || ((uintptr_t)w & 15) || lda % 8 || lda < K)
    return (int)hipErrorInvalidValue;
  switch (f) {
    case 4: return launch_then<4>(p, then, s);
    case 5: return launch_then<5>(p, then, s);
    case 6: return launch_then<6>(p, then, s);
    case 8: return launch_then<8>(p, then, s);
  }
  return (int)hipErrorInvalidValue;
}

// The same with the product as it lies in y [planes][M][N].
K8S_API int k8s_add_rows(const float* y, int planes, K8S_ADD_PARAMS, hipStream_t s) {
  using namespace k8s::padd;
  const AddArgs p = add_args(K8S_ADD_NAMES);
  if (!args_ok(p, then) || !y || ((uintptr_t)y & 15) || planes < 1) return (int)hipErrorInvalidValue;
  switch (then) {
    case kNothing: hipLaunchKernelGGL((add_rows_kernel<kNothing>), dim3(M), dim3(256), 0, s, p, y, planes); break;
    case kDyt: hipLaunchKernelGGL((add_rows_kernel<kDyt>), dim3(M), dim3(256), 0, s, p, y, planes); break;
    default: hipLaunchKernelGGL((add_rows_kernel<kScaled>), dim3(M), dim3(256), 0, s, p, y, planes); break;
  }
  return (int)hipGetLastError();
}
