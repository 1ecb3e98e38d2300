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
// Tiles of 32 F rows x 256 columns, one 512-thread workgroup a compute unit; F is chosen by how the tiles fill whole waves of 256
// (ops/linear.py: add_plan).  K comes in tiles of 64 by LDS-DMA, three of them staged (two where the rows leave no room), and is
// worked off in two phases, W's columns 0 - 127 and 128 - 255: a wave multiplies 16 F rows x 32 columns a phase and reads its rows'
// fragments once a tile.  Waves 4 - 7 run one barrier behind waves 0 - 3, so that on every SIMD one of two waves issues matrix
// instructions while the other reads fragments and asks for tiles.  In slots between barriers, u the K tile:
//   waves 0 - 3:  4u  read X0, W0    4u+1  multiply    4u+2  read W1            4u+3  multiply
//   waves 4 - 7:                     4u+1  read X1, W0  4u+2  multiply          4u+3  read W1      4u+4  multiply
// A slot's reads have ended when the next slot has (the multiplication waits for them).  So a buffer of tile u takes its next tile
// from slot 4u+2 (X0: read by waves 0 - 3 alone), 4u+3 (X1, W0) and 4u+5 (W1); each wave asks in its reading slots, W by halves of
// the waves.  A wave waits for its own share of what is read next in the reading slot before: FLY counts what it has asked for
// since.  Past the last tile the last one is asked for again, into a buffer that nobody reads, so that the counts hold.
//
// What bounds it: with 256-row tiles the power limit (1.4 PFLOP/s); with 128 and 160 rows the fragments' way out of LDS, a
// phase's 12 to 14 reads a wave in front of 16 to 20 matrix instructions (1.15 - 1.2 PFLOP/s, what the library's tiles of that size
// do).  us of product and pass / of this with tanh, 2048 x 2048 and 2048 x 8192 at 2600, 4096, 4850, 6144, 10000, 16384 rows:
//   44 / 40, 58 / 46, 68 / 54, 70 / 64, 114 / 111, 181 / 161;   110 / 108, 143 / 129, 158 / 142, 177 / 172, 340 / 289, 428 / 414;
// with the norm left to the product behind 42 / 36, 57 / 41, 68 / 49, 70 / 59, 114 / 99, 175 / 146;   110 / 104, 138 / 124, 155 /
// 138, 175 / 167, 341 / 280, 425 / 398.  tanh is 5 to 11 us of it a wave of tiles: vector instructions while the matrix units wait.
// The residual asked for in front of the last tile's products, with that tile's code of its own, changed nothing (registers).
#include <type_traits>

#include "common.h"

namespace k8s {
namespace padd {

constexpr int BN = 256, BK = 64, ROW_B = 2 * BK;          // a staged row: 128 bytes
constexpr int GM = 4;                                     // row tiles of a group that shares its columns' weights

typedef __attribute__((address_space(3))) void lds_void_t;
__device__ __forceinline__ void glds16(const uint16_t* src, unsigned char* lds_dst) {
  __builtin_amdgcn_global_load_lds(src, (lds_void_t*)lds_dst, 16, 0, 0);
}
__device__ __forceinline__ void bar() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}
template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ float last_lane(float v) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ void lds_bar() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  bar();
}

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
  constexpr int BM = 32 * F, HM = 16 * F;                  // rows of a tile, of a half
  constexpr int NB = F <= 5 ? 3 : 2;                       // staged K tiles
  constexpr int XA = (2 * F + 3) / 4;                      // DMA instructions of a wave for its half of X
  constexpr int XB = HM * ROW_B, WB = 128 * ROW_B, BUF = 2 * XB + 2 * WB;
  constexpr int LDS = NB * BUF > HM * 1024 ? NB * BUF : HM * 1024;
  static_assert(LDS <= 160 * 1024);
  __shared__ __attribute__((aligned(1024))) unsigned char sm[LDS];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wv >> 2, wc = wv & 3;
  int tm, tn;
  {
    const int T = p.n_mt * p.n_nt, b = blockIdx.x, xcd = b & 7, q = T >> 3, r = T & 7;
    const int t = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (b >> 3);
    const int gsz = GM * p.n_nt, first = t / gsz * GM, gm = min(p.n_mt - first, GM);
    tm = first + (t % gsz) % gm;
    tn = (t % gsz) / gm;
  }
  const int M = p.M, N = p.N, K = p.K, m0 = tm * BM, nt = K / BK;

  // ---- what this wave stages: its own half of X, a part of both halves of W
  const uint16_t* xs[XA];
  uint32_t xd[XA];
#pragma unroll
  for (int i = 0; i < XA; ++i) {
    const int j = min(4 * i + wc, 2 * F - 1), R = 8 * j + (lane >> 3);      // (past the last: the last again)
    xs[i] = p.a + (size_t)min(m0 + HM * wr + R, M - 1) * p.lda + 8 * ((lane & 7) ^ ((R >> 1) & 7));
    xd[i] = wr * XB + j * 1024;
  }
  const uint16_t* wsrc[2][2];
  uint32_t wd[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int j = 8 * wr + 2 * wc + i, R = 8 * j + (lane >> 3), rho = R & 31;
    const int col = 32 * (R >> 5) + 8 * ((rho >> 2) & 3) + 4 * (rho >> 4) + (rho & 3);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      wsrc[h][i] = p.w + (size_t)(tn * BN + 128 * h + col) * K + 8 * ((lane & 7) ^ ((R >> 1) & 7));
    wd[i] = 2 * XB + j * 1024;
  }
  auto put_x = [&](int v, int buf) {
    const int kt = min(v, nt - 1) * BK;
#pragma unroll
    for (int i = 0; i < XA; ++i) glds16(xs[i] + kt, sm + buf * BUF + xd[i]);
  };
  auto put_w = [&](int h, int v, int buf) {
    const int kt = min(v, nt - 1) * BK;
#pragma unroll
    for (int i = 0; i < 2; ++i) glds16(wsrc[h][i] + kt, sm + buf * BUF + h * WB + wd[i]);
  };
  const int frow = lane & 15, fhi = lane >> 4;
  const int f0 = frow * ROW_B + 16 * (fhi ^ ((frow >> 1) & 7));
  f32x4 acc[2][F][2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[h][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 xf[F][2], wf[2][2];
  auto read_x = [&](int buf) {
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        xf[i][ks] = *reinterpret_cast<const bf16x8*>(sm + buf * BUF + wr * XB + 16 * i * ROW_B + (f0 ^ (64 * ks)));
  };
  auto read_w = [&](int h, int buf) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        wf[j][ks] = *reinterpret_cast<const bf16x8*>(sm + buf * BUF + 2 * XB + h * WB + (32 * wc + 16 * j) * ROW_B + (f0 ^ (64 * ks)));
  };
  auto mul = [&](auto H) {
    constexpr int h = decltype(H)::value;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[h][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j][ks], xf[i][ks], acc[h][i][j], 0, 0, 0);
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  auto run = [&](auto WR) {
    constexpr bool second = decltype(WR)::value;
    // DMA instructions of this wave that may be in flight behind what is read next
    constexpr int FLY = (second ? 2 : 0) + (NB == 3 ? 6 + 2 * XA : 2 + XA);
    put_x(0, 0);
    put_w(0, 0, 0);
    put_w(1, 0, 0);
    put_x(1, 1);
    if constexpr (NB == 3) {
      put_w(0, 1, 1);
      put_w(1, 1, 1);
      put_x(2, 2);
    }
    if constexpr (second) put_w(0, NB - 1, NB - 1);
    vm_wait<FLY>();
    bar();
    if constexpr (second) bar();
    int b = 0, bl = NB - 1;                                 // the buffers of tiles u and u - 1
    for (int u = 0; u < nt; ++u) {
      read_x(b);
      read_w(0, b);
      put_w(second, u - 1 + NB, bl);
      vm_wait<FLY>();
      bar();
      mul(H0{});
      bar();
      read_w(1, b);
      if constexpr (!second) put_w(1, u - 1 + NB, bl);
      put_x(u + NB, b);
      if constexpr (second) put_w(0, u + NB, b);
      vm_wait<FLY>();
      bar();
      mul(H1{});
      bar();
      bl = b;
      b = b + 1 == NB ? 0 : b + 1;
    }
    if constexpr (!second) bar();
  };
  if (wr == 0)
    run(std::false_type{});
  else
    run(std::true_type{});
  vm_wait<0>();                                             // no DMA is in flight when the buffers get another use

  // ---- epilogue: acc[h][i][j][v] = row m0 + HM wr + 16 i + frow, column 256 tn + 128 h + 32 wc + 8 fhi + 4 j + v.
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
    if (wr != half) return;
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int r = 16 * i + frow, c = (128 * h + 32 * wc + 8 * fhi + 4 * j) >> 2;
          *reinterpret_cast<f32x4*>(sm + r * 1024 + 16 * (c ^ frow)) = acc[h][i][j];
        }
  };
  auto finish = [&](int half) {
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int r = 8 * i + wv, m = row(half, i);
      f32x4 v = *reinterpret_cast<const f32x4*>(sm + r * 1024 + 16 * (lane ^ (r & 15)));
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
