// Portions of several tokens through the matrix-state recurrences of matrix_mem.hip (the gated delta rule and the matrix
// memory; definitions there), in tiles of 16 tokens on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32: fp32 operands
// and sums, as the token-by-token form has them).
//
// With S [D][V] the state in front of a tile, G_i the product of the decays up to and with token i of the tile (per key
// channel for the delta rule, one number for the memory) and G_(j,i] the product over j < t <= i:
//   delta rule:   A_ij = beta_i sum_d k_i k_j G_(j,i]  (j < i),   P_ij = sum_d q_i k_j G_(j,i]  (j <= i)
//                 U = (I + A)^-1 diag(beta) (V - (K G) S),   O = (Q G) S + P U,   S <- G_15 S + (K G_(j,15])^T U
//   memory:       P_ij = (q_i . k_j) G_(j,i] w_j,            O = (Q G) S + P V,   S <- G_15 S + (K G_(j,15] w_j)^T V
// (w the input factor; the normaliser is one more column whose values are 1).
//
// tile_*_kernel, one workgroup per (tile, head), all tiles at once: Q G, K G, (K G_(j,15])^T, P, T = (I + A)^-1 diag(beta)
// and G_15 into a workspace.  The products over (j, i] are formed by multiplying decays, never as ratios or exponentials of
// differences, so that they hold for any decay; T by forward substitution.  A value that is not finite reaches its own and
// later tokens, never earlier ones (lower_rows), as token by token.
// tile_state_kernel, one workgroup per (segment, head, 64 columns), walks the tiles of its segment.  A wave holds the state
// of 16 columns in accumulators: tile dt, rows d = 16 dt + 4 hq + i, column r (lane = 16 hq + r).  A contraction may take
// its index in any order that both operands agree on, so register i of accumulator dt IS the second operand of the step
// that takes rows 16 dt + i + {0, 4, 8, 12}: neither the state nor U is ever moved between lanes.  The next tile's
// operands but one are fetched into registers while the current one is computed, one barrier per tile.
//
// What bounds it: the chain of tiles.  Per tile and wave 3 D / 4 + 8 matrix instructions of 32 cycles (56 at D = 64,
// 0.75 us) on one wave per SIMD, and around them the way of a tile's operands through LDS: 1.8 us per tile where one
// workgroup has a CU to itself.  Two tiles of lead cover the way from memory.  Sixteen tokens because a larger tile adds
// products over its pairs and shortens nothing: the state's own products, 3 D V per token, are the same.
// 16 heads, D 64, V 128, 8 sequences of 2048 tokens: delta rule 2.70 ms (in chunks of 64 tokens, token by token within
// them, twice) -> 0.14 (tile_delta, 239 MB written) + 0.23 ms;  memory 1.33 -> 0.09 + 0.25 ms.  64 sequences of about 390:
// 2.13 -> 0.24 + 0.35 and 1.75 -> 0.14 + 0.36 ms.  Error against 64 bits as before: 1.6e-7 -> 1.7e-7, 5.9e-6 -> 6.0e-6.
#include "common.h"

namespace k8s {

constexpr int kTs = 16;          // tokens per tile

// floats of a (tile, head) in the workspace, in this order
template <int D, int KIND>
struct TileWs {
  static constexpr int q = 0;                                   // [16][D]
  static constexpr int k = 16 * D;                              // [16][D] (delta rule)
  static constexpr int kt = KIND == 0 ? 32 * D : 16 * D;        // [D][16]
  static constexpr int p = kt + 16 * D;                         // [16][16]
  static constexpr int t = p + 256;                             // [16][16] (delta rule)
  static constexpr int e = KIND == 0 ? t + 256 : t;             // [D]
  static constexpr int all = e + D;
};

// the same parts in LDS, rows padded by 4 against bank conflicts
template <int D, int KIND>
struct TileLds {
  using W = TileWs<D, KIND>;
  static constexpr int ld = D + 4, lt = kTs + 4;
  static constexpr int k = kTs * ld, kt = k + (KIND == 0 ? kTs * ld : 0), p = kt + D * lt, t = p + kTs * lt,
                       e = t + (KIND == 0 ? kTs * lt : 0), all = e + D;
  static __device__ __forceinline__ int of(int i) {      // where float i (a multiple of 4) of the workspace goes
    if (i < W::kt) return i / D * ld + i % D;             // q rows, then k rows
    if (i < W::e) return kt + (i - W::kt) / kTs * lt + (i - W::kt) % kTs;
    return e + i - W::e;
  }
};

struct TileArgs {
  const void* x;               // rows: q | k | v ...
  long xs;                     // row stride
  const float* a;              // [T][H D] (delta rule)
  const float* rate;
  const float* dt_bias;
  const float* beta;
  int bs;
  const float* ab;             // [T][H][3] (memory)
  const int* tiles;            // [n][4]: segment, first row, rows, -
  const int* seg_row0;         // [n_seg + 1]
  const int* seg_tile0;        // [n_seg + 1]
  float* ws;
  float* state;
  float* nstate;
  const int* seg_pos0;
  const int* seg_slot;
  float* out;
  float* nq;
  float* spare;                // 256 floats behind the tiles' workspace
  int H, G, V;
  float unit_eps;
};

template <typename T>
__device__ __forceinline__ float tld(const T* p, size_t i);
template <>
__device__ __forceinline__ float tld<float>(const float* p, size_t i) { return p[i]; }
template <>
__device__ __forceinline__ float tld<uint16_t>(const uint16_t* p, size_t i) { return bf2f(p[i]); }

// sum over 16 neighbouring lanes, left in all of them
__device__ __forceinline__ float row_sum16(float v) {
#define K8S_ROR(n) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x120 + n, 0xf, 0xf, true))
  K8S_ROR(8);
  K8S_ROR(4);
  K8S_ROR(2);
  K8S_ROR(1);
#undef K8S_ROR
  return v;
}

__device__ __forceinline__ float tsoftplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// the columns of (Q G), (K G) and the rows of (K G_(j,15])^T, G_15: thread d < D of the first 128 walks the tile forwards,
// of the last 128 backwards.  WK: the memory's per-token input factors [16] (null: none).
template <int D, int KIND>
__device__ __forceinline__ void tile_prefix(const float* sq, const float* sk, const float* sg, int ld, int gstep,
                                            const float* wk, float* w) {
  using W = TileWs<D, KIND>;
  const int tid = threadIdx.x, d = tid & 127;
  if (d >= D) return;
  if (tid < 128) {
    float g = 1.f;
#pragma unroll
    for (int t = 0; t < kTs; ++t) {
      g *= sg[t * gstep + (gstep > 1 ? d : 0)];
      w[W::q + t * D + d] = sq[t * ld + d] * g;
      if (KIND == 0) w[W::k + t * D + d] = sk[t * ld + d] * g;
    }
    w[W::e + d] = g;
  } else {
    float g = 1.f;
    float o[kTs];
#pragma unroll
    for (int t = kTs - 1; t >= 0; --t) {
      o[t] = sk[t * ld + d] * g * (wk ? wk[t] : 1.f);
      g *= sg[t * gstep + (gstep > 1 ? d : 0)];
    }
#pragma unroll
    for (int t = 0; t < kTs; t += 4) *reinterpret_cast<f32x4*>(w + W::kt + d * kTs + t) = f32x4{o[t], o[t + 1], o[t + 2], o[t + 3]};
  }
}

template <int D, typename TA>
__global__ void __launch_bounds__(256) tile_delta_kernel(TileArgs p) {
  using W = TileWs<D, 0>;
  constexpr int LD = D + 4, LA = kTs + 4;
  __shared__ __attribute__((aligned(16))) float sq[kTs * LD], sk[kTs * LD], sg[kTs * LD], sA[kTs * LA], sP[kTs * LA];
  __shared__ float sf[2 * kTs], sb[kTs];
  const int it = blockIdx.x, hh = blockIdx.y, tid = threadIdx.x;
  const int r0 = p.tiles[it * 4 + 1], n = p.tiles[it * 4 + 2];
  const int H = p.H, kvh = hh / (H / p.G), GD = p.G * D;
  const TA* x = (const TA*)p.x;
  const float rate = p.rate[hh];
  for (int e = tid; e < kTs * D; e += 256) {
    const int t = e / D, d = e - t * D;
    float q = 0.f, k = 0.f, g = 1.f;
    if (t < n) {
      const size_t row = (size_t)(r0 + t) * p.xs;
      q = tld(x, row + kvh * D + d);
      k = tld(x, row + GD + kvh * D + d);
      g = expf(-rate * tsoftplus(p.a[(size_t)(r0 + t) * H * D + hh * D + d] + p.dt_bias[hh * D + d]));
    }
    sq[t * LD + d] = q;
    sk[t * LD + d] = k;
    sg[t * LD + d] = g;
  }
  if (tid < kTs) sb[tid] = tid < n ? 1.f / (1.f + expf(-p.beta[(size_t)(r0 + tid) * p.bs + hh])) : 0.f;
  for (int e = tid; e < kTs * LA; e += 256) {
    sA[e] = 0.f;
    sP[e] = 0.f;
  }
  __syncthreads();
  {  // unit-length factors: eight lanes per (token, q or k)
    const int pr = tid >> 3, sub = tid & 7;
    const float* src = (pr & 1 ? sk : sq) + (pr >> 1) * LD;
    float ss = 0.f;
    for (int d = sub; d < D; d += 8) ss = fmaf(src[d], src[d], ss);
    ss += __shfl_xor(ss, 1, 64);
    ss += __shfl_xor(ss, 2, 64);
    ss += __shfl_xor(ss, 4, 64);
    if (sub == 0) sf[pr] = (pr & 1 ? 1.f : 1.f / sqrtf((float)D)) / sqrtf(ss + p.unit_eps);
  }
  __syncthreads();
  for (int e = tid; e < kTs * D; e += 256) {
    const int t = e / D, d = e - t * D;
    sq[t * LD + d] *= sf[2 * t];
    sk[t * LD + d] *= sf[2 * t + 1];
  }
  __syncthreads();
  float* w = p.ws + ((size_t)it * H + hh) * W::all;
  tile_prefix<D, 0>(sq, sk, sg, LD, LD, nullptr, w);
  {  // 16 lanes per j carry k_j through the decays of the tokens behind it
    const int j = tid >> 4, l = tid & 15, j0 = (tid >> 6) * 4;
    constexpr int M = D / 16;
    float c[M];
#pragma unroll
    for (int m = 0; m < M; ++m) c[m] = sk[j * LD + l + 16 * m];
    for (int i = j0; i < kTs; ++i) {
      float ka = 0.f, qa = 0.f;
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const int o = i * LD + l + 16 * m;
        if (i > j) c[m] *= sg[o];
        ka = fmaf(sk[o], c[m], ka);
        qa = fmaf(sq[o], c[m], qa);
      }
      ka = row_sum16(ka);
      qa = row_sum16(qa);
      if (l == 0 && i >= j) {
        sP[i * LA + j] = qa;
        if (i > j) sA[i * LA + j] = ka * sb[i];
      }
    }
  }
  __syncthreads();
  w[W::p + tid] = sP[(tid >> 4) * LA + (tid & 15)];
  if (tid < kTs) {   // column c of the inverse by forward substitution
    float t[kTs];
#pragma unroll
    for (int i = 0; i < kTs; ++i) {
      float v = i == tid ? sb[tid] : 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) v = fmaf(-sA[i * LA + j], t[j], v);
      t[i] = v;
      w[W::t + i * kTs + tid] = v;
    }
  }
}

template <int D>
__global__ void __launch_bounds__(256) tile_memory_kernel(TileArgs p) {
  using W = TileWs<D, 1>;
  constexpr int LD = D + 4;
  __shared__ __attribute__((aligned(16))) float sq[kTs * LD], sk[kTs * LD];
  __shared__ float sf[kTs], sw[kTs];
  const int it = blockIdx.x, hh = blockIdx.y, tid = threadIdx.x;
  const int r0 = p.tiles[it * 4 + 1], n = p.tiles[it * 4 + 2];
  const int H = p.H, HD = H * D;
  const float* x = (const float*)p.x;
  for (int e = tid; e < kTs * D; e += 256) {
    const int t = e / D, d = e - t * D;
    const float* row = x + (size_t)(r0 + t) * p.xs + hh * D + d;
    sq[t * LD + d] = t < n ? row[0] : 0.f;
    sk[t * LD + d] = t < n ? row[HD] : 0.f;
  }
  if (tid < kTs) {
    const float* ab = p.ab + ((size_t)(r0 + tid) * H + hh) * 3;
    sf[tid] = tid < n ? ab[0] : 1.f;
    sw[tid] = tid < n ? ab[1] : 0.f;
  }
  __syncthreads();
  float* w = p.ws + ((size_t)it * H + hh) * W::all;
  tile_prefix<D, 1>(sq, sk, sf, LD, 1, sw, w);
  const int i = tid >> 4, j = tid & 15;
  float s = 0.f;
  if (j <= i) {
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int d = 0; d < D; d += 4) {
      const f32x4 q = *reinterpret_cast<const f32x4*>(sq + i * LD + d), k = *reinterpret_cast<const f32x4*>(sk + j * LD + d);
#pragma unroll
      for (int m = 0; m < 4; ++m) a[m] = fmaf(q[m], k[m], a[m]);
    }
    float g = sw[j];
    for (int t = j + 1; t <= i; ++t) g *= sf[t];
    s = ((a[0] + a[1]) + (a[2] + a[3])) * g;
  }
  w[W::p + tid] = s;
}

// Whether none of this lane's four numbers is infinite or NaN.
__device__ __forceinline__ bool finite4(const f32x4& v) {
  const float z = (v[0] * 0.f + v[1] * 0.f) + (v[2] * 0.f + v[3] * 0.f);
  return z == z;
}

// c + A B for a lower triangular A [16][16] (af: its operand), row i from the rows of B up to i alone: a zero above the
// diagonal times a number that is not finite would be NaN in the rows of earlier tokens.
__device__ __forceinline__ f32x4 lower_rows(const f32x4& af, const f32x4& b, const f32x4& c, int hq) {
  f32x4 out = c;
#pragma unroll 1
  for (int i = 0; i < kTs; ++i) {
    f32x4 t = c;
#pragma unroll
    for (int e = 0; e < 4; ++e) t = __builtin_amdgcn_mfma_f32_16x16x4f32(af[e], 4 * hq + e <= i ? b[e] : 0.f, t, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = 4 * hq + e == i ? t[e] : out[e];
  }
  return out;
}

template <int D, int KIND, typename TA>
__global__ void __launch_bounds__(256) tile_state_kernel(TileArgs p) {
  using W = TileWs<D, KIND>;
  using M = TileLds<D, KIND>;
  constexpr int ND = D / 16, LD = M::ld, LT = M::lt, kBuf = M::all, oK = M::k, oT = M::kt, oP = M::p, oI = M::t, oE = M::e;
  constexpr int NP = W::all / 4, B = (NP + 255) / 256;          // 16-byte pieces of a tile's operands, per thread
  extern __shared__ __attribute__((aligned(16))) float lds[];   // two of kBuf
  const int sg = blockIdx.x, hh = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, r = lane & 15, hq = lane >> 4, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = p.H, V = p.V, X = KIND == 1 ? 1 : 0;
  const int vcol = blockIdx.z * 64 + 16 * wv + r;
  const bool own = vcol < V + X, norm = KIND == 1 && vcol == V;
  const int c0 = p.seg_tile0[sg], c1 = p.seg_tile0[sg + 1], row0 = p.seg_row0[sg], row1 = p.seg_row0[sg + 1];
  const size_t so = (size_t)p.seg_slot[sg] * H + hh;
  float* st = norm ? p.nstate + so * D : p.state + so * D * V + vcol;
  const int sstep = norm ? 1 : V;
  const bool fresh = p.seg_pos0[sg] == 0;
  f32x4 S[ND];
#pragma unroll
  for (int dt = 0; dt < ND; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[dt][i] = (own && !fresh) ? st[(size_t)(16 * dt + 4 * hq + i) * sstep] : 0.f;
  const TA* xv = (const TA*)p.x + (KIND == 0 ? 2 * p.G * D : 2 * H * D) + (size_t)hh * V + min(vcol, V - 1);
  // Every load and store of the walk is issued by every lane, whatever the tile (rows past the end read the last one, the
  // pieces past the last repeat it, results that nobody wants go to a spare place): with a branch around one of them the
  // number of accesses in flight is no longer known and each wait becomes one for all of them.
  float* op = norm ? p.nq + (size_t)row0 * H + hh : p.out + ((size_t)row0 * H + hh) * V + vcol;
  const size_t ostep = norm ? H : (size_t)H * V;
  float* spare = p.spare + tid;
  int piece[B], into[B];
#pragma unroll
  for (int b = 0; b < B; ++b) {
    piece[b] = 4 * min(tid + 256 * b, NP - 1);
    into[b] = M::of(piece[b]);
  }
  struct Part {                                  // a tile's operands on their way, and this lane's values
    f32x4 w[B];
    TA v[4];
  };
  auto fetch = [&](int c, Part& f) {
    const float* w = p.ws + ((size_t)c * H + hh) * W::all;
#pragma unroll
    for (int b = 0; b < B; ++b) f.w[b] = *reinterpret_cast<const f32x4*>(w + piece[b]);
#pragma unroll
    for (int i = 0; i < 4; ++i) f.v[i] = xv[(size_t)min(row0 + kTs * (c - c0) + 4 * hq + i, row1 - 1) * p.xs];
  };
  // one tile: its operands into LDS, the next but one's on their way, then the products
  auto step = [&](int c, Part& f) {
    float* b = lds + ((c - c0) & 1) * kBuf;      // (last read two tiles ago: one barrier lies between)
#pragma unroll
    for (int k = 0; k < B; ++k) *reinterpret_cast<f32x4*>(b + into[k]) = f.w[k];
    const int r0 = row0 + kTs * (c - c0), n = row1 - r0;
    f32x4 U;
#pragma unroll
    for (int i = 0; i < 4; ++i) U[i] = own && 4 * hq + i < n ? (norm ? 1.f : tld(f.v, i)) : 0.f;
    __syncthreads();
    fetch(min(c + 2, c1 - 1), f);
    f32x4 O = {0.f, 0.f, 0.f, 0.f}, R = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) {
      const f32x4 qf = *reinterpret_cast<const f32x4*>(b + r * LD + 16 * dt + 4 * hq);
      f32x4 kf;
      if (KIND == 0) kf = *reinterpret_cast<const f32x4*>(b + oK + r * LD + 16 * dt + 4 * hq);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (KIND == 0) R = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i], S[dt][i], R, 0, 0, 0);
        O = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[i], S[dt][i], O, 0, 0, 0);
      }
    }
    if (KIND == 0) {
      const f32x4 tf = *reinterpret_cast<const f32x4*>(b + oI + r * LT + 4 * hq);
      R = U - R;
      U = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) U = __builtin_amdgcn_mfma_f32_16x16x4f32(tf[i], R[i], U, 0, 0, 0);
    }
    const f32x4 pf = *reinterpret_cast<const f32x4*>(b + oP + r * LT + 4 * hq), Oq = O;
#pragma unroll
    for (int i = 0; i < 4; ++i) O = __builtin_amdgcn_mfma_f32_16x16x4f32(pf[i], U[i], O, 0, 0, 0);
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) {
      const f32x4 ef = *reinterpret_cast<const f32x4*>(b + oE + 16 * dt + 4 * hq);
      const f32x4 tf = *reinterpret_cast<const f32x4*>(b + oT + (16 * dt + r) * LT + 4 * hq);
#pragma unroll
      for (int i = 0; i < 4; ++i) S[dt][i] *= ef[i];
#pragma unroll
      for (int i = 0; i < 4; ++i) S[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(tf[i], U[i], S[dt], 0, 0, 0);
    }
    // Rare: the two triangular products row by row (the state takes in every token either way).  Behind the state's own
    // products, off the chain from tile to tile.
    if (__any(!finite4(U) || (KIND == 0 && !finite4(R)))) {
      if (KIND == 0) U = lower_rows(*reinterpret_cast<const f32x4*>(b + oI + r * LT + 4 * hq), R, f32x4{0.f, 0.f, 0.f, 0.f}, hq);
      O = lower_rows(*reinterpret_cast<const f32x4*>(b + oP + r * LT + 4 * hq), U, Oq, hq);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 4 * hq + i;
      *(own && t < n ? op + (size_t)(r0 - row0 + t) * ostep : spare) = O[i];
    }
  };
  Part fa, fb;
  if (c0 >= c1) return;                          // a segment without rows
  fetch(c0, fa);
  fetch(min(c0 + 1, c1 - 1), fb);
  for (int c = c0; c < c1; c += 2) {
    step(c, fa);
    if (c + 1 < c1) step(c + 1, fb);
  }
  if (own) {
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) st[(size_t)(16 * dt + 4 * hq + i) * sstep] = S[dt][i];
  }
}

template <int D, int KIND, typename TA>
static int launch_tile_state(const TileArgs& p, int n_seg, int n_tiles, hipStream_t s) {
  if constexpr (KIND == 0)
    hipLaunchKernelGGL((tile_delta_kernel<D, TA>), dim3(n_tiles, p.H), dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((tile_memory_kernel<D>), dim3(n_tiles, p.H), dim3(256), 0, s, p);
  constexpr int lds = 2 * TileLds<D, KIND>::all * sizeof(float);
  auto k = tile_state_kernel<D, KIND, TA>;
  if (lds > 48 * 1024 && hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds))
    return (int)hipGetLastError();
  hipLaunchKernelGGL(k, dim3(n_seg, p.H, (p.V + KIND + 63) / 64), dim3(256), lds, s, p);
  return (int)hipGetLastError();
}

template <int KIND, typename TA>
static int launch_tiles(const TileArgs& p, int D, int n_seg, int n_tiles, hipStream_t s) {
  switch (D) {
    case 16: return launch_tile_state<16, KIND, TA>(p, n_seg, n_tiles, s);
    case 32: return launch_tile_state<32, KIND, TA>(p, n_seg, n_tiles, s);
    case 64: return launch_tile_state<64, KIND, TA>(p, n_seg, n_tiles, s);
    case 96: return launch_tile_state<96, KIND, TA>(p, n_seg, n_tiles, s);
    case 128: return launch_tile_state<128, KIND, TA>(p, n_seg, n_tiles, s);
    default: return (int)hipErrorInvalidValue;
  }
}

template <int KIND>
static int ws_floats(int D) {
  switch (D) {
    case 16: return TileWs<16, KIND>::all;
    case 32: return TileWs<32, KIND>::all;
    case 64: return TileWs<64, KIND>::all;
    case 96: return TileWs<96, KIND>::all;
    case 128: return TileWs<128, KIND>::all;
    default: return 0;
  }
}

}  // namespace k8s

using namespace k8s;

// floats per (tile, head), and 256 more in all, that the tiled form of the delta rule (kind 0) or the matrix memory (kind 1)
// works in;
// 0: it does not take these sizes
K8S_API int k8s_tile_state_ws(int kind, int D) { return kind == 0 ? ws_floats<0>(D) : ws_floats<1>(D); }

// gated delta rule, arguments as k8s_gated_delta; tiles [n][4] cut every segment into tiles of 16 rows, seg_tile0 [n_seg + 1]
K8S_API int k8s_gated_delta_tiles(const void* qkv, int dt, const float* a, const float* rate, const float* dt_bias,
                                  const float* beta, int bs, float* state, const int* seg_row0,
                                  const int* seg_pos0, const int* seg_slot, float* out, int n_seg, int H, int G, int D,
                                  int V, float unit_eps, hipStream_t s,
                                  const int* tiles, int n_tiles, const int* seg_tile0, float* ws) {
  if (n_seg <= 0 || n_tiles <= 0) return 0;
  if (G < 1 || H % G || V < 1 || !k8s_tile_state_ws(0, D) || !tiles || !seg_tile0 || !ws) return (int)hipErrorInvalidValue;
  TileArgs p{};
  p.x = qkv;
  p.xs = 2L * G * D + (long)H * V;
  p.a = a;
  p.rate = rate;
  p.dt_bias = dt_bias;
  p.beta = beta;
  p.bs = bs;
  p.state = state;
  p.seg_row0 = seg_row0;
  p.seg_pos0 = seg_pos0;
  p.seg_slot = seg_slot;
  p.out = out;
  p.H = H;
  p.G = G;
  p.V = V;
  p.unit_eps = unit_eps;
  p.tiles = tiles;
  p.seg_tile0 = seg_tile0;
  p.ws = ws;
  p.spare = ws + (size_t)n_tiles * H * k8s_tile_state_ws(0, D);
  return dt == 0 ? launch_tiles<0, uint16_t>(p, D, n_seg, n_tiles, s) : launch_tiles<0, float>(p, D, n_seg, n_tiles, s);
}

namespace k8s {
// matrix memory between its gates and its denominators (matrix_mem.hip): raw read-outs S^T q and n.q of every token
int matrix_memory_tiles(const float* x, int xs, const float* ab, float* state, float* nstate, const int* seg_row0,
                        const int* seg_pos0, const int* seg_slot, float* nq, float* out, int n_seg, int H, int D, int V, hipStream_t s,
                        const int* tiles, int n_tiles, const int* seg_tile0, float* ws) {
  if (!k8s_tile_state_ws(1, D) || n_tiles <= 0 || !seg_tile0 || !ws) return (int)hipErrorInvalidValue;
  TileArgs p{};
  p.x = x;
  p.xs = xs;
  p.ab = ab;
  p.state = state;
  p.nstate = nstate;
  p.seg_row0 = seg_row0;
  p.seg_pos0 = seg_pos0;
  p.seg_slot = seg_slot;
  p.out = out;
  p.nq = nq;
  p.H = H;
  p.G = H;
  p.V = V;
  p.tiles = tiles;
  p.seg_tile0 = seg_tile0;
  p.ws = ws;
  p.spare = ws + (size_t)n_tiles * H * k8s_tile_state_ws(1, D);
  return launch_tiles<1, float>(p, D, n_seg, n_tiles, s);
}
}  // namespace k8s
