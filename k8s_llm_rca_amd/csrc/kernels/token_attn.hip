// Attention of single tokens (decode rows) over paged keys, bf16 on v_mfma_f32_16x16x32_bf16: for the masked layers
// (masked_attn.hip) and the latent ones (latent_attn.hip).
//
// One token has one position, so the tile of 16 query rows those kernels give to tokens goes to the HEADS that share a
// key head here: up to 16 heads read a key's bytes once.  A workgroup owns (row, key head, part of the row's keys) and
// its waves take the part's 32-key blocks in turn (wave w: blocks w, w + NW, ..), each with an online softmax of its own;
// the waves' maxima, sums and outputs meet in LDS and are added in wave order.  A row whose keys fit one part is
// finished there (sink, gate, rounding); otherwise token_merge_kernel joins the parts with the same arithmetic.  Blocks,
// waves and parts follow from positions alone, so a row's bits do not depend on the step it is in.
//
// What bounds it: the chain row -> page -> keys -> scores -> join of some 5 us, and that one compute unit takes cold keys
// in at 20 to 30 KB a us (as fragments; tok_turn), far below its share of the caches' rate.  So parts are small (256 masked
// or 128 latent keys: 128 KB of keys and values and 144 KB), and a merge of 3.5 us pays from the second part on.  16 heads
// over 2 of 128 / 16 heads over latents of 256 + 64, us with the merge, and in brackets what a tile of 16 tokens per wave
// (masked) and a wave per 256 keys (latent) took in engine steps of about that size, all with fragments' loads: 1 row at 100
// keys 5.3 / 8.5 (8.4 / 13.5), 8 rows at 1500 10.7 / 12.5 (26 / 36), 64 rows at 400 12.3 / 14.3 (28 / 35).
#include "common.h"
#include "key_runs.h"
#include "state_step.h"

namespace k8s {

constexpr float kTokLog2e = 1.4426950408889634f;

struct TokOut {
  const float* sink;      // [H] or null
  const float* gate;      // rows of stride gs, column h, or null
  int gs;
  uint16_t* out;          // element (row, h, c) at row * ost + h * osh + c
  float* out32;           // the same in fp32 instead
  long ost, osh;
  float* po;              // [items][H][parts][V]: a part's unnormalised output
  float* pml;             // [items][H][parts][2]: its maximum (log2 units) and denominator
  int H, n_parts;
  int hs;                 // heads of one workgroup are hs apart (score maps: theirs lie [head][map])
};

// 1 / denominator (sink included) times the gate; w: the factor of the outputs
__device__ __forceinline__ float tok_finish(const TokOut& a, int row, int head, float m, float l, float& w) {
  const float sk = a.sink ? a.sink[head] * kTokLog2e : -INFINITY;
  const float M = fmaxf(m, sk);
  w = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
  const float L = l * w + (a.sink ? __builtin_amdgcn_exp2f(sk - M) : 0.f);
  const float g = a.gate ? 1.f / (1.f + expf(-a.gate[(size_t)row * a.gs + head])) : 1.f;
  return L == 0.f ? 0.f : g / L;                           // (NaN stays NaN)
}

__device__ __forceinline__ void tok_store4(const TokOut& a, int row, int head, int c, const f32x4& v) {
  const size_t o = (size_t)row * a.ost + (size_t)head * a.osh + c;       // V, the strides: multiples of 16
  if (a.out32)
    *reinterpret_cast<f32x4*>(a.out32 + o) = v;
  else
    *reinterpret_cast<u16x4*>(a.out + o) = u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
}

template <int NW, int V>
struct TokLds {
  static constexpr int P = V + 4;    // row pitch: the four rows a store instruction writes lie 16 banks apart
  alignas(16) float o[NW][16][P];
  float ml[NW][16][2];
};

// The waves' heads -> LDS -> out or a part.  m, l: of head lane & 15, l already summed over the lane quarters.
// o[dt][i]: head 4 (lane >> 4) + i, column 16 dt + (lane & 15).  A wave without a block brings m = -inf and zeros.
// Four columns a thread and every wave's numbers read at once: with a column a thread and a loop over the waves the join
// was the larger part of the kernel (latent, 32 keys a part: 18.9 us).
template <int NW, int ND>
__device__ __forceinline__ void tok_join(TokLds<NW, ND * 16>& s, const TokOut& a, int row, int head0, int nh, int part,
                                         float m, float l, const f32x4 (&o)[ND]) {
  constexpr int V = ND * 16;
  const int lane = threadIdx.x & 63, r = lane & 15, hq = lane >> 4, wv = threadIdx.x >> 6;
  if (hq == 0) {
    s.ml[wv][r][0] = m;
    s.ml[wv][r][1] = l;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (4 * hq + i < nh) {
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) s.o[wv][4 * hq + i][16 * dt + r] = o[dt][i];
    }
  __syncthreads();
  for (int e = threadIdx.x; e < nh * (V / 4); e += 64 * NW) {
    const int hh = e / (V / 4), c = 4 * (e % (V / 4)), head = head0 + hh * a.hs;
    float mw[NW], lw[NW];
    f32x4 ow[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      mw[w] = s.ml[w][hh][0];
      lw[w] = s.ml[w][hh][1];
      ow[w] = *reinterpret_cast<const f32x4*>(&s.o[w][hh][c]);
    }
    float M = mw[0], L = 0.f;
#pragma unroll
    for (int w = 1; w < NW; ++w) M = fmaxf(M, mw[w]);
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = mw[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw[w] - M);   // -inf: no visible key
      L = fmaf(lw[w], f, L);
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[k] = fmaf(ow[w][k], f, acc[k]);
    }
    if (a.n_parts > 1) {
      const size_t pi = ((size_t)blockIdx.x * a.H + head) * a.n_parts + part;
      *reinterpret_cast<f32x4*>(a.po + pi * V + c) = acc;
      if (c == 0) {
        a.pml[pi * 2] = M;
        a.pml[pi * 2 + 1] = L;
      }
    } else {
      float w;
      const float f = tok_finish(a, row, head, M, L, w);
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[k] *= w * f;
      tok_store4(a, row, head, c, acc);
    }
  }
}

// a part without keys
__device__ __forceinline__ void tok_empty(const TokOut& a, int head0, int nh, int part) {
  if ((int)threadIdx.x < nh) {
    float* ml = a.pml + (((size_t)blockIdx.x * a.H + head0 + threadIdx.x * a.hs) * a.n_parts + part) * 2;
    ml[0] = -INFINITY;
    ml[1] = 0.f;
  }
}

// One workgroup per (row, head).  Group j of V / 4 threads adds the parts j, j + S, .. (S groups), the groups' sums are
// added in order.  Nothing but the sum waits for anything: the first parts are on their way while the maxima arrive.
__global__ void __launch_bounds__(256) token_merge_kernel(TokOut a, const int* __restrict__ items, int V) {
  constexpr int U = 4;
  __shared__ f32x4 sum[256];
  const int it = blockIdx.x / a.H, head = blockIdx.x % a.H, lane = threadIdx.x & 63, np = a.n_parts;
  const int row = items[it * 4 + 1], W = V / 4, S = 256 / W, j = threadIdx.x / W, c = threadIdx.x % W;
  const size_t p0 = (size_t)blockIdx.x * np;
  const f32x4* po = reinterpret_cast<const f32x4*>(a.po + p0 * V) + c;
  const float* ml = a.pml + p0 * 2;
  const bool on = j < S;
  f32x4 v[U];
  float mv[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int p = j + S * u;
    const bool has = on && p < np;
    v[u] = po[(size_t)(has ? p : 0) * W];
    mv[u] = has ? ml[p * 2] : -INFINITY;
  }
  float M = -INFINITY, L = 0.f;
  for (int p = lane; p < np; p += 64) M = fmaxf(M, ml[p * 2]);
  M = wave_max(M);
  for (int p = lane; p < np; p += 64) {
    const float m = ml[p * 2];                             // -inf: no visible key, or no score that is a number
    L = fmaf(ml[p * 2 + 1], m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M), L);
  }
  L = wave_sum(L);
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  auto add = [&](const f32x4& x, float m) {
    if (m == -INFINITY) return;                            // a part without a visible key (its output was not written)
    const float f = __builtin_amdgcn_exp2f(m - M);
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[k] = fmaf(x[k], f, acc[k]);
  };
#pragma unroll
  for (int u = 0; u < U; ++u) add(v[u], mv[u]);
  if (on)
    for (int p = j + S * U; p < np; p += S) add(po[(size_t)p * W], ml[p * 2]);
  sum[threadIdx.x] = acc;
  __syncthreads();
  if (j > 0) return;
  for (int g = 1; g < S; ++g) acc += sum[g * W + c];
  float w;
  const float f = tok_finish(a, row, head, M, L, w);
#pragma unroll
  for (int k = 0; k < 4; ++k) acc[k] *= w * f;
  tok_store4(a, row, head, 4 * c, acc);
}

// The same and, in the same launch, the merged heads out of latent space (head_proj_kernel, small_proj.hip, K -> N by w [H][K][N]):
// out[row][h][n] = sum_k bf16(merged[h][k]) w[h][k][n], every bit that of the two launches.  Of a handful of rows both are a launch
// and one trip to memory; here the parts, their maxima and the weights are on their way together.  A workgroup has 64 columns of
// one head and TR rows, which it merges itself: a thread four entries of a row, all parts of them at once.  K = TR's threads x 4.
// us with the attention in front, both launches / this, 16 heads 256 -> 128, at 2, 5, 9, 16 parts:  1 row 13.5 / 10.8, 13.6 / 10.9,
// 13.5 / 10.8, 14.0 / 11.5;  7 rows 16.1 / 12.1, 16.2 / 12.6, 16.3 / 12.9, 17.0 / 14.1;  16 rows 16.1 / 12.3, 16.4 / 13.3, 17.6 / 14.2,
// 19.5 / 16.7;  64 rows 18.6 / 14.7, 26.0 / 22.9, 32.3 / 29.7, 40.8 / 38.8.
template <int TR, int NP, int K>
__global__ void __launch_bounds__(256) token_merge_proj_kernel(TokOut a, const int* __restrict__ items, int n_items,
                                                               const uint16_t* __restrict__ w, int N) {
  constexpr int W = K / 4, S = 256 / W, KG = K / 8;        // S: groups of parts, as in token_merge_kernel
  static_assert(TR * W <= 256 && TR <= 4 && NP <= 64);
  __shared__ float xs[K > 512 ? K * TR : 512 * TR], fac[TR][NP], fin[TR];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, n0 = blockIdx.x * 64, h = blockIdx.y, t0 = blockIdx.z * TR;
  const int nt = min(TR, n_items - t0), np = a.n_parts, c = 2 * (tid & 31), kg = tid >> 5;
  const int t = tid / W, c4 = tid % W;
  const size_t p0 = ((size_t)(t0 + min(t, nt - 1)) * a.H + h) * np;
  const f32x4* po = reinterpret_cast<const f32x4*>(a.po + p0 * K) + c4;
  f32x4 v[NP];
  if (t < nt) {
#pragma unroll
    for (int p = 0; p < NP; ++p) v[p] = po[(size_t)(p < np ? p : 0) * W];
  }
  float m = -INFINITY, l = 0.f;
  if (wv < nt && lane < np) {
    const float* ml = a.pml + (((size_t)(t0 + wv) * a.H + h) * np + lane) * 2;
    m = ml[0], l = ml[1];
  }
  const uint16_t* wp = w + ((size_t)h * K + (size_t)kg * KG) * N + n0 + c;
  uint32_t wq[KG];
#pragma unroll
  for (int u = 0; u < KG; ++u) wq[u] = *reinterpret_cast<const uint32_t*>(wp + (size_t)u * N);
  if (wv < nt) {                                           // wave -> row: the parts' factors
    const float M = wave_max(m), f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
    const float L = wave_sum(fmaf(l, f, 0.f));
    if (lane < NP) fac[wv][lane] = m == -INFINITY ? -1.f : f;        // -1: no visible key, its output was not written
    if (lane == 0) {
      float wf;
      const float g = tok_finish(a, items[(t0 + wv) * 4 + 1], h, M, L, wf);
      fin[wv] = wf * g;
    }
  }
  __syncthreads();
  if (t < TR) {
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
    if (t < nt) {
#pragma unroll
      for (int g = 0; g < S; ++g) {
        f32x4 one = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = g; p < NP; p += S) {
          const float f = fac[t][p];
          if (p < np && f != -1.f) {
#pragma unroll
            for (int k = 0; k < 4; ++k) one[k] = fmaf(v[p][k], f, one[k]);
          }
        }
        if (g == 0)
          acc = one;
        else
          acc += one;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[k] = bf2f(f2bf(acc[k] * fin[t]));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) xs[(4 * c4 + k) * TR + t] = acc[k];
  }
  __syncthreads();
  float acc[TR][2] = {};
#pragma unroll
  for (int u = 0; u < KG; ++u) {
    const float w0 = bf2f((uint16_t)wq[u]), w1 = bf2f((uint16_t)(wq[u] >> 16));
    const float* x = xs + (kg * KG + u) * TR;
#pragma unroll
    for (int i = 0; i < TR; ++i) {
      acc[i][0] = fmaf(x[i], w0, acc[i][0]);
      acc[i][1] = fmaf(x[i], w1, acc[i][1]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TR; ++i) {
    xs[(kg * TR + i) * 64 + c] = acc[i][0];
    xs[(kg * TR + i) * 64 + c + 1] = acc[i][1];
  }
  __syncthreads();
  for (int e = tid; e < nt * 64; e += 256) {
    float r = 0.f;
#pragma unroll
    for (int g = 0; g < 8; ++g) r += xs[g * TR * 64 + e];
    a.out[(size_t)items[(t0 + e / 64) * 4 + 1] * a.ost + (size_t)h * a.osh + n0 + e % 64] = f2bf(r);
  }
}

template <int K>
static int launch_merge_proj(const TokOut& a, const int* items, int rows, const uint16_t* w, int N, hipStream_t s) {
#define K8S_MP(TR, NP)                                                                                                        \
  {                                                                                                                           \
    hipLaunchKernelGGL((token_merge_proj_kernel<TR, NP, K>), dim3(N / 64, a.H, (rows + TR - 1) / TR), dim3(256), 0, s, a, items, rows, \
                       w, N);                                                                                                 \
    return (int)hipGetLastError();                                                                                            \
  }
  if (rows == 1) {
    if (a.n_parts <= 4) K8S_MP(1, 4)
    if (a.n_parts <= 9) K8S_MP(1, 9)
    K8S_MP(1, 16)
  }
  if (a.n_parts <= 4) K8S_MP(4, 4)
  if (a.n_parts <= 9) K8S_MP(4, 9)
  K8S_MP(4, 16)
#undef K8S_MP
}

__device__ __forceinline__ bf16x8 tld16(const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }

// TURN: keys and values are loaded with lane 4 r + h at piece h of row r, so that four lanes beside each other read 64 bytes of
// a line; the fragment wants them in lane 16 h + r (from: 4 (4 r + h), the byte address of the lane that has this lane's).
// Loaded where the fragment wants them, four neighbours read four rows and each is a lookup of its own in the first-level
// cache.  That counts where a compute unit has one or two workgroups, each a chain of such loads; where others run meanwhile
// the exchanges through LDS cost more than the lookups.  us with the merge, as fragments / turned, in a replayed chain:
// masked, 16 heads over 2 of 128, 7 rows at 1000 keys 11.2 / 9.6, 64 at 2000 35 / 35; 16 over 16 of 64, 16 rows at 200 (256
// workgroups) 6.3 / 6.0, 32 at 200 (512) 8.1 / 7.3, 16 at 512 (768) 13.0 / 13.9, 64 at 512 30 / 34; 8 over 8 of 64 + 128 7.4 / 7.7
// and of 128 + 128 8.2 / 8.4 at 4 and 7 rows.  Latent, 16 heads of 256 + 64, 7 rows at 1000 12.3 / 10.8, 32 at 512 (160) 13.9 /
// 12.4, 16 at 2000 (256) 13.6 / 13.9, 64 at 512 (320) 18.6 / 19.3; of 512 + 64 18.3 / 15.4, 39 / 41 at 64 rows; of 64 + 32
// 7.5 / 7.7.
template <bool TURN>
__device__ __forceinline__ bf16x8 tok_turn(bf16x8 v, int from) {
  if constexpr (TURN) {
    int w[4];
    __builtin_memcpy(w, &v, 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = __builtin_amdgcn_ds_bpermute(from, w[i]);
    __builtin_memcpy(&v, w, 16);
  }
  return v;
}

constexpr int kTurnMasked = 512, kTurnLatent = 255, kTurnLong = 192;      // workgroups up to which it pays (kTurnLong: R > 256)

// Scores p[8] (log2 units, keys 8 h .. 8 h + 7 of head lane & 15; -inf: not seen) -> the running maximum and sum, the
// weights as the value product's operand; the output is rescaled only where a head's maximum moved.
template <int ND>
__device__ __forceinline__ void tok_softmax(const float (&p)[8], int hq, float& m, float& l, f32x4 (&o)[ND], bf16x8& pf) {
  float cmax = p[0];
#pragma unroll
  for (int j = 1; j < 8; ++j) cmax = fmaxf(cmax, p[j]);
  cmax = fmaxf(cmax, __shfl_xor(cmax, 16, 64));
  cmax = fmaxf(cmax, __shfl_xor(cmax, 32, 64));
  const bool grow = cmax > m;
  const float mn = grow ? cmax : m, ms = mn == -INFINITY ? 0.f : mn;
  float ps = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float e = __builtin_amdgcn_exp2f(p[j] - ms);
    ps += e;
    pf[j] = (__bf16)e;
  }
  if (__any(grow)) {
    const float alpha = __builtin_amdgcn_exp2f(m - ms);
    l *= alpha;
    m = mn;
    float ai[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ai[i] = __shfl(alpha, 4 * hq + i, 64);
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[dt][i] *= ai[i];
  }
  l += ps;
}

// The rows as their projection left them (fp32 planes: q | k | v), for the form that prepares them itself.
struct TokPrep {
  const float* x;         // [planes][T][qs], planes pstep apart
  const float* bias;      // [(H + G) D + G V] or null
  const float* q_w;       // [D] or null: the norm's weights
  const float* k_w;
  const float* cs;        // [T][rot]: cos | sin
  const float* v_other;   // [T][G V] or null: v = (1 - lam) v + lam v_other
  float* v_keep;          // [T][G V] or null: v as projected
  const int* slots;
  uint16_t* vc;           // [pages][BS][G V] or null
  size_t pstep;
  int qs, planes, rot, norm;
  float eps, lam;
};

// LDS written before is there for the whole workgroup; leaves loads from memory in flight
__device__ __forceinline__ void step_barrier_lds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// What a thread prepares of a row: asked for first, used once the keys are on their way (more than four planes: added as they
// come).  The arithmetic of attn_prep_half_kernel and write_values (masked_attn.hip).
struct TokRow {
  static constexpr int NP = 4;
  f32x4 a[NP], b[NP], wa, wb, ba, bb, co, si;
  __device__ __forceinline__ static f32x4 any4(const float* p) {      // of any alignment
    f32x4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
  }
  __device__ __forceinline__ static void ask(const TokPrep& p, const float* x, f32x4 (&v)[NP]) {
    if (p.planes <= NP) {
#pragma unroll
      for (int k = 0; k < NP; ++k) v[k] = *reinterpret_cast<const f32x4*>(x + min(k, p.planes - 1) * p.pstep);
    } else {
      v[0] = sum_planes4(x, p.pstep, p.planes);
    }
  }
  __device__ __forceinline__ static f32x4 sum(const TokPrep& p, const f32x4 (&v)[NP]) {
    f32x4 t = v[0];
#pragma unroll
    for (int k = 1; k < NP; ++k)
      if (k < p.planes && p.planes <= NP) t += v[k];
    return t;
  }
  __device__ __forceinline__ void ask_head(const TokPrep& p, int row, int c0, int ia, int ib, bool turn, const float* w,
                                           int half) {
    const float* x = p.x + (size_t)row * p.qs + c0;
    ask(p, x + ia, a);
    ask(p, x + ib, b);
    wa = wb = f32x4{1.f, 1.f, 1.f, 1.f};
    ba = bb = co = si = f32x4{0.f, 0.f, 0.f, 0.f};
    if (w) wa = any4(w + ia), wb = any4(w + ib);
    if (p.bias) ba = any4(p.bias + c0 + ia), bb = any4(p.bias + c0 + ib);
    if (turn) {
      const float* c = p.cs + (size_t)row * p.rot + ia;
      co = *reinterpret_cast<const f32x4*>(c), si = *reinterpret_cast<const f32x4*>(c + half);
    }
  }
  __device__ __forceinline__ void ask_value(const TokPrep& p, int row, int c0, size_t vo) {
    ask(p, p.x + (size_t)row * p.qs + c0, a);
    ba = wa = f32x4{0.f, 0.f, 0.f, 0.f};
    if (p.bias) ba = any4(p.bias + c0);
    if (p.v_other) wa = *reinterpret_cast<const f32x4*>(p.v_other + vo);
  }
  template <int LPH>
  __device__ __forceinline__ void head(const TokPrep& p, int D, bool turn, u16x4& ha, u16x4& hb) const {
    f32x4 va = sum(p, a), vb = sum(p, b);
    if (p.bias) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        va[k] += ba[k];
        vb[k] += bb[k];
      }
    }
    if (turn) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float ua = va[k], ub = vb[k];
        va[k] = ua * co[k] - ub * si[k];
        vb[k] = ub * co[k] + ua * si[k];
      }
    }
    float rn = 1.f;
    if (p.norm) {
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k) ss = fmaf(va[k], va[k], fmaf(vb[k], vb[k], ss));
#pragma unroll
      for (int o = 1; o < LPH; o <<= 1) ss += __shfl_xor(ss, o, 64);
      rn = 1.f / sqrtf(ss / (float)D + p.eps);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      ha[k] = f2bf(va[k] * (rn * wa[k]));
      hb[k] = f2bf(vb[k] * (rn * wb[k]));
    }
  }
  __device__ __forceinline__ u16x4 value(const TokPrep& p, size_t vo, bool store) const {
    f32x4 v = sum(p, a);
    if (p.bias) v += ba;
    if (p.v_keep && store) *reinterpret_cast<f32x4*>(p.v_keep + vo) = v;
    u16x4 h;
#pragma unroll
    for (int k = 0; k < 4; ++k) h[k] = f2bf(p.v_other ? mix_value(p.lam, v[k], wa[k]) : v[k]);
    return h;
  }
};

struct MaskTokArgs {
  const uint16_t* q;      // [T][H * D] (H: heads x maps)
  uint16_t* kc;           // [pages][BS][G * maps * D]  (written by the form that prepares)
  uint16_t* vt;           // [pages][G * V][BS]
  const int* bt;
  int maxb;
  const int* items;       // [rows][4]: segment, row, 1, position
  int G, BS, chunk, window, keep_first, part_blocks, most;   // a part: part_blocks, or more where most parts are too few
  float scale, softcap;
  TokOut t;
  TokPrep p;
};

// grid (rows, key heads (x maps) x groups of 16 of their heads, parts); a part is a run of the row's list of 32-key blocks
// (kept first tokens, then the window's or chunk's).
//
// PREP (steps in which every sequence has one row): the pass between the projection and the attention (attn_prep_half_kernel,
// masked_attn.hip: planes, bias, rotation, norm, the caches' rows) is made here, where it was a launch of 4 us with a handful
// of workgroups.  Every workgroup prepares its own heads' queries; the one whose part ends with the row's position also its
// key and value, which it writes to the pages and puts into the fragments of its last block itself.  The row is asked for in
// front of the pages and keys, which are on their way while it is prepared.  The arithmetic, and every bit, is the pass's.
//
// ONE: no wave has more than one block (a part has at most as many blocks as there are waves, and no row more parts than the
// launch: n_parts < most).  One block's registers instead of two's (104 for 250) let a second workgroup onto the compute unit,
// which otherwise waits out each one's chain.  us before / this, with the preparation and the merge, 16 heads over 2 of 128:
// 1 row at 100 keys 7.0 / 6.7, 64 at 512 15.8 / 15.7, 64 at 1500 32.5 / 27.5, 200 at 900 62.7 / 49.0;  32 over 8 of 128, 7 at
// 1500 23.0 / 19.3, 64 at 512 45.3 / 36.7;  12 over 3 of 64 + 128, 64 at 512 20.6 / 17.4.
//
// MEM: workgroups behind the attention's (grid z from n_parts on, two heads each) take the matrix memory of the same rows
// (state_step.h), which a layer has beside it: neither waits for the other, and each alone leaves most of the chip idle.
// us of both launches / of this, 16 heads over 2 of 128 beside 16 of 64 x 128: 1 row at 100 keys 11.1 / 7.1, 5 at 1100 15.9 / 11.8, 64
// at 450 34.7 / 31.5.
struct NoMemory {
  struct Args {};
  static constexpr bool on = false;
  struct Lds {};
};
template <int LV, int DR>
struct WithMemory {
  using Args = StepArgs;
  static constexpr bool on = true;
  using Lds = StepLds<1, LV, DR, false>;
  static __device__ __forceinline__ void run(const StepArgs& m, int z, Lds (&lds)[2]) {
    const int h0 = 2 * (z * gridDim.y + blockIdx.y), half = threadIdx.x >> 8, h = h0 + half;
    if (h0 >= m.H) return;                                 // (the whole workgroup)
    state_step_head<1, LV, DR, float, uint16_t, float, false>(m, blockIdx.x, min(h, m.H - 1), 0, 1, threadIdx.x & 255, h < m.H,
                                                              lds[half]);
  }
};

template <int NDC, int NV, bool CAP, int NW, bool TURN, bool PREP, bool ONE, typename MEM = NoMemory>
__global__ void __launch_bounds__(64 * NW, ONE ? 4 : 1) masked_attn_token_kernel(MaskTokArgs a, typename MEM::Args m2) {
  constexpr int D = NDC * 32, V = NV * 16;
  __shared__ TokLds<NW, V> lds;
  __shared__ __attribute__((aligned(16))) uint16_t qs[PREP ? 16 * D : 8], ks[PREP ? D : 8], vs[PREP ? V : 8];
  if constexpr (MEM::on) {
    static_assert(NW == 8 && 2 * sizeof(typename MEM::Lds) <= sizeof(lds), "two heads in the attention's LDS");
    if ((int)blockIdx.z >= a.t.n_parts)
      return MEM::run(m2, blockIdx.z - a.t.n_parts, reinterpret_cast<typename MEM::Lds(&)[2]>(lds));
  }
  const int lane = threadIdx.x & 63, r = lane & 15, hq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sg = a.items[blockIdx.x * 4], row = a.items[blockIdx.x * 4 + 1], pos = a.items[blockIdx.x * 4 + 3];
  const int H = a.t.H, M = a.t.hs, hpg = H / (a.G * M), nhc = (hpg + 15) / 16, g = blockIdx.y / nhc, hc = blockIdx.y % nhc;
  const int gv = g / M, head0 = (gv * hpg + 16 * hc) * M + g % M, nh = min(16, hpg - 16 * hc), NK = a.G * M * D,
            NVt = a.G * V;
  const int keep = a.window > 0 ? a.keep_first : 0;
  const KeyRuns k0 = key_runs(pos, a.chunk, a.window, a.keep_first);
  const int lo_al = k0.lo & ~31, a_beg = k0.a0 & ~31;
  const int a_end = a.window > 0 ? min(lo_al, (a.keep_first + 31) & ~31) : a_beg;
  const int nblkA = max(0, (a_end - a_beg) >> 5), nblk = nblkA + ((pos - lo_al) >> 5) + 1;
  const int pb = max(a.part_blocks, (nblk + a.most - 1) / a.most), b_lo = (int)blockIdx.z * pb;
  const int nb = min(nblk, b_lo + pb) - b_lo;
  if (nb <= 0) {                                           // the whole workgroup (parts of a longer row's step)
    tok_empty(a.t, head0, nh, blockIdx.z);
    return;
  }
  // ---- the row as projected: D / 8 neighbouring threads a head of q or k, four entries of v a thread
  constexpr int LPH = D / 8;
  const int tid = threadIdx.x, kt = nh * LPH, vt0 = kt + LPH;        // the first threads of k and of v
  const bool ends = PREP && b_lo + nb == nblk, heads = PREP && tid < (ends ? vt0 : kt);
  const bool vals = ends && tid >= vt0 && tid < vt0 + V / 4;
  const int j = tid % LPH, half = PREP ? a.p.rot >> 1 : 0, sl = ends ? a.p.slots[row] : -1;
  const bool isk = tid >= kt, turn = PREP && 8 * j < a.p.rot;
  const int pa = turn ? 4 * j : 8 * j, pb2 = turn ? pa + half : pa + 4;
  const int c0 = isk ? (H + g) * D : (head0 + tid / LPH) * D, vc0 = (H + a.G) * D + gv * V + 4 * (tid - vt0);
  TokRow tr;
  if constexpr (PREP) {
    if (heads)
      tr.ask_head(a.p, row, c0, pa, pb2, turn, isk ? a.p.k_w : a.p.q_w, half);
    else if (vals)
      tr.ask_value(a.p, row, vc0, (size_t)row * NVt + gv * V + 4 * (tid - vt0));
  }
  bf16x8 qf[NDC];
  if constexpr (!PREP) {
    const uint16_t* qp = a.q + (size_t)row * H * D + (size_t)(head0 + min(r, nh - 1) * M) * D;
#pragma unroll
    for (int cc = 0; cc < NDC; ++cc) qf[cc] = tld16(qp + 32 * cc + 8 * hq);
  }
  float m = -INFINITY, l = 0.f;
  f32x4 o[NV];
#pragma unroll
  for (int dt = 0; dt < NV; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float sc2 = a.scale * kTokLog2e, cap2 = a.softcap * kTokLog2e, icap = a.softcap > 0.f ? a.scale / a.softcap : 0.f;
  const int* pages = a.bt + (size_t)sg * a.maxb;
  const int my = (nb - wv + NW - 1) / NW;                  // this wave's blocks (<= 0: none)
  // lane i holds the first key, the page and the place in it of the wave's block base + i
  int base = 0, kbv = 0, pgv = 0, ofv = 0;
  auto fill = [&](int k) {
    base = k;
    const int bi = b_lo + wv + NW * (k + lane);
    kbv = bi < nblkA ? a_beg + 32 * bi : lo_al + 32 * (bi - nblkA);
    const int pi = kbv / a.BS;
    ofv = kbv - pi * a.BS;
    pgv = k + lane < my ? pages[pi] : 0;
  };
  fill(0);
  const int lr = TURN ? lane >> 2 : r, lh = TURN ? lane & 3 : hq, from = 4 * (4 * r + hq);
  constexpr int U = ONE ? 1 : 2;      // blocks of a wave in flight
  bf16x8 kf[U][2][NDC], vf[U][NV];
  int kb[U], page = 0, off = 0;
  auto load_k = [&](int u, int k) {
    if (!ONE && k - base == 64) fill(k);
    kb[u] = __shfl(kbv, k - base, 64);
    page = __shfl(pgv, k - base, 64), off = __shfl(ofv, k - base, 64);
    const uint16_t* kp = a.kc + ((size_t)page * a.BS + off) * NK + g * D + 8 * lh;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int cc = 0; cc < NDC; ++cc) kf[u][t][cc] = tld16(kp + (size_t)(8 * (lr >> 2) + 4 * t + (lr & 3)) * NK + 32 * cc);
  };
  auto load_v = [&](int u) {
    const uint16_t* vp = a.vt + ((size_t)page * NVt + (size_t)gv * V) * a.BS + off + 8 * lh;
#pragma unroll
    for (int dt = 0; dt < NV; ++dt) vf[u][dt] = tld16(vp + (size_t)(16 * dt + lr) * a.BS);
  };
  auto load = [&](int u, int k) {
    load_k(u, k);
    load_v(u);
  };
  if constexpr (ONE) {
    if (my > 0) load_k(0, 0);
    if (!PREP && my > 0) load_v(0);
  } else {
    if (my > 0) load(0, 0);
    if (my > 1) load(1, 1);
  }
  if constexpr (PREP) {
    if (heads) {
      u16x4 ha, hb;
      tr.head<LPH>(a.p, D, turn, ha, hb);
      uint16_t* to = isk ? ks : qs + (tid / LPH) * D;
      *reinterpret_cast<u16x4*>(to + pa) = ha;
      *reinterpret_cast<u16x4*>(to + pb2) = hb;
      if (isk && sl >= 0 && hc == 0) {
        uint16_t* kp = a.kc + (size_t)sl * NK + g * D;
        *reinterpret_cast<u16x4*>(kp + pa) = ha;
        *reinterpret_cast<u16x4*>(kp + pb2) = hb;
      }
    } else if (vals) {
      const int c = gv * V + 4 * (tid - vt0);
      const u16x4 v = tr.value(a.p, (size_t)row * NVt + c, hc == 0);
      *reinterpret_cast<u16x4*>(vs + 4 * (tid - vt0)) = v;
      if (sl >= 0 && hc == 0) {
        uint16_t* vp = a.vt + ((size_t)(sl / a.BS) * NVt + c) * a.BS + sl % a.BS;
#pragma unroll
        for (int k = 0; k < 4; ++k) vp[(size_t)k * a.BS] = v[k];
        if (a.p.vc) *reinterpret_cast<u16x4*>(a.p.vc + (size_t)sl * NVt + c) = v;
      }
    }
    if (ONE && my > 0) load_v(0);
    step_barrier_lds();
#pragma unroll
    for (int cc = 0; cc < NDC; ++cc) qf[cc] = *reinterpret_cast<const bf16x8*>(qs + min(r, nh - 1) * D + 32 * cc + 8 * hq);
  }
  // the row's own key and value into the fragments of the block that holds its position
  auto own = [&](int u) {
    if (!PREP || sl < 0 || kb[u] + 32 <= pos) return;
    const int at = pos - kb[u];
#pragma unroll
    for (int t = 0; t < 2; ++t)
      if (8 * (lr >> 2) + 4 * t + (lr & 3) == at) {
#pragma unroll
        for (int cc = 0; cc < NDC; ++cc) kf[u][t][cc] = *reinterpret_cast<const bf16x8*>(ks + 32 * cc + 8 * lh);
      }
    if (lh == at >> 3) {
#pragma unroll
      for (int dt = 0; dt < NV; ++dt) {
        const __bf16 v = __builtin_bit_cast(__bf16, vs[16 * dt + lr]);
#pragma unroll
        for (int i = 0; i < 8; ++i) vf[u][dt][i] = i == (at & 7) ? v : vf[u][dt][i];
      }
    }
  };
  const int cq_lo = a.chunk > 0 ? (pos / a.chunk) * a.chunk : 0, wq_lo = a.window > 0 ? pos - a.window + 1 : 0;
  for (int k = 0; k < my; k += ONE ? my : 2) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k + u >= my) break;
      own(u);
      float p[8];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int cc = 0; cc < NDC; ++cc)
          s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tok_turn<TURN>(kf[u][t][cc], from), qf[cc], s, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) p[4 * t + i] = s[i];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = kb[u] + 8 * hq + j;
        if (CAP) {                                         // cap tanh(x), tanh(x) = 1 - 2 / (1 + e^(2x)), in log2 units
          const float e = __builtin_amdgcn_exp2f(fminf(p[j] * icap * (2.f * kTokLog2e), 60.f));
          p[j] = cap2 * (1.f - 2.f * __builtin_amdgcn_rcpf(1.f + e));
        } else {
          p[j] *= sc2;
        }
        p[j] = key <= pos && key >= cq_lo && (key >= wq_lo || key < keep) ? p[j] : -INFINITY;
      }
      bf16x8 pf;
      tok_softmax<NV>(p, hq, m, l, o, pf);
#pragma unroll
      for (int dt = 0; dt < NV; ++dt)
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf, tok_turn<TURN>(vf[u][dt], from), o[dt], 0, 0, 0);
      if (!ONE && k + u + 2 < my) load(u, k + u + 2);
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  tok_join<NW, NV>(lds, a.t, row, head0, nh, blockIdx.z, m, l, o);
}

struct LatTokArgs {
  const uint16_t* qa;     // element (row, h, c) at row * qst + h * qsh + c
  long qst, qsh;
  const uint16_t* qr;     // [T][H][32 NP]
  const uint16_t* c;      // [pages][BS][R + 32 NP]
  const uint16_t* ct;     // [pages][R][BS]
  const int* bt;
  int maxb;
  const int* items;       // [rows][4]: segment, row, 1, position
  int BS, window, part, most;   // a part: `part` keys, or more where most parts are too few
  float scale_log2;
  TokOut t;
};

// grid (rows, parts, groups of 16 heads); parts are ranges of the key index (a row's first one is that of its first
// visible key).  ONE as above, for R from 192 on: R 256 + 64, 16 heads, 1 row at 20 keys 5.9 / 5.5 us, 64 rows at 512 14.9 /
// 15.2, at 1500 35.3 / 31.4, 200 at 900 67.9 / 57.0;  R 512 + 64 1 row at 100 12.3 / 11.3, 64 at 512 24.9 / 24.2;  below, where
// the registers let several workgroups on anyway, R 128 + 32 7 rows at 700 9.2 / 9.6.  (All values asked for in front of the
// scores: 7 rows at 700 11.2 / 11.4.)
template <int NR, int NP, int NW, bool TURN, bool ONE>
__global__ void __launch_bounds__(64 * NW, ONE ? 2 : 1) latent_attn_token_kernel(LatTokArgs a) {
  constexpr int R = NR * 32, ND = R / 16, NC = NR + NP, RW = R + 32 * NP, NH = ND / 2;
  __shared__ TokLds<NW, R> lds;
  const int lane = threadIdx.x & 63, r = lane & 15, hq = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sg = a.items[blockIdx.x * 4], row = a.items[blockIdx.x * 4 + 1], pos = a.items[blockIdx.x * 4 + 3];
  const int H = a.t.H, head0 = 16 * blockIdx.z, nh = min(16, H - head0);
  const int lo = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  const int first = lo / a.part * a.part, part = max(a.part, ((pos + a.most - first) / a.most + 31) & ~31);
  const int p0 = first + (int)blockIdx.y * part, k_begin = max(lo, p0), k_end = min(pos + 1, p0 + part);
  if (k_begin >= k_end) {                                  // the whole workgroup
    tok_empty(a.t, head0, nh, blockIdx.y);
    return;
  }
  const int kb0 = k_begin & ~31, nb = (k_end - kb0 + 31) >> 5;
  bf16x8 qf[NC];
  const size_t hl = head0 + min(r, nh - 1);
#pragma unroll
  for (int cc = 0; cc < NC; ++cc)
    qf[cc] = tld16(cc < NR ? a.qa + row * a.qst + hl * a.qsh + 32 * cc + 8 * hq
                           : a.qr + ((size_t)row * H + hl) * (32 * NP) + 32 * (cc - NR) + 8 * hq);
  float m = -INFINITY, l = 0.f;
  f32x4 o[ND];
#pragma unroll
  for (int dt = 0; dt < ND; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int* pages = a.bt + (size_t)sg * a.maxb;
  const int lr = TURN ? lane >> 2 : r, lh = TURN ? lane & 3 : hq, from = 4 * (4 * r + hq);
  for (int b = wv; b < nb; b += ONE ? nb : NW) {
    const int kb = kb0 + 32 * b, page = pages[kb / a.BS], off = kb % a.BS;
    const uint16_t* cp = a.c + (size_t)page * a.BS * RW;
    const uint16_t* tp = a.ct + (size_t)page * R * a.BS + (size_t)lr * a.BS + off + 8 * lh;
    bf16x8 kf[2][NC], vf[ND];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int cc = 0; cc < NC; ++cc)
        kf[t][cc] = tld16(cp + (size_t)(off + 8 * (lr >> 2) + 4 * t + (lr & 3)) * RW + 32 * cc + 8 * lh);
#pragma unroll
    for (int dt = 0; dt < NH; ++dt) vf[dt] = tld16(tp + (size_t)(16 * dt) * a.BS);
    float p[8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int cc = 0; cc < NC; ++cc)
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tok_turn<TURN>(kf[t][cc], from), qf[cc], s, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kb + 8 * hq + 4 * t + i;
        p[4 * t + i] = key < k_end && key >= k_begin ? s[i] * a.scale_log2 : -INFINITY;
      }
    }
    // the second half of the values takes the registers the keys leave
#pragma unroll
    for (int dt = NH; dt < ND; ++dt) vf[dt] = tld16(tp + (size_t)(16 * dt) * a.BS);
    bf16x8 pf;
    tok_softmax<ND>(p, hq, m, l, o, pf);
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf, tok_turn<TURN>(vf[dt], from), o[dt], 0, 0, 0);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  tok_join<NW, ND>(lds, a.t, row, head0, nh, blockIdx.y, m, l, o);
}

template <int NDC, int NV, int NW, bool PREP, bool ONE>
static int launch_mask_tok_nw(const MaskTokArgs& a, int rows, hipStream_t s) {
  const int hpg = a.t.H / (a.G * a.t.hs);
  const dim3 grid(rows, a.G * a.t.hs * ((hpg + 15) / 16), a.t.n_parts);
  auto k = a.softcap > 0.f ? masked_attn_token_kernel<NDC, NV, true, NW, false, PREP, ONE>
                           : masked_attn_token_kernel<NDC, NV, false, NW, false, PREP, ONE>;
  if constexpr (NV == 2 * NDC && (NDC == 2 || NW == 8))      // keys as long as values, heads that share keys or are of 64
    if ((long)rows * grid.y * grid.z <= kTurnMasked)
      k = a.softcap > 0.f ? masked_attn_token_kernel<NDC, NV, true, NW, true, PREP, ONE>
                          : masked_attn_token_kernel<NDC, NV, false, NW, true, PREP, ONE>;
  hipLaunchKernelGGL(k, grid, dim3(64 * NW), 0, s, a, NoMemory::Args{});
  if (a.t.n_parts > 1)
    hipLaunchKernelGGL(token_merge_kernel, dim3(rows * a.t.H), dim3(256), 0, s, a.t, a.items, NV * 16);
  return (int)hipGetLastError();
}

// Waves by the sizes of a head and by whether heads share keys, by nothing that changes from step to step (a row's bits):
// eight, so that a part's blocks are on their way together;  four with 64 + 64 numbers a key, whose registers let more
// workgroups onto a compute unit;  two where every head has keys of its own, for its many workgroups.  us at 1 / 64 rows,
// eight waves / this / tiles of 16 tokens:  16 heads over 16 of 128, 1 key 3.8 / 3.8 / 6.6 and 12.9 / 8.0 / 7.3, 200 keys
// 6.6 / 7.5 / 20 and 28 / 24 / 32, 4000 keys 11.1 / 12.2 / 37 and 480 / 399 / 442;  12 over 6 of 64 at 4000 keys 64 rows
// 122 / 78 / 94;  4 over 4 of 64 8.5 / 8.7 / 25 and 75 / 45 / 65.
template <int NDC, int NV, bool PREP>
static int launch_mask_tok_as(const MaskTokArgs& a, int rows, hipStream_t s) {
  if constexpr (NDC == 2 && NV == 4)
    return launch_mask_tok_nw<NDC, NV, 4, PREP, false>(a, rows, s);
  else if (a.t.H == a.G * a.t.hs)
    return launch_mask_tok_nw<NDC, NV, 2, PREP, false>(a, rows, s);
  else
    return a.t.n_parts < a.most && a.part_blocks <= 8 ? launch_mask_tok_nw<NDC, NV, 8, PREP, true>(a, rows, s)
                                                      : launch_mask_tok_nw<NDC, NV, 8, PREP, false>(a, rows, s);
}
template <int NDC, int NV>
static int launch_mask_tok(const MaskTokArgs& a, int rows, hipStream_t s) {
  if constexpr (NDC != 3)
    if (a.p.x) return launch_mask_tok_as<NDC, NV, true>(a, rows, s);
  return launch_mask_tok_as<NDC, NV, false>(a, rows, s);
}

static int mask_tok_any(const MaskTokArgs& a, int D, int V, int rows, hipStream_t s) {
  if (D == 96) return launch_mask_tok<3, 6>(a, rows, s);
  if (D == 64 && V == 64) return launch_mask_tok<2, 4>(a, rows, s);
  if (D == 64 && V == 128) return launch_mask_tok<2, 8>(a, rows, s);
  if (D == 128 && V == 64) return launch_mask_tok<4, 4>(a, rows, s);
  return launch_mask_tok<4, 8>(a, rows, s);
}

template <int NDC, int NV>
static int launch_mask_memory(const MaskTokArgs& a, const StepArgs& m, int MD, int rows, hipStream_t s) {
  const int hpg = a.t.H / a.G, y = a.G * ((hpg + 15) / 16), z = ((m.H + 1) / 2 + y - 1) / y;
  const dim3 grid(rows, y, a.t.n_parts + z);
  const bool turn = NV == 2 * NDC && (long)rows * y * a.t.n_parts <= kTurnMasked;
#define K8S_MM(LV, DR)                                                                                                  \
  if (m.V == 4 * LV && MD == DR * (256 / LV)) {                                                                         \
    using MEM = WithMemory<LV, DR>;                                                                                     \
    hipLaunchKernelGGL((turn ? masked_attn_token_kernel<NDC, NV, false, 8, NV == 2 * NDC, true, true, MEM>              \
                             : masked_attn_token_kernel<NDC, NV, false, 8, false, true, true, MEM>),                    \
                       grid, dim3(512), 0, s, a, m);                                                                    \
    if (a.t.n_parts > 1)                                                                                                \
      hipLaunchKernelGGL(token_merge_kernel, dim3(rows * a.t.H), dim3(256), 0, s, a.t, a.items, NV * 16);               \
    return (int)hipGetLastError();                                                                                      \
  }
  K8S_MM(32, 8)
  K8S_MM(16, 8)
  K8S_MM(16, 4)
#undef K8S_MM
  return (int)hipErrorInvalidValue;
}

template <int NR, int NP>
static void launch_lat_tok_np(const LatTokArgs& a, int rows, hipStream_t s) {
  constexpr int NW = 4;
  const dim3 grid(rows, a.t.n_parts, (a.t.H + 15) / 16);
  auto k = latent_attn_token_kernel<NR, NP, NW, false, false>;
  if constexpr (NR >= 6) {
    const bool one = a.t.n_parts < a.most && a.part <= 32 * NW;
    if ((long)rows * grid.y * grid.z <= (NR > 8 ? kTurnLong : kTurnLatent))
      k = one ? latent_attn_token_kernel<NR, NP, NW, true, true> : latent_attn_token_kernel<NR, NP, NW, true, false>;
    else if (one)
      k = latent_attn_token_kernel<NR, NP, NW, false, true>;
  }
  hipLaunchKernelGGL(k, grid, dim3(64 * NW), 0, s, a);
}

template <int NR>
static int launch_lat_tok(const LatTokArgs& a, int np, int rows, hipStream_t s) {
  switch (np) {
    case 0: launch_lat_tok_np<NR, 0>(a, rows, s); break;
    case 1: launch_lat_tok_np<NR, 1>(a, rows, s); break;
    case 2: launch_lat_tok_np<NR, 2>(a, rows, s); break;
    default: return (int)hipErrorInvalidValue;
  }
  if (a.t.n_parts > 1 && a.t.out)
    hipLaunchKernelGGL(token_merge_kernel, dim3(rows * a.t.H), dim3(256), 0, s, a.t, a.items, NR * 32);
  return (int)hipGetLastError();
}

}  // namespace k8s

using namespace k8s;

K8S_API int k8s_masked_attn_mfma_ok(int H, int G, int D, int V);
K8S_API int k8s_latent_attn_mfma_ok(int R, int RP);

// items [rows][4]; n_parts > 1: po [rows][H][n_parts][V], pml [rows][H][n_parts][2]
K8S_API int k8s_masked_attn_token(const void* q, const void* kc, const void* vt, const int* bt, int maxb,
                                  const int* items, int rows, const float* sink, const float* gate, int gs, void* out,
                                  int H, int G, int D, int V, int BS, int chunk, int window, int keep_first, float scale,
                                  float softcap, hipStream_t s, int part_blocks, int most, int n_parts, float* pml,
                                  float* po, int maps, int out_f32) {
  if (rows <= 0) return 0;
  if (!k8s_masked_attn_mfma_ok(H, G, D, V) || BS % 32 || chunk < 0 || window < 0 || keep_first < 0 || n_parts < 1 ||
      part_blocks < 1 || maps < 1 || most < 1 || n_parts > most || (n_parts > 1 && (!pml || !po)))
    return (int)hipErrorInvalidValue;
  MaskTokArgs a;
  a.q = (const uint16_t*)q; a.kc = (uint16_t*)kc; a.vt = (uint16_t*)vt; a.bt = bt; a.maxb = maxb;
  a.items = items; a.G = G; a.BS = BS; a.chunk = chunk; a.window = window; a.keep_first = keep_first;
  a.part_blocks = part_blocks; a.most = most; a.scale = scale; a.softcap = softcap;
  a.t.sink = sink; a.t.gate = gate; a.t.gs = gs; a.t.out = out_f32 ? nullptr : (uint16_t*)out;
  a.t.out32 = out_f32 ? (float*)out : nullptr; a.t.ost = (long)H * maps * V; a.t.osh = V;
  a.t.po = po; a.t.pml = pml; a.t.H = H * maps; a.t.n_parts = n_parts; a.t.hs = maps;
  a.p = TokPrep{};
  return mask_tok_any(a, D, V, rows, s);
}

// The same on rows as their projection left them, every row the only one of its sequence (TokPrep): what k8s_attn_prep_half
// and k8s_masked_attn_token give.  D 64 or 128, qs and pstep multiples of 4, rot a multiple of 8 with its table, x / kc / cs /
// v_other / v_keep 16-byte aligned; vc may be null.
#define K8S_PREP_PARAMS                                                                                                     \
  const float *x, int qs, int planes, long pstep, const float *bias, const float *q_w, const float *k_w, float eps, int norm,  \
      const float *cs, int rot, float lam, const float *v_other, float *v_keep, const int *slots, void *vc, void *kc, void *vt, \
      const int *bt, int maxb, const int *items, int rows, const float *sink, const float *gate, int gs, void *out, int H,      \
      int G, int D, int V, int BS, int chunk, int window, int keep_first, float scale, float softcap, hipStream_t s,            \
      int part_blocks, int most, int n_parts, float *pml, float *po
#define K8S_PREP_NAMES                                                                                                    \
  x, qs, planes, pstep, bias, q_w, k_w, eps, norm, cs, rot, lam, v_other, v_keep, slots, vc, kc, vt, bt, maxb, items, rows, \
      sink, gate, gs, out, H, G, D, V, BS, chunk, window, keep_first, scale, softcap, s, part_blocks, most, n_parts, pml, po
static bool prep_args(MaskTokArgs& a, K8S_PREP_PARAMS) {
  (void)s;
  auto off = [](const void* p) { return ((uintptr_t)p & 15) != 0; };
  if (!k8s_masked_attn_mfma_ok(H, G, D, V) || D == 96 || BS % 32 || chunk < 0 || window < 0 || keep_first < 0 || n_parts < 1 ||
      part_blocks < 1 || most < 1 || n_parts > most || (n_parts > 1 && (!pml || !po)) || !x || qs % 4 || planes < 1 ||
      (planes > 1 && pstep % 4) || rot < 0 || rot > D || rot % 8 || (rot && !cs) || norm < 0 || norm > 1 || !slots || !kc ||
      !vt || off(x) || off(cs) || off(kc) || off(v_other) || off(v_keep) || ((uintptr_t)vc & 7))
    return false;
  a.q = nullptr; a.kc = (uint16_t*)kc; a.vt = (uint16_t*)vt; a.bt = bt; a.maxb = maxb;
  a.items = items; a.G = G; a.BS = BS; a.chunk = chunk; a.window = window; a.keep_first = keep_first;
  a.part_blocks = part_blocks; a.most = most; a.scale = scale; a.softcap = softcap;
  a.t.sink = sink; a.t.gate = gate; a.t.gs = gs; a.t.out = (uint16_t*)out; a.t.out32 = nullptr;
  a.t.ost = (long)H * V; a.t.osh = V; a.t.po = po; a.t.pml = pml; a.t.H = H; a.t.n_parts = n_parts; a.t.hs = 1;
  a.p = TokPrep{x, bias, q_w, k_w, cs, v_other, v_keep, slots, (uint16_t*)vc, (size_t)pstep, qs, planes, rot, norm, eps, lam};
  return true;
}

K8S_API int k8s_masked_attn_token_prep(K8S_PREP_PARAMS) {
  if (rows <= 0) return 0;
  MaskTokArgs a;
  return prep_args(a, K8S_PREP_NAMES) ? mask_tok_any(a, D, V, rows, s) : (int)hipErrorInvalidValue;
}

// The same and k8s_memory_step of the same rows (its x: `mx`, bf16 out) in one launch.  Heads share keys (H > G), no softcap,
// D and V not both 64, n_parts < most, part_blocks <= 8.
K8S_API int k8s_masked_attn_memory(K8S_PREP_PARAMS, const float* mx, int mxs, const float* gate_bias, float cap, float* state,
                                   float* nstate, float* mstate, const int* pos0, const int* slot, const float* mgate, int mgs,
                                   const float* mw, int mwh, void* mout, int MH, int MD, int MV, float meps, float den_eps) {
  if (rows <= 0) return 0;
  MaskTokArgs a;
  if (!prep_args(a, K8S_PREP_NAMES) || H <= G || softcap > 0.f || n_parts >= most || part_blocks > 8 || MH < 1 || !mx || !state ||
      !nstate || !mstate || !pos0 || !slot || !mgate || !mout)
    return (int)hipErrorInvalidValue;
  const StepArgs m = memory_args(mx, mxs, gate_bias, cap, state, nstate, mstate, pos0, slot, mgate, mgs, mw, mwh, mout, MH, MV, meps,
                                 den_eps);
  if (D == 128 && V == 128) return launch_mask_memory<4, 8>(a, m, MD, rows, s);
  if (D == 64 && V == 128) return launch_mask_memory<2, 8>(a, m, MD, rows, s);
  if (D == 128 && V == 64) return launch_mask_memory<4, 4>(a, m, MD, rows, s);
  return (int)hipErrorInvalidValue;
}

// items [rows][4]; n_parts > 1: po [rows][H][n_parts][R], pml [rows][H][n_parts][2], and without out they are left to
// k8s_latent_merge_proj
K8S_API int k8s_latent_attn_token(const void* qa, long qst, long qsh, const void* qr, int RP, const void* c, const void* ct,
                                  const int* bt, int maxb, const int* items, int rows, const float* gate, int ldg,
                                  const float* sink, void* out, long ost, long osh, float* po, float* pml, int n_parts,
                                  int part, int most, int H, int R, int BS, int window, float scale, hipStream_t s) {
  if (rows <= 0) return 0;
  if (!k8s_latent_attn_mfma_ok(R, RP) || BS % 32 || H <= 0 || n_parts < 1 || n_parts > most || part <= 0 || part % 32 ||
      (RP && !qr) || window < 0 || qst % 8 || qsh % 8 || (n_parts > 1 && (!pml || !po)) || (n_parts == 1 && !out))
    return (int)hipErrorInvalidValue;
  LatTokArgs a;
  a.qa = (const uint16_t*)qa; a.qst = qst; a.qsh = qsh; a.qr = (const uint16_t*)qr; a.c = (const uint16_t*)c;
  a.ct = (const uint16_t*)ct; a.bt = bt; a.maxb = maxb; a.items = items; a.BS = BS; a.window = window; a.part = part;
  a.most = most;
  a.scale_log2 = scale * kTokLog2e;
  a.t.sink = sink; a.t.gate = gate; a.t.gs = ldg; a.t.out = (uint16_t*)out; a.t.out32 = nullptr; a.t.ost = ost;
  a.t.osh = osh; a.t.po = po; a.t.pml = pml; a.t.H = H; a.t.n_parts = n_parts; a.t.hs = 1;
  switch (R / 32) {
    case 1: return launch_lat_tok<1>(a, RP / 32, rows, s);
    case 2: return launch_lat_tok<2>(a, RP / 32, rows, s);
    case 3: return launch_lat_tok<3>(a, RP / 32, rows, s);
    case 4: return launch_lat_tok<4>(a, RP / 32, rows, s);
    case 6: return launch_lat_tok<6>(a, RP / 32, rows, s);
    case 8: return launch_lat_tok<8>(a, RP / 32, rows, s);
    case 12: return launch_lat_tok<12>(a, RP / 32, rows, s);
    case 16: return launch_lat_tok<16>(a, RP / 32, rows, s);
    default: return (int)hipErrorInvalidValue;
  }
}

// out[row][h] = merged[row][h] . w[h] of the parts that k8s_latent_attn_token left (2 to 16 of them): w [H][R][N], R 128 or 256, N a
// multiple of 64; po on 16 bytes, w on 4.
K8S_API int k8s_latent_merge_proj(const float* po, const float* pml, int n_parts, const int* items, int rows, const float* gate, int ldg,
                                  const float* sink, const void* w, void* out, long ost, long osh, int H, int R, int N,
                                  hipStream_t s) {
  if (rows <= 0) return 0;
  if (!po || !pml || !items || !w || !out || n_parts < 2 || n_parts > 16 || H < 1 || (R != 128 && R != 256) || N < 64 || N % 64 ||
      ((uintptr_t)po & 15) || ((uintptr_t)w & 3))
    return (int)hipErrorInvalidValue;
  TokOut t{};
  t.sink = sink; t.gate = gate; t.gs = ldg; t.out = (uint16_t*)out; t.ost = ost; t.osh = osh;
  t.po = const_cast<float*>(po); t.pml = const_cast<float*>(pml); t.H = H; t.n_parts = n_parts; t.hs = 1;
  return R == 128 ? launch_merge_proj<128>(t, items, rows, (const uint16_t*)w, N, s)
                  : launch_merge_proj<256>(t, items, rows, (const uint16_t*)w, N, s);
}
