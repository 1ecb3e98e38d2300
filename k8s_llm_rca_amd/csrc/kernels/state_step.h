// One token per sequence through a matrix state, with what stands around it: the reply steps of the gated delta rule and the
// matrix memory (matrix_mem.hip) and of the decaying linear attention (mixer_ops.hip), same arithmetic, in one launch each
// (state_step.hip) or, of the matrix memory, in further workgroups of the attention beside it (token_attn.hip).
//
// KIND 0, delta rule:  q, k to unit length, decays and beta from their gates,  S <- g S;  u = beta (v - S^T k);
//   S <- S + k u^T;  o = S^T q,  then the head's norm, its weight and the output gate.
// KIND 1, matrix memory:  the exponential gates and their running maximum,  S <- f S + i k v^T, n likewise,
//   o = S^T q / max(|n.q|, e^-m),  then the head's norm, weight and gate.
// KIND 2, decaying attention:  silu of q, k, v,  S <- d S + k v^T;  o = S^T q, times the norm's weight and the output gate.
//   The norm spans all heads, which no workgroup sees: the sum of squares of every head goes to ssp, and
//   whoever adds the output projection to the residual divides by the root mean square (the factor is one per row).
//
// A workgroup has a head of one sequence (V = 4 LV, D = DR RG), or of KIND 2 a slice of its columns; a thread four neighbouring columns of DR rows RG apart, so a
// wave's accesses to the state are whole lines.  Nothing waits for anything but the state's address: rows,
// gates and state are asked for together.  What bounds it: the state's bytes, read and written once (64 KB a head each way):
// where every unit has a head, memory (KIND 2 with a workgroup a head of 128 x 128, 16 sequences of 16 heads: 7.2 us, of which a launch
// takes 2.6);  with fewer, the rate of a unit, 48 to 68 KB a us of both (7 and 1 sequences 5.3 and 4.5 us).  A step reads the model's weights between two visits to a state, so that no cache holds it: it is
// read and written without a place in the second-level cache (non-temporal), which would else have its written lines to give back
// when the kernel ends.  us as ordinary / non-temporal accesses of states no cache holds:  KIND 2, 16 heads of 128 x 128, 1, 7, 16, 32,
// 64 sequences 3.7 / 3.3, 6.1 / 4.7, 9.9 / 6.9, 17.9 / 12.8, 34 / 26 (5.2 TB/s; either alone 33 and 28);  KIND 1, 16 of 64 x 128,
// 1, 5, 16, 32, 64 4.6 / 4.3, 5.1 / 4.7, 6.9 / 5.5, 10.6 / 7.7, 19.3 / 15.1;  KIND 0 5.1 / 4.7, 5.5 / 5.0, 7.1 / 5.8, 10.9 / 7.9, 18.3 /
// 14.4;  8 of 64 x 64 at 64 7.2 / 5.6 and 7.5 / 6.0.
#pragma once
#include "common.h"
#include "gates.h"

namespace k8s {

struct StepArgs {
  const void* x;          // KIND 0: [T] q [G][D] | k [G][D] | v [H][V];  1: q [H][D] | k | v [H][V] | . | i [H] | f [H];  2: q | k | v
  int xs;
  const float* a;         // KIND 0: [T][H D], before bias and softplus
  const float* rate;      // KIND 0: [H];  2: the decays [H]
  const float* bias;      // KIND 0: [H D];  1: [2 H] = (i | f)
  const float* beta;      // KIND 0: rows of stride bs
  int bs;
  float cap;              // KIND 1
  float* state;           // [slots][H][D][V]
  float* nstate;          // [slots][H][D]
  float* mstate;          // [slots][H]
  const int* pos0;
  const int* slot;
  const void* gate;       // rows of stride gs, column h V + c
  int gs;
  const float* w;         // h wh + c, or null
  int wh;
  float eps, unit_eps, den_eps;
  void* out;              // [T][H V]
  float* ssp;             // KIND 2: [T][H][slices]
  int H, G, V;
  const float* lr;        // LOW: rows of stride bs, ra entries for the decays' gates, rg for the output's
  const uint16_t* la;     // LOW: [H D][ra]
  const uint16_t* lg;     // LOW: [H V][rg]
  int ra, rg;
};
constexpr int kLowMax = 128;              // LOW: ra and rg, at most

template <typename T>
__device__ __forceinline__ float ss_ld(const T* p);
template <>
__device__ __forceinline__ float ss_ld<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float ss_ld<uint16_t>(const uint16_t* p) { return bf2f(*p); }
__device__ __forceinline__ f32x4 ss_ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 ss_ld4(const uint16_t* p) {
  const u16x4 v = *reinterpret_cast<const u16x4*>(p);
  return f32x4{bf2f(v[0]), bf2f(v[1]), bf2f(v[2]), bf2f(v[3])};
}
__device__ __forceinline__ void ss_st4(float* p, const f32x4& v) { *reinterpret_cast<f32x4*>(p) = v; }
__device__ __forceinline__ void ss_st4(uint16_t* p, const f32x4& v) {
  *reinterpret_cast<u16x4*>(p) = u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
}
template <typename TA>
__device__ __forceinline__ float ss_silu(float z);
template <>
__device__ __forceinline__ float ss_silu<float>(float z) { return z / (1.f + expf(-z)); }
template <>
__device__ __forceinline__ float ss_silu<uint16_t>(float z) { return bf2f(f2bf(silu_hw(z))); }

// four columns' sums over the row groups of 256 threads: lanes of equal lv within a wave, then the waves in order
template <int LV>
__device__ __forceinline__ f32x4 sum_rows(f32x4 v, f32x4 (*red)[LV], int tid) {
  const int lane = tid & 63;
#pragma unroll
  for (int o = LV; o < 64; o <<= 1)
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] += __shfl_xor(v[k], o, 64);
  if (lane < LV) red[tid >> 6][lane] = v;
  __syncthreads();
  const int lv = tid % LV;
  f32x4 s = red[0][lv];
#pragma unroll
  for (int w = 1; w < 4; ++w) s += red[w][lv];
  return s;
}

// LOW (KIND 0): the two products of low rank in front (low_rank_pair, small_proj.hip) are made here, by every workgroup for its
// own head, where they were a launch: a thread has a quarter of K of a column of each 64, asked for in front of the state
// (16 heads of 64 x 128, ranks of 64, 1 and 5 sequences: 7.4 -> 6.4 us, 8.9 -> 7.5).  The sums are low_rank_pair's, to the bit.
template <int KIND, int LV, int DR, bool LOW>
struct StepLds {
  static constexpr int D = DR * (256 / LV);
  f32x4 red[2][4][LV];
  float sq[D], sk[D], sg[KIND == 0 ? D : 1], sc[3][4];
  float lx[LOW ? 2 * kLowMax : 1], lp[LOW ? 4 : 1][LOW ? D + 4 * LV : 1];
};

// Threads tid of 256 take row it's head hh (its columns from 4 LV z on); all of a workgroup come here, those without a head of
// their own (!on) write nothing.
template <int KIND, int LV, int DR, typename TA, typename TO, typename TG, bool LOW>
__device__ __forceinline__ void state_step_head(const StepArgs& a, int it, int hh, int z, int nz, int tid, bool on,
                                                StepLds<KIND, LV, DR, LOW>& lds) {
  constexpr int RG = 256 / LV, D = DR * RG, CB = (D + 4 * LV) / 64;
  static_assert(!LOW || KIND == 0);
  static_assert(D <= 256, "a thread per entry of q and k");
  auto& lx = lds.lx;
  auto& lp = lds.lp;
  auto& sq = lds.sq;
  auto& sk = lds.sk;
  auto& sg = lds.sg;
  auto& sc = lds.sc;
  auto& red = lds.red;
  const int lv = tid % LV, rg = tid / LV, wv = tid >> 6;
  const int H = a.H, V = a.V, c = 4 * (z * LV + lv);
  const TA* row = (const TA*)a.x + (size_t)it * a.xs;
  const int slot = a.slot[it];
  const bool fresh = a.pos0[it] == 0;
  const int kv = KIND == 0 ? a.G * D : H * D, kh = KIND == 0 ? hh / (H / a.G) : hh;
  float q = 0.f, k = 0.f, n = 0.f, g = 0.f;
  float lxv = 0.f;
  u16x8 lwv[LOW ? CB : 1][kLowMax / 32];
  if constexpr (LOW) {
    if (tid < a.ra + a.rg) lxv = a.lr[(size_t)it * a.bs + tid];
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const bool dec = b < D / 64;
      const int col = 64 * b + (tid & 63), K = dec ? a.ra : a.rg;
      const uint16_t* lw = (dec ? a.la + (size_t)(hh * D + col) * K : a.lg + (size_t)(hh * V + col - D) * K) + wv * (K / 4);
#pragma unroll
      for (int p = 0; p < kLowMax / 32; ++p)
        if (32 * p < K) lwv[b][p] = *reinterpret_cast<const u16x8*>(lw + 8 * p);
    }
  }
  if (tid < D) {
    q = ss_ld(row + kh * D + tid);
    k = ss_ld(row + kv + kh * D + tid);
    if (KIND == 0) g = LOW ? a.bias[hh * D + tid] : a.a[((size_t)it * H + hh) * D + tid] + a.bias[hh * D + tid];
    if (KIND == 1 && !fresh) n = a.nstate[((size_t)slot * H + hh) * D + tid];
  }
  f32x4 v = ss_ld4(row + 2 * kv + hh * V + c);
  float* st = a.state + ((size_t)slot * H + hh) * D * V + c;
  f32x4 S[DR];
#pragma unroll
  for (int i = 0; i < DR; ++i) S[i] = fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : ldw_nt<f32x4>(st + (size_t)(rg + RG * i) * V);
  f32x4 gt = f32x4{0.f, 0.f, 0.f, 0.f}, w = f32x4{1.f, 1.f, 1.f, 1.f};
  if (tid < LV) {
    if (!LOW) gt = ss_ld4((const TG*)a.gate + (size_t)it * a.gs + hh * V + c);
    if (a.w) w = ss_ld4(a.w + hh * a.wh + c);
  }
  if constexpr (LOW) {
    if (tid < a.ra + a.rg) lx[tid] = bf2f(f2bf(lxv));
    __syncthreads();
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const int KG = (b < D / 64 ? a.ra : a.rg) / 4;
      const float* xs = lx + (b < D / 64 ? 0 : a.ra) + wv * KG;
      float s = 0.f;
#pragma unroll
      for (int p = 0; p < kLowMax / 32; ++p)
        if (8 * p < KG) {
#pragma unroll
          for (int j = 0; j < 8; ++j) s = fmaf(xs[8 * p + j], bf2f(lwv[b][p][j]), s);
        }
      lp[wv][64 * b + (tid & 63)] = s;
    }
    __syncthreads();
    if (tid < D) {
      float s = 0.f;
#pragma unroll
      for (int u = 0; u < 4; ++u) s += lp[u][tid];
      g = s + g;
    }
    if (tid < LV) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float s = 0.f;
#pragma unroll
        for (int u = 0; u < 4; ++u) s += lp[u][D + c + j];
        gt[j] = s;
      }
    }
  }
  float fa = 1.f, ia = 1.f, m = 0.f;
  if (KIND == 1) {
    const float m0 = fresh ? 0.f : a.mstate[(size_t)slot * H + hh];
    const TA* gr = row + 2 * kv + 2 * H * V;
    const float gi = a.cap * tanhf((ss_ld(gr + hh) + a.bias[hh]) / a.cap);
    const float gf = logsigmoid_f(a.cap * tanhf((ss_ld(gr + H + hh) + a.bias[H + hh]) / a.cap));
    m = gf + fmaxf(m0, gi - gf);
    fa = expf(gf + m0 - m);
    ia = expf(gi - m);
  } else if (KIND == 2) {
    fa = a.rate[hh];
    q = ss_silu<TA>(q);
    k = ss_silu<TA>(k);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = ss_silu<TA>(v[j]);
  }
  if (tid < D) {
    sq[tid] = q;
    sk[tid] = k;
    if (KIND == 0) sg[tid] = expf(-a.rate[hh] * softplus_f(g));
  }
  if (KIND == 0) {
    const float qq = wave_sum(q * q), kk = wave_sum(k * k);
    if ((tid & 63) == 0) {
      sc[0][wv] = qq;
      sc[1][wv] = kk;
    }
  }
  if (KIND == 1) {
    n = fa * n + k * ia;
    if (on && tid < D) a.nstate[((size_t)slot * H + hh) * D + tid] = n;
    const float nq = wave_sum(n * q);
    if ((tid & 63) == 0) sc[2][wv] = nq;
  }
  __syncthreads();                                         // (mstate has been read by every thread)
  if (KIND == 1 && on && tid == 0) a.mstate[(size_t)slot * H + hh] = m;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  float of = 1.f;                                          // the factor of the read-out
  if (KIND == 0) {
    const float kf = 1.f / sqrtf(sc[1][0] + sc[1][1] + sc[1][2] + sc[1][3] + a.unit_eps);
    of = 1.f / sqrtf((float)D) / sqrtf(sc[0][0] + sc[0][1] + sc[0][2] + sc[0][3] + a.unit_eps);
    f32x4 ks = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < DR; ++i) {
      const float gd = sg[rg + RG * i], kd = sk[rg + RG * i];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        S[i][j] *= gd;
        ks[j] = fmaf(S[i][j], kd, ks[j]);
      }
    }
    ks = sum_rows<LV>(ks, red[0], tid);
    const float beta = sigmoid_f(a.beta[(size_t)it * a.bs + hh]);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = beta * (v[j] - ks[j] * kf) * kf;
  }
#pragma unroll
  for (int i = 0; i < DR; ++i) {
    const float kd = sk[rg + RG * i], qd = sq[rg + RG * i];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (KIND == 0)
        S[i][j] = fmaf(kd, v[j], S[i][j]);
      else
        S[i][j] = fmaf(fa, S[i][j], kd * (KIND == 1 ? ia * v[j] : v[j]));
      acc[j] = fmaf(S[i][j], qd, acc[j]);
    }
    if (on) __builtin_nontemporal_store(S[i], reinterpret_cast<f32x4*>(st + (size_t)(rg + RG * i) * V));
  }
  acc = sum_rows<LV>(acc, red[1], tid);
  if (tid >= 64) return;
  float mu = 1.f;
  if (KIND == 1) {
    const float qs = 1.f / sqrtf((float)D), nq = sc[2][0] + sc[2][1] + sc[2][2] + sc[2][3];
    mu = qs / (fmaxf(fabsf(nq * qs), expf(-m)) + a.den_eps);
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    acc[j] *= of;
    ss = fmaf(acc[j] * mu, acc[j] * mu, ss);
  }
#pragma unroll
  for (int o = 1; o < LV; o <<= 1) ss += __shfl_xor(ss, o, 64);
  if (tid >= LV || !on) return;
  const float rn = KIND == 2 ? 1.f : mu / sqrtf(ss / (float)V + a.eps);
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = acc[j] * rn * w[j] * sigmoid_f(gt[j]);
  ss_st4((TO*)a.out + (size_t)it * H * V + hh * V + c, acc);
  if (KIND == 2 && tid == 0) a.ssp[((size_t)it * H + hh) * nz + z] = ss;
}

// KIND 1
inline StepArgs memory_args(const float* x, int xs, const float* gate_bias, float cap, float* state, float* nstate, float* mstate,
                            const int* pos0, const int* slot, const float* gate, int gs, const float* w, int wh, void* out, int H,
                            int V, float eps, float den_eps) {
  StepArgs p{};
  p.x = x; p.xs = xs; p.bias = gate_bias; p.cap = cap; p.state = state; p.nstate = nstate; p.mstate = mstate; p.pos0 = pos0;
  p.slot = slot; p.gate = gate; p.gs = gs; p.w = w; p.wh = wh; p.eps = eps; p.den_eps = den_eps; p.out = out; p.H = H;
  p.G = H; p.V = V;
  return p;
}

}  // namespace k8s
