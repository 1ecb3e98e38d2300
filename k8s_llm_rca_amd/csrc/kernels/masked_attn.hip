// Softmax attention over a paged key / value cache under a position mask, behind a pass that prepares
// q and k.
//
// attn_prep:  rows of the joint projection (fp32: q [H][D] | k [G][D] | v [NV], row stride qs)
//   + bias;  q, k rotated on their first `rot` entries per head (entry i with i + rot / 2, or with rot_pairs
//   entry 2i with 2i + 1; angle pos * f_i with f_i = base^(-2 i / rot) or from a table of doubles, the product
//   formed in double; cos and sin times rot_amp; rot_cs: the step's table of them, made once for all layers);  norm 1: q, k divided by the head's root mean square (eps inside
//   the root) behind the rotation and multiplied by a weight [D] where given;  norm 2: q and k each divided by
//   the root mean square of the WHOLE projection (all heads at once) and multiplied by a weight of that size,
//   in front of the rotation;  q multiplied by the position's temperature 1 + tq_coef ln(floor((pos + 1) /
//   tq_every) + 1) (tq_every > 0);  v optionally kept as projected (v_keep) and mixed with another layer's
//   values of the same token, (1 - lam) v + lam v_other;  k and v written to their pages (and v to the
//   transposed twin), q written as activations.  The values start at column v_col of the row: behind the
//   keys, or AT the keys (the values are the keys as projected).  G = 0: a layer that reads another layer's
//   pages prepares its queries only.  H and G count heads of D entries: a layer with several score maps per
//   head passes maps * heads.
//
// masked attention:  position i sees j <= i with  (chunk > 0:  i / chunk == j / chunk)  and
//   (window > 0:  i - j < window  or  j < keep_first).  s = scale q.k, then softcap tanh(s / softcap) for
//   softcap > 0.  A sink adds exp(sink_h) to head h's denominator.  Head h's output may be multiplied by
//   sigmoid(gate[t][h]).  Query head h reads key / value head h / (H / G).  With M > 1 score maps per head, q
//   holds H M heads laid out [h][m] and the key pages G M heads [g][m]: map m of head h scores against key
//   head (h / (H / G)) M + m and applies its weights to value head h / (H / G); the output is [T][H][M][V],
//   each map's result by itself (fp32 where the caller joins the maps).
//   The visible keys of a row are two runs, [a0, a1) (kept first tokens) and [lo, pos].  The kernels: rows_attn.hip
//   (vector pipes, any size and type), mask_prompt.hip and token_attn.hip (bf16 on the matrix cores: portions of prompts,
//   single tokens).
//
// Pages: kc [pages][BS][G D], vc [pages][BS][G V], vt [pages][G V][BS]; a token's slot = page * BS + offset.
// Scores, weights and accumulation are fp32; TA (bf16 as uint16_t, or float) is the type of q, the pages
// and the output.
#include "common.h"
#include "rope_rows.h"
#include "key_runs.h"

namespace k8s {

template <typename T>
__device__ __forceinline__ void sta(T* p, size_t i, float v);
template <>
__device__ __forceinline__ void sta<float>(float* p, size_t i, float v) { p[i] = v; }
template <>
__device__ __forceinline__ void sta<uint16_t>(uint16_t* p, size_t i, float v) { p[i] = f2bf(v); }

constexpr int kPrepPer = 8;    // entries of a head per lane: D <= 512

template <typename TA>
__global__ void __launch_bounds__(256) attn_prep_kernel(const float* __restrict__ qkv, int qs,
                                                        const float* __restrict__ bias, int H, int G, int D, int NV,
                                                        const int* __restrict__ positions,
                                                        const int* __restrict__ slots, TA* __restrict__ kc,
                                                        TA* __restrict__ vc, TA* __restrict__ vt, int BS,
                                                        TA* __restrict__ q_out, int norm, const float* __restrict__ q_w,
                                                        const float* __restrict__ k_w, float eps, int rot, float base,
                                                        float lam, const float* __restrict__ v_other,
                                                        float* __restrict__ v_keep, int upr, int v_col, float tq_coef,
                                                        int tq_every, const double* __restrict__ rot_freq,
                                                        float rot_amp, int rot_pairs,
                                                        const float* __restrict__ rot_cs) {
  extern __shared__ float sm[];   // [rot]: cos | sin;  [upr][D]: the heads of one round
  __shared__ float red[16];
  const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int half = rot >> 1;
  float* cs = sm;
  if (rot && rot_cs) {
    for (int i = tid; i < rot; i += 256) cs[i] = rot_cs[(size_t)r * rot + i];
  } else if (rot) {
    const double lb = log((double)base), p = (double)positions[r];
    for (int i = tid; i < half; i += 256) {
      const double ang = p * (rot_freq ? rot_freq[i] : exp(-(double)(2 * i) / (double)rot * lb));
      cs[i] = (float)cos(ang) * rot_amp;
      cs[half + i] = (float)sin(ang) * rot_amp;
    }
  }
  const int sl = slots[r];
  const int NQ = H * D, NK = G * D, units = H + G;
  const float* row = qkv + (size_t)r * qs;
  const float tq = tq_every > 0 ? 1.f + tq_coef * logf((float)((positions[r] + 1) / tq_every) + 1.f) : 1.f;
  // norm 2: 1 / rms of the whole q and of the whole k projection
  float rq = 1.f, rk = 1.f;
  if (norm == 2) {
    float sq = 0.f, sk = 0.f;
    for (int i = tid; i < NQ; i += 256) {
      const float v = row[i] + (bias ? bias[i] : 0.f);
      sq = fmaf(v, v, sq);
    }
    for (int i = tid; i < NK; i += 256) {
      const float v = row[NQ + i] + (bias ? bias[NQ + i] : 0.f);
      sk = fmaf(v, v, sk);
    }
    rq = 1.f / sqrtf(block_sum(sq, red) / (float)NQ + eps);
    if (NK) rk = 1.f / sqrtf(block_sum(sk, red) / (float)NK + eps);
  }
  // rounds of upr heads (all of the row's q and k heads where LDS holds them: one barrier pair per row):
  // the round's heads are loaded, then every wave works on its own
  for (int u0 = 0; u0 < units; u0 += upr) {
    const int u1 = min(units, u0 + upr);
    for (int u = u0 + wv; u < u1; u += 4) {
      float* buf = sm + rot + (u - u0) * D;
      for (int d = lane; d < D; d += 64) {
        float v = row[u * D + d] + (bias ? bias[u * D + d] : 0.f);
        if (norm == 2) v *= u < H ? rq * (q_w ? q_w[u * D + d] : 1.f) : rk * (k_w ? k_w[(u - H) * D + d] : 1.f);
        buf[d] = v;
      }
    }
    __syncthreads();
    for (int u = u0 + wv; u < u1; u += 4) {
      const float* buf = sm + rot + (u - u0) * D;
      float val[kPrepPer];
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < kPrepPer; ++i) {
        const int d = lane + 64 * i;
        float xv = 0.f;
        if (d < D) {
          xv = buf[d];
          if (rot_pairs && d < rot) {
            const int j = d >> 1;
            xv = (d & 1) ? xv * cs[j] + buf[d - 1] * cs[half + j] : xv * cs[j] - buf[d + 1] * cs[half + j];
          } else if (d < half) {
            xv = xv * cs[d] - buf[d + half] * cs[half + d];
          } else if (d < rot) {
            const int j = d - half;
            xv = xv * cs[j] + buf[j] * cs[half + j];
          }
        }
        val[i] = xv;
        ss = fmaf(xv, xv, ss);
      }
      float rn = 1.f;
      if (norm == 1) rn = 1.f / sqrtf(wave_sum(ss) / (float)D + eps);
      const float* wgt = norm == 1 ? (u < H ? q_w : k_w) : nullptr;
      if (u < H) rn *= tq;
#pragma unroll
      for (int i = 0; i < kPrepPer; ++i) {
        const int d = lane + 64 * i;
        if (d < D) {
          const float o = val[i] * rn * (wgt ? wgt[d] : 1.f);
          if (u < H)
            sta(q_out, (size_t)r * NQ + u * D + d, o);
          else if (sl >= 0)
            sta(kc, (size_t)sl * NK + (u - H) * D + d, o);
        }
      }
    }
    if (u1 < units) __syncthreads();
  }
  const int page = sl >= 0 ? sl / BS : 0, off = sl >= 0 ? sl - page * BS : 0;
  for (int c = tid; c < NV; c += 256) {
    float v = row[v_col + c] + (bias ? bias[v_col + c] : 0.f);
    if (v_keep) v_keep[(size_t)r * NV + c] = v;
    if (v_other) v = (1.f - lam) * v + lam * v_other[(size_t)r * NV + c];
    if (sl >= 0) {
      if (vc) sta(vc, (size_t)sl * NV + c, v);
      if (vt) sta(vt, ((size_t)page * NV + c) * BS + off, v);
    }
  }
}

__global__ void __launch_bounds__(256) rope_table_kernel(const int* __restrict__ positions,
                                                         const double* __restrict__ freq, float amp,
                                                         float* __restrict__ cs, size_t n, int half) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) rope_entry(positions, freq, amp, cs, half, i);
}

template <typename TA>
__device__ __forceinline__ void sta4(TA* p, size_t i, const f32x4& v);
template <>
__device__ __forceinline__ void sta4<float>(float* p, size_t i, const f32x4& v) { *reinterpret_cast<f32x4*>(p + i) = v; }
template <>
__device__ __forceinline__ void sta4<uint16_t>(uint16_t* p, size_t i, const f32x4& v) {
  *reinterpret_cast<u16x4*>(p + i) = u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
}

// The value columns of TR rows from r0 (nr of them exist) to their pages: row-major, and a column of TR rows whose slots
// are neighbours of one page to the transposed page in one store.  MIX: kept as projected (v_keep) and mixed
// with another layer's (v_other) on the way, where these are given.
template <typename TA, int TR, bool MIX>
__device__ __forceinline__ void write_values(const float* __restrict__ x, int qs, int r0, int nr, int NV, int v_col,
                                             const float* __restrict__ bias, const int* __restrict__ slots,
                                             TA* __restrict__ vc, TA* __restrict__ vt, int BS, int tid, int threads,
                                             float lam, const float* __restrict__ v_other, float* __restrict__ v_keep,
                                             int planes = 1, size_t pstep = 0) {
  if (NV == 0) return;
  const int s0 = slots[r0];
  bool run = TR > 1 && nr == TR && s0 >= 0 && s0 % BS + TR <= BS;              // then a page holds all TR
  for (int k = 1; k < nr; ++k) run = run && slots[r0 + k] == s0 + k;
  for (int c = tid; c < NV; c += threads) {
    const float vb = bias ? bias[v_col + c] : 0.f;
    float v[TR], vo[TR];
#pragma unroll
    for (int k = 0; k < TR; ++k) {
      const int kk = min(k, nr - 1);
      v[k] = sum_planes(x + (size_t)(r0 + kk) * qs + v_col + c, pstep, TR == 1 ? planes : 1) + vb;
      vo[k] = MIX && v_other ? v_other[(size_t)(r0 + kk) * NV + c] : 0.f;
    }
    if (MIX) {
#pragma unroll
      for (int k = 0; k < TR; ++k)
        if (k < nr) {
          const size_t o = (size_t)(r0 + k) * NV + c;
          if (v_keep) v_keep[o] = v[k];
          if (v_other) v[k] = mix_value(lam, v[k], vo[k]);
        }
    }
    if (vt && run) {
      const int page = s0 / BS;
      TA* o = vt + ((size_t)page * NV + c) * BS + (s0 - page * BS);
      TA t[TR];
#pragma unroll
      for (int k = 0; k < TR; ++k) sta(t, k, v[k]);
      __builtin_memcpy(o, t, sizeof(t));                   // of any alignment: a sequence's rows start anywhere in a tile
    } else if (vt) {
#pragma unroll
      for (int k = 0; k < TR; ++k) {
        const int sl = k < nr ? slots[r0 + k] : -1;
        if (sl >= 0) sta(vt, ((size_t)(sl / BS) * NV + c) * BS + sl % BS, v[k]);
      }
    }
    if (vc) {
#pragma unroll
      for (int k = 0; k < TR; ++k) {
        const int sl = k < nr ? slots[r0 + k] : -1;
        if (sl >= 0) sta(vc, (size_t)sl * NV + c, v[k]);
      }
    }
  }
}

// The preparation where a row's entries do not meet beyond their rotation pair (2i, 2i + 1): no norm, no bias,
// cos | sin from the table.  A thread takes four neighbouring entries -- two pairs -- at a time straight from
// memory to memory (no LDS).  A workgroup takes TR rows; value column c of TR rows whose slots are
// neighbours of one page goes to the transposed page in one store.
template <typename TA, int TR>
__global__ void __launch_bounds__(256) attn_prep_pairs_kernel(const float* __restrict__ x, int qs, int NQ, int NK, int NV,
                                                              int D, int v_col, const int* __restrict__ slots,
                                                              TA* __restrict__ kc, TA* __restrict__ vc,
                                                              TA* __restrict__ vt, int BS, TA* __restrict__ q_out,
                                                              int rot, const float* __restrict__ cs, int T) {
  const int r0 = blockIdx.x * TR, tid = threadIdx.x, nv = (NQ + NK) >> 2, half = rot >> 1;
  const int nr = min(TR, T - r0);
  for (int i = tid; i < nr * nv; i += 256) {
    const int rr = i / nv, c = (i - rr * nv) << 2, r = r0 + rr;
    f32x4 v = *reinterpret_cast<const f32x4*>(x + (size_t)r * qs + c);
    const int d = c % D;
#pragma unroll
    for (int k = 0; k < 4; k += 2)
      if (d + k < rot) {
        const float* p = cs + (size_t)r * rot + ((d + k) >> 1);
        const float co = p[0], si = p[half], a = v[k], b = v[k + 1];
        v[k] = a * co - b * si;
        v[k + 1] = b * co + a * si;
      }
    if (c < NQ) {
      sta4(q_out, (size_t)r * NQ + c, v);
    } else {
      const int sl = slots[r];
      if (sl >= 0) sta4(kc, (size_t)sl * NK + (c - NQ), v);
    }
  }
  write_values<TA, TR, false>(x, qs, r0, nr, NV, v_col, nullptr, slots, vc, vt, BS, tid, 256, 0.f, nullptr, nullptr);
}

// four neighbours of a float array of any alignment
__device__ __forceinline__ f32x4 any4(const float* p) {
  f32x4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}

// The preparation with rotation halves (i with i + rot / 2), biases and a norm per head behind the rotation, cos | sin from
// the table:  D / 8 neighbouring lanes (a power of two) hold a head, each two groups of four entries -- rotated ones and
// their partners, or eight neighbours behind the rotated part -- so the rotation needs no exchange, the norm a few
// cross-lane sums, and every access is 16 bytes.  16 heads of 128 over 2 with values mixed across layers, 16384 rows: 226 us
// (attn_prep_kernel: a row's heads through LDS, a double-precision angle per pair where they are rotated) -> 73 us, one
// row 15 -> 3.0 us.  TR = 1 (few rows): a row over several
// workgroups, its values in some of their own: one pass of loads, and one compute unit does not take all its planes in
// (one row, four planes: 5.2 -> 4.1 us in a reply step).
constexpr int kPrepRow = 128;
template <typename TA, int TR, bool MIX>
__global__ void __launch_bounds__(256) attn_prep_half_kernel(const float* __restrict__ x, int qs, int H, int G, int NV, int D,
                                                             int v_col, const float* __restrict__ bias,
                                                             const int* __restrict__ slots, TA* __restrict__ kc,
                                                             TA* __restrict__ vc, TA* __restrict__ vt, int BS,
                                                             TA* __restrict__ q_out, int rot, const float* __restrict__ cs,
                                                             int norm, const float* __restrict__ q_w,
                                                             const float* __restrict__ k_w, float eps, int T, float lam,
                                                             const float* __restrict__ v_other,
                                                             float* __restrict__ v_keep, int planes, size_t pstep) {
  const int r0 = blockIdx.x * TR, tid = threadIdx.x, half = rot >> 1, lph = D >> 3, units = H + G;
  const int nr = min(TR, T - r0), n = units * lph;
  // TR = 1: the first workgroups of a row have its heads, 128 threads each, the others its values
  const int hb = TR == 1 ? (n + kPrepRow - 1) / kPrepRow : 1, heads = TR == 1 ? hb * kPrepRow : 256;
  const int at = TR == 1 ? (int)blockIdx.y * kPrepRow + tid : tid;
  for (int i = at; i < nr * n && at < heads; i += heads) {
    const int rr = i / n, u = (i - rr * n) / lph, j = i & (lph - 1), r = r0 + rr;
    const bool turn = 8 * j < rot;
    const int a = turn ? 4 * j : 8 * j, b = turn ? a + half : a + 4;
    const float* p = x + (size_t)r * qs + u * D;
    f32x4 va = sum_planes4(p + a, pstep, TR == 1 ? planes : 1), vb = sum_planes4(p + b, pstep, TR == 1 ? planes : 1);
    // the norm's weights with the row (entry by entry behind the norm they were half of the time)
    const float* w = u < H ? q_w : k_w;
    f32x4 wa = f32x4{1.f, 1.f, 1.f, 1.f}, wb = wa;
    if (w) {
      wa = any4(w + a);
      wb = any4(w + b);
    }
    if (bias) {
      const f32x4 ba = any4(bias + u * D + a), bb = any4(bias + u * D + b);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        va[k] += ba[k];
        vb[k] += bb[k];
      }
    }
    if (turn) {
      const float* c = cs + (size_t)r * rot + a;
      const f32x4 co = *reinterpret_cast<const f32x4*>(c), si = *reinterpret_cast<const f32x4*>(c + half);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float ua = va[k], ub = vb[k];
        va[k] = ua * co[k] - ub * si[k];
        vb[k] = ub * co[k] + ua * si[k];
      }
    }
    float rn = 1.f;
    if (norm) {
      float ss = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k) ss = fmaf(va[k], va[k], fmaf(vb[k], vb[k], ss));
      for (int o = 1; o < lph; o <<= 1) ss += __shfl_xor(ss, o, 64);
      rn = 1.f / sqrtf(ss / (float)D + eps);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      va[k] *= rn * wa[k];
      vb[k] *= rn * wb[k];
    }
    if (u < H) {
      const size_t o = ((size_t)r * H + u) * D;
      sta4(q_out, o + a, va);
      sta4(q_out, o + b, vb);
    } else {
      const int sl = slots[r];
      if (sl >= 0) {
        const size_t o = ((size_t)sl * G + u - H) * D;
        sta4(kc, o + a, va);
        sta4(kc, o + b, vb);
      }
    }
  }
  if (TR > 1)
    write_values<TA, TR, MIX>(x, qs, r0, nr, NV, v_col, bias, slots, vc, vt, BS, tid, 256, lam, v_other, v_keep);
  else if (at >= heads)
    write_values<TA, TR, MIX>(x, qs, r0, nr, NV, v_col, bias, slots, vc, vt, BS, at - heads,
                              (gridDim.y - hb) * kPrepRow, lam, v_other, v_keep, planes, pstep);
}


}  // namespace k8s

using namespace k8s;

K8S_API int k8s_attn_prep(const float* qkv, int qs, const float* bias, int H, int G, int D, int NV, const int* positions,
                          const int* slots, void* kc, void* vc, void* vt, int BS, void* q_out, int dt, int norm,
                          const float* q_w, const float* k_w, float eps, int rot, float base, float lam,
                          const float* v_other, float* v_keep, int T, hipStream_t s, int v_col, float tq_coef,
                          int tq_every, const double* rot_freq, float rot_amp, int rot_pairs,
                          const float* rot_cs) {
  if (T <= 0) return 0;
  if (H < 1 || G < 0 || D < 1 || D > 64 * kPrepPer || NV < 0 || rot < 0 || rot > D || (rot & 1) || BS < 1 ||
      norm < 0 || norm > 2 || v_col < 0 || tq_every < 0 || (G > 0 && !kc) || (NV > 0 && !vc && !vt))
    return (int)hipErrorInvalidValue;
  const int units = H + G;
  const int upr = (size_t)(rot + units * D) * sizeof(float) <= 64 * 1024 ? units : 4;    // heads per round
  const size_t lds = (size_t)(rot + upr * D) * sizeof(float);
  if (dt == 0)
    hipLaunchKernelGGL((attn_prep_kernel<uint16_t>), dim3(T), dim3(256), lds, s, qkv, qs, bias, H, G, D, NV, positions,
                       slots, (uint16_t*)kc, (uint16_t*)vc, (uint16_t*)vt, BS, (uint16_t*)q_out, norm, q_w, k_w, eps, rot,
                       base, lam, v_other, v_keep, upr, v_col, tq_coef, tq_every, rot_freq, rot_amp, rot_pairs,
                       rot_cs);
  else
    hipLaunchKernelGGL((attn_prep_kernel<float>), dim3(T), dim3(256), lds, s, qkv, qs, bias, H, G, D, NV, positions, slots,
                       (float*)kc, (float*)vc, (float*)vt, BS, (float*)q_out, norm, q_w, k_w, eps, rot, base, lam,
                       v_other, v_keep, upr, v_col, tq_coef, tq_every, rot_freq, rot_amp, rot_pairs,
                       rot_cs);
  return (int)hipGetLastError();
}

K8S_API int k8s_rope_table(const int* positions, const double* freq, float amp, float* cs, int T, int half, hipStream_t s) {
  if (T <= 0 || half <= 0) return 0;
  const size_t n = (size_t)T * half;
  hipLaunchKernelGGL(rope_table_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, positions, freq, amp, cs, n,
                     half);
  return (int)hipGetLastError();
}

// D and qs multiples of 4, x / q_out / kc 16-byte aligned (8 for bf16 outputs); rot 0 needs no table
K8S_API int k8s_attn_prep_pairs(const float* x, int qs, int H, int G, int D, int NV, int v_col, const int* slots,
                                void* kc, void* vc, void* vt, int BS, void* q_out, int dt, int rot, const float* cs,
                                int T, hipStream_t s) {
  if (T <= 0) return 0;
  if (H < 1 || G < 0 || D < 4 || D % 4 || qs % 4 || rot < 0 || rot > D || rot % 2 || (rot && !cs) || NV < 0 || v_col < 0 ||
      BS < 1 || (G > 0 && !kc) || (NV > 0 && !vc && !vt) || ((uintptr_t)x & 15))
    return (int)hipErrorInvalidValue;
#define K8S_PP(TA, TR)                                                                                             \
  hipLaunchKernelGGL((attn_prep_pairs_kernel<TA, TR>), dim3((T + TR - 1) / TR), dim3(256), 0, s, x, qs, H * D, G * D, NV, \
                     D, v_col, slots, (TA*)kc, (TA*)vc, (TA*)vt, BS, (TA*)q_out, rot, cs, T)
  if (dt == 0) {
    if (T > 1024) K8S_PP(uint16_t, 8);
    else K8S_PP(uint16_t, 1);
  } else {
    if (T > 1024) K8S_PP(float, 8);
    else K8S_PP(float, 1);
  }
#undef K8S_PP
  return (int)hipGetLastError();
}

// D 8, 16, .. 512 (powers of two), qs a multiple of 4, rot a multiple of 8 with its table, x / q_out / kc / cs 16-byte
// aligned (8 for bf16 outputs); norm 0 / 1 as in k8s_attn_prep.  planes > 1 (T <= 1024): x is the sum of as many, pstep
// (a multiple of 4) numbers apart
K8S_API int k8s_attn_prep_half(const float* x, int qs, int H, int G, int D, int NV, int v_col, const float* bias,
                               const int* slots, void* kc, void* vc, void* vt, int BS, void* q_out, int dt, int rot,
                               const float* cs, int norm, const float* q_w, const float* k_w, float eps, int T,
                               hipStream_t s, float lam, const float* v_other, float* v_keep, int planes, long pstep) {
  if (T <= 0) return 0;
  if (H < 1 || G < 0 || D < 8 || D > 512 || (D & (D - 1)) || qs % 4 || rot < 0 || rot > D || rot % 8 || (rot && !cs) ||
      NV < 0 || v_col < 0 || BS < 1 || (G > 0 && !kc) || (NV > 0 && !vc && !vt) || norm < 0 || norm > 1 ||
      planes < 1 || (planes > 1 && (T > 1024 || pstep % 4)) || ((uintptr_t)x & 15) || ((uintptr_t)cs & 15))
    return (int)hipErrorInvalidValue;
  const int row_groups = ((H + G) * (D / 8) + kPrepRow - 1) / kPrepRow + (NV + kPrepRow - 1) / kPrepRow;
#define K8S_PH(TA, TR, MIX)                                                                                             \
  hipLaunchKernelGGL((attn_prep_half_kernel<TA, TR, MIX>), dim3((T + TR - 1) / TR, TR == 1 ? row_groups : 1), dim3(TR == 1 ? kPrepRow : 256), 0, s, x, qs, H, G, NV, D, \
                     v_col, bias, slots, (TA*)kc, (TA*)vc, (TA*)vt, BS, (TA*)q_out, rot, cs, norm, q_w, k_w, eps, T, lam, \
                     v_other, v_keep, planes, pstep)
#define K8S_PH_T(TA)                                   \
  if (v_other || v_keep) {                             \
    if (T > 1024) K8S_PH(TA, 8, true);                 \
    else K8S_PH(TA, 1, true);                          \
  } else {                                             \
    if (T > 1024) K8S_PH(TA, 8, false);                \
    else K8S_PH(TA, 1, false);                         \
  }
  if (dt == 0) {
    K8S_PH_T(uint16_t)
  } else {
    K8S_PH_T(float)
  }
#undef K8S_PH_T
#undef K8S_PH
  return (int)hipGetLastError();
}

// 1 when the matrix-core kernels (mask_prompt.hip, token_attn.hip) take these sizes (bf16 only)
K8S_API int k8s_masked_attn_mfma_ok(int H, int G, int D, int V) {
  return H >= 1 && G >= 1 && H % G == 0 && (((D == 64 || D == 128) && (V == 64 || V == 128)) || (D == 96 && V == 96));
}
