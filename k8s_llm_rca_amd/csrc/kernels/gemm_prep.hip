// An attention layer's input product of many rows together with the pass behind it (attn_prep_half_kernel, masked_attn.hip):
//   x = A . W^T = q [H][D] | k [G][D] | v [G][V] | rest,   + bias;  q and k rotated (entry i with i + rot / 2, cos | sin from the
//   table) and divided by their head's root mean square (times a weight);  v kept as projected and mixed with another layer's;
//   q written as activations, k and v (transposed, and as it is where asked for) to their pages, the rest as it is in fp32.
//
// The pass read 10 KB of fp32 a row and wrote 5 KB of activations (16 heads over 2 of 128) behind a product that wrote the 10 KB:  of
// both only the activations are left.  The tiles are gemm_add's (row_tiles.h); every tile of columns is of one kind (H D, G D and G V are
// multiples of 256), the last one of the rest may end early.  In a tile of heads W's rows are staged in an order that gives a lane
// four neighbouring rotation pairs of a head, which need no exchange; the head's sum of squares meets over four lanes and, through LDS, over
// the head's waves.  A tile of values or of the rest passes through LDS, half at a time: a thread takes eight tokens of a value's
// column for its page, a wave whole rows of the rest.
//
// What bounds it: the product (row_tiles.h) and the epilogue, which the matrix units wait for.  us at 4096 rows of 16 heads over 2 of 128,
// K 2048, product and pass 65 (with values to mix 71) / whole rows through LDS with the rotation and the norm as exchanges 69 (75) / pairs
// in a lane 59 (77) / the values' slots and their other layer's asked for ahead 52 (54);  at 16384 237 (248) / 229 / 195 / 176 (176): 0.98
// PFLOP/s.  More sizes: ops/linear.py, prep_plan.
#include "key_runs.h"
#include "row_tiles.h"

namespace k8s {
namespace padd {

struct PrepArgs {
  const uint16_t* a;     // [M][lda]
  const uint16_t* w;     // [N][K]
  const float* bias;     // [nq + nk + nv] or null
  const float* cs;       // [M][rot]: cos | sin, or null
  const float* q_w;      // [D] or null
  const float* k_w;
  const float* v_other;  // [M][nv] or null
  float* v_keep;         // [M][nv] or null
  const int* slots;      // [M]
  uint16_t* q;           // [M][nq]
  uint16_t* kc;          // [pages][BS][nk]
  uint16_t* vt;          // [pages][nv][BS]
  uint16_t* vc;          // [pages][BS][nv] or null
  float* rest;           // [M][ldr]
  float eps, lam;
  int lda, ldr, M, N, K, nq, nk, nv, D, rot, norm, BS, n_mt, n_nt;
};

template <int F>
__global__ void __launch_bounds__(512, 1) gemm_prep_kernel(PrepArgs p) {
  using Tile = RowTile<F>;
  constexpr int HM = Tile::HM, RW = HM / 8;                 // rows of a half, of it a wave's
  constexpr int U = 4;                                      // fragments whose tables are asked for at once
  __shared__ __attribute__((aligned(1024))) unsigned char sm[Tile::LDS];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wv >> 2, wc = wv & 3;
  int tm, tn;
  tile_of(p.n_mt, p.n_nt, tm, tn);
  const int M = p.M, m0 = tm * Tile::BM, n0 = tn * BN, nqk = p.nq + p.nk, nqkv = nqk + p.nv;
  const bool heads = n0 < nqk, isq = n0 < p.nq, vals = !heads && n0 < nqkv;
  // A head's pair t is (t, t + rot / 2) where it is rotated, else two others of its entries; a lane has four neighbouring pairs
  const int half = p.rot >> 1, gap = (p.D >> 1) - half, slabs = p.D >> 5;           // (32 columns of a wave: a slab)
  auto entry = [&](int t, int second) { return t < half ? t + second * half : p.rot + t - half + second * gap; };
  f32x4 acc[2][F][2];
  Tile::product(p.a, p.lda, p.w, M, p.K, m0, sm, acc, [&](int h, int R) {
    const int slab = R >> 5, in = slab & (slabs - 1);
    const int c = heads ? 128 * h + 32 * (slab - in) + entry(16 * in + (R & 15), (R >> 4) & 1) : eight_columns(h, R);
    return min(n0 + c, p.N - 1);
  });
  lds_bar();                                                // (every wave has read its last fragments)

  if (heads) {
    const int frow = lane & 15, fhi = lane >> 4, in = wc & (slabs - 1), t0 = 16 * in + 4 * fhi;
    const int d0 = entry(t0, 0), d1 = entry(t0, 1), hd = 32 * (wc - in);           // hd: the head's first column in the half
    const bool turn = t0 < half;
    auto row = [&](int i) { return m0 + HM * wr + 16 * i + frow; };
    float* const red = reinterpret_cast<float*>(sm) + wr * HM * 8;                   // [HM][2][4]: the slabs' sums of squares
    f32x4 b[2][2], hw[2];
    hw[0] = hw[1] = f32x4{1.f, 1.f, 1.f, 1.f};
    const float* w = isq ? p.q_w : p.k_w;
    if (w) hw[0] = *reinterpret_cast<const f32x4*>(w + d0), hw[1] = *reinterpret_cast<const f32x4*>(w + d1);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        b[h][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (p.bias) b[h][j] = *reinterpret_cast<const f32x4*>(p.bias + n0 + 128 * h + hd + (j ? d1 : d0));
      }
#pragma unroll
    for (int i0 = 0; i0 < F; i0 += U) {
      f32x4 co[U], si[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        co[u] = f32x4{1.f, 1.f, 1.f, 1.f}, si[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (turn) {
          const float* c = p.cs + (size_t)min(row(min(i0 + u, F - 1)), M - 1) * p.rot + t0;
          co[u] = *reinterpret_cast<const f32x4*>(c), si[u] = *reinterpret_cast<const f32x4*>(c + half);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u;
        if (i >= F) break;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 x = acc[h][i][0] + b[h][0], y = acc[h][i][1] + b[h][1];
          f32x4 xr = x, yr = y;
          if (turn) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              xr[k] = x[k] * co[u][k] - y[k] * si[u][k];
              yr[k] = y[k] * co[u][k] + x[k] * si[u][k];
            }
          }
          acc[h][i][0] = xr, acc[h][i][1] = yr;
          float ss = 0.f;
#pragma unroll
          for (int k = 0; k < 4; ++k) ss = fmaf(xr[k], xr[k], fmaf(yr[k], yr[k], ss));
          ss += __shfl_xor(ss, 16, 64);
          ss += __shfl_xor(ss, 32, 64);
          if (fhi == 0) red[((16 * i + frow) * 2 + h) * 4 + wc] = ss;
        }
      }
    }
    lds_bar();
#pragma unroll
    for (int i = 0; i < F; ++i) {
      const int m = row(i);
      const int sl = isq || m >= M ? 0 : p.slots[m];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float rn = 1.f;
        if (p.norm) {
          const f32x4 s = *reinterpret_cast<const f32x4*>(red + ((16 * i + frow) * 2 + h) * 4);
          const float ss = p.D == 128 ? s[0] + s[1] + s[2] + s[3] : wc < 2 ? s[0] + s[1] : s[2] + s[3];
          rn = 1.f / sqrtf(ss / (float)p.D + p.eps);
        }
        u16x4 o[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int k = 0; k < 4; ++k) o[j][k] = f2bf(acc[h][i][j][k] * (rn * hw[j][k]));
        const int c = n0 + 128 * h + hd;
        if (m >= M || sl < 0) continue;
        uint16_t* to = isq ? p.q + (size_t)m * p.nq + c : p.kc + (size_t)sl * p.nk + (c - p.nq);
        *reinterpret_cast<u16x4*>(to + d0) = o[0];
        *reinterpret_cast<u16x4*>(to + d1) = o[1];
      }
    }
    return;
  }

  // Values: a thread has a column, eight rows at a time, which go to a page at once where they are neighbours of one.  The other
  // layer's values and the slots (lane: row of the half) are asked for in front of the half's results.
  const int c1 = threadIdx.x & 255, col = n0 - nqk + c1, g0 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  constexpr int VF = F == 8 ? 4 : F;                        // groups of rows whose values are held (registers)
  float vo[VF][8];
  int sv[2];
  auto ask_other = [&](int hf, int i0) {
    if (p.v_other)
#pragma unroll
      for (int it = 0; it < VF; ++it)
#pragma unroll
        for (int k = 0; k < 8; ++k)
          vo[it][k] = p.v_other[(size_t)min(m0 + HM * hf + 8 * (2 * (i0 + it) + g0) + k, M - 1) * p.nv + col];
  };
  auto ask_values = [&](int hf) {
#pragma unroll
    for (int q = 0; q < 2; ++q) sv[q] = p.slots[min(m0 + HM * hf + 64 * q + lane, M - 1)];
    ask_other(hf, 0);
  };
  auto finish_values = [&](int hf) {
    const float bias = p.bias ? p.bias[n0 + c1] : 0.f;
    // (a loop: the second groups' values are asked for when the first ones are done with)
#pragma unroll 1
    for (int i0 = 0; i0 < F; i0 += VF) {
      if (i0) ask_other(hf, i0);
#pragma unroll
      for (int it = 0; it < VF; ++it) {
        const int g = 2 * (i0 + it) + g0, r = m0 + HM * hf + 8 * g, n = min(8, M - r);
        if (n <= 0) break;
        int sl[8];
        u16x8 h;
#pragma unroll
        for (int k = 0; k < 8; ++k) sl[k] = __builtin_amdgcn_readlane(g < 8 ? sv[0] : sv[1], (8 * g + k) & 63);
        bool run = n == 8 && sl[0] >= 0 && sl[0] % p.BS + 8 <= p.BS;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const int rr = 8 * g + k;
          float v = *reinterpret_cast<const float*>(sm + rr * 1024 + 16 * ((c1 >> 2) ^ (rr & 15)) + 4 * (c1 & 3)) + bias;
          run = run && sl[k] == sl[0] + k;
          if (p.v_keep && k < n) p.v_keep[(size_t)(r + k) * p.nv + col] = v;
          if (p.v_other) v = mix_value(p.lam, v, vo[it][k]);
          h[k] = f2bf(v);
          if (p.vc && k < n && sl[k] >= 0) p.vc[(size_t)sl[k] * p.nv + col] = h[k];
        }
        if (run) {
          __builtin_memcpy(p.vt + ((size_t)(sl[0] / p.BS) * p.nv + col) * p.BS + sl[0] % p.BS, &h, 16);      // (of any alignment)
        } else {
#pragma unroll
          for (int k = 0; k < 8; ++k)
            if (k < n && sl[k] >= 0) p.vt[((size_t)(sl[k] / p.BS) * p.nv + col) * p.BS + sl[k] % p.BS] = h[k];
        }
      }
    }
  };
  auto finish_rest = [&](int hf) {
    const int c0 = n0 + 4 * lane;
    if (c0 >= p.N) return;
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int m = m0 + HM * hf + 8 * i + wv;
      if (m < M) *reinterpret_cast<f32x4*>(p.rest + (size_t)m * p.ldr + (c0 - nqkv)) = Tile::get(sm, 8 * i + wv);
    }
  };
  for (int hf = 0; hf < 2; ++hf) {
    if (vals) ask_values(hf);
    if (hf) lds_bar();                                      // (the first half is read)
    if (wr == hf) Tile::put(sm, acc);
    lds_bar();
    if (vals)
      finish_values(hf);
    else
      finish_rest(hf);
  }
}

template <int F>
static int launch_prep(PrepArgs p, hipStream_t s) {
  p.n_mt = (p.M + 32 * F - 1) / (32 * F);
  p.n_nt = (p.N + BN - 1) / BN;
  hipLaunchKernelGGL((gemm_prep_kernel<F>), dim3(p.n_mt * p.n_nt), dim3(512), 0, s, p);
  return (int)hipGetLastError();
}

}  // namespace padd
}  // namespace k8s

using namespace k8s;

// f: rows of a tile / 32 (4, 5, 6, 8).  nq, nk, nv multiples of 256, N of 4, K of 64; D 64 or 128, rot 0 or 8 times a power of two up to
// D with cs; rest (where N is more than the three) rows of ldr, a multiple of 4.  All on 16 bytes but slots, q, kc, vc (8) and vt (2).
K8S_API int k8s_gemm_prep(const void* a, int lda, const void* w, int M, int N, int K, int f, const float* bias, const float* cs, int rot,
                          int norm, const float* q_w, const float* k_w, float eps, float lam, const float* v_other, float* v_keep,
                          const int* slots, void* q, void* kc, void* vt, void* vc, int BS, int nq, int nk, int nv, int D, float* rest,
                          int ldr, hipStream_t s) {
  using namespace k8s::padd;
  auto off = [](const void* t, int n) { return ((uintptr_t)t % n) != 0; };
  const int over = N - nq - nk - nv;
  if (M <= 0 || K <= 0 || K % BK || N <= 0 || N % 4 || nq < BN || nk < BN || nv < BN || nq % BN || nk % BN || nv % BN || over < 0 ||
      (D != 64 && D != 128) || nq % D || nk % D || rot < 0 || rot > D || (rot && (rot < 8 || (rot & (rot - 1)) || !cs)) || BS < 1 ||
      (over && (!rest || ldr < over || ldr % 4)) || norm < 0 || norm > 1 || !a || !w || lda < K || lda % 8 || !slots || !q || !kc || !vt ||
      off(a, 16) || off(w, 16) || off(bias, 16) || off(cs, 16) || off(q_w, 16) || off(k_w, 16) || off(v_other, 16) || off(v_keep, 16) ||
      off(rest, 16) || off(q, 8) || off(kc, 8) || off(vc, 8))
    return (int)hipErrorInvalidValue;
  const PrepArgs p{(const uint16_t*)a, (const uint16_t*)w, bias, cs, q_w, k_w, v_other, v_keep, slots, (uint16_t*)q, (uint16_t*)kc,
                   (uint16_t*)vt, (uint16_t*)vc, rest, eps, lam, lda, ldr, M, N, K, nq, nk, nv, D, rot, norm, BS, 0, 0};
  switch (f) {
    case 4: return launch_prep<4>(p, s);
    case 5: return launch_prep<5>(p, s);
    case 6: return launch_prep<6>(p, s);
    case 8: return launch_prep<8>(p, s);
  }
  return (int)hipErrorInvalidValue;
}
