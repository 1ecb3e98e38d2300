// Prompt portions of the masked attention (masked_attn.hip: causal, chunked, windowed with kept first tokens, sinks,
// capped scores, output gates, score maps) with the heads of a key head as rows of one tile.
//
// A workgroup is 4 waves x 32 rows (token, head of the key head): 128 / heads tokens.  Keys go in blocks of 64 whose
// 32-key halves do not cross a page (BS % 32 == 0), fetched into registers while the block before is computed and parked in LDS (two
// buffers, one barrier per block), so a byte of K and V leaves the caches once per 128 rows.  v_mfma_f32_32x32x16_bf16,
// swapped: S^T = K Q^T, a lane owns query row lane & 31; MFMA row rho of a 32-key half stands for key
// 16 (reg >> 3) + 8 hi + (reg & 7), reg = (rho & 3) + 4 (rho >> 3), hi = (rho >> 2) & 1, so that a lane's score
// registers 8 s .. 8 s + 7 are the weights operand of O^T = V^T P^T as they stand.  LDS rows are padded by 16 bytes: the
// 16 rows a quarter wave reads 16 bytes of lie in different banks for D = 64, 96 and 128 alike.
//
// Few tiles behind many keys: a tile's blocks are cut into parts, a workgroup each, whose outputs a second kernel joins
// (n_parts; 500 rows at 8000 keys, 16 heads over 2 of 128: 211 -> 62 us).
//
// Zero weights times values that are not finite are NaN in rows that do not see their keys.  A tile that ends with a result
// that is not finite walks its keys once more (CARE): in blocks that some token does not see whole, such values are parked
// as zeros, and added behind the walk where they are seen.  (Looking at every block's values on the way cost 3.5 %.)
//
// What bounds it: matrix and vector instructions of two waves a SIMD in turn (240 registers).  Eight prompts of 2048, 16
// heads over 2 of 128, us alone in a loop: causal 230 = 598 TFLOP/s, a window of 1024 175 = 590, chunks of 1024 with capped
// scores 168 = 410 (an exponential and a reciprocal more per score);  between a prompt's other kernels, whose traffic has
// taken the caches, the latter two 190 to 220 and 183 to 186.  Tiles of 16 tokens x 2 heads a wave with operands from the caches
// took 681, 485 and 418: every wave fetched its keys itself.
#include <type_traits>

#include "common.h"
#include "key_runs.h"

namespace k8s {

struct MaskPromptArgs {
  const uint16_t* q;      // [T][H M D]
  const uint16_t* kc;     // [pages][BS][G M D]
  const uint16_t* vt;     // [pages][G V][BS]
  const int* bt;
  int maxb;
  const int* items;       // [n][4]: segment, first row, tokens (<= max(1, 128 / (H / G))), position of the first token
  int n_items;
  const float* sink;      // [H M] or null
  const float* gate;      // rows of stride gs, column h, or null
  int gs;
  uint16_t* out;          // [T][H M V]
  float* out32;           // the same in fp32 instead
  int H, G, M, BS, chunk, window, keep_first;    // H: heads (each with M maps)
  float scale, softcap;
  // few tiles: a tile's blocks are split over grid.y workgroups of part_blocks each, whose results a merge joins
  int n_parts, part_blocks, row_base;            // row_base: the first tile's first row
  float* po;              // [rows][H M][n_parts][V]
  float* pml;             // [rows][H M][n_parts][2]
};

// of a pair of bf16 numbers: bits 15 and 31 set where one is infinite or NaN (an exponent of ones)
__device__ __forceinline__ uint32_t mp_wild(uint32_t v) { return ((v & 0x7f807f80u) + 0x00800080u) & 0x80008000u; }

__device__ __forceinline__ int mp_key(int reg, int hi) { return 16 * (reg >> 3) + 8 * hi + (reg & 7); }

// HALF: BS is an odd multiple of 32, a block's halves may lie in two pages.
template <int ND, int NV, int NW, bool CAP, bool HALF>
__global__ void __launch_bounds__(64 * NW, ND == 4 && NV == 2 ? 3 : 2) mask_prompt_kernel(MaskPromptArgs a) {
  constexpr int D = ND * 16, V = NV * 32, TH = 64 * NW, KP = D * 2 + 16, VP = 144;
  constexpr int KC = 64 * D / 8 / TH, VC = V * 8 / TH;      // 16-byte chunks per thread and block
  static_assert(64 * D / 8 % TH == 0 && V * 8 % TH == 0, "whole chunks per thread");
  constexpr float kLog2e = 1.4426950408889634f;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2][64 * KP + V * VP];
  __shared__ int wild[NW];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 31, hi = lane >> 5;
  // key heads (and groups of 128 of their heads) next to each other, the last items first: they see the most keys
  const int hpg = a.H / a.G, hw = min(hpg, 32 * NW), nhc = (hpg + hw - 1) / hw, per = a.G * a.M * nhc;
  const int kh = blockIdx.x % per / nhc, hc = blockIdx.x % nhc, gv = kh / a.M, mp = kh % a.M;
  const int item = a.n_items - 1 - blockIdx.x / per;
  const int sg = a.items[item * 4], row0 = a.items[item * 4 + 1], ntok = a.items[item * 4 + 2],
            pos0 = a.items[item * 4 + 3];
  const int HM = a.H * a.M, NK = a.G * a.M * D, NVt = a.G * V;
  const int grow = w * 32 + r, tt = grow / hw, hh = hc * hw + grow % hw, head = (gv * hpg + hh) * a.M + mp;
  const bool valid = tt < ntok && hh < hpg;
  const int pos = pos0 + tt, pos_last = pos0 + ntok - 1;
  const int limit = valid ? pos : -1;                       // last visible key
  const int cq_lo = a.chunk > 0 ? (pos / a.chunk) * a.chunk : 0;
  const int wq_lo = a.window > 0 ? pos - a.window + 1 : 0;
  const int keep = a.window > 0 ? a.keep_first : 0;
  // the wave's first and last token: a block that both see whole needs no mask
  const int wt0 = w * 32 / hw, wt1 = min(ntok - 1, (w * 32 + 31) / hw);
  const bool full = (w * 32 + 31) / hw < ntok;              // every row of the wave is a token's
  const int wp0 = pos0 + wt0, wp1 = pos0 + wt1;
  const int cl_lo = a.chunk > 0 ? (wp1 / a.chunk) * a.chunk : 0, wl_lo = a.window > 0 ? wp1 - a.window + 1 : 0;
  const int cw_lo = a.chunk > 0 ? (wp0 / a.chunk) * a.chunk : 0, ww_lo = a.window > 0 ? wp0 - a.window + 1 : 0;
  // the tile's key blocks: kept first tokens [a_beg, a_end), then [lo_al, pos_last]
  const KeyRuns k0 = key_runs(pos0, a.chunk, a.window, a.keep_first);
  const int lo_al = k0.lo & ~63, a_beg = k0.a0 & ~63;
  const int a_end = a.window > 0 ? min(lo_al, (a.keep_first + 63) & ~63) : a_beg;
  const int nblkA = max(0, (a_end - a_beg) >> 6), nblk = nblkA + ((pos_last - lo_al) >> 6) + 1;
  const int b_lo = blockIdx.y * a.part_blocks, b_hi = (int)blockIdx.y == a.n_parts - 1 ? nblk : min(nblk, b_lo + a.part_blocks);
  const size_t part = (((size_t)(row0 + tt - a.row_base) * HM + head) * a.n_parts + blockIdx.y);
  if (b_lo >= b_hi) {                                       // the whole workgroup: a part without blocks
    if (valid && hi == 0) {
      a.pml[part * 2] = -INFINITY;
      a.pml[part * 2 + 1] = 0.f;
    }
    return;
  }
  const int* pages = a.bt + (size_t)sg * a.maxb;
  auto block_at = [&](int bi) { return bi < nblkA ? a_beg + 64 * bi : lo_al + 64 * (bi - nblkA); };

  bf16x8 qf[ND];
  const uint16_t* qp = a.q + (size_t)(row0 + (valid ? tt : 0)) * HM * D + (size_t)(valid ? head : mp) * D + 8 * hi;
#pragma unroll
  for (int s = 0; s < ND; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + 16 * s);
  f32x16 o[NV];
  float m, l;
  // a scale that is not positive is applied before the mask and the maximum, a positive one in the exponent
  const float sc1 = a.scale * kLog2e, sc2 = sc1 > 0.f ? sc1 : 1.f, cap2 = a.softcap * kLog2e, icap = CAP ? 2.f * kLog2e * a.scale / a.softcap : 0.f;

  bf16x8 stg[KC + VC];
  auto load = [&](int kb, int pg0, int pg1) {
    const int of0 = kb % a.BS, of1 = HALF ? (kb + 32) % a.BS : 0;
    const uint16_t* kp = a.kc + ((size_t)pg0 * a.BS + of0) * NK + kh * D;
    const uint16_t* vp = a.vt + ((size_t)pg0 * NVt + (size_t)gv * V) * a.BS + of0;
    const uint16_t* k1 = HALF ? a.kc + ((size_t)pg1 * a.BS + of1 - 32) * NK + kh * D : kp;
    const uint16_t* v1 = HALF ? a.vt + ((size_t)pg1 * NVt + (size_t)gv * V) * a.BS + of1 - 32 : vp;
#pragma unroll
    for (int i = 0; i < KC; ++i) {
      const int c = tid + TH * i, key = c / (D / 8);
      stg[i] = *reinterpret_cast<const bf16x8*>((HALF && key >= 32 ? k1 : kp) + (size_t)key * NK + 8 * (c % (D / 8)));
    }
#pragma unroll
    for (int i = 0; i < VC; ++i) {
      const int c = tid + TH * i;
      stg[KC + i] = *reinterpret_cast<const bf16x8*>((HALF && (c & 4) ? v1 : vp) + (size_t)(c >> 3) * a.BS + 8 * (c & 7));
    }
  };
  // the pages of a block's halves (a second half past the last key reads the first's)
  auto page0 = [&](int kb) { return pages[kb / a.BS]; };
  auto page1 = [&](int kb) { return HALF ? pages[(kb + 32 <= pos_last ? kb + 32 : kb) / a.BS] : 0; };
  const int tl_lo = a.chunk > 0 ? (pos_last / a.chunk) * a.chunk : 0, tw_lo = a.window > 0 ? pos_last - a.window + 1 : 0;
  auto open = [&](int kb) { return kb + 63 <= pos0 && kb >= tl_lo && (kb >= tw_lo || kb + 64 <= keep); };
  auto park = [&](int b, int kb, auto care) {
    if constexpr (decltype(care)::value) {
      if (!open(kb)) {
        uint32_t x[4 * VC];
        __builtin_memcpy(x, stg + KC, sizeof(x));
#pragma unroll
        for (int i = 0; i < 4 * VC; ++i) x[i] &= ~((mp_wild(x[i]) >> 15) * 0xffffu);
        __builtin_memcpy(stg + KC, x, sizeof(x));
      }
    }
#pragma unroll
    for (int i = 0; i < KC; ++i) {
      const int c = tid + TH * i;
      *reinterpret_cast<bf16x8*>(lds[b] + (c / (D / 8)) * KP + 16 * (c % (D / 8))) = stg[i];
    }
#pragma unroll
    for (int i = 0; i < VC; ++i) {
      const int c = tid + TH * i;
      *reinterpret_cast<bf16x8*>(lds[b] + 64 * KP + (c >> 3) * VP + 16 * (c & 7)) = stg[KC + i];
    }
  };
  const int krow = mp_key((r & 3) + 4 * (r >> 3), (r >> 2) & 1);   // the key of this lane's MFMA row in a 32-key half
  // the queries are there before the loop: its waits count the block loads alone
#pragma unroll
  for (int s = 0; s < ND; ++s) asm volatile("" ::"v"(qf[s]));
  auto walk = [&](auto care) {
#pragma unroll
    for (int dt = 0; dt < NV; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[dt][i] = 0.f;
    m = a.sink && valid && a.n_parts == 1 ? a.sink[head] * kLog2e : -INFINITY;
    l = 0.f;
    int kb_next = block_at(min(b_lo + 1, b_hi - 1)), pg0 = page0(kb_next), pg1 = page1(kb_next);
    {
      const int kb = block_at(b_lo);
      load(kb, page0(kb), page1(kb));
      park(b_lo & 1, kb, care);
    }
    __syncthreads();
    for (int bi = b_lo; bi < b_hi; ++bi) {
      const int kb = block_at(bi);
      // the page of the block after the next, while this one is computed (the last ones are read again: every load is
      // unconditional, so the count of loads in flight is known)
      const int kb_after = block_at(min(bi + 2, b_hi - 1)), pa0 = page0(kb_after), pa1 = page1(kb_after);
      load(kb_next, pg0, pg1);
      // a wave all of whose tokens come before the block, or after its window or chunk, has nothing to do
      const bool live = wt0 < ntok && kb <= wp1 && kb + 63 >= cw_lo && (kb + 63 >= ww_lo || kb < keep);
      if (live) {
        const unsigned char *kl = lds[bi & 1], *vl = kl + 64 * KP;
        f32x16 sc[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
          const unsigned char* kr = kl + (32 * kt + krow) * KP + 16 * hi;
          f32x16 acc;
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
          for (int s = 0; s < ND; ++s)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(kr + 32 * s), qf[s], acc, 0, 0, 0);
          sc[kt] = acc;
        }
        if (CAP) {                                            // cap tanh(x), tanh(x) = 1 - 2 / (1 + e^(2x)), in log2 units
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const float e = __builtin_amdgcn_exp2f(fminf(sc[kt][i] * icap, 60.f));
              sc[kt][i] = cap2 * (1.f - 2.f * __builtin_amdgcn_rcpf(1.f + e));
            }
        } else if (!(sc1 > 0.f)) {
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int i = 0; i < 16; ++i) sc[kt][i] *= sc1;
        }
        if (!(full && kb + 63 <= wp0 && kb >= cl_lo && (kb >= wl_lo || kb + 64 <= keep))) {
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const int key = kb + 32 * kt + mp_key(i, hi);
              const bool ok = key <= limit && key >= cq_lo && (key >= wq_lo || key < keep);
              sc[kt][i] = ok ? sc[kt][i] : -INFINITY;
            }
        }
        float cmax = sc[0][0];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int i = 0; i < 16; ++i) cmax = fmaxf(cmax, sc[kt][i]);
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32, 64));
        // the reference moves only where a row's maximum outgrows it by 2^8: weights up to 256, exact in the sums, and most
        // blocks leave the outputs alone
        const float mc = CAP ? cmax : cmax * sc2;
        const bool upd = mc > m + 8.f;
        const float mn = upd ? mc : m, sub = mn == -INFINITY ? 0.f : -mn;
        bf16x8 pf[2][2];
        float ps = 0.f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const float x = sc[kt][8 * s + j], e = __builtin_amdgcn_exp2f(CAP ? x + sub : fmaf(x, sc2, sub));
              ps += e;
              pf[kt][s][j] = (__bf16)e;
            }
        if (__any(upd)) {
          const float alpha = upd ? __builtin_amdgcn_exp2f(m - mn) : 1.f;
          l *= alpha;
          m = mn;
#pragma unroll
          for (int dt = 0; dt < NV; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[dt][i] *= alpha;
        }
        l += ps;
#pragma unroll
        for (int dt = 0; dt < NV; ++dt) {
          const unsigned char* vr = vl + (32 * dt + r) * VP + 16 * hi;
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int s = 0; s < 2; ++s)
              o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(vr + 64 * kt + 32 * s),
                                                              pf[kt][s], o[dt], 0, 0, 0);
        }
      }
      park((bi + 1) & 1, kb_next, care);
      kb_next = kb_after;
      pg0 = pa0;
      pg1 = pa1;
      __syncthreads();
    }
  };
  walk(std::false_type{});
  float z = 0.f;
#pragma unroll
  for (int dt = 0; dt < NV; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) z = fmaf(o[dt][i], 0.f, z);
  const bool any = __any(z != z);
  if (lane == 0) wild[w] = any;
  __syncthreads();
  bool care = false;
#pragma unroll
  for (int i = 0; i < NW; ++i) care |= wild[i] != 0;
  if (care) walk(std::true_type{});
  if (!valid) return;
  l += __shfl_xor(l, 32, 64);
  if (care) {                                               // (a weight above zero leaves infinity and NaN what they are)
    for (int bi = b_lo; bi < b_hi; ++bi) {
      const int kb = block_at(bi);
      if (open(kb)) continue;
      for (int key = kb; key < min(kb + 64, limit + 1); ++key) {
        if (key < cq_lo || (key < wq_lo && key >= keep)) continue;
        const uint16_t* vp = a.vt + ((size_t)pages[key / a.BS] * NVt + (size_t)gv * V + 4 * hi) * a.BS + key % a.BS;
#pragma unroll
        for (int dt = 0; dt < NV; ++dt)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const uint16_t v = vp[(size_t)(32 * dt + 8 * (i >> 2) + (i & 3)) * a.BS];
            if (mp_wild(v)) o[dt][i] += bf2f(v);
          }
      }
    }
  }
  if (a.n_parts > 1) {
    if (hi == 0) {
      a.pml[part * 2] = m;
      a.pml[part * 2 + 1] = l;
    }
    float* po = a.po + part * V + 4 * hi;
#pragma unroll
    for (int dt = 0; dt < NV; ++dt)
#pragma unroll
      for (int i = 0; i < 16; i += 4)
        *reinterpret_cast<f32x4*>(po + 32 * dt + 2 * i) = f32x4{o[dt][i], o[dt][i + 1], o[dt][i + 2], o[dt][i + 3]};
    return;
  }
  if (a.sink) l += __builtin_amdgcn_exp2f(a.sink[head] * kLog2e - m);
  float f = 1.f / l;
  if (a.gate) f *= 1.f / (1.f + __expf(-a.gate[(size_t)(row0 + tt) * a.gs + head]));
  const size_t ob = (size_t)(row0 + tt) * HM * V + (size_t)head * V + 4 * hi;   // o[dt][i]: dim 32 dt + 8 (i >> 2) + 4 hi + (i & 3)
#pragma unroll
  for (int dt = 0; dt < NV; ++dt)
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      const size_t oo = ob + 32 * dt + 2 * i;
      if (a.out32)
        *reinterpret_cast<f32x4*>(a.out32 + oo) = f32x4{o[dt][i] * f, o[dt][i + 1] * f, o[dt][i + 2] * f, o[dt][i + 3] * f};
      else
        *reinterpret_cast<u16x4*>(a.out + oo) =
            u16x4{f2bf(o[dt][i] * f), f2bf(o[dt][i + 1] * f), f2bf(o[dt][i + 2] * f), f2bf(o[dt][i + 3] * f)};
    }
}

// Joins the parts of a (row, head).  S threads share four of its columns (W such groups to a row), each takes every S-th part;
// theirs are joined in order.  S = 1 where the parts are few; eight for the many parts of few rows.
template <int S>
__global__ void __launch_bounds__(256) mask_prompt_merge_kernel(MaskPromptArgs a, size_t n4, int W) {
  constexpr float kLog2e = 1.4426950408889634f;
  __shared__ f32x4 sacc[S > 1 ? 256 : 1];
  __shared__ float sml[S > 1 ? 256 : 1][2];
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) / S;
  const int s = threadIdx.x % S, HM = a.H * a.M, n = a.n_parts;
  const bool on = i < n4;
  const size_t rh = (on ? i : 0) / W, row = a.row_base + rh / HM;
  const int head = rh % HM, c = (on ? i : 0) - rh * W;
  const float* ml = a.pml + rh * n * 2;
  const f32x4* po = reinterpret_cast<const f32x4*>(a.po) + rh * n * W + c;
  float M = -INFINITY, L = 0.f;
#pragma unroll 8
  for (int p = s; p < n; p += S) M = fmaxf(M, ml[2 * p]);
  if (S == 1 && a.sink) M = fmaxf(M, a.sink[head] * kLog2e);
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  const float Ms = M == -INFINITY ? 0.f : M;
#pragma unroll 8
  for (int p = s; p < n; p += S) {
    const float l = ml[2 * p + 1], f = __builtin_amdgcn_exp2f(ml[2 * p] - Ms);
    const f32x4 v = po[(size_t)p * W];
    L = fmaf(l, f, L);
#pragma unroll
    for (int k = 0; k < 4; ++k) acc[k] = l == 0.f ? acc[k] : fmaf(v[k], f, acc[k]);   // (l 0: a part this row sees no key of)
  }
  if (S > 1) {
    sacc[threadIdx.x] = acc;
    sml[threadIdx.x][0] = M;
    sml[threadIdx.x][1] = L;
    __syncthreads();
    if (s > 0) return;
    if (a.sink) M = fmaxf(M, a.sink[head] * kLog2e);
#pragma unroll
    for (int k = 1; k < S; ++k) M = fmaxf(M, sml[threadIdx.x + k][0]);
  }
  if (!on) return;
  const float Mt = M == -INFINITY ? 0.f : M;
  if (S > 1) {
    L = 0.f;
    acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < S; ++k) {
      const float f = __builtin_amdgcn_exp2f(sml[threadIdx.x + k][0] - Mt), l = sml[threadIdx.x + k][1];
      L = fmaf(l, f, L);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = l == 0.f ? acc[j] : fmaf(sacc[threadIdx.x + k][j], f, acc[j]);
    }
  }
  if (a.sink) L += __builtin_amdgcn_exp2f(a.sink[head] * kLog2e - Mt);
  float f = 1.f / L;
  if (a.gate) f *= 1.f / (1.f + __expf(-a.gate[row * a.gs + head]));
  const size_t o = (row * HM + head) * W * 4 + 4 * c;
  if (a.out32)
    *reinterpret_cast<f32x4*>(a.out32 + o) = f32x4{acc[0] * f, acc[1] * f, acc[2] * f, acc[3] * f};
  else
    *reinterpret_cast<u16x4*>(a.out + o) = u16x4{f2bf(acc[0] * f), f2bf(acc[1] * f), f2bf(acc[2] * f), f2bf(acc[3] * f)};
}

template <int ND, int NV, int NW>
static int launch_mp(const MaskPromptArgs& a, int rows, hipStream_t s) {
  const int hpg = a.H / a.G, hw = hpg < 32 * NW ? hpg : 32 * NW;
  const dim3 grid(a.n_items * a.G * a.M * ((hpg + hw - 1) / hw), a.n_parts);
#define K8S_MP(CAP, HALF) \
  hipLaunchKernelGGL((mask_prompt_kernel<ND, NV, NW, CAP, HALF>), grid, dim3(64 * NW), 0, s, a)
  if (a.softcap > 0.f) {
    if (a.BS % 64) K8S_MP(true, true);
    else K8S_MP(true, false);
  } else {
    if (a.BS % 64) K8S_MP(false, true);
    else K8S_MP(false, false);
  }
#undef K8S_MP
  if (a.n_parts == 1) return (int)hipGetLastError();
  const size_t n4 = (size_t)rows * a.H * a.M * NV * 8;
  if (a.n_parts <= 8)
    hipLaunchKernelGGL(mask_prompt_merge_kernel<1>, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, a, n4, NV * 8);
  else
    hipLaunchKernelGGL(mask_prompt_merge_kernel<8>, dim3((unsigned)((n4 + 31) / 32)), dim3(256), 0, s, a, n4, NV * 8);
  return (int)hipGetLastError();
}

}  // namespace k8s

using namespace k8s;

K8S_API int k8s_masked_attn_mfma_ok(int H, int G, int D, int V);

// Items of up to max(1, 128 / (H / G)) tokens.  n_parts > 1: the items are the rows row_base .. row_base + rows of the step,
// each tile's list of 64-key blocks is cut into parts of part_blocks (the last part takes what is left);
// po [rows][H maps][n_parts][V], pml [.. ][2].
K8S_API int k8s_masked_attn_prompt(const void* q, const void* kc, const void* vt, const int* bt, int maxb, const int* items,
                                   int n_items, const float* sink, const float* gate, int gs, void* out, int H, int G,
                                   int D, int V, int BS, int chunk, int window, int keep_first, float scale, float softcap,
                                   hipStream_t s, int maps, int out_f32, int n_parts, int part_blocks, int row_base, int rows,
                                   float* po, float* pml) {
  if (n_items <= 0) return 0;
  if (!k8s_masked_attn_mfma_ok(H, G, D, V) || BS % 32 || chunk < 0 || window < 0 || keep_first < 0 || maps < 1 ||
      n_parts < 1 || (n_parts > 1 && (part_blocks < 1 || rows < 1 || row_base < 0 || !po || !pml)))
    return (int)hipErrorInvalidValue;
  MaskPromptArgs a;
  a.q = (const uint16_t*)q; a.kc = (const uint16_t*)kc; a.vt = (const uint16_t*)vt; a.bt = bt; a.maxb = maxb;
  a.items = items; a.n_items = n_items; a.sink = sink; a.gate = gate; a.gs = gs;
  a.out = out_f32 ? nullptr : (uint16_t*)out; a.out32 = out_f32 ? (float*)out : nullptr;
  a.H = H; a.G = G; a.M = maps; a.BS = BS; a.chunk = chunk; a.window = window; a.keep_first = keep_first;
  a.scale = scale; a.softcap = softcap;
  a.n_parts = n_parts; a.part_blocks = n_parts > 1 ? part_blocks : 1 << 30; a.row_base = row_base; a.po = po; a.pml = pml;
  if (D == 96) return launch_mp<6, 3, 4>(a, rows, s);
  if (D == 64 && V == 64) return launch_mp<4, 2, 4>(a, rows, s);
  if (D == 64 && V == 128) return launch_mp<4, 4, 4>(a, rows, s);
  if (D == 128 && V == 64) return launch_mp<8, 2, 4>(a, rows, s);
  return launch_mp<8, 4, 4>(a, rows, s);
}
