// Attention over a paged LATENT cache (one vector of R numbers per token, shared
// by every head): the keys' and values' up-projections are moved to the query and
// output side, so a head's query is qa[h] = W_uk[h]^T q[h] (R numbers), its
// score against token j is scale * qa[h] . c_j, and its output in latent space
// is sum_j p_j c_j; the caller applies W_uv[h] afterwards.  All heads of a token
// read the same keys once.  Causal softmax in fp32; the optional per-head output gate
// sigmoid(gate[t][h]) is applied here (it commutes with W_uv).
//
// A cache row may hold RP more numbers behind the latent, a key part shared by all heads (the rotated
// one): a head's query then has RP more entries qr[t][h] and the score is scale * (qa[h] . c_j + qr[h] . k_j);
// the values stay the latents alone.  window > 0: position i sees j with i - j < window.  sink (optional) [H]:
// exp(sink_h) is added to head h's denominator, without a key or a value.
//
// Rows are addressed through the step's segments (seq_ops.hip): row r of segment
// s is the token at position seg_pos0[s] + r - seg_row0[s] and sees keys 0 .. that
// position, read through block table row s ([n_seg][maxb] pages of BS tokens).  This file: the matrix-core form;
// rows_attn.hip has the one on the vector pipes.
#include "common.h"

namespace k8s {

// ---------------------------------------------------------------------------
// MFMA form (bf16): v_mfma_f32_16x16x32_bf16, one wave per work item.
//
// The latents are cached twice: c [pages][BS][R] (a key's R numbers contiguous:
// the QK^T operand) and ct [pages][R][BS] (8 consecutive keys of one latent
// column contiguous: the PV operand), as the K / transposed-V pages of the
// head-wise attention kernels.  A wave owns MT tiles of 16 query rows; a tile is
// TPM consecutive tokens x HC heads (HC = min(H, 16), TPM = 16 / HC), so all its
// rows read the same keys.  Keys go in chunks of 32 (never across a page:
// BS % 32 == 0).  Swapped QK^T (S^T = C Q^T): a lane owns ONE query row
// (lane & 15) and 8 of its key scores; MFMA row rho of key tile t holds key
// 8 (rho >> 2) + 4 t + (rho & 3), so lane quarter h ends with keys 8h .. 8h + 7,
// the k-slots of the PV operand: P moves from accumulator to operand in place.
//
// Items ([n][4] int32: segment, first row, tokens, position of the first row's
// token) are made on the host from the step's segments: a wave walks every key its
// rows see and writes the gated, normalised output.  Decode rows: token_attn.hip.
//
// NP: 32-number chunks of the cache row behind the latent (a score-only key part): row width R + 32 NP.
constexpr float kLog2e = 1.4426950408889634f;

struct LatArgs {
  const uint16_t* qa;     // element (t, h, c) at t * qst + h * qsh + c
  long qst, qsh;
  const uint16_t* qr;     // [T][H][32 NP]
  const uint16_t* c;      // [pages][BS][R + 32 NP]
  const uint16_t* ct;     // [pages][R][BS]
  const int* bt;
  int maxb;
  const int* items;
  int n_items;
  const float* gate;      // or null
  int ldg;
  const float* sink;      // [H] or null
  int window;             // 0: every key up to the row's own position
  uint16_t* out;          // element (t, h, c) at t * ost + h * osh + c
  long ost, osh;
  int H, HC, TPM, BS;
  float scale_log2;
};

typedef __attribute__((address_space(3))) void lds_void_t;

__device__ __forceinline__ bf16x8 ld16(const uint16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }

// One tile of 16 query rows meets 32 keys (scores s[2], keys kb + 8 h + 4 t + i): online softmax in log2 units.
// The weights go to pf (the PV product's operand); the accumulator o is rescaled only where a maximum moved.
template <int ND>
__device__ __forceinline__ void lat_softmax(const f32x4 (&s)[2], float scale_log2, bool open, int kb, int h, int lo,
                                            int limit, float& m, float& l, f32x4 (&o)[ND], bf16x8& pf) {
  float p[8];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) p[4 * t + i] = s[t][i] * scale_log2;
  if (!open) {                                             // (a wave-uniform branch)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int key = kb + 8 * h + j;
      p[j] = key < limit && key >= lo ? p[j] : -INFINITY;
    }
  }
  float cmax = p[0];
#pragma unroll
  for (int j = 1; j < 8; ++j) cmax = fmaxf(cmax, p[j]);
  cmax = fmaxf(cmax, __shfl_xor(cmax, 16, 64));
  cmax = fmaxf(cmax, __shfl_xor(cmax, 32, 64));
  const bool grow = cmax > m;
  const float mn = grow ? cmax : m, ms = mn == -INFINITY ? 0.f : mn;    // -inf: a row that has seen no key yet
  float psum = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float e = __builtin_amdgcn_exp2f(p[j] - ms);
    psum += e;
    pf[j] = (__bf16)e;
  }
  if (__any(grow)) {
    const float alpha = __builtin_amdgcn_exp2f(m - ms);
    l *= alpha;
    m = mn;
    float ar[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ar[i] = __shfl(alpha, 4 * h + i, 64);
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[dt][i] *= ar[i];
  }
  l += psum;
}

// Prompt portions: the four waves of a workgroup own four consecutive items of ONE
// segment (the host pads every segment's items to a multiple of four with empty
// ones), so they read the same keys.  A chunk's operand fragments do not depend on
// the item: kf[t][cc] and vf[dt] go from global memory to LDS once per workgroup, without
// a register between (a quarter by each wave) -- slot f holds the 64
// lanes' 16 bytes, row by row, a row's four pieces swapped so that reads are
// conflict-free -- and are read by all four waves.  Two buffers: chunk i + 1 is asked for when chunk i begins and its page number
// one chunk earlier; one barrier per chunk.
//
// What bounds it: one tile of 16 rows uses a fragment once, so a wave waits for LDS between its batches, and beside 576
// cycles of matrix instructions a chunk has some 480 of softmax.  16384 rows of 16 heads over a window of 1024 keys, R 256 +
// 64: 596 us with fragments through registers and two reads in flight, 550 with LDS-DMA, batches of eight and the page number
// early (4 and 12 a batch the same), 453 with a row's 64 bytes in four lanes that follow each other (in fragment order they
// lie 16 apart and each is a lookup of its own in the first-level cache); 3517 and 4351 rows 107 -> 96 -> 87 and 183 -> 157
// -> 149.  Not quicker: two tiles a wave and one wave a SIMD (669 before the last change), eight waves to a workgroup that
// share the keys of 8 items (495: all wait at one barrier), a row's 128 bytes in eight lanes (465).
// With two tiles (R up to 128) a fragment is used twice and more workgroups share a compute unit, so that registers count: us
// through registers / batches of 8 / 4 / 2: 16 heads of R 64, two of 4000 rows 208 / 247 / 234 / 187; 24 heads of 96, 3000 rows
// behind 1000 199 / 270 / 185 / 184; 16 heads of 96 + 64, 16 of 700 73 / 68 / 65 / 57.
template <int NR, int NP, int MT, int OCC>
__global__ void __launch_bounds__(256, OCC) latent_attn_mfma_lds_kernel(LatArgs a) {
  constexpr int R = NR * 32, ND = R / 16, NC = NR + NP, RW = R + 32 * NP, NF = 2 * NC + ND, NFW = (NF + 3) / 4;
  constexpr int BATCH = MT > 1 ? 2 : 8;                       // fragments that are read from LDS at once
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  bf16x8* frag = reinterpret_cast<bf16x8*>(lds_raw);          // [2][NF][64]
  __shared__ int kend_s[4], kbeg_s[4];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, h = lane >> 4;
  // ... and the LAST items of the range first: they see the most keys, so the short ones fill the tail
  const int per = gridDim.x >> 3;
  const int blk = (gridDim.x & 7) == 0 ? (blockIdx.x & 7) * per + (per - 1 - (blockIdx.x >> 3))
                                       : gridDim.x - 1 - blockIdx.x;
  const int item0 = blk * 4;
  if (item0 >= a.n_items) return;                              // whole workgroup
  const int item = item0 + wv;
  const int sg = a.items[item0 * 4];
  const int row0 = a.items[item * 4 + 1], ntok = a.items[item * 4 + 2], pos0 = a.items[item * 4 + 3];
  const int hc = blockIdx.z;
  if (lane == 0) {
    kend_s[wv] = ntok > 0 ? pos0 + ntok : 0;
    kbeg_s[wv] = ntok > 0 ? (a.window > 0 ? max(0, pos0 - a.window + 1) : 0) : 0x7fffffff;
  }
  __syncthreads();
  const int k_end = max(max(kend_s[0], kend_s[1]), max(kend_s[2], kend_s[3]));
  const int k_beg = min(min(kbeg_s[0], kbeg_s[1]), min(kbeg_s[2], kbeg_s[3])) & ~31;
  const int tl = r / a.HC, hl = r - tl * a.HC, head = hc * a.HC + hl;
  bf16x8 qf[MT][NC];
  int limit[MT], lo[MT];
  f32x4 o[MT][ND];
  float m[MT], l[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int ti = mt * a.TPM + tl;
    const bool valid = tl < a.TPM && ti < ntok && head < a.H;
    limit[mt] = valid ? pos0 + ti + 1 : 0;
    lo[mt] = a.window > 0 ? pos0 + ti - a.window + 1 : 0;
    const size_t rq = row0 + (valid ? ti : 0), hq = valid ? head : 0;
#pragma unroll
    for (int cc = 0; cc < NC; ++cc) {
      qf[mt][cc] = ld16(cc < NR ? a.qa + rq * a.qst + hq * a.qsh + 32 * cc + 8 * h
                                : a.qr + (rq * a.H + hq) * (32 * NP) + 32 * (cc - NR) + 8 * h);
      if (!valid)
#pragma unroll
        for (int j = 0; j < 8; ++j) qf[mt][cc][j] = (__bf16)0.f;
    }
#pragma unroll
    for (int dt = 0; dt < ND; ++dt) o[mt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[mt] = (a.sink && valid) ? a.sink[head] * kLog2e : -INFINITY;
    l[mt] = 0.f;
  }
  const int* pages = a.bt + (size_t)sg * a.maxb;
  // this wave's share of a chunk's fragments, f = wv + 4 i, straight into LDS (lane l's 16 bytes at 16 l of the slot): four
  // lanes take a row's 64 bytes, in an order that spreads a column of eight rows over all banks; a fragment's lane reads at
  const int lr = lane >> 2, lh = (lane & 3) ^ ((lr >> 1) & 3);
  const int at = 4 * r + (h ^ ((r >> 1) & 3));
  auto fetch = [&](int kb, int page, int buf) {
    const int off = kb % a.BS;
    const uint16_t* cp = a.c + (size_t)page * a.BS * RW;
    const uint16_t* tp = a.ct + (size_t)page * R * a.BS;
#pragma unroll
    for (int i = 0; i < NFW; ++i) {
      const int f = wv + 4 * i;
      if (NF % 4 && f >= NF) continue;
      const uint16_t* src;
      if (f < 2 * NC) {
        const int t = f / NC, cc = f - t * NC;
        src = cp + (size_t)(off + 8 * (lr >> 2) + 4 * t + (lr & 3)) * RW + 32 * cc + 8 * lh;
      } else {
        src = tp + (size_t)(16 * (f - 2 * NC) + lr) * a.BS + off + 8 * lh;
      }
      __builtin_amdgcn_global_load_lds(src, (lds_void_t*)(frag + ((size_t)buf * NF + f) * 64), 16, 0, 0);
    }
  };
  auto landed = [&]() {                                       // this wave's share is there; then every wave's
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto page_of = [&](int kb) { return pages[min(kb, k_end - 1) / a.BS]; };
  int page = 0;
  if (k_beg < k_end) {
    fetch(k_beg, page_of(k_beg), 0);
    page = page_of(k_beg + 32);
  }
  // The fragments in the order of their use: keys (both tiles in turn), then values; batches, the next one asked for
  // once the first of a batch is there -- the compiler waits for all LDS reads in flight where LDS-DMA is about.
  auto slot = [](int j) { return j < 2 * NC ? (j & 1) * NC + (j >> 1) : j; };
  int buf = 0;
  for (int kb = k_beg; kb < k_end; kb += 32, buf ^= 1) {
    landed();                                                 // (and nobody reads the other buffer any more)
    if (kb + 32 < k_end) fetch(kb + 32, page, buf ^ 1);
    page = page_of(kb + 64);                                  // there with that chunk
    const bf16x8* fb = frag + (size_t)buf * NF * 64 + at;
    const bool open = kb + 31 <= pos0 && (a.window <= 0 || kb >= pos0 + ntok - a.window);
    f32x4 s[MT][2];
    bf16x8 pf[MT], fr[2][BATCH];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) s[mt][0] = s[mt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto read = [&](int b) {
#pragma unroll
      for (int i = 0; i < BATCH; ++i)
        if (b * BATCH + i < NF) fr[b & 1][i] = fb[slot(b * BATCH + i) * 64];
    };
    read(0);
#pragma unroll
    for (int b = 0; b * BATCH < NF; ++b) {
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        const int j = b * BATCH + i;
        if (j >= NF) continue;
        if (j == 2 * NC) {
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            lat_softmax<ND>(s[mt], a.scale_log2, open, kb, h, lo[mt], limit[mt], m[mt], l[mt], o[mt], pf[mt]);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          if (j < 2 * NC)
            s[mt][j & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fr[b & 1][i], qf[mt][j >> 1], s[mt][j & 1], 0, 0, 0);
          else
            o[mt][j - 2 * NC] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[mt], fr[b & 1][i], o[mt][j - 2 * NC], 0, 0, 0);
        }
        if (i == 0) {
          __builtin_amdgcn_sched_barrier(0);
          if ((b + 1) * BATCH < NF) read(b + 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    float lt = l[mt];
    lt += __shfl_xor(lt, 16, 64);
    lt += __shfl_xor(lt, 32, 64);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = 4 * h + i;
      const int qtl = q / a.HC, qhl = q - qtl * a.HC, qhead = hc * a.HC + qhl, ti = mt * a.TPM + qtl;
      const float lq = __shfl(lt, q, 64), mq = __shfl(m[mt], q, 64);
      if (!(qtl < a.TPM && ti < ntok && qhead < a.H)) continue;
      const float g = a.gate ? 1.f / (1.f + expf(-a.gate[(size_t)(row0 + ti) * a.ldg + qhead])) : 1.f;
      const float ls = a.sink ? lq + __builtin_amdgcn_exp2f(a.sink[qhead] * kLog2e - mq) : lq;
      const float sc = ls > 0.f ? g / ls : 0.f;
      uint16_t* op = a.out + (size_t)(row0 + ti) * a.ost + (size_t)qhead * a.osh + r;
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) op[16 * dt] = f2bf(o[mt][dt][i] * sc);
    }
  }
}

template <int NR, int NP>
static int launch_lat_np(const LatArgs& a, int n_head_chunks, hipStream_t s) {
  int nblk = (a.n_items + 3) / 4;
  if (nblk > 8) nblk = (nblk + 7) & ~7;   // a multiple of the XCD count (the kernels' item remap)
  const dim3 grid(nblk, 1, n_head_chunks);
  if (a.n_items % 4) return (int)hipErrorInvalidValue;   // prompt items come in fours per segment
  constexpr size_t lds = 2 * (size_t)(4 * NR + 2 * NP) * 64 * 16;  // two buffers of 2 (NR + NP) + R / 16 KiB
  // tiles per wave and waves per SIMD by register need: two tiles while two waves still fit a SIMD
  // (R <= 128), one tile and two waves at R = 192 / 256, one and one above
  constexpr int MT = NR <= 4 ? 2 : 1, OCC = NR <= 8 ? 2 : 1;
  auto k = latent_attn_mfma_lds_kernel<NR, NP, MT, OCC>;
  if (lds > 48 * 1024 && hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds))
    return (int)hipGetLastError();
  hipLaunchKernelGGL(k, grid, dim3(256), lds, s, a);
  return (int)hipGetLastError();
}

template <int NR>
static int launch_lat(const LatArgs& a, int np, int n_head_chunks, hipStream_t s) {
  switch (np) {
    case 0: return launch_lat_np<NR, 0>(a, n_head_chunks, s);
    case 1: return launch_lat_np<NR, 1>(a, n_head_chunks, s);
    case 2: return launch_lat_np<NR, 2>(a, n_head_chunks, s);
    default: return (int)hipErrorInvalidValue;
  }
}

}  // namespace k8s

// 0: the MFMA kernels do not take latent rank R; else the tiles per wave for prompt portions (2 up to R = 128).
// RP: the score-only numbers of a cache row behind the latent (a multiple of 32 up to 64).
K8S_API int k8s_latent_attn_mfma_ok(int R, int RP) {
  if (RP != 0 && RP != 32 && RP != 64) return 0;
  switch (R) {
    case 32: case 64: case 96: case 128: return 2;
    case 192: case 256: case 384: case 512: return 1;
    default: return 0;
  }
}

// Items of up to k8s_latent_attn_mfma_ok() * (16 / min(H, 16)) tokens, in fours per segment.
K8S_API int k8s_latent_attn_mfma(const void* qa, const void* c, const void* ct, const int* bt, int maxb,
                                 const int* items, int n_items, const float* gate, int ldg, void* out, int H, int R,
                                 int BS, float scale, hipStream_t s, long qst, long qsh, const void* qr, int RP, long ost, long osh,
                                 int window, const float* sink) {
  if (n_items <= 0) return 0;
  if (!k8s_latent_attn_mfma_ok(R, RP) || BS % 32 || H <= 0 || (RP && !qr) || window < 0 ||
      qst % 8 || qsh % 8)
    return (int)hipErrorInvalidValue;
  k8s::LatArgs a;
  a.qst = qst; a.qsh = qsh; a.qr = (const uint16_t*)qr; a.ost = ost; a.osh = osh; a.window = window; a.sink = sink;
  a.qa = (const uint16_t*)qa; a.c = (const uint16_t*)c; a.ct = (const uint16_t*)ct; a.bt = bt; a.maxb = maxb;
  a.items = items; a.n_items = n_items; a.gate = gate; a.ldg = ldg; a.out = (uint16_t*)out;
  a.H = H; a.HC = H < 16 ? H : 16; a.TPM = 16 / a.HC; a.BS = BS; a.scale_log2 = scale * k8s::kLog2e;
  const int nhc = (H + a.HC - 1) / a.HC;
  int rc;
  switch (R / 32) {
    case 1: rc = k8s::launch_lat<1>(a, RP / 32, nhc, s); break;
    case 2: rc = k8s::launch_lat<2>(a, RP / 32, nhc, s); break;
    case 3: rc = k8s::launch_lat<3>(a, RP / 32, nhc, s); break;
    case 4: rc = k8s::launch_lat<4>(a, RP / 32, nhc, s); break;
    case 6: rc = k8s::launch_lat<6>(a, RP / 32, nhc, s); break;
    case 8: rc = k8s::launch_lat<8>(a, RP / 32, nhc, s); break;
    case 12: rc = k8s::launch_lat<12>(a, RP / 32, nhc, s); break;
    case 16: rc = k8s::launch_lat<16>(a, RP / 32, nhc, s); break;
    default: return (int)hipErrorInvalidValue;
  }
  return rc;
}
