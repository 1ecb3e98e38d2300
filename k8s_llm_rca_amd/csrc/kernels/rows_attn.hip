// Softmax attention of single rows over paged keys and values on the vector pipes, fp32 arithmetic: fp32 models, and head
// sizes the matrix-core kernels do not take.  The masks are masked_attn.hip's, the latent form latent_attn.hip's: there all
// heads share a cache row of W = R + RP numbers, which is the key, and whose first R numbers are the value.
//
// A row's visible keys are cut into parts of 128 by their place in its own key range.  Within a part the scores of up to
// eight heads (two where workgroups are few) of one key head meet in LDS -- four (two) lanes beside each other have a
// key, so that they read the same 16 bytes of it, and a quarter (half) of the heads each -- then their softmax, then a
// thread walks the part's keys for one value column and the heads again.  Parts are joined in order with fixed
// multiply-adds, by the workgroup itself where there are rows enough to fill the chip, by a second kernel where few rows are
// spread over a workgroup per part: both do the same arithmetic, so a row's result does not depend on how the prompt was cut
// or on what else is in the step.
//
// What bounds it (prompts in fp32 with whole tiles go to rows_attn_mfma_kernel): the scores -- lookups of the first-level
// cache, one for every key that four neighbouring lanes read -- and
// latency at few rows, for which reason the heads and the parts are spread over workgroups.  622 rows of two prompts, 16
// heads, 256 + 64 numbers and 2 key heads of 128, median of both: a lane a key, four keys in four lanes, 150 us; three
// workgroups a compute unit by their registers and 16 values on their way 126; two lanes a key 106; four lanes a key, two
// keys each, and four workgroups 98 (one register spilled; three without a spill 105).  fp32, 16 heads over 2 of 128, two
// rows at 340 keys: 980 us (a workgroup per row, all heads one after the other, the scores formed twice) -> 28 us; 666 rows
// of two prompts: 1451 -> 122 us; latent (16 heads, 256 + 64 numbers): 706 -> 39 and 719 -> 196 us.
#include "common.h"
#include "key_runs.h"
#include <type_traits>

namespace k8s {

constexpr int kRaKeys = 128;    // keys of a part
constexpr int kRaHeads = 8;     // heads of a workgroup
constexpr int kRaFew = 2;       // of one that has a single part, where few of them run
constexpr int kRaAsk = 16;      // values of a column asked for together with eight heads

template <typename T>
__device__ __forceinline__ float rld(const T* p, size_t i);
template <>
__device__ __forceinline__ float rld<float>(const float* p, size_t i) { return p[i]; }
template <>
__device__ __forceinline__ float rld<uint16_t>(const uint16_t* p, size_t i) { return bf2f(p[i]); }
template <typename T>
__device__ __forceinline__ void rst(T* p, size_t i, float v);
template <>
__device__ __forceinline__ void rst<float>(float* p, size_t i, float v) { p[i] = v; }
template <>
__device__ __forceinline__ void rst<uint16_t>(uint16_t* p, size_t i, float v) { p[i] = f2bf(v); }
__device__ __forceinline__ f32x4 rld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 rld4(const uint16_t* p) {
  const u16x4 v = *reinterpret_cast<const u16x4*>(p);
  return f32x4{bf2f(v[0]), bf2f(v[1]), bf2f(v[2]), bf2f(v[3])};
}

struct RowsArgs {
  const void* q;               // entry d < D1 of head h of row t at t * qst + h * qsh + d
  long qst, qsh;
  const float* q2;             // entries D1 .. D1 + D2 at (t * H + h) * D2 (latent form)
  int D1, D2;
  const void* kc;              // a key's entries of key head i at slot * ks + i * D
  const void* vc;              // a value's of value head g at slot * vs + g * V
  int ks, vs;
  const int* bt;
  int maxb;
  const int* row_seg;
  const int* seg_row0;
  const int* seg_pos0;
  const float* sink;
  const float* gate;
  int gs;
  void* out;                   // entry c of head h of row t at t * ost + h * osh + c
  long ost, osh;
  int H, G, M, V, BS;          // H counts heads x maps
  int row_base, chunk, window, keep_first;
  float scale, softcap;
  float* po;                   // [T][H][n_parts][V], null: the workgroup joins the parts
  float* pml;                  // [T][H][n_parts][2]
  int n_parts;
};

// (m, l) and the outputs of a further part; both maxima may be -inf (no key yet, a part whose scores all are)
__device__ __forceinline__ void ra_join(float& m, float& l, float mp, float lp, float& a, float& b) {
  const float mn = fmaxf(m, mp), ms = mn == -INFINITY ? 0.f : mn;
  a = expf(m - ms);
  b = expf(mp - ms);
  l = fmaf(l, a, __fmul_rn(lp, b));
  m = mn;
}
__device__ __forceinline__ float ra_join_out(float o, float a, float op, float b) { return fmaf(o, a, __fmul_rn(op, b)); }

// PART: a workgroup has one part (p.po).  FEW: and there are few of them, each a chain of latencies, so that all the registers
// are its own: every value of the part is asked for before the scores, and 16 pieces of a key at a time instead of 2; and two
// heads a workgroup, for with eight the multiply-adds and LDS reads of one compute unit are as long as the chain.  The sums are
// those of the other forms.  Reply steps of two rows at 340 keys, both attentions, median of a trace: 35.8 us -> 31.3
// (registers) -> 16.9 (two heads) -> 14.5 (two lanes a key).
// Few: up to 512 workgroups of two heads over fp32 pages and 256 over bf16 ones, which need more registers: what runs at
// once.  Past that they go in turns and read each key four times as often.  us with the merge, eight heads / two, 16 heads
// over 2 of 128: 7 rows at 800 keys (392) 25.7 / 23.6 fp32, 26.1 / 28.4 bf16; 12 at 700 (576) 25.6 / 28.6, 25.4 / 36.0; 32 heads
// over 2 of 64: 32 rows at 500 (2048) 23.4 / 44.7, 23.3 / 77.0; 4 at 500 (256) 21.3 / 19.6, 22.1 / 20.3.
template <typename TQ, typename TC, typename TO, bool VEC, bool PART, bool FEW>
__global__ void __launch_bounds__(256, FEW ? 1 : 4) rows_attn_kernel(RowsArgs p) {
  constexpr int NH = FEW ? kRaFew : kRaHeads;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int D = p.D1 + p.D2, V = p.V, hpg = p.H / (p.G * p.M);
  const int HB = min(hpg, NH), nhb = (hpg + HB - 1) / HB, nvb = (V + 255) / 256;
  float* sq = sm;                                   // [HB][D4]
  const int D4 = ((D + 3) & ~3) + 4;                // (neighbouring heads' rows in different banks)
  float* sp = sq + HB * D4;                         // [HB][128]
  float* sl = sp + HB * kRaKeys;                    // [HB][2]: m, l of the part
  int* ss = reinterpret_cast<int*>(sl + 2 * HB);    // [128]: cache slots
  const int r = p.row_base + blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int gi = blockIdx.y;
  const int vb = gi % nvb;
  gi /= nvb;
  const int hb = gi % nhb, gm = gi / nhb, g = gm / p.M;
  const int nh = min(HB, hpg - hb * HB);
  auto head = [&](int i) { return (g * hpg + hb * HB + i) * p.M + gm % p.M; };
  const int sg = p.row_seg[r], pos = p.seg_pos0[sg] + r - p.seg_row0[sg];
  const KeyRuns kr = key_runs(pos, p.chunk, p.window, p.keep_first);
  const int x_lo = PART ? blockIdx.z * kRaKeys : 0, x_hi = PART ? min(kr.total, x_lo + kRaKeys) : kr.total;
  if (x_lo >= x_hi) return;
  const int* bt = p.bt + (size_t)sg * p.maxb;
  for (int i = tid; i < nh * D; i += 256) {
    const int h = i / D, d = i - h * D;
    sq[h * D4 + d] = d < p.D1 ? rld((const TQ*)p.q, (size_t)r * p.qst + (size_t)head(h) * p.qsh + d)
                              : p.q2[((size_t)r * p.H + head(h)) * p.D2 + d - p.D1];
  }
  // this thread's value column and heads
  const int v0 = vb * 256, vc = min(V - v0, 256), tpc = 256 / vc, hs = tid / vc, col = tid - hs * vc;
  const bool own = hs < tpc;
  const TC* kbase = (const TC*)p.kc + (size_t)gm * D;
  const TC* vbase = (const TC*)p.vc + (size_t)g * V + v0 + col;
  float m[NH], l[NH], o[NH];      // of head hs + k tpc
#pragma unroll
  for (int k = 0; k < NH; ++k) {
    const int h = hs + k * tpc;
    const bool on = own && h < nh && p.sink && !PART;
    m[k] = on ? p.sink[head(h)] : -INFINITY;
    l[k] = on ? 1.f : 0.f;
    o[k] = 0.f;
  }
  for (int x0 = x_lo; x0 < x_hi; x0 += kRaKeys) {
    const int nk = min(kRaKeys, x_hi - x0);
    __syncthreads();                                // the part before is read no more
    if (tid < kRaKeys) {
      const int j = kr.key(x0 + min(tid, nk - 1));
      ss[tid] = bt[j / p.BS] * p.BS + j % p.BS;
    }
    __syncthreads();
    TC vall[FEW ? kRaKeys : 1];
    if constexpr (FEW) {
      if (own) {
#pragma unroll
        for (int j = 0; j < kRaKeys; ++j) vall[j] = vbase[(size_t)ss[j] * p.vs];      // (past nk: the last one again)
      }
    }
    {  // scores: HL lanes beside each other have a key (KX of them), each every HL-th head
      constexpr int HL = FEW ? 2 : 4, KW = 64 / HL, KX = kRaKeys / (4 * KW), HP = NH / HL;
      const int x = wv * KW + lane / HL, h0 = lane % HL;
      if (wv * KW < nk && h0 < nh) {
        const TC* kp[KX];
#pragma unroll
        for (int i = 0; i < KX; ++i) kp[i] = kbase + (size_t)ss[x + 4 * KW * i] * p.ks;
        const float* q0 = sq + h0 * D4;
        const float* qh[HP];
#pragma unroll
        for (int k = 0; k < HP; ++k) qh[k] = h0 + HL * k < nh ? q0 + HL * k * D4 : q0;
        float a[HP][KX] = {};
        if (VEC) {
#pragma unroll (FEW ? 16 : 2)
          for (int d = 0; d < D; d += 4) {
            f32x4 kv[KX];
#pragma unroll
            for (int i = 0; i < KX; ++i) kv[i] = rld4(kp[i] + d);
#pragma unroll
            for (int k = 0; k < HP; ++k) {
              const f32x4 qv = *reinterpret_cast<const f32x4*>(qh[k] + d);
#pragma unroll
              for (int i = 0; i < KX; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) a[k][i] = fmaf(qv[e], kv[i][e], a[k][i]);
            }
          }
        } else {
          for (int d = 0; d < D; ++d)
#pragma unroll
            for (int i = 0; i < KX; ++i) {
              const float kv = rld(kp[i], d);
#pragma unroll
              for (int k = 0; k < HP; ++k) a[k][i] = fmaf(qh[k][d], kv, a[k][i]);
            }
        }
#pragma unroll
        for (int k = 0; k < HP; ++k)
#pragma unroll
          for (int i = 0; i < KX; ++i)
            if (h0 + HL * k < nh) {
              float s = a[k][i] * p.scale;
              if (p.softcap > 0.f) s = p.softcap * tanhf(s / p.softcap);
              const int xi = x + 4 * KW * i;
              sp[(h0 + HL * k) * kRaKeys + xi] = xi < nk ? s : -INFINITY;
            }
      } else if (h0 < nh) {
        for (int h = h0; h < nh; h += HL)
          for (int i = 0; i < KX; ++i) sp[h * kRaKeys + x + 4 * KW * i] = -INFINITY;
      }
    }
    __syncthreads();
    for (int h = wv; h < nh; h += 4) {              // the part's softmax, a wave per head
      const float s0 = sp[h * kRaKeys + lane], s1 = sp[h * kRaKeys + 64 + lane];
      const float mp = wave_max(fmaxf(s0, s1)), ms = mp == -INFINITY ? 0.f : mp;
      const float e0 = expf(s0 - ms), e1 = expf(s1 - ms);
      sp[h * kRaKeys + lane] = e0;
      sp[h * kRaKeys + 64 + lane] = e1;
      const float lp = wave_sum(e0 + e1);
      if (lane == 0) {
        sl[2 * h] = mp;
        sl[2 * h + 1] = lp;
      }
    }
    __syncthreads();
    if (own) {
      float op[NH];
#pragma unroll
      for (int k = 0; k < NH; ++k) op[k] = 0.f;
      auto with = [&](int j, const float (&v)[4]) {  // keys j .. j + 3 of the part
#pragma unroll
        for (int k = 0; k < NH; ++k) {
          const int h = hs + k * tpc;
          if (h < nh) {
            const f32x4 w = *reinterpret_cast<const f32x4*>(sp + h * kRaKeys + j);
#pragma unroll
            for (int e = 0; e < 4; ++e) op[k] = fmaf(w[e], v[e], op[k]);
          }
        }
      };
      // (weights past nk are zero, and zero times an infinity would be NaN)
      if constexpr (FEW) {
#pragma unroll
        for (int j = 0; j < kRaKeys; j += 4)
          if (j < nk) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = j + e < nk ? rld(vall + j + e, 0) : 0.f;
            with(j, v);
          }
      } else {
        auto four = [&](int j, int n) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = e < n ? rld(vbase, (size_t)ss[j + e] * p.vs) : 0.f;
          with(j, v);
        };
        const int nk4 = nk & ~3;
        int j4 = 0;
        for (; j4 + kRaAsk <= nk4; j4 += kRaAsk) {          // their values on their way together
          float v[kRaAsk / 4][4];
#pragma unroll
          for (int e = 0; e < kRaAsk; ++e) v[e / 4][e % 4] = rld(vbase, (size_t)ss[j4 + e] * p.vs);
#pragma unroll
          for (int e = 0; e < kRaAsk; e += 4) with(j4 + e, v[e / 4]);
        }
        for (; j4 < nk4; j4 += 4) four(j4, 4);
        if (nk4 < nk) four(nk4, nk - nk4);
      }
#pragma unroll
      for (int k = 0; k < NH; ++k) {
        const int h = hs + k * tpc;
        if (h < nh) {
          if constexpr (PART) {
            const size_t at = ((size_t)blockIdx.x * p.H + head(h)) * p.n_parts + blockIdx.z;
            p.po[at * V + v0 + col] = op[k];
            if (col == 0 && vb == 0) {
              p.pml[at * 2] = sl[2 * h];
              p.pml[at * 2 + 1] = sl[2 * h + 1];
            }
          } else {
            float a, b;
            ra_join(m[k], l[k], sl[2 * h], sl[2 * h + 1], a, b);
            o[k] = ra_join_out(o[k], a, op[k], b);
          }
        }
      }
    }
  }
  if (PART || !own) return;
#pragma unroll
  for (int k = 0; k < NH; ++k) {
    const int h = hs + k * tpc;
    if (h < nh) {
      const int hh = head(h);
      float v = o[k] / l[k];
      if (p.gate) v *= 1.f / (1.f + expf(-p.gate[(size_t)r * p.gs + hh]));
      rst((TO*)p.out, (size_t)r * p.ost + (size_t)hh * p.osh + v0 + col, v);
    }
  }
}

// The same sums on the matrix units, fp32 throughout, for workgroups that walk all parts of a row: 16 heads are the rows of a
// tile, and its columns 16 keys, then 16 value columns.  A v_mfma_f32_16x16x4_f32 adds its four products one after the other,
// each with the rounding of a multiply-add, so a score and a value are the chains of rows_attn_kernel, to the bit.
// For that the four numbers of an instruction have to stand beside each other in the key: four lanes read 64 bytes of a key, so
// that it is looked up once per 16 numbers, and lane swaps turn the 4 x 4 of them.  Queries and weights stand in LDS as the lanes
// want them, four instructions' in 16 bytes.
// What bounds it: the chain of a part (slots, keys, softmax, values) with four to five workgroups a compute unit to cover it;
// matrix instructions are a third of the time (with 8 heads of a key half of each is empty).  us of rows_attn_kernel / here, 622
// rows of two prompts: 16 heads, 256 + 64 numbers 116 / 59;  16 heads over 2 of 128 67 / 42, over 16 of 64 190 / 121.  The
// next part's slots and the first 32 keys' values asked for in front of the scores: 65 -> 60 and 45 -> 42, 300 single rows at
// 500 keys 119 -> 82.  Eight waves, a tile of keys each: 69 and 51 (fewer workgroups at once), and with half of them for
// the values 65 and 64.
constexpr int kRmKeys = kRaKeys + 4;    // a head's weights in LDS: 16 heads' neighbours in 64 banks

// Where entry or key i of 16 stands in LDS: the four of an instruction's lane behind each other.
__device__ __forceinline__ int rm_at(int i) { return (i & ~15) | (i & 3) << 2 | (i >> 2 & 3); }

__device__ __forceinline__ void rm_turn(float& a, float& b, bool far) {
  const auto t = far ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                     : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(t[0]);
  b = __uint_as_float(t[1]);
}

template <int NE>
__global__ void __launch_bounds__(256, 4) rows_attn_mfma_kernel(RowsArgs p) {
  using cols = float __attribute__((ext_vector_type(NE)));
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int D = p.D1 + p.D2, V = p.V, hpg = p.H / (p.G * p.M), nhb = (hpg + 15) / 16, D4 = D + 4;
  constexpr int kAhead = 8;                         // times four keys: whose values are on their way together
  const int nvb = V / (64 * NE);
  float* sq = sm;                                   // [16][D4]
  float* sp = sq + 16 * D4;                         // [16][kRmKeys]
  float* sl = sp + 16 * kRmKeys;                    // [16][2]: m, l of the part
  int* slots = reinterpret_cast<int*>(sl + 32);     // [2][128]: cache slots of this part and the next
  const int r = p.row_base + blockIdx.x, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c16 = lane & 15, kg = lane >> 4;
  int gi = blockIdx.y;
  const int vb = gi % nvb;
  gi /= nvb;
  const int hb = gi % nhb, gm = gi / nhb, g = gm / p.M;
  const int nh = min(16, hpg - hb * 16);
  auto head = [&](int i) { return (g * hpg + hb * 16 + i) * p.M + gm % p.M; };
  const int sg = p.row_seg[r], pos = p.seg_pos0[sg] + r - p.seg_row0[sg];
  const KeyRuns kr = key_runs(pos, p.chunk, p.window, p.keep_first);
  const int* bt = p.bt + (size_t)sg * p.maxb;
  auto slot = [&](int x) {                          // (past the last key: that one again)
    const int j = kr.key(min(x, kr.total - 1));
    return bt[j / p.BS] * p.BS + j % p.BS;
  };
  if (tid < kRaKeys) slots[tid] = slot(tid);
  for (int i = tid; i < nh * D; i += 256) {
    const int h = i / D, d = i - h * D;
    sq[h * D4 + rm_at(d)] = d < p.D1 ? ((const float*)p.q)[(size_t)r * p.qst + (size_t)head(h) * p.qsh + d]
                                     : p.q2[((size_t)r * p.H + head(h)) * p.D2 + d - p.D1];
  }
  const int col = (vb * 4 + wv) * 16 * NE + c16 * NE;
  const float* kbase = (const float*)p.kc + (size_t)gm * D + 4 * kg;
  const float* vbase = (const float*)p.vc + (size_t)g * V + col;
  float m[4], l[4];                                 // of head 4 kg + i
  f32x4 o[NE];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool on = 4 * kg + i < nh && p.sink;
    m[i] = on ? p.sink[head(4 * kg + i)] : -INFINITY;
    l[i] = on ? 1.f : 0.f;
  }
#pragma unroll
  for (int e = 0; e < NE; ++e) o[e] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int x0 = 0, par = 0; x0 < kr.total; x0 += kRaKeys, par ^= 1) {
    const int nk = min(kRaKeys, kr.total - x0);
    const int* ss = slots + par * kRaKeys;
    __syncthreads();                                // slots (and queries) are there, the part before is read no more
    const int next = tid < kRaKeys && x0 + kRaKeys < kr.total ? slot(x0 + kRaKeys + tid) : 0;
    cols v[kAhead];                               // the first values, asked for in front of the scores
#pragma unroll
    for (int u = 0; u < kAhead; ++u) v[u] = *reinterpret_cast<const cols*>(vbase + (size_t)ss[4 * u + kg] * p.vs);
    {  // scores of keys 16 wv .. and 64 + 16 wv ..
      f32x4 a[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      const int x = 16 * wv + c16;
      const float* k0 = kbase + (size_t)ss[x] * p.ks;
      const float* k1 = kbase + (size_t)ss[x + 64] * p.ks;
      const float* qh = sq + c16 * D4 + 4 * kg;
      auto tiles = [&](auto both) {
        constexpr int NT = decltype(both)::value ? 2 : 1;
#pragma unroll 4
        for (int d = 0; d < D; d += 16) {
          f32x4 t[NT];
          t[0] = rld4(k0 + d);
          if constexpr (NT == 2) t[1] = rld4(k1 + d);
          const f32x4 qv = *reinterpret_cast<const f32x4*>(qh + d);
#pragma unroll
          for (int f = 0; f < NT; ++f) {
            float t0 = t[f][0], t1 = t[f][1], t2 = t[f][2], t3 = t[f][3];
            rm_turn(t0, t2, true);
            rm_turn(t1, t3, true);
            rm_turn(t0, t1, false);
            rm_turn(t2, t3, false);
            t[f] = f32x4{t0, t1, t2, t3};
          }
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int f = 0; f < NT; ++f) a[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[e], t[f][e], a[f], 0, 0, 0);
        }
      };
      if (64 + 16 * wv < nk)
        tiles(std::true_type{});
      else if (16 * wv < nk)
        tiles(std::false_type{});
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float s = a[f][i] * p.scale;
          if (p.softcap > 0.f) s = p.softcap * tanhf(s / p.softcap);
          sp[(4 * kg + i) * kRmKeys + rm_at(x) + 64 * f] = x + 64 * f < nk ? s : -INFINITY;
        }
    }
    if (tid < kRaKeys) slots[(par ^ 1) * kRaKeys + tid] = next;
    __syncthreads();
    for (int h = wv; h < nh; h += 4) {              // the part's softmax, a wave per head
      float* w = sp + h * kRmKeys + rm_at(lane);
      const float s0 = w[0], s1 = w[64];
      const float mp = wave_max(fmaxf(s0, s1)), ms = mp == -INFINITY ? 0.f : mp;
      const float e0 = expf(s0 - ms), e1 = expf(s1 - ms);
      w[0] = e0;
      w[64] = e1;
      const float lp = wave_sum(e0 + e1);
      if (lane == 0) {
        sl[2 * h] = mp;
        sl[2 * h + 1] = lp;
      }
    }
    __syncthreads();
    f32x4 op[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) op[e] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float* wp = sp + c16 * kRmKeys + 4 * kg;
    f32x4 w;
    for (int j0 = 0; j0 < nk; j0 += 4 * kAhead) {
      if (j0) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = *reinterpret_cast<const cols*>(vbase + (size_t)ss[j0 + 4 * u + kg] * p.vs);
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int j = j0 + 4 * u;
        if (j >= nk) break;
        if (u % 4 == 0) w = *reinterpret_cast<const f32x4*>(wp + j);
#pragma unroll
        for (int e = 0; e < NE; ++e)                // (weights past nk are zero, and zero times an infinity would be NaN)
          op[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u % 4], j + kg < nk ? v[u][e] : 0.f, op[e], 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int h = 4 * kg + i;
      if (h < nh) {
        float a, b;
        ra_join(m[i], l[i], sl[2 * h], sl[2 * h + 1], a, b);
#pragma unroll
        for (int e = 0; e < NE; ++e) o[e][i] = ra_join_out(o[e][i], a, op[e][i], b);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int h = 4 * kg + i;
    if (h < nh) {
      const int hh = head(h);
      cols v;
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        v[e] = o[e][i] / l[i];
        if (p.gate) v[e] *= 1.f / (1.f + expf(-p.gate[(size_t)r * p.gs + hh]));
      }
      *reinterpret_cast<cols*>((float*)p.out + (size_t)r * p.ost + (size_t)hh * p.osh + col) = v;
    }
  }
}

// Wherever whole tiles of 16 entries and 64 value columns are read and written by 16 bytes, at any number of heads a key, most of
// a tile empty or not: us of rows_attn_kernel / this at 622 rows, 64 entries, 1, 2, 4 heads a key 190 / 121, 102 / 71, 62 / 48;
// latent, 1 head of 64 + 16 31 / 19, 3 of 256 + 64 61 / 50, 40 of 512 + 64 (329 rows) 251 / 159;  one row at 100 keys, 16
// heads over 2 of 128 17.6 / 11.7, latent 27 / 21.
static bool rows_mfma_ok(const RowsArgs& p) {
  const int D = p.D1 + p.D2;
  return !p.po && D % 16 == 0 && D <= 1024 && p.V % 64 == 0 && p.ks % 4 == 0 && p.vs % 4 == 0 &&
         p.ost % 4 == 0 && p.osh % 4 == 0 && (((uintptr_t)p.kc | (uintptr_t)p.vc | (uintptr_t)p.out) & 15) == 0;
}

static int launch_rows_mfma(const RowsArgs& p, int T, hipStream_t s) {
  const int hpg = p.H / (p.G * p.M), ne = p.V % 256 == 0 ? 4 : p.V % 128 == 0 ? 2 : 1;
  const size_t lds = sizeof(float) * (16 * ((size_t)p.D1 + p.D2 + 4) + 16 * kRmKeys + 32 + 2 * kRaKeys);
  auto k = ne == 4 ? rows_attn_mfma_kernel<4> : ne == 2 ? rows_attn_mfma_kernel<2> : rows_attn_mfma_kernel<1>;
  if (lds > 48 * 1024 && hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds))
    return (int)hipGetLastError();
  hipLaunchKernelGGL(k, dim3(T, p.G * p.M * ((hpg + 15) / 16) * (p.V / (64 * ne))), dim3(256), lds, s, p);
  return (int)hipGetLastError();
}

// joins the parts of a (row, head) in order
template <typename TO>
__global__ void __launch_bounds__(256) rows_attn_merge_kernel(RowsArgs p) {
  const int r = p.row_base + blockIdx.x, hh = blockIdx.y;
  const int sg = p.row_seg[r], pos = p.seg_pos0[sg] + r - p.seg_row0[sg];
  const int n = (key_runs(pos, p.chunk, p.window, p.keep_first).total + kRaKeys - 1) / kRaKeys;
  const size_t at = ((size_t)blockIdx.x * p.H + hh) * p.n_parts;
  for (int c = threadIdx.x; c < p.V; c += blockDim.x) {
    float m = p.sink ? p.sink[hh] : -INFINITY, l = p.sink ? 1.f : 0.f, o = 0.f;
    for (int k = 0; k < n; ++k) {
      float a, b;
      ra_join(m, l, p.pml[(at + k) * 2], p.pml[(at + k) * 2 + 1], a, b);
      o = ra_join_out(o, a, p.po[(at + k) * p.V + c], b);
    }
    float v = o / l;
    if (p.gate) v *= 1.f / (1.f + expf(-p.gate[(size_t)r * p.gs + hh]));
    rst((TO*)p.out, (size_t)r * p.ost + (size_t)hh * p.osh + c, v);
  }
}

template <typename TQ, typename TC, typename TO>
static int launch_rows(const RowsArgs& p, int T, hipStream_t s) {
  if (sizeof(TQ) == 4 && sizeof(TC) == 4 && sizeof(TO) == 4 && rows_mfma_ok(p)) return launch_rows_mfma(p, T, s);
  const int D = p.D1 + p.D2, hpg = p.H / (p.G * p.M), z = p.po ? p.n_parts : 1;
  auto groups = [&](int most) { return p.G * p.M * ((hpg + most - 1) / most) * ((p.V + 255) / 256); };
  const bool few = p.po && (long)T * groups(kRaFew) * z <= (sizeof(TC) == 4 ? 512 : 256);
  const int most = few ? kRaFew : kRaHeads, HB = hpg < most ? hpg : most;
  const size_t lds = sizeof(float) * ((size_t)HB * ((D + 3) / 4 * 4 + 4) + HB * kRaKeys + 2 * HB + kRaKeys);
  const dim3 grid(T, groups(most), z);
  // four numbers of a key at a time where every key starts on such a border
  const bool vec = D % 4 == 0 && p.ks % 4 == 0 && ((uintptr_t)p.kc & (4 * sizeof(TC) - 1)) == 0;
  auto k = few    ? (vec ? rows_attn_kernel<TQ, TC, TO, true, true, true> : rows_attn_kernel<TQ, TC, TO, false, true, true>)
           : p.po ? (vec ? rows_attn_kernel<TQ, TC, TO, true, true, false> : rows_attn_kernel<TQ, TC, TO, false, true, false>)
                  : (vec ? rows_attn_kernel<TQ, TC, TO, true, false, false>
                         : rows_attn_kernel<TQ, TC, TO, false, false, false>);
  if (lds > 48 * 1024 && hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds))
    return (int)hipGetLastError();
  hipLaunchKernelGGL(k, grid, dim3(256), lds, s, p);
  if (p.po)
    hipLaunchKernelGGL((rows_attn_merge_kernel<TO>), dim3(T, p.H), dim3(p.V >= 256 ? 256 : (p.V + 63) / 64 * 64), 0, s, p);
  return (int)hipGetLastError();
}

}  // namespace k8s

using namespace k8s;

// n_parts > 0: a workgroup per part of 128 visible keys (n_parts: at least the parts of the row that sees most), joined from
// po [T][H maps][n_parts][V] and pml [.. ][2]; 0: a workgroup walks all parts
K8S_API int k8s_masked_attn_rows(const void* q, const void* kc, const void* vc, const int* block_tables, int maxb,
                                 const int* row_seg, const int* seg_row0, const int* seg_pos0, const float* sink,
                                 const float* gate, int gs, void* out, int T, int H, int G, int D, int V, int BS,
                                 int chunk, int window, int keep_first, float scale, float softcap, int dt,
                                 hipStream_t s, int maps, int out_f32, int n_parts, float* po, float* pml) {
  if (T <= 0) return 0;
  if (maps < 1) return (int)hipErrorInvalidValue;
  const int HQ = H * maps;
  // the sizes callers may count on, all within this kernel's LDS: 8192 outputs a row; queries, 64 scores and two sums a head
  // in 64 KB
  if (H < 1 || G < 1 || H % G || D < 1 || V < 1 || HQ * V > 8192 || chunk < 0 || window < 0 || keep_first < 0 ||
      (size_t)(HQ * D + HQ * 64 + 2 * HQ) * sizeof(float) > 64 * 1024 || (n_parts > 0 && (!po || !pml)))
    return (int)hipErrorInvalidValue;
  RowsArgs p{};
  p.q = q;
  p.qst = (long)HQ * D;
  p.qsh = D;
  p.D1 = D;
  p.kc = kc;
  p.vc = vc;
  p.ks = G * maps * D;
  p.vs = G * V;
  p.bt = block_tables;
  p.maxb = maxb;
  p.row_seg = row_seg;
  p.seg_row0 = seg_row0;
  p.seg_pos0 = seg_pos0;
  p.sink = sink;
  p.gate = gate;
  p.gs = gs;
  p.out = out;
  p.ost = (long)HQ * V;
  p.osh = V;
  p.H = HQ;
  p.G = G;
  p.M = maps;
  p.V = V;
  p.BS = BS;
  p.chunk = chunk;
  p.window = window;
  p.keep_first = keep_first;
  p.scale = scale;
  p.softcap = softcap;
  p.n_parts = n_parts;
  p.po = n_parts > 0 ? po : nullptr;
  p.pml = pml;
  if (dt == 0 && out_f32) return launch_rows<uint16_t, uint16_t, float>(p, T, s);
  if (dt == 0) return launch_rows<uint16_t, uint16_t, uint16_t>(p, T, s);
  return launch_rows<float, float, float>(p, T, s);
}

// Rows row_base .. row_base + n_rows of the step.  dt: 0 = bf16 cache and output, 1 = fp32.
K8S_API int k8s_latent_attn_rows(const float* qa, const void* cache, const int* bt, int maxb, const int* row_seg,
                                 const int* seg_row0, const int* seg_pos0, const float* gate, int ldg, void* out,
                                 int row_base, int n_rows, int H, int R, int BS, float scale, int dt,
                                 hipStream_t s, long qst, long qsh, const float* qr, int RP, long ost, long osh,
                                 int window, const float* sink, int n_parts, float* po, float* pml) {
  if (n_rows <= 0) return 0;
  if (H <= 0 || R <= 0 || R > 2048 || RP < 0 || (RP && !qr) || window < 0 || (n_parts > 0 && (!po || !pml)))
    return (int)hipErrorInvalidValue;
  // the sizes callers may count on, all within this kernel's LDS: the queries of as many heads as make 2048 numbers beside 32
  // cache rows and their scores in 160 KB
  const size_t hg = 2048 / R < H ? (2048 / R < 64 ? 2048 / R : 64) : (H < 64 ? H : 64);
  if ((hg * (R + RP) + 32 * (size_t)(R + RP + 1) + 35 * hg) * sizeof(float) > 160 * 1024) return (int)hipErrorInvalidValue;
  RowsArgs p{};
  p.q = qa;
  p.qst = qst;
  p.qsh = qsh;
  p.q2 = qr;
  p.D1 = R;
  p.D2 = RP;
  p.kc = cache;
  p.vc = cache;
  p.ks = R + RP;
  p.vs = R + RP;
  p.bt = bt;
  p.maxb = maxb;
  p.row_seg = row_seg;
  p.seg_row0 = seg_row0;
  p.seg_pos0 = seg_pos0;
  p.sink = sink;
  p.gate = gate;
  p.gs = ldg;
  p.out = out;
  p.ost = ost;
  p.osh = osh;
  p.H = H;
  p.G = 1;
  p.M = 1;
  p.V = R;
  p.BS = BS;
  p.row_base = row_base;
  p.window = window;
  p.scale = scale;
  p.n_parts = n_parts;
  p.po = n_parts > 0 ? po : nullptr;
  p.pml = pml;
  return dt == 0 ? launch_rows<float, uint16_t, uint16_t>(p, n_rows, s) : launch_rows<float, float, float>(p, n_rows, s);
}
