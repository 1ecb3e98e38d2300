// Dynamic Tanh norm around an fp32 residual stream, and the squared ReLU.
//
//   dyt(x) = tanh(alpha x) * w + b   per element: no mean, no variance, nothing couples a row's entries.
// So the residual add, the norm of the new residual and the cast for the next GEMM are ONE elementwise
// pass: x is read and written once (fp32), the sublayer outputs are read once (fp32), the activations
// written once (TA: bf16 as uint16_t, or float).  Four consecutive columns per thread where the width
// allows 16-byte accesses.
#include "common.h"
#include "rope_rows.h"

namespace k8s {

template <typename T>
__device__ __forceinline__ float ldd(const T* p, size_t i);
template <>
__device__ __forceinline__ float ldd<float>(const float* p, size_t i) { return p[i]; }
template <>
__device__ __forceinline__ float ldd<uint16_t>(const uint16_t* p, size_t i) { return bf2f(p[i]); }
template <typename T>
__device__ __forceinline__ void std_(T* p, size_t i, float v);
template <>
__device__ __forceinline__ void std_<float>(float* p, size_t i, float v) { p[i] = v; }
template <>
__device__ __forceinline__ void std_<uint16_t>(uint16_t* p, size_t i, float v) { p[i] = f2bf(v); }

template <typename T>
__device__ __forceinline__ void st4(T* p, size_t i, const float (&v)[4]);
template <>
__device__ __forceinline__ void st4<float>(float* p, size_t i, const float (&v)[4]) {
  *reinterpret_cast<f32x4*>(p + i) = f32x4{v[0], v[1], v[2], v[3]};
}
template <>
__device__ __forceinline__ void st4<uint16_t>(uint16_t* p, size_t i, const float (&v)[4]) {
  *reinterpret_cast<u16x4*>(p + i) = u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
}

// x += sy * y + sy2 * y2 (y, y2 optional, each the sum of yp / yp2 planes);  out = tanh(alpha x) w + b (w optional).
// n4 = T * W / 4.
template <typename TA>
__global__ void __launch_bounds__(256) add_dyt4_kernel(float* __restrict__ x, const float* __restrict__ y, float sy,
                                                       const float* __restrict__ y2, float sy2, float alpha,
                                                       const float* __restrict__ w, const float* __restrict__ b,
                                                       TA* __restrict__ out, size_t n4, int W, int yp, int yp2) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (size_t)gridDim.x * blockDim.x) {
    const size_t e = i * 4;
    const int c = (int)(e % (size_t)W);
    f32x4 xv = *reinterpret_cast<const f32x4*>(x + e);
    if (y) {
      const f32x4 yv = sum_planes4(y + e, n4 * 4, yp);
#pragma unroll
      for (int k = 0; k < 4; ++k) xv[k] = fmaf(sy, yv[k], xv[k]);
      if (y2) {
        const f32x4 zv = sum_planes4(y2 + e, n4 * 4, yp2);
#pragma unroll
        for (int k = 0; k < 4; ++k) xv[k] = fmaf(sy2, zv[k], xv[k]);
      }
      *reinterpret_cast<f32x4*>(x + e) = xv;
    }
    if (w) {
      const f32x4 wv = *reinterpret_cast<const f32x4*>(w + c), bv = *reinterpret_cast<const f32x4*>(b + c);
      float o[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] = fmaf(tanhf(alpha * xv[k]), wv[k], bv[k]);
      st4(out, e, o);
    }
  }
}

template <typename TA>
__global__ void __launch_bounds__(256) add_dyt1_kernel(float* __restrict__ x, const float* __restrict__ y, float sy,
                                                       const float* __restrict__ y2, float sy2, float alpha,
                                                       const float* __restrict__ w, const float* __restrict__ b,
                                                       TA* __restrict__ out, size_t n, int W, int yp, int yp2) {
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (size_t)gridDim.x * 256) {
    const int c = (int)(e % (size_t)W);
    float xv = x[e];
    if (y) {
      xv = fmaf(sy, sum_planes(y + e, n, yp), xv);
      if (y2) xv = fmaf(sy2, sum_planes(y2 + e, n, yp2), xv);
      x[e] = xv;
    }
    if (w) std_(out, e, fmaf(tanhf(alpha * xv), w[c], b[c]));
  }
}

// x = embed[id] * scale;  out = dyt(x) (w optional).  One workgroup per row; those past the T rows: rope_rows.h.
template <typename TE, typename TA>
__global__ void __launch_bounds__(256) embed_scale_dyt_kernel(const int* __restrict__ ids, const TE* __restrict__ embed,
                                                              float scale, float* __restrict__ x, float alpha,
                                                              const float* __restrict__ w, const float* __restrict__ b,
                                                              TA* __restrict__ out, int W, int T, RopeTables rt) {
  if ((int)blockIdx.x >= T) return rope_block(rt, T);
  const size_t o = (size_t)blockIdx.x * W, src = (size_t)ids[blockIdx.x] * W;
  for (int c = threadIdx.x; c < W; c += 256) {
    const float xv = ldd(embed, src + c) * scale;
    x[o + c] = xv;
    if (w) std_(out, o + c, fmaf(tanhf(alpha * xv), w[c], b[c]));
  }
}

// The same with four neighbouring columns per thread (16384 rows of 2048 106 -> 50 us, one row 10.3 -> 2.4).
__device__ __forceinline__ f32x4 ldd4(const float* p, size_t i) { return *reinterpret_cast<const f32x4*>(p + i); }
__device__ __forceinline__ f32x4 ldd4(const uint16_t* p, size_t i) {
  const u16x4 v = *reinterpret_cast<const u16x4*>(p + i);
  return f32x4{bf2f(v[0]), bf2f(v[1]), bf2f(v[2]), bf2f(v[3])};
}
template <typename TE, typename TA>
__global__ void __launch_bounds__(512) embed_scale_dyt4_kernel(const int* __restrict__ ids, const TE* __restrict__ embed,
                                                               float scale, float* __restrict__ x, float alpha,
                                                               const float* __restrict__ w, const float* __restrict__ b,
                                                               TA* __restrict__ out, int W, int T, RopeTables rt) {
  if ((int)blockIdx.x >= T) return rope_block(rt, T);
  const size_t o = (size_t)blockIdx.x * W, src = (size_t)ids[blockIdx.x] * W;
  for (int c = 4 * threadIdx.x; c < W; c += 4 * blockDim.x) {
    f32x4 v = ldd4(embed, src + c), wv = f32x4{0.f, 0.f, 0.f, 0.f}, bv = wv;
    if (w) {
      wv = ldd4(w, c);
      bv = ldd4(b, c);
    }
    float r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] *= scale;
      r[k] = fmaf(tanhf(alpha * v[k]), wv[k], bv[k]);
    }
    *reinterpret_cast<f32x4*>(x + o + c) = v;
    if (w) st4(out, o + c, r);
  }
}

template <typename TA>
__global__ void __launch_bounds__(256) relu_sq_kernel(const TA* __restrict__ u, TA* __restrict__ out, size_t n) {
  for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (size_t)gridDim.x * 256) {
    const float v = fmaxf(ldd(u, e), 0.f);
    std_(out, e, v * v);
  }
}

template <>
__global__ void __launch_bounds__(256) relu_sq_kernel<uint16_t>(const uint16_t* __restrict__ u,
                                                                uint16_t* __restrict__ out, size_t n) {
  const size_t n8 = n / 8;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (size_t)gridDim.x * 256) {
    const u16x8 a = *reinterpret_cast<const u16x8*>(u + i * 8);
    u16x8 r;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float v = fmaxf(bf2f(a[k]), 0.f);
      r[k] = f2bf(v * v);
    }
    *reinterpret_cast<u16x8*>(out + i * 8) = r;
  }
  if (blockIdx.x == 0)
    for (size_t e = n8 * 8 + threadIdx.x; e < n; e += 256) {
      const float v = fmaxf(bf2f(u[e]), 0.f);
      out[e] = f2bf(v * v);
    }
}

static int grid_for(size_t items) {
  const size_t g = (items + 255) / 256;
  return (int)(g < 1 ? 1 : (g > 8192 ? 8192 : g));
}

}  // namespace k8s

using namespace k8s;

K8S_API int k8s_add_dyt(float* x, const float* y, float sy, const float* y2, float sy2, float alpha, const float* w,
                        const float* b, void* out, int odt, int T, int W, hipStream_t s, int yp, int yp2) {
  if (T <= 0 || W <= 0) return 0;
  if ((w == nullptr) != (out == nullptr) || (w && !b) || (y2 && !y) || yp < 1 || yp2 < 1) return (int)hipErrorInvalidValue;
  const size_t n = (size_t)T * W;
  if (W % 4 == 0) {
    // few rows: a wave per workgroup, so that more compute units take the planes in (one row, eight planes of 2048:
    // 4.4 -> 3.8 us in a reply step)
    const int th = n / 4 <= 64 * 1024 ? 64 : 256;
    const int g4 = th == 64 ? (int)((n / 4 + 63) / 64) : grid_for(n / 4);
    if (odt == 0)
      hipLaunchKernelGGL((add_dyt4_kernel<uint16_t>), dim3(g4), dim3(th), 0, s, x, y, sy, y2, sy2, alpha, w,
                         b, (uint16_t*)out, n / 4, W, yp, yp2);
    else
      hipLaunchKernelGGL((add_dyt4_kernel<float>), dim3(g4), dim3(th), 0, s, x, y, sy, y2, sy2, alpha, w, b,
                         (float*)out, n / 4, W, yp, yp2);
  } else {
    if (odt == 0)
      hipLaunchKernelGGL((add_dyt1_kernel<uint16_t>), dim3(grid_for(n)), dim3(256), 0, s, x, y, sy, y2, sy2, alpha, w, b,
                         (uint16_t*)out, n, W, yp, yp2);
    else
      hipLaunchKernelGGL((add_dyt1_kernel<float>), dim3(grid_for(n)), dim3(256), 0, s, x, y, sy, y2, sy2, alpha, w, b,
                         (float*)out, n, W, yp, yp2);
  }
  return (int)hipGetLastError();
}

K8S_API int k8s_embed_scale_dyt(const int* ids, const void* embed, int edt, float scale, float* x, float alpha,
                                const float* w, const float* b, void* out, int odt, int T, int W, hipStream_t s,
                                const int* pos, const double* freq0, float amp0, int half0,
                                float* cs0, const double* freq1, float amp1, int half1, float* cs1) {
  if (T <= 0 || W <= 0) return 0;
  if ((w == nullptr) != (out == nullptr) || (w && !b)) return (int)hipErrorInvalidValue;
  const RopeTables rt{pos, {freq0, freq1}, {cs0, cs1}, {amp0, amp1}, {half0, half1}};
  if (!rope_tables_ok(rt)) return (int)hipErrorInvalidValue;
  const bool by4 = W % 4 == 0 && (((uintptr_t)embed | (uintptr_t)x | (uintptr_t)w | (uintptr_t)b | (uintptr_t)out) & 15) == 0;
  const int t4 = W > 2048 - 256 ? 512 : (W / 4 + 63) / 64 * 64;
#define K8S_EMB(TE, TA)                                                                                                 \
  if (by4)                                                                                                              \
    hipLaunchKernelGGL((embed_scale_dyt4_kernel<TE, TA>), dim3(T + rope_blocks(rt, T, t4)), dim3(t4), 0, s, ids,        \
                       (const TE*)embed, scale, x, alpha, w, b, (TA*)out, W, T, rt);                                    \
  else                                                                                                                  \
    hipLaunchKernelGGL((embed_scale_dyt_kernel<TE, TA>), dim3(T + rope_blocks(rt, T, 256)), dim3(256), 0, s, ids,         \
                       (const TE*)embed, scale, x, alpha, w, b, (TA*)out, W, T, rt)
  if (edt == 0 && odt == 0) {
    K8S_EMB(uint16_t, uint16_t);
  } else if (edt == 0) {
    K8S_EMB(uint16_t, float);
  } else if (odt == 0) {
    K8S_EMB(float, uint16_t);
  } else {
    K8S_EMB(float, float);
  }
#undef K8S_EMB
  return (int)hipGetLastError();
}

K8S_API int k8s_relu_sq(const void* u, void* out, long n, int dt, hipStream_t s) {
  if (n <= 0) return 0;
  if (dt == 0)
    hipLaunchKernelGGL((relu_sq_kernel<uint16_t>), dim3(grid_for((size_t)n / 8 + 1)), dim3(256), 0, s,
                       (const uint16_t*)u, (uint16_t*)out, (size_t)n);
  else
    hipLaunchKernelGGL((relu_sq_kernel<float>), dim3(grid_for((size_t)n)), dim3(256), 0, s, (const float*)u,
                       (float*)out, (size_t)n);
  return (int)hipGetLastError();
}
