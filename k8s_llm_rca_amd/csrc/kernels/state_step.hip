// The launches of one token per sequence through a matrix state (state_step.h).
#include "state_step.h"

namespace k8s {

template <int KIND, int LV, int DR, typename TA, typename TO, typename TG, bool LOW>
__global__ void __launch_bounds__(256) state_step_kernel(StepArgs a) {
  __shared__ StepLds<KIND, LV, DR, LOW> lds;
  state_step_head<KIND, LV, DR, TA, TO, TG, LOW>(a, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.z, threadIdx.x, true, lds);
}

template <int KIND, typename TA, typename TO, typename TG, bool LOW = false>
static int launch_step(const StepArgs& a, int n, int D, hipStream_t s, int slices = 1) {
  const dim3 grid(n, a.H, slices);
  const int V = a.V / slices;      // of a workgroup
#define K8S_ST(LV, DR) hipLaunchKernelGGL((state_step_kernel<KIND, LV, DR, TA, TO, TG, LOW>), grid, dim3(256), 0, s, a)
  if (V == 128 && D == 128)
    K8S_ST(32, 16);
  else if (V == 128 && D == 64)
    K8S_ST(32, 8);
  else if (V == 64 && D == 128)
    K8S_ST(16, 8);
  else if (V == 64 && D == 64)
    K8S_ST(16, 4);
  else if constexpr (KIND == 2) {
    if (V == 32 && D == 128)
      K8S_ST(8, 4);
    else if (V == 32 && D == 64)
      K8S_ST(8, 2);
    else
      return (int)hipErrorInvalidValue;
  } else
    return (int)hipErrorInvalidValue;
#undef K8S_ST
  return (int)hipGetLastError();
}

}  // namespace k8s

using namespace k8s;

// n sequences of one token each (rows 0 .. n - 1).  Rows, gates, weights and states in 16-byte accesses: pitches and column
// offsets multiples of 4, pointers of 16 bytes.  V = 64 or 128, D = 64 or 128.
K8S_API int k8s_delta_step(const void* qkv, int dt, const float* a, const float* rate, const float* dt_bias,
                           const float* beta, int bs, float* state, const int* pos0, const int* slot, const float* gate,
                           int gs, const float* w, int wh, void* out, int n, int H, int G, int D, int V, float eps,
                           float unit_eps, hipStream_t s) {
  if (n <= 0) return 0;
  StepArgs p{};
  p.x = qkv; p.xs = 2 * G * D + H * V; p.a = a; p.rate = rate; p.bias = dt_bias; p.beta = beta; p.bs = bs; p.state = state;
  p.pos0 = pos0; p.slot = slot; p.gate = gate; p.gs = gs; p.w = w; p.wh = wh; p.eps = eps; p.unit_eps = unit_eps;
  p.out = out; p.H = H; p.G = G; p.V = V;
  return dt == 0 ? launch_step<0, uint16_t, uint16_t, float>(p, n, D, s) : launch_step<0, float, float, float>(p, n, D, s);
}

// The same in bf16 with a = bf16(lr[., 0 .. ra)) . la^T, the gate = bf16(lr[., ra .. ra + rg)) . lg^T and beta behind them in the
// same rows (stride ls): k8s_low_rank_pair and k8s_delta_step, to the bit.  ra, rg: 32, 64, 96 or 128; la, lg 16-byte aligned.
K8S_API int k8s_delta_step_low(const void* qkv, const float* lr, int ls, int ra, int rg, const void* la, const void* lg,
                               const float* rate, const float* dt_bias, float* state, const int* pos0, const int* slot,
                               const float* w, int wh, void* out, int n, int H, int G, int D, int V, float eps,
                               float unit_eps, hipStream_t s) {
  if (n <= 0) return 0;
  auto off = [](int k, const void* p) { return k < 32 || k > kLowMax || k % 32 || !p || ((uintptr_t)p & 15); };
  if (off(ra, la) || off(rg, lg) || !lr || ls < ra + rg + H || G < 1 || H % G) return (int)hipErrorInvalidValue;
  StepArgs p{};
  p.x = qkv; p.xs = 2 * G * D + H * V; p.rate = rate; p.bias = dt_bias; p.beta = lr + ra + rg; p.bs = ls; p.state = state;
  p.pos0 = pos0; p.slot = slot; p.w = w; p.wh = wh; p.eps = eps; p.unit_eps = unit_eps; p.out = out; p.H = H; p.G = G; p.V = V;
  p.lr = lr; p.ra = ra; p.rg = rg; p.la = (const uint16_t*)la; p.lg = (const uint16_t*)lg;
  return launch_step<0, uint16_t, uint16_t, float, true>(p, n, D, s);
}

K8S_API int k8s_memory_step(const float* x, int xs, const float* gate_bias, float cap, float* state, float* nstate,
                            float* mstate, const int* pos0, const int* slot, const float* gate, int gs, const float* w,
                            int wh, void* out, int odt, int n, int H, int D, int V, float eps, float den_eps, hipStream_t s) {
  if (n <= 0) return 0;
  const StepArgs p = memory_args(x, xs, gate_bias, cap, state, nstate, mstate, pos0, slot, gate, gs, w, wh, out, H, V, eps, den_eps);
  return odt == 0 ? launch_step<1, float, uint16_t, float>(p, n, D, s) : launch_step<1, float, float, float>(p, n, D, s);
}

// ssp [n][H][slices]; slices: workgroups of a head, 1, 2 or 4 (32 columns or more each)
K8S_API int k8s_decay_step(const void* x, int xs, int dt, const float* decay, float* state, const int* pos0, const int* slot,
                           const void* gate, int gs, const float* w, void* out, float* ssp, int n, int H, int D, int V,
                           hipStream_t s, int slices) {
  if (n <= 0) return 0;
  if (slices < 1 || V % slices) return (int)hipErrorInvalidValue;
  StepArgs p{};
  p.x = x; p.xs = xs; p.rate = decay; p.state = state; p.pos0 = pos0; p.slot = slot; p.gate = gate; p.gs = gs; p.w = w;
  p.wh = V; p.out = out; p.ssp = ssp; p.H = H; p.G = H; p.V = V;
  return dt == 0 ? launch_step<2, uint16_t, uint16_t, uint16_t>(p, n, D, s, slices)
                 : launch_step<2, float, float, float>(p, n, D, s, slices);
}
