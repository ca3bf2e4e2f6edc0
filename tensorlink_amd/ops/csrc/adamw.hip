// Fused AdamW step for gfx950.
//
// Replaces the reference's per-module torch.optim step executed on each
// worker (tensorlink/ml/worker.py:1279-1297). The Python-side optimizer
// flattens a stage's parameters into ONE contiguous buffer, so the whole
// stage steps in a single launch (cf. the plan's "one fused HIP Adam
// kernel launch per stage rank").
//
// param: bf16 or fp32 [n]; grad: same dtype as param; exp_avg/exp_avg_sq:
// fp32 [n]. Decoupled weight decay, bias correction — matches
// torch.optim.AdamW numerics (fp32 math throughout).

#include "common.hpp"

namespace {

constexpr int BLOCK = 256;

struct AdamArgs {
  float lr, beta1, beta2, eps, weight_decay, bc1, bc2;
};

// one element; p, m and v are updated
DEVINLINE void adam(const AdamArgs& a, float g, float& p, float& m,
                    float& v) {
  m = m * a.beta1 + (1.f - a.beta1) * g;
  v = v * a.beta2 + (1.f - a.beta2) * g * g;
  const float denom = sqrtf(v / a.bc2) + a.eps;
  p = p * (1.f - a.lr * a.weight_decay) - a.lr * (m / a.bc1) / denom;
}

DEVINLINE float ld(const bf16* p) { return bf2f(*p); }
DEVINLINE float ld(const float* p) { return *p; }
DEVINLINE void st(bf16* p, float x) { *p = f2bf(x); }
DEVINLINE void st(float* p, float x) { *p = x; }

// any alignment: one element per thread
template <typename T>
__global__ __launch_bounds__(BLOCK) void adamw_kernel(
    T* __restrict__ param, const T* __restrict__ grad, float* __restrict__ m,
    float* __restrict__ v, int64_t n, AdamArgs a) {
  const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (i >= n) return;
  float p = ld(param + i), mi = m[i], vi = v[i];
  adam(a, ld(grad + i), p, mi, vi);
  m[i] = mi;
  v[i] = vi;
  st(param + i, p);
}

// 16-byte aligned buffers: eight elements per thread, 16 bytes per access;
// each is read and written once a step, so past the caches. Bound by HBM.
template <typename T>
__global__ __launch_bounds__(BLOCK) void adamw_vec_kernel(
    T* __restrict__ param, const T* __restrict__ grad, float* __restrict__ m,
    float* __restrict__ v, int64_t n, AdamArgs a) {
  const int64_t i0 = ((int64_t)blockIdx.x * BLOCK + threadIdx.x) * 8;
  if (i0 + 8 > n) {
    for (int64_t i = i0; i < n; ++i) {
      float p = ld(param + i), mi = m[i], vi = v[i];
      adam(a, ld(grad + i), p, mi, vi);
      m[i] = mi;
      v[i] = vi;
      st(param + i, p);
    }
    return;
  }
  constexpr int W = sizeof(T) / 2;           // 16-byte words of 8 elements
  using f32x4 = __attribute__((ext_vector_type(4))) float;
  f32x4 pw[W], gw[W], mw[2], vw[2];
#pragma unroll
  for (int w = 0; w < W; ++w) {
    pw[w] = __builtin_nontemporal_load(
        reinterpret_cast<const f32x4*>(param + i0) + w);
    gw[w] = __builtin_nontemporal_load(
        reinterpret_cast<const f32x4*>(grad + i0) + w);
  }
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    mw[w] = __builtin_nontemporal_load(
        reinterpret_cast<const f32x4*>(m + i0) + w);
    vw[w] = __builtin_nontemporal_load(
        reinterpret_cast<const f32x4*>(v + i0) + w);
  }
  T ps[8], gs[8];
  __builtin_memcpy(ps, pw, sizeof(ps));
  __builtin_memcpy(gs, gw, sizeof(gs));
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float p = ld(ps + j), mi = mw[j >> 2][j & 3], vi = vw[j >> 2][j & 3];
    adam(a, ld(gs + j), p, mi, vi);
    mw[j >> 2][j & 3] = mi;
    vw[j >> 2][j & 3] = vi;
    st(ps + j, p);
  }
  __builtin_memcpy(pw, ps, sizeof(ps));
#pragma unroll
  for (int w = 0; w < W; ++w)
    __builtin_nontemporal_store(pw[w],
                                reinterpret_cast<f32x4*>(param + i0) + w);
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    __builtin_nontemporal_store(mw[w], reinterpret_cast<f32x4*>(m + i0) + w);
    __builtin_nontemporal_store(vw[w], reinterpret_cast<f32x4*>(v + i0) + w);
  }
}

template <typename T>
void launch(void* param, const void* grad, void* m, void* v, int64_t n,
            const AdamArgs& a, hipStream_t stream) {
  const bool aligned =
      (((uintptr_t)param | (uintptr_t)grad | (uintptr_t)m | (uintptr_t)v) &
       15) == 0;
  const int64_t work = aligned ? (n + 7) / 8 : n;
  const dim3 grid((uint32_t)((work + BLOCK - 1) / BLOCK)), block(BLOCK);
  if (aligned)
    hipLaunchKernelGGL(adamw_vec_kernel<T>, grid, block, 0, stream, (T*)param,
                       (const T*)grad, (float*)m, (float*)v, n, a);
  else
    hipLaunchKernelGGL(adamw_kernel<T>, grid, block, 0, stream, (T*)param,
                       (const T*)grad, (float*)m, (float*)v, n, a);
}

}  // namespace

extern "C" {

void tl_adamw(void* param, const void* grad, void* m, void* v, int64_t n,
              int is_bf16, float lr, float beta1, float beta2, float eps,
              float weight_decay, int step, hipStream_t stream) {
  if (n <= 0) return;
  const AdamArgs a{lr, beta1, beta2, eps, weight_decay,
                   1.f - powf(beta1, (float)step),
                   1.f - powf(beta2, (float)step)};
  if (is_bf16)
    launch<bf16>(param, grad, m, v, n, a, stream);
  else
    launch<float>(param, grad, m, v, n, a, stream);
}

}  // extern "C"
