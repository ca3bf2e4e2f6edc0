// Training rows of layers with layer norms and biases, bf16 with fp32 sums
// (gfx950).
//
//   tl_bias_grad     the column sums of dy; with z also dz = dy gelu'(z)
//                    (tanh form) and the sums of dz, in the same pass.
//   tl_layernorm_fwd r = x + a (rounded; optional), y = LayerNorm(r) w + b.
//   tl_layernorm_bwd the gradient of r: LayerNorm's plus, where there is one,
//                    the gradient that comes along r itself; and the slabs of
//                    dw and db.
//
// All bound by their rows' way through memory or, at 2048 rows, by the launch.
// Column sums leave one fp32 slab per block of rows, added side by side by
// tl_reduce_partials. us at 2048 rows, before (a pass for each of the parts)
// -> now, the slabs' sums of 3.7 included: bias of 768 to 3072 columns 14 -> 7,
// activation and bias of 3072 25 -> 17, norm of 768 with its add 11 -> 6
// forward, with the add of the gradients 24 -> 15 backward.

#include "common.hpp"

namespace {

constexpr int BLOCK = 256;
constexpr int CW = 128, RW = 16;     // columns of a block, rows side by side

DEVINLINE float gelu_grad(float x) {
  const float b = 0.7978845608f, k = 0.044715f;
  const float u = b * (x + k * x * x * x);
  const float t = 1.f - 2.f / (__expf(2.f * u) + 1.f);
  return 0.5f * (1.f + t) +
         0.5f * x * (1.f - t * t) * b * (1.f + 3.f * k * x * x);
}

template <int GELU>
__global__ __launch_bounds__(BLOCK) void bias_grad_kernel(
    const bf16* __restrict__ dy, const bf16* __restrict__ z,
    bf16* __restrict__ dz, float* __restrict__ partial, int64_t M, int N,
    int per) {
  __shared__ float lds[RW][CW + 4];
  const int g = threadIdx.x / 16, l = threadIdx.x % 16;
  const int c = blockIdx.x * CW + l * 8;
  const int64_t r0 = (int64_t)blockIdx.y * per;
  const int64_t r1 = min(M, r0 + per);
  float acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0.f;
  if (c < N)
    for (int64_t r = r0 + g; r < r1; r += RW) {
      bf16x8 v = *reinterpret_cast<const bf16x8*>(dy + r * N + c);
      if (GELU) {
        const bf16x8 vz = *reinterpret_cast<const bf16x8*>(z + r * N + c);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          v.v[j] = f2bf(bf2f(v.v[j]) * gelu_grad(bf2f(vz.v[j])));
        *reinterpret_cast<bf16x8*>(dz + r * N + c) = v;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] += bf2f(v.v[j]);
    }
#pragma unroll
  for (int j = 0; j < 8; ++j) lds[g][l * 8 + j] = acc[j];
  __syncthreads();
  const int n = blockIdx.x * CW + threadIdx.x;
  if (threadIdx.x < CW && n < N) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < RW; ++i) s += lds[i][threadIdx.x];
    partial[(int64_t)blockIdx.y * N + n] = s;
  }
}

// one wave per row, 512 columns per ITER
template <int ITERS>
__global__ __launch_bounds__(BLOCK) void layernorm_fwd_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ a,
    const bf16* __restrict__ w, const bf16* __restrict__ b,
    bf16* __restrict__ r_out, bf16* __restrict__ y, float* __restrict__ mean,
    float* __restrict__ rstd, int64_t M, int W, float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  float f[ITERS][8], s = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * 64 + lane) * 8;
    if (c < W) {
      bf16x8 v = *reinterpret_cast<const bf16x8*>(x + row * W + c);
      if (a) {
        const bf16x8 va = *reinterpret_cast<const bf16x8*>(a + row * W + c);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          v.v[j] = f2bf(bf2f(v.v[j]) + bf2f(va.v[j]));
        *reinterpret_cast<bf16x8*>(r_out + row * W + c) = v;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) s += f[it][j] = bf2f(v.v[j]);
    }
  }
  const float mu = wave_reduce_sum(s) / W;
  float q = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it)
    if ((it * 64 + lane) * 8 < W)
#pragma unroll
      for (int j = 0; j < 8; ++j) q += (f[it][j] - mu) * (f[it][j] - mu);
  const float rs = rsqrtf(wave_reduce_sum(q) / W + eps);
  if (lane == 0) {
    mean[row] = mu;
    rstd[row] = rs;
  }
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * 64 + lane) * 8;
    if (c < W) {
      const bf16x8 vw = *reinterpret_cast<const bf16x8*>(w + c);
      const bf16x8 vb = *reinterpret_cast<const bf16x8*>(b + c);
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o.v[j] = f2bf((f[it][j] - mu) * rs * bf2f(vw.v[j]) + bf2f(vb.v[j]));
      *reinterpret_cast<bf16x8*>(y + row * W + c) = o;
    }
  }
}

// partial [grid, 2 W]: dw, db
template <int ITERS>
__global__ __launch_bounds__(BLOCK) void layernorm_bwd_kernel(
    const bf16* __restrict__ dy, const bf16* __restrict__ dr,
    const bf16* __restrict__ r, const bf16* __restrict__ w,
    const float* __restrict__ mean, const float* __restrict__ rstd,
    bf16* __restrict__ dx, float* __restrict__ partial, int64_t M, int W) {
  __shared__ float lds[4][ITERS * 512];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float dw[ITERS][8], db[ITERS][8], fw[ITERS][8];
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * 64 + lane) * 8;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      dw[it][j] = db[it][j] = 0.f;
      fw[it][j] = c < W ? bf2f(w[c + j]) : 0.f;
    }
  }
  for (int64_t row = (int64_t)blockIdx.x * 4 + wave; row < M;
       row += (int64_t)gridDim.x * 4) {
    const float mu = mean[row], rs = rstd[row];
    float g[ITERS][8], xh[ITERS][8], sg = 0.f, sgx = 0.f;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int c = (it * 64 + lane) * 8;
      if (c < W) {
        const bf16x8 vd = *reinterpret_cast<const bf16x8*>(dy + row * W + c);
        const bf16x8 vr = *reinterpret_cast<const bf16x8*>(r + row * W + c);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float d = bf2f(vd.v[j]);
          xh[it][j] = (bf2f(vr.v[j]) - mu) * rs;
          dw[it][j] += d * xh[it][j];
          db[it][j] += d;
          g[it][j] = d * fw[it][j];
          sg += g[it][j];
          sgx += g[it][j] * xh[it][j];
        }
      }
    }
    sg = wave_reduce_sum(sg) / W;
    sgx = wave_reduce_sum(sgx) / W;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int c = (it * 64 + lane) * 8;
      if (c < W) {
        bf16x8 o, vr;
        if (dr) vr = *reinterpret_cast<const bf16x8*>(dr + row * W + c);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float d = (g[it][j] - sg - xh[it][j] * sgx) * rs;
          o.v[j] = f2bf(dr ? d + bf2f(vr.v[j]) : d);
        }
        *reinterpret_cast<bf16x8*>(dx + row * W + c) = o;
      }
    }
  }
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    __syncthreads();
#pragma unroll
    for (int it = 0; it < ITERS; ++it)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        lds[wave][(it * 64 + lane) * 8 + j] = half ? db[it][j] : dw[it][j];
    __syncthreads();
    for (int c = threadIdx.x; c < W; c += BLOCK)
      partial[((int64_t)blockIdx.x * 2 + half) * W + c] =
          lds[0][c] + lds[1][c] + lds[2][c] + lds[3][c];
  }
}

}  // namespace

extern "C" {

// rows of a block of tl_bias_grad, so that some 1024 blocks share the sums
int tl_bias_grad_rows(int64_t M, int N) {
  const int64_t slabs = 1024 / cdiv(N, CW) + 1;
  const int64_t per = (M + slabs - 1) / slabs;
  return (int)((per + RW - 1) / RW * RW);
}

// N a multiple of 8; partial [ceil(M / per), N]; z and dz null: sums of dy
void tl_bias_grad(const void* dy, const void* z, void* dz, void* partial,
                  int64_t M, int N, int per, hipStream_t stream) {
  const dim3 grid(cdiv(N, CW), (uint32_t)((M + per - 1) / per));
  if (z)
    hipLaunchKernelGGL(bias_grad_kernel<1>, grid, dim3(BLOCK), 0, stream,
                       (const bf16*)dy, (const bf16*)z, (bf16*)dz,
                       (float*)partial, M, N, per);
  else
    hipLaunchKernelGGL(bias_grad_kernel<0>, grid, dim3(BLOCK), 0, stream,
                       (const bf16*)dy, nullptr, nullptr, (float*)partial, M,
                       N, per);
}

// W a multiple of 8, at most 2048
#define TL_LN(KERNEL, GRID, ...)                                             \
  switch (cdiv(W, 512)) {                                                    \
    case 1: hipLaunchKernelGGL(KERNEL<1>, GRID, dim3(BLOCK), 0, stream,      \
                               __VA_ARGS__); break;                          \
    case 2: hipLaunchKernelGGL(KERNEL<2>, GRID, dim3(BLOCK), 0, stream,      \
                               __VA_ARGS__); break;                          \
    case 3: hipLaunchKernelGGL(KERNEL<3>, GRID, dim3(BLOCK), 0, stream,      \
                               __VA_ARGS__); break;                          \
    case 4: hipLaunchKernelGGL(KERNEL<4>, GRID, dim3(BLOCK), 0, stream,      \
                               __VA_ARGS__); break;                          \
    default: break;                                                          \
  }

void tl_layernorm_fwd(const void* x, const void* a, const void* w,
                      const void* b, void* r_out, void* y, void* mean,
                      void* rstd, int64_t M, int W, float eps,
                      hipStream_t stream) {
  const dim3 grid((uint32_t)((M + 3) / 4));
  TL_LN(layernorm_fwd_kernel, grid, (const bf16*)x, (const bf16*)a,
        (const bf16*)w, (const bf16*)b, (bf16*)r_out, (bf16*)y, (float*)mean,
        (float*)rstd, M, W, eps)
}

// partial [blocks, 2, W]
void tl_layernorm_bwd(const void* dy, const void* dr, const void* r,
                      const void* w, const void* mean, const void* rstd,
                      void* dx, void* partial, int64_t M, int W, int blocks,
                      hipStream_t stream) {
  const dim3 grid(blocks);
  TL_LN(layernorm_bwd_kernel, grid, (const bf16*)dy, (const bf16*)dr,
        (const bf16*)r, (const bf16*)w, (const float*)mean,
        (const float*)rstd, (bf16*)dx, (float*)partial, M, W)
}
#undef TL_LN

}  // extern "C"
