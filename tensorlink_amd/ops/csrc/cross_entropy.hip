// Shifted causal-LM cross entropy on bf16 logits (gfx950).
//
// Row (b, s) of the logits [B, S, V] has the label labels[b, s + 1]; rows
// without one (the last of a sequence, ignored labels) count for nothing.
// Bound by the logits' way through HBM: the forward pass reads them once (a
// running maximum and sum per lane, in fp32), the backward pass reads them
// once more and writes the gradient in their own layout and type. Rows of odd
// length start anywhere, so each has a scalar head up to its first 16 bytes.
//
// 4 x 512 x 50257: shifted copy, conversion to fp32, log-softmax, selection
// and all of it backwards were 1050 us in 12 launches, and are 200 us in three
// (49 us forward, 4.2 TB/s; 146 us backward, 2.8 TB/s).

#include <cstdint>

#include "common.hpp"

namespace {

constexpr int BLOCK = 512;
constexpr int NW = BLOCK / WAVE_SIZE;

// calls f(index, values, count) for the row's elements, eight at a time
template <typename F>
DEVINLINE void for_row(const bf16* row, int V, F f) {
  const int head =
      min(V, (int)((16 - (reinterpret_cast<uintptr_t>(row) & 15)) & 15) / 2);
  const int body = (V - head) / 8, tail = head + body * 8;
  for (int i = threadIdx.x; i < body; i += BLOCK)
    f(head + i * 8, *reinterpret_cast<const bf16x8*>(row + head + i * 8), 8);
  const int t = threadIdx.x;                 // at most 7 + 7 are left
  const int i = t < head ? t : tail + t - head;
  if (i < V && t < head + V - tail) {
    bf16x8 v;
    v.v[0] = row[i];
    f(i, v, 1);
  }
}

constexpr int64_t NONE = INT64_MIN;

// label of a row, NONE without one
DEVINLINE int64_t label_of(const int64_t* labels, int64_t row, int S,
                           int64_t ignore) {
  if (row % S == S - 1) return NONE;
  const int64_t l = labels[row + 1];
  return l == ignore ? NONE : l;
}

__global__ __launch_bounds__(BLOCK) void ce_fwd_kernel(
    const bf16* __restrict__ logits, const int64_t* __restrict__ labels,
    float* __restrict__ lse, float* __restrict__ loss, int S, int V,
    int64_t ignore) {
  __shared__ float red_m[NW], red_s[NW];
  const int64_t row = blockIdx.x;
  const int64_t l = label_of(labels, row, S, ignore);
  if (l == NONE) {
    if (threadIdx.x == 0) loss[row] = 0.f;
    return;
  }
  const bf16* x = logits + row * V;
  float m = -INFINITY, s = 0.f;
  auto merge = [](float& m, float& s, float m2, float s2) {
    const float n = fmaxf(m, m2), z = n == -INFINITY ? 0.f : n;
    s = s * __expf(m - z) + s2 * __expf(m2 - z);
    m = n;
  };
  for_row(x, V, [&](int, const bf16x8& v, int n) {
    float f[8], n8 = m;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      f[j] = j < n ? bf2f(v.v[j]) : -INFINITY;
      n8 = fmaxf(n8, f[j]);
    }
    const float z = n8 == -INFINITY ? 0.f : n8;
    s *= __expf(m - z);
#pragma unroll
    for (int j = 0; j < 8; ++j) s += __expf(f[j] - z);
    m = n8;
  });
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    merge(m, s, __shfl_xor(m, off, WAVE_SIZE), __shfl_xor(s, off, WAVE_SIZE));
  if (threadIdx.x % WAVE_SIZE == 0) {
    red_m[threadIdx.x / WAVE_SIZE] = m;
    red_s[threadIdx.x / WAVE_SIZE] = s;
  }
  __syncthreads();
  if (threadIdx.x) return;
  for (int w = 1; w < NW; ++w) merge(m, s, red_m[w], red_s[w]);
  const float z = m + logf(s);
  lse[row] = z;
  // a label outside of the vocabulary has no loss to speak of
  loss[row] = l >= 0 && l < V ? z - bf2f(x[l]) : NAN;
}

// out[0] the mean over the rows with a label, out[1] their number
__global__ __launch_bounds__(BLOCK) void ce_mean_kernel(
    const int64_t* __restrict__ labels, const float* __restrict__ loss,
    float* __restrict__ out, int64_t rows, int S, int64_t ignore) {
  __shared__ float red[2][NW];
  float sum = 0.f, n = 0.f;
  for (int64_t r = threadIdx.x; r < rows; r += BLOCK) {
    sum += loss[r];
    n += label_of(labels, r, S, ignore) == NONE ? 0.f : 1.f;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sum += __shfl_xor(sum, off, WAVE_SIZE);
    n += __shfl_xor(n, off, WAVE_SIZE);
  }
  if (threadIdx.x % WAVE_SIZE == 0) {
    red[0][threadIdx.x / WAVE_SIZE] = sum;
    red[1][threadIdx.x / WAVE_SIZE] = n;
  }
  __syncthreads();
  if (threadIdx.x) return;
  for (int w = 1; w < NW; ++w) {
    sum += red[0][w];
    n += red[1][w];
  }
  out[0] = sum / n;
  out[1] = n;
}

__global__ __launch_bounds__(BLOCK) void ce_bwd_kernel(
    const bf16* __restrict__ logits, const int64_t* __restrict__ labels,
    const float* __restrict__ lse, const float* __restrict__ mean,
    const float* __restrict__ dloss, bf16* __restrict__ dx, int S, int V,
    int64_t ignore) {
  const int64_t row = blockIdx.x;
  const int64_t l = label_of(labels, row, S, ignore);
  const float z = l == NONE ? 0.f : lse[row];
  const float scale = l == NONE ? 0.f : dloss[0] / mean[1];
  bf16* d = dx + row * V;
  // both tensors' rows start at the same offset from 16 bytes
  for_row(logits + row * V, V, [&](int i, const bf16x8& v, int n) {
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float p = l == NONE ? 0.f : __expf(bf2f(v.v[j]) - z);
      o.v[j] = f2bf((i + j == l ? p - 1.f : p) * scale);
    }
    if (n == 8)
      *reinterpret_cast<bf16x8*>(d + i) = o;
    else
      d[i] = o.v[0];
  });
}

}  // namespace

extern "C" {

// logits [B, S, V] bf16, labels [B, S]; lse, loss [B S], mean [2]
void tl_ce_fwd(const void* logits, const void* labels, void* lse, void* loss,
               void* mean, int64_t rows, int S, int V, int64_t ignore,
               hipStream_t stream) {
  hipLaunchKernelGGL(ce_fwd_kernel, dim3((uint32_t)rows), dim3(BLOCK), 0,
                     stream, (const bf16*)logits, (const int64_t*)labels,
                     (float*)lse, (float*)loss, S, V, ignore);
  hipLaunchKernelGGL(ce_mean_kernel, dim3(1), dim3(BLOCK), 0, stream,
                     (const int64_t*)labels, (const float*)loss, (float*)mean,
                     rows, S, ignore);
}

// logits and dx with the same offset from 16 bytes
void tl_ce_bwd(const void* logits, const void* labels, const void* lse,
               const void* mean, const void* dloss, void* dx, int64_t rows,
               int S, int V, int64_t ignore, hipStream_t stream) {
  hipLaunchKernelGGL(ce_bwd_kernel, dim3((uint32_t)rows), dim3(BLOCK), 0,
                     stream, (const bf16*)logits, (const int64_t*)labels,
                     (const float*)lse, (const float*)mean,
                     (const float*)dloss, (bf16*)dx, S, V, ignore);
}

}  // extern "C"
