// What stands between the products of a decoder layer, one launch each
// (gfx950). At decode sizes every launch costs 4 to 5 us whatever it does, so
// these kernels take a product's fp32 cuts as they are (skinny_gemm.hip,
// gemm_tiled.hip: summed in order, plus bias, rounded to bf16, which is what
// the reduce kernel writes) instead of its reduced rows.
//
//   add_norm     residual add and RMSNorm: after the output projection, and
//                after the down projection with the NEXT layer's norm.
//   rope_append  (optional) RMSNorm per head of q and k, RoPE, and the append
//                of k and v to a contiguous or paged cache.
//
// Bound by the launch: a decode layer (3584 wide, one row) had reduce, add,
// norm, reduce + bias, conversion of the frequencies, rope + append, length
// + 1 and reduce as launches of 2 to 6 us, and now has three of 4 to 5. Four
// layers and the head of it: 717 -> 666 us; with norms per head (two copies,
// two norms and a concatenation more), two layers at 48 rows: 742 -> 674 us.

#include "common.hpp"

namespace {

constexpr int BLOCK = 256;
constexpr int NW = BLOCK / WAVE_SIZE;

// eight values of a product's row at column c, as the reduce kernel rounds
// them; NS 0: the row is there in bf16
struct Rows {
  const bf16* x;              // [M, N], or null
  const float* partial;       // [n_split, M, N]
  const bf16* bias;           // [N] or null (with partial)
  int64_t MN;
  int N, n_split;
  DEVINLINE void get(int64_t row, int c, float (&f)[8]) const {
    if (x) {
      const bf16x8 v = *reinterpret_cast<const bf16x8*>(x + row * N + c);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = bf2f(v.v[j]);
      return;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = 0.f;
    const float* p = partial + row * N + c;
#pragma unroll 4
    for (int s = 0; s < n_split; ++s, p += MN) {
      const float4 a = *reinterpret_cast<const float4*>(p);
      const float4 b = *reinterpret_cast<const float4*>(p + 4);
      f[0] += a.x; f[1] += a.y; f[2] += a.z; f[3] += a.w;
      f[4] += b.x; f[5] += b.y; f[6] += b.z; f[7] += b.w;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (bias) f[j] += bf2f(bias[c + j]);
      f[j] = bf2f(f2bf(f[j]));
    }
  }
};

// r = product + residual, y = RMSNorm(r) * w. ROUNDED: the norm sees r as it
// is stored, else the fp32 sum. w null: no norm.
template <int ITERS>
__global__ __launch_bounds__(BLOCK) void add_norm_kernel(
    Rows rows, const bf16* __restrict__ residual, const bf16* __restrict__ w,
    bf16* __restrict__ r_out, bf16* __restrict__ y, int rounded, float eps) {
  __shared__ float lds[NW];
  const int H = rows.N;
  const int64_t row = blockIdx.x;
  float vals[ITERS][8];
  float sumsq = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * BLOCK + threadIdx.x) * 8;
    if (c < H) {
      rows.get(row, c, vals[it]);
      const bf16x8 vr =
          *reinterpret_cast<const bf16x8*>(residual + row * H + c);
      bf16x8 out;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float f = vals[it][j] + bf2f(vr.v[j]);
        out.v[j] = f2bf(f);
        vals[it][j] = rounded ? bf2f(out.v[j]) : f;
        sumsq += vals[it][j] * vals[it][j];
      }
      *reinterpret_cast<bf16x8*>(r_out + row * H + c) = out;
    }
  }
  if (!w) return;
  const float rstd = rsqrtf(block_reduce_sum<NW>(sumsq, lds) / H + eps);
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int c = (it * BLOCK + threadIdx.x) * 8;
    if (c < H) {
      const bf16x8 vw = *reinterpret_cast<const bf16x8*>(w + c);
      bf16x8 out;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        out.v[j] = f2bf(vals[it][j] * rstd * bf2f(vw.v[j]));
      *reinterpret_cast<bf16x8*>(y + row * H + c) = out;
    }
  }
}

struct RopeArgs {
  bf16* q_out;                // [T, Hq, D]
  bf16 *k_cache, *v_cache;    // [B, Hkv, Smax, D], or pools of 128 positions
  const int* positions;       // [T]
  const void* inv_freq;       // [D / 2] fp32 or bf16
  const int* table;           // [B, bt_stride] or null
  const bf16 *qw, *kw;        // [D] norm weights, or null
  int S, Hq, Hkv, D, Smax, bt_stride, freq_bf16;
  float eps;
};

// Up to 64 lanes per head, eight elements of either half each (with norms
// D / 16 lanes, a power of two, so that a lane has all it needs); one wave per
// block, so that a single token still spreads over several CUs.
__global__ __launch_bounds__(WAVE_SIZE) void rope_append_rows_kernel(
    Rows rows, RopeArgs a) {
  const int64_t token = blockIdx.x;
  const int D = a.D, D2 = D / 2, L = min(D / 16, WAVE_SIZE);
  const int HPB = WAVE_SIZE / L;
  const int g = threadIdx.x / L, h = blockIdx.y * HPB + g;
  if (g >= HPB || h >= a.Hq + 2 * a.Hkv) return;
  const int pos = a.positions[token];
  const bool rotate = h < a.Hq + a.Hkv;
  bf16* dst;
  if (h < a.Hq) {
    dst = a.q_out + (token * a.Hq + h) * D;
  } else {
    const int hk = rotate ? h - a.Hq : h - a.Hq - a.Hkv;
    bf16* pool = rotate ? a.k_cache : a.v_cache;
    const int64_t b = token / a.S;
    if (a.table) {
      const int page = a.table[b * a.bt_stride + (pos >> 7)];
      dst = pool + (((int64_t)page * a.Hkv + hk) * 128 + (pos & 127)) * D;
    } else {
      dst = pool + ((b * a.Hkv + hk) * a.Smax + pos) * D;
    }
  }
  const bf16* w = !rotate ? nullptr : h < a.Hq ? a.qw : a.kw;
  for (int d = threadIdx.x % L * 8; d < D2; d += L * 8) {
    float x1[8], x2[8];
    rows.get(token, h * D + d, x1);
    rows.get(token, h * D + d + D2, x2);
    if (w) {
      float sumsq = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) sumsq += x1[j] * x1[j] + x2[j] * x2[j];
      for (int off = L / 2; off > 0; off >>= 1)
        sumsq += __shfl_xor(sumsq, off, WAVE_SIZE);
      const float rstd = rsqrtf(sumsq / D + a.eps);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        x1[j] = bf2f(f2bf(x1[j] * rstd * bf2f(w[d + j])));
        x2[j] = bf2f(f2bf(x2[j] * rstd * bf2f(w[d + D2 + j])));
      }
    }
    if (rotate) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float f =
            a.freq_bf16 ? bf2f(static_cast<const bf16*>(a.inv_freq)[d + j])
                        : static_cast<const float*>(a.inv_freq)[d + j];
        float c, s;
        __sincosf((float)pos * f, &s, &c);
        const float a1 = x1[j], a2 = x2[j];
        x1[j] = a1 * c - a2 * s;
        x2[j] = a2 * c + a1 * s;
      }
    }
    bf16x8 o1, o2;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      o1.v[j] = f2bf(x1[j]);
      o2.v[j] = f2bf(x2[j]);
    }
    *reinterpret_cast<bf16x8*>(dst + d) = o1;
    *reinterpret_cast<bf16x8*>(dst + d + D2) = o2;
  }
}

}  // namespace

extern "C" {

// x [M, H] bf16, or null and partial [n_split, M, H]; w and y null: no norm.
// H a multiple of 8, at most 16384.
void tl_add_norm(const void* x, const void* partial, int n_split,
                 const void* residual, const void* w, void* r_out, void* y,
                 int64_t M, int H, int rounded, float eps,
                 hipStream_t stream) {
  if (M <= 0) return;
  const Rows rows{(const bf16*)x, (const float*)partial, nullptr, M * H, H,
                  n_split};
#define CASE(I)                                                              \
  case I:                                                                    \
    hipLaunchKernelGGL(add_norm_kernel<I>, dim3((uint32_t)M), dim3(BLOCK),   \
                       0, stream, rows, (const bf16*)residual,               \
                       (const bf16*)w, (bf16*)r_out, (bf16*)y, rounded,      \
                       eps);                                                 \
    break;
  switch (cdiv(H, BLOCK * 8)) {
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
    default: break;
  }
#undef CASE
}

// x [T, (Hq + 2 Hkv) D] bf16, or null and partial (with bias or null). D a
// multiple of 16; with qw and kw D / 16 a power of two, at most 64.
void tl_rope_append_rows(const void* x, const void* partial, int n_split,
                         const void* bias, void* q_out, void* k_cache,
                         void* v_cache, const void* positions,
                         const void* inv_freq, int freq_bf16,
                         const void* table, int bt_stride, const void* qw,
                         const void* kw, float eps, int64_t T, int S, int Hq,
                         int Hkv, int D, int Smax, hipStream_t stream) {
  if (T <= 0) return;
  const int N = (Hq + 2 * Hkv) * D;
  const Rows rows{(const bf16*)x, (const float*)partial, (const bf16*)bias,
                  T * N, N, n_split};
  const RopeArgs a{(bf16*)q_out, (bf16*)k_cache, (bf16*)v_cache,
                   (const int*)positions, inv_freq, (const int*)table,
                   (const bf16*)qw, (const bf16*)kw, S, Hq, Hkv, D, Smax,
                   bt_stride, freq_bf16, eps};
  const int hpb = D >= 1024 ? 1 : WAVE_SIZE / (D / 16);
  hipLaunchKernelGGL(rope_append_rows_kernel,
                     dim3((uint32_t)T, cdiv(Hq + 2 * Hkv, hpb)),
                     dim3(WAVE_SIZE), 0, stream, rows, a);
}

}  // extern "C"
