// Skinny-M GEMM for the decode path: out[M,N] = x[M,K] @ W[N,K]^T (+bias),
// M <= 64.
//
// torch Linear stores W as [N, K] row-major, so both operands are
// k-contiguous. At decode M the GEMM is pure W-streaming: what bounds it is
// how many bytes of W are in flight and how few launches surround it.
//
// A block covers 64 rows of W and all rows of x. Both go to LDS by
// global_load_lds (128 or 256 contiguous bytes per row, 16-byte slots permuted by
// row, so the ds_read_b128 meet no conflicts), three steps of XK k ahead in
// four buffers. The copies are counted: a step waits for the oldest only, with
// one barrier. W through registers instead is 64 bytes per row and load, and
// the compiler then drains all copies at each use. A wave owns 16 rows of W
// (the A operand, so a lane ends with four neighbouring columns of a row).
// Grid (N/64, n_split): K is cut in 2 or 4 where N/64 leaves CUs without a
// block (fp32 partials + reduce kernel), at multiples of 256.
//
// Measured on MI355X, 1 / 16 / 64 rows, reduce included (before: W through
// registers, one step ahead, a barrier that drained it): 3584 x 18944 44 / 45
// / 53 -> 28 / 28 / 35 us (4.9 TB/s), 4096 x 12288 46 / 47 / 53 -> 21 / 22 /
// 25, 4608 x 3584 19 / 19 / 22 -> 11 / 11 / 15, 152064 x 3584 241 / 253 / 291
// -> 179 / 186 / 225 (6.1 TB/s). Cuts inside the block, each with a wave's own
// buffers and no partials, were slower (44 us on 3584 x 18944).
//
// Contract with gemm_tiled.hip: every row sums K in 32-wide
// mfma_f32_16x16x32_bf16 steps in order within a cut, and the cuts in order.

#include "common.hpp"

namespace {

constexpr int BLOCK = 256;

using f32x4 = __attribute__((ext_vector_type(4))) float;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

template <int N>
DEVINLINE void waitcnt_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

constexpr int NB = 4;                // buffers

// XK k per step. GLU: W is [gate; up] of N / 2 rows each and a wave owns eight
// rows of either at the same columns; out [M, N / 2] = silu(gate) up, of the
// two rounded to bf16 as the product alone would be.
template <int MT, int XK, int SPLIT, int GLU>
__global__ __launch_bounds__(BLOCK) void skinny_gemm_kernel(
    const bf16* __restrict__ x,     // [M, K]
    const bf16* __restrict__ w,     // [N, K]
    const bf16* __restrict__ bias,  // [N] or null
    bf16* __restrict__ out,         // [M, N]
    float* __restrict__ partial,    // [n_split, M, N] when SPLIT
    int M, int N, int K, int k_per) {
  constexpr int R = MT * 16 + 64;            // rows of a buffer: x, then w
  constexpr int SL = XK / 8, RPC = 64 / SL;  // slots of a row, rows of a copy
  constexpr int CPW = R / RPC / 4;           // copies per wave
  static_assert(CPW * RPC * 4 == R);
  auto turn = [](int r) { return SL == 16 ? r & 15 : (r >> 1) & 7; };
  __shared__ bf16 lds[NB][R][XK];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, quad = lane >> 4;
  const int n0 = GLU ? blockIdx.x * 32 + wave * 8
                     : blockIdx.x * 64 + wave * 16;
  const int kb = SPLIT ? blockIdx.y * k_per : 0;
  const int ke = SPLIT ? min(K, kb + k_per) : K;

  const bf16* src[CPW];
  int off[CPW];
#pragma unroll
  for (int g = 0; g < CPW; ++g) {
    const int r = (wave * CPW + g) * RPC + lane / SL, wr = r - MT * 16;
    const int64_t wrow =
        GLU ? blockIdx.x * 32 + (wr >> 4) * 8 + (wr & 7) +
                  (wr & 8 ? N / 2 : 0)
            : blockIdx.x * 64 + wr;
    src[g] = wr < 0 ? x + (int64_t)min(r, M - 1) * K : w + wrow * K;
    off[g] = (lane % SL ^ turn(r)) * 8;
  }
  auto copy = [&](int i) {
    const int k0 = kb + i * XK;
#pragma unroll
    for (int g = 0; g < CPW; ++g)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(
              src[g] + min(k0 + off[g], K - 8)),
          (__attribute__((address_space(3))) void*)(
              &lds[i & (NB - 1)][(wave * CPW + g) * RPC][0]),
          16, 0, 0);
  };
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto product = [&](int buf, int t) {       // 32 k
    const int s = ((t * 4 + quad) ^ turn(col)) * 8;
    const bf16x8_t wf = *reinterpret_cast<const bf16x8_t*>(
        &lds[buf][MT * 16 + wave * 16 + col][s]);
#pragma unroll
    for (int m = 0; m < MT; ++m)
      acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          wf, *reinterpret_cast<const bf16x8_t*>(&lds[buf][m * 16 + col][s]),
          acc[m], 0, 0, 0);
  };
  const int whole = (ke - kb) / XK;
  const int ns = (ke - kb + XK - 1) / XK;
  auto arrive = [&](int i) {                 // step i is in LDS, i - 1 free
    if (i + 2 < ns)
      waitcnt_vm<2 * CPW>();
    else if (i + 1 < ns)
      waitcnt_vm<CPW>();
    else
      waitcnt_vm<0>();
    __builtin_amdgcn_s_barrier();
    if (i + 3 < ns) copy(i + 3);
  };
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (i < ns) copy(i);
  for (int i = 0; i < whole; ++i) {
    arrive(i);
#pragma unroll
    for (int t = 0; t < XK / 32; ++t) product(i & (NB - 1), t);
  }
  if (whole < ns) {                          // less than a step is left
    arrive(whole);
    for (int t = 0; t < (ke - kb - whole * XK) / 32; ++t)
      product(whole & (NB - 1), t);
  }

  if (GLU) {                                 // quads 0, 1 gate, 2, 3 up
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      bf16x4_t o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float g = bf2f(f2bf(acc[m][r]));
        const float u = __shfl_xor(g, 32, 64);
        o[r] = (__bf16)(g / (1.f + __expf(-g)) * u);
      }
      const int row = m * 16 + col;
      if (quad < 2 && row < M)
        *reinterpret_cast<bf16x4_t*>(out + (int64_t)row * (N / 2) + n0 +
                                     quad * 4) = o;
    }
    return;
  }
  // lane: columns n0 + quad * 4 + 0..3 of row m * 16 + col
  const int n = n0 + quad * 4;
  f32x4 b = (f32x4){0.f, 0.f, 0.f, 0.f};
  if (!SPLIT && bias) {
#pragma unroll
    for (int r = 0; r < 4; ++r) b[r] = bf2f(bias[n + r]);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = m * 16 + col;
    if (row >= M) continue;
    if (SPLIT) {
      *reinterpret_cast<f32x4*>(
          partial + ((int64_t)blockIdx.y * M + row) * N + n) = acc[m];
    } else {
      bf16x4_t o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = (__bf16)(acc[m][r] + b[r]);
      *reinterpret_cast<bf16x4_t*>(out + (int64_t)row * N + n) = o;
    }
  }
}

// N is a multiple of 64: four columns per thread
__global__ __launch_bounds__(BLOCK) void skinny_reduce_kernel(
    const float* __restrict__ partial, const bf16* __restrict__ bias,
    bf16* __restrict__ out, int64_t MN, int N, int n_split) {
  const int64_t i = ((int64_t)blockIdx.x * BLOCK + threadIdx.x) * 4;
  if (i >= MN) return;
  f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < n_split; ++s)
    acc += *reinterpret_cast<const f32x4*>(partial + s * MN + i);
  bf16x4_t o;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float b = bias ? bf2f(bias[i % N + r]) : 0.f;
    o[r] = (__bf16)(bias ? acc[r] + b : acc[r]);
  }
  *reinterpret_cast<bf16x4_t*>(out + i) = o;
}

}  // namespace

extern "C" {

// out = the sum over the cuts, in order, plus bias
void tl_gemm_reduce(const void* partial, const void* bias, void* out,
                    int64_t MN, int N, int n_split, hipStream_t stream) {
  hipLaunchKernelGGL(skinny_reduce_kernel,
                     dim3((uint32_t)((MN / 4 + BLOCK - 1) / BLOCK)),
                     dim3(BLOCK), 0, stream, (const float*)partial,
                     (const bf16*)bias, (bf16*)out, MN, N, n_split);
}

// partial: scratch [n_split * M * N] floats (only used when n_split > 1; out
// null then: the cuts are left for the caller to sum)
//
// Uncut products of more than 16 rows have blocks enough for two per CU, which
// steps of 64 k leave the LDS for (151936 x 4096, 32 / 48 / 64 rows: 252 / 270
// / 284 us with steps of 128, 246 / 260 / 272 with 64); with cuts, or for 16
// rows, longer steps are as good or better (6144 x 4096, 32 rows: 14.7, 15.3).
void tl_skinny_gemm(const void* x, const void* w, const void* bias,
                    void* out, void* partial, int M, int N, int K,
                    int n_split, int k_per, hipStream_t stream) {
  const dim3 grid(N / 64, n_split), block(BLOCK);
#define TL_SG(MT, XK)                                                            \
  do {                                                                       \
    if (n_split > 1)                                                         \
      hipLaunchKernelGGL((skinny_gemm_kernel<MT, XK, 1, 0>), grid, block, 0,        \
                         stream, (const bf16*)x, (const bf16*)w, nullptr,    \
                         nullptr, (float*)partial, M, N, K, k_per);          \
    else                                                                     \
      hipLaunchKernelGGL((skinny_gemm_kernel<MT, XK, 0, 0>), grid, block, 0,        \
                         stream, (const bf16*)x, (const bf16*)w,             \
                         (const bf16*)bias, (bf16*)out, nullptr, M, N, K,    \
                         K);                                                 \
  } while (0)
  if (M <= 16) {
    TL_SG(1, 128);
  } else if (n_split == 1) {
    if (M <= 32) TL_SG(2, 64);
    else TL_SG(4, 64);
  } else {
    if (M <= 32) TL_SG(2, 128);
    else if (M <= 48) TL_SG(3, 128);
    else TL_SG(4, 128);
  }
#undef TL_SG
  if (n_split > 1 && out)
    tl_gemm_reduce(partial, bias, out, (int64_t)M * N, N, n_split, stream);
}

// out [M, N / 2] = silu(x gate^T) (x up^T), w = [gate; up] [N, K]; M <= 64,
// N a multiple of 64. Against the product and the activation as two launches
// (the library's, 37888 x 3584 / 28672 x 4096): 1 row 55 / 61 -> 50 / 45 us, 32
// rows 57 / 54 -> 55 / 46, 64 rows 64 / 55 -> 66 / 52: above 32 rows the caller
// has N / 64 blocks fit one round of two per CU.
void tl_skinny_glu(const void* x, const void* w, void* out, int M, int N,
                   int K, hipStream_t stream) {
#define TL_SG(MT, XK)                                                        \
  hipLaunchKernelGGL((skinny_gemm_kernel<MT, XK, 0, 1>), dim3(N / 64),       \
                     dim3(BLOCK), 0, stream, (const bf16*)x, (const bf16*)w, \
                     nullptr, (bf16*)out, nullptr, M, N, K, K)
  if (M <= 16) TL_SG(1, 128);
  else if (M <= 32) TL_SG(2, 64);
  else TL_SG(4, 64);
#undef TL_SG
}

}  // extern "C"
