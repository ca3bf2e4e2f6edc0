// Tiled serving GEMM for mid-M (65 <= M <= ~512): out[M,N] = x[M,K] @
// W[N,K]^T (+bias). Companion to skinny_gemm.hip (M <= 64): SAME per-row
// accumulation semantics — K in 32-wide mfma_f32_16x16x32_bf16 steps in
// order, f32 accumulators, the same cuts of K summed in the same order — so a
// row's result is bitwise IDENTICAL for any M and either kernel. That
// property is what lets chunked prefill, speculative verify, batched decode
// and plain generate produce equal tokens (the serving engine's exact-greedy
// guarantee); do not change the order here without changing skinny_gemm.hip
// to match.
//
// BM rows of x times BN rows of W per block, BM / 32 waves of 64 x BN/2. Both
// panels go to LDS by global_load_lds with NB - 1 steps of 64 k in flight, one
// counted wait and one barrier per step. 16-byte slots are permuted by row on
// the source address ((row >> 1) & 7: the 16 rows of a fragment read cover the
// 256 bytes of the banks once). W is the A operand, so a lane ends with four
// neighbouring columns of a row. Blocks go round robin over the 8 XCDs; each
// XCD takes a contiguous stretch of tiles, row tiles first, so that the row
// tiles of a panel of W meet in one L2.
//
// What bounds it is how long a CU's lines take, of which it has some 64 in
// flight: 480 cycles on the average, W from HBM and x from L2 (3584 x 18944,
// 512 rows, 256 x 128: the copies alone take 72 of 85 us, the products alone
// 46; more buffers change nothing, a larger tile does).
//
// Measured on MI355X, 128 / 333 / 512 rows, reduce included (before: 128 or
// 256 rows x 64, one step ahead, K in 8 cuts): 3584 x 3584 17 / 36 / 42 -> 16
// / 29 / 31 us, 3584 x 18944 46 / 108 / 121 -> 46 / 87 / 89, 4608 x 3584 22 /
// 38 / 44 -> 20 / 28 / 39. All cuts in one block instead of partials was
// slower (3584 x 18944, 512 rows: 171 us).

#include "common.hpp"

namespace {

constexpr int XK = 64;

using f32x4 = __attribute__((ext_vector_type(4))) float;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

// counted VMEM wait with a compile-time immediate — invisible to hipcc's
// waitcnt pass, so the glds pipeline is not drained at barriers
template <int N>
DEVINLINE void waitcnt_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int BM, int BN, int NB, int SPLIT>
__global__ __launch_bounds__(BM * 2) void gemm_tiled_kernel(
    const bf16* __restrict__ x,     // [M, K]
    const bf16* __restrict__ w,     // [N, K]
    const bf16* __restrict__ bias,  // [N] or null
    bf16* __restrict__ out,         // [M, N]
    float* __restrict__ partial,    // [n_split, M, N] when SPLIT
    int M, int N, int K, int k_per, int n_split) {
  constexpr int NM = BM / 64;                // waves along the rows
  constexpr int CPW = (BM + BN) / (NM * 16); // copies of 8 rows per wave
  constexpr int NT = BN / 32;                // 16-column tiles per wave
  __shared__ bf16 lds[NB][BM + BN][XK];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, quad = lane >> 4;
  const int nm = (M + BM - 1) / BM, np = (N + BN - 1) / BN;
  const int per = gridDim.x >> 3;            // the grid is a multiple of 8
  int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const int m0 = id % nm * BM;
  id /= nm;
  const int n0 = id % np * BN, cut = id / np;
  if (cut >= (SPLIT ? n_split : 1)) return;
  const int kb = SPLIT ? cut * k_per : 0;
  const int ke = SPLIT ? min(K, kb + k_per) : K;

  const bf16* src[CPW];
  int off[CPW];
#pragma unroll
  for (int g = 0; g < CPW; ++g) {
    const int r = (wave * CPW + g) * 8 + (lane >> 3);
    src[g] = r < BM ? x + (int64_t)min(m0 + r, M - 1) * K
                    : w + (int64_t)min(n0 + r - BM, N - 1) * K;
    off[g] = ((lane & 7) ^ ((r >> 1) & 7)) * 8;
  }
  auto copy = [&](int i, int buf) {
    const int k0 = kb + i * XK;
#pragma unroll
    for (int g = 0; g < CPW; ++g)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(
              src[g] + min(k0 + off[g], K - 8)),
          (__attribute__((address_space(3))) void*)(
              &lds[buf][(wave * CPW + g) * 8][0]),
          16, 0, 0);
  };
  const int wm = (wave & (NM - 1)) * 64, wn = wave / NM * (BN / 2);
  f32x4 acc[NT][4];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto product = [&](int buf, int t) {       // 32 k
    const int s = ((t * 4 + quad) ^ (col >> 1)) * 8;
    bf16x8_t xf[4], wf[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
      wf[i] = *reinterpret_cast<const bf16x8_t*>(
          &lds[buf][BM + wn + i * 16 + col][s]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      xf[j] = *reinterpret_cast<const bf16x8_t*>(
          &lds[buf][wm + j * 16 + col][s]);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            wf[i], xf[j], acc[i][j], 0, 0, 0);
  };
  const int whole = (ke - kb) / XK;
  const int ns = (ke - kb + XK - 1) / XK;
  int cur = 0;                               // buffer of the step
  auto arrive = [&](int i) {                 // step i is in LDS, i - 1 free
    if (NB > 3 && i + 2 < ns)
      waitcnt_vm<2 * CPW>();
    else if (NB > 2 && i + 1 < ns)
      waitcnt_vm<CPW>();
    else
      waitcnt_vm<0>();
    __builtin_amdgcn_s_barrier();
    if (i + NB - 1 < ns) copy(i + NB - 1, cur ? cur - 1 : NB - 1);
  };
#pragma unroll
  for (int i = 0; i < NB - 1; ++i)
    if (i < ns) copy(i, i);
  for (int i = 0; i < whole; ++i) {
    arrive(i);
#pragma unroll
    for (int t = 0; t < XK / 32; ++t) product(cur, t);
    cur = cur == NB - 1 ? 0 : cur + 1;
  }
  if (whole < ns) {                          // 32 are left
    arrive(whole);
    product(cur, 0);
  }

#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int n = n0 + wn + i * 16 + quad * 4;
    if (n >= N) continue;                    // N is a multiple of 64
    f32x4 b = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (!SPLIT && bias) {
#pragma unroll
      for (int r = 0; r < 4; ++r) b[r] = bf2f(bias[n + r]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = m0 + wm + j * 16 + col;
      if (row >= M) continue;
      if (SPLIT) {
        *reinterpret_cast<f32x4*>(partial + ((int64_t)cut * M + row) * N +
                                  n) = acc[i][j];
      } else {
        bf16x4_t o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (__bf16)(acc[i][j][r] + b[r]);
        *reinterpret_cast<bf16x4_t*>(out + (int64_t)row * N + n) = o;
      }
    }
  }
}

}  // namespace

extern "C" {

void tl_gemm_reduce(const void* partial, const void* bias, void* out,
                    int64_t MN, int N, int n_split, hipStream_t stream);

// partial: scratch [n_split * M * N] floats (only used when n_split > 1; out
// null then: the cuts are left for the caller to sum).
//
// The tile is the one that needs no second round of blocks: 128 x 64 with four
// buffers (one block per CU) while that makes at most 256 blocks, else 128 x
// 128 with four. Beyond that 256 x 128 with three buffers where it has no more
// rows of padding than 128 (each panel of W then goes to half as many CUs),
// else 128 x 128 with two buffers and two blocks per CU. us on 3584 x 18944 in
// 4 cuts, in that order: 128 rows 46 / 61 / 78 / 85, 256 rows 85 / 65 / 86 /
// 83, 333 rows - / 109 / 88 / 87, 512 rows 155 / 115 / 89 / 101.
//
// Very wide N has many rounds anyway: 256 x 128 from 129 rows, 128 x 256 where
// that saves 128 rows of padding, 128 x 128 with four buffers below. us on
// 152064 x 3584, 256 x 128 / 128 x 256 / 128 x 128: 128 rows 325 / 261 / 250,
// 256 rows 342 / 387 / 423, 333 rows 607 / 511 / 570, 512 rows 628 / 713 / 773
// (before, 256 x 256 with two buffers: 256 rows 354, 333 rows 594, 512 rows
// 627; 128 rows on 128 x 128 with two buffers 269).
void tl_gemm_tiled(const void* x, const void* w, const void* bias, void* out,
                   void* partial, int M, int N, int K, int n_split,
                   int k_per, hipStream_t stream) {
  auto blocks = [&](int bm, int bn) {
    return cdiv(M, bm) * cdiv(N, bn) * n_split;
  };
#define TL_GT1(BM, BN, NB, SP)                                               \
  hipLaunchKernelGGL((gemm_tiled_kernel<BM, BN, NB, SP>),                    \
                     dim3((uint32_t)(cdiv(blocks(BM, BN), 8) * 8)),          \
                     dim3(BM * 2), 0, stream, (const bf16*)x,                \
                     (const bf16*)w, (const bf16*)bias, (bf16*)out,          \
                     (float*)partial, M, N, K, k_per, n_split)
#define TL_GT(BM, BN, NB)                                                    \
  do {                                                                       \
    if (n_split > 1) TL_GT1(BM, BN, NB, 1); else TL_GT1(BM, BN, NB, 0);      \
  } while (0)
  const bool even = cdiv(M, 256) * 2 == cdiv(M, 128);
  if (N >= 65536 && n_split == 1) {
    if (M <= 128) TL_GT(128, 128, 4);
    else if (even) TL_GT(256, 128, 3);
    else TL_GT(128, 256, 3);
  } else if (blocks(128, 64) <= 256) {
    TL_GT(128, 64, 4);
  } else if (blocks(128, 128) <= 256) {
    TL_GT(128, 128, 4);
  } else if (even) {
    TL_GT(256, 128, 3);
  } else {
    TL_GT(128, 128, 2);
  }
#undef TL_GT
#undef TL_GT1
  if (n_split > 1 && out)
    tl_gemm_reduce(partial, bias, out, (int64_t)M * N, N, n_split, stream);
}

}  // extern "C"
