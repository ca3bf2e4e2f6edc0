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
// 128 rows of x times BN rows of W per block, four waves of 64 x BN/2. At
// these M a step's products (512 cycles per wave at BN 128) are much shorter
// than the way of its operands from HBM, so both panels go to LDS by
// global_load_lds with NB - 1 steps of 64 k in flight (96 KB at BN 128), one
// counted wait and one barrier per step. 16-byte slots are permuted by row on
// the source address ((row >> 1) & 7: the 16 rows of a fragment read cover
// the 256 bytes of the banks once). W is the A operand, so a lane ends with
// four neighbouring columns of a row. Blocks go round robin over the 8 XCDs;
// each XCD takes a contiguous stretch of tiles, row tiles first, so that the
// row tiles of a panel of W meet in one L2.
//
// Measured on MI355X, 128 / 333 / 512 rows, reduce included (before: 128 or
// 256 rows x 64, one step ahead, K in 8 cuts): 3584 x 3584 17 / 36 / 42 -> 16
// / 29 / 33 us, 3584 x 18944 46 / 108 / 121 -> 46 / 86 / 101, 4608 x 3584 22 /
// 38 / 44 -> 20 / 28 / 43. All cuts in one block instead of partials was
// slower (3584 x 18944, 512 rows: 171 us).

#include "common.hpp"

namespace {

constexpr int BLOCK = 256;
constexpr int BM = 128, XK = 64;

using f32x4 = __attribute__((ext_vector_type(4))) float;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

// counted VMEM wait with a compile-time immediate — invisible to hipcc's
// waitcnt pass, so the glds pipeline is not drained at barriers
template <int N>
DEVINLINE void waitcnt_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int BN, int NB, int SPLIT>
__global__ __launch_bounds__(BLOCK) void gemm_tiled_kernel(
    const bf16* __restrict__ x,     // [M, K]
    const bf16* __restrict__ w,     // [N, K]
    const bf16* __restrict__ bias,  // [N] or null
    bf16* __restrict__ out,         // [M, N]
    float* __restrict__ partial,    // [n_split, M, N] when SPLIT
    int M, int N, int K, int k_per, int n_split) {
  constexpr int CPW = (BM + BN) / 32;        // copies of 8 rows per wave
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
  auto copy = [&](int i) {
    const int k0 = kb + i * XK;
#pragma unroll
    for (int g = 0; g < CPW; ++g)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(
              src[g] + min(k0 + off[g], K - 8)),
          (__attribute__((address_space(3))) void*)(
              &lds[i & (NB - 1)][(wave * CPW + g) * 8][0]),
          16, 0, 0);
  };
  const int wm = (wave & 1) * 64, wn = (wave >> 1) * (BN / 2);
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
  auto arrive = [&](int i) {                 // step i is in LDS, i - 1 free
    if (NB > 3 && i + 2 < ns)
      waitcnt_vm<2 * CPW>();
    else if (NB > 2 && i + 1 < ns)
      waitcnt_vm<CPW>();
    else
      waitcnt_vm<0>();
    __builtin_amdgcn_s_barrier();
    if (i + NB - 1 < ns) copy(i + NB - 1);
  };
#pragma unroll
  for (int i = 0; i < NB - 1; ++i)
    if (i < ns) copy(i);
  for (int i = 0; i < whole; ++i) {
    arrive(i);
#pragma unroll
    for (int t = 0; t < XK / 32; ++t) product(i & (NB - 1), t);
  }
  if (whole < ns) {                          // 32 are left
    arrive(whole);
    product(whole & (NB - 1), 0);
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

// Big-tile variant for very wide N (lm_head): 256x256 block tile, 8 waves
// (2M x 4N quadrants of 128x64), 128 KB LDS, 1 block/CU. With more than 128
// rows the products are what bounds it, and a wave's 12 fragment reads serve
// 32 MFMAs against 8 for 16 above. Same per-row K accumulation as the rest
// of the family, K in one piece. Handles N % 256 != 0 (lm_head 151936) with
// clamped W loads + guarded stores.
template <int HAS_BIAS>
__global__ __launch_bounds__(512, 1) void gemm_tiled_sq_kernel(
    const bf16* __restrict__ x,     // [M, K]
    const bf16* __restrict__ w,     // [N, K]
    const bf16* __restrict__ bias,  // [N] or null
    bf16* __restrict__ out,         // [M, N]
    int M, int N, int K) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;          // 0..7
  const int col = lane & 15;
  const int quad = lane >> 4;
  const int wm = wave >> 2;                   // 0..1: 128-row band
  const int wn = wave & 3;                    // 0..3: 64-col band
  const int m_base = blockIdx.z * 256;

  const int k_begin = 0, k_end = K;

  __shared__ bf16 lds[2][256 + 256][64];

  f32x4 acc[32];
#pragma unroll
  for (int m = 0; m < 32; ++m) acc[m] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int l8 = lane >> 3, c8 = lane & 7;

  // x: 32 chunks of 8 rows -> 4 per wave; W: 32 chunks -> 4 per wave
#define GS_GLDS_TILE(bufi, k0)                                              \
  if ((k0) < k_end) {                                                       \
    _Pragma("unroll") for (int g = 0; g < 4; ++g) {                         \
      const int chunk = wave * 4 + g;                                       \
      const int row = chunk * 8 + l8;                                       \
      const int xr = min(m_base + row, M - 1);                              \
      const int kc = min((k0) + (c8 ^ (row & 7)) * 8, K - 8);               \
      auto gsrc = (const __attribute__((address_space(1))) void*)(          \
          x + (int64_t)xr * K + kc);                                        \
      auto ldst = (__attribute__((address_space(3))) void*)(                \
          &lds[bufi][chunk * 8][0]);                                        \
      __builtin_amdgcn_global_load_lds(gsrc, ldst, 16, 0, 0);               \
    }                                                                       \
    _Pragma("unroll") for (int g = 0; g < 4; ++g) {                         \
      const int wchunk = wave * 4 + g;                                      \
      const int wr = wchunk * 8 + l8;                                       \
      const int gr = min((int)blockIdx.x * 256 + wr, N - 1);                \
      const int kc = min((k0) + (c8 ^ (wr & 7)) * 8, K - 8);                \
      auto gsrc = (const __attribute__((address_space(1))) void*)(          \
          w + (int64_t)gr * K + kc);                                        \
      auto ldst = (__attribute__((address_space(3))) void*)(                \
          &lds[bufi][256 + wchunk * 8][0]);                                 \
      __builtin_amdgcn_global_load_lds(gsrc, ldst, 16, 0, 0);               \
    }                                                                       \
  }

  GS_GLDS_TILE(0, k_begin);
  int buf = 0;
  for (int k0 = k_begin; k0 < k_end; k0 += 64) {
    if (k0 + 64 < k_end) {
      GS_GLDS_TILE(buf ^ 1, k0 + 64);
      waitcnt_vm<8>();                        // tile t landed; t+1 out
    } else {
      waitcnt_vm<0>();
    }
    __builtin_amdgcn_s_barrier();
    const int tile_k = min(64, k_end - k0);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      if (kk * 32 < tile_k) {
        bf16x8_t bfrag[4], afrag[8];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
          const int wrow = wn * 64 + nt * 16 + col;
          const int wslot = (kk * 4 + quad) ^ (wrow & 7);
          bfrag[nt] = *reinterpret_cast<const bf16x8_t*>(
              &lds[buf][256 + wrow][wslot * 8]);
        }
#pragma unroll
        for (int mt = 0; mt < 8; ++mt) {
          const int row = wm * 128 + mt * 16 + col;
          const int slot = (kk * 4 + quad) ^ (row & 7);
          afrag[mt] = *reinterpret_cast<const bf16x8_t*>(
              &lds[buf][row][slot * 8]);
        }
#pragma unroll
        for (int mt = 0; mt < 8; ++mt)
#pragma unroll
          for (int nt = 0; nt < 4; ++nt)
            acc[mt * 4 + nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                afrag[mt], bfrag[nt], acc[mt * 4 + nt], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    buf ^= 1;
  }
#undef GS_GLDS_TILE

#pragma unroll
  for (int mt = 0; mt < 8; ++mt) {
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const int oc = blockIdx.x * 256 + wn * 64 + nt * 16 + col;
      if (oc < N) {
        const float b = HAS_BIAS ? bf2f(bias[oc]) : 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int orow = m_base + wm * 128 + mt * 16 + quad * 4 + r;
          if (orow < M) {
            out[(int64_t)orow * N + oc] = f2bf(acc[mt * 4 + nt][r] + b);
          }
        }
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
// The tile is the one that needs no second round of blocks: BN 64 with four
// buffers (one block per CU) while that makes at most 256 blocks, else BN 128
// with four, else BN 128 with two buffers and two blocks per CU. us on 3584 x
// 18944 in 4 cuts, BN 64 / 128 / 128 two buffers: 128 rows 46 / 61 / 85, 256
// rows 85 / 65 / 83, 512 rows 155 / 115 / 101; on 37888 x 3584 uncut, 65 rows
// 81 / 79 / 69.
void tl_gemm_tiled(const void* x, const void* w, const void* bias, void* out,
                   void* partial, int M, int N, int K, int n_split,
                   int k_per, hipStream_t stream) {
  if (N >= 65536 && n_split == 1 && M > 128) {
    const dim3 grid(cdiv(N, 256), 1, cdiv(M, 256)), block(512);
    if (bias)
      hipLaunchKernelGGL(gemm_tiled_sq_kernel<1>, grid, block, 0, stream,
                         (const bf16*)x, (const bf16*)w, (const bf16*)bias,
                         (bf16*)out, M, N, K);
    else
      hipLaunchKernelGGL(gemm_tiled_sq_kernel<0>, grid, block, 0, stream,
                         (const bf16*)x, (const bf16*)w, nullptr, (bf16*)out,
                         M, N, K);
    return;
  }
  const int nm = cdiv(M, BM);
  const int b64 = nm * cdiv(N, 64) * n_split;
  const int b128 = nm * cdiv(N, 128) * n_split;
#define TL_GT(BN, NB, SP, BLOCKS)                                            \
  hipLaunchKernelGGL((gemm_tiled_kernel<BN, NB, SP>),                        \
                     dim3((uint32_t)(cdiv(BLOCKS, 8) * 8)), dim3(BLOCK), 0,  \
                     stream, (const bf16*)x, (const bf16*)w,                 \
                     (const bf16*)bias, (bf16*)out, (float*)partial, M, N,   \
                     K, k_per, n_split)
  if (b64 <= 256) {
    if (n_split > 1) TL_GT(64, 4, 1, b64); else TL_GT(64, 4, 0, b64);
  } else if (b128 <= 256) {
    if (n_split > 1) TL_GT(128, 4, 1, b128); else TL_GT(128, 4, 0, b128);
  } else {
    if (n_split > 1) TL_GT(128, 2, 1, b128); else TL_GT(128, 2, 0, b128);
  }
#undef TL_GT
  if (n_split > 1 && out)
    tl_gemm_reduce(partial, bias, out, (int64_t)M * N, N, n_split, stream);
}

}  // extern "C"
