// Grouped expert products with stacked experts on MFMA (gfx950, bf16): the
// two ends of the range around moe_gemm.hip.
//
// out[p][n] = sum_k x[tok ? tok[p] : p][k] w[e][n][k] for the pairs p of
// expert e (seg[e] <= p < seg[e + 1]).
//
// tl_moe_tiles (prompts): 128 pairs x 128 columns per block, four waves of
// 64 x 64. Both panels go to LDS by direct loads (global_load_lds, rows
// gathered through tok), double-buffered over 64-wide k steps; the 16-byte
// slots of a row are permuted by the row number on the source address, and
// the fragment reads apply the same permutation. The tile list is implicit:
// the grid has an upper bound of tiles (P / 128 + E), a block finds its
// expert with a wave-wide scan over the segments and leaves if there is
// none. Consecutive tiles go to one XCD, columns first, so an expert's
// weights and a tile's rows are read from that XCD's L2. The weight is the
// A operand, so a lane ends with four neighbouring columns of one row. The
// k order per row is that of moe_gemm.hip.
// tl_moe_tiles_any is the same for experts behind a pointer table, in bf16 or
// fp8 (converted to bf16 on the way to LDS, which takes registers between
// the load and the store), and for gate and up in one pass: the weight panel
// then holds 64 gate and 64 up rows, a wave has both of its columns, and
// silu(gate) * up is written, 64 columns per block.
//
// tl_moe_rows (decoding): few pairs per expert. A block covers 16 columns of
// one expert; its four waves take a quarter of K each, straight from global
// memory (all loads of a quarter are in flight before the first product),
// and meet in LDS.

#include "common.hpp"

namespace {

constexpr int BLOCK = 256;
constexpr int BM = 128, BN = 128, BK = 64;

using f32x4 = __attribute__((ext_vector_type(4))) float;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

struct alignas(8) bf16x4 {
  bf16 v[4];
};

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

DEVINLINE bf16x8_t from_fp8(uint32_t a, uint32_t b) {      // exact
  const bf16x2_t p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.f, false);
  const bf16x2_t p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.f, true);
  const bf16x2_t p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, false);
  const bf16x2_t p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, true);
  return (bf16x8_t){p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// addresses from the pointer table are global memory (not flat)
using u32x4 = __attribute__((ext_vector_type(4))) uint32_t;
template <typename T>
DEVINLINE T load_global(const char* p) {
  return *reinterpret_cast<const __attribute__((address_space(1))) T*>(
      reinterpret_cast<uint64_t>(p));
}

template <int FP8, int GATED>
__global__ __launch_bounds__(BLOCK, 2) void moe_tile_kernel(
    const bf16* __restrict__ x, const int* __restrict__ tok,
    const int* __restrict__ seg, const uint64_t* __restrict__ w_ptrs,
    const bf16* __restrict__ w, const uint64_t* __restrict__ s_ptrs,
    bf16* __restrict__ out, int E, int N, int K, int n_tiles) {
  constexpr int CN = GATED ? BN / 2 : BN;         // columns of out per block
  __shared__ bf16 lds[2][BM + BN][BK];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // blocks go round-robin over the 8 XCDs: give each a contiguous stretch
  const int per = gridDim.x / 8;                  // grid is a multiple of 8
  const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  const int nt = (N + CN - 1) / CN;
  const int mt = id / nt, n0 = (id - mt * nt) * CN;
  if (mt >= n_tiles) return;
  // expert and row tile of the mt-th tile
  int e = -1, mb = 0, run = 0;
  for (int eb = 0; eb < E; eb += 64) {
    const int ee = eb + lane;
    const int c =
        ee < E ? (seg[ee + 1] - seg[ee] + BM - 1) / BM : 0;
    int inc = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(inc, off, WAVE_SIZE);
      if (lane >= off) inc += o;
    }
    const int tot = __shfl(inc, 63, WAVE_SIZE);
    if (mt < run + tot) {
      const unsigned long long m = __ballot(mt < run + inc);
      const int l = __ffsll((long long)m) - 1;
      e = eb + l;
      mb = mt - run - __shfl(inc - c, l, WAVE_SIZE);
      break;
    }
    run += tot;
  }
  if (e < 0) return;
  const int m0 = seg[e] + mb * BM;
  const int rows = min(BM, seg[e + 1] - m0);
  const char* we = reinterpret_cast<const char*>(
      w_ptrs ? w_ptrs[e]
             : reinterpret_cast<uint64_t>(w + (int64_t)e * N * K *
                                                  (GATED ? 2 : 1)));
  // weight row behind row r of the panel
  auto w_row = [&](int r) -> int64_t {
    if (GATED && r >= CN) return (int64_t)N + min(n0 + r - CN, N - 1);
    return min(n0 + r, N - 1);
  };

  // wave w loads 8-row groups: of the 32 (x rows, then w rows) 8w .. 8w+7,
  // with fp8 of the 16 x groups 4w .. 4w+3
  constexpr int NG = FP8 ? 4 : 8;
  const int l8 = lane >> 3, c8 = lane & 7;
  const bf16* src[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int r = (wave * NG + g) * 8 + l8;
    if (r < BM) {
      const int p = m0 + min(r, rows - 1);
      src[g] = x + (int64_t)(tok ? tok[p] : p) * K;
    } else {
      src[g] = reinterpret_cast<const bf16*>(we) + w_row(r - BM) * K;
    }
  }
#define MT_LOAD(bufi, k0)                                                   \
  _Pragma("unroll") for (int g = 0; g < NG; ++g) {                          \
    const int r8 = (wave * NG + g) * 8;                                     \
    const int kc = min((k0) + (c8 ^ l8) * 8, K - 8);                        \
    __builtin_amdgcn_global_load_lds(                                       \
        (const __attribute__((address_space(1))) void*)(src[g] + kc),       \
        (__attribute__((address_space(3))) void*)(&lds[bufi][r8][0]), 16, 0, \
        0);                                                                 \
  }
  // fp8 weights: a thread takes 32 k of one panel row through registers
  const int fr = threadIdx.x >> 1, fh = threadIdx.x & 1;
  const char* fsrc = FP8 ? we + w_row(fr) * K : nullptr;
  u32x4 fv[2];
  auto f8_load = [&](int k0) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
      fv[t] = load_global<u32x4>(fsrc + min(k0 + fh * 32 + t * 16, K - 16));
  };
  auto f8_store = [&](int bufi) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      bf16* row = &lds[bufi][BM + fr][0];
      const int s = fh * 4 + t * 2;
      *reinterpret_cast<bf16x8_t*>(row + ((s ^ (fr & 7)) * 8)) =
          from_fp8(fv[t][0], fv[t][1]);
      *reinterpret_cast<bf16x8_t*>(row + (((s + 1) ^ (fr & 7)) * 8)) =
          from_fp8(fv[t][2], fv[t][3]);
    }
  };

  const int col = lane & 15, quad = lane >> 4;
  const int wm = (wave & 1) * 64, wn = (wave >> 1) * (GATED ? 32 : 64);
  // panel row of the wave's n tile i: gated tiles 0, 1 gate and 2, 3 up
  auto n_row = [&](int i) {
    return GATED ? wn + (i & 1) * 16 + (i >> 1) * CN : wn + i * 16;
  };
  f32x4 acc[4][4];                       // [n tile][m tile]
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  MT_LOAD(0, 0)
  if (FP8) {
    f8_load(0);
    f8_store(0);
  }
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += BK) {
    sync_lds_copies();
    if (k0 + BK < K) {
      MT_LOAD(buf ^ 1, k0 + BK)
      if (FP8) f8_load(k0 + BK);
    }
    const bool whole = k0 + BK <= K;     // else 32 are left
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      if (kk && !whole) break;
      const int slot = FP8 && whole ? quad * 2 + kk : kk * 4 + quad;
      const int s = (slot ^ (col & 7)) * 8;
      bf16x8_t xf[4], wf[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        xf[i] = *reinterpret_cast<const bf16x8_t*>(
            &lds[buf][wm + i * 16 + col][s]);
        wf[i] = *reinterpret_cast<const bf16x8_t*>(
            &lds[buf][BM + n_row(i) + col][s]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              wf[i], xf[j], acc[i][j], 0, 0, 0);
    }
    if (FP8 && k0 + BK < K) f8_store(buf ^ 1);
    buf ^= 1;
  }
#undef MT_LOAD
  float sc[4][4];
  if (FP8) {
    const char* sp = reinterpret_cast<const char*>(s_ptrs[e]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sc[i][r] = load_global<float>(sp + w_row(n_row(i) + quad * 4 + r) * 4);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int m = wm + j * 16 + col;
    if (m >= rows) continue;
#pragma unroll
    for (int i = 0; i < (GATED ? 2 : 4); ++i) {
      const int n = n0 + wn + i * 16 + quad * 4;
      if (n >= N) continue;              // N is a multiple of 32
      bf16x4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = FP8 ? acc[i][j][r] * sc[i][r] : acc[i][j][r];
        if (GATED) {                     // both rounded to bf16 first
          const float u = FP8 ? acc[i + 2][j][r] * sc[i + 2][r]
                              : acc[i + 2][j][r];
          const float g = bf2f(f2bf(v));
          v = g / (1.f + __expf(-g)) * bf2f(f2bf(u));
        }
        o.v[r] = f2bf(v);
      }
      *reinterpret_cast<bf16x4*>(out + (int64_t)(m0 + m) * N + n) = o;
    }
  }
}

// KS: 32-wide k steps per wave and pass
template <int KS>
__global__ __launch_bounds__(BLOCK) void moe_rows_kernel(
    const bf16* __restrict__ x, const int* __restrict__ tok,
    const int* __restrict__ seg, const bf16* __restrict__ w,
    bf16* __restrict__ out, int N, int K) {
  __shared__ float red[4][16][17];
  const int e = blockIdx.y, n0 = blockIdx.x * 16;
  const int p0 = seg[e], mt = seg[e + 1] - p0;
  if (mt <= 0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, quad = lane >> 4;
  const int steps = K / 32;
  const bf16* wr = w + ((int64_t)e * N + n0 + col) * K + quad * 8;
  for (int mb = 0; mb < mt; mb += 16) {
    const int p = p0 + min(mb + col, mt - 1);
    const bf16* xr = x + (int64_t)(tok ? tok[p] : p) * K + quad * 8;
    f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int s0 = wave * KS; s0 < steps; s0 += 4 * KS) {
      bf16x8_t wf[KS], xf[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int k = min(s0 + s, steps - 1) * 32;
        wf[s] = *reinterpret_cast<const bf16x8_t*>(wr + k);
        xf[s] = *reinterpret_cast<const bf16x8_t*>(xr + k);
      }
#pragma unroll
      for (int s = 0; s < KS; ++s)
        if (s0 + s < steps)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s], xf[s], acc, 0,
                                                        0, 0);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][quad * 4 + r][col] = acc[r];
    __syncthreads();
    // thread (row m, column n) of the 16 x 16 tile
    const int m = threadIdx.x >> 4, n = threadIdx.x & 15;
    if (mb + m < mt) {
      float s = 0.f;
#pragma unroll
      for (int u = 0; u < 4; ++u) s += red[u][n][m];
      out[(int64_t)(p0 + mb + m) * N + n0 + n] = f2bf(s);
    }
  }
}

}  // namespace

extern "C" {

// N a multiple of 64 (gated: of 32), K of 32; w_ptrs null: bf16 stacked
void tl_moe_tiles_any(const void* x, const void* tok, const void* seg,
                      const void* w_ptrs, const void* w, const void* s_ptrs,
                      void* out, int64_t P, int E, int N, int K, int fp8,
                      int gated, hipStream_t stream) {
  if (P <= 0) return;
  // every segment adds at most one partly filled tile
  const int tiles = (int)(P / BM + (P < E ? P : E));
  const int cn = gated ? BN / 2 : BN;
  const int blocks = tiles * ((N + cn - 1) / cn);
#define TL_MT(F, G)                                                          \
  hipLaunchKernelGGL((moe_tile_kernel<F, G>), dim3((blocks + 7) / 8 * 8),    \
                     dim3(BLOCK), 0, stream, (const bf16*)x,                 \
                     (const int*)tok, (const int*)seg,                       \
                     (const uint64_t*)w_ptrs, (const bf16*)w,                \
                     (const uint64_t*)s_ptrs, (bf16*)out, E, N, K, tiles)
  if (fp8) {
    if (gated) TL_MT(1, 1); else TL_MT(1, 0);
  } else {
    if (gated) TL_MT(0, 1); else TL_MT(0, 0);
  }
#undef TL_MT
}

void tl_moe_tiles(const void* x, const void* tok, const void* seg,
                  const void* w, void* out, int P, int E, int N, int K,
                  hipStream_t stream) {
  tl_moe_tiles_any(x, tok, seg, nullptr, w, nullptr, out, P, E, N, K, 0, 0,
                   stream);
}

// N a multiple of 16, K of 32
void tl_moe_rows(const void* x, const void* tok, const void* seg,
                 const void* w, void* out, int P, int E, int N, int K,
                 hipStream_t stream) {
  if (P <= 0) return;
  dim3 grid(N / 16, E), block(BLOCK);
  const int per = (K / 32 + 3) / 4;      // k steps of a wave
#define TL_MR(KS)                                                            \
  hipLaunchKernelGGL(moe_rows_kernel<KS>, grid, block, 0, stream,            \
                     (const bf16*)x, (const int*)tok, (const int*)seg,       \
                     (const bf16*)w, (bf16*)out, N, K)
  if (per <= 1) TL_MR(1);
  else if (per <= 2) TL_MR(2);
  else if (per <= 3) TL_MR(3);
  else if (per <= 4) TL_MR(4);
  else TL_MR(8);
#undef TL_MR
}

}  // extern "C"
