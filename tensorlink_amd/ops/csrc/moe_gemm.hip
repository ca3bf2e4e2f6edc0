// Grouped expert GEMM for MoE serving (gfx950): out[p] = x[tok[p]] @ W[e]^T
// for every (token, expert) pair p, pairs sorted by expert into segments
// (seg[e] <= p < seg[e + 1]). Expert weights come through a device pointer
// table (no stacked copy) or stacked; they may be bf16 or fp8 e4m3 (OCP),
// which the matrix cores take after an exact conversion to bf16, with the
// per-channel scale applied to the fp32 sums. Capture-safe.
//
// Few pairs per expert: the time is that of reading the weights once. A wave
// owns 16 weight rows (the A operand, so a lane ends with four neighbouring
// columns of one pair), loads them straight into registers a step ahead, and
// shares up to 64 pairs' rows in LDS with the block's other waves; a step is
// 256 wide, so barriers are few and 4 KB to 8 KB per wave are in flight. With
// GATED the 16 rows are 8 gate and 8 up rows and the wave writes silu(gate) *
// up, both rounded to bf16 first. Many pairs: moe_tiles.hip.
//
// Measured on MI355X, us for the gated product 1536 x 2048 and the product
// 2048 x 768 of 128 experts, 8 pairs a token (before: a barrier per 64 k, fp8
// by table lookups, the activation in a kernel of its own):
//   tokens            64           512         2400 (bf16: tiles)
//   bf16  before   190 +  93    210 + 109    633 + 268
//         now      152 +  76    179 + 101    341 + 185
//   fp8   before   182 +  70    194 +  82    498 + 242
//         now       86 +  45    114 +  67    345 + 174
// One group (fp8 linear layers) of 3584 x 18944: 16 rows 287 -> 70 us, 64
// rows 293 -> 85 us, 512 rows 2313 -> 231 us (tiles). Loads through the
// table's integers as flat loads cost 15 to 30%.
//
// Contract: K is summed in 64-wide chunks, two mfma_f32_16x16x32_bf16 each,
// in order, by this kernel and by moe_tiles.hip: a pair's row has the same
// bits however many pairs there are. The first product of a chunk takes k =
// 8 q + 0..7 of quad q in bf16, 16 q + 0..7 in fp8 (one 16-byte load).

#include "common.hpp"

namespace {

constexpr int BLOCK = 256;

using f32x4 = __attribute__((ext_vector_type(4))) float;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// 8 fp8 -> bf16, exact
DEVINLINE bf16x8_t from_fp8(uint32_t a, uint32_t b) {
  const bf16x2_t p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.f, false);
  const bf16x2_t p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 1.f, true);
  const bf16x2_t p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, false);
  const bf16x2_t p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 1.f, true);
  return (bf16x8_t){p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// The weights' addresses come as integers: say that they are global memory,
// or flat loads are made, which count as LDS accesses too.
template <typename T>
DEVINLINE T load_global(const char* p) {
  return *reinterpret_cast<const __attribute__((address_space(1))) T*>(
      reinterpret_cast<uint64_t>(p));
}
using u32x4 = __attribute__((ext_vector_type(4))) uint32_t;
using u32x2 = __attribute__((ext_vector_type(2))) uint32_t;
DEVINLINE uint4 load16(const char* p) {
  const u32x4 v = load_global<u32x4>(p);
  return make_uint4(v[0], v[1], v[2], v[3]);
}
DEVINLINE uint2 load8(const char* p) {
  const u32x2 v = load_global<u32x2>(p);
  return make_uint2(v[0], v[1]);
}

struct MoeArgs {
  const bf16* x;              // [T, K] rows
  const int* tok;             // [P] row of x, or null: row p
  const int* seg;             // [E + 1]
  const uint64_t* w_ptrs;     // [E] weights [N, K] (gated [2N, K]), or null
  const bf16* w;              // stacked bf16
  const uint64_t* s_ptrs;     // [E] fp32 scale per weight row (fp8)
  bf16* out;                  // [P, N]
  int N, K;
};

// lane: rows quad * 4 + r of the wave's 16, pair m * 16 + col
template <int FP8, int GATED, int MT>
DEVINLINE void finish(const MoeArgs& a, const f32x4 (&acc)[MT], int m0,
                      int rows, const float sc[4], int c0) {
  const int lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int p = m * 16 + col;
    bf16x4_t o;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      o[r] = (__bf16)(FP8 ? acc[m][r] * sc[r] : acc[m][r]);
      if (GATED) {                           // up sits 32 lanes on
        const float g = (float)o[r], u = __shfl_xor(g, 32, WAVE_SIZE);
        o[r] = (__bf16)(g / (1.f + __expf(-g)) * u);
      }
    }
    if (p < rows && (!GATED || quad < 2))
      *reinterpret_cast<bf16x4_t*>(a.out + (int64_t)(m0 + p) * a.N + c0 +
                                   quad * 4) = o;
  }
}

// The pairs' rows in LDS, shared by the block's four waves: XK wide steps,
// double-buffered, 16-byte slots permuted by row.
constexpr int XK = 256;

template <int FP8, int GATED, int MT>
DEVINLINE void rows_pass(const MoeArgs& a, const char* wr, int m0, int rows,
                        float sc[4], int c0, bf16 (*xs)[64][XK]) {
  const int lane = threadIdx.x & 63, col = lane & 15, quad = lane >> 4;
  const int wave = threadIdx.x >> 6;
  // a copy moves two rows; wave w takes 2 MT of the 8 MT
  const bf16* src[2 * MT];
#pragma unroll
  for (int g = 0; g < 2 * MT; ++g) {
    const int r = (wave * 2 * MT + g) * 2 + (lane >> 5);
    const int p = m0 + min(r, rows - 1);
    src[g] = a.x + (int64_t)(a.tok ? a.tok[p] : p) * a.K;
  }
  auto copy = [&](int buf, int k0) {
#pragma unroll
    for (int g = 0; g < 2 * MT; ++g) {
      const int r0 = (wave * 2 * MT + g) * 2, r = r0 + (lane >> 5);
      const int k = min(k0 + ((lane & 31) ^ (r & 15)) * 8, a.K - 8);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(src[g] + k),
          (__attribute__((address_space(3))) void*)(&xs[buf][r0][0]), 16, 0,
          0);
    }
  };
  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto xf = [&](int buf, int m, int slot) {
    return *reinterpret_cast<const bf16x8_t*>(
        &xs[buf][m * 16 + col][(slot ^ col) * 8]);
  };
  constexpr int NC = XK / 64, WN = FP8 ? 1 : 2;
  uint4 wv[NC][WN];
  auto wload = [&](int k0) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int t = 0; t < WN; ++t)
        wv[c][t] = load16(wr + (k0 + c * 64) * (FP8 ? 1 : 2) + t * 64 +
                          quad * 16);
  };
  auto product = [&](const uint4& lo, const uint4& hi, int t, int slot,
                     int buf) {
    bf16x8_t wf;
    if (FP8)
      wf = t ? from_fp8(lo.z, lo.w) : from_fp8(lo.x, lo.y);
    else
      wf = __builtin_bit_cast(bf16x8_t, t ? hi : lo);
#pragma unroll
    for (int m = 0; m < MT; ++m)
      acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          wf, xf(buf, m, slot), acc[m], 0, 0, 0);
  };
  auto slot_of = [&](int c, int t) {
    return c * 8 + (FP8 ? quad * 2 + t : t * 4 + quad);
  };
  copy(0, 0);
  if (XK <= a.K) wload(0);
  int buf = 0, k0 = 0;
  for (; k0 + XK <= a.K; k0 += XK) {
    uint4 wc[NC][WN];
    sync_lds_copies();
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int t = 0; t < WN; ++t) wc[c][t] = wv[c][t];
    if (k0 + XK < a.K) copy(buf ^ 1, k0 + XK);
    if (k0 + 2 * XK <= a.K) wload(k0 + XK);
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int t = 0; t < 2; ++t)
        product(wc[c][0], wc[c][WN - 1], t, slot_of(c, t), buf);
    buf ^= 1;
  }
  if (k0 < a.K) {                            // less than a step is left
    sync_lds_copies();
    int c = 0;
    for (; k0 + 64 <= a.K; k0 += 64, ++c) {
      const char* w = wr + k0 * (FP8 ? 1 : 2) + quad * 16;
      const uint4 lo = load16(w), hi = FP8 ? lo : load16(w + 64);
#pragma unroll
      for (int t = 0; t < 2; ++t) product(lo, hi, t, slot_of(c, t), buf);
    }
    if (k0 < a.K) {                          // 32: k = 8 q + 0..7
      uint4 v;
      if (FP8) {
        const uint2 u = load8(wr + k0 + quad * 8);
        v = make_uint4(u.x, u.y, 0, 0);
      } else {
        v = load16(wr + k0 * 2 + quad * 16);
      }
      product(v, v, 0, c * 8 + quad, buf);
    }
  }
  __syncthreads();                           // the next pass copies anew
  finish<FP8, GATED, MT>(a, acc, m0, rows, sc, c0);
}

template <int FP8, int GATED>
__global__ __launch_bounds__(BLOCK) void moe_gemm_kernel(MoeArgs a) {
  __shared__ bf16 xs[2][64][XK];
  const int e = blockIdx.y;
  const int m0 = a.seg[e], mt = a.seg[e + 1] - m0;
  if (mt <= 0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, quad = lane >> 4;
  constexpr int CW = GATED ? 8 : 16;         // columns per wave
  const int c0 = (blockIdx.x * 4 + wave) * CW;
  auto row_of = [&](int i) {                 // weight row of the wave's i-th
    return GATED && i >= 8 ? a.N + c0 + i - 8 : c0 + i;
  };
  const char* base = reinterpret_cast<const char*>(
      a.w_ptrs ? a.w_ptrs[e]
               : reinterpret_cast<uint64_t>(a.w + (int64_t)e * a.N * a.K *
                                                      (GATED ? 2 : 1)));
  const char* wr = base + (int64_t)row_of(col) * a.K * (FP8 ? 1 : 2);
  float sc[4] = {1.f, 1.f, 1.f, 1.f};
  if (FP8) {
    const char* s = reinterpret_cast<const char*>(a.s_ptrs[e]);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      sc[r] = load_global<float>(s + (int64_t)row_of(quad * 4 + r) * 4);
  }
  for (int mb = 0; mb < mt; mb += 64) {
    const int rows = min(64, mt - mb);
    if (rows <= 16)
      rows_pass<FP8, GATED, 1>(a, wr, m0 + mb, rows, sc, c0, xs);
    else if (rows <= 32)
      rows_pass<FP8, GATED, 2>(a, wr, m0 + mb, rows, sc, c0, xs);
    else
      rows_pass<FP8, GATED, 4>(a, wr, m0 + mb, rows, sc, c0, xs);
  }
}

}  // namespace

extern "C" {

void tl_moe_tiles_any(const void* x, const void* tok, const void* seg,
                      const void* w_ptrs, const void* w, const void* s_ptrs,
                      void* out, int64_t P, int E, int N, int K, int fp8,
                      int gated, hipStream_t stream);

// N: columns of out, a multiple of 64 (gated: of 32); K a multiple of 32.
// w_ptrs [E], or null and w stacked (bf16). P: an upper bound of the pairs.
// Tiles of 128 pairs pay once an expert has about half of one in bf16 (32
// pairs 179 + 101 against 200 + 108 us, 64 pairs 277 + 132 against 229 + 132),
// in fp8, where their weights pass through registers, once it has more than
// one (64 pairs 183 against 232 us, 150 pairs 345 against 331; one group of
// 128 rows on 3584 x 18944 166 against 223, of 256 rows 328 against 225).
void tl_moe_gemm(const void* x, const void* tok, const void* seg,
                 const void* w_ptrs, const void* w, const void* s_ptrs,
                 void* out, int64_t P, int E, int N, int K, int fp8,
                 int gated, hipStream_t stream) {
  if (P <= 0) return;
  if (fp8 ? P >= 160 * (int64_t)E : P >= 48 * (int64_t)E && P >= 1024) {
    tl_moe_tiles_any(x, tok, seg, w_ptrs, w, s_ptrs, out, P, E, N, K, fp8,
                     gated, stream);
    return;
  }
  const MoeArgs a{(const bf16*)x, (const int*)tok, (const int*)seg,
                  (const uint64_t*)w_ptrs, (const bf16*)w,
                  (const uint64_t*)s_ptrs, (bf16*)out, N, K};
  const dim3 grid(N / (gated ? 32 : 64), E), block(BLOCK);
#define TL_MG(F, G)                                                          \
  hipLaunchKernelGGL((moe_gemm_kernel<F, G>), grid, block, 0, stream, a)
  if (fp8) {
    if (gated) TL_MG(1, 1); else TL_MG(1, 0);
  } else {
    if (gated) TL_MG(0, 1); else TL_MG(0, 0);
  }
#undef TL_MG
}

}  // extern "C"
