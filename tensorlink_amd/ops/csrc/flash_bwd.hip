// Causal GQA flash-attention BACKWARD on gfx950 MFMA (training path).
//
// P is recomputed from the forward's logsumexp. As in the forward
// (prefill_attn.hip) every score tile is formed in the orientation in which
// its accumulator registers are the B operand of the next product, so
// neither P nor dS passes through LDS; the other operand comes from the
// transposing LDS reads of a tile that is there already.
//
//   prep   one pass over dO and O: Delta = rowsum(dO * O), and the logsumexp
//          in log2 units, both padded to whole query tiles (padding rows get
//          +inf, which makes their P zero).
//   dK/dV  block = 4 waves x 32 keys, K and V of a wave in registers; 64-row
//          tiles of Q and dO stream through LDS, double-buffered:
//            S = Q K^T   dP = dO V^T         (a lane owns one key)
//            dV^T += dO^T P     dK^T += Q^T dS
//          The query heads of a kv head are cut into `parts` blocks where
//          the key tiles alone leave CUs idle; their fp32 sums are then
//          added in order.
//   dQ     block = 4 waves x 32 queries; 64-row tiles of K and V:
//            S^T = K Q^T  dP^T = V dO^T      (a lane owns one query)
//            dQ^T += K^T dS^T
//
// The 7 products take 32 + 24 MFMAs per 32 x 32 scores and wave; the LDS
// reads (32 and 24 KB) need as many cycles. dQ keeps two waves per SIMD to
// overlap the two. dK/dV with D 128 needs 324 registers to have more than
// one operand read ahead of its product: with one wave per SIMD it takes 438
// us at 1 x 4096 rows, 32/8 heads, within 256 registers and two waves 643.
//
// Measured on MI355X, causal, prep included (before: 16x16x32 tiles, P and
// dS through LDS, Delta from library calls): 2 x 2048 rows, 28/4 heads, D
// 128, 2330 -> 374 us; 4 x 512 rows, 12 heads, D 64, 95 -> 41 us.
// All accumulation in f32; inputs/outputs bf16 except lse f32.

#include "common.hpp"

namespace {

constexpr int NW = 4;        // waves per block, 32 keys or rows each
constexpr int BM = NW * 32;
constexpr int BT = 64;       // rows of a streamed tile

using f32x16 = __attribute__((ext_vector_type(16))) float;
using f32x4 = __attribute__((ext_vector_type(4))) float;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

constexpr float LOG2E = 1.4426950408889634f;

struct BwdArgs {
  const bf16 *q, *k, *v, *dout, *out;
  const float* lse;           // [B, Hq, S]
  float *l2, *delta;          // [B, Hq, Sp]
  bf16 *dq, *dk, *dv;
  float *pk, *pv;             // parts > 1: [parts, B, S, Hkv, D]
  int B, S, Sp, Hq, Hkv, causal, parts;
  float scale;
};

// 16-byte slot permutation within a tile row: 16 rows at one slot (the b128
// row reads) and four rows at 64 bytes (the transposing reads) both cover
// all banks once.
template <int D>
DEVINLINE int perm(int row) {
  return D == 128 ? (((row & 3) << 2) | ((row >> 2) & 3))
                  : ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
}

// blocks go round robin over the 8 XCDs: give each XCD its own groups where
// their number allows, so that a group's tiles are read from one L2
DEVINLINE void block_of(int id, int groups, int* group, int* tile) {
  if ((groups & 7) == 0) {
    const int per = groups >> 3, r = id >> 3;
    *group = (id & 7) * per + r % per;
    *tile = r / per;
  } else {
    *group = id % groups;
    *tile = id / groups;
  }
}

// Copies 64 rows of two operands to LDS; rows past the end repeat the last.
template <int D>
struct Tile {
  static constexpr int SL = D / 8, RPC = 64 / SL, CPW = BT / RPC / NW;
  int off[CPW], row[CPW], wave;
  DEVINLINE void init(int lane, int w) {
    wave = w;
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
      row[i] = (w * CPW + i) * RPC + lane / SL;
      off[i] = ((lane % SL) ^ perm<D>(row[i])) * 8;
    }
  }
  DEVINLINE void copy(const bf16* a, const bf16* b, int stride, int left,
                      bf16 (*la)[D], bf16 (*lb)[D]) const {
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
      const int o = min(row[i], left - 1) * stride + off[i];
      const int r0 = (wave * CPW + i) * RPC;
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(a + o),
          (__attribute__((address_space(3))) void*)(&la[r0][0]), 16, 0, 0);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(b + o),
          (__attribute__((address_space(3))) void*)(&lb[r0][0]), 16, 0, 0);
    }
  }
};

// Byte offsets of a lane's reads of a tile: row operand (row l32, slots
// 2c + half) and transposed operand (rows 8u + 4 half + i, 32 columns n). The
// slot permutation is an xor, so c, n and u are xors on one offset each; a
// register per c and (n, u) would spill in the dK/dV kernel, hence fresh().
template <int D>
struct Reads {
  unsigned row, col;
  DEVINLINE void init(int lane) {
    const int half = lane >> 5, l32 = lane & 31;
    row = l32 * D * 2 + ((half ^ perm<D>(l32)) * 16);
    const int e = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
    const int r = half * 4 + ((lane >> 2) & 3);
    col = r * D * 2 + ((e ^ perm<D>(r)) * 16) + (lane & 1) * 8;
  }
  static DEVINLINE unsigned fresh(unsigned x) {
    asm volatile("" : "+v"(x));              // not to be hoisted
    return x;
  }
  static DEVINLINE bf16x8_t rows(const bf16* t, unsigned at, int c) {
    return *reinterpret_cast<const bf16x8_t*>(
        reinterpret_cast<const char*>(t) + (at ^ (c * 32)));
  }
  static DEVINLINE bf16x8_t cols(const bf16* t, unsigned at, int n) {
    typedef __attribute__((address_space(3))) bf16x4_t* l4;
    const char* p = reinterpret_cast<const char*>(t);
    const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
        (l4)(p + (at ^ (n * 64))));
    const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
        (l4)(p + (at ^ (n * 64 + 32)) + 16 * D));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

template <int N>
DEVINLINE void clear(f32x16 (&x)[N]) {
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) x[n][r] = 0.f;
}

#define MFMA(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0)

// D / 8 lanes per row, 8 elements each
template <int D>
__global__ __launch_bounds__(256) void attn_bwd_prep_kernel(BwdArgs a) {
  constexpr int L = D / 8;
  const int64_t at =
      (int64_t)blockIdx.x * (256 / L) + threadIdx.x / L;   // (b, s, h)
  if (at >= (int64_t)a.B * a.Sp * a.Hq) return;
  const int h = (int)(at % a.Hq);
  const int s = (int)((at / a.Hq) % a.Sp), b = (int)(at / a.Hq / a.Sp);
  const int64_t to = ((int64_t)b * a.Hq + h) * a.Sp + s;
  float sum = 0.f;
  if (s < a.S) {
    const int64_t from = (((int64_t)b * a.S + s) * a.Hq + h) * D +
                         (threadIdx.x % L) * 8;
    const bf16x8_t x = *reinterpret_cast<const bf16x8_t*>(a.dout + from);
    const bf16x8_t y = *reinterpret_cast<const bf16x8_t*>(a.out + from);
#pragma unroll
    for (int j = 0; j < 8; ++j) sum += (float)x[j] * (float)y[j];
  }
  sum = group_reduce_sum<L>(sum);
  if (threadIdx.x % L) return;
  const float l =
      s < a.S ? a.lse[((int64_t)b * a.Hq + h) * a.S + s] : -1e30f;
  a.l2[to] = l <= -1e29f ? INFINITY : l * LOG2E;
  a.delta[to] = sum;
}

// ------------------------------ dK / dV ------------------------------
template <int D>
__global__ __launch_bounds__(NW * 64, D == 128 ? 1 : 2) void attn_bwd_dkv_kernel(BwdArgs a) {
  constexpr int KS = D / 16, NV = D / 32;
  __shared__ bf16 lds[2][2][BT][D];          // [buffer][q|do]
  __shared__ float ld[2][2][BT];             // [buffer][l2|delta]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, l32 = lane & 31;
  const int G = a.Hq / a.Hkv, gp = (G + a.parts - 1) / a.parts;
  int grp, kt;
  block_of(blockIdx.x, a.B * a.Hkv * a.parts, &grp, &kt);
  const int part = grp % a.parts, bh = grp / a.parts;
  const int b = bh / a.Hkv, hkv = bh - b * a.Hkv;
  const int k0 = kt * BM, key0 = k0 + wave * 32, key = key0 + l32;
  const int g_end = min(G, (part + 1) * gp);

  bf16x8_t kf[KS], vf[KS];
  {
    const int64_t o =
        (((int64_t)b * a.S + min(key, a.S - 1)) * a.Hkv + hkv) * D + half * 8;
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      kf[c] = *reinterpret_cast<const bf16x8_t*>(a.k + o + c * 16);
      vf[c] = *reinterpret_cast<const bf16x8_t*>(a.v + o + c * 16);
    }
  }
  f32x16 dk[NV], dv[NV];
  clear(dk);
  clear(dv);
  Tile<D> tile;
  tile.init(lane, wave);
  Reads<D> rd;
  rd.init(lane);
  const float c2 = a.scale * LOG2E;

  // (head, query tile) pairs in one sequence, so the copies run ahead
  const int qt0 = a.causal ? k0 / BT : 0, nt = (a.S + BT - 1) / BT - qt0;
  const int n = (g_end - part * gp) * nt;
  auto copy = [&](int i, int buf) {
    const int h = hkv * G + part * gp + i / nt, t0 = (qt0 + i % nt) * BT;
    const int64_t o = (((int64_t)b * a.S + t0) * a.Hq + h) * D;
    tile.copy(a.q + o, a.dout + o, a.Hq * D, a.S - t0, lds[buf][0],
              lds[buf][1]);
    if (wave < 2) {
      const float* src = (wave ? a.delta : a.l2) +
                         ((int64_t)b * a.Hq + h) * a.Sp + t0 + lane;
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)src,
          (__attribute__((address_space(3))) void*)(&ld[buf][wave][0]), 4, 0,
          0);
    }
  };
  if (n > 0) copy(0, 0);
  for (int i = 0; i < n; ++i) {
    const int buf = i & 1;
    sync_lds_copies();         // this tile has landed; the other is free
    if (i + 1 < n) copy(i + 1, buf ^ 1);
    const int t0 = (qt0 + i % nt) * BT;
#pragma unroll
    for (int qs = 0; qs < BT; qs += 32) {
      if (a.causal && t0 + qs + 31 < key0) continue;
      const bf16* qt = &lds[buf][0][qs][0];
      const bf16* dt = &lds[buf][1][qs][0];
      const unsigned ra = rd.fresh(rd.row), ca = rd.fresh(rd.col);
      f32x16 s[1], dp[1];
      clear(s);
      clear(dp);
#pragma unroll
      for (int c = 0; c < KS; ++c) s[0] = MFMA(rd.rows(qt, ra, c), kf[c], s[0]);
#pragma unroll
      for (int c = 0; c < KS; ++c)
        dp[0] = MFMA(rd.rows(dt, ra, c), vf[c], dp[0]);
      bf16x8_t p[2], ds[2];
      const bool diag = a.causal && t0 + qs < key0 + 31;
#pragma unroll
      for (int g = 0; g < 4; ++g) {          // queries 8 g + 4 half + j
        const f32x4 l = *reinterpret_cast<const f32x4*>(
            &ld[buf][0][qs + g * 8 + half * 4]);
        const f32x4 de = *reinterpret_cast<const f32x4*>(
            &ld[buf][1][qs + g * 8 + half * 4]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = g * 4 + j;
          float e = __builtin_amdgcn_exp2f(fmaf(s[0][r], c2, -l[j]));
          if (diag && key > t0 + qs + g * 8 + half * 4 + j) e = 0.f;
          p[r >> 3][r & 7] = (__bf16)e;
          ds[r >> 3][r & 7] = (__bf16)(e * (dp[0][r] - de[j]));
        }
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int m = 0; m < NV; ++m) {
          dv[m] = MFMA(rd.cols(dt + t * 16 * D, ca, m), p[t], dv[m]);
          dk[m] = MFMA(rd.cols(qt + t * 16 * D, ca, m), ds[t], dk[m]);
        }
    }
  }

  // lane: its key's elements 32 m + 8 g + 4 half + 0..3
  if (key >= a.S) return;
  const int64_t o =
      (((int64_t)b * a.S + key) * a.Hkv + hkv) * D + half * 4;
  const int64_t po = (int64_t)part * a.B * a.S * a.Hkv * D + o;
#pragma unroll
  for (int m = 0; m < NV; ++m)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 x, y;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[j] = dk[m][g * 4 + j] * a.scale;
        y[j] = dv[m][g * 4 + j];
      }
      const int e = m * 32 + g * 8;
      if (a.parts > 1) {
        *reinterpret_cast<f32x4*>(a.pk + po + e) = x;
        *reinterpret_cast<f32x4*>(a.pv + po + e) = y;
      } else {
        *reinterpret_cast<bf16x4_t*>(a.dk + o + e) =
            __builtin_convertvector(x, bf16x4_t);
        *reinterpret_cast<bf16x4_t*>(a.dv + o + e) =
            __builtin_convertvector(y, bf16x4_t);
      }
    }
}

__global__ __launch_bounds__(256) void attn_bwd_sum_kernel(BwdArgs a,
                                                           int64_t n) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  const float* src = blockIdx.y ? a.pv : a.pk;
  f32x4 x = *reinterpret_cast<const f32x4*>(src + i);
  for (int p = 1; p < a.parts; ++p)
    x += *reinterpret_cast<const f32x4*>(src + p * n + i);
  *reinterpret_cast<bf16x4_t*>((blockIdx.y ? a.dv : a.dk) + i) =
      __builtin_convertvector(x, bf16x4_t);
}

// -------------------------------- dQ ---------------------------------
template <int D>
__global__ __launch_bounds__(NW * 64, 2) void attn_bwd_dq_kernel(BwdArgs a) {
  constexpr int KS = D / 16, NV = D / 32;
  __shared__ bf16 lds[2][2][BT][D];          // [buffer][k|v]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, l32 = lane & 31;
  const int n_qt = (a.S + BM - 1) / BM;
  int bh, qt;
  block_of(blockIdx.x, a.B * a.Hq, &bh, &qt);
  qt = n_qt - 1 - qt;                        // most keys first
  const int b = bh / a.Hq, h = bh - b * a.Hq, hkv = h / (a.Hq / a.Hkv);
  const int q0 = qt * BM, w0 = q0 + wave * 32, row = w0 + l32;

  bf16x8_t qf[KS], df[KS];
  {
    const int64_t o =
        (((int64_t)b * a.S + min(row, a.S - 1)) * a.Hq + h) * D + half * 8;
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      qf[c] = *reinterpret_cast<const bf16x8_t*>(a.q + o + c * 16);
      df[c] = *reinterpret_cast<const bf16x8_t*>(a.dout + o + c * 16);
    }
  }
  const int64_t lo = ((int64_t)b * a.Hq + h) * a.Sp + min(row, a.Sp - 1);
  const float l = a.l2[lo], de = a.delta[lo];
  f32x16 dq[NV];
  clear(dq);
  Tile<D> tile;
  tile.init(lane, wave);
  Reads<D> rd;
  rd.init(lane);
  const float c2 = a.scale * LOG2E;
  const int kv_end = a.causal ? min(a.S, q0 + BM) : a.S;
  const int n = (kv_end + BT - 1) / BT;
  auto copy = [&](int i, int buf) {
    const int64_t o = (((int64_t)b * a.S + i * BT) * a.Hkv + hkv) * D;
    tile.copy(a.k + o, a.v + o, a.Hkv * D, a.S - i * BT, lds[buf][0],
              lds[buf][1]);
  };
  copy(0, 0);
  for (int i = 0; i < n; ++i) {
    const int buf = i & 1, t0 = i * BT;
    sync_lds_copies();         // this tile has landed; the other is free
    if (i + 1 < n) copy(i + 1, buf ^ 1);
#pragma unroll
    for (int ks = 0; ks < BT; ks += 32) {
      if (t0 + ks >= a.S || (a.causal && t0 + ks > w0 + 31)) continue;
      const bf16* kt = &lds[buf][0][ks][0];
      const bf16* vt = &lds[buf][1][ks][0];
      const unsigned ra = rd.fresh(rd.row), ca = rd.fresh(rd.col);
      f32x16 s[1], dp[1];
      clear(s);
      clear(dp);
#pragma unroll
      for (int c = 0; c < KS; ++c) s[0] = MFMA(rd.rows(kt, ra, c), qf[c], s[0]);
#pragma unroll
      for (int c = 0; c < KS; ++c)
        dp[0] = MFMA(rd.rows(vt, ra, c), df[c], dp[0]);
      bf16x8_t ds[2];
      const bool edge =
          (a.causal && t0 + ks + 31 > w0) || t0 + ks + 32 > a.S;
      const int lim = a.causal ? min(row, a.S - 1) : a.S - 1;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float e = __builtin_amdgcn_exp2f(fmaf(s[0][r], c2, -l));
        if (edge && t0 + ks + 8 * (r >> 2) + 4 * half + (r & 3) > lim)
          e = 0.f;
        ds[r >> 3][r & 7] = (__bf16)(e * (dp[0][r] - de));
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int m = 0; m < NV; ++m)
          dq[m] = MFMA(rd.cols(kt + t * 16 * D, ca, m), ds[t], dq[m]);
    }
  }
  if (row >= a.S) return;
  bf16* op = a.dq + (((int64_t)b * a.S + row) * a.Hq + h) * D + half * 4;
#pragma unroll
  for (int m = 0; m < NV; ++m)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 x;
#pragma unroll
      for (int j = 0; j < 4; ++j) x[j] = dq[m][g * 4 + j] * a.scale;
      *reinterpret_cast<bf16x4_t*>(op + m * 32 + g * 8) =
          __builtin_convertvector(x, bf16x4_t);
    }
}
#undef MFMA

template <int D>
void launch(const BwdArgs& a, hipStream_t stream) {
  const int64_t rows = (int64_t)a.B * a.Sp * a.Hq;
  const int rpb = 256 / (D / 8), tiles = cdiv(a.S, BM);
  hipLaunchKernelGGL((attn_bwd_prep_kernel<D>),
                     dim3((uint32_t)((rows + rpb - 1) / rpb)), dim3(256), 0,
                     stream, a);
  hipLaunchKernelGGL((attn_bwd_dkv_kernel<D>),
                     dim3((uint32_t)(tiles * a.B * a.Hkv * a.parts)),
                     dim3(NW * 64), 0, stream, a);
  if (a.parts > 1) {
    const int64_t n = (int64_t)a.B * a.S * a.Hkv * D;
    hipLaunchKernelGGL(attn_bwd_sum_kernel,
                       dim3((uint32_t)((n / 4 + 255) / 256), 2), dim3(256), 0,
                       stream, a, n);
  }
  hipLaunchKernelGGL((attn_bwd_dq_kernel<D>),
                     dim3((uint32_t)(tiles * a.B * a.Hq)), dim3(NW * 64), 0,
                     stream, a);
}

}  // namespace

extern "C" {

// Query rows are padded to whole tiles in l2 and delta.
int tl_attn_bwd_rows(int S) { return cdiv(S, BT) * BT; }

// Blocks per kv head and key tile: two blocks per CU keep the chip busy, and
// a kv head's query heads are cut until there are that many (2 x 2048 rows, 4
// kv heads: 128 key tiles).
int tl_attn_bwd_parts(int B, int S, int Hq, int Hkv) {
  const int G = Hq / Hkv;
  const int64_t blocks = (int64_t)cdiv(S, BM) * B * Hkv;
  int parts = 1;
  while (parts < G && blocks * parts < 512) ++parts;
  return cdiv(G, cdiv(G, parts));            // none of them empty
}

// l2, delta: fp32 scratch [B, Hq, tl_attn_bwd_rows(S)]; pk, pv: fp32 scratch
// [parts, B, S, Hkv, D], unused with one part.
void tl_attn_bwd(const void* q, const void* k, const void* v,
                 const void* dout, const void* out, const void* lse,
                 void* l2, void* delta, void* dq, void* dk, void* dv,
                 void* pk, void* pv, int B, int S, int Hq, int Hkv, int D,
                 float scale, int causal, int parts, hipStream_t stream) {
  if (B <= 0 || S <= 0 || Hq <= 0) return;
  const BwdArgs a{(const bf16*)q, (const bf16*)k, (const bf16*)v,
                  (const bf16*)dout, (const bf16*)out, (const float*)lse,
                  (float*)l2, (float*)delta, (bf16*)dq, (bf16*)dk, (bf16*)dv,
                  (float*)pk, (float*)pv, B, S, tl_attn_bwd_rows(S), Hq, Hkv,
                  causal, parts, scale};
  if (D == 128) launch<128>(a, stream);
  else if (D == 64) launch<64>(a, stream);
}

}  // extern "C"
