// Causal GQA flash-attention forward (prefill) on gfx950 MFMA.
//
// Replaces the reference's HF SDPA-inside-eager-blocks prefill
// (tensorlink/ml/worker.py:330-335).
//
// The scores are formed transposed, S^T = K Q^T, with 32x32x16 MFMAs: a lane
// then holds 32 keys of ONE query, so the row maximum and sum are in-lane
// reductions plus one exchange with lane ^ 32, and the accumulator registers
// ARE the B operand of O^T = V^T P^T once the keys of a 16-key step are
// counted in the accumulator's order (4h..4h+3, 8+4h..8+4h+3 for lane half
// h). ds_read_b64_tr_b16 delivers V^T in exactly that order, so P never
// leaves the registers. What bounds it: the matrix cores, the exponentials
// (16 per lane and 32 keys) and the LDS reads (32 KB per wave and 64 keys)
// each need about 1000 cycles per 64-key tile and wave, so the block keeps
// two waves per SIMD to overlap them.
//
//   wave = 32 query rows; block = NW waves; K and V tiles of 64 keys, double
//   buffered, copied by global_load_lds (16-byte slots permuted by key row on
//   the source address, so neither the b128 K reads nor the transposing V
//   reads meet bank conflicts).
//
// A row's result depends on its own keys only: tiles start at key 0 whatever
// the query tile, and the running maximum is a per-row decision. With
// SPLIT, keys are cut at multiples of SEG into grid slices that a second
// kernel merges in order; a row of one slice keeps its bits (exp2(0) = 1).
//
// Measured on MI355X (D 128, causal; before: 16x16x32 tiles with P through
// LDS, library attention from 4096 rows on): 1 x 7001 rows, 32/8 heads, 1284
// -> 440 us (912 TFLOP/s); 32 x 512, 28/4 heads, 408 -> 128 us; 512 rows over
// 3968 keys 223 -> 53 us; 1 x 333 rows 24 -> 12 us. Blocks of 8 waves are
// within 10% on either side (4096 rows 167 -> 151 us, 512 rows 128 -> 144),
// of 2 waves slower everywhere but at 4 x 512 rows of D 64 (12.1 -> 11.4).
//
// q [B,Sq,Hq,D]; k, v rows of D at (batch, head, token) strides, or pages
// [n_pages,Hkv,128,D] with a block table; out [B,Sq,Hq,D].

#include "common.hpp"

namespace {

constexpr int BN = 64;       // keys per tile
constexpr int NW = 4;        // waves per block
constexpr int SEG = 1024;    // keys per slice when the keys are split

using f32x16 = __attribute__((ext_vector_type(16))) float;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;

struct PrefillArgs {
  const bf16* q;
  const bf16* k;
  const bf16* v;
  const int* table;           // [B, bt_stride] pages, or null
  bf16* out;
  float* lse;                 // [B, Hq, Sq] or null
  float* po;                  // SPLIT: [nseg, B, Sq, Hq, D]
  float* pml;                 // SPLIT: [nseg, B, Sq, Hq, 2] (log2 max, sum)
  int64_t kbs, khs;           // batch and head strides of k and v
  int kts;                    // token stride
  int B, Sq, Skv, q_off, Hq, Hkv, bt_stride, causal, n_qt;
  float scale;
};

// 16-byte slot permutations within a row of D elements (8 or 16 slots): K
// rows are read 16 at a time at one slot, V four rows at a time over 64
// bytes. A 64-element row is half of the 256 bytes that the banks span.
template <int D>
DEVINLINE int k_perm(int row) {
  return D == 128 ? (row & 15) : ((row >> 1) & 7);
}
template <int D>
DEVINLINE int v_perm(int row) {
  return D == 128 ? (((row & 3) << 2) | ((row >> 2) & 3))
                  : ((((row >> 1) & 1) << 2) | ((row >> 2) & 3));
}

template <int D, int SPLIT>
__global__ __launch_bounds__(NW * 64, 2) void prefill_attn_kernel(
    PrefillArgs a) {
  constexpr int BM = NW * 32;
  constexpr int SL = D / 8;                  // 16-byte slots per row
  constexpr int RPC = 64 / SL;               // rows per 1 KB copy
  constexpr int CPW = BN / RPC / NW;         // copies per wave and operand
  constexpr int KS = D / 16;                 // QK steps
  constexpr int NV = D / 32;                 // dv tiles
  static_assert(CPW >= 1, "");

  __shared__ bf16 lds[2][2][BN][D];          // [buffer][k|v]

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, l32 = lane & 31;

  // Late query tiles first: under the causal mask they have the most keys.
  // Heads are cut into 8 stretches, one per XCD (blocks go round robin), so
  // that a kv head's query heads meet in one L2.
  const int n_bh = a.B * a.Hq;
  const int id = blockIdx.x;
  int bh, qt;
  if ((n_bh & 7) == 0) {
    const int per = n_bh >> 3, r = id >> 3;
    bh = (id & 7) * per + r % per;
    qt = a.n_qt - 1 - r / per;
  } else {
    bh = id % n_bh;
    qt = a.n_qt - 1 - id / n_bh;
  }
  const int b = bh / a.Hq, h = bh - b * a.Hq;
  const int hkv = h / (a.Hq / a.Hkv);
  const int q0 = qt * BM, w0 = q0 + wave * 32;

  int kv_end = a.causal ? min(a.Skv, a.q_off + q0 + BM) : a.Skv;
  int kv_begin = 0;
  if (SPLIT) {
    kv_begin = blockIdx.y * SEG;
    if (kv_begin >= kv_end) return;
    kv_end = min(kv_end, kv_begin + SEG);
  }

  // ---- Q: B operand, query l32, all KS steps; scale folded into exp2 ----
  const int row = w0 + l32;
  bf16x8_t qf[KS];
  {
    const bf16* qp =
        a.q + (((int64_t)b * a.Sq + min(row, a.Sq - 1)) * a.Hq + h) * D +
        half * 8;
#pragma unroll
    for (int c = 0; c < KS; ++c)
      qf[c] = *reinterpret_cast<const bf16x8_t*>(qp + c * 16);
  }
  float c2 = a.scale * LOG2E;
  if (c2 < 0.f) {                            // exact: flip the query's sign
    c2 = -c2;
#pragma unroll
    for (int c = 0; c < KS; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[c][j] = -qf[c][j];
  }
  c2 = fmaxf(c2, 1e-30f);
  const int qpos = a.q_off + row;            // this lane's last key

  // ---- copies: chunk c = rows c * RPC.., lane -> (row, slot) ----
  const int crow = lane / SL, cslot = lane % SL;
  int koff[CPW], voff[CPW], lrow[CPW];
#pragma unroll
  for (int i = 0; i < CPW; ++i) {
    lrow[i] = (wave * CPW + i) * RPC + crow;
    koff[i] = (cslot ^ k_perm<D>(lrow[i])) * 8;
    voff[i] = (cslot ^ v_perm<D>(lrow[i])) * 8;
  }
  const int64_t base = (int64_t)b * a.kbs + (int64_t)hkv * a.khs;

  auto copy = [&](int buf, int kt0) {
    int64_t tb;
    if (a.table) {
      const int page = a.table[(int64_t)b * a.bt_stride + (kt0 >> 7)];
      tb = ((int64_t)page * a.Hkv + hkv) * 128 * D + (int64_t)(kt0 & 127) * D;
    } else {
      tb = base + (int64_t)kt0 * a.kts;
    }
    const bf16* kp = a.k + tb;
    const bf16* vp = a.v + tb;
    const int last = a.Skv - 1 - kt0;        // rows past the end repeat it
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
      const int ro = min(lrow[i], last) * a.kts;
      const int r0 = (wave * CPW + i) * RPC;
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(kp + ro + koff[i]),
          (__attribute__((address_space(3))) void*)(&lds[buf][0][r0][0]), 16,
          0, 0);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(vp + ro + voff[i]),
          (__attribute__((address_space(3))) void*)(&lds[buf][1][r0][0]), 16,
          0, 0);
    }
  };

  float m_run = -1e30f, l_run = 0.f;         // log2 units; l of this half
  f32x16 o[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[n][r] = 0.f;

  // element offsets of the transposing V reads: rows 16 ks + 8 u + 4 half + i
  const int vi = (lane >> 2) & 3;
  const int ve = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
  int vaddr[NV][2];
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = u * 8 + half * 4 + vi;
      vaddr[n][u] =
          r * D + (((n * 4 + ve) ^ v_perm<D>(r)) * 8) + (lane & 1) * 4;
    }
  int kaddr[KS];
#pragma unroll
  for (int c = 0; c < KS; ++c)
    kaddr[c] = l32 * D + (((c * 2 + half) ^ k_perm<D>(l32)) * 8);

  copy(0, kv_begin);
  int buf = 0;
  for (int kt0 = kv_begin; kt0 < kv_end; kt0 += BN) {
    sync_lds_copies();         // this tile has landed; the other is free
    if (kt0 + BN < kv_end) copy(buf ^ 1, kt0 + BN);
    // whole tile past this wave's last key: nothing to add
    if (!a.causal || kt0 <= a.q_off + w0 + 31) {
      const bf16* kl = &lds[buf][0][0][0];
      const bf16* vl = &lds[buf][1][0][0];
      f32x16 s[2];
#pragma unroll
      for (int n = 0; n < 2; ++n) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[n][r] = 0.f;
#pragma unroll
        for (int c = 0; c < KS; ++c) {
          const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(
              kl + n * 32 * D + kaddr[c]);
          s[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[c], s[n], 0,
                                                         0, 0);
        }
      }
      // ---- mask, only where the tile meets the diagonal or the end ----
      if ((a.causal && kt0 + BN - 1 > a.q_off + w0) || kt0 + BN > a.Skv) {
        const int lim = a.causal ? min(qpos, a.Skv - 1) : a.Skv - 1;
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = kt0 + n * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
            if (key > lim) s[n][r] = -INFINITY;
          }
      }
      float mx = s[0][0];
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[n][r]);
      {
        const unsigned u = __float_as_uint(mx);
        const auto e = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        mx = fmaxf(__uint_as_float(e[0]), __uint_as_float(e[1])) * c2;
      }
      // The reference maximum moves only when it is exceeded by 2^8: P and
      // the sums stay far inside the fp32 range, and O is rarely rescaled.
      const bool up = mx > m_run + 8.f;
      if (__any(up)) {
        const float alpha =
            up ? __builtin_amdgcn_exp2f(m_run - mx) : 1.f;
        m_run = up ? mx : m_run;
        l_run *= alpha;
#pragma unroll
        for (int n = 0; n < NV; ++n)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[n][r] *= alpha;
      }
      bf16x8_t p[4];
      float ps[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float e =
              __builtin_amdgcn_exp2f(fmaf(s[n][r], c2, -m_run));
          ps[r & 3] += e;
          p[n * 2 + (r >> 3)][r & 7] = (__bf16)e;
        }
      l_run += (ps[0] + ps[1]) + (ps[2] + ps[3]);
      // ---- O^T += V^T P^T ----
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
#pragma unroll
        for (int n = 0; n < NV; ++n) {
          typedef __attribute__((address_space(3))) bf16x4_t* l4;
          const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (l4)(vl + ks * 16 * D + vaddr[n][0]));
          const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (l4)(vl + ks * 16 * D + vaddr[n][1]));
          const bf16x8_t vf =
              __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          o[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, p[ks], o[n], 0,
                                                         0, 0);
        }
      }
    }
    buf ^= 1;
  }

  // ---- epilogue: lane holds dv n * 32 + 8 g + 4 half + 0..3 of its row ----
  const float l = l_run + __shfl_xor(l_run, 32, WAVE_SIZE);
  if (row >= a.Sq) return;
  if (SPLIT) {
    const int64_t at = (((int64_t)blockIdx.y * a.B + b) * a.Sq + row) * a.Hq +
                       h;
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<float4*>(a.po + at * D + n * 32 + g * 8 +
                                   half * 4) =
            make_float4(o[n][g * 4], o[n][g * 4 + 1], o[n][g * 4 + 2],
                        o[n][g * 4 + 3]);
    if (half == 0)
      *reinterpret_cast<float2*>(a.pml + at * 2) = make_float2(m_run, l);
    return;
  }
  const float linv = l > 0.f ? 1.f / l : 0.f;
  bf16* op = a.out + (((int64_t)b * a.Sq + row) * a.Hq + h) * D + half * 4;
#pragma unroll
  for (int n = 0; n < NV; ++n)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bf16x4_t w;
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = (__bf16)(o[n][g * 4 + r] * linv);
      *reinterpret_cast<bf16x4_t*>(op + n * 32 + g * 8) = w;
    }
  if (a.lse && half == 0)
    a.lse[((int64_t)b * a.Hq + h) * a.Sq + row] =
        l > 0.f ? (m_run + __log2f(l)) * LN2 : -1e30f;
}

// One wave per (b, row, head): the row's own slices in key order.
template <int D>
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t n = (int64_t)a.B * a.Sq * a.Hq;
  const int64_t at = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (at >= n) return;
  const int row = (int)((at / a.Hq) % a.Sq);
  const int last = a.causal ? min(a.q_off + row, a.Skv - 1) : a.Skv - 1;
  const int ns = last / SEG + 1;
  float m = -1e30f;
  for (int s = 0; s < ns; ++s) m = fmaxf(m, a.pml[(s * n + at) * 2]);
  constexpr int E = D / 64;
  float l = 0.f, o[E];
#pragma unroll
  for (int e = 0; e < E; ++e) o[e] = 0.f;
  for (int s = 0; s < ns; ++s) {
    const float2 ml = *reinterpret_cast<const float2*>(a.pml +
                                                       (s * n + at) * 2);
    const float f = __builtin_amdgcn_exp2f(ml.x - m);
    l += ml.y * f;
    const float* p = a.po + (s * n + at) * D + lane * E;
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] += p[e] * f;
  }
  const float linv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e)
    a.out[at * D + lane * E + e] = f2bf(o[e] * linv);
}

template <int D>
void launch(const PrefillArgs& a, int nseg, hipStream_t stream) {
  const dim3 grid((uint32_t)(a.n_qt * a.B * a.Hq), nseg), block(NW * 64);
  if (nseg > 1) {
    hipLaunchKernelGGL((prefill_attn_kernel<D, 1>), grid, block, 0, stream, a);
    const int64_t n = (int64_t)a.B * a.Sq * a.Hq;
    hipLaunchKernelGGL((prefill_merge_kernel<D>),
                       dim3((uint32_t)((n + 3) / 4)), dim3(256), 0, stream,
                       a);
  } else {
    hipLaunchKernelGGL((prefill_attn_kernel<D, 0>), grid, block, 0, stream, a);
  }
}

}  // namespace

extern "C" {

// Slices of the keys. Only calls of up to 512 rows are cut: a prompt's
// portion of 512 rows has 4 query tiles per head, which leave most of the
// 256 CUs idle (512 rows over 3968 keys, 28 heads: 112 blocks against 448).
// The cut is by key position, so portions of any size give a row the same
// bits; longer calls fill the chip without it.
int tl_prefill_segments(int Sq, int Skv) {
  return Sq <= 512 ? cdiv(Skv, SEG) : 1;
}

// po, pml: fp32 scratch for the slices, [nseg, B, Sq, Hq, D] and
// [nseg, B, Sq, Hq, 2]; null: keys are not cut (always so with lse).
void tl_prefill_attn(const void* q, const void* k, const void* v,
                     const void* table, void* out, void* lse, void* po,
                     void* pml, int64_t kbs, int64_t khs, int kts, int B,
                     int Sq, int Skv, int q_off, int Hq, int Hkv, int D,
                     float scale, int causal, int bt_stride,
                     hipStream_t stream) {
  if (B <= 0 || Sq <= 0 || Hq <= 0) return;
  const PrefillArgs a{(const bf16*)q, (const bf16*)k, (const bf16*)v,
                      (const int*)table, (bf16*)out, (float*)lse, (float*)po,
                      (float*)pml, kbs, khs, kts, B, Sq, Skv, q_off, Hq, Hkv,
                      bt_stride, causal, cdiv(Sq, NW * 32), scale};
  const int nseg = po ? tl_prefill_segments(Sq, Skv) : 1;
  if (D == 128) launch<128>(a, nseg, stream);
  else if (D == 64) launch<64>(a, nseg, stream);
}

}  // extern "C"
