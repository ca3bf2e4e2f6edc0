// MFMA decode attention for gfx950.
//
// One block serves all G <= 16 query heads of one kv head over one slice of a
// sequence, so K and V are read once. What bounds it is how many bytes of K
// and V are in flight: every wave copies tiles of 32 keys to LDS buffers of
// its own with global_load_lds, one tile ahead, waits for its own copies only
// and meets the others once, at the end.
//
// The scores are formed transposed, S^T = K Q^T (16x16x32 MFMA, a lane holds 8
// keys of ONE head), so the row maximum is in-lane plus two exchanges, and the
// accumulators of two 16-key tiles ARE the B operand of O^T = V^T P^T once its
// 32 keys are counted as 4q..4q+3, 16+4q..16+4q+3 for quad q; V^T comes in
// that order from ds_read_b64_tr_b16. P does not pass through LDS.
//
// Flash-decode SPLIT: a long row is cut into slices (tl_split_for_len) in
// blocks that write (m, l, o) partials; a combine kernel merges them in order.
//
// Measured on MI355X, D 128 (before: 16-key tiles, K loaded where it is used,
// V through LDS stores, no copy in flight over a tile): 1 sequence of 513 keys,
// 4 kv heads, 16.5 -> 8.6 us; 8 of 1000, 8 kv heads, 32 -> 14; 48 of 1958 96
// -> 74 (5.2 TB/s); 256 of 577, 4 kv heads, 66 -> 62 (4.9 TB/s); 2 of 32400 84
// -> 63.

#include "common.hpp"

namespace {

constexpr int NWAVE = 4;
constexpr int KT = 32;            // keys per tile

using f32x4 = __attribute__((ext_vector_type(4))) float;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr float LOG2E = 1.4426950408889634f;

// 16-byte slot permutations within a row of D elements: K is read 16 rows at
// one slot, V four rows at 32 bytes (the quads' row groups alternate halves).
template <int D>
DEVINLINE int k_perm(int row) {
  return D == 128 ? (row & 15) : ((row >> 1) & 7);
}
template <int D>
DEVINLINE int v_perm(int row) {
  return D == 128 ? (((row & 3) << 1) | (((row >> 2) & 1) << 3))
                  : ((((row >> 1) & 1) << 1) | (((row >> 2) & 1) << 2));
}

// Transposed reads of 32 keys x 4 tiles of 16 columns; the wait is inside, as
// a read in flight must not have its registers reused.
struct VFrag {
  uint64_t lo[4], hi[4];
};
template <int OFF>
DEVINLINE VFrag read_v(const unsigned (&a)[4]) {
  VFrag f;
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\t"
      "ds_read_b64_tr_b16 %4, %8 offset:%12\n\t"
      "ds_read_b64_tr_b16 %1, %9\n\t"
      "ds_read_b64_tr_b16 %5, %9 offset:%12\n\t"
      "ds_read_b64_tr_b16 %2, %10\n\t"
      "ds_read_b64_tr_b16 %6, %10 offset:%12\n\t"
      "ds_read_b64_tr_b16 %3, %11\n\t"
      "ds_read_b64_tr_b16 %7, %11 offset:%12\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(f.lo[0]), "=&v"(f.lo[1]), "=&v"(f.lo[2]), "=&v"(f.lo[3]),
        "=&v"(f.hi[0]), "=&v"(f.hi[1]), "=&v"(f.hi[2]), "=&v"(f.hi[3])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "n"(OFF)
      : "memory");
  return f;
}

template <int N>
DEVINLINE void waitcnt_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// out layout when SPLIT_MODE: partial [B, Hq, n_split, D] float, ml [B, Hq,
// n_split, 2] float (m in log2 units, l); else bf16 out directly.
// PAGED: k_cache/v_cache are page pools [n_pages, Hkv, 128, D] and
// block_table [B, bt_stride] maps position/128 -> page id.
template <int D, int SPLIT_MODE, int PAGED>
__global__ __launch_bounds__(NWAVE * 64) void decode_attn_mfma_kernel(
    const bf16* __restrict__ q,        // [B, Hq, D]
    const bf16* __restrict__ k_cache,  // [B, Hkv, Smax, D] (or pool)
    const bf16* __restrict__ v_cache,
    const int* __restrict__ seq_lens,  // [B]
    const int* __restrict__ block_table,
    bf16* __restrict__ out,            // [B, Hq, D]
    float* __restrict__ partial,
    float* __restrict__ partial_ml,
    int Hq, int Hkv, int Smax, float scale, int n_split, int bt_stride,
    int per_row, int len_add) {
  constexpr int KCH = D / 32;        // MFMA k-chunks for QK^T
  constexpr int NV = D / 16;         // 16-column tiles of V
  constexpr int SL = D / 8, RPC = 64 / SL;   // slots per row, rows per copy
  constexpr int CP = KT / RPC;               // copies per operand and tile
  const int b = blockIdx.x, hkv = blockIdx.y, split = blockIdx.z;
  const int G = Hq / Hkv, h0 = hkv * G;
  const int L = seq_lens[b] + len_add;

  // per_row: this ROW's slices come from its own length (batch composition
  // must not change a row's accumulation — exact-greedy guarantee); the
  // launch z-width n_split is a host-side upper bound, surplus blocks exit.
  const int ns_row = per_row ? tl_split_for_len(L) : n_split;
  if (split >= ns_row) return;
  const int per_split = (L + ns_row * KT - 1) / (ns_row * KT) * KT;
  const int k_begin = split * per_split;
  const int k_end = min(L, k_begin + per_split);

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, quad = lane >> 4;

  __shared__ union alignas(16) {
    bf16 buf[NWAVE][2][2][KT][D];            // [wave][buffer][k|v]
    struct {
      float o[NWAVE][16][D + 4];
      float m[NWAVE][16], l[NWAVE][16];
    } red;
  } lds;

  // B operand: q of head col (zero past G), scale in exp2 units
  bf16x8_t qf[KCH];
  {
    const bf16* qrow =
        q + ((int64_t)b * Hq + h0 + (col < G ? col : 0)) * D + quad * 8;
#pragma unroll
    for (int c = 0; c < KCH; ++c) {
      qf[c] = *reinterpret_cast<const bf16x8_t*>(qrow + c * 32);
      if (col >= G)
#pragma unroll
        for (int j = 0; j < 8; ++j) qf[c][j] = (__bf16)0.f;
    }
  }
  float c2 = scale * LOG2E;
  if (c2 < 0.f) {                            // exact: flip the query's sign
    c2 = -c2;
#pragma unroll
    for (int c = 0; c < KCH; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) qf[c][j] = -qf[c][j];
  }
  c2 = fmaxf(c2, 1e-30f);

  // pages of this slice: lane i holds the i-th of 64 (8192 keys) at a time
  int pages = 0, page0 = k_begin >> 7;
  auto load_pages = [&]() {
    if (PAGED && k_begin < k_end)
      pages = block_table[b * bt_stride +
                          min(page0 + lane, (k_end - 1) >> 7)];
  };
  load_pages();

  const int crow = lane / SL, cslot = lane % SL;
  int koff[CP], voff[CP];
#pragma unroll
  for (int i = 0; i < CP; ++i) {
    const int r = i * RPC + crow;
    koff[i] = (cslot ^ k_perm<D>(r)) * 8;
    voff[i] = (cslot ^ v_perm<D>(r)) * 8;
  }
  auto copy = [&](int bufi, int t0) {
    int64_t base;
    if (PAGED) {
      if ((t0 >> 7) - page0 >= 64) {
        page0 += 64;
        load_pages();
      }
      const int page = __builtin_amdgcn_readlane(pages, (t0 >> 7) - page0);
      base = (((int64_t)page * Hkv + hkv) * 128 + (t0 & 127)) * D;
    } else {
      base = (((int64_t)b * Hkv + hkv) * Smax + t0) * D;
    }
    const bf16* kp = k_cache + base;
    const bf16* vp = v_cache + base;
    const int last = k_end - 1 - t0;         // keys past the end repeat it
#pragma unroll
    for (int i = 0; i < CP; ++i) {
      const int ro = min(i * RPC + crow, last) * D;
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(kp + ro + koff[i]),
          (__attribute__((address_space(3))) void*)(
              &lds.buf[wave][bufi][0][i * RPC][0]),
          16, 0, 0);
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(vp + ro + voff[i]),
          (__attribute__((address_space(3))) void*)(
              &lds.buf[wave][bufi][1][i * RPC][0]),
          16, 0, 0);
    }
  };

  // V^T reads: rows 4 quad + (lane >> 2) & 3 (and 16 on), columns 16 n
  unsigned vaddr[NV];
  {
    const int r = quad * 4 + ((lane >> 2) & 3);
    const unsigned base =
        (unsigned)(uintptr_t)(&lds.buf[wave][0][1][0][0]) + r * D * 2 +
        (lane & 1) * 8;
#pragma unroll
    for (int n = 0; n < NV; ++n)
      vaddr[n] = base + (((n * 2 + ((lane & 3) >> 1)) ^ v_perm<D>(r)) * 16);
  }

  float m_run = -1e30f, l_run = 0.f;         // log2 units; l of this lane
  f32x4 o[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) o[n] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // ---- each wave takes every NWAVE'th tile ----
  if (k_begin + wave * KT < k_end) copy(0, k_begin + wave * KT);
  int buf = 0;
  for (int t0 = k_begin + wave * KT; t0 < k_end; t0 += NWAVE * KT) {
    const int next = t0 + NWAVE * KT;
    if (next < k_end) {
      copy(buf ^ 1, next);
      waitcnt_vm<2 * CP>();
    } else {
      waitcnt_vm<0>();
    }
    f32x4 s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[h] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < KCH; ++c) {
        const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(
            &lds.buf[wave][buf][0][h * 16 + col]
                    [((c * 4 + quad) ^ k_perm<D>(col)) * 8]);
        s[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[c], s[h], 0, 0,
                                                       0);
      }
    }
    if (t0 + KT > k_end) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (t0 + h * 16 + quad * 4 + r >= k_end) s[h][r] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[h][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE_SIZE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE_SIZE)) * c2;
    // the reference maximum moves only when it is exceeded by 2^8 (a
    // decision of the head's own lanes): P and the sums stay far inside fp32
    const bool up = mx > m_run + 8.f;
    if (__any(up)) {
      const float alpha = up ? __builtin_amdgcn_exp2f(m_run - mx) : 1.f;
      m_run = up ? mx : m_run;
      l_run *= alpha;
#pragma unroll
      for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[n][r] *= alpha;
    }
    bf16x8_t p;
    float ps = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = __builtin_amdgcn_exp2f(fmaf(s[h][r], c2, -m_run));
        ps += e;
        p[h * 4 + r] = (__bf16)e;
      }
    l_run += ps;
#pragma unroll
    for (int g = 0; g < NV / 4; ++g) {
      unsigned a[4];
#pragma unroll
      for (int n = 0; n < 4; ++n) a[n] = vaddr[g * 4 + n] + buf * (2 * KT * D * 2);
      const VFrag f = read_v<16 * D * 2>(a);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const uint64_t w[2] = {f.lo[n], f.hi[n]};
        bf16x8_t vf;
        __builtin_memcpy(&vf, w, 16);
        o[g * 4 + n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            vf, p, o[g * 4 + n], 0, 0, 0);
      }
    }
    buf ^= 1;                // read_v has waited for all reads of this buffer
  }

  // ---- wave partials -> LDS: lane has columns 16 n + 4 quad + r of head col
  l_run += __shfl_xor(l_run, 16, WAVE_SIZE);
  l_run += __shfl_xor(l_run, 32, WAVE_SIZE);
  __syncthreads();                           // all buffers are free
#pragma unroll
  for (int n = 0; n < NV; ++n)
    *reinterpret_cast<f32x4*>(&lds.red.o[wave][col][n * 16 + quad * 4]) = o[n];
  if (quad == 0) {
    lds.red.m[wave][col] = m_run;
    lds.red.l[wave][col] = l_run;
  }
  __syncthreads();

  // ---- final merge across waves; write out ----
  for (int i = threadIdx.x; i < G * D; i += NWAVE * 64) {
    const int g = i / D, d = i - g * D;
    float m_tot = lds.red.m[0][g];
#pragma unroll
    for (int w = 1; w < NWAVE; ++w) m_tot = fmaxf(m_tot, lds.red.m[w][g]);
    float l_tot = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < NWAVE; ++w) {
      const float f = __builtin_amdgcn_exp2f(lds.red.m[w][g] - m_tot);
      l_tot += lds.red.l[w][g] * f;
      acc += lds.red.o[w][g][d] * f;
    }
    if (SPLIT_MODE) {
      const int64_t base = (((int64_t)b * Hq + h0 + g) * n_split + split);
      partial[base * D + d] = acc;
      if (d == 0) {
        partial_ml[base * 2] = m_tot;
        partial_ml[base * 2 + 1] = l_tot;
      }
    } else {
      out[((int64_t)b * Hq + h0 + g) * D + d] =
          f2bf(acc / fmaxf(l_tot, 1e-30f));
    }
  }
}

// combine kernel: merge this row's ns_row partials per (b, h). A row
// whose ns_row == 1 reduces to f = exp(0) = 1 scales — bitwise equal to
// the direct-write path.
template <int D>
__global__ __launch_bounds__(128) void decode_attn_combine_kernel(
    const float* __restrict__ partial, const float* __restrict__ partial_ml,
    const int* __restrict__ seq_lens, bf16* __restrict__ out, int Hq,
    int n_split, int per_row, int len_add) {
  const int bh = blockIdx.x;                    // b * Hq + h
  const int d = threadIdx.x;                    // [0, D)
  const int ns_row =
      per_row ? tl_split_for_len(seq_lens[bh / Hq] + len_add) : n_split;
  __shared__ float sm[64], sl[64];
  if (threadIdx.x < ns_row) {
    sm[threadIdx.x] = partial_ml[((int64_t)bh * n_split + threadIdx.x) * 2];
    sl[threadIdx.x] = partial_ml[((int64_t)bh * n_split + threadIdx.x) * 2 + 1];
  }
  __syncthreads();
  float m_tot = -1e30f;
  for (int s = 0; s < ns_row; ++s) m_tot = fmaxf(m_tot, sm[s]);
  float l_tot = 0.f, o = 0.f;
  for (int s = 0; s < ns_row; ++s) {
    const float f = __builtin_amdgcn_exp2f(sm[s] - m_tot);
    l_tot += sl[s] * f;
    o += partial[((int64_t)bh * n_split + s) * D + d] * f;
  }
  out[(int64_t)bh * D + d] = f2bf(o / fmaxf(l_tot, 1e-30f));
}

}  // namespace

extern "C" {

// scratch: partial floats [B*Hq*n_split*D] + ml [B*Hq*n_split*2]; pass
// nullptr when n_split == 1.
void tl_decode_attn_mfma(const void* q, const void* k_cache,
                         const void* v_cache, const void* seq_lens,
                         const void* block_table, void* out,
                         void* partial, void* partial_ml, int B, int Hq,
                         int Hkv, int Smax, int D, float scale, int n_split,
                         int bt_stride, int per_row, int len_add,
                         hipStream_t stream) {
  dim3 grid(B, Hkv, n_split), block(NWAVE * 64);
#define LAUNCH(DD, SM, PG)                                                   \
  hipLaunchKernelGGL((decode_attn_mfma_kernel<DD, SM, PG>), grid, block, 0,  \
                     stream, (const bf16*)q, (const bf16*)k_cache,           \
                     (const bf16*)v_cache, (const int*)seq_lens,             \
                     (const int*)block_table, (bf16*)out,                    \
                     (float*)partial, (float*)partial_ml, Hq, Hkv, Smax,     \
                     scale, n_split, bt_stride, per_row, len_add)
#define PICK(DD)                                                             \
  do {                                                                       \
    if (block_table) {                                                       \
      if (n_split == 1) LAUNCH(DD, 0, 1); else LAUNCH(DD, 1, 1);             \
    } else {                                                                 \
      if (n_split == 1) LAUNCH(DD, 0, 0); else LAUNCH(DD, 1, 0);             \
    }                                                                        \
  } while (0)
  if (D == 128) PICK(128);
  else if (D == 64) PICK(64);
#undef PICK
#undef LAUNCH
  if (n_split > 1) {
    dim3 cgrid(B * Hq), cblock(D);
    if (D == 128)
      hipLaunchKernelGGL((decode_attn_combine_kernel<128>), cgrid, cblock, 0,
                         stream, (const float*)partial,
                         (const float*)partial_ml, (const int*)seq_lens,
                         (bf16*)out, Hq, n_split, per_row, len_add);
    else
      hipLaunchKernelGGL((decode_attn_combine_kernel<64>), cgrid, cblock, 0,
                         stream, (const float*)partial,
                         (const float*)partial_ml, (const int*)seq_lens,
                         (bf16*)out, Hq, n_split, per_row, len_add);
  }
}

}  // extern "C"
