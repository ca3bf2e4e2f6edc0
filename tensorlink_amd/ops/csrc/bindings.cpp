// Python bindings for the tensorlink_amd CDNA4 kernel library.
// Host-side glue only — every kernel lives in the sibling .hip files and is
// reached through an extern "C" launcher taking raw pointers + hipStream_t.

#include <torch/extension.h>

#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

extern "C" {
void tl_rmsnorm_fwd(const void* x, const void* residual, const void* w,
                    void* y, void* r_out, void* rstd, int64_t N, int H,
                    float eps, hipStream_t stream);
void tl_rmsnorm_bwd(const void* dy, const void* x, const void* w,
                    const void* rstd, void* dx, void* dw, void* dw_partial,
                    int n_blocks, int64_t N, int H, hipStream_t stream);
void tl_rope(void* q, void* k, const void* positions, const void* inv_freq,
             int64_t T, int Hq, int Hkv, int D, float sign,
             hipStream_t stream);
void tl_swiglu_fwd(const void* gate, const void* up, void* out, int64_t n,
                   hipStream_t stream);
void tl_swiglu_bwd(const void* dout, const void* gate, const void* up,
                   void* dgate, void* dup, int64_t n, hipStream_t stream);
void tl_adamw(void* param, const void* grad, void* m, void* v, int64_t n,
              int is_bf16, float lr, float beta1, float beta2, float eps,
              float weight_decay, int step, hipStream_t stream);
void tl_decode_attn(const void* q, const void* k_cache, const void* v_cache,
                    const void* seq_lens, void* out, int B, int Hq, int Hkv,
                    int Smax, int D, float scale, hipStream_t stream);
int tl_prefill_segments(int Sq, int Skv);
void tl_prefill_attn(const void* q, const void* k, const void* v,
                     const void* table, void* out, void* lse, void* po,
                     void* pml, int64_t kbs, int64_t khs, int kts, int B,
                     int Sq, int Skv, int q_off, int Hq, int Hkv, int D,
                     float scale, int causal, int bt_stride,
                     hipStream_t stream);
void tl_swiglu_fused(const void* gu, void* out, int64_t N, int I,
                     hipStream_t stream);
void tl_swiglu_fused_bwd(const void* dout, const void* gu, void* dgu,
                         int64_t N, int I, hipStream_t stream);
void tl_rope_rows(void* qkv, void* q, void* k, void* v, const void* positions,
                  const void* inv_freq, int64_t T, int Hq, int Hkv, int D,
                  int bwd, hipStream_t stream);
void tl_skinny_glu(const void* x, const void* w, void* out, int M, int N,
                   int K, hipStream_t stream);
void tl_ce_fwd(const void* logits, const void* labels, void* lse, void* loss,
               void* mean, int64_t rows, int S, int V, int64_t ignore,
               hipStream_t stream);
void tl_ce_bwd(const void* logits, const void* labels, const void* lse,
               const void* mean, const void* dloss, void* dx, int64_t rows,
               int S, int V, int64_t ignore, hipStream_t stream);
void tl_reduce_partials(const void* partials, void* out, int P, int64_t H,
                        hipStream_t stream);
int tl_bias_grad_rows(int64_t M, int N);
void tl_bias_grad(const void* dy, const void* z, void* dz, void* partial,
                  int64_t M, int N, int per, hipStream_t stream);
void tl_layernorm_fwd(const void* x, const void* a, const void* w,
                      const void* b, void* r_out, void* y, void* mean,
                      void* rstd, int64_t M, int W, float eps,
                      hipStream_t stream);
void tl_layernorm_bwd(const void* dy, const void* dr, const void* r,
                      const void* w, const void* mean, const void* rstd,
                      void* dx, void* partial, int64_t M, int W, int blocks,
                      hipStream_t stream);
void tl_add_norm(const void* x, const void* partial, int n_split,
                 const void* residual, const void* w, void* r_out, void* y,
                 int64_t M, int H, int rounded, float eps,
                 hipStream_t stream);
void tl_rope_append_rows(const void* x, const void* partial, int n_split,
                         const void* bias, void* q_out, void* k_cache,
                         void* v_cache, const void* positions,
                         const void* inv_freq, int freq_bf16,
                         const void* table, int bt_stride, const void* qw,
                         const void* kw, float eps, int64_t T, int S, int Hq,
                         int Hkv, int D, int Smax, hipStream_t stream);
void tl_decode_attn_mfma(const void* q, const void* k_cache,
                         const void* v_cache, const void* seq_lens,
                         const void* block_table, void* out,
                         void* partial, void* partial_ml, int B, int Hq,
                         int Hkv, int Smax, int D, float scale, int n_split,
                         int bt_stride, int per_row, int len_add,
                         hipStream_t stream);
void tl_skinny_gemm(const void* x, const void* w, const void* bias,
                    void* out, void* partial, int M, int N, int K,
                    int n_split, int k_per, hipStream_t stream);
void tl_gemm_tiled(const void* x, const void* w, const void* bias, void* out,
                   void* partial, int M, int N, int K, int n_split,
                   int k_per, hipStream_t stream);
void tl_sample(const void* logits, const void* temps, const void* top_ps,
               const void* top_ks, const void* pres, const void* freqs,
               void* counts, const void* seeds, const void* ctr, void* out,
               uint64_t seed_base, int B, int V, hipStream_t stream);
void tl_bump_counter(void* ctr, hipStream_t stream);
int tl_prefill_segments(int Sq, int Skv);
void tl_prefill_attn(const void* q, const void* k, const void* v,
                     const void* table, void* out, void* lse, void* po,
                     void* pml, int64_t kbs, int64_t khs, int kts, int B,
                     int Sq, int Skv, int q_off, int Hq, int Hkv, int D,
                     float scale, int causal, int bt_stride,
                     hipStream_t stream);
void tl_swiglu_fused(const void* gu, void* out, int64_t N, int I,
                     hipStream_t stream);
void tl_decode_attn_mfma(const void* q, const void* k_cache,
                         const void* v_cache, const void* seq_lens,
                         const void* block_table, void* out,
                         void* partial, void* partial_ml, int B, int Hq,
                         int Hkv, int Smax, int D, float scale, int n_split,
                         int bt_stride, int per_row, int len_add,
                         hipStream_t stream);
void tl_skinny_gemm(const void* x, const void* w, const void* bias,
                    void* out, void* partial, int M, int N, int K,
                    int n_split, int k_per, hipStream_t stream);
void tl_gemm_tiled(const void* x, const void* w, const void* bias, void* out,
                   void* partial, int M, int N, int K, int n_split,
                   int k_per, hipStream_t stream);
void tl_sample(const void* logits, const void* temps, const void* top_ps,
               const void* top_ks, const void* pres, const void* freqs,
               void* counts, const void* seeds, const void* ctr, void* out,
               uint64_t seed_base, int B, int V, hipStream_t stream);
void tl_bump_counter(void* ctr, hipStream_t stream);
void tl_moe_gemm(const void* x, const void* tok_idx, const void* seg_off,
                 const void* w_ptrs, const void* s_ptrs, void* out, int E,
                 int N, int K, int fp8, hipStream_t stream);
int tl_attn_bwd_rows(int S);
int tl_attn_bwd_parts(int B, int S, int Hq, int Hkv);
void tl_attn_bwd(const void* q, const void* k, const void* v,
                 const void* dout, const void* out, const void* lse,
                 void* l2, void* delta, void* dq, void* dk, void* dv,
                 void* pk, void* pv, int B, int S, int Hq, int Hkv, int D,
                 float scale, int causal, int parts, hipStream_t stream);
}

namespace {

hipStream_t cur_stream() {
  return c10::hip::getCurrentHIPStream().stream();
}

// host copy of tl_split_for_len (common.hpp — keep in sync; this file is
// compiled by plain g++ so it cannot include the device header)
int tl_split_for_len(int L) {
  int ns = 1;
  while (ns < 16 && L > 1024 * ns) ns <<= 1;
  return ns;
}

#define CHECK_IN(t, d)                                              \
  TORCH_CHECK((t).is_cuda(), #t " must be on GPU");                 \
  TORCH_CHECK((t).is_contiguous(), #t " must be contiguous");       \
  TORCH_CHECK((t).scalar_type() == (d), #t " wrong dtype")

using torch::Tensor;

std::vector<Tensor> rmsnorm_fwd(Tensor x, c10::optional<Tensor> residual,
                                Tensor w, double eps, bool save_rstd) {
  CHECK_IN(x, torch::kBFloat16);
  CHECK_IN(w, torch::kBFloat16);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0, "H must be divisible by 8");
  const int64_t N = x.numel() / H;
  auto y = torch::empty_like(x);
  Tensor rstd, r_out;
  if (save_rstd) rstd = torch::empty({N}, x.options().dtype(torch::kFloat));
  const void* res_ptr = nullptr;
  void* rout_ptr = nullptr;
  if (residual.has_value()) {
    CHECK_IN(residual.value(), torch::kBFloat16);
    r_out = torch::empty_like(x);
    res_ptr = residual->data_ptr();
    rout_ptr = r_out.data_ptr();
  }
  tl_rmsnorm_fwd(x.data_ptr(), res_ptr, w.data_ptr(), y.data_ptr(), rout_ptr,
                 save_rstd ? rstd.data_ptr() : nullptr, N, H, (float)eps,
                 cur_stream());
  std::vector<Tensor> outs = {y};
  if (residual.has_value()) outs.push_back(r_out);
  if (save_rstd) outs.push_back(rstd);
  return outs;
}

std::vector<Tensor> rmsnorm_bwd(Tensor dy, Tensor x, Tensor w, Tensor rstd) {
  CHECK_IN(dy, torch::kBFloat16);
  CHECK_IN(x, torch::kBFloat16);
  CHECK_IN(w, torch::kBFloat16);
  CHECK_IN(rstd, torch::kFloat);
  const int H = x.size(-1);
  const int64_t N = x.numel() / H;
  const int n_blocks = (int)std::min<int64_t>(N, 512);
  auto dx = torch::empty_like(x);
  auto dw = torch::empty_like(w);
  auto partial = torch::empty({n_blocks, (int64_t)H},
                              x.options().dtype(torch::kFloat));
  tl_rmsnorm_bwd(dy.data_ptr(), x.data_ptr(), w.data_ptr(), rstd.data_ptr(),
                 dx.data_ptr(), dw.data_ptr(), partial.data_ptr(), n_blocks,
                 N, H, cur_stream());
  return {dx, dw};
}

void rope_(Tensor q, Tensor k, Tensor positions, Tensor inv_freq,
           double sign) {
  CHECK_IN(q, torch::kBFloat16);
  CHECK_IN(k, torch::kBFloat16);
  CHECK_IN(positions, torch::kInt);
  CHECK_IN(inv_freq, torch::kFloat);
  const int D = q.size(-1);
  const int Hq = q.size(-2);
  const int Hkv = k.size(-2);
  const int64_t T = q.numel() / ((int64_t)Hq * D);
  TORCH_CHECK(k.numel() / ((int64_t)Hkv * D) == T, "q/k token mismatch");
  TORCH_CHECK(positions.numel() == T, "positions size mismatch");
  tl_rope(q.data_ptr(), k.data_ptr(), positions.data_ptr(),
          inv_freq.data_ptr(), T, Hq, Hkv, D, (float)sign, cur_stream());
}

Tensor swiglu_fwd(Tensor gate, Tensor up) {
  CHECK_IN(gate, torch::kBFloat16);
  CHECK_IN(up, torch::kBFloat16);
  TORCH_CHECK(gate.numel() % 8 == 0, "numel must be divisible by 8");
  auto out = torch::empty_like(gate);
  tl_swiglu_fwd(gate.data_ptr(), up.data_ptr(), out.data_ptr(), gate.numel(),
                cur_stream());
  return out;
}

std::vector<Tensor> swiglu_bwd(Tensor dout, Tensor gate, Tensor up) {
  CHECK_IN(dout, torch::kBFloat16);
  auto dg = torch::empty_like(gate);
  auto du = torch::empty_like(up);
  tl_swiglu_bwd(dout.data_ptr(), gate.data_ptr(), up.data_ptr(), dg.data_ptr(),
                du.data_ptr(), gate.numel(), cur_stream());
  return {dg, du};
}

void adamw_(Tensor param, Tensor grad, Tensor m, Tensor v, double lr,
            double beta1, double beta2, double eps, double weight_decay,
            int64_t step) {
  TORCH_CHECK(param.is_cuda() && param.is_contiguous());
  TORCH_CHECK(m.scalar_type() == torch::kFloat &&
              v.scalar_type() == torch::kFloat);
  TORCH_CHECK(grad.scalar_type() == param.scalar_type());
  const bool is_bf16 = param.scalar_type() == torch::kBFloat16;
  TORCH_CHECK(is_bf16 || param.scalar_type() == torch::kFloat);
  tl_adamw(param.data_ptr(), grad.data_ptr(), m.data_ptr(), v.data_ptr(),
           param.numel(), is_bf16 ? 1 : 0, (float)lr, (float)beta1,
           (float)beta2, (float)eps, (float)weight_decay, (int)step,
           cur_stream());
}

Tensor decode_attn(Tensor q, Tensor k_cache, Tensor v_cache, Tensor seq_lens,
                   double scale, int64_t n_split,
                   c10::optional<Tensor> block_table, int64_t len_add) {
  CHECK_IN(q, torch::kBFloat16);
  CHECK_IN(k_cache, torch::kBFloat16);
  CHECK_IN(v_cache, torch::kBFloat16);
  CHECK_IN(seq_lens, torch::kInt);
  const int B = q.size(0), Hq = q.size(1), D = q.size(2);
  const int Hkv = k_cache.size(1), Smax = k_cache.size(2);
  const int G = Hq / Hkv;
  const void* bt = nullptr;
  int bt_stride = 0;
  if (block_table.has_value()) {
    CHECK_IN(block_table.value(), torch::kInt);
    TORCH_CHECK(G <= 16, "paged decode requires GQA group <= 16");
    TORCH_CHECK(k_cache.size(2) == 128, "paged pool PAGE must be 128");
    bt = block_table->data_ptr();
    bt_stride = block_table->size(1);
  }
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
  TORCH_CHECK(Hq % Hkv == 0, "GQA requires Hq % Hkv == 0");
  auto out = torch::empty_like(q);
  const bool legacy = (getenv("TL_DECODE_LEGACY") != nullptr || G > 16) &&
                      bt == nullptr;
  if (legacy) {
    if (len_add) seq_lens = seq_lens + len_add;
    tl_decode_attn(q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                   seq_lens.data_ptr(), out.data_ptr(), B, Hq, Hkv, Smax, D,
                   (float)scale, cur_stream());
    return out;
  }
  int per_row = 0;
  if (n_split <= 0) {
    // auto: per-ROW split from each row's own length (tl_split_for_len,
    // common.hpp) so a sequence's numerics are batch-independent; the
    // launch z-width comes from a batch-shape-free host bound on L
    // (cache capacity), no device sync needed.
    per_row = 1;
    const int upper = bt ? bt_stride * 128 : Smax;
    n_split = tl_split_for_len(upper);
  }
  TORCH_CHECK(n_split <= 64, "n_split too large");
  Tensor partial, partial_ml;
  void *pp = nullptr, *pml = nullptr;
  if (n_split > 1) {
    partial = torch::empty({(int64_t)B * Hq * n_split * D},
                           q.options().dtype(torch::kFloat));
    partial_ml = torch::empty({(int64_t)B * Hq * n_split * 2},
                              q.options().dtype(torch::kFloat));
    pp = partial.data_ptr();
    pml = partial_ml.data_ptr();
  }
  tl_decode_attn_mfma(q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                      seq_lens.data_ptr(), bt, out.data_ptr(), pp, pml, B,
                      Hq, Hkv, Smax, D, (float)scale, (int)n_split,
                      bt_stride, per_row, (int)len_add, cur_stream());
  return out;
}

// k, v: a tensor of rows of D at the given (batch, head, token) strides, or
// page pools with a table. Split keys go through fp32 partials.
Tensor prefill_run(const Tensor& q, const Tensor& k, const Tensor& v,
                   const int* table, int bt_stride, int64_t kbs, int64_t khs,
                   int64_t kts, int64_t Skv, int64_t Hkv, double scale,
                   bool causal, int64_t q_off, float* lse) {
  const int64_t B = q.size(0), Sq = q.size(1), Hq = q.size(2), D = q.size(3);
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
  TORCH_CHECK(Hkv > 0 && Hq % Hkv == 0, "GQA requires Hq % Hkv == 0");
  TORCH_CHECK(kts <= INT_MAX / 64, "token stride too large");
  auto out = torch::empty_like(q);
  if (Skv == 0) {                            // no keys: zeros
    out.zero_();
    return out;
  }
  const int nseg = lse ? 1 : tl_prefill_segments((int)Sq, (int)Skv);
  Tensor po, pml;
  if (nseg > 1) {
    const auto f32 = q.options().dtype(torch::kFloat);
    po = torch::empty({nseg * B * Sq * Hq * D}, f32);
    pml = torch::empty({nseg * B * Sq * Hq * 2}, f32);
  }
  tl_prefill_attn(q.data_ptr(), k.data_ptr(), v.data_ptr(), table,
                  out.data_ptr(), lse, nseg > 1 ? po.data_ptr() : nullptr,
                  nseg > 1 ? pml.data_ptr() : nullptr, kbs, khs, (int)kts,
                  (int)B, (int)Sq, (int)Skv, (int)q_off, (int)Hq, (int)Hkv,
                  (int)D, (float)scale, causal ? 1 : 0, bt_stride, cur_stream());
  return out;
}

Tensor prefill_attn(Tensor q, Tensor k, Tensor v, double scale, bool causal,
                    int64_t q_off) {
  CHECK_IN(q, torch::kBFloat16);
  CHECK_IN(k, torch::kBFloat16);
  CHECK_IN(v, torch::kBFloat16);
  const int64_t Skv = k.size(1), Hkv = k.size(2), D = q.size(3);
  TORCH_CHECK(q_off + q.size(1) <= Skv || !causal, "q_off + Sq must fit Skv");
  return prefill_run(q, k, v, nullptr, 0, Skv * Hkv * D, D, Hkv * D, Skv, Hkv,
                     scale, causal, q_off, nullptr);
}

std::vector<Tensor> prefill_attn_lse(Tensor q, Tensor k, Tensor v,
                                     double scale, bool causal) {
  CHECK_IN(q, torch::kBFloat16);
  CHECK_IN(k, torch::kBFloat16);
  CHECK_IN(v, torch::kBFloat16);
  const int64_t Skv = k.size(1), Hkv = k.size(2), D = q.size(3);
  auto lse = torch::empty({q.size(0), q.size(2), q.size(1)},
                          q.options().dtype(torch::kFloat));
  auto out = prefill_run(q, k, v, nullptr, 0, Skv * Hkv * D, D, Hkv * D, Skv,
                         Hkv, scale, causal, 0, (float*)lse.data_ptr());
  return {out, lse};
}

// Causal attention of q's rows (positions kv_len - Sq ..) over the first
// kv_len positions of a cache, read in place: [B,Hkv,Smax,D] or page pools.
Tensor prefill_attn_cache(Tensor q, Tensor k_cache, Tensor v_cache,
                          c10::optional<Tensor> table, int64_t kv_len,
                          double scale) {
  CHECK_IN(q, torch::kBFloat16);
  CHECK_IN(k_cache, torch::kBFloat16);
  CHECK_IN(v_cache, torch::kBFloat16);
  const int64_t Sq = q.size(1), D = q.size(3);
  const int64_t Hkv = k_cache.size(1), Smax = k_cache.size(2);
  TORCH_CHECK(k_cache.size(3) == D && v_cache.sizes() == k_cache.sizes(),
              "cache shape mismatch");
  TORCH_CHECK(Sq > 0 && Sq <= kv_len, "kv_len must cover the query rows");
  const int* bt = nullptr;
  int bt_stride = 0;
  if (table.has_value()) {
    CHECK_IN(table.value(), torch::kInt);
    TORCH_CHECK(Smax == 128, "paged pool PAGE must be 128");
    TORCH_CHECK(table->size(0) == q.size(0) && table->size(1) * 128 >= kv_len,
                "table too small");
    bt = table->data_ptr<int>();
    bt_stride = (int)table->size(1);
  } else {
    TORCH_CHECK(k_cache.size(0) == q.size(0) && kv_len <= Smax,
                "cache too small");
  }
  return prefill_run(q, k_cache, v_cache, bt, bt_stride, Hkv * Smax * D,
                     Smax * D, D, kv_len, Hkv, scale, true, kv_len - Sq,
                     nullptr);
}

std::vector<Tensor> attn_bwd(Tensor q, Tensor k, Tensor v, Tensor dout,
                             Tensor out, Tensor lse, double scale,
                             bool causal) {
  CHECK_IN(q, torch::kBFloat16);
  CHECK_IN(k, torch::kBFloat16);
  CHECK_IN(v, torch::kBFloat16);
  CHECK_IN(dout, torch::kBFloat16);
  CHECK_IN(out, torch::kBFloat16);
  CHECK_IN(lse, torch::kFloat);
  const int B = q.size(0), S = q.size(1), Hq = q.size(2), D = q.size(3);
  const int Hkv = k.size(2);
  TORCH_CHECK(k.size(1) == S, "training attention needs Sq == Skv");
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64 or 128");
  TORCH_CHECK(Hkv > 0 && Hq % Hkv == 0, "GQA requires Hq % Hkv == 0");
  TORCH_CHECK(v.sizes() == k.sizes() && k.size(0) == B && k.size(3) == D &&
                  dout.sizes() == q.sizes() && out.sizes() == q.sizes() &&
                  lse.numel() == (int64_t)B * Hq * S,
              "attention backward: shape mismatch");
  auto dq = torch::empty_like(q);
  auto dk = torch::empty_like(k);
  auto dv = torch::empty_like(v);
  const auto f32 = q.options().dtype(torch::kFloat);
  auto rows = torch::empty({2, (int64_t)B * Hq * tl_attn_bwd_rows(S)}, f32);
  const int parts = tl_attn_bwd_parts(B, S, Hq, Hkv);
  Tensor sums;
  if (parts > 1) sums = torch::empty({2, parts * k.numel()}, f32);
  tl_attn_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(),
              out.data_ptr(), lse.data_ptr(), rows[0].data_ptr(),
              rows[1].data_ptr(), dq.data_ptr(), dk.data_ptr(),
              dv.data_ptr(), parts > 1 ? sums[0].data_ptr() : nullptr,
              parts > 1 ? sums[1].data_ptr() : nullptr, B, S, Hq, Hkv, D,
              (float)scale, causal ? 1 : 0, parts, cur_stream());
  return {dq, dk, dv};
}

Tensor swiglu_fused(Tensor gu) {
  CHECK_IN(gu, torch::kBFloat16);
  const int64_t I2 = gu.size(-1);
  TORCH_CHECK(I2 % 16 == 0, "fused width must be divisible by 16");
  const int64_t I = I2 / 2;
  const int64_t N = gu.numel() / I2;
  auto sizes = gu.sizes().vec();
  sizes.back() = I;
  auto out = torch::empty(sizes, gu.options());
  tl_swiglu_fused(gu.data_ptr(), out.data_ptr(), N, (int)I, cur_stream());
  return out;
}

Tensor swiglu_fused_bwd(Tensor dout, Tensor gu) {
  CHECK_IN(dout, torch::kBFloat16);
  CHECK_IN(gu, torch::kBFloat16);
  const int64_t I2 = gu.size(-1);
  TORCH_CHECK(I2 % 16 == 0 && dout.numel() * 2 == gu.numel() &&
                  dout.size(-1) * 2 == I2,
              "dout must be half as wide as gate_up, a multiple of 8");
  auto dgu = torch::empty_like(gu);
  tl_swiglu_fused_bwd(dout.data_ptr(), gu.data_ptr(), dgu.data_ptr(),
                      gu.numel() / std::max<int64_t>(I2, 1), (int)(I2 / 2),
                      cur_stream());
  return dgu;
}

// fused projection rows [T, (Hq + 2 Hkv) D] -> rotated q, k, and v
std::vector<Tensor> rope_split(Tensor qkv, Tensor positions, Tensor inv_freq,
                               int64_t Hq, int64_t Hkv) {
  CHECK_IN(qkv, torch::kBFloat16);
  CHECK_IN(positions, torch::kInt);
  CHECK_IN(inv_freq, torch::kFloat);
  const int64_t T = qkv.size(0), D = inv_freq.numel() * 2;
  TORCH_CHECK(qkv.dim() == 2 && qkv.size(1) == (Hq + 2 * Hkv) * D &&
                  D % 16 == 0 && positions.numel() == T,
              "qkv width mismatch");
  auto q = torch::empty({T, Hq, D}, qkv.options());
  auto k = torch::empty({T, Hkv, D}, qkv.options());
  auto v = torch::empty_like(k);
  tl_rope_rows(qkv.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
               positions.data_ptr(), inv_freq.data_ptr(), T, (int)Hq,
               (int)Hkv, (int)D, 0, cur_stream());
  return {q, k, v};
}

// its backward
Tensor rope_merge(Tensor dq, Tensor dk, Tensor dv, Tensor positions,
                  Tensor inv_freq) {
  CHECK_IN(dq, torch::kBFloat16);
  CHECK_IN(dk, torch::kBFloat16);
  CHECK_IN(dv, torch::kBFloat16);
  CHECK_IN(positions, torch::kInt);
  CHECK_IN(inv_freq, torch::kFloat);
  const int64_t T = dq.size(0), Hq = dq.size(1), Hkv = dk.size(1);
  const int64_t D = inv_freq.numel() * 2;
  TORCH_CHECK(dq.dim() == 3 && dq.size(2) == D && D % 16 == 0 &&
                  dk.size(0) == T && dk.size(2) == D &&
                  dv.sizes() == dk.sizes() && positions.numel() == T,
              "gradient shapes mismatch");
  auto out = torch::empty({T, (Hq + 2 * Hkv) * D}, dq.options());
  tl_rope_rows(out.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
               positions.data_ptr(), inv_freq.data_ptr(), T, (int)Hq,
               (int)Hkv, (int)D, 1, cur_stream());
  return out;
}

static void check_ce(const Tensor& logits, const Tensor& labels) {
  CHECK_IN(logits, torch::kBFloat16);
  CHECK_IN(labels, torch::kLong);
  TORCH_CHECK(logits.dim() == 3 && labels.dim() == 2 &&
                  labels.size(0) == logits.size(0) &&
                  labels.size(1) == logits.size(1) && logits.numel() > 0 &&
                  logits.size(2) < (1 << 30) && labels.size(1) < (1 << 30) &&
                  labels.numel() < (1ll << 31),
              "logits [B, S, V] and labels [B, S] mismatch");
}

// (mean loss over the labelled rows, log-sum-exp [B, S], [mean, count])
std::vector<Tensor> ce_fwd(Tensor logits, Tensor labels, int64_t ignore) {
  check_ce(logits, labels);
  auto f32 = logits.options().dtype(torch::kFloat);
  auto lse = torch::empty(labels.sizes(), f32);
  auto loss = torch::empty(labels.sizes(), f32);
  auto mean = torch::empty({2}, f32);
  tl_ce_fwd(logits.data_ptr(), labels.data_ptr(), lse.data_ptr(),
            loss.data_ptr(), mean.data_ptr(), labels.numel(),
            (int)labels.size(1), (int)logits.size(2), ignore, cur_stream());
  return {mean.select(0, 0), lse, mean};
}

Tensor ce_bwd(Tensor logits, Tensor labels, Tensor lse, Tensor mean,
              Tensor dloss, int64_t ignore) {
  check_ce(logits, labels);
  CHECK_IN(lse, torch::kFloat);
  CHECK_IN(mean, torch::kFloat);
  CHECK_IN(dloss, torch::kFloat);
  TORCH_CHECK(lse.numel() == labels.numel() && mean.numel() == 2 &&
                  dloss.numel() == 1,
              "saved shapes mismatch");
  // rows of any length: the gradient starts at the logits' offset from 16
  const int64_t off = (int64_t)(((uintptr_t)logits.data_ptr() & 15) / 2);
  auto buf = torch::empty({off + logits.numel()}, logits.options());
  auto dx = buf.narrow(0, off, logits.numel()).view(logits.sizes());
  tl_ce_bwd(logits.data_ptr(), labels.data_ptr(), lse.data_ptr(),
            mean.data_ptr(), dloss.data_ptr(), dx.data_ptr(), labels.numel(),
            (int)labels.size(1), (int)logits.size(2), ignore, cur_stream());
  return dx;
}

// projection rows [T, (Hq + 2 Hkv) D] to q, k and v, and back
std::vector<Tensor> rows_split(Tensor qkv, int64_t Hq, int64_t Hkv,
                               int64_t D) {
  CHECK_IN(qkv, torch::kBFloat16);
  TORCH_CHECK(qkv.dim() == 2 && qkv.size(1) == (Hq + 2 * Hkv) * D &&
                  D % 16 == 0,
              "qkv width mismatch");
  const int64_t T = qkv.size(0);
  auto q = torch::empty({T, Hq, D}, qkv.options());
  auto k = torch::empty({T, Hkv, D}, qkv.options());
  auto v = torch::empty_like(k);
  tl_rope_rows(qkv.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
               nullptr, nullptr, T, (int)Hq, (int)Hkv, (int)D, 0,
               cur_stream());
  return {q, k, v};
}

Tensor rows_merge(Tensor dq, Tensor dk, Tensor dv) {
  CHECK_IN(dq, torch::kBFloat16);
  CHECK_IN(dk, torch::kBFloat16);
  CHECK_IN(dv, torch::kBFloat16);
  TORCH_CHECK(dq.dim() == 3 && dk.dim() == 3 && dk.size(0) == dq.size(0) &&
                  dk.size(2) == dq.size(2) && dv.sizes() == dk.sizes() &&
                  dq.size(2) % 16 == 0,
              "gradient shapes mismatch");
  const int64_t T = dq.size(0), Hq = dq.size(1), Hkv = dk.size(1);
  const int64_t D = dq.size(2);
  auto out = torch::empty({T, (Hq + 2 * Hkv) * D}, dq.options());
  tl_rope_rows(out.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(),
               nullptr, nullptr, T, (int)Hq, (int)Hkv, (int)D, 1,
               cur_stream());
  return out;
}

// {column sums of dy}, or with z {dz = dy gelu'(z), column sums of dz}
std::vector<Tensor> bias_grad(Tensor dy, c10::optional<Tensor> z) {
  CHECK_IN(dy, torch::kBFloat16);
  const int64_t N = dy.size(-1), M = N ? dy.numel() / N : 0;
  TORCH_CHECK(M > 0 && N % 8 == 0, "rows must be a multiple of 8 wide");
  const int per = tl_bias_grad_rows(M, (int)N);
  const int P = (int)((M + per - 1) / per);
  auto partial = torch::empty({P, N}, dy.options().dtype(torch::kFloat));
  auto db = torch::empty({N}, dy.options());
  Tensor dz;
  if (z.has_value()) {
    CHECK_IN(z.value(), torch::kBFloat16);
    TORCH_CHECK(z->sizes() == dy.sizes(), "shapes differ");
    dz = torch::empty_like(dy);
  }
  tl_bias_grad(dy.data_ptr(), z.has_value() ? z->data_ptr() : nullptr,
               z.has_value() ? dz.data_ptr() : nullptr, partial.data_ptr(),
               M, (int)N, per, cur_stream());
  tl_reduce_partials(partial.data_ptr(), db.data_ptr(), P, N, cur_stream());
  if (z.has_value()) return {dz, db};
  return {db};
}

static int64_t check_ln(const Tensor& x, const Tensor& w) {
  CHECK_IN(x, torch::kBFloat16);
  CHECK_IN(w, torch::kBFloat16);
  const int64_t W = x.size(-1);
  TORCH_CHECK(W % 8 == 0 && W <= 2048 && w.numel() == W && x.numel() > 0,
              "rows must be a multiple of 8 wide, at most 2048");
  return W;
}

// (y, mean, rstd) or with a (y, mean, rstd, r = x + a)
std::vector<Tensor> layernorm_fwd(Tensor x, c10::optional<Tensor> a, Tensor w,
                                  Tensor b, double eps) {
  const int64_t W = check_ln(x, w), M = x.numel() / W;
  CHECK_IN(b, torch::kBFloat16);
  TORCH_CHECK(b.numel() == W, "norm bias size mismatch");
  auto f32 = x.options().dtype(torch::kFloat);
  auto y = torch::empty_like(x);
  auto mean = torch::empty({M}, f32), rstd = torch::empty({M}, f32);
  Tensor r;
  if (a.has_value()) {
    CHECK_IN(a.value(), torch::kBFloat16);
    TORCH_CHECK(a->sizes() == x.sizes(), "shapes differ");
    r = torch::empty_like(x);
  }
  tl_layernorm_fwd(x.data_ptr(), a.has_value() ? a->data_ptr() : nullptr,
                   w.data_ptr(), b.data_ptr(),
                   a.has_value() ? r.data_ptr() : nullptr, y.data_ptr(),
                   mean.data_ptr(), rstd.data_ptr(), M, (int)W, (float)eps,
                   cur_stream());
  if (a.has_value()) return {y, mean, rstd, r};
  return {y, mean, rstd};
}

// (gradient of r, dw, db); dr: what comes along r itself
std::vector<Tensor> layernorm_bwd(Tensor dy, c10::optional<Tensor> dr,
                                  Tensor r, Tensor w, Tensor mean,
                                  Tensor rstd) {
  const int64_t W = check_ln(r, w), M = r.numel() / W;
  CHECK_IN(dy, torch::kBFloat16);
  CHECK_IN(mean, torch::kFloat);
  CHECK_IN(rstd, torch::kFloat);
  TORCH_CHECK(dy.sizes() == r.sizes() && mean.numel() == M &&
                  rstd.numel() == M,
              "saved shapes mismatch");
  if (dr.has_value()) {
    CHECK_IN(dr.value(), torch::kBFloat16);
    TORCH_CHECK(dr->sizes() == r.sizes(), "shapes differ");
  }
  const int blocks = (int)std::min<int64_t>(256, (M + 3) / 4);
  auto dx = torch::empty_like(r);
  auto partial = torch::empty({blocks, 2 * W},
                              r.options().dtype(torch::kFloat));
  auto dwb = torch::empty({2, W}, r.options());
  tl_layernorm_bwd(dy.data_ptr(), dr.has_value() ? dr->data_ptr() : nullptr,
                   r.data_ptr(), w.data_ptr(), mean.data_ptr(),
                   rstd.data_ptr(), dx.data_ptr(), partial.data_ptr(), M,
                   (int)W, blocks, cur_stream());
  tl_reduce_partials(partial.data_ptr(), dwb.data_ptr(), blocks, 2 * W,
                     cur_stream());
  return {dx, dwb.select(0, 0), dwb.select(0, 1)};
}

// Split-K policy SHARED by the streaming (M<=64) and tiled (M>64) GEMM
// kernels. It depends only on (N, K) — never M — so a row's accumulation
// (split boundaries + s-ordered reduce) is bitwise identical at every M:
// the serving engine's exact-greedy guarantee rests on this.
// split-block target (~blocks before M/z tiling); env-tunable for
// in-pipeline A/B — read ONCE so the policy stays (N,K)-pure in-process
static int gemm_split_target() {
  static int t = [] {
    const char* e = getenv("TL_GEMM_SPLIT_TARGET");
    return e ? atoi(e) : 256;
  }();
  return t;
}

struct GemmSplit {
  int n, k_per;
};

// 1, 2 or 4 cuts of whole 256s of K, at most one block per CU: a block keeps
// three steps in flight, which streams W at full rate, and every further cut
// costs its fp32 partials a round trip (3584 x 18944, 1 / 256 / 512 rows: 4
// cuts 28 / 65 / 101 us, 8 cuts 30 / 65 / 117).
static GemmSplit gemm_split(int N, int K) {
  const int steps = (K + 255) / 256, panels = N / 64;
  const int most = gemm_split_target() / panels;
  const int n = std::min(most >= 4 ? 4 : most >= 2 ? 2 : 1, steps);
  if (n <= 1) return {1, K};
  const int per = (steps + n - 1) / n;
  return {(steps + per - 1) / per, per * 256};
}

// x W^T of the family: bf16 rows in `out`, or its cuts in `partial` where the
// caller sums them (cuts set) and there are any.
struct Product {
  Tensor out, partial;
  int n_split = 1;
  const void* rows() const { return out.defined() ? out.data_ptr() : nullptr; }
  const void* cuts() const {
    return partial.defined() ? partial.data_ptr() : nullptr;
  }
};

Product run_gemm(const Tensor& x, const Tensor& w,
                 const c10::optional<Tensor>& bias, bool cuts) {
  CHECK_IN(x, torch::kBFloat16);
  CHECK_IN(w, torch::kBFloat16);
  const int K = x.size(-1);
  const int64_t M = x.numel() / K;
  const int N = w.size(0);
  TORCH_CHECK(w.size(1) == K, "K mismatch");
  TORCH_CHECK(K % 32 == 0 && N % 64 == 0, "unsupported shape");
  const void* bp = nullptr;
  if (bias.has_value()) {
    CHECK_IN(bias.value(), torch::kBFloat16);
    bp = bias->data_ptr();
  }
  const auto [n_split, k_per] = gemm_split(N, K);
  Product p;
  p.n_split = n_split;
  if (n_split > 1)
    p.partial = torch::empty({(int64_t)n_split * M * N},
                             x.options().dtype(torch::kFloat));
  if (!cuts || n_split == 1) {
    auto sizes = x.sizes().vec();
    sizes.back() = N;
    p.out = torch::empty(sizes, x.options());
  }
  void* op = p.out.defined() ? p.out.data_ptr() : nullptr;
  void* pp = n_split > 1 ? p.partial.data_ptr() : nullptr;
  if (M <= 64)
    tl_skinny_gemm(x.data_ptr(), w.data_ptr(), bp, op, pp, (int)M, N, K,
                   n_split, k_per, cur_stream());
  else
    tl_gemm_tiled(x.data_ptr(), w.data_ptr(), bp, op, pp, (int)M, N, K,
                  n_split, k_per, cur_stream());
  return p;
}

Tensor skinny_gemm(Tensor x, Tensor w, c10::optional<Tensor> bias) {
  return run_gemm(x, w, bias, false).out;
}

// silu(x gate^T) (x up^T) with w = [gate; up], at most 64 rows
Tensor skinny_glu(Tensor x, Tensor w) {
  CHECK_IN(x, torch::kBFloat16);
  CHECK_IN(w, torch::kBFloat16);
  const int64_t K = x.size(-1), M = x.numel() / K, N = w.size(0);
  TORCH_CHECK(w.dim() == 2 && w.size(1) == K, "K mismatch");
  TORCH_CHECK(M <= 64 && K % 32 == 0 && N % 64 == 0, "unsupported shape");
  auto sizes = x.sizes().vec();
  sizes.back() = N / 2;
  auto out = torch::empty(sizes, x.options());
  if (M > 0)
    tl_skinny_glu(x.data_ptr(), w.data_ptr(), out.data_ptr(), (int)M, (int)N,
                  (int)K, cur_stream());
  return out;
}

// r = x (+ residual), y = RMSNorm(r) w; y undefined without w
std::vector<Tensor> add_norm_run(const Product& p, const Tensor& residual,
                                 const c10::optional<Tensor>& w, double eps,
                                 bool rounded) {
  CHECK_IN(residual, torch::kBFloat16);
  const int64_t H = residual.size(-1), M = residual.numel() / H;
  TORCH_CHECK(H % 8 == 0 && H <= 16384, "width must be a multiple of 8");
  auto r = torch::empty_like(residual);
  Tensor y;
  if (w.has_value()) {
    CHECK_IN(w.value(), torch::kBFloat16);
    TORCH_CHECK(w->numel() == H, "norm weight size mismatch");
    y = torch::empty_like(residual);
  }
  tl_add_norm(p.rows(), p.cuts(), p.n_split, residual.data_ptr(),
              w.has_value() ? w->data_ptr() : nullptr, r.data_ptr(),
              w.has_value() ? y.data_ptr() : nullptr, M, (int)H,
              rounded ? 1 : 0, (float)eps, cur_stream());
  if (w.has_value()) return {y, r};
  return {r};
}

std::vector<Tensor> add_norm(Tensor x, Tensor residual,
                             c10::optional<Tensor> w, double eps,
                             bool rounded) {
  CHECK_IN(x, torch::kBFloat16);
  TORCH_CHECK(x.sizes() == residual.sizes(), "shapes differ");
  Product p;
  p.out = x;
  return add_norm_run(p, residual, w, eps, rounded);
}

std::vector<Tensor> linear_add_norm(Tensor x, Tensor weight, Tensor residual,
                                    c10::optional<Tensor> w, double eps,
                                    bool rounded) {
  TORCH_CHECK(residual.size(-1) == weight.size(0) &&
                  residual.numel() / residual.size(-1) ==
                      x.numel() / x.size(-1),
              "residual shape mismatch");
  Product p = run_gemm(x, weight, c10::nullopt, true);
  if (p.out.defined()) p.partial = Tensor();
  return add_norm_run(p, residual, w, eps, rounded);
}

Tensor rope_append_run(const Product& p, const Tensor& like,
                       const c10::optional<Tensor>& bias, Tensor& k_cache,
                       Tensor& v_cache, const Tensor& positions,
                       const Tensor& inv_freq, int64_t S, int64_t Hq,
                       int64_t Hkv, const c10::optional<Tensor>& table,
                       const c10::optional<Tensor>& qw,
                       const c10::optional<Tensor>& kw, double eps,
                       int64_t T) {
  CHECK_IN(k_cache, torch::kBFloat16);
  CHECK_IN(v_cache, torch::kBFloat16);
  CHECK_IN(positions, torch::kInt);
  TORCH_CHECK(inv_freq.is_cuda() && inv_freq.is_contiguous() &&
                  (inv_freq.scalar_type() == torch::kFloat ||
                   inv_freq.scalar_type() == torch::kBFloat16),
              "inv_freq must be fp32 or bf16 on GPU");
  const int64_t D = k_cache.size(3), Smax = k_cache.size(2);
  TORCH_CHECK(v_cache.sizes() == k_cache.sizes() && k_cache.size(1) == Hkv,
              "cache shapes mismatch");
  TORCH_CHECK(D % 16 == 0, "D must be divisible by 16");
  TORCH_CHECK(inv_freq.numel() * 2 == D && positions.numel() == T,
              "positions or inv_freq size mismatch");
  TORCH_CHECK(T % S == 0, "T must be divisible by S");
  const int* bt = nullptr;
  int bt_stride = 0;
  if (table.has_value()) {
    CHECK_IN(table.value(), torch::kInt);
    TORCH_CHECK(Smax == 128, "paged pool PAGE must be 128");
    TORCH_CHECK(table->size(0) * S == T, "table batch mismatch");
    bt = table->data_ptr<int>();
    bt_stride = (int)table->size(1);
  } else {
    TORCH_CHECK(k_cache.size(0) * S == T, "cache batch mismatch");
  }
  const void *qp = nullptr, *kp = nullptr;
  if (qw.has_value()) {
    CHECK_IN(qw.value(), torch::kBFloat16);
    TORCH_CHECK(kw.has_value(), "q and k norms go together");
    CHECK_IN(kw.value(), torch::kBFloat16);
    TORCH_CHECK(qw->numel() == D && kw->numel() == D &&
                    D <= 1024 && ((D / 16) & (D / 16 - 1)) == 0,
                "norms need D / 16 to be a power of two up to 64");
    qp = qw->data_ptr();
    kp = kw->data_ptr();
  }
  auto q = torch::empty({T, Hq, D}, like.options());
  tl_rope_append_rows(p.rows(), p.cuts(), p.n_split,
                      bias.has_value() ? bias->data_ptr() : nullptr,
                      q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                      positions.data_ptr(), inv_freq.data_ptr(),
                      inv_freq.scalar_type() == torch::kBFloat16 ? 1 : 0, bt,
                      bt_stride, qp, kp, (float)eps, T, (int)S, (int)Hq,
                      (int)Hkv, (int)D, (int)Smax, cur_stream());
  return q;
}

// qkv: [T, (Hq + 2 Hkv) D] fused projection output (q | k | v per row).
// Returns (normed and) rotated q [T, Hq, D]; k and v land in the caches.
Tensor rope_append_(Tensor qkv, Tensor k_cache, Tensor v_cache,
                    Tensor positions, Tensor inv_freq, int64_t S, int64_t Hq,
                    int64_t Hkv, c10::optional<Tensor> block_table,
                    c10::optional<Tensor> qw, c10::optional<Tensor> kw,
                    double eps) {
  CHECK_IN(qkv, torch::kBFloat16);
  TORCH_CHECK(qkv.size(-1) == (Hq + 2 * Hkv) * k_cache.size(3),
              "qkv width mismatch");
  Product p;
  p.out = qkv;
  return rope_append_run(p, qkv, c10::nullopt, k_cache, v_cache, positions,
                         inv_freq, S, Hq, Hkv, block_table, qw, kw, eps,
                         qkv.numel() / qkv.size(-1));
}

// The fused projection itself in front of it.
Tensor linear_rope_append_(Tensor x, Tensor weight,
                           c10::optional<Tensor> bias, Tensor k_cache,
                           Tensor v_cache, Tensor positions, Tensor inv_freq,
                           int64_t S, int64_t Hq, int64_t Hkv,
                           c10::optional<Tensor> block_table,
                           c10::optional<Tensor> qw,
                           c10::optional<Tensor> kw, double eps) {
  TORCH_CHECK(weight.size(0) == (Hq + 2 * Hkv) * k_cache.size(3) &&
                  (!bias.has_value() || bias->numel() == weight.size(0)),
              "qkv width mismatch");
  Product p = run_gemm(x, weight, bias, true);
  const bool done = p.out.defined();         // bias is in there
  if (done) p.partial = Tensor();
  return rope_append_run(p, x, done ? c10::nullopt : bias, k_cache, v_cache,
                         positions, inv_freq, S, Hq, Hkv, block_table, qw, kw,
                         eps, x.numel() / x.size(-1));
}

Tensor sample_tokens(Tensor logits, Tensor temps, Tensor top_ps,
                     Tensor top_ks, Tensor pres, Tensor freqs,
                     c10::optional<Tensor> counts,
                     c10::optional<Tensor> seeds,
                     c10::optional<Tensor> counter, int64_t seed_base) {
  CHECK_IN(logits, torch::kBFloat16);
  CHECK_IN(temps, torch::kFloat);
  CHECK_IN(top_ps, torch::kFloat);
  CHECK_IN(top_ks, torch::kInt);
  CHECK_IN(pres, torch::kFloat);
  CHECK_IN(freqs, torch::kFloat);
  const int B = logits.size(0);
  const int V = logits.size(1);
  void* cnt = nullptr;
  if (counts.has_value()) {
    CHECK_IN(counts.value(), torch::kInt);
    TORCH_CHECK(counts->size(0) == B && counts->size(1) == V,
                "counts must be [B, V]");
    cnt = counts->data_ptr();
  }
  const void* sd = nullptr;
  if (seeds.has_value()) {
    CHECK_IN(seeds.value(), torch::kLong);
    sd = seeds->data_ptr();
  }
  const void* ct = nullptr;
  if (counter.has_value()) {
    CHECK_IN(counter.value(), torch::kLong);
    ct = counter->data_ptr();
  }
  auto out = torch::empty({B}, logits.options().dtype(torch::kLong));
  tl_sample(logits.data_ptr(), temps.data_ptr(), top_ps.data_ptr(),
            top_ks.data_ptr(), pres.data_ptr(), freqs.data_ptr(), cnt, sd,
            ct, out.data_ptr(), (uint64_t)seed_base, B, V, cur_stream());
  return out;
}

void bump_sample_counter(Tensor ctr) {
  CHECK_IN(ctr, torch::kLong);
  tl_bump_counter(ctr.data_ptr(), cur_stream());
}

}  // namespace

void register_mix_ops(pybind11::module& mod);  // bindings_mix.cpp
void register_seq_ops(pybind11::module& mod);  // bindings_seq.cpp
void register_ssm_ops(pybind11::module& mod);  // bindings_ssm.cpp
void register_gla_ops(pybind11::module& mod);  // bindings_gla.cpp
void register_delta_ops(pybind11::module& mod);  // bindings_delta.cpp

PYBIND11_MODULE(TORCH_EXTENSION_NAME, mod) {
  register_mix_ops(mod);
  register_seq_ops(mod);
  register_ssm_ops(mod);
  register_gla_ops(mod);
  register_delta_ops(mod);
  mod.def("rope_append_", &rope_append_,
          "(norm +) RoPE rotate + KV-cache append from fused-QKV rows",
          py::arg("qkv"), py::arg("k_cache"), py::arg("v_cache"),
          py::arg("positions"), py::arg("inv_freq"), py::arg("S"),
          py::arg("Hq"), py::arg("Hkv"), py::arg("block_table"),
          py::arg("qw") = py::none(), py::arg("kw") = py::none(),
          py::arg("eps") = 0.0);
  mod.def("linear_rope_append_", &linear_rope_append_,
          "fused-QKV projection with rope_append_ on its cuts");
  mod.def("add_norm", &add_norm, "residual add (+ RMSNorm)");
  mod.def("linear_add_norm", &linear_add_norm,
          "projection, residual add (+ RMSNorm)");
  mod.def("swiglu_fused", &swiglu_fused, "silu-mul on fused [.,2I] rows");
  mod.def("skinny_glu", &skinny_glu,
          "decode-M SwiGLU of a fused gate and up projection");
  mod.def("skinny_gemm", &skinny_gemm, "decode-M GEMM: x @ W^T + bias");
  mod.def("rmsnorm_fwd", &rmsnorm_fwd, "fused RMSNorm fwd (+residual)");
  mod.def("rmsnorm_bwd", &rmsnorm_bwd, "RMSNorm bwd");
  mod.def("rope_", &rope_, "in-place RoPE apply");
  mod.def("swiglu_fwd", &swiglu_fwd, "silu(gate)*up");
  mod.def("swiglu_bwd", &swiglu_bwd, "SwiGLU bwd");
  mod.def("adamw_", &adamw_, "fused AdamW step");
  mod.def("swiglu_fused_bwd", &swiglu_fused_bwd,
          "gradient of swiglu_fused as one tensor");
  mod.def("ce_fwd", &ce_fwd, "shifted causal-LM cross entropy");
  mod.def("ce_bwd", &ce_bwd, "its gradient in the logits' layout");
  mod.def("rows_split", &rows_split, "projection rows to q, k, and v");
  mod.def("rows_merge", &rows_merge, "its backward");
  mod.def("bias_grad", &bias_grad, "column sums (and GELU's gradient)");
  mod.def("layernorm_fwd", &layernorm_fwd, "(add and) LayerNorm");
  mod.def("layernorm_bwd", &layernorm_bwd, "its backward");
  mod.def("rope_split", &rope_split,
          "fused projection rows to rotated q, k, and v");
  mod.def("rope_merge", &rope_merge,
          "gradients of q, k, v rotated back into projection rows");
  mod.def("decode_attn", &decode_attn, "GQA decode attention over KV cache",
          py::arg("q"), py::arg("k_cache"), py::arg("v_cache"),
          py::arg("seq_lens"), py::arg("scale"), py::arg("n_split"),
          py::arg("block_table"), py::arg("len_add") = 0);
  mod.def("prefill_attn", &prefill_attn, "causal GQA prefill attention");
  mod.def("prefill_attn_cache", &prefill_attn_cache,
          "the same with K and V read from a cache in place");
  mod.def("sample_tokens", &sample_tokens,
          "fused penalties/temperature/top-k/top-p sampling, one block/row");
  mod.def("bump_sample_counter", &bump_sample_counter,
          "advance the graph-safe sampling RNG counter");
  mod.def("prefill_attn_lse", &prefill_attn_lse,
          "causal GQA prefill attention returning (out, logsumexp)");
  mod.def("attn_bwd", &attn_bwd,
          "flash-attention backward: (dq, dk, dv) from the saved out and lse");
}
