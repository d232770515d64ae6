// pybind bindings for the polyrl_amd CDNA4 kernel suite.
#include <torch/extension.h>
#include <vector>

void rmsnorm(torch::Tensor out, torch::Tensor x, torch::Tensor weight,
             double eps);
void fused_add_rmsnorm(torch::Tensor out, torch::Tensor residual,
                       torch::Tensor x, torch::Tensor weight, double eps);
void silu_mul(torch::Tensor out, torch::Tensor gate, torch::Tensor up);
torch::Tensor linear_rows(torch::Tensor x, torch::Tensor w);
torch::Tensor linear_swiglu(torch::Tensor x, torch::Tensor w);
bool linear_rows_pays(long M, long N, long K);
std::vector<long> product_rows(long M, long cols, long K, long least);
void linear_rows_add(torch::Tensor out, torch::Tensor x, torch::Tensor w);
bool linear_joint_takes(const torch::Tensor& x, const std::vector<torch::Tensor>& ws);
std::vector<torch::Tensor> linear_joint(torch::Tensor x, std::vector<torch::Tensor> ws);
bool linear_gated_takes(const torch::Tensor& x, const torch::Tensor& wg,
                        const torch::Tensor& wu);
bool linear_wgrad_pair_takes(const torch::Tensor& dy0, const torch::Tensor& dy1,
                             const torch::Tensor& x);
std::vector<torch::Tensor> linear_wgrad_pair(torch::Tensor dy0, torch::Tensor dy1,
                                             torch::Tensor x);
std::vector<torch::Tensor> linear_gated(torch::Tensor x, torch::Tensor wg,
                                        torch::Tensor wu, bool keep);
bool linear_dgrad_sum_takes(const std::vector<torch::Tensor>& dys,
                            const std::vector<torch::Tensor>& ws);
torch::Tensor linear_dgrad_sum(std::vector<torch::Tensor> dys,
                               std::vector<torch::Tensor> ws);
void linear_rows_into(torch::Tensor& out, const torch::Tensor& x,
                      const torch::Tensor& w);
void rope_inplace(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
                  torch::Tensor cos_tab, torch::Tensor sin_tab);
void rope_kv_append(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                    torch::Tensor positions, torch::Tensor cos_tab,
                    torch::Tensor sin_tab, torch::Tensor k_cache,
                    torch::Tensor v_cache, torch::Tensor slot_mapping);
void gather_logprobs(torch::Tensor out_lp, torch::Tensor out_ent,
                     torch::Tensor logits, torch::Tensor labels,
                     bool want_entropy);
void sample(torch::Tensor out_tokens, torch::Tensor out_logprobs,
            torch::Tensor logits, torch::Tensor temperature,
            torch::Tensor top_k, torch::Tensor top_p, int64_t seed,
            bool no_filter, torch::Tensor seed_dev);
void kv_cache_append(torch::Tensor k_cache, torch::Tensor v_cache,
                     torch::Tensor k, torch::Tensor v,
                     torch::Tensor slot_mapping);
void paged_attention_decode(torch::Tensor out, torch::Tensor q,
                            torch::Tensor k_cache, torch::Tensor v_cache,
                            torch::Tensor page_table,
                            torch::Tensor context_lens, double scale);
void varlen_prefill_attention(torch::Tensor out, torch::Tensor q,
                              torch::Tensor k, torch::Tensor v,
                              torch::Tensor cu_seqlens_q,
                              torch::Tensor cu_seqlens_k,
                              torch::Tensor tile_seq, torch::Tensor tile_q0,
                              double scale, bool causal, torch::Tensor lse);
void varlen_attention_backward(
    torch::Tensor dq, torch::Tensor dk, torch::Tensor dv,
    torch::Tensor q, torch::Tensor k, torch::Tensor v,
    torch::Tensor out, torch::Tensor dout, torch::Tensor lse,
    torch::Tensor cu_seqlens_q, torch::Tensor cu_seqlens_k,
    torch::Tensor tile_seq, torch::Tensor tile_k0,
    double scale, bool causal, bool use_v2);
std::vector<torch::Tensor> rmsnorm_train_fwd(torch::Tensor x,
                                             torch::Tensor res,
                                             torch::Tensor w, double eps);
std::vector<torch::Tensor> rmsnorm_train_bwd(torch::Tensor dy,
                                             torch::Tensor dh,
                                             torch::Tensor h,
                                             torch::Tensor w,
                                             torch::Tensor rstd);
void silu_mul_bwd(torch::Tensor dgate, torch::Tensor dup, torch::Tensor dy,
                  torch::Tensor gate, torch::Tensor up);
void gather_logprobs_train_fwd(torch::Tensor out_lp, torch::Tensor out_lse,
                               torch::Tensor logits, torch::Tensor labels);
torch::Tensor gather_logprobs_train_bwd(torch::Tensor logits,
                                        torch::Tensor labels,
                                        torch::Tensor lse,
                                        torch::Tensor dlp);
torch::Tensor rope_train_apply(torch::Tensor x, torch::Tensor cos_t,
                               torch::Tensor sin_t, bool backward);
torch::Tensor pack_lengths(torch::Tensor mask, torch::Tensor pos);
std::vector<torch::Tensor> pack_rows(torch::Tensor mask, torch::Tensor ids,
                                     torch::Tensor pos, torch::Tensor cu,
                                     int64_t total, int64_t padded, int64_t lo,
                                     int64_t hi);
torch::Tensor gather_rows(torch::Tensor x, torch::Tensor map);
torch::Tensor embed_grad(torch::Tensor dy, torch::Tensor ids, int64_t V);
torch::Tensor tuned_linear_fwd(torch::Tensor x, torch::Tensor w);
long tuned_linear_pick(long M, long N, long K);
torch::Tensor tuned_linear_dgrad(torch::Tensor dy, torch::Tensor w);
torch::Tensor tuned_linear_wgrad(torch::Tensor dy, torch::Tensor x);
torch::Tensor linear_wgrad(torch::Tensor dy, torch::Tensor x);
torch::Tensor linear_dgrad(torch::Tensor dy, torch::Tensor w);
void varlen_attention_backward_v3(
    torch::Tensor dq, torch::Tensor dk, torch::Tensor dv,
    torch::Tensor q, torch::Tensor k, torch::Tensor v,
    torch::Tensor out, torch::Tensor dout, torch::Tensor lse,
    torch::Tensor cu_seqlens_q, torch::Tensor cu_seqlens_k,
    torch::Tensor t64_seq, torch::Tensor t64_q0,
    double scale, bool causal);

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rmsnorm", &rmsnorm, "RMSNorm (bf16, CDNA4)");
  m.def("fused_add_rmsnorm", &fused_add_rmsnorm,
        "residual-add + RMSNorm, residual updated in place");
  m.def("silu_mul", &silu_mul, "SiLU(gate) * up");
  m.def("linear_rows", &linear_rows, "x W^T of prompts");
  m.def("linear_joint_takes", &linear_joint_takes, "linear_joint for a product each");
  m.def("linear_joint", &linear_joint, "x W^T of several weights");
  m.def("linear_wgrad_pair_takes", &linear_wgrad_pair_takes,
        "linear_wgrad_pair for a product each");
  m.def("linear_wgrad_pair", &linear_wgrad_pair, "dY0^T X and dY1^T X");
  m.def("linear_gated_takes", &linear_gated_takes, "linear_gated for a product each");
  m.def("linear_gated", &linear_gated, "silu(x Wg^T) * (x Wu^T), and both products");
  m.def("linear_dgrad_sum_takes", &linear_dgrad_sum_takes,
        "linear_dgrad_sum for a product each");
  m.def("linear_dgrad_sum", &linear_dgrad_sum, "the sum of dY_p W_p");
  m.def("linear_rows_into", &linear_rows_into, "x W^T, W's rows in 8s");
  m.def("linear_rows_add", &linear_rows_add, "out += x W^T, rounded once");
  m.def("linear_rows_pays", &linear_rows_pays, "linear_rows for the library's product");
  m.def("product_rows", &product_rows, "row parts of a product's tiles, their cost");
  m.def("linear_swiglu", &linear_swiglu, "SiLU(x Wg^T) * (x Wu^T)");
  m.def("rope_inplace", &rope_inplace, "NEOX RoPE in place (table-driven)");
  m.def("rope_kv_append", &rope_kv_append,
        "NEOX RoPE in place on q, k + paged KV cache rows, one launch");
  m.def("gather_logprobs", &gather_logprobs,
        "log-softmax gather at labels (+optional entropy)");
  m.def("sample", &sample,
        "fused temperature/top-k/top-p sampling + logprob capture");
  m.def("kv_cache_append", &kv_cache_append, "paged KV cache scatter-append");
  m.def("paged_attention_decode", &paged_attention_decode,
        "paged decode attention (GQA, bf16)");
  m.def("varlen_prefill_attention", &varlen_prefill_attention,
        "varlen causal prefill attention (MFMA, bf16; optional LSE out)");
  m.def("varlen_attention_backward", &varlen_attention_backward,
        "varlen causal flash-attention backward (MFMA, bf16)");
  m.def("rmsnorm_train_fwd", &rmsnorm_train_fwd,
        "trainer RMSNorm fwd (+optional fused residual): y, h, rstd");
  m.def("rmsnorm_train_bwd", &rmsnorm_train_bwd,
        "trainer RMSNorm bwd: dx, dw(fp32)");
  m.def("silu_mul_bwd", &silu_mul_bwd, "silu(gate)*up backward, one pass");
  m.def("gather_logprobs_train_fwd", &gather_logprobs_train_fwd,
        "training logprob gather: lp + logsumexp (bf16 logits)");
  m.def("gather_logprobs_train_bwd", &gather_logprobs_train_bwd,
        "dlogits = dlp * (onehot - softmax), one pass");
  m.def("rope_train_apply", &rope_train_apply,
        "trainer NEOX RoPE (one pass; backward = rotate by -theta)");
  m.def("pack_lengths", &pack_lengths,
        "real tokens of a padded batch's rows, their largest positions");
  m.def("pack_rows", &pack_rows,
        "packed tokens and positions, packed rows of places and back");
  m.def("gather_rows", &gather_rows, "rows that a map names, zeros where none");
  m.def("embed_grad", &embed_grad, "embedding gradient, fp32 sums in row order");
  m.def("tuned_linear_fwd", &tuned_linear_fwd,
        "Y = X W^T via hipBLASLt with per-shape in-process algo search");
  m.def("tuned_linear_pick", &tuned_linear_pick,
        "what tuned_linear_fwd found: 1 the kernel, 0 an algorithm, -1 nothing yet");
  m.def("tuned_linear_dgrad", &tuned_linear_dgrad, "dX = dY W: the kernel where it is the faster, else algo-pinned");
  m.def("tuned_linear_wgrad", &tuned_linear_wgrad,
        "dW = dY^T X: the kernel for many rows, else algo-pinned");
  m.def("linear_wgrad", &linear_wgrad, "dW = dY^T X, the kernel");
  m.def("linear_dgrad", &linear_dgrad, "dX = dY W, the kernel");
  m.def("varlen_attention_backward_v3", &varlen_attention_backward_v3,
        "varlen flash-attention backward v3 (atomic-free dkv+dq split, "
        "head_dim 64/128)");
}
