// The autograd nodes, as functions of the tensors and Python objects the package's `*Fn.apply` take. Each returns what the
// node's forward returns; gradients are wired when the caller's grad mode is on and an input requires one.
#pragma once
#include "ops.hpp"

namespace tfb {

using OptTensor = std::optional<Tensor>;
using Tensors = std::vector<Tensor>;

Tensor rmsnorm_node(const Tensor& x, const OptTensor& w, double eps);
Tensors rmsnorm_pass_node(const Tensor& x, const OptTensor& w, double eps, std::optional<double> y8_scale, bool bytes_only);
Tensors add_rmsnorm_node(const Tensor& x, const Tensor& res, const OptTensor& w, double eps);
Tensors block_head_node(const Tensor& x, const Tensor& x0, const Tensor& l1, const Tensor& l2, const OptTensor& skip, const OptTensor& l3,
                        double eps);
Tensors mix_tail_node(const Tensor& x, const Tensor& lam, int64_t T);
Tensor relu2_node(const Tensor& x);
Tensor linear_node(const Tensor& x, const Tensor& w, const OptTensor& res);
Tensor linear8_node(const Tensor& x, const Tensor& w, PyObject* state, std::optional<double> x_scale, const OptTensor& x8,
                    const OptTensor& res);
Tensor attention_node(const Tensor& q, const Tensor& k, const Tensor& v, double scale, int64_t band);
Tensor rope_attention_node(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t n_head, double scale);
Tensor rope_norm_node(const Tensor& x, const Tensor& cos, const Tensor& sin, double eps);
Tensor rope_norm_attention_node(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t n_head, double scale, double eps,
                                int64_t band, bool heads);   // [B, T, C], or [B, T, H, D]
Tensor qkv_rope_attention_node(const Tensor& x, const Tensor& w, const Tensor& cos, const Tensor& sin, int64_t n_head, double scale);
Tensor mlp8_node(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj, PyObject* state, const OptTensor& x8, const OptTensor& res);
Tensor nr_mlp_node(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj, PyObject* state, double eps);
Tensor mlp_fused_node(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj);
Tensors moe_node(const Tensor& h, const Tensor& router, const Tensor& w_fc, const Tensor& w_proj, PyObject* state, int64_t topk,
                 const OptTensor& bias, const std::vector<double>& aux_weights, int64_t capacity, PyObject* info);
Tensor lm_head_loss_node(const Tensor& x, const Tensor& W, const Tensor& targets, double softcap, bool mean);
Tensor fused_loss_node(const Tensor& logits, const Tensor& targets, double softcap);
Tensor reduced_loss_node(const Tensor& logits, const Tensor& targets, bool mean, double softcap);
Tensor embedding_node(const Tensor& idx, const Tensor& w);

// The amax partials a norm backward hangs on the gradient tensor it wrote, with the tensor's version counter, and their
// retrieval while g2 is still that memory and nothing has been written to it since (nullptr otherwise; a new reference).
void attach_amax(const Tensor& t, PyObject* amax);
PyObject* amax_hint(const Tensor& g, const Tensor& g2);

}  // namespace tfb
