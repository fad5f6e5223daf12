// Attention layers of the encoder path, with the reference's class names and call
// signatures:
//   layers::MultiHeadedAttention            turbo_transformers/layers/multi_headed_attention.h:25-129
//   layers::BertAttention                   turbo_transformers/layers/bert_attention.h:25-47
//   layers::MultiHeadedAttentionSmartBatch  turbo_transformers/layers/multi_headed_attention_smart_batch.h:25-137
// MultiHeadedAttention also covers the decoder-side forms of the reference class: "context"
// attention over an encoder memory (separate q/k/v projections, memory_keys/memory_values cache),
// self attention with a growing self_keys/self_values cache, pre-LayerNorm and post_add_input.
//
// Device pipeline of one call (9 -> 6 launches by folding the memory-bound ops into GEMM
// epilogues):
//   QKV GEMM  + bias + head split            -> q,k,v [B,h,S,d]      (gemm012_fused + SplitAddBiasTranspose)
//   QK^T batched GEMM, alpha = 1/sqrt(d)     -> score [B,h,S,S]      (batch_gemm3)
//   mask + softmax in place                                           (ApplyMaskAndSoftmax)
//   P V batched GEMM storing [B,S,h,d]       -> ctx   [B,S,H]         (batch_gemm4 + TransposeForScore)
//   output GEMM                              -> out   [B,S,H]         (gemm5)
//   AddBiasLayerNorm(out, input) in place                             (AddBiasLayerNorm)
#pragma once

#include <algorithm>
#include <initializer_list>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "core/tensor.h"
#include "layers/bert_layers.h"
#include "layers/exchange_memory.h"
#include "layers/packed_weight.h"

namespace turbo_transformers {
namespace layers {

class MultiHeadedAttention {
 public:
  MultiHeadedAttention(core::Tensor k_weight, core::Tensor k_bias, core::Tensor v_weight, core::Tensor v_bias,
                       core::Tensor q_weight, core::Tensor q_bias, core::Tensor dense_weight, core::Tensor dense_bias,
                       core::Tensor qkv_weight, core::Tensor qkv_bias, int64_t num_attention_heads)
      : k_weight_(std::move(k_weight)), k_bias_(std::move(k_bias)), v_weight_(std::move(v_weight)),
        v_bias_(std::move(v_bias)), q_weight_(std::move(q_weight)), q_bias_(std::move(q_bias)),
        dense_weight_(std::move(dense_weight)), dense_bias_(std::move(dense_bias)), qkv_weight_(std::move(qkv_weight)),
        qkv_bias_(std::move(qkv_bias)), layernorm_gamma_(nullptr), layernorm_beta_(nullptr),
        num_attention_heads_(num_attention_heads) {}

  MultiHeadedAttention(core::Tensor k_weight, core::Tensor k_bias, core::Tensor v_weight, core::Tensor v_bias,
                       core::Tensor q_weight, core::Tensor q_bias, core::Tensor dense_weight, core::Tensor dense_bias,
                       core::Tensor qkv_weight, core::Tensor qkv_bias, core::Tensor layernorm_gamma,
                       core::Tensor layernorm_beta, int64_t num_attention_heads)
      : k_weight_(std::move(k_weight)), k_bias_(std::move(k_bias)), v_weight_(std::move(v_weight)),
        v_bias_(std::move(v_bias)), q_weight_(std::move(q_weight)), q_bias_(std::move(q_bias)),
        dense_weight_(std::move(dense_weight)), dense_bias_(std::move(dense_bias)), qkv_weight_(std::move(qkv_weight)),
        qkv_bias_(std::move(qkv_bias)), layernorm_gamma_(std::move(layernorm_gamma)),
        layernorm_beta_(std::move(layernorm_beta)), num_attention_heads_(num_attention_heads) {}

  void EnforceShapeAndType() const;

  // query [B,F,H]; key/value [B,T,H] (read by "context" attention only); attention_mask additive fp32,
  // [B,1,1,T] / [B,1,T] (per key) or [B,F,T], or empty; output [B,F,H]; att_score [B,h,F,T] (may be
  // nullptr: then the probabilities stay internal).  layer_cache entries are [B,h,len,d] or empty.
  void operator()(const core::Tensor& key_tensor, const core::Tensor& value_tensor, const core::Tensor& query_tensor,
                  const core::Tensor& attention_mask, const std::string& attn_type, core::Tensor* output,
                  core::Tensor* att_score, std::unordered_map<std::string, core::Tensor*> layer_cache,
                  bool pre_layernorm = false, bool post_layernorm = false, bool post_add_input = false,
                  bool is_trans_weight = false) const {
    Forward(key_tensor, value_tensor, query_tensor, attention_mask, attn_type, output, att_score, std::move(layer_cache), pre_layernorm,
            post_layernorm, post_add_input, is_trans_weight, {}, *this);
  }

  // The whole attention core runs as one kernel when nobody asks for the probabilities
  // (head size 64, additive key mask broadcast over the query rows).
  // batch, seq, heads: the shape of the batch (fp32 takes the fused kernel only where it pays: everywhere if `in_halves`, which it runs
  // in on a packed batch or one whose V the caller keeps transposed)
  static bool UseFusedCore(const core::Tensor& attention_mask, const core::Tensor* att_score, int64_t head_dim, int dtype,
                           int64_t batch = 0, int64_t seq = 0, int64_t heads = 0, bool in_halves = false);

  WeightRange qkv_weight() const { return qkv_packed_.Range(qkv_weight_); }
  WeightRange dense_weight() const { return dense_packed_.Range(dense_weight_); }

 protected:
  // operator(); `ahead`: what the layer and the following ones read after the attention core (WeightsAhead).
  // `lender`: whose tensors hold Q, K, V, the context ... during the call: those of this layer, or of another one of the stack that
  // runs.  With its own each layer of an encoder writes and reads 4 x rows x hidden values in memory that the last-level cache (256 MB) has
  // seen a whole pass ago, and pushes the weights out of it: us per forward, own / of one layer, base: fp16 20 x 100 tokens 932 / 886, 12 x 64
  // 592 / 527, int8 20 x 128 1356 / 1223.  A layer that is called by itself has its own.
  void Forward(const core::Tensor& key_tensor, const core::Tensor& value_tensor, const core::Tensor& query_tensor,
               const core::Tensor& attention_mask, const std::string& attn_type, core::Tensor* output, core::Tensor* att_score,
               std::unordered_map<std::string, core::Tensor*> layer_cache, bool pre_layernorm, bool post_layernorm,
               bool post_add_input, bool is_trans_weight, const std::vector<WeightRange>& ahead, const MultiHeadedAttention& lender) const;

  // Per-call intermediates, reused across calls (Reshape keeps a buffer that is large enough).
  struct Scratch {
    core::Tensor q, k, v, k_grown, v_grown, kv_bias, ctx, partial, score, ln_query;
    std::mutex mutex;  // from a call's first launch that writes here to its last that reads; all launches are on one stream
  };

  // A key/value cache that the attention core extends: [past | new] along the sequence into the grown tensors.
  struct CacheGrowth {
    const core::Tensor *k_past, *v_past;
    core::Tensor *k_grown, *v_grown;
  };
  // The one-kernel core that also returns the probabilities (head size 64, up to TTMI_PROBS_MAX_KEYS keys).
  bool UseProbsCore(int64_t head_dim, int64_t keys, std::initializer_list<const core::Tensor*> tensors) const;

  // The whole call as one launch (ttmi_decoder_attention): a token each of a few sequences, over a growing cache or a projected memory, with
  // LayerNorm in front and the input added behind; false: nothing was done.
  bool AsOneLaunch(const core::Tensor& query_tensor, const core::Tensor& attention_mask, bool is_self, core::Tensor* output, core::Tensor* att_score,
                   const std::unordered_map<std::string, core::Tensor*>& layer_cache, bool is_trans_weight) const;

  // Attention core and output projection as one launch, the heads' parts of it added up by the LayerNorm behind.
  bool UseProjectingCore(const core::Tensor& query_tensor, const WeightRef& wo, int64_t batch, int64_t seq, int64_t v_pitch, int dtype) const;

  // Everything after q/k/v exist, shared by the dense and the smart-batch layers.
  // `fused_core`: the one-kernel attention core runs; `v_pitch` > 0: v holds V transposed, [B,h,d,v_pitch].
  // `seq` query positions against `key_seq` key positions held in k / v ([B,h,key_seq,d]); with `grow` the first of them
  // are in its past tensors instead, and k / v hold the rest.
  void AttentionTail(Scratch& scratch, const core::Tensor& query_tensor, const core::Tensor& attention_mask, core::Tensor* output,
                     core::Tensor* att_score, int64_t batch, int64_t seq, int64_t key_seq, const core::Tensor& k,
                     const core::Tensor& v, const std::vector<int64_t>* seq_list, bool fused_core, int64_t v_pitch,
                     bool post_layernorm, bool post_add_input, bool is_trans_weight, const CacheGrowth* grow = nullptr,
                     const std::vector<WeightRange>& ahead = {}) const;

  core::Tensor k_weight_, k_bias_, v_weight_, v_bias_, q_weight_, q_bias_;
  core::Tensor dense_weight_, dense_bias_, qkv_weight_, qkv_bias_;
  core::Tensor layernorm_gamma_, layernorm_beta_;
  int64_t num_attention_heads_;

  PackedWeight qkv_packed_, dense_packed_, q_packed_, k_packed_, v_packed_, kv_packed_;
  mutable Scratch scratch_;
  mutable ExchangeMemory exchange_;
  mutable std::mutex mutex_;  // the layer keeps per-call state, like the reference (…attention.cpp:32,272)
};

class BertAttention : public MultiHeadedAttention {
 public:
  BertAttention(core::Tensor qkv_weight, core::Tensor qkv_bias, core::Tensor dense_weight, core::Tensor dense_bias,
                core::Tensor layer_norm_weight, core::Tensor layer_norm_bias, int64_t num_attention_heads)
      : MultiHeadedAttention(core::Tensor(nullptr), core::Tensor(nullptr), core::Tensor(nullptr), core::Tensor(nullptr),
                             core::Tensor(nullptr), core::Tensor(nullptr), std::move(dense_weight), std::move(dense_bias),
                             std::move(qkv_weight), std::move(qkv_bias), std::move(layer_norm_weight),
                             std::move(layer_norm_bias), num_attention_heads) {
    EnforceShapeAndType();
  }
  void EnforceShapeAndType() const;

  void operator()(const core::Tensor& input_tensor, const core::Tensor& attention_mask, core::Tensor* output,
                  core::Tensor* attn = nullptr, bool is_trans_weight = false) const {
    (*this)(input_tensor, attention_mask, output, attn, is_trans_weight, {});
  }
  void operator()(const core::Tensor& input_tensor, const core::Tensor& attention_mask, core::Tensor* output, core::Tensor* attn,
                  bool is_trans_weight, const std::vector<WeightRange>& ahead, const BertAttention* lender = nullptr) const;

  int64_t heads() const { return num_attention_heads_; }
  ExchangeMemory& exchange() const { return exchange_; }  // of the encoder whose first layer this is
  int64_t hidden() const { return dense_weight_.shape(0); }
  DLDataType dtype() const { return dense_weight_.dtype(); }
  // QKV weight [3H,H], bias, output weight [H,H], bias, LayerNorm gamma and beta
  void AppendParameters(std::vector<const void*>* to) const {
    to->insert(to->end(), {qkv_packed_.Get(qkv_weight_, false).data, qkv_bias_.raw(), dense_packed_.Get(dense_weight_, false).data,
                           dense_bias_.raw(), layernorm_gamma_.raw(), layernorm_beta_.raw()});
  }
};

class MultiHeadedAttentionSmartBatch : public MultiHeadedAttention {
 public:
  using MultiHeadedAttention::MultiHeadedAttention;

  // query [1, sum(len), H] packed; attention_mask [B,1,max_len] (-1e9 on pad keys) or empty;
  // output [1, sum(len), H]; att_score [B,h,max_len,max_len] (padded).
  void operator()(const core::Tensor& key_tensor, const core::Tensor& value_tensor, const core::Tensor& query_tensor,
                  const core::Tensor& attention_mask, const std::string& attn_type, core::Tensor* output,
                  core::Tensor* att_score, std::unordered_map<std::string, core::Tensor*> layer_cache,
                  const std::vector<int64_t>& query_seq_len_list, const std::vector<int64_t>& key_seq_len_list,
                  bool pre_layernorm = false, bool post_layernorm = false, bool post_add_input = false,
                  bool is_trans_weight = false) const {
    Forward(key_tensor, value_tensor, query_tensor, attention_mask, attn_type, output, att_score, layer_cache, query_seq_len_list,
            pre_layernorm, post_layernorm, post_add_input, is_trans_weight, {}, *this);
  }
  // self attention, post-LayerNorm, no extra residual, as a layer of an encoder
  void operator()(const core::Tensor& input_tensor, const core::Tensor& attention_mask, core::Tensor* output,
                  const std::vector<int64_t>& seq_len_list, const std::vector<WeightRange>& ahead,
                  const MultiHeadedAttentionSmartBatch& lender) const {
    Forward(input_tensor, input_tensor, input_tensor, attention_mask, "self", output, nullptr, {}, seq_len_list, false, true, false, false,
            ahead, lender);
  }

 private:
  void Forward(const core::Tensor& key_tensor, const core::Tensor& value_tensor, const core::Tensor& query_tensor,
               const core::Tensor& attention_mask, const std::string& attn_type, core::Tensor* output, core::Tensor* att_score,
               const std::unordered_map<std::string, core::Tensor*>& layer_cache, const std::vector<int64_t>& query_seq_len_list,
               bool pre_layernorm, bool post_layernorm, bool post_add_input, bool is_trans_weight,
               const std::vector<WeightRange>& ahead, const MultiHeadedAttentionSmartBatch& lender) const;
};

// One layer of an encoder.
template <typename Attention>
struct EncoderLayer {
  const Attention* attention;
  const BertIntermediate* intermediate;
  const BertOutput* output;
};
// The whole stack as one launch (ttmi_encoder_chain) for up to 16 rows in 16-bit types: a block of the matrix instruction, and one row for each
// of a workgroup's sixteen wavefronts to normalise.  A stack has the bits of its layers run so one by one, whose sums differ from those of the
// sub-layers' own launches: whoever runs whole layers comes here (a stack, a layer of it, the C++ model), so that a model's result does not depend on how it is
// asked for.  (A form of two blocks, us per forward layer by layer / as one launch: fp16 base 1 x 17 305 / 263, 1 x 32 304 / 277, bf16 large 2 x 16 720 /
// 689, is not built.)  false: nothing was done.  `hidden` [batch,seq,H], `mask` additive fp32 per key or empty; `out` may be `hidden` or lie over it.
bool RunEncoderChain(const std::vector<EncoderLayer<BertAttention>>& layers, const core::Tensor& hidden, const core::Tensor& mask,
                     core::Tensor* out);

// What the attention core of each layer may read ahead: the layer's other weights and the next layer's first one.  Nothing
// for weights that stay in the last-level cache (256 MB) from one pass to the next: up to 200 MB of them products run as fast as
// with one weight over and over, of 640 MB 128 x 2304 x 768 in fp32 halves takes 10.4 instead of 8.2 us.  The tensors of a call
// (Q, K, V, context, four of hidden states, two fp32 slices of a product and the intermediate one: rows x (12 x hidden + ffn)) take their
// part of the cache.  From 200 MiB of both on they are read ahead: us per forward without / with, fp16 base (170 MB of weights), 20 x 100 tokens 848 /
// 791, 40 x 128 1573 / 1518; large bf16 (604 MB), 1 x 128 928 / 880, 8 x 128 1601 / 1517.
// Between 195 MB and there weights may leave the cache or not.  Of 640, 768 and 896 columns in 16 bits they do: fp16 base 9 x 128 (198 MB)
// 663 / 629, 11 x 128 731 / 692, 3 x 512 843 / 791, bf16 12 x 128 835 / 734, 13 layers 6 x 128 (203 MB) 600 / 576, 17 of 768 / ffn 1536 16 x 128 1030 /
// 933.  Of 512, 1024 and 1280 they do not, nor in fp32, and reading them costs what a layer holds (6, 25, 39 and from 13 MB): 29 layers of 512 12 x
// 128 1219 / 1229, 7 of 1024 in fp16 6 x 128 426 / 444, 4 of 1280 8 x 128 328 / 342, 6 of 768 in fp32 4 x 128 404 / 428 and 2 x 300 468 / 503,
// 14 of 512 in fp32 8 x 128 806 / 859.  Nor do they where the tensors are few: 13 layers of 768 in fp16 2 x 300 (15 MB of
// them) 564 / 631, 1 x 500 (12 MB) 563 / 609, 14 1 x 300 526 / 556, 5 of 1280 1 x 128 207 / 222.  Below 195 MB in all: base 1 x
// 387 (182 MB) 470 / 535, 4 x 128 457 / 481, 8 x 128 (195 MB) between 587 / 584 and 612 / 587 from process to process.
// Nor for up to 32 rows: those products request all of a workgroup's share of the weights at once (fp32 the fp32 weights as they are), so
// reading ahead is no sooner, and the attention launch waits for it.  us per forward of large bf16 (600 MB), without / with: 1 x 8 tokens 666 /
// 711, 1 x 10 677 / 713, 1 x 20 728 / 748, 1 x 32 715 / 726, 2 x 16 719 / 750, 3 x 10 751 / 854, 8 x 4 809 / 811, 32 x 1 822 / 821; fp16 the same.
bool WeightsLeaveCache(int64_t bytes, int64_t rows, int64_t width, int64_t ffn, int64_t element_size);
template <typename Attention>
std::vector<std::vector<WeightRange>> WeightsAhead(const std::vector<EncoderLayer<Attention>>& layers, const core::Tensor& hidden) {
  std::vector<std::vector<WeightRange>> ahead(layers.size());
  int64_t bytes = 0, ffn = 0;
  for (size_t i = 0; i < layers.size(); ++i) {
    ahead[i] = {layers[i].attention->dense_weight(), layers[i].intermediate->weight(), layers[i].output->weight()};
    const WeightRange qkv = layers[i].attention->qkv_weight();
    for (const WeightRange& r : ahead[i]) bytes += r.bytes;
    bytes += qkv.bytes;
    ffn = std::max(ffn, layers[i].intermediate->out_features());
    if (i > 0) ahead[i - 1].push_back(qkv);
  }
  const int64_t width = hidden.shape(-1), rows = width > 0 ? hidden.numel() / width : 0;
  if (!WeightsLeaveCache(bytes, rows, width, ffn, (int64_t)hidden.element_size())) ahead.assign(layers.size(), {});
  return ahead;
}

}  // namespace layers
}  // namespace turbo_transformers
