#include "layers/multi_headed_attention.h"

#include <algorithm>
#include <cmath>

#include "core/device_context.h"
#include "layers/kernels.h"
#include "ttmi.h"

namespace turbo_transformers {
namespace layers {

using core::DeviceContext;
using core::Tensor;

static void* Stream() { return DeviceContext::GetInstance().stream(); }

void MultiHeadedAttention::EnforceShapeAndType() const {
  TT_ENFORCE(!qkv_weight_.is_null() && !qkv_bias_.is_null(), "self attention needs the fused qkv weight and bias");
  TT_ENFORCE_EQ(qkv_weight_.n_dim(), (size_t)2, "qkv_weight must be a matrix");
  TT_ENFORCE_EQ(dense_weight_.n_dim(), (size_t)2, "dense_weight must be a matrix");
  TT_ENFORCE_EQ(dense_weight_.shape(0), dense_weight_.shape(1), "dense_weight must be [hidden, hidden]");
  const int64_t hidden = dense_weight_.shape(0);
  TT_ENFORCE_EQ(qkv_weight_.numel(), 3 * hidden * hidden, "qkv_weight must hold 3*hidden*hidden elements");
  TT_ENFORCE_EQ(qkv_bias_.numel(), 3 * hidden, "qkv_bias must hold 3*hidden elements");
  TT_ENFORCE_EQ(dense_bias_.numel(), hidden, "dense_bias must hold hidden elements");
  TT_ENFORCE(num_attention_heads_ > 0 && hidden % num_attention_heads_ == 0, "hidden must be a multiple of the head count");
  TT_ENFORCE(core::SameDataType(qkv_weight_.dtype(), dense_weight_.dtype()), "weights must share one element type");
}

void BertAttention::EnforceShapeAndType() const {
  MultiHeadedAttention::EnforceShapeAndType();
  TT_ENFORCE(!layernorm_gamma_.is_null() && !layernorm_beta_.is_null(), "BertAttention needs LayerNorm parameters");
  TT_ENFORCE_EQ(layernorm_gamma_.numel(), dense_weight_.shape(0), "LayerNorm weight size mismatch");
  TT_ENFORCE_EQ(layernorm_beta_.numel(), dense_weight_.shape(0), "LayerNorm bias size mismatch");
}

bool MultiHeadedAttention::UseFusedCore(const Tensor& attention_mask, const Tensor* att_score, int64_t head_dim, int dtype,
                                        int64_t batch, int64_t seq, int64_t heads, bool in_halves) {
  bool mask_is_key_mask = true;
  if (!attention_mask.is_null()) {
    mask_is_key_mask = attention_mask.n_dim() == 2 || (attention_mask.n_dim() == 3 && attention_mask.shape(1) == 1) ||
                       (attention_mask.n_dim() == 4 && attention_mask.shape(2) == 1);
  }
  bool dtype_ok = dtype == TTMI_F16 || dtype == TTMI_BF16;
  if (dtype == TTMI_F32 && batch > 0) {
    // On the fp32 instruction (a dense batch with V row-major) the kernel is bound by the matrix pipe: a wavefront's 32 queries cost 3.4 us
    // per 64 keys.  It beats the three launches of the chain (18 us) when the sequence is short or when there are wavefronts for half
    // the SIMDs (1024 on this chip).
    const int64_t wave_blocks = batch * heads * ((seq + 31) / 32);
    // In fp16 halves it takes half of that and always wins: dense with V transposed few long sequences have the form that splits the keys
    // (1 x 512: 18 against 34 us); packed, us per forward of base, chain / kernel: 1 x 200 tokens 910 / 760, 1 x 512 1332 / 1136, 150 and
    // 140 992 / 791, 4 x 130 1253 / 1014, 300, 20 and 10 1210 / 921, 3 x 350 1949 / 1384, 8 x 160 1690 / 1342.
    dtype_ok = in_halves || seq <= 128 || wave_blocks >= 512;
  }
  return att_score == nullptr && head_dim == 64 && dtype_ok && mask_is_key_mask;
}

bool MultiHeadedAttention::UseProbsCore(int64_t head_dim, int64_t keys, std::initializer_list<const Tensor*> tensors) const {
  bool aligned = true;
  for (const Tensor* t : tensors) aligned = aligned && reinterpret_cast<uintptr_t>(t->raw()) % 16 == 0;
  return head_dim == 64 && keys > 0 && keys <= TTMI_PROBS_MAX_KEYS && aligned;
}

bool MultiHeadedAttention::UseProjectingCore(const Tensor& query_tensor, const WeightRef& wo, int64_t batch, int64_t seq, int64_t v_pitch, int dtype) const {
  // us per forward of fp16 base, separate / projecting: 1 x 10 tokens 332 / 306, 1 x 32 343 / 311, 2 x 20 366 / 348, 1 x 64 368 / 352, 4 x
  // 16 369 / 360, 1 x 100 437 / 444, 8 x 16 422 / 468.
  // A workgroup takes 32 queries of a head and 128 columns, and computes their attention again for each 128: beyond the two that
  // fit a CU at a time it is more work than the product, and from one per CU on the fp32 slices, one a head, have to be small.
  // Attention to LayerNorm, separate / projecting, weights from HBM, heads x batch x tokens (workgroups): 4 x 64 x 1 (512) 9.1 / 7.4,
  // 8 x 16 x 4 (512) 9.6 / 8.2, 12 x 6 x 10 (432) 10.4 / 9.9, 12 x 8 x 4 (576) 10.1 / 11.7, 12 x 64 x 1 (4608) 11.2 / 36.7; 14 x 1 x 64 (196) 10.7 /
  // 10.5, 16 x 2 x 20 (256) 11.2 / 9.9, 14 x 3 x 21 (294, 3.2 MB of slices) 11.1 / 11.4, 16 x 2 x 33 (512, 4.3 MB) 11.6 / 12.3.
  // Beyond 1024 columns the kernel that sums takes several turns for a row: 20 x 1 x 32 13.0 / 12.3, 24 x 1 x 8 12.0 / 13.3, 32 x 1 x 64 12.8 / 25.3,
  // 64 x 1 x 64 20.8 / 78.9.
  constexpr int64_t kMostRows = 64, kMostColumns = 1024, kSmallSlices = 600 * 1000;
  const int64_t tokens = batch * seq, hidden = query_tensor.shape(-1), heads = num_attention_heads_;
  const int64_t workgroups = (seq + 31) / 32 * batch * heads * ((hidden + 127) / 128), cus = DeviceContext::GetInstance().compute_units();
  const bool wins = tokens <= kMostRows && hidden <= kMostColumns &&
                    (workgroups <= cus || (workgroups <= 2 * cus && heads * tokens * hidden <= kSmallSlices));
  bool aligned = true;
  for (const void* p : {query_tensor.raw(), wo.data, dense_bias_.raw(), layernorm_gamma_.raw(), layernorm_beta_.raw()})
    aligned = aligned && reinterpret_cast<uintptr_t>(p) % 16 == 0;
  return (dtype == TTMI_F16 || dtype == TTMI_BF16) && v_pitch > 0 && wins && aligned;
}

static int64_t RoundUp8(int64_t n) { return (n + 7) / 8 * 8; }

// score -> softmax -> P V -> merge heads -> output projection -> bias (+input) (+LayerNorm)
void MultiHeadedAttention::AttentionTail(Scratch& scratch, const Tensor& query_tensor, const Tensor& attention_mask, Tensor* output,
                                         Tensor* att_score, int64_t batch, int64_t seq, int64_t key_seq, const Tensor& k,
                                         const Tensor& v, const std::vector<int64_t>* seq_list, bool fused_core, int64_t v_pitch,
                                         bool post_layernorm, bool post_add_input, bool is_trans_weight,
                                         const CacheGrowth* grow, const std::vector<WeightRange>& ahead) const {
  const int dt = kernels::DeviceDType(query_tensor);
  const DLDeviceType dev = query_tensor.device_type();
  const int dev_id = query_tensor.device_id();
  const int64_t hidden = query_tensor.shape(-1), heads = num_attention_heads_, d = hidden / heads;
  const int64_t tokens = query_tensor.numel() / hidden;

  const float scaler = 1.0f / std::sqrt(static_cast<float>(d));
  const WeightRef wo = dense_packed_.Get(dense_weight_, is_trans_weight);
  const void* ahead_data[TTMI_MAX_AHEAD];
  int64_t ahead_bytes[TTMI_MAX_AHEAD];
  const size_t ranges = std::min(ahead.size(), (size_t)TTMI_MAX_AHEAD);
  for (size_t i = 0; i < ranges; ++i) ahead_data[i] = ahead[i].data, ahead_bytes[i] = ahead[i].bytes;
  if (fused_core && seq_list == nullptr && post_layernorm && !post_add_input && UseProjectingCore(query_tensor, wo, batch, seq, v_pitch, dt)) {
    if (!attention_mask.is_null()) TT_ENFORCE_EQ(attention_mask.numel(), batch * seq, "attention mask has the wrong size");
    TT_ENFORCE_EQ(seq, key_seq, "the fused core is for self attention without a key/value cache");
    float* partial = scratch.partial.Reshape<float>({heads, tokens, hidden}, dev, dev_id, "gemm5/slices/Reshape");
    TT_DEVICE_CALL(ttmi_attention_projection(scratch.q.raw(), k.raw(), v.raw(), attention_mask.is_null() ? nullptr : attention_mask.data<float>(),
                                             wo.data, partial, batch, heads, seq, d, v_pitch, scaler, dt, ahead_data,
                                             ahead_bytes, (int64_t)ranges, Stream()));
    output->ReshapeAs(query_tensor.dtype(), {query_tensor.shape(0), query_tensor.shape(1), hidden}, dev, dev_id, "gemm5/Reshape");
    kernels::AddSlicesLayerNorm(scratch.partial, query_tensor, dense_bias_, layernorm_gamma_, layernorm_beta_, output, 1e-12f);
    return;
  }
  scratch.ctx.ReshapeAs(query_tensor.dtype(), {tokens, hidden}, dev, dev_id, "batch_gemm4/Reshape");

  // Nobody asked for the probabilities: run the whole core as one kernel; the [B,h,S,S] scores
  // never reach HBM.
  if (fused_core) {
    const float* mask = nullptr;
    if (!attention_mask.is_null()) {
      TT_ENFORCE_EQ(attention_mask.numel(), batch * seq, "attention mask has the wrong size");
      mask = attention_mask.data<float>();
    }
    TT_ENFORCE_EQ(seq, key_seq, "the fused core is for self attention without a key/value cache");
    const int32_t* cu = nullptr;
    if (seq_list != nullptr) cu = DeviceContext::GetInstance().GetSeqPlan(*seq_list).cu_seqlens;
    TT_DEVICE_CALL(ttmi_fused_attention_ahead(scratch.q.raw(), k.raw(), v.raw(), mask, scratch.ctx.mutable_raw(), cu, batch, heads, seq, d,
                                              v_pitch, scaler, dt, ahead_data, ahead_bytes, (int64_t)ranges, Stream()));
  } else {
  Tensor* score = att_score != nullptr ? att_score : &scratch.score;
  // score is [B,h,F,T]: F = query positions, T = key positions (they differ for context attention
  // and when a key/value cache has been prepended)
  const int64_t F = seq, T = key_seq;
  score->ReshapeAs(query_tensor.dtype(), {batch, heads, F, T}, dev, dev_id, "batch_gemm3/Reshape");
  // One kernel for the chain below: 8 hypotheses x 100 keys 4.5 against 14.8 us (fp16), 64 x 64 queries x 256 keys 32
  // against 42; with thousands of workgroups the chain's larger tiles win (32 x 512 x 512: 212 against 201 us).
  const int64_t workgroups = batch * heads * ((F + 31) / 32);
  if (grow != nullptr || (seq_list == nullptr && batch * heads < 65536 && workgroups <= 4096 && UseProbsCore(d, T, {&k, &v}))) {
    const float* mask = nullptr;
    bool per_query = false;
    if (!attention_mask.is_null()) {
      per_query = !(attention_mask.n_dim() == 2 || (attention_mask.n_dim() == 3 && attention_mask.shape(1) == 1) ||
                    (attention_mask.n_dim() == 4 && attention_mask.shape(2) == 1));
      mask = attention_mask.data<float>();
      TT_ENFORCE_EQ(attention_mask.numel(), per_query ? batch * F * T : batch * T, "attention mask has the wrong size");
    }
    TT_DEVICE_CALL(ttmi_attention_with_probs(
        scratch.q.raw(), grow ? grow->k_past->raw() : nullptr, grow ? grow->v_past->raw() : nullptr, grow ? grow->k_past->shape(2) : 0,
        k.raw(), v.raw(), grow ? grow->k_grown->mutable_raw() : nullptr, grow ? grow->v_grown->mutable_raw() : nullptr, mask,
        per_query ? 1 : 0, score->mutable_raw(), scratch.ctx.mutable_raw(), batch, heads, F, T, d, scaler, dt, Stream()));
  } else {
  // batch_gemm3: score[b,h] = scaler * q[b,h] k[b,h]^T   (multi_headed_attention.cpp:328-330)
  TT_DEVICE_CALL(ttmi_gemm_strided_batched(scratch.q.raw(), k.raw(), score->mutable_raw(), F, T, d, d, d, T, F * d, T * d, F * T,
                                           batch * heads, 1, scaler, 0.f, dt, Stream()));
  kernels::ApplyMaskAndSoftmax(score, attention_mask, 1.0f);

  if (seq_list == nullptr) {
    // batch_gemm4 with the [B,h,F,d] -> [B,F,h,d] transpose folded into the store (:345-354)
    TT_DEVICE_CALL(ttmi_gemm_batched_heads(score->raw(), v.raw(), scratch.ctx.mutable_raw(), F, d, T, T, d, hidden, heads,
                                           heads * F * T, F * T, heads * T * d, T * d, F * hidden, d, batch, 0, 1.f, 0.f, dt,
                                           Stream()));
  } else {
    // padded P V, then drop the pad rows while merging heads (…smart_batch.cpp:385-392)
    Tensor& padded = scratch.ln_query;  // free at this point of the call
    padded.ReshapeAs(query_tensor.dtype(), {batch, heads, seq, d}, dev, dev_id, "ApplyMaskAndSoftmax/Reshape");
    TT_DEVICE_CALL(ttmi_gemm_strided_batched(score->raw(), v.raw(), padded.mutable_raw(), seq, d, seq, seq, d, d, seq * seq,
                                             seq * d, seq * d, batch * heads, 0, 1.f, 0.f, dt, Stream()));
    kernels::TransposeForScorePad(&scratch.ctx, padded, *seq_list);
  }
  }  // chain
  }  // unfused core

  output->ReshapeAs(query_tensor.dtype(), {query_tensor.shape(0), query_tensor.shape(1), hidden}, dev, dev_id, "gemm5/Reshape");
  if (!post_add_input && post_layernorm) {
    // gemm5 then AddBiasLayerNorm(query, bias, gamma, beta, out), eps 1e-12 (:359-371)
    kernels::GemmAddBiasLayerNorm(scratch.ctx, wo, hidden, query_tensor, dense_bias_, layernorm_gamma_, layernorm_beta_, output, 1e-12f);
  } else {
    ttmi_epilogue_args args{};
    args.bias = dense_bias_.raw();
    args.residual = post_add_input ? query_tensor.raw() : nullptr;
    TT_DEVICE_CALL(ttmi_gemm_fused(scratch.ctx.raw(), wo.data, output->mutable_raw(), tokens, hidden, hidden, hidden, hidden, hidden,
                                   post_add_input ? TTMI_EPI_BIAS_RESIDUAL : TTMI_EPI_BIAS, &args, wo.DTypeFor(dt), Stream()));
  }
}

// One projection followed by AddBiasTransposeForScore, as one GEMM: x[B,S,H] W + b -> [B,h,S,d]
// (multi_headed_attention.cpp:73-88, :107-150).
static void ProjectToHeads(const Tensor& x, const WeightRef& packed_w, const Tensor& bias, int64_t heads, Tensor* out,
                           const char* name) {
  const int64_t batch = x.shape(0), seq = x.shape(1), hidden = x.shape(2), d = hidden / heads;
  out->ReshapeAs(x.dtype(), {batch, heads, seq, d}, x.device_type(), x.device_id(), name);
  ttmi_epilogue_args args{};
  args.bias = bias.raw();
  args.q = out->mutable_raw();
  args.seq = seq;
  args.heads = heads;
  args.head_dim = d;
  TT_DEVICE_CALL(ttmi_gemm_fused(x.raw(), packed_w.data, nullptr, batch * seq, hidden, hidden, hidden, hidden, hidden,
                                 TTMI_EPI_QKV_SPLIT, &args, packed_w.DTypeFor(kernels::DeviceDType(x)), Stream()));
}

static bool CacheHas(const std::unordered_map<std::string, Tensor*>& cache, const char* key) {
  auto it = cache.find(key);
  return it != cache.end() && it->second != nullptr && !it->second->is_null();
}

// cache[key] = a copy of `src` (multi_headed_attention.cpp:216-229)
static void StoreInCache(std::unordered_map<std::string, Tensor*>& cache, const char* key, const Tensor& src, const char* name) {
  auto it = cache.find(key);
  TT_ENFORCE(it != cache.end() && it->second != nullptr, "layer_cache has no entry %s", key);
  std::vector<int64_t> shape;
  for (size_t i = 0; i < src.n_dim(); ++i) shape.push_back(src.shape((int)i));
  it->second->ReshapeAs(src.dtype(), shape, src.device_type(), src.device_id(), name);
  core::CopyBytes(it->second->mutable_raw(), src.device_type(), src.raw(), src.device_type(),
                  (size_t)src.numel() * src.element_size());
}

bool MultiHeadedAttention::AsOneLaunch(const Tensor& query_tensor, const Tensor& attention_mask, bool is_self, Tensor* output, Tensor* att_score,
                                       const std::unordered_map<std::string, Tensor*>& layer_cache, bool is_trans_weight) const {
  const int dt = kernels::DeviceDType(query_tensor);
  if (query_tensor.shape(0) > TTMI_CHAIN_MAX_ROWS || query_tensor.shape(1) != 1 || att_score == nullptr) return false;
  const char *key_name = is_self ? "self_keys" : "memory_keys", *value_name = is_self ? "self_values" : "memory_values";
  if (!CacheHas(layer_cache, key_name) || !CacheHas(layer_cache, value_name)) return false;
  const Tensor &k_past = *layer_cache.at(key_name), &v_past = *layer_cache.at(value_name);
  const int64_t batch = query_tensor.shape(0), hidden = query_tensor.shape(2), heads = num_attention_heads_, past = k_past.shape(2);
  const int64_t keys = is_self ? past + 1 : past, width = is_self ? 3 * hidden : hidden;
  if (past < 1 || v_past.shape(2) != past || layernorm_gamma_.numel() != hidden || layernorm_beta_.numel() != hidden) return false;
  int64_t bytes = 0;
  TT_DEVICE_CALL(ttmi_decoder_chain_workspace(batch, heads, hidden, width, keys, dt, &bytes));
  if (bytes == 0) return false;
  const float* mask = nullptr;
  if (!attention_mask.is_null()) {
    if (attention_mask.numel() != batch * keys) return false;
    mask = attention_mask.data<float>();
  }
  if (is_self) MultiHeadedAttention::EnforceShapeAndType();
  for (const Tensor* t : {&q_weight_, &k_weight_, &v_weight_, &q_bias_, &k_bias_, &v_bias_})
    if (!is_self && t->is_null()) return false;
  const Tensor &in_weight = is_self ? qkv_weight_ : q_weight_, &in_bias = is_self ? qkv_bias_ : q_bias_;
  if (in_weight.numel() != width * hidden || in_bias.numel() != width) return false;
  const void* w_in = (is_self ? qkv_packed_ : q_packed_).Get(in_weight, is_trans_weight).data;
  const void* w_out = dense_packed_.Get(dense_weight_, is_trans_weight).data;
  const DLDeviceType dev = query_tensor.device_type();
  const int dev_id = query_tensor.device_id();
  uintptr_t bits = 0;
  for (const void* p : {query_tensor.raw(), layernorm_gamma_.raw(), layernorm_beta_.raw(), w_in, in_bias.raw(), w_out, dense_bias_.raw(), k_past.raw(), v_past.raw()})
    bits |= reinterpret_cast<uintptr_t>(p);
  if ((bits & 15) != 0) return false;
  Tensor out_apart(nullptr), probs_apart(nullptr);
  Tensor* const out = kernels::ResultBeside(output, {&query_tensor, &attention_mask, &k_past, &v_past}, &out_apart, query_tensor.dtype(), {batch, 1, hidden},
                                            dev, dev_id, "gemm5/Reshape");
  Tensor* const probs = kernels::ResultBeside(att_score, {&query_tensor, &attention_mask, &k_past, &v_past, out}, &probs_apart, query_tensor.dtype(),
                                              {batch, heads, 1, keys}, dev, dev_id, "batch_gemm3/Reshape");
  if (reinterpret_cast<uintptr_t>(out->raw()) % 16 != 0) return false;
  Tensor k_grown(nullptr), v_grown(nullptr);
  if (is_self) {
    k_grown.ReshapeAs(query_tensor.dtype(), {batch, heads, keys, hidden / heads}, dev, dev_id, "self/self_key/Reshape");
    v_grown.ReshapeAs(query_tensor.dtype(), {batch, heads, keys, hidden / heads}, dev, dev_id, "self/self_value/Reshape");
  }
  exchange_.Use(bytes, dev, dev_id, [&](void* memory, int turn) {
    TT_DEVICE_CALL(ttmi_decoder_attention(query_tensor.raw(), layernorm_gamma_.raw(), layernorm_beta_.raw(), 1e-6f, w_in, in_bias.raw(), w_out,
                                          dense_bias_.raw(), k_past.raw(), v_past.raw(), is_self ? k_grown.mutable_raw() : nullptr,
                                          is_self ? v_grown.mutable_raw() : nullptr, mask, probs->mutable_raw(), out->mutable_raw(), memory, turn, batch, heads, hidden,
                                          keys, 1.0f / std::sqrt(static_cast<float>(hidden / heads)), dt, 0, 0, Stream()));
  });
  if (out != output) *output = std::move(out_apart);
  if (probs != att_score) *att_score = std::move(probs_apart);
  if (is_self) {
    *layer_cache.at(key_name) = std::move(k_grown);
    *layer_cache.at(value_name) = std::move(v_grown);
  }
  return true;
}

void MultiHeadedAttention::Forward(const Tensor& key_tensor, const Tensor& value_tensor, const Tensor& query_tensor,
                                   const Tensor& attention_mask, const std::string& attn_type, Tensor* output,
                                   Tensor* att_score, std::unordered_map<std::string, Tensor*> layer_cache,
                                   bool pre_layernorm, bool post_layernorm, bool post_add_input, bool is_trans_weight,
                                   const std::vector<WeightRange>& ahead, const MultiHeadedAttention& lender) const {
  std::lock_guard<std::mutex> g(mutex_);
  Scratch& scratch = lender.scratch_;
  std::lock_guard<std::mutex> use(scratch.mutex);
  const bool is_self = attn_type == "self";
  TT_ENFORCE(is_self || attn_type == "context", "attn_type should be context or self.");
  TT_ENFORCE_EQ(query_tensor.n_dim(), (size_t)3, "The query_tensors should be a matrix with shape [batch_size, query_seq_len, hidden_size].");
  TT_ENFORCE(output != nullptr, "output must not be null");
  kernels::RequireGpu(query_tensor, "MultiHeadedAttention");
  TT_ENFORCE_EQ(dense_weight_.n_dim(), (size_t)2, "dense_weight must be a matrix");

  const int64_t batch = query_tensor.shape(0), seq = query_tensor.shape(1), hidden = query_tensor.shape(2);
  TT_ENFORCE_EQ(hidden, dense_weight_.shape(0), "hidden size of the input and of the weights differ");
  TT_ENFORCE(core::SameDataType(query_tensor.dtype(), dense_weight_.dtype()), "input and weights must share one element type");
  const int64_t heads = num_attention_heads_, d = hidden / heads;
  TT_ENFORCE(heads > 0 && hidden % heads == 0, "hidden must be a multiple of the head count");
  const int dt = kernels::DeviceDType(query_tensor);
  const DLDeviceType dev = query_tensor.device_type();
  const int dev_id = query_tensor.device_id();
  for (const auto& kv : layer_cache) {
    if (kv.second == nullptr || kv.second->is_null()) continue;
    kernels::RequireGpu(*kv.second, "layer_cache");
    TT_ENFORCE(core::SameDataType(kv.second->dtype(), query_tensor.dtype()), "layer_cache[%s] and the query differ in element type", kv.first.c_str());
    TT_ENFORCE(kv.second->n_dim() == 4 && kv.second->shape(0) == batch && kv.second->shape(1) == heads && kv.second->shape(3) == d,
               "layer_cache[%s] must be [batch, heads, len, head_dim]", kv.first.c_str());
  }

  if (pre_layernorm) TT_ENFORCE(!layernorm_gamma_.is_null() && !layernorm_beta_.is_null(), "pre_layernorm needs LayerNorm parameters");
  if (pre_layernorm && post_add_input && AsOneLaunch(query_tensor, attention_mask, is_self, output, att_score, layer_cache, is_trans_weight)) return;
  // a projection of the query, with LayerNorm in front where asked for (:66-80, :190-199 -- eps is 1e-6 there)
  auto project_query = [&](const WeightRef& packed_w, int64_t n, const ttmi_epilogue_args& args) {
    if (pre_layernorm) {
      kernels::LayerNormGemm(query_tensor, layernorm_gamma_, layernorm_beta_, 1e-6f, &scratch.ln_query, packed_w, nullptr, n,
                             TTMI_EPI_QKV_SPLIT, args);
    } else {
      TT_DEVICE_CALL(ttmi_gemm_fused(query_tensor.raw(), packed_w.data, nullptr, batch * seq, n, hidden, hidden, hidden, n,
                                     TTMI_EPI_QKV_SPLIT, &args, packed_w.DTypeFor(dt), Stream()));
    }
  };

  const Tensor* k_used = &scratch.k;
  const Tensor* v_used = &scratch.v;
  int64_t v_pitch = 0;
  bool fused_core = false;
  // What a call adds to the layer cache is computed into fresh tensors and moved there: no copy.
  auto fresh = [&](int64_t len, const char* name) {
    Tensor t(nullptr);
    t.ReshapeAs(query_tensor.dtype(), {batch, heads, len, d}, dev, dev_id, name);
    return t;
  };
  auto move_to_cache = [&](const char* key, Tensor& t) -> const Tensor* {
    auto it = layer_cache.find(key);
    TT_ENFORCE(it != layer_cache.end() && it->second != nullptr, "layer_cache has no entry %s", key);
    *it->second = std::move(t);
    return it->second;
  };
  Tensor k_cache(nullptr), v_cache(nullptr);
  CacheGrowth growth{};
  if (is_self) {
    MultiHeadedAttention::EnforceShapeAndType();
    // with the fused core V is kept transposed, [B,h,d,pitch]: its tiles are then plain copies.
    // A key/value cache needs the row-major layout (it is appended along the sequence).
    const bool fused_self = layer_cache.empty() && UseFusedCore(attention_mask, att_score, d, dt, batch, seq, heads, true);
    if (fused_self) v_pitch = RoundUp8(seq);
    fused_core = fused_self;
    scratch.q.ReshapeAs(query_tensor.dtype(), {batch, heads, seq, d}, dev, dev_id, "self/q/Reshape");
    const bool past_k = CacheHas(layer_cache, "self_keys"), past_v = CacheHas(layer_cache, "self_values");
    Tensor* k_new = &scratch.k;  // where the projection puts keys and values
    Tensor* v_new = &scratch.v;
    if (!layer_cache.empty() && !past_k && !past_v) {
      k_cache = fresh(seq, "self/self_key/Reshape");
      v_cache = fresh(seq, "self/self_value/Reshape");
      k_new = &k_cache;
      v_new = &v_cache;
    } else {
    scratch.k.ReshapeAs(query_tensor.dtype(), {batch, heads, seq, d}, dev, dev_id, "self/k/Reshape");
    if (v_pitch > 0) scratch.v.ReshapeAs(query_tensor.dtype(), {batch, heads, d, v_pitch}, dev, dev_id, "self/v/Reshape");
    else scratch.v.ReshapeAs(query_tensor.dtype(), {batch, heads, seq, d}, dev, dev_id, "self/v/Reshape");
    }
    // gemm012_fused + SplitAddBiasTransposeForScore in one launch (:199-203)
    ttmi_epilogue_args args{};
    args.bias = qkv_bias_.raw();
    args.q = scratch.q.mutable_raw();
    args.k = k_new->mutable_raw();
    args.v = v_new->mutable_raw();
    args.seq = seq;
    args.heads = heads;
    args.head_dim = d;
    args.v_seq_pitch = v_pitch;
    project_query(qkv_packed_.Get(qkv_weight_, is_trans_weight), 3 * hidden, args);
    // decoder self attention: earlier keys/values come first (:205-214), the grown tensors go back (:216-229)
    auto prepend = [&](const char* key, Tensor* cur, Tensor* grown, const char* name) {
      if (!CacheHas(layer_cache, key)) return;
      const Tensor& past = *layer_cache.at(key);
      const int64_t past_len = past.shape(2);
      grown->ReshapeAs(query_tensor.dtype(), {batch, heads, past_len + seq, d}, dev, dev_id, name);
      TT_DEVICE_CALL(ttmi_concat(past.raw(), cur->raw(), grown->mutable_raw(), batch * heads, past_len * d, seq * d, dt, Stream()));
      std::swap(*cur, *grown);
    };
    if (k_new == &k_cache) {
      k_used = move_to_cache("self_keys", k_cache);
      v_used = move_to_cache("self_values", v_cache);
    } else if (past_k && past_v && batch * heads < 65536 && layer_cache.at("self_keys")->shape(2) > 0 &&
               layer_cache.at("self_keys")->shape(2) == layer_cache.at("self_values")->shape(2) &&
               UseProbsCore(d, layer_cache.at("self_keys")->shape(2) + seq, {layer_cache.at("self_keys"), layer_cache.at("self_values")})) {
      // the attention core reads [past | new] in place and writes the grown cache on the way
      const int64_t total = layer_cache.at("self_keys")->shape(2) + seq;
      k_cache = fresh(total, "self/self_key/Reshape");
      v_cache = fresh(total, "self/self_value/Reshape");
      growth = CacheGrowth{layer_cache.at("self_keys"), layer_cache.at("self_values"), &k_cache, &v_cache};
    } else {
      prepend("self_keys", &scratch.k, &scratch.k_grown, "self/keys/Concat");
      prepend("self_values", &scratch.v, &scratch.v_grown, "self/values/Concat");
    }
    if (!layer_cache.empty() && k_used == &scratch.k && growth.k_grown == nullptr) {
      StoreInCache(layer_cache, "self_keys", scratch.k, "self/self_key/Reshape");
      StoreInCache(layer_cache, "self_values", scratch.v, "self/self_value/Reshape");
    }
  } else {
    TT_ENFORCE(!q_weight_.is_null() && !k_weight_.is_null() && !v_weight_.is_null() && !q_bias_.is_null() && !k_bias_.is_null() &&
                   !v_bias_.is_null(), "context attention needs the separate q/k/v weights and biases");
    scratch.q.ReshapeAs(query_tensor.dtype(), {batch, heads, seq, d}, dev, dev_id, "context/AddBiasTransposeForScore/q_out2/Reshape");
    ttmi_epilogue_args args{};
    args.bias = q_bias_.raw();
    args.q = scratch.q.mutable_raw();
    args.seq = seq;
    args.heads = heads;
    args.head_dim = d;
    project_query(q_packed_.Get(q_weight_, is_trans_weight), hidden, args);
    if (CacheHas(layer_cache, "memory_keys") && CacheHas(layer_cache, "memory_values")) {
      // the encoder memory was projected at an earlier step (:90-105); used in place, no copy
      k_used = layer_cache.at("memory_keys");
      v_used = layer_cache.at("memory_values");
    } else {
      TT_ENFORCE_EQ(key_tensor.n_dim(), (size_t)3, "The key_tensor should be a matrix with shape [batch_size, key_seq_len, hidden_size].");
      TT_ENFORCE_EQ(value_tensor.n_dim(), (size_t)3, "The value_tensor should be a matrix with shape [batch_size, key_seq_len, hidden_size].");
      kernels::RequireGpu(key_tensor, "MultiHeadedAttention");
      kernels::RequireGpu(value_tensor, "MultiHeadedAttention");
      TT_ENFORCE(key_tensor.shape(0) == batch && value_tensor.shape(0) == batch && key_tensor.shape(1) == value_tensor.shape(1) &&
                     key_tensor.shape(2) == hidden && value_tensor.shape(2) == hidden,
                 "key and value must be [batch_size, key_seq_len, hidden_size]");
      TT_ENFORCE(core::SameDataType(key_tensor.dtype(), query_tensor.dtype()) && core::SameDataType(value_tensor.dtype(), query_tensor.dtype()),
                 "key, value and query must share one element type");
      const bool keep = !layer_cache.empty();  // :128-150
      Tensor *k_out = keep ? &k_cache : &scratch.k, *v_out = keep ? &v_cache : &scratch.v;
      // Keys and values are usually projections of the same memory: then one product against both weights, whose tiles fill the
      // last round of workgroups better than two launches do (fp32 800 x 768: 2 x 16.3 us, together 23.3 and 2 for the bias, which is
      // joined on each call because it is read where the caller keeps it).
      const bool shared = key_tensor.raw() == value_tensor.raw() && !is_trans_weight && k_weight_.n_dim() == 2 && k_weight_.shape(1) == hidden &&
                          k_weight_.numel() == v_weight_.numel() && k_bias_.numel() == hidden && v_bias_.numel() == hidden;
      if (shared) {
        const int64_t len = key_tensor.shape(1);
        k_out->ReshapeAs(query_tensor.dtype(), {batch, heads, len, d}, dev, dev_id, "context/keys/AddBiasTransposeForScore/Reshape");
        v_out->ReshapeAs(query_tensor.dtype(), {batch, heads, len, d}, dev, dev_id, "context/values/AddBiasTransposeForScore/Reshape");
        scratch.kv_bias.ReshapeAs(query_tensor.dtype(), {2 * hidden}, dev, dev_id, "context/kv_bias/Reshape");
        TT_DEVICE_CALL(ttmi_concat(k_bias_.raw(), v_bias_.raw(), scratch.kv_bias.mutable_raw(), 1, hidden, hidden, dt, Stream()));
        ttmi_epilogue_args kv{};
        kv.bias = scratch.kv_bias.raw();
        kv.q = k_out->mutable_raw();
        kv.k = v_out->mutable_raw();
        kv.seq = len;
        kv.heads = heads;
        kv.head_dim = d;
        const WeightRef both = kv_packed_.GetPair(k_weight_, v_weight_);
        TT_DEVICE_CALL(ttmi_gemm_fused(key_tensor.raw(), both.data, nullptr, batch * len, 2 * hidden, hidden, hidden, hidden,
                                       2 * hidden, TTMI_EPI_QKV_SPLIT, &kv, both.DTypeFor(dt), Stream()));
      } else {
        ProjectToHeads(key_tensor, k_packed_.Get(k_weight_, is_trans_weight), k_bias_, heads, k_out, "context/keys/AddBiasTransposeForScore/Reshape");
        ProjectToHeads(value_tensor, v_packed_.Get(v_weight_, is_trans_weight), v_bias_, heads, v_out, "context/values/AddBiasTransposeForScore/Reshape");
      }
      if (keep) {
        k_used = move_to_cache("memory_keys", k_cache);
        v_used = move_to_cache("memory_values", v_cache);
      }
    }
  }
  const bool growing = growth.k_grown != nullptr;
  const int64_t key_seq = fused_core ? seq : growing ? k_cache.shape(2) : k_used->shape(2);
  TT_ENFORCE_EQ(fused_core ? seq : growing ? v_cache.shape(2) : v_used->shape(2), key_seq, "keys and values differ in length");

  AttentionTail(scratch, query_tensor, attention_mask, output, att_score, batch, seq, key_seq, *k_used, *v_used, nullptr, fused_core, v_pitch,
                post_layernorm, post_add_input, is_trans_weight, growing ? &growth : nullptr, ahead);
  if (growing) {
    move_to_cache("self_keys", k_cache);
    move_to_cache("self_values", v_cache);
  }
}

void BertAttention::operator()(const Tensor& input_tensor, const Tensor& attention_mask, Tensor* output, Tensor* attn,
                               bool is_trans_weight, const std::vector<WeightRange>& ahead, const BertAttention* lender) const {
  // bert_attention.cpp:29-47: self attention, post-LayerNorm, no extra residual
  std::unordered_map<std::string, Tensor*> dummy{};
  Forward(input_tensor, input_tensor, input_tensor, attention_mask, "self", output, attn, dummy, false /* pre_layernorm */,
          true /* post_layernorm */, false /* post_add_input */, is_trans_weight, ahead,
          lender != nullptr ? *lender : *this);
}

bool WeightsLeaveCache(int64_t bytes, int64_t rows, int64_t width, int64_t ffn, int64_t element_size) {
  constexpr int64_t kMB = 1000 * 1000, kLeaves = 200ll << 20, kMayLeave = 195 * kMB;
  if (rows <= 32) return false;
  const int64_t tensors = rows * (12 * width + ffn) * element_size, layer = (4 * width * width + 2 * width * ffn) * element_size;
  if (bytes + tensors > kLeaves) return true;
  return bytes + tensors > kMayLeave && element_size == 2 && tensors > 18 * kMB && layer > 8 * kMB && layer < 22 * kMB;
}

void MultiHeadedAttentionSmartBatch::Forward(const Tensor& key_tensor, const Tensor& value_tensor, const Tensor& query_tensor,
                                             const Tensor& attention_mask, const std::string& attn_type, Tensor* output,
                                             Tensor* att_score, const std::unordered_map<std::string, Tensor*>& layer_cache,
                                             const std::vector<int64_t>& query_seq_len_list, bool pre_layernorm, bool post_layernorm,
                                             bool post_add_input, bool is_trans_weight, const std::vector<WeightRange>& ahead,
                                             const MultiHeadedAttentionSmartBatch& lender) const {
  std::lock_guard<std::mutex> g(mutex_);
  Scratch& scratch = lender.scratch_;
  std::lock_guard<std::mutex> use(scratch.mutex);
  TT_ENFORCE(attn_type == "self", "only attn_type \"self\" is built (\"context\" belongs to the decoder path)");
  TT_ENFORCE(layer_cache.empty(), "layer_cache belongs to the decoder path and is not built");
  TT_ENFORCE(!pre_layernorm, "pre_layernorm is not built for the smart-batch layer");
  TT_ENFORCE_EQ(query_tensor.n_dim(), (size_t)3, "The query_tensors should be a matrix with shape [1, sum_query_seq_len, hidden_size].");
  TT_ENFORCE_EQ(query_tensor.shape(0), (int64_t)1, "a packed batch has leading dimension 1");
  TT_ENFORCE(output != nullptr, "output must not be null");
  kernels::RequireGpu(query_tensor, "MultiHeadedAttentionSmartBatch");
  MultiHeadedAttention::EnforceShapeAndType();
  (void)key_tensor;
  (void)value_tensor;

  auto plan = DeviceContext::GetInstance().GetSeqPlan(query_seq_len_list);
  TT_ENFORCE_EQ(query_tensor.shape(1), plan.total, "The query_tensor shape 1 should be the sum of seq_len_list.");
  const int64_t hidden = query_tensor.shape(2), heads = num_attention_heads_, d = hidden / heads;
  TT_ENFORCE_EQ(hidden, dense_weight_.shape(0), "hidden size of the input and of the weights differ");
  TT_ENFORCE(core::SameDataType(query_tensor.dtype(), qkv_weight_.dtype()), "input and weights must share one element type");
  const int dt = kernels::DeviceDType(query_tensor);
  const DLDeviceType dev = query_tensor.device_type();
  const int dev_id = query_tensor.device_id();
  const int64_t batch = plan.batch, max_seq = plan.max_seq;

  // Padded q,k,v; the QKV GEMM scatters bias-added rows of the packed input into them.  The
  // unfused core multiplies whole padded tensors, so pad rows must be exactly 0 there
  // (transpose.cpp:504-522); the fused kernel never reads a pad row, so nothing is cleared.
  // V stays row-major here: the transposed store needs the row map and a division per group of eight packed rows,
  // and that costs the QKV GEMM more than the scatter costs the attention kernel (20 requests, 6275 tokens:
  // 2.50 against 2.39 ms per forward).
  const bool fused_core = UseFusedCore(attention_mask, att_score, d, dt, batch, max_seq, heads, true);
  Tensor* qkv[3] = {&scratch.q, &scratch.k, &scratch.v};
  const char* names[3] = {"self/q/Reshape", "self/k/Reshape", "self/v/Reshape"};
  for (int i = 0; i < 3; ++i) {
    qkv[i]->ReshapeAs(query_tensor.dtype(), {batch, heads, max_seq, d}, dev, dev_id, names[i]);
    if (fused_core) continue;
    const size_t bytes = (size_t)qkv[i]->numel() * qkv[i]->element_size();
    TT_DEVICE_CALL(ttmi_memset_zero(qkv[i]->mutable_raw(), (bytes + 3) / 4 * 4  /* capacity is rounded to 512 B */, Stream()));
  }
  ttmi_epilogue_args args{};
  args.bias = qkv_bias_.raw();
  args.q = scratch.q.mutable_raw();
  args.k = scratch.k.mutable_raw();
  args.v = scratch.v.mutable_raw();
  args.seq = max_seq;
  args.heads = heads;
  args.head_dim = d;
  args.token_rows = plan.token_rows;
  args.batch = batch;
  const WeightRef wqkv = qkv_packed_.Get(qkv_weight_, is_trans_weight);
  TT_DEVICE_CALL(ttmi_gemm_fused(query_tensor.raw(), wqkv.data, nullptr, plan.total, 3 * hidden, hidden, hidden, hidden, 3 * hidden,
                                 TTMI_EPI_QKV_SPLIT_PAD, &args, wqkv.DTypeFor(dt), Stream()));

  AttentionTail(scratch, query_tensor, attention_mask, output, att_score, batch, max_seq, max_seq, scratch.k, scratch.v, &query_seq_len_list, fused_core, 0,
                post_layernorm, post_add_input, is_trans_weight, nullptr, ahead);
}

bool RunEncoderChain(const std::vector<EncoderLayer<BertAttention>>& layers, const Tensor& hidden, const Tensor& mask, Tensor* out) {
  if (layers.empty() || hidden.is_null() || !hidden.is_gpu() || hidden.n_dim() != 3) return false;
  const BertAttention& first = *layers[0].attention;
  const int64_t batch = hidden.shape(0), seq = hidden.shape(1), width = hidden.shape(2), rows = batch * seq;
  const int64_t heads = first.heads(), ffn = layers[0].intermediate->out_features(), count = (int64_t)layers.size();
  const int dt = core::ToDeviceDType(hidden.dtype());
  if (batch < 1 || seq < 1 || first.hidden() != width) return false;
  int64_t bytes = 0;
  TT_DEVICE_CALL(ttmi_encoder_chain_workspace(count, rows, heads, width, ffn, dt, &bytes));
  if (bytes <= 0) return false;
  for (const auto& l : layers) {
    const bool same = l.attention->heads() == heads && l.attention->hidden() == width && l.intermediate->in_features() == width &&
                      l.intermediate->out_features() == ffn && l.output->in_features() == ffn && l.output->out_features() == width &&
                      core::SameDataType(l.attention->dtype(), hidden.dtype()) && core::SameDataType(l.intermediate->dtype(), hidden.dtype()) &&
                      core::SameDataType(l.output->dtype(), hidden.dtype());
    if (!same) return false;
  }
  const float* additive = nullptr;
  if (!mask.is_null()) {
    if (!MultiHeadedAttention::UseFusedCore(mask, nullptr, width / heads, dt) || mask.numel() != rows) return false;
    additive = mask.data<float>();
  }
  std::vector<const void*> parameters;
  parameters.reserve(12 * layers.size());
  for (const auto& l : layers) {
    l.attention->AppendParameters(&parameters);
    l.intermediate->AppendParameters(&parameters);
    l.output->AppendParameters(&parameters);
  }
  const float* input32 = hidden.shadow() != nullptr ? hidden.shadow()->data<float>() : nullptr;
  uintptr_t bits = reinterpret_cast<uintptr_t>(hidden.raw()) | reinterpret_cast<uintptr_t>(input32);
  for (const void* p : parameters) bits |= reinterpret_cast<uintptr_t>(p);
  if ((bits & 15) != 0) return false;
  const DLDeviceType dev = hidden.device_type();
  const int dev_id = hidden.device_id();
  // A workgroup that starts late reads the input late: where the result would lie over it (the same tensor, or one place in a plan for both) it gets
  // memory of its own, so that a call has the bits that it has elsewhere.
  Tensor apart(nullptr);
  Tensor* const target = kernels::ResultBeside(out, {&hidden, &mask}, &apart, hidden.dtype(), {batch, seq, width}, dev, dev_id, "BERTEmbedding/Reshape");
  void* const result = target->mutable_raw();
  float* const result32 = kernels::KeepsFp32Residual(*target) ? target->EnsureShadow()->mutableData<float>() : nullptr;
  if (reinterpret_cast<uintptr_t>(result) % 16 != 0) return false;
  first.exchange().Use(bytes, dev, dev_id, [&](void* memory, int turn) {
    TT_DEVICE_CALL(ttmi_encoder_chain(parameters.data(), hidden.raw(), input32, additive, result, result32, memory, turn, count, batch, seq, heads, width,
                                      ffn, 1e-12f, dt, 0, 0, Stream()));
  });
  if (target != out) *out = std::move(apart);
  return true;
}

}  // namespace layers
}  // namespace turbo_transformers
