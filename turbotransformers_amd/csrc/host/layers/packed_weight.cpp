#include "layers/packed_weight.h"

#include "core/device_context.h"
#include "layers/kernels.h"
#include "ttmi.h"

namespace turbo_transformers {
namespace layers {

WeightRef PackedWeight::Pack(std::initializer_list<const core::Tensor*> parts) const {
  const core::Tensor& w = **parts.begin();
  const int64_t K = w.shape(0), N = w.shape(1), rows = N * (int64_t)parts.size();
  const int dtype = core::ToDeviceDType(w.dtype());
  void* stream = core::DeviceContext::GetInstance().stream();
  const bool split = dtype == TTMI_F32 && K > 0 && K % TTMI_PACKED_WEIGHT_K == 0;
  if (split) packed_.ReshapeAs(w.dtype(), {TTMI_PACKED_WEIGHT_FLOATS(rows, K)}, w.device_type(), w.device_id(), "PackedWeight");
  else packed_.ReshapeAs(w.dtype(), {rows, K}, w.device_type(), w.device_id(), "PackedWeight");
  char* at = static_cast<char*>(packed_.mutable_raw());
  for (const core::Tensor* part : parts) {
    TT_DEVICE_CALL(ttmi_transpose_2d(part->raw(), at, K, N, dtype, stream));
    at += (size_t)(K * N) * w.element_size();
  }
  if (split) TT_DEVICE_CALL(ttmi_split_weights(packed_.mutable_raw(), rows, K, stream));
  dtype_ = split ? TTMI_F32_PACKED : dtype;
  return {packed_.raw(), dtype_};
}

WeightRef PackedWeight::Get(const core::Tensor& w, bool is_trans_weight) const {
  TT_ENFORCE_EQ(w.n_dim(), (size_t)2, "weights must be 2-D");
  kernels::RequireGpu(w, "weight");
  if (is_trans_weight) return {w.raw(), core::ToDeviceDType(w.dtype())};
  std::lock_guard<std::mutex> lock(mutex_);
  if (source_ == w.raw() && !packed_.is_null()) return {packed_.raw(), dtype_};
  const WeightRef ref = Pack({&w});
  source_ = w.raw();
  return ref;
}

WeightRange PackedWeight::Range(const core::Tensor& w) const {
  std::lock_guard<std::mutex> lock(mutex_);
  if (source_ != w.raw() || packed_.is_null()) return {};
  const int64_t bytes = w.numel() * (int64_t)w.element_size();
  // (the halves of an fp32 weight lie behind its values, which are read for tiles outside their window only)
  return {static_cast<const char*>(packed_.raw()) + (dtype_ == TTMI_F32_PACKED ? bytes : 0), bytes};
}

WeightRef PackedWeight::GetPair(const core::Tensor& w, const core::Tensor& v) const {
  TT_ENFORCE(w.n_dim() == 2 && v.n_dim() == 2 && w.shape(0) == v.shape(0) && w.shape(1) == v.shape(1), "a pair of weights has one shape");
  TT_ENFORCE(core::SameDataType(w.dtype(), v.dtype()), "a pair of weights has one element type");
  kernels::RequireGpu(w, "weight");
  kernels::RequireGpu(v, "weight");
  std::lock_guard<std::mutex> lock(mutex_);
  if (source_ == w.raw() && second_source_ == v.raw() && !packed_.is_null()) return {packed_.raw(), dtype_};
  const WeightRef ref = Pack({&w, &v});
  source_ = w.raw();
  second_source_ = v.raw();
  return ref;
}

}  // namespace layers
}  // namespace turbo_transformers
