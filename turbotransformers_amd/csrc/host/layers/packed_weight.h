// The MFMA GEMM kernels want every weight K-contiguous, i.e. [out, in] ("trans" layout),
// while the reference API hands layers [in, out] matrices unless is_trans_weight is set.
// PackedWeight produces the [out, in] form once, on the first call that needs it, and
// afterwards only returns the pointer.  fp32 weights get what ttmi_split_weights adds.
#pragma once

#include <initializer_list>
#include <mutex>

#include "core/tensor.h"
#include "ttmi.h"

namespace turbo_transformers {
namespace layers {

// A weight as the products take it.
struct WeightRef {
  const void* data;
  int dtype;
  // ... beside an input of the given type
  int DTypeFor(int input) const { return input == TTMI_F32 && dtype == TTMI_F32_PACKED ? TTMI_F32_PACKED : input; }
};

// The bytes of a weight that a product reads.
struct WeightRange {
  const void* data = nullptr;
  int64_t bytes = 0;
};

class PackedWeight {
 public:
  // W as [N, K]; `w` is [K, N] when !is_trans_weight, [N, K] (used as it is) otherwise.
  WeightRef Get(const core::Tensor& w, bool is_trans_weight) const;
  // [w; v] as [2 N, K] for two weights [K, N] that are applied to the same rows.
  WeightRef GetPair(const core::Tensor& w, const core::Tensor& v) const;
  // What products of `w` [K, N] read; empty before the first Get.
  WeightRange Range(const core::Tensor& w) const;
  // Output width N of `w` under the given layout.
  static int64_t OutDim(const core::Tensor& w, bool is_trans_weight) { return is_trans_weight ? w.shape(0) : w.shape(1); }
  static int64_t InDim(const core::Tensor& w, bool is_trans_weight) { return is_trans_weight ? w.shape(1) : w.shape(0); }

 private:
  WeightRef Pack(std::initializer_list<const core::Tensor*> parts) const;  // [K, N] each, one below the other
  mutable std::mutex mutex_;  // two threads may make the first call of one layer object together
  mutable core::Tensor packed_;
  mutable const void* source_ = nullptr;
  mutable const void* second_source_ = nullptr;
  mutable int dtype_ = 0;
};

}  // namespace layers
}  // namespace turbo_transformers
