// The memory through which the steps of a call that runs as one launch pass their rows (ttmi_encoder_chain, ttmi_decoder_attention,
// ttmi_decoder_feed_forward): its parts take turns from call to call of the layer that holds it, and go with it.
#pragma once

#include <mutex>

#include "core/device_context.h"
#include "core/tensor.h"
#include "ttmi.h"

namespace turbo_transformers {
namespace layers {

class ExchangeMemory {
 public:
  // launch(memory, turn) queues one call
  template <typename Launch>
  void Use(int64_t bytes, DLDeviceType device, int device_id, const Launch& launch) {
    std::lock_guard<std::mutex> lock(mutex_);
    void* const stream = core::DeviceContext::GetInstance().stream();
    float* const memory = memory_.Reshape<float>({bytes / 4}, device, device_id, "chain/exchange");
    int capturing = 0;
    TT_DEVICE_CALL(ttmi_stream_capturing(stream, &capturing));
    if (capturing) {  // replayed in an order that is not known here
      launch(memory, 2);
      return;
    }
    if (prepared_ != bytes) TT_DEVICE_CALL(ttmi_chain_prepare(memory, bytes, stream));
    prepared_ = 0;  // (until the call is queued)
    launch(memory, turn_);
    turn_ = 1 - turn_;
    prepared_ = bytes;
  }

 private:
  std::mutex mutex_;
  core::Tensor memory_{nullptr};
  int64_t prepared_ = 0;  // bytes
  int turn_ = 0;
};

}  // namespace layers
}  // namespace turbo_transformers
