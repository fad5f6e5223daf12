// The memory through which the steps of a call that runs as one launch pass their rows (ttmi_encoder_chain, ttmi_decoder_attention,
// ttmi_decoder_feed_forward): two of its parts take turns from call to call of the layer that holds it, two from one recorded call to the next, and all of it goes
// with the layer.  Calls of another size have memory of their own, so that a recorded call, replayed between them, writes nothing that they count on, and its
// memory stays where it is.  (The sizes do not depend on the rows: there is one, but for encoders, which may be run by the stack and by the layer.)
#pragma once

#include <list>
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
    Memory* m = nullptr;
    for (Memory& known : memory_)
      if (known.bytes == bytes && known.device_id == device_id) m = &known;
    if (m == nullptr) {
      memory_.emplace_back();
      m = &memory_.back();
      m->bytes = bytes, m->device_id = device_id;
    }
    float* const memory = m->words.Reshape<float>({bytes / 4}, device, device_id, "chain/exchange");
    int capturing = 0;
    TT_DEVICE_CALL(ttmi_stream_capturing(stream, &capturing));
    if (capturing) {  // replayed in an order that is not known here: such launches count themselves
      if (!m->prepared) TT_DEVICE_CALL(ttmi_chain_prepare(memory, bytes, stream));  // (recorded too: each replay finds all parts as they should be)
      launch(memory, 2);
      return;
    }
    if (!m->prepared) TT_DEVICE_CALL(ttmi_chain_prepare(memory, bytes, stream));
    m->prepared = false;  // (until the call is queued)
    launch(memory, m->turn);
    m->turn = 1 - m->turn;
    m->prepared = true;
  }

 private:
  struct Memory {
    core::Tensor words{nullptr};
    int64_t bytes = 0;
    int device_id = 0, turn = 0;
    bool prepared = false;
  };
  std::mutex mutex_;
  std::list<Memory> memory_;
};

}  // namespace layers
}  // namespace turbo_transformers
