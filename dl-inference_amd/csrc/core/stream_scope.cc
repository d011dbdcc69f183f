// The stream of the running graph (StreamScope, include/dli/tensor.h) and the caching allocator.
#include <ATen/ATen.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>

#include <stdexcept>
#include <string>

#include "dli/tensor.h"
#include "dli_hip.h"

namespace dli {
namespace {

struct Current {
  void* stream = nullptr;
  bool active = false;
};
thread_local Current current;

// The scope's stream is not the one that orders the allocator's reuse on this device.
bool foreign(int device_id) {
  if (!current.active) return false;
  const auto device = static_cast<c10::DeviceIndex>(device_id);
  return static_cast<void*>(c10::hip::getCurrentHIPStream(device).stream()) != current.stream;
}

bool capturing() {
  int captured = 0;
  if (dli_hip_stream_is_capturing(current.stream, &captured) != 0)
    throw std::runtime_error(std::string("stream capture state: ") + dli_hip_last_error());
  return captured != 0;
}

}  // namespace

StreamScope::StreamScope(void* stream) : previous_(current.stream), active_(current.active) {
  current = {stream, true};
}

StreamScope::~StreamScope() { current = {previous_, active_}; }

bool StreamScope::allowsScratch(int device_id) { return !foreign(device_id) || !capturing(); }

void StreamScope::use(const at::Tensor& tensor, int device_id) {
  if (!foreign(device_id) || capturing()) return;
  c10::hip::HIPCachingAllocator::recordStream(
      tensor.storage().data_ptr(),
      c10::hip::getStreamFromExternal(static_cast<hipStream_t>(current.stream),
                                      static_cast<c10::DeviceIndex>(device_id)));
}

}  // namespace dli
