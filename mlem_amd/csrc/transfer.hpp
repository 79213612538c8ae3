// transfer.hpp — host memory (or a file) to the device through pinned buffers.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <functional>

namespace mlem {

// Copy `bytes` produced by produce(dst, offset, n) to device memory, in chunks
// through pinned buffers; several threads produce and enqueue chunks at a time
// where the range is large (produce is then called concurrently). Returns when
// the copy is complete; an exception of produce is thrown on.
using Produce = std::function<void(void* dst, uint64_t offset, uint64_t n)>;
void stream_to_device(void* dst, uint64_t bytes, int device, hipStream_t s,
                      const Produce& produce);

}  // namespace mlem
