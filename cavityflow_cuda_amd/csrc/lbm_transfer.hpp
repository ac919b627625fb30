// Copies between device and host memory (lbm_transfer.cpp).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace lbm {

struct Segment {
    void* host;
    void* device;
    size_t bytes;
};

// Copies the segments (at least one) on the stream. Large copies of pageable
// memory go through pinned buffers and several threads. To the host it returns
// with the copies complete; to the device the host memory may be reused once
// the stream has been waited for.
hipError_t transfer(const Segment* segments, size_t count, bool to_host, hipStream_t st);
inline hipError_t transfer(void* host, void* device, size_t bytes, bool to_host, hipStream_t st)
{
    const Segment s{host, device, bytes};
    return transfer(&s, 1, to_host, st);
}

// Whether transfer takes that way for so many bytes of this memory.
bool ring_pays(const void* host, size_t bytes, size_t segments);

}  // namespace lbm
