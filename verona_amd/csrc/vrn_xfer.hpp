// vrn_xfer.hpp -- copies between pageable host arrays and the device.
//
// The runtime moves pageable memory at 27 to 29 GB/s to the device and 17 GB/s
// from it (one thread staging), pinned memory at 57 GB/s both ways.  Large copies
// therefore go through pinned staging slots here, filled and emptied by a few
// threads while the link moves the neighbouring slots; small ones, and
// memory that the runtime knows, go to the runtime directly.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace vrn_xfer {

// Every handle that copies holds the staging memory: it is allocated by the
// first large copy and freed with the last handle.
void retain();
void release();
struct Hold {
    Hold() { retain(); }
    ~Hold() { release(); }
    Hold(const Hold &) = delete;
    Hold &operator=(const Hold &) = delete;
};

// Copy n bytes in the order of stream s.  h2d returns once the host array has
// been read (a large one: also once it has arrived), d2h once it has been
// written.
hipError_t h2d(void *dev, const void *host, size_t n, hipStream_t s);
hipError_t d2h(void *host, const void *dev, size_t n, hipStream_t s);

}  // namespace vrn_xfer
