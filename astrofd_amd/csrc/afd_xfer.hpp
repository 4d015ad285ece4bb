// afd_xfer.hpp -- host <-> device copies of whole arrays through pinned staging and a few host threads.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace afd {

// One reference per context: the staging memory and the threads are made by the first large copy,
// shared by every context of the process (any device), and given back with the last reference.
void xfer_retain();
void xfer_release();

// A context's own pinned block of PIN_BLOCK bytes (null: none to be had, or none free and `lock` false).
// Closed contexts leave up to two for the next ones (locking and unlocking one takes 30 us, which a caller
// that opens contexts beside one it holds would pay each time); the last reference gives them back.
constexpr size_t PIN_BYTES = size_t(512) << 10, PIN_BLOCK = 2 * PIN_BYTES + 4096;
char *xfer_pin_get(bool lock);
void xfer_pin_put(char *block);

// Copy `bytes` between pageable host memory and device memory in stream order on `s` (a stream of the
// current device) and wait for it: on return the host memory may be read or reused.  wait false: the
// host memory is left alone until the caller has waited for the stream, so the copy need not.
hipError_t xfer_d2h(void *host, const void *dev, size_t bytes, hipStream_t s, bool wait = true);
hipError_t xfer_h2d(void *dev, const void *host, size_t bytes, hipStream_t s, bool wait = true);

}  // namespace afd
