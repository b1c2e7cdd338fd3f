// Device allocations.
#pragma once

#include <stddef.h>

namespace lgx {

// bytes (at least one) of device memory, uninitialised.  When none is left,
// every device scene's spare blocks (device.h) are given back first; throws
// if that is not enough.  Freed with hipFree.
void* device_alloc(size_t bytes);

} // namespace lgx
