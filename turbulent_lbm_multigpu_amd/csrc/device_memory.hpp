// device_memory.hpp -- device allocation shared by the runtime and the server.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

// hipMalloc on the current device; where memory is short, the second buffers
// that solvers on this device keep for fused steps are freed first.
hipError_t lbm_device_malloc(void **p, size_t bytes);
