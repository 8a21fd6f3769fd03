// device_memory.hpp -- device allocation shared by the runtime and the server.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

// hipMalloc on the current device; where memory is short, the second buffers
// that solvers on this device keep for fused steps are freed first.
hipError_t lbm_device_malloc(void **p, size_t bytes);

struct lbm_solver;

// rho[cells] and j[3][cells] of the whole domain as float, whatever the
// storage (rounded to the storage's compute type first), in one transfer.
int lbm_solver_moments_float(lbm_solver *s, float *rho, float *j);
