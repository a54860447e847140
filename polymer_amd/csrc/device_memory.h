// device_memory.h -- device allocations of the library (polyeri.hip).  Every
// one goes through these functions, so that memory which the work pool keeps
// idle is never the reason why one fails.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

// hipMalloc on the current device; where it fails, once more after the
// device's idle work buffers have been given back.
hipError_t polyeri_device_malloc(void** p, size_t bytes);
// Work buffers kept between calls (work_pool.h): a block of the current
// device, and its return once no stream uses it.
int polyeri_work_get(void** p, size_t bytes);
void polyeri_work_put(void* p);
