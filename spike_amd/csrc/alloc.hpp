// alloc.hpp -- device memory, for every translation unit of the library.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace spk {

// hipMalloc; when memory is short, once more after the idle memory of closed networks has gone
// back to the device (a caller finds the memory that it would find without any kept).  A failure
// leaves nothing in the thread's last error: the runtime keeps a failed call's error past the
// calls that succeed after it, and the check behind the next launch would report it.
hipError_t device_malloc(void** p, size_t bytes);

}  // namespace spk

// For tests of what happens when memory runs out: `pass` further requests are served, then
// `count` are refused (a request that is tried twice counts twice).
extern "C" void spk_refuse_allocations(int pass, int count);
