// A HIP runtime for host tests on a machine without a GPU: memory is host
// memory, copies are memcpy, a launch runs nothing and is written down.  The
// library's own objects are linked against it (tests/test_launches.py).
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <functional>
#include <string>

namespace fake {

struct Launch {
    std::string kernel;  // mangled name
    dim3 grid, block;
    void **args;  // the kernel's arguments, for the time of the call
};

// Called for each launch that is not refused.
extern std::function<void(const Launch &)> on_launch;
// Launches of kernels whose name holds this are refused (empty: none).
extern std::string refuse;
// hipFuncSetAttribute fails.
extern bool refuse_attributes;
// Device bytes there are (hipMalloc fails past them), in use, and the most so far.
extern size_t memory, used, peak;
// Bytes of the block that begins at p.
size_t size_of(const void *p);

}  // namespace fake
