// Fixed device scratch of the no-allocation entry point (noalloc.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace moert {

// Bytes of the scratch: a 256-byte header (unused), then the split partials of up to 64 query heads x 64 splits x 66
// floats.
constexpr size_t kNoallocHeader = 256;
constexpr size_t kNoallocScratchBytes = kNoallocHeader + (size_t)64 * 64 * 66 * 4;  // 1,081,600

// The scratch's device address on the current device (taken once per device with hipGetSymbolAddress); null on
// failure with the error in *err.
void* noalloc_scratch(hipError_t* err);

}  // namespace moert
