// device_errors.h — the error flags that kernels raise, and what rtx_sync says of them.  Plain functions, no GPU.
#pragma once
#include <stdint.h>

#include "../../include/rtx.h"

namespace rtx {

// bits of DeviceState::error_flags
constexpr uint32_t kErrStackOverflow = 1u;    // a ray needed more stack entries than its launch has
constexpr uint32_t kErrSortTimeout = 2u;      // the sort's look-back wait ran out
constexpr uint32_t kErrBadAs = 4u;            // a traced structure is not one
constexpr uint32_t kErrCollapseTimeout = 8u;  // the collapse's wait for its queue ran out

struct DeviceError {
    int code;
    const char* text;
};

// The error of the first flag in this order; RTX_SUCCESS without one.
inline DeviceError device_error(uint32_t flags) {
    if (!flags) return {RTX_SUCCESS, ""};
    if (flags & kErrStackOverflow) return {RTX_ERROR_STACK_OVERFLOW, "traversal stack overflow"};
    if (flags & kErrSortTimeout) return {RTX_ERROR_DEVICE_LOST, "radix sort look-back timed out"};
    if (flags & kErrCollapseTimeout) return {RTX_ERROR_DEVICE_LOST, "the build's collapse queue timed out"};
    return {RTX_ERROR_INVALID_AS, "device reported an invalid acceleration structure"};
}

}  // namespace rtx
