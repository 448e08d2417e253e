// trace_rules.h — rules of the traversal that need no GPU: plain functions of sizes, the same on host and device.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define RTX_RULE __host__ __device__ __forceinline__
#else
#define RTX_RULE inline
#endif

namespace rtx {

// Whether a lane whose stack pointer is sp takes an entry from a stack of `entries`.  Not from an empty stack, and not
// after pushes past its end, which are dropped but counted (so that the step's overflow check sees them): entry sp - 1
// is then no entry of this lane, and lies beyond its part of the spill area.
RTX_RULE bool pops_entry(uint32_t sp, uint32_t entries) { return sp - 1u < entries; }

}  // namespace rtx
