// sort.h — stable radix sort of (key, uint32 value) pairs on a HIP stream.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rtx {

// Scratch bytes needed to sort n pairs with key_bytes-byte keys (4 or 8).
uint64_t sort_scratch_bytes(uint32_t n, int key_bytes);
// How many of them, at the end, are there for the look-back words of tiles smaller than 4,096 keys.
uint64_t sort_small_tile_bytes(uint32_t n, int key_bytes);

// Sort keys[0..n) ascending, carrying vals; input values are ignored and replaced by the original indices
// (the sorted permutation).  Stable.  err_flags receives kErrSortTimeout if a look-back spin ran out.
hipError_t sort_pairs_u32(uint32_t* keys, uint32_t* vals, uint32_t n, void* scratch, uint32_t* err_flags,
                          hipStream_t stream);
// key_bits: the keys' bits above are zero.
hipError_t sort_pairs_u64(uint64_t* keys, uint32_t* vals, uint32_t n, void* scratch, uint32_t* err_flags,
                          hipStream_t stream, int key_bits = 64);

}  // namespace rtx
