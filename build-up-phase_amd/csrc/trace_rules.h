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

// ---- launches ---------------------------------------------------------------------------------------------------

// A CU's LDS, and the unit it is given out in: 128 of them, so that 16 blocks of up to 10,240 B fit.
constexpr uint32_t kCuLdsBytes = 160u * 1024u;
constexpr uint32_t kLdsUnit = 1280u;
constexpr uint32_t kCuSimds = 4;

// LDS of the traversal kernels beside the stack and the rays, but for their lean form: the octant table of a block, and
// 512 B a wave for the triangle tasks (8 B of each lane).
constexpr uint32_t kOctTableBytes = 2048;
constexpr uint32_t kTaskLaneBytes = 8;

// What a launch of the persistent traversal kernels asks for.
struct TraceShape {
    uint32_t block_size;
    uint32_t blocks_per_cu;
    uint32_t grid;            // blocks: blocks_per_cu on every CU
    uint32_t waves_per_simd;  // that the kernel variant's registers allow at least
    uint32_t lane_bytes;      // LDS of a lane: its stack entries, and its world ray where the kernel keeps it there
    uint32_t start_blocks;    // blocks of a CU that can start at once beside what runs already
};

// Blocks of a launch that a CU holds at once.
RTX_RULE uint32_t resident_blocks(const TraceShape& s, uint32_t lds_bytes) {
    const uint32_t units = (lds_bytes + kLdsUnit - 1u) / kLdsUnit;
    const uint32_t by_lds = units ? kCuLdsBytes / kLdsUnit / units : s.blocks_per_cu;
    const uint32_t by_waves = kCuSimds * s.waves_per_simd / (s.block_size / 64u);
    const uint32_t most = by_lds < by_waves ? by_lds : by_waves;
    return s.blocks_per_cu < most ? s.blocks_per_cu : most;
}

// Ray ids per chunk of a launch of n rays on `waves` waves, of which first_waves own their first chunk.  Automatic: at
// most one ray per lane of those is spread over all of them (a wave of few rays diverges less, and the launch lasts as
// long as its slowest wave); otherwise 64, or for single rays 256 when every wave gets at least 8 chunks.  Fetches count
// where rays are cheap: a 7680x4320 film of two quads 437 us with 64, 391 us with 256, 16.7M rays that all miss 239 and
// 218 us; where they are not, 256 is even (16.7M rays over 20M triangles) or up to 3% slower (3M to 16M any-hit rays
// 1%, camera rays that all enter small meshes 865 and 893 us).  Whole paths are too uneven for that: 4 samples of the
// 1080p Cornell box 13.6 ms with 256, 13.0 ms with 64.
RTX_RULE uint32_t rays_per_chunk(uint32_t configured, uint32_t n, uint32_t waves, uint32_t first_waves, bool paths) {
    if (configured >= 64u) return configured;
    if (first_waves && (uint64_t)n <= (uint64_t)first_waves * 64u)
        return n ? (n + first_waves - 1u) / first_waves : 1u;
    return !paths && (uint64_t)n >= (uint64_t)waves * 64u * 8u ? 256u : 64u;
}

struct TracePlan {
    uint32_t grid;         // blocks launched
    uint32_t lds;          // dynamic LDS of a block
    uint32_t first_waves;  // waves whose first chunk is their own
    bool lean;             // the kernel form without the octant table and the tasks in LDS
    bool queues;           // rays are left for the queues
};

// The plan of a launch of n rays (0: the count is on the device).
//   lean         where the table and the tasks would cost a CU a block, and for five waves per SIMD, whose shapes fill
//                the LDS with their stacks.  With both in all launches 720p path tracing took 10.1 ms on 20 blocks of
//                one wave per CU (12 or 13 of them fitted) and 7.9 ms on 16 with 16 stack entries each; lean 7.2 and
//                6.3 ms.  Where they fit (256 x 4), the table's byte read instead of 16 vector instructions per node
//                step and the tasks through LDS instead of five permutes are 2% and 1% faster
//   first_waves  only waves that start at once own rays.  The blocks beyond start as others retire, when the queues
//                have run dry, and would only then begin with theirs: on 32 blocks of 256 per CU, of which 4 or 5
//                start, 4M incoherent rays took 1.83 ms and 720p path tracing 9.3 ms, now 1.22 and 7.2 ms
//   grid         no more waves than rays
RTX_RULE TracePlan plan_trace(const TraceShape& s, uint32_t ray_chunk, uint32_t n, bool paths) {
    TracePlan p;
    const uint32_t waves_block = s.block_size / 64u;
    p.lds = s.lane_bytes * s.block_size;
    const uint32_t tasks = kTaskLaneBytes * s.block_size;
    uint32_t resident = resident_blocks(s, p.lds);
    p.lean = s.waves_per_simd >= 5u || resident_blocks(s, p.lds + tasks + kOctTableBytes) < resident;
    if (!p.lean) p.lds += tasks;
    p.grid = s.grid;
    if (n && ray_chunk < 64u && (n - 1u) / waves_block < p.grid) p.grid = (n - 1u) / waves_block + 1u;
    if (s.start_blocks < resident) resident = s.start_blocks;
    const uint32_t at_once = s.grid / s.blocks_per_cu * resident;
    p.first_waves = (at_once < p.grid ? at_once : p.grid) * waves_block;
    const uint64_t chunk = rays_per_chunk(ray_chunk, n, p.grid * waves_block, p.first_waves, paths);
    p.queues = !n || chunk * p.first_waves < n;
    return p;
}

}  // namespace rtx
