// sort.hip — stable onesweep LSD radix sort of (key, uint32 value) pairs for gfx950.
//
// Method: Adinets & Merrill 2022, "Onesweep: A Faster Least Significant Digit Radix Sort for GPUs".
//   1. one pass over the keys builds the 256-bin histogram of every 8-bit digit (LDS-privatised);
//   2. one 256-thread block turns the histograms into digit start offsets;
//   3. per digit pass, each block takes a tile of keys (tile id from an atomic ticket, so every tile it
//      waits for belongs to a block that is already running), ranks its keys stably in LDS using 64-lane
//      ballots, publishes its per-digit counts and resolves its global offsets with decoupled look-back,
//      stages the tile in LDS in digit order and writes it out in runs.
// Up to one tile of keys is sorted by one block in one launch, the digit passes going back and forth in LDS.
// The look-back spin is bounded: past the limit the block raises kErrSortTimeout and finishes.
#include "rtx_internal.h"
#include "sort.h"

namespace rtx {

namespace {

constexpr int kSortBlock = 256;
// Keys per thread: 16 (4,096-key tiles); below kLargeFrom keys 4 (1,024-key tiles), so that more blocks share a pass.
// A pass with 4 and with 16: 32,768 keys 8.2 and 13 us, 65,536 9.6 and 13.5, 131,072 11.6 and 14.4, 262,144 15.1 and
// 15.7, 655K 28 and 20 (the look-back of small tiles goes over four times as many).  They cross near 270,000 keys; the
// line below gives away at most 3 us a pass between.
constexpr int kItemsLarge = 16, kItemsSmall = 4;
constexpr uint32_t kLargeFrom = 1u << 17;
constexpr uint32_t kOneBlock = kSortBlock * kItemsLarge;
uint32_t tile_keys(uint32_t n) { return (uint32_t)kSortBlock * (uint32_t)(n >= kLargeFrom ? kItemsLarge : kItemsSmall); }
constexpr int kRadix = 256;
constexpr uint32_t kFlagAgg = 1u << 30;
constexpr uint32_t kFlagInc = 2u << 30;
constexpr uint32_t kValMask = (1u << 30) - 1u;
constexpr int kSpinLimit = 1 << 22;

template <typename K>
__global__ __launch_bounds__(256) void hist_kernel(const K* __restrict__ keys, uint32_t n, int passes,
                                                   uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[8][kRadix];
    for (int i = threadIdx.x; i < 8 * kRadix; i += blockDim.x) (&h[0][0])[i] = 0;
    __syncthreads();
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        K k = keys[i];
        for (int p = 0; p < passes; ++p) atomicAdd(&h[p][(uint32_t)(k >> (8 * p)) & 255u], 1u);
    }
    __syncthreads();
    for (int p = 0; p < passes; ++p)
        for (int d = threadIdx.x; d < kRadix; d += blockDim.x)
            if (h[p][d]) atomicAdd(&hist[p * kRadix + d], h[p][d]);
}

__global__ __launch_bounds__(256) void scan_hist_kernel(const uint32_t* __restrict__ hist, int passes,
                                                        uint32_t* __restrict__ start) {
    __shared__ uint32_t s[kRadix];
    int t = threadIdx.x;
    for (int p = 0; p < passes; ++p) {
        uint32_t c = hist[p * kRadix + t];
        s[t] = c;
        __syncthreads();
        for (int off = 1; off < kRadix; off <<= 1) {
            uint32_t v = t >= off ? s[t - off] : 0u;
            __syncthreads();
            s[t] += v;
            __syncthreads();
        }
        start[p * kRadix + t] = s[t] - c;
        __syncthreads();
    }
}

__global__ void fill_u32_kernel(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__device__ __forceinline__ uint32_t status_load(uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void status_store(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Ranks of a tile's keys by one digit.  A wave takes ITEMS x 64 consecutive keys, 64 at a time, and counts its digits in
// its own row of LDS: the lanes of one digit find each other by ballots, take their places after the wave's count so far,
// and the first of them moves the count on.  (A row of counts shared by the waves, with two barriers per 64 keys of each,
// took twice as long.)
struct RankLds {
    uint32_t cnt[4][kRadix];  // counts of each wave, then its first place
    uint32_t excl[kRadix];    // digits' first places in the tile
    uint32_t sum[4];
};

// Returns the count of digit threadIdx.x in the tile; rank[i] is the place among the tile's keys of that digit.
template <typename K, int ITEMS>
__device__ __forceinline__ uint32_t rank_tile(RankLds& R, const K* key, const bool* valid, int shift, uint32_t* rank) {
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int k = 0; k < 4; ++k) R.cnt[k][t] = 0;
    __syncthreads();
    volatile uint32_t* const mine = R.cnt[w];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t d = (uint32_t)(key[i] >> shift) & 255u;
        uint64_t peers = __ballot(valid[i]);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t bits = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bits : ~bits;
        }
        const uint32_t lr = (uint32_t)__popcll(peers & lt_mask);
        const uint32_t before = mine[d];
        rank[i] = before + lr;
        if (valid[i] && lr == 0) mine[d] = before + (uint32_t)__popcll(peers);
    }
    __syncthreads();
    // digit t: the waves' first places, and the exclusive prefix over the digits
    const uint32_t c0 = R.cnt[0][t], c1 = R.cnt[1][t], c2 = R.cnt[2][t], c3 = R.cnt[3][t];
    const uint32_t count = c0 + c1 + c2 + c3;
    R.cnt[0][t] = 0;
    R.cnt[1][t] = c0;
    R.cnt[2][t] = c0 + c1;
    R.cnt[3][t] = c0 + c1 + c2;
    uint32_t incl = count;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(incl, off);
        if (lane >= off) incl += v;
    }
    if (lane == 63) R.sum[w] = incl;
    __syncthreads();
    uint32_t base = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) base += k < w ? R.sum[k] : 0u;
    R.excl[t] = base + incl - count;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) rank[i] += R.cnt[w][(uint32_t)(key[i] >> shift) & 255u];
    __syncthreads();
    return count;
}

template <typename K, int ITEMS>
__global__ __launch_bounds__(kSortBlock) void onesweep_kernel(const K* __restrict__ keys_in,
                                                              const uint32_t* __restrict__ vals_in,
                                                              K* __restrict__ keys_out, uint32_t* __restrict__ vals_out,
                                                              uint32_t n, int shift,
                                                              const uint32_t* __restrict__ digit_start,
                                                              uint32_t* __restrict__ status,
                                                              uint32_t* __restrict__ tile_counter,
                                                              uint32_t* __restrict__ err_flags) {
    constexpr int kTile = kSortBlock * ITEMS;
    __shared__ uint32_t s_tile;
    __shared__ RankLds R;
    __shared__ uint32_t s_global[kRadix];
    __shared__ K s_keys[kTile];
    __shared__ uint32_t s_vals[kTile];

    const int t = threadIdx.x;
    if (t == 0) s_tile = atomicAdd(tile_counter, 1u);
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint64_t tile_start = (uint64_t)tile * kTile;
    const uint64_t first = tile_start + (uint64_t)(t >> 6) * (64 * ITEMS) + (t & 63);

    K key[ITEMS];
    uint32_t val[ITEMS];
    uint32_t rank[ITEMS];
    bool valid[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint64_t idx = first + 64u * i;
        valid[i] = idx < n;
        key[i] = valid[i] ? keys_in[idx] : (K)0;
        val[i] = valid[i] ? (vals_in ? vals_in[idx] : (uint32_t)idx) : 0u;
    }
    const uint32_t count = rank_tile<K, ITEMS>(R, key, valid, shift, rank);

    // decoupled look-back for digit t
    {
        uint32_t* st = status + (uint64_t)tile * kRadix + t;
        uint32_t excl = 0;
        if (tile == 0) {
            status_store(st, kFlagInc | count);
        } else {
            status_store(st, kFlagAgg | count);
            int64_t p = (int64_t)tile - 1;
            int spins = 0;
            while (p >= 0) {
                uint32_t v = status_load(status + (uint64_t)p * kRadix + t);
                uint32_t f = v & ~kValMask;
                if (f == 0u) {
                    if (++spins > kSpinLimit) {
                        atomicOr(err_flags, kErrSortTimeout);
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                    continue;
                }
                excl += v & kValMask;
                if (f == kFlagInc) break;
                --p;
            }
            status_store(st, kFlagInc | ((excl + count) & kValMask));
        }
        s_global[t] = digit_start[t] + excl;
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (valid[i]) {
            const uint32_t pos = R.excl[(uint32_t)(key[i] >> shift) & 255u] + rank[i];
            s_keys[pos] = key[i];
            s_vals[pos] = val[i];
        }
    }
    __syncthreads();
    const uint64_t rem = (uint64_t)n - tile_start;
    const uint32_t tile_n = rem < (uint64_t)kTile ? (uint32_t)rem : (uint32_t)kTile;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        uint32_t pos = (uint32_t)i * kSortBlock + t;
        if (pos < tile_n) {
            K k = s_keys[pos];
            uint32_t d = (uint32_t)(k >> shift) & 255u;
            uint32_t o = s_global[d] + (pos - R.excl[d]);
            if (o < n) {  // only false after a look-back timeout (reported through err_flags)
                keys_out[o] = k;
                vals_out[o] = s_vals[pos];
            }
        }
    }
}

// At most one tile of keys: every pass in one block.
template <typename K, int ITEMS>
__global__ __launch_bounds__(kSortBlock) void one_block_sort_kernel(K* __restrict__ keys, uint32_t* __restrict__ vals,
                                                                    uint32_t n, int passes) {
    constexpr int kTile = kSortBlock * ITEMS;
    __shared__ RankLds R;
    __shared__ K s_keys[kTile];
    __shared__ uint32_t s_vals[kTile];
    const int t = threadIdx.x;
    const uint32_t first = (uint32_t)(t >> 6) * (64 * ITEMS) + (t & 63);
    K key[ITEMS];
    uint32_t val[ITEMS], rank[ITEMS];
    bool valid[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        val[i] = first + 64u * i;
        valid[i] = val[i] < n;
        key[i] = valid[i] ? keys[val[i]] : (K)0;
    }
    for (int p = 0; p < passes; ++p) {
        rank_tile<K, ITEMS>(R, key, valid, 8 * p, rank);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (valid[i]) {
                const uint32_t pos = R.excl[(uint32_t)(key[i] >> (8 * p)) & 255u] + rank[i];
                s_keys[pos] = key[i];
                s_vals[pos] = val[i];
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (valid[i]) {
                key[i] = s_keys[first + 64u * i];
                val[i] = s_vals[first + 64u * i];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (valid[i]) {
            keys[first + 64u * i] = key[i];
            vals[first + 64u * i] = val[i];
        }
    }
}

}  // namespace

uint64_t sort_scratch_bytes(uint32_t n, int key_bytes) {
    uint64_t tiles = ((uint64_t)n + tile_keys(n) - 1) / tile_keys(n);
    int passes = key_bytes;  // 8-bit digits
    uint64_t b = 0;
    b += align_up((uint64_t)n * key_bytes, 256);       // alternate keys
    b += align_up((uint64_t)n * 4, 256);               // alternate values
    b += align_up((uint64_t)passes * kRadix * 4, 256); // histograms
    b += align_up((uint64_t)passes * kRadix * 4, 256); // digit starts
    b += align_up((uint64_t)passes * 4, 256);          // tile counters
    b += align_up((uint64_t)passes * tiles * kRadix * 4, 256);  // look-back status
    return b;
}

uint64_t sort_small_tile_bytes(uint32_t n, int key_bytes) {
    constexpr uint64_t large = (uint64_t)kSortBlock * kItemsLarge;
    const uint64_t tiles = ((uint64_t)n + tile_keys(n) - 1) / tile_keys(n), least = (n + large - 1) / large;
    return (uint64_t)key_bytes * (tiles - least) * kRadix * 4;
}

template <typename K>
static hipError_t sort_pairs_impl(K* keys, uint32_t* vals, uint32_t n, int passes, void* scratch,
                                  uint32_t* err_flags, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    if (n <= kOneBlock) {
        if (n <= kSortBlock)
            one_block_sort_kernel<K, 1><<<1, kSortBlock, 0, stream>>>(keys, vals, n, passes);
        else if (n <= kSortBlock * kItemsSmall)
            one_block_sort_kernel<K, kItemsSmall><<<1, kSortBlock, 0, stream>>>(keys, vals, n, passes);
        else
            one_block_sort_kernel<K, kItemsLarge><<<1, kSortBlock, 0, stream>>>(keys, vals, n, passes);
        return hipGetLastError();
    }
    const bool large = n >= kLargeFrom;
    uint64_t tiles = ((uint64_t)n + tile_keys(n) - 1) / tile_keys(n);
    uint8_t* p = (uint8_t*)scratch;
    K* keys_alt = (K*)p;
    p += align_up((uint64_t)n * sizeof(K), 256);
    uint32_t* vals_alt = (uint32_t*)p;
    p += align_up((uint64_t)n * 4, 256);
    uint32_t* hist = (uint32_t*)p;
    p += align_up((uint64_t)sizeof(K) * kRadix * 4, 256);
    uint32_t* start = (uint32_t*)p;
    p += align_up((uint64_t)sizeof(K) * kRadix * 4, 256);
    uint32_t* counters = (uint32_t*)p;
    p += align_up((uint64_t)sizeof(K) * 4, 256);
    uint32_t* status = (uint32_t*)p;
    // hist, start, counters and status are contiguous: clear them with one fill
    uint64_t clear_words = ((uint8_t*)status - (uint8_t*)hist) / 4 + (uint64_t)passes * tiles * kRadix;
    fill_u32_kernel<<<1024, 256, 0, stream>>>(hist, clear_words, 0u);
    int hist_blocks = (int)std::min<uint64_t>(1024, (n + 4095) / 4096);
    hist_kernel<K><<<hist_blocks, 256, 0, stream>>>(keys, n, passes, hist);
    scan_hist_kernel<<<1, 256, 0, stream>>>(hist, passes, start);
    K* kin = keys;
    K* kout = keys_alt;
    uint32_t* vin = nullptr;
    uint32_t* vout = vals_alt;
    for (int pass = 0; pass < passes; ++pass) {
        uint32_t* st = status + (uint64_t)pass * tiles * kRadix;
        if (large)
            onesweep_kernel<K, kItemsLarge><<<(unsigned)tiles, kSortBlock, 0, stream>>>(
                kin, vin, kout, vout, n, 8 * pass, start + pass * kRadix, st, counters + pass, err_flags);
        else
            onesweep_kernel<K, kItemsSmall><<<(unsigned)tiles, kSortBlock, 0, stream>>>(
                kin, vin, kout, vout, n, 8 * pass, start + pass * kRadix, st, counters + pass, err_flags);
        std::swap(kin, kout);
        vin = vout;
        vout = (vout == vals_alt) ? vals : vals_alt;
    }
    // an even number of passes leaves keys in `keys` and values in `vals`
    return hipGetLastError();
}

hipError_t sort_pairs_u32(uint32_t* keys, uint32_t* vals, uint32_t n, void* scratch, uint32_t* err_flags,
                          hipStream_t stream) {
    return sort_pairs_impl<uint32_t>(keys, vals, n, 4, scratch, err_flags, stream);
}

hipError_t sort_pairs_u64(uint64_t* keys, uint32_t* vals, uint32_t n, void* scratch, uint32_t* err_flags,
                          hipStream_t stream, int key_bits) {
    // an even number of passes over the digits that keys of key_bits bits have
    return sort_pairs_impl<uint64_t>(keys, vals, n, (key_bits + 15) / 16 * 2, scratch, err_flags, stream);
}

}  // namespace rtx
