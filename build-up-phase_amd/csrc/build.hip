// build.hip — LBVH builder for BLAS (triangles) and TLAS (instances) on gfx950.
//
// Replaces the driver build behind vkCmdBuildAccelerationStructuresKHR (main.cpp:808 for the BLAS,
// main.cpp:932 for the TLAS).  Pipeline, all on the context stream:
//   prep      one thread per primitive: fetch + transform triangle vertices (BLAS) or read the 64-B instance
//             record, invert its transform in FP64 and bound the BLAS root box in world space (TLAS);
//             writes a 64-B leaf record, the primitive box, and the centroid bounds (ordered-int atomics)
//   morton    30-bit (uint32) or 63-bit (uint64) Morton code of each box centroid
//   sort      stable onesweep radix sort of (code, primitive index)                         [sort.hip]
//   karras    binary radix tree over the sorted codes (Karras 2012), one thread per internal node
//   refit     bottom-up boxes and treelet refinement: subtrees of up to kSubtree primitives a wave each in LDS, then the
//             nodes above them, the second thread to reach a node merging its children (atomic arrival count)
//   collapse  top-down conversion to 8-wide nodes: each node adopts the children that the SAH-optimal choice gives it,
//             places them by octant, quantises their boxes to 8 bits per plane and gives them consecutive slots; the
//             nodes above the subtrees through a queue, then the subtrees a wave each.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "build.h"
#include "rtx_internal.h"
#include "sort.h"

namespace rtx {

namespace {

struct Box {
    float lo[3], hi[3];
};

__device__ __forceinline__ float box_area(const float* b) {
    float dx = b[3] - b[0], dy = b[4] - b[1], dz = b[5] - b[2];
    if (!(dx >= 0.0f) || !(dy >= 0.0f) || !(dz >= 0.0f)) return 0.0f;
    return dx * dy + dy * dz + dz * dx;
}

// Geometry transform at build time: x' = ((m00*x + m01*y) + m02*z) + m03 with separate roundings
// (this file is compiled with -ffp-contract=off).
__device__ __forceinline__ void xform_vertex(const float* m, const float* v, float* o) {
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        float a = m[4 * r + 0] * v[0];
        float b = m[4 * r + 1] * v[1];
        float c = m[4 * r + 2] * v[2];
        float s = a + b;
        s = s + c;
        s = s + m[4 * r + 3];
        o[r] = s;
    }
}

// Centroid bounds as ordered integers: kBoundSlots copies of 6 words (min xyz, max xyz), each on a line of its own, that
// the blocks take in turn; readers merge them.  (With one copy the atomics on its words, 10 ns each in turn, took as
// long as the rest of the kernels that bound centroids.)  Batched builds have 6 words per BLAS instead.
constexpr uint32_t kBoundSlots = 32;
constexpr uint32_t kBoundStride = 32;  // words

struct Bounds {
    uint32_t lo[3] = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu};
    uint32_t hi[3] = {0u, 0u, 0u};
    __device__ void add(const float* c) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const uint32_t o = float_to_ordered(c[a]);
            lo[a] = o < lo[a] ? o : lo[a];
            hi[a] = o > hi[a] ? o : hi[a];
        }
    }
    // over `lanes` lanes (a power of two)
    __device__ void merge_lanes(int lanes) {
        for (int off = lanes / 2; off > 0; off >>= 1) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const uint32_t l = (uint32_t)__shfl_xor((int)lo[a], off), h = (uint32_t)__shfl_xor((int)hi[a], off);
                lo[a] = l < lo[a] ? l : lo[a];
                hi[a] = h > hi[a] ? h : hi[a];
            }
        }
    }
    // a whole wave's bounds to 6 words
    __device__ void publish(uint32_t* cb) {
        merge_lanes(64);
        const uint32_t lane = __lane_id();
        if (lo[0] == 0xFFFFFFFFu && hi[0] == 0u) return;  // nothing added
        if (lane < 3u) atomicMin(&cb[lane], lane == 0 ? lo[0] : (lane == 1 ? lo[1] : lo[2]));
        else if (lane < 6u) atomicMax(&cb[lane], lane == 3 ? hi[0] : (lane == 4 ? hi[1] : hi[2]));
    }
};

// All threads of a 256-thread block: their bounds to the block's slot.
__device__ void publish_block(Bounds b, uint32_t* cb) {
    __shared__ uint32_t s[6];
    if (threadIdx.x < 6) s[threadIdx.x] = (threadIdx.x < 3) ? 0xFFFFFFFFu : 0u;
    __syncthreads();
    b.publish(s);
    __syncthreads();
    uint32_t* slot = cb + kBoundStride * (blockIdx.x % kBoundSlots);
    if (threadIdx.x < 3) {
        if (s[threadIdx.x] != 0xFFFFFFFFu) atomicMin(&slot[threadIdx.x], s[threadIdx.x]);
    } else if (threadIdx.x < 6) {
        if (s[threadIdx.x] != 0u) atomicMax(&slot[threadIdx.x], s[threadIdx.x]);
    }
}

// The merged bounds for all threads of a block, in 6 words of LDS.
__device__ void load_bounds(const uint32_t* __restrict__ cb, uint32_t* s) {
    if (threadIdx.x < 64u) {
        Bounds b;
        if (threadIdx.x < kBoundSlots) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                b.lo[a] = cb[kBoundStride * threadIdx.x + a];
                b.hi[a] = cb[kBoundStride * threadIdx.x + 3 + a];
            }
        }
        b.merge_lanes(64);
        if (threadIdx.x == 0) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                s[a] = b.lo[a];
                s[3 + a] = b.hi[a];
            }
        }
    }
    __syncthreads();
}

// Words that a build starts from: the bounds' slots, and the 16 words of counters (zero).
__global__ __launch_bounds__(256) void init_build_kernel(uint32_t* __restrict__ cb, uint32_t* __restrict__ misc) {
    for (uint32_t i = threadIdx.x; i < kBoundSlots * kBoundStride; i += 256u)
        cb[i] = i % kBoundStride < 3u ? 0xFFFFFFFFu : 0u;
    if (threadIdx.x < 16u) misc[threadIdx.x] = 0u;
}

// prim_blas != nullptr: batched build (per-primitive BLAS id out, per-BLAS centroid bounds).  A block takes `per`
// consecutive primitives; its bounds go out once, or where a batch goes on to the next BLAS.  Bound by HBM: 136 B per
// triangle (12 indices, 36 vertices, 88 written); 4M triangles 143 us = 3.8 TB/s, against 412 us with the six LDS atomics
// per thread and six global ones per 256 triangles that the bounds used to take.
__global__ __launch_bounds__(256) void prep_tris_kernel(const GeomDesc* __restrict__ geoms, int ngeom, uint32_t n,
                                                        TriSlot* __restrict__ leaves, float* __restrict__ boxes,
                                                        uint32_t* __restrict__ cbounds,
                                                        uint32_t* __restrict__ prim_blas, uint32_t per) {
    Bounds bounds;
    uint32_t bounds_blas = 0xFFFFFFFFu;
    const uint64_t first = (uint64_t)blockIdx.x * per;
    const uint32_t end = (uint32_t)(first + per < n ? first + per : n);
    for (uint64_t at = first; at < end; at += 256u) {
        const uint32_t i = (uint32_t)at + threadIdx.x;
        uint32_t blas = 0;
        bool valid = false;
        float cen[3] = {0, 0, 0};
        if (i < end) {
            int lo = 0, hi = ngeom - 1;
            while (lo < hi) {
                int mid = (lo + hi + 1) >> 1;
                if (geoms[mid].prim_base <= i) lo = mid; else hi = mid - 1;
            }
            const GeomDesc g = geoms[lo];
            uint32_t p = i - g.prim_base;
            blas = g.blas;
            if (prim_blas) prim_blas[i] = blas;
            TriSlot t;
            valid = true;
            if (g.type == RTX_GEOMETRY_TYPE_AABBS) {
                // VkAabbPositionsKHR: min xyz, max xyz; inactive when NaN or min > max
                const float* src = (const float*)(g.vtx + (uint64_t)p * g.stride);
#pragma unroll
                for (int k = 0; k < 6; ++k) t.v[k] = src[k];
                t.v[6] = t.v[7] = t.v[8] = 0.0f;
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    valid = valid && isfinite(t.v[a]) && isfinite(t.v[3 + a]) && t.v[a] <= t.v[3 + a];
            } else {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    uint32_t vi = g.idx[3 * (uint64_t)p + k];
                    float v[3];
                    if (vi > g.max_vertex) {
                        valid = false;
                        v[0] = v[1] = v[2] = 0.0f;
                    } else {
                        const float* src = (const float*)(g.vtx + (uint64_t)(vi + g.first_vertex) * g.stride);
                        v[0] = src[0];
                        v[1] = src[1];
                        v[2] = src[2];
                    }
                    if (g.xform) {
                        float o[3];
                        xform_vertex(g.xform, v, o);
                        t.v[3 * k] = o[0];
                        t.v[3 * k + 1] = o[1];
                        t.v[3 * k + 2] = o[2];
                    } else {
                        t.v[3 * k] = v[0];
                        t.v[3 * k + 1] = v[1];
                        t.v[3 * k + 2] = v[2];
                    }
                }
#pragma unroll
                for (int k = 0; k < 9; ++k) valid = valid && isfinite(t.v[k]);
            }
            t.prim = p;
            t.geom = g.geom_local;
            t.bits = (valid ? kTriValid : 0u) | ((g.flags & RTX_GEOMETRY_OPAQUE_BIT) ? 0u : kTriNonOpaque) |
                     (g.type == RTX_GEOMETRY_TYPE_AABBS ? kTriAabb : 0u);
            t.pad[0] = t.pad[1] = t.pad[2] = t.pad[3] = 0u;
            leaves[i] = t;
            float* b = boxes + 6 * (uint64_t)i;
            if (valid) {
                const bool aabb = g.type == RTX_GEOMETRY_TYPE_AABBS;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    float l = aabb ? t.v[a] : fminf(t.v[a], fminf(t.v[3 + a], t.v[6 + a]));
                    float h = aabb ? t.v[3 + a] : fmaxf(t.v[a], fmaxf(t.v[3 + a], t.v[6 + a]));
                    b[a] = l;
                    b[3 + a] = h;
                    float s = l + h;
                    cen[a] = s * 0.5f;
                }
            } else {
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    b[a] = INFINITY;
                    b[3 + a] = -INFINITY;
                }
            }
        }
        if (!prim_blas) {
            if (valid) bounds.add(cen);
            continue;
        }
        const uint64_t in = __ballot(i < end);
        if (!in) continue;
        const uint32_t b0 = (uint32_t)__shfl((int)blas, __ffsll((unsigned long long)in) - 1);
        if (b0 != bounds_blas) {
            if (bounds_blas != 0xFFFFFFFFu) bounds.publish(cbounds + 6 * (uint64_t)bounds_blas);
            bounds = Bounds();
            bounds_blas = b0;
        }
        if (valid && blas == b0) {
            bounds.add(cen);
        } else if (valid) {  // a wave that straddles a boundary
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const uint32_t o = float_to_ordered(cen[a]);
                atomicMin(&cbounds[6 * (uint64_t)blas + a], o);
                atomicMax(&cbounds[6 * (uint64_t)blas + 3 + a], o);
            }
        }
    }
    if (!prim_blas)
        publish_block(bounds, cbounds);
    else if (bounds_blas != 0xFFFFFFFFu)
        bounds.publish(cbounds + 6 * (uint64_t)bounds_blas);
}
// Consecutive primitives per block: at most 2,048 blocks, which fill the chip.
uint32_t prep_chunk(uint32_t n) { return ((n + 255u) / 256u + 2047u) / 2048u * 256u; }

__device__ void invert3x4_d(const double* m, double* inv) {
    double a = m[0], b = m[1], c = m[2], d = m[4], e = m[5], f = m[6], g = m[8], h = m[9], i = m[10];
    double A = e * i - f * h, B = -(d * i - f * g), C = d * h - e * g;
    double det = a * A + b * B + c * C;
    double r = 1.0 / det;
    inv[0] = A * r;
    inv[1] = -(b * i - c * h) * r;
    inv[2] = (b * f - c * e) * r;
    inv[4] = B * r;
    inv[5] = (a * i - c * g) * r;
    inv[6] = -(a * f - c * d) * r;
    inv[8] = C * r;
    inv[9] = -(a * h - b * g) * r;
    inv[10] = (a * e - b * d) * r;
#pragma unroll
    for (int row = 0; row < 3; ++row)
        inv[4 * row + 3] = -(inv[4 * row + 0] * m[3] + inv[4 * row + 1] * m[7] + inv[4 * row + 2] * m[11]);
}

__device__ __forceinline__ float round_down_f(double x) {
    float f = (float)x;
    if ((double)f > x) f = nextafterf(f, -INFINITY);
    return f;
}
__device__ __forceinline__ float round_up_f(double x) {
    float f = (float)x;
    if ((double)f < x) f = nextafterf(f, INFINITY);
    return f;
}

// World box of an instance: the union of its BLAS's second-level boxes (the root's leaf children, and the
// children of its internal children), each decoded from the 8-bit planes with the FP32 operations the traversal
// uses (so it encloses what they enclose) and transformed corner by corner in FP64.  For a rotated instance this
// is much tighter than the transformed root box, and every ray that misses it skips the instance's FP64 entry.
// A BLAS whose nodes do not check out falls back to the root box.
__device__ void add_world_box(const double* m, const float* blo, const float* bhi, double* lo, double* hi) {
    for (int c = 0; c < 8; ++c) {
        const double p[3] = {(double)((c & 1) ? bhi[0] : blo[0]), (double)((c & 2) ? bhi[1] : blo[1]),
                             (double)((c & 4) ? bhi[2] : blo[2])};
        for (int a = 0; a < 3; ++a) {
            const double w = m[4 * a] * p[0] + m[4 * a + 1] * p[1] + m[4 * a + 2] * p[2] + m[4 * a + 3];
            lo[a] = fmin(lo[a], w);
            hi[a] = fmax(hi[a], w);
        }
    }
}

__device__ void decode_child_box(const Node8* nd, int k, const float* rlo, const float* qs, float* blo, float* bhi) {
    for (int a = 0; a < 3; ++a) {
        const float p = fmaf((float)nd->pq[a], qs[a], rlo[a]);
        const float sc = __uint_as_float((uint32_t)nd->e[a] << 23);
        blo[a] = fmaf((float)nd->qlo[a][k], sc, p);
        bhi[a] = fmaf((float)nd->qhi[a][k], sc, p);
    }
}

// By a whole wave: lane 8 k + j takes grandchild j of child k.
__device__ void instance_world_box(const AsHeader* h, const double* m, double* lo, double* hi) {
    const uint32_t k = __lane_id() >> 3, j = __lane_id() & 7u;
    const uint8_t* slots = (const uint8_t*)h + kHeaderBytes;
    const Node8* root = (const Node8*)slots;
    const float rlo[3] = {h->lo[0], h->lo[1], h->lo[2]}, qs[3] = {h->qscale[0], h->qscale[1], h->qscale[2]};
    const uint32_t nslots = h->slot_count;
    bool ok = root->vmask != 0 && root->base < nslots;
    const bool present = (root->vmask >> k) & 1u, internal = present && ((root->imask >> k) & 1u);
    const uint32_t cs = root->base + (uint32_t)__popc(root->vmask & ((1u << k) - 1u));
    const Node8* c = (const Node8*)(slots + (uint64_t)cs * kSlotBytes);
    if (ok && internal) ok = cs < nslots && c->vmask != 0;
    float blo[3], bhi[3];
    if (!__all(ok)) {
        if (__lane_id() == 0) add_world_box(m, h->lo, h->hi, lo, hi);
    } else if (internal) {
        if ((c->vmask >> j) & 1u) {
            decode_child_box(c, (int)j, rlo, qs, blo, bhi);
            add_world_box(m, blo, bhi, lo, hi);
        }
    } else if (present && j == 0) {
        decode_child_box(root, (int)k, rlo, qs, blo, bhi);
        add_world_box(m, blo, bhi, lo, hi);
    }
    for (int off = 32; off > 0; off >>= 1)
        for (int a = 0; a < 3; ++a) {
            lo[a] = fmin(lo[a], __shfl_xor(lo[a], off));
            hi[a] = fmax(hi[a], __shfl_xor(hi[a], off));
        }
}

// A wave per instance (a thread per instance took 41 us for three instances: one lane went through the 64 boxes of the
// BLAS's second level in turn).
__global__ __launch_bounds__(256) void prep_instances_kernel(const rtx_instance* __restrict__ inst, uint32_t n,
                                                             InstSlot* __restrict__ leaves,
                                                             InstanceInfo* __restrict__ table,
                                                             float* __restrict__ boxes,
                                                             uint32_t* __restrict__ cbounds,
                                                             uint32_t* __restrict__ max_blas_depth,
                                                             uint32_t* __restrict__ content_out) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t waves = gridDim.x * 4u;
    uint32_t content = 0, depth = 0;
    Bounds bounds;
    for (uint32_t i = blockIdx.x * 4u + (threadIdx.x >> 6); i < n; i += waves) {
        const rtx_instance r = inst[i];
        bool valid = false;
        double m[12];
        for (int k = 0; k < 12; ++k) m[k] = (double)(&r.transform[0][0])[k];
        double inv[12];
        invert3x4_d(m, inv);
        const uint32_t flags = r.sbt_offset_and_flags >> 24;
        float box[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
        bool ok = r.blas_address != 0 && (r.blas_address & 255u) == 0 && isfinite(inv[0]) && isfinite(inv[5]) &&
                  isfinite(inv[10]);
        if (ok) {
            const AsHeader* h = (const AsHeader*)r.blas_address;
            ok = h->magic == kMagicBlas && h->prim_count > 0 && h->slot_count > 0;
            if (ok) {
                double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
                instance_world_box(h, m, lo, hi);
                double ext = 0;
                for (int a = 0; a < 3; ++a) ext = fmax(ext, fmax(fabs(lo[a]), fabs(hi[a])) + (hi[a] - lo[a]));
                const double pad = ext * 0x1p-20;
                for (int a = 0; a < 3; ++a) {
                    box[a] = round_down_f(lo[a] - pad);
                    box[3 + a] = round_up_f(hi[a] + pad);
                }
                depth = h->max_depth > depth ? h->max_depth : depth;
                content |= h->content | ((flags & RTX_INSTANCE_FORCE_NO_OPAQUE_BIT) ? kContentNonOpaque : 0u);
                valid = true;
            }
        }
        if (lane == 0) {
            InstanceInfo info;
            InstSlot s;
            for (int k = 0; k < 12; ++k) {
                info.inv[k] = inv[k];
                s.inv[k] = (float)inv[k];
            }
            info.custom = r.custom_index_and_mask & 0xFFFFFFu;
            info.mask = r.custom_index_and_mask >> 24;
            info.sbt_offset = r.sbt_offset_and_flags & 0xFFFFFFu;
            info.flags = flags;
            info.blas = r.blas_address;
            info.pad = 0;
            s.blas = r.blas_address;
            s.instance_id = i;
            s.mask = info.mask | (flags << 8);
            leaves[i] = s;
            table[i] = info;
            float cen[3];
            for (int a = 0; a < 3; ++a) {
                boxes[6 * (uint64_t)i + a] = box[a];
                boxes[6 * (uint64_t)i + 3 + a] = box[3 + a];
                const float s2 = box[a] + box[3 + a];
                cen[a] = s2 * 0.5f;
            }
            if (valid) bounds.add(cen);
        }
    }
    // one atomic per wave for the depth and the content bits
    if (lane == 0 && depth) atomicMax(max_blas_depth, depth);
    if (lane == 0 && content) atomicOr(content_out, content);
    publish_block(bounds, cbounds);
}

__global__ __launch_bounds__(256) void box_bounds_kernel(const float* __restrict__ boxes, uint32_t n,
                                                         uint32_t* __restrict__ cbounds) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    float cen[3] = {0, 0, 0};
    bool valid = false;
    if (i < n) {
        const float* b = boxes + 6 * (uint64_t)i;
        valid = b[0] <= b[3] && b[1] <= b[4] && b[2] <= b[5];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            float s = b[a] + b[3 + a];
            cen[a] = s * 0.5f;
        }
    }
    Bounds bounds;
    if (valid) bounds.add(cen);
    publish_block(bounds, cbounds);
}

__device__ __forceinline__ uint32_t quant_axis(float c, float cmin, float scale, uint32_t maxq) {
    float f = (c - cmin) * scale;
    if (!(f > 0.0f)) return 0u;
    if (f >= (float)maxq) return maxq;
    return (uint32_t)f;
}

template <typename K>
__global__ __launch_bounds__(256) void morton_kernel(const float* __restrict__ boxes, uint32_t n,
                                                     const uint32_t* __restrict__ slots, K* __restrict__ keys) {
    __shared__ uint32_t cbounds[6];
    load_bounds(slots, cbounds);
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    constexpr bool k64 = sizeof(K) == 8;
    const float cells = k64 ? 2097152.0f : 1024.0f;
    const uint32_t maxq = k64 ? 2097151u : 1023u;
    const float* b = boxes + 6 * (uint64_t)i;
    uint32_t q[3];
    bool valid = b[0] <= b[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float cmin = ordered_to_float(cbounds[a]);
        float cmax = ordered_to_float(cbounds[3 + a]);
        float ext = cmax - cmin;
        float scale = ext > 0.0f ? cells / ext : 0.0f;
        float s = b[a] + b[3 + a];
        float c = s * 0.5f;
        q[a] = quant_axis(c, cmin, scale, maxq);
    }
    K code;
    if (k64)
        code = (K)((spread21(q[0]) << 2) | (spread21(q[1]) << 1) | spread21(q[2]));
    else
        code = (K)((spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]));
    keys[i] = valid ? code : (K)~(K)0;
}

// Batched builds: key = BLAS id << 30 | 30-bit Morton code over that BLAS's centroid bounds, so that a stable
// sort groups the BLASes and every BLAS becomes one subtree of the binary radix tree.
__global__ __launch_bounds__(256) void morton_batch_kernel(const float* __restrict__ boxes, uint32_t n,
                                                           const uint32_t* __restrict__ cbounds,
                                                           const uint32_t* __restrict__ prim_blas,
                                                           uint64_t* __restrict__ keys) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t blas = prim_blas[i];
    const uint32_t* cb = cbounds + 6 * (uint64_t)blas;
    const float* b = boxes + 6 * (uint64_t)i;
    uint32_t q[3];
    const bool valid = b[0] <= b[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float cmin = ordered_to_float(cb[a]);
        float cmax = ordered_to_float(cb[3 + a]);
        float ext = cmax - cmin;
        float scale = ext > 0.0f ? 1024.0f / ext : 0.0f;
        float s = b[a] + b[3 + a];
        float c = s * 0.5f;
        q[a] = quant_axis(c, cmin, scale, 1023u);
    }
    const uint32_t code = valid ? ((spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2])) : 0x3FFFFFFFu;
    keys[i] = ((uint64_t)blas << 30) | code;
}

constexpr uint32_t kMixedBlas = 0xFFFFFFFFu;

template <typename K>
__device__ __forceinline__ int karras_delta(const K* keys, int64_t n, int64_t i, int64_t j) {
    if (j < 0 || j >= n) return -1;
    K a = keys[i], b = keys[j];
    constexpr int kb = (int)sizeof(K) * 8;
    if (a == b) return kb + __clz((uint32_t)(i ^ j));
    if (sizeof(K) == 8) return __clzll((unsigned long long)(a ^ b));
    return __clz((uint32_t)(a ^ b));
}

// cnt: primitives below each internal node.  node_blas != nullptr (batched builds): the BLAS that owns all primitives
// of internal node i, or kMixedBlas.
template <typename K>
__global__ __launch_bounds__(256) void karras_kernel(const K* __restrict__ keys, uint32_t n, int32_t* __restrict__ left,
                                                     int32_t* __restrict__ right, int32_t* __restrict__ parent,
                                                     uint32_t* __restrict__ cnt,
                                                     uint32_t* __restrict__ node_blas = nullptr) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i == 0) parent[0] = -1;
    if (i >= (int64_t)n - 1) return;
    int64_t N = n;
    int d = (karras_delta(keys, N, i, i + 1) - karras_delta(keys, N, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = karras_delta(keys, N, i, i - d);
    int64_t lmax = 2;
    while (karras_delta(keys, N, i, i + lmax * d) > dmin) lmax *= 2;
    int64_t l = 0;
    for (int64_t t = lmax / 2; t >= 1; t /= 2)
        if (karras_delta(keys, N, i, i + (l + t) * d) > dmin) l += t;
    int64_t j = i + l * d;
    int dnode = karras_delta(keys, N, i, j);
    int64_t s = 0;
    int64_t t = l;
    do {
        t = (t + 1) / 2;
        if (s + t <= l && karras_delta(keys, N, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int64_t gamma = i + s * d + (d < 0 ? -1 : 0);
    int64_t lo = i < j ? i : j, hi = i < j ? j : i;
    int32_t lc = (lo == gamma) ? (int32_t)(-1 - gamma) : (int32_t)gamma;
    int32_t rc = (hi == gamma + 1) ? (int32_t)(-1 - (gamma + 1)) : (int32_t)(gamma + 1);
    left[i] = lc;
    right[i] = rc;
    cnt[i] = (uint32_t)(hi - lo + 1);
    parent[lc >= 0 ? lc : (N - 1) + (-1 - lc)] = (int32_t)i;
    parent[rc >= 0 ? rc : (N - 1) + (-1 - rc)] = (int32_t)i;
    if (node_blas) {
        const uint64_t blo = (uint64_t)keys[lo] >> 30, bhi = (uint64_t)keys[hi] >> 30;
        node_blas[i] = blo == bhi ? (uint32_t)blo : kMixedBlas;
    }
}

// Batched builds: the root of BLAS b is its topmost node whose primitives all belong to b (a leaf for a
// one-triangle BLAS).  Runs over the 2n-1 nodes before the refit; the refinement never moves these roots.
__global__ __launch_bounds__(256) void blas_roots_kernel(uint32_t n, const uint64_t* __restrict__ keys,
                                                         const int32_t* __restrict__ parent,
                                                         const uint32_t* __restrict__ node_blas,
                                                         int32_t* __restrict__ roots) {
    const uint64_t k = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (k >= 2ull * n - 1) return;
    uint32_t b;
    int32_t code;
    if (k < (uint64_t)n - 1) {
        b = node_blas[k];
        code = (int32_t)k;
    } else {
        const uint64_t pos = k - (n - 1);
        b = (uint32_t)(keys[pos] >> 30);
        code = -1 - (int32_t)pos;
    }
    if (b == kMixedBlas) return;
    const int32_t p = parent[k];
    if (p < 0 || node_blas[p] == kMixedBlas) roots[b] = code;
}

__device__ __forceinline__ float load_coherent(const float* p) {
    return __uint_as_float(__hip_atomic_load((const uint32_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ void store_coherent(float* p, float v) {
    __hip_atomic_store((uint32_t*)p, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint32_t load_coherent_u32(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_coherent_u32(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int32_t load_coherent_i32(const int32_t* p) {
    return (int32_t)load_coherent_u32((const uint32_t*)p);
}
__device__ __forceinline__ void store_coherent_i32(int32_t* p, int32_t v) {
    store_coherent_u32((uint32_t*)p, (uint32_t)v);
}

// ---- bottom-up refit with SAH treelet refinement ------------------------------------------------------------
//
// Node numbering: internal nodes 0..n-2, leaves n-1+pos (sorted position); a child code c >= 0 is internal node
// c, c < 0 the leaf at position -1-c.  Per internal node the pass keeps the box, the SAH cost of its subtree
// (sum of internal-node surface areas, the only term a restructuring can change), the primitive count and the
// height (leaves: cost 0, count 1, height 0).  The node cost is area + (cost(left) + cost(right)).
//
// When a node with at least min_prims primitives is complete, a whole wave restructures the treelet below it (Karras &
// Aila 2013, "Fast Parallel Construction of High-Quality Bounding Volume Hierarchies"):
//   formation  start from the node's two children and open the internal treelet leaf with the largest surface
//              area (lowest slot on ties) until there are 7 leaves; the node and the 5 opened nodes are the
//              treelet's 6 internal nodes
//   DP         over the 127 leaf subsets S in order of size: cost(S) = area(S) + min over splits {P, S\P} of
//              (cost(P) + cost(S\P)), P containing the lowest leaf of S; ties go to the smallest P
//   rebuild    only on a strict cost decrease and when the treelet height does not grow (so the whole tree
//              keeps the radix tree's depth bound): breadth-first from S = all leaves, internal
//              nodes reused in formation order.
// A treelet covers only nodes of its root's finished subtree and is processed after that subtree is final, so
// the result does not depend on the order in which waves finish.
//
// A pass has two launches.  subtree_refine_kernel: a wave takes a maximal subtree of at most kSubtree primitives into
// LDS and works through it level by level, deepest first.  refit_refine_kernel: the nodes above, a thread per subtree
// climbing from its root; the second thread to reach a node (atomic arrival count) merges its children.  There the
// cross-wave hand-off uses agent-scope atomic loads and stores (coherent across XCDs without L2 write-back fences): a
// wave waits for its stores to complete (s_waitcnt) before it bumps a parent's arrival count.
constexpr int kTreeletLeaves = 7;
constexpr uint32_t kTreeletNodes = kTreeletLeaves - 1;

// The DP's work of one wave, per lane.  A subset S of size K has 2^(K-1) - 1 splits {P, S\P} with P holding S's lowest
// leaf; kSplitLanes[K] consecutive lanes share a subset (1 for K <= 4, 2 for K = 5, 8 for K = 6) and take its splits
// in turn, in order of P.  split[t][lane]: the byte offsets of cost[P] (low half) and cost[S\P] (high half) of the
// lane's split in step t, offsets of cost[0] (infinite) where it has none; steps of size K from kSplitStep[K].
// subset[w][lane]: byte K - 2 of the two words: the subset whose result the lane writes (0: none).
constexpr uint32_t kSplitLanes[7] = {0, 0, 1, 1, 1, 2, 8};
constexpr uint32_t kSplitStep[8] = {0, 0, 0, 1, 4, 11, 19, 23};
constexpr uint32_t kSplitSteps = 23;
struct SplitTable {
    uint32_t split[kSplitSteps][64];
    uint32_t subset[2][64];
};
constexpr uint32_t bits7(uint32_t v) {
    uint32_t c = 0;
    for (; v; v &= v - 1u) ++c;
    return c;
}
constexpr SplitTable make_split_table() {
    SplitTable T{};
    for (uint32_t K = 2; K <= 6; ++K) {
        uint32_t sub = 0;
        for (uint32_t S = 1; S < 128; ++S) {
            if (bits7(S) != K) continue;
            const uint32_t low = S & (0u - S), rest = S ^ low;
            const uint32_t first = sub * kSplitLanes[K];
            T.subset[(K - 2) / 4][first] |= S << (8 * ((K - 2) & 3));
            uint32_t q = 0;  // the proper subsets of rest in increasing order
            for (uint32_t i = 0; i < (1u << (K - 1)) - 1u; ++i) {
                const uint32_t P = low | q;
                T.split[kSplitStep[K] + i / kSplitLanes[K]][first + i % kSplitLanes[K]] = (4u * P) | (4u * (S ^ P)) << 16;
                q = (q - rest) & rest;
            }
            ++sub;
        }
    }
    return T;
}
__constant__ SplitTable kSplitTable = make_split_table();

// A lane's part of the table, loaded once per wave.
struct SplitRegs {
    uint32_t split[kSplitSteps];
    uint32_t subset[2];
};
__device__ __forceinline__ void load_splits(SplitRegs& r) {
    const uint32_t lane = threadIdx.x;
#pragma unroll
    for (uint32_t t = 0; t < kSplitSteps; ++t) r.split[t] = kSplitTable.split[t][lane];
    r.subset[0] = kSplitTable.subset[0][lane];
    r.subset[1] = kSplitTable.subset[1][lane];
}

// One treelet in LDS: its leaves and internal nodes (codes of the caller), the leaves' boxes and values, the DP.
struct TreeletLds {
    float cost[128];  // of every subset; its surface area until the DP reaches it
    uint8_t part[128];
    float box[kTreeletLeaves + 1][6];
    uint32_t lcnt[kTreeletLeaves], lhgt[kTreeletLeaves];
    int32_t leaf[kTreeletLeaves];
    int32_t pool[kTreeletNodes];
};

// The restructured treelet (wave-uniform): node i (0 = the root, breadth-first) covers leaf subset (sets >> 8 i) & 255,
// its children are 4-bit codes in byte i of kids (child 0 low): node index, or 8 + leaf; heights in bytes.
struct TreeletPlan {
    uint64_t sets, kids, heights;
    float total;
    bool commit;
};

// DP steps of subset size K.
template <uint32_t K>
__device__ __forceinline__ void treelet_dp_size(TreeletLds& T, const SplitRegs& r) {
    constexpr uint32_t G = kSplitLanes[K];
    const uint8_t* const cost = (const uint8_t*)T.cost;
    float best = INFINITY;
    uint32_t bp = 0;  // offset of the best P; no finite split: 0
#pragma unroll
    for (uint32_t t = kSplitStep[K]; t < kSplitStep[K + 1]; ++t) {
        const uint32_t p = r.split[t] & 0xFFFFu;
        const float c = *(const float*)(cost + p) + *(const float*)(cost + (r.split[t] >> 16));
        if (c < best) {
            best = c;
            bp = p;
        }
    }
#pragma unroll
    for (uint32_t off = G / 2; off > 0; off >>= 1) {
        const float oc = __shfl_xor(best, (int)off);
        const uint32_t op = (uint32_t)__shfl_xor((int)bp, (int)off);
        if (oc < best || (oc == best && op < bp)) {
            best = oc;
            bp = op;
        }
    }
    const uint32_t S = (r.subset[(K - 2) / 4] >> (8 * ((K - 2) & 3))) & 255u;
    if (S) {
        T.cost[S] = T.cost[S] + best;
        T.part[S] = (uint8_t)(bp >> 2);
    }
    __syncthreads();
}

// Whole-wave solution of the treelet staged in T (boxes, counts, heights, and cost[1 << j] of its leaves).
__device__ __forceinline__ TreeletPlan treelet_solve(TreeletLds& T, const SplitRegs& r, float old_cost, uint32_t old_h) {
    const uint32_t lane = threadIdx.x;
    TreeletPlan plan;
    plan.sets = plan.kids = plan.heights = 0;
    plan.total = old_cost;
    plan.commit = false;
    // surface areas: lane S for subset S of leaves 0..5, then with leaf 6 for subset 64 + S
    {
        float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
        for (int j = 0; j < kTreeletLeaves - 1; ++j)
            if (lane & (1u << j)) {
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    b[a] = fminf(b[a], T.box[j][a]);
                    b[3 + a] = fmaxf(b[3 + a], T.box[j][3 + a]);
                }
            }
        const float a0 = box_area(b);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            b[a] = fminf(b[a], T.box[kTreeletLeaves - 1][a]);
            b[3 + a] = fmaxf(b[3 + a], T.box[kTreeletLeaves - 1][3 + a]);
        }
        const float a1 = box_area(b);
        if (lane & (lane - 1u)) T.cost[lane] = a0;
        if (lane) T.cost[64u + lane] = a1;
        if (lane == 0) T.cost[0] = INFINITY;
    }
    __syncthreads();
    treelet_dp_size<2>(T, r);
    treelet_dp_size<3>(T, r);
    treelet_dp_size<4>(T, r);
    treelet_dp_size<5>(T, r);
    treelet_dp_size<6>(T, r);
    // all 7 leaves: the 63 splits containing leaf 0, one per lane; the lowest lane with the least cost has the smallest P
    const uint32_t p7 = 1u | (lane << 1);
    const float c7 = lane < 63u ? T.cost[p7] + T.cost[127u ^ p7] : INFINITY;
    float m = c7;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fminf(m, __shfl_xor(m, off));
    const uint64_t at = __ballot(c7 == m && lane < 63u);
    const float total = T.cost[127] + m;
    if (!(total < old_cost) || !at) return plan;
    const uint32_t P7 = 1u | ((uint32_t)__ffsll((unsigned long long)at) - 1u) << 1;
    // rebuild, breadth-first, on wave-uniform values
    uint64_t sets = 127u, kids = 0;
    uint32_t nodes = 1;
#pragma unroll
    for (uint32_t i = 0; i < kTreeletNodes; ++i) {
        const uint32_t S = (uint32_t)(sets >> (8 * i)) & 127u;
        const uint32_t P =
            i == 0 ? P7 : (uint32_t)__builtin_amdgcn_readfirstlane((int)T.part[S]);
        if (i >= nodes || P == 0u || (P & S) != P || P == S) return plan;  // no finite split was found
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t C = h ? S ^ P : P;
            uint32_t code;
            if ((C & (C - 1u)) == 0u) {
                code = 8u + (uint32_t)__ffs((int)C) - 1u;
            } else {
                code = nodes;
                sets |= (uint64_t)C << (8 * nodes);
                ++nodes;
            }
            kids |= (uint64_t)code << (8 * i + 4 * h);
        }
    }
    uint64_t lh = 0, heights = 0;
#pragma unroll
    for (int j = 0; j < kTreeletLeaves; ++j)
        lh |= (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)T.lhgt[j]) << (8 * j);
#pragma unroll
    for (int i = (int)kTreeletNodes - 1; i >= 0; --i) {
        uint32_t hc[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t code = (uint32_t)(kids >> (8 * i + 4 * h)) & 15u;
            hc[h] = (uint32_t)((code & 8u ? lh : heights) >> (8 * (code & 7u))) & 255u;
        }
        heights |= (uint64_t)(1u + (hc[0] > hc[1] ? hc[0] : hc[1])) << (8 * i);
    }
    plan.sets = sets;
    plan.kids = kids;
    plan.heights = heights;
    plan.commit = (heights & 255u) <= old_h;
    if (plan.commit) plan.total = total;
    return plan;
}

__device__ __forceinline__ int32_t plan_child(const TreeletLds& T, const TreeletPlan& plan, uint32_t i, int h) {
    const uint32_t code = (uint32_t)(plan.kids >> (8 * i + 4 * h)) & 15u;
    return code & 8u ? T.leaf[code & 7u] : T.pool[code];
}

// Box and primitive count of plan node i.
__device__ __forceinline__ uint32_t plan_bounds(const TreeletLds& T, uint32_t S, float* b) {
    uint32_t np = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        b[k] = INFINITY;
        b[3 + k] = -INFINITY;
    }
#pragma unroll
    for (int j = 0; j < kTreeletLeaves; ++j)
        if (S & (1u << j)) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                b[a] = fminf(b[a], T.box[j][a]);
                b[3 + a] = fmaxf(b[3 + a], T.box[j][3 + a]);
            }
            np += T.lcnt[j];
        }
    return np;
}

__device__ __forceinline__ uint64_t node_index(uint32_t n, int32_t c) {
    return c >= 0 ? (uint64_t)c : (uint64_t)n - 1 + (uint64_t)(-1 - c);
}

__device__ __forceinline__ float coherent_area(const float* nboxes, uint64_t i) {
    float b[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) b[k] = load_coherent(nboxes + 6 * i + k);
    return box_area(b);
}

// Treelet formation for root R, by one lane: open the largest-area internal treelet leaf until there are 7
// leaves; false when fewer than 7 primitives lie below R (nothing to restructure).  The lanes of a wave form their
// treelets at the same time: their roots were completed in the same step, so none is an ancestor of another and their
// subtrees - everything a formation reads and a restructuring writes - are disjoint.  children(c, l, r, al, ar): node
// c's children and their areas (-1 for leaves, which have negative codes).
struct TreeletForm {
    int32_t leaf[kTreeletLeaves];
    int32_t pool[kTreeletNodes];
};

template <typename Children>
__device__ __forceinline__ bool treelet_form(int32_t R, Children children, TreeletForm& out) {
    int32_t lf[kTreeletLeaves];
    float la[kTreeletLeaves];
    out.pool[0] = R;
    children(R, lf[0], lf[1], la[0], la[1]);
#pragma unroll
    for (int k = 2; k < kTreeletLeaves; ++k) {
        int best = -1;
        float ba = -1.0f;
        int32_t c = 0;
#pragma unroll
        for (int j = 0; j < k; ++j)
            if (la[j] > ba) {
                ba = la[j];
                best = j;
                c = lf[j];
            }
        if (best < 0) return false;
        out.pool[k - 1] = c;
        int32_t l, r;
        float al, ar;
        children(c, l, r, al, ar);
#pragma unroll
        for (int j = 0; j < k; ++j)
            if (j == best) {
                lf[j] = l;
                la[j] = al;
            }
        lf[k] = r;
        la[k] = ar;
    }
#pragma unroll
    for (int j = 0; j < kTreeletLeaves; ++j) out.leaf[j] = lf[j];
    return true;
}

__device__ __forceinline__ void stage_form(TreeletLds& T, const TreeletForm& f) {
#pragma unroll
    for (int j = 0; j < kTreeletLeaves; ++j) T.leaf[j] = f.leaf[j];
#pragma unroll
    for (uint32_t j = 0; j < kTreeletNodes; ++j) T.pool[j] = f.pool[j];
}

// Whole-wave treelet restructuring below internal node R (uniform arguments) from its formation, which lane
// `owner` holds in `f`, in global memory.  Returns R's cost and height afterwards through new_cost / new_h.
__device__ __forceinline__ void treelet_optimize(TreeletLds& T, const SplitRegs& sr, uint32_t n, float old_cost,
                                                 uint32_t old_h, uint32_t owner, const TreeletForm& f, int32_t* left,
                                                 int32_t* right, int32_t* parent, float* nboxes, float* cost,
                                                 uint32_t* cnt, uint32_t* hgt, float& new_cost, uint32_t& new_h) {
    const uint32_t lane = threadIdx.x;
    __syncthreads();
    if (lane == owner) stage_form(T, f);
    __syncthreads();
    if (lane < (uint32_t)kTreeletLeaves) {
        const int32_t c = T.leaf[lane];
        const uint64_t bi = node_index(n, c);
#pragma unroll
        for (int k = 0; k < 6; ++k) T.box[lane][k] = load_coherent(nboxes + 6 * bi + k);
        T.cost[1u << lane] = c >= 0 ? load_coherent(cost + c) : 0.0f;
        T.lcnt[lane] = c >= 0 ? load_coherent_u32(cnt + c) : 1u;
        T.lhgt[lane] = c >= 0 ? load_coherent_u32(hgt + c) : 0u;
    }
    __syncthreads();
    const TreeletPlan plan = treelet_solve(T, sr, old_cost, old_h);
    new_cost = old_cost;
    new_h = old_h;
    if (!plan.commit) return;
    if (lane < kTreeletNodes) {
        const int32_t x = T.pool[lane];
        const int32_t c0 = plan_child(T, plan, lane, 0), c1 = plan_child(T, plan, lane, 1);
        store_coherent_i32(left + x, c0);
        store_coherent_i32(right + x, c1);
        store_coherent_i32(parent + node_index(n, c0), x);
        store_coherent_i32(parent + node_index(n, c1), x);
        if (lane > 0) {  // the root's box is unchanged; its cost and height are published by its owner
            const uint32_t S = (uint32_t)(plan.sets >> (8 * lane)) & 127u;
            float b[6];
            const uint32_t np = plan_bounds(T, S, b);
#pragma unroll
            for (int k = 0; k < 6; ++k) store_coherent(nboxes + 6 * (uint64_t)x + k, b[k]);
            store_coherent(cost + x, T.cost[S]);
            store_coherent_u32(cnt + x, np);
            store_coherent_u32(hgt + x, (uint32_t)(plan.heights >> (8 * lane)) & 255u);
        }
    }
    new_cost = plan.total;
    new_h = (uint32_t)plan.heights & 255u;
}

// ---- subtrees in LDS ------------------------------------------------------------------------------------------
//
// A maximal subtree of at most kSubtree primitives as one wave holds it: internal nodes 0 .. nint - 1 breadth-first
// from the root, primitives at kSubtree + 0 .. (local ids), each with its code in the binary tree.
// 112: 9.6 KB of LDS, so that 16 waves share a CU, the four per SIMD that 128 registers allow.  The two rounds over 15.5M
// triangles of 64 meshes take 9.5 + 2.4 ms (subtrees + the nodes above); when they took 11.0 + 2.5, it was 11.1 + 3.0
// with 96 primitives and 14.8 + 2.2 with 128.
constexpr uint32_t kSubtree = 112;
struct SubtreeLds {
    int32_t code[2 * kSubtree];
    uint32_t kids[kSubtree];          // local ids of the children, 16 bits each
    uint16_t level[kSubtree + 1];     // first node of each breadth-first level
};

// Loads the codes and links of the subtree below `root` (an internal node).
__device__ __forceinline__ void load_subtree(SubtreeLds& U, int32_t root, const int32_t* __restrict__ left,
                                             const int32_t* __restrict__ right, uint32_t& nint, uint32_t& nleaf,
                                             uint32_t& nlevel) {
    const uint32_t lane = threadIdx.x;
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    __syncthreads();
    if (lane == 0) {
        U.code[0] = root;
        U.level[0] = 0;
    }
    __syncthreads();
    nint = 1;
    nleaf = 0;
    nlevel = 0;
    for (uint32_t a = 0; a < nint;) {
        const uint32_t end = nint;  // the level is [a, end)
        ++nlevel;
        if (lane == 0) U.level[nlevel] = (uint16_t)end;
        for (; a < end; a += 64u) {
            const bool on = a + lane < end;
            int32_t c[2] = {0, 0};
            if (on) {
                const int32_t x = U.code[a + lane];
                c[0] = left[x];
                c[1] = right[x];
            }
            uint32_t id[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint64_t mi = __ballot(on && c[h] >= 0), ml = __ballot(on && c[h] < 0);
                id[h] = c[h] >= 0 ? nint + (uint32_t)__popcll(mi & below)
                                  : kSubtree + nleaf + (uint32_t)__popcll(ml & below);
                nint += (uint32_t)__popcll(mi);
                nleaf += (uint32_t)__popcll(ml);
                if (on) U.code[id[h]] = c[h];
            }
            if (on) U.kids[a + lane] = id[0] | id[1] << 16;
        }
        a = end;
        __syncthreads();
    }
}

// Lists the maximal subtrees of at most kSubtree primitives (internal node or leaf codes) and clears the arrival
// counts of the nodes above them.  A block looks at kFindNodes nodes and takes its places in the list at once (an atomic
// on one word costs about 10 ns in turn: one per listed node took 1.1 ms on 15.5M triangles).  queue: an empty place for
// each of the nodes above, which the collapse queues its tasks in.
constexpr uint32_t kFindNodes = 4096;
constexpr uint64_t kNoTask = ~0ull;
__global__ __launch_bounds__(256) void find_subtrees_kernel(uint32_t n, const int32_t* __restrict__ left,
                                                            const int32_t* __restrict__ right,
                                                            const uint32_t* __restrict__ cnt,
                                                            uint32_t* __restrict__ arrivals,
                                                            int32_t* __restrict__ list, uint32_t* __restrict__ count,
                                                            uint64_t* __restrict__ queue,
                                                            uint32_t* __restrict__ queue_size) {
    __shared__ uint32_t s_at, s_base, s_above, s_above_base;
    if (n == 1 || cnt[0] <= kSubtree) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            list[0] = n == 1 ? -1 : 0;
            *count = 1;
        }
        return;
    }
    const uint32_t first = blockIdx.x * kFindNodes;
    uint32_t above = 0;  // bit t: this thread's t-th node lies above the listed subtrees
    uint32_t want = 0;
    if (threadIdx.x == 0) s_at = s_above = 0;
    __syncthreads();
#pragma unroll
    for (uint32_t t = 0; t < kFindNodes / 256u; ++t) {
        const uint32_t i = first + t * 256u + threadIdx.x;
        if (i >= n - 1 || cnt[i] <= kSubtree) continue;
        arrivals[i] = 0;
        above |= 1u << t;
        const int32_t l = left[i], r = right[i];
        want += (l < 0 || cnt[l] <= kSubtree ? 1u : 0u) + (r < 0 || cnt[r] <= kSubtree ? 1u : 0u);
    }
    uint32_t at = want ? atomicAdd(&s_at, want) : 0u;
    const uint32_t nabove = queue ? (uint32_t)__popc(above) : 0u;
    uint32_t qat = nabove ? atomicAdd(&s_above, nabove) : 0u;
    __syncthreads();
    if (threadIdx.x == 0) {
        s_base = s_at ? atomicAdd(count, s_at) : 0u;
        s_above_base = s_above ? atomicAdd(queue_size, s_above) : 0u;
    }
    __syncthreads();
    qat += s_above_base;
    for (uint32_t k = 0; k < nabove; ++k) queue[qat + k] = kNoTask;
    if (!want) return;
    at += s_base;
    for (; above; above &= above - 1u) {
        const uint32_t i = first + ((uint32_t)__ffs((int)above) - 1u) * 256u + threadIdx.x;
        const int32_t l = left[i], r = right[i];
        if (l < 0 || cnt[l] <= kSubtree) list[at++] = l;
        if (r < 0 || cnt[r] <= kSubtree) list[at++] = r;
    }
}

struct RefineArgs {
    uint32_t n;
    int32_t* left;
    int32_t* right;
    int32_t* parent;
    const uint32_t* order;
    const float* prim_boxes;  // boxes of the primitives, for the first pass; nullptr: nboxes holds the leaves' boxes
    float* nboxes;
    float* cost;
    uint32_t* cnt;
    uint32_t* hgt;
    uint32_t* arrivals;
    uint32_t min_prims;  // 0xFFFFFFFF: plain refit
    const uint32_t* node_blas;
    const int32_t* list;  // subtree roots and their number
    const uint32_t* count;
};

// Refit and refinement of the listed subtrees, one wave each.  A pass whose every node went through global memory
// (agent-scope loads that miss the L2, about 16 dependent ones per treelet) took 18.0 and 12.3 ms for the two rounds on
// 15.5M triangles, 4.4 ms for the first one on 4M; here the links and boxes of a subtree are read once.  What bounds it
// now: the instructions of the treelets (about 600 VALU and 450 SALU each) at four waves per SIMD.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void subtree_refine_kernel(RefineArgs a) {
    __shared__ SubtreeLds U;
    __shared__ float ubox[2 * kSubtree][6];
    __shared__ TreeletLds T;
    __shared__ float ucost[kSubtree], uarea[kSubtree];
    __shared__ uint32_t ucnt[kSubtree], uhgt[kSubtree];
    const uint32_t lane = threadIdx.x;
    SplitRegs sr;
    load_splits(sr);
    const uint32_t count = *a.count;
    for (uint32_t ti = blockIdx.x; ti < count; ti += gridDim.x) {
        const int32_t root = a.list[ti];
        if (root < 0) {
            if (a.prim_boxes && lane < 6u) {
                const uint64_t pos = (uint64_t)(-1 - root);
                a.nboxes[6 * ((uint64_t)a.n - 1 + pos) + lane] = a.prim_boxes[6 * (uint64_t)a.order[pos] + lane];
            }
            continue;
        }
        uint32_t nint, nleaf, nlevel;
        load_subtree(U, root, a.left, a.right, nint, nleaf, nlevel);
        for (uint32_t i = lane; i < nleaf; i += 64u) {
            const uint64_t pos = (uint64_t)(-1 - U.code[kSubtree + i]);
            float* nb = a.nboxes + 6 * ((uint64_t)a.n - 1 + pos);
            const float* src = a.prim_boxes ? a.prim_boxes + 6 * (uint64_t)a.order[pos] : nb;
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                const float v = src[k];
                ubox[kSubtree + i][k] = v;
                if (a.prim_boxes) nb[k] = v;
            }
        }
        __syncthreads();
        auto children = [&](int32_t c, int32_t& l, int32_t& r, float& al, float& ar) {
            const uint32_t k = U.kids[c];
            const uint32_t kl = k & 0xFFFFu, kr = k >> 16;
            // leaves as negative codes: -1 - local id
            l = kl >= kSubtree ? -1 - (int32_t)kl : (int32_t)kl;
            r = kr >= kSubtree ? -1 - (int32_t)kr : (int32_t)kr;
            al = kl >= kSubtree ? -1.0f : uarea[kl];
            ar = kr >= kSubtree ? -1.0f : uarea[kr];
        };
        for (uint32_t lv = nlevel; lv-- > 0;) {
            const uint32_t end = U.level[lv + 1];
            for (uint32_t at = U.level[lv]; at < end; at += 64u) {
                const uint32_t x = at + lane;
                bool need = false;
                float ccost = 0.0f;
                uint32_t chgt = 0;
                if (x < end) {
                    const uint32_t k = U.kids[x], l = k & 0xFFFFu, r = k >> 16;
                    float b[6];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        b[c] = fminf(ubox[l][c], ubox[r][c]);
                        b[3 + c] = fmaxf(ubox[l][3 + c], ubox[r][3 + c]);
                    }
#pragma unroll
                    for (int c = 0; c < 6; ++c) ubox[x][c] = b[c];
                    const bool il = l < kSubtree, ir = r < kSubtree;
                    const float area = box_area(b);
                    ccost = area + ((il ? ucost[l] : 0.0f) + (ir ? ucost[r] : 0.0f));
                    const uint32_t ccnt = (il ? ucnt[l] : 1u) + (ir ? ucnt[r] : 1u);
                    const uint32_t hl = il ? uhgt[l] : 0u, hr = ir ? uhgt[r] : 0u;
                    chgt = 1u + (hl > hr ? hl : hr);
                    ucost[x] = ccost;
                    uarea[x] = area;
                    ucnt[x] = ccnt;
                    uhgt[x] = chgt;
                    // batched builds never restructure across BLASes
                    need = ccnt >= a.min_prims && (!a.node_blas || a.node_blas[U.code[x]] != kMixedBlas);
                }
                __syncthreads();
                TreeletForm form;
                uint64_t todo = __ballot(need && treelet_form((int32_t)x, children, form));
                while (todo) {
                    const int L = __ffsll((unsigned long long)todo) - 1;
                    todo &= todo - 1;
                    const float rc = __shfl(ccost, L);
                    const uint32_t rh = (uint32_t)__shfl((int)chgt, L);
                    if ((int)lane == L) stage_form(T, form);
                    __syncthreads();
                    if (lane < (uint32_t)kTreeletLeaves) {
                        const int32_t c = T.leaf[lane];
                        const uint32_t id = c >= 0 ? (uint32_t)c : (uint32_t)(-1 - c);
                        T.leaf[lane] = (int32_t)id;
#pragma unroll
                        for (int k = 0; k < 6; ++k) T.box[lane][k] = ubox[id][k];
                        T.cost[1u << lane] = c >= 0 ? ucost[id] : 0.0f;
                        T.lcnt[lane] = c >= 0 ? ucnt[id] : 1u;
                        T.lhgt[lane] = c >= 0 ? uhgt[id] : 0u;
                    }
                    __syncthreads();
                    const TreeletPlan plan = treelet_solve(T, sr, rc, rh);
                    if (plan.commit && lane < kTreeletNodes) {
                        const uint32_t y = (uint32_t)T.pool[lane];
                        U.kids[y] = (uint32_t)plan_child(T, plan, lane, 0) | (uint32_t)plan_child(T, plan, lane, 1) << 16;
                        uhgt[y] = (uint32_t)(plan.heights >> (8 * lane)) & 255u;
                        if (lane == 0) {
                            ucost[y] = plan.total;
                        } else {
                            const uint32_t S = (uint32_t)(plan.sets >> (8 * lane)) & 127u;
                            float b[6];
                            ucnt[y] = plan_bounds(T, S, b);
#pragma unroll
                            for (int k = 0; k < 6; ++k) ubox[y][k] = b[k];
                            uarea[y] = box_area(b);
                            ucost[y] = T.cost[S];
                        }
                    }
                    __syncthreads();
                }
            }
        }
        for (uint32_t i = lane; i < nint; i += 64u) {
            const int32_t x = U.code[i];
            const uint32_t k = U.kids[i];
            const int32_t c0 = U.code[k & 0xFFFFu], c1 = U.code[k >> 16];
            a.left[x] = c0;
            a.right[x] = c1;
            a.parent[node_index(a.n, c0)] = x;
            a.parent[node_index(a.n, c1)] = x;
#pragma unroll
            for (int c = 0; c < 6; ++c) a.nboxes[6 * (uint64_t)x + c] = ubox[i][c];
            a.cost[x] = ucost[i];
            a.cnt[x] = ucnt[i];
            a.hgt[x] = uhgt[i];
        }
    }
}

// Treelet refinement rounds: default kTreeletRounds, none under PREFER_FAST_BUILD, RTX_BUILD_TREELET_ROUNDS_*
// overrides both, NO_TREELET disables; round r restructures nodes with at least kTreeletMinPrims[r] primitives.
// (The two rounds take 12 ms on 15.5M triangles; each buys 0.5-1.5% of closest-hit speed on the query scenes.)
constexpr int kTreeletRounds = 2;
constexpr uint32_t kTreeletMinPrims[3] = {7, 14, 28};
int treelet_rounds(uint32_t flags, uint32_t n) {
    if ((flags & RTX_BUILD_NO_TREELET_BIT) || n < (uint32_t)kTreeletLeaves) return 0;
    const uint32_t r = (flags >> RTX_BUILD_TREELET_ROUNDS_SHIFT) & 3u;
    if (r) return (int)r;
    return (flags & RTX_BUILD_PREFER_FAST_BUILD_BIT) ? 0 : kTreeletRounds;
}

// Refit and refinement of the nodes above the listed subtrees, one wave per block, one subtree per lane; with no list
// (an update's refit, whose kept hierarchy has no counts) of the whole tree, one leaf per lane.
__global__ __launch_bounds__(64) void refit_refine_kernel(RefineArgs a) {
    __shared__ TreeletLds T;
    const uint32_t lane = threadIdx.x;
    const uint32_t n = a.n;
    SplitRegs sr;
    load_splits(sr);
    auto children = [&](int32_t c, int32_t& l, int32_t& r, float& al, float& ar) {
        l = load_coherent_i32(a.left + c);
        r = load_coherent_i32(a.right + c);
        al = l >= 0 ? coherent_area(a.nboxes, (uint64_t)l) : -1.0f;
        ar = r >= 0 ? coherent_area(a.nboxes, (uint64_t)r) : -1.0f;
    };
    // a wave takes a batch of subtrees: as few as the waves of the launch allow, since it works on its lanes' treelets
    // one after another
    const uint32_t count = a.list ? *a.count : n;
    const uint32_t share = (count - 1u) / gridDim.x + 1u;
    const uint32_t batch = a.list && share < 64u ? share : 64u;
    for (uint32_t first = blockIdx.x * batch; first < count; first += gridDim.x * batch) {
        bool active = lane < batch && first + lane < count;
        float cur[6] = {0, 0, 0, 0, 0, 0};
        float ccost = 0.0f;
        uint32_t ccnt = 1, chgt = 0;
        uint64_t self = 0;
        int32_t node = -1;
        if (active) {
            const int32_t c = a.list ? a.list[first + lane] : -1 - (int32_t)(first + lane);
            self = node_index(n, c);
            const float* src = a.list ? a.nboxes + 6 * self : a.prim_boxes + 6 * (uint64_t)a.order[first + lane];
#pragma unroll
            for (int k = 0; k < 6; ++k) cur[k] = src[k];
            if (!a.list) {
#pragma unroll
                for (int k = 0; k < 6; ++k) store_coherent(a.nboxes + 6 * self + k, cur[k]);
            }
            if (c >= 0) {
                ccost = a.cost[c];
                ccnt = a.cnt[c];
                chgt = a.hgt[c];
            }
            node = load_coherent_i32(a.parent + self);
        }
        // the vote stands in the loop's single latch: with two latches (after the last `if`, and past it) the compiler
        // may nest the loop, and the lanes without a node would leave it while the others still work as a wave
        for (bool any = __any(active); any; any = __any(active)) {
            bool own = false;
            if (active) {
                if (node < 0) {
                    active = false;
                } else {
                    __atomic_signal_fence(__ATOMIC_SEQ_CST);
                    __builtin_amdgcn_s_waitcnt(0);
                    __atomic_signal_fence(__ATOMIC_SEQ_CST);
                    const uint32_t old = __hip_atomic_fetch_add(&a.arrivals[node], 1u, __ATOMIC_RELAXED,
                                                                __HIP_MEMORY_SCOPE_AGENT);
                    if (old == 0u) {
                        active = false;
                    } else {
                        own = true;
                        const int32_t l = load_coherent_i32(a.left + node), r = load_coherent_i32(a.right + node);
                        const uint64_t li = node_index(n, l), ri = node_index(n, r);
                        const bool self_left = li == self;
                        const int32_t sc = self_left ? r : l;
                        const uint64_t sib = self_left ? ri : li;
                        const float scost = sc >= 0 ? load_coherent(a.cost + sc) : 0.0f;
                        const uint32_t scnt = sc >= 0 ? load_coherent_u32(a.cnt + sc) : 1u;
                        const uint32_t shgt = sc >= 0 ? load_coherent_u32(a.hgt + sc) : 0u;
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            cur[k] = fminf(cur[k], load_coherent(a.nboxes + 6 * sib + k));
                            cur[3 + k] = fmaxf(cur[3 + k], load_coherent(a.nboxes + 6 * sib + 3 + k));
                        }
                        const float cl = self_left ? ccost : scost, cr = self_left ? scost : ccost;
                        ccost = box_area(cur) + (cl + cr);
                        ccnt += scnt;
                        chgt = 1u + (chgt > shgt ? chgt : shgt);
                    }
                }
            }
            // batched builds never restructure across BLASes
            const bool root = own && ccnt >= a.min_prims && (!a.node_blas || a.node_blas[node] != kMixedBlas);
            // every lane with a treelet root forms its treelet at once (the dependent child / box loads overlap),
            // then the wave restructures them one after another
            TreeletForm form;
            uint64_t need = __ballot(root && treelet_form(node, children, form));
            while (need) {
                const int L = __ffsll((unsigned long long)need) - 1;
                need &= need - 1;
                const float rc = __shfl(ccost, L);
                const uint32_t rh = (uint32_t)__shfl((int)chgt, L);
                float nc;
                uint32_t nh;
                treelet_optimize(T, sr, n, rc, rh, (uint32_t)L, form, a.left, a.right, a.parent, a.nboxes, a.cost,
                                 a.cnt, a.hgt, nc, nh);
                if ((int)lane == L) {
                    ccost = nc;
                    chgt = nh;
                }
            }
            if (own) {
#pragma unroll
                for (int k = 0; k < 6; ++k) store_coherent(a.nboxes + 6 * (uint64_t)node + k, cur[k]);
                store_coherent(a.cost + node, ccost);
                store_coherent_u32(a.cnt + node, ccnt);
                store_coherent_u32(a.hgt + node, chgt);
                self = (uint64_t)node;
                node = load_coherent_i32(a.parent + node);
            }
        }
    }
}

// ---- costs of the 8-wide collapse ------------------------------------------------------------------------------
//
// The SAH-optimal collapse of the binary tree into 8-wide nodes (Ylitie, Karras & Laine 2017, section 4), for
// this layout's leaves (one primitive per child slot).  C(x, j), j = 1..8, is the least cost of the subtree of
// x spread over at most j child slots of its parent:
//   leaf:      C(x, j) = c_leaf * A(x)
//   internal:  D(x, j) = min over k in [1, j-1] of C(l, k) + C(r, j - k)        (x dissolved into j slots)
//              C(x, 1) = A(x) + D(x, W)                                         (x becomes a wide node)
//              C(x, j) = min(C(x, j - 1), D(x, j)),  j >= 2
// computed bottom-up: the listed subtrees a wave each in LDS, then the nodes above (second arrival merges, as the
// refit).  The collapse then takes, for each wide node x, the children that D(x, W) picks.  W is the build's node width
// (8, or 2..7 from RTX_BUILD_MAX_WIDTH): narrower trees use the same 64-B node with fewer children.
//
// wdec[x], 4 bits for each j = 2..8: the left child's slot count k that D(x, j) takes, and 8 where D(x, j) beats
// C(x, j - 1).  Along with the costs go the slots that the choice takes in all (the primitives with a box and the wide
// nodes) and its depth in wide nodes, so that the collapse of a subtree knows its place before it starts: sub[x], for
// the nodes of the listed subtrees: slots below x as a wide node (8 bits) | wide nodes from x down << 8 | depth << 16.
__device__ __forceinline__ bool box_valid(const float* b) { return b[0] <= b[3] && b[1] <= b[4] && b[2] <= b[5]; }

struct WideRow {
    float c[8];
    uint64_t slots, depth;  // a byte for each j (slots: listed subtrees only)
};

// Row j = 2..W.. of x from its children's rows; returns wdec, and in `dissolved` the row of D(x, W).
__device__ __forceinline__ uint32_t wide_merge(const WideRow& l, const WideRow& r, float area, bool valid, int width,
                                               WideRow& out, uint32_t& slots_below) {
    float d[9];
    uint32_t k[9];
    uint32_t dec = 0;
#pragma unroll
    for (int j = 2; j <= 8; ++j) {
        d[j] = INFINITY;
        k[j] = 1;
#pragma unroll
        for (int i = 1; i < j; ++i) {
            const float c = l.c[i - 1] + r.c[j - i - 1];
            if (c < d[j]) {
                d[j] = c;
                k[j] = (uint32_t)i;
            }
        }
    }
    float dw = d[8];
    uint32_t kw = k[8];
#pragma unroll
    for (int j = 2; j < 8; ++j)
        if (j == width) {
            dw = d[j];
            kw = k[j];
        }
    auto at = [](uint64_t v, uint32_t j) { return (uint32_t)(v >> (8 * (j - 1))) & 255u; };
    auto both = [&](uint32_t j, uint32_t kk, uint32_t& sl, uint32_t& de) {
        sl = at(l.slots, kk) + at(r.slots, j - kk);
        const uint32_t a = at(l.depth, kk), b = at(r.depth, j - kk);
        de = a > b ? a : b;
    };
    uint32_t sl, de;
    both((uint32_t)width, kw, sl, de);
    slots_below = sl;
    sl = valid ? 1u + sl : 0u;
    de = valid ? 1u + de : 0u;
    out.c[0] = area + dw;
    out.slots = sl;
    out.depth = de;
#pragma unroll
    for (uint32_t j = 2; j <= 8; ++j) {
        const bool split = d[j] < out.c[j - 2];
        dec |= (k[j] | (split ? 8u : 0u)) << (4 * (j - 2));
        out.c[j - 1] = fminf(out.c[j - 2], d[j]);
        if (split) both(j, k[j], sl, de);
        out.slots |= (uint64_t)(sl & 255u) << (8 * (j - 1));
        out.depth |= (uint64_t)(de & 255u) << (8 * (j - 1));
    }
    return dec;
}

__device__ __forceinline__ void wide_leaf(const float* b, float c_leaf, WideRow& t) {
    const float a = c_leaf * box_area(b);
#pragma unroll
    for (int j = 0; j < 8; ++j) t.c[j] = a;
    t.slots = box_valid(b) ? 0x0101010101010101ull : 0ull;
    t.depth = 0;
}

struct CostArgs {
    uint32_t n;
    const int32_t* left;
    const int32_t* right;
    const int32_t* parent;
    const float* nboxes;
    float* wc;        // rows of the listed roots and the nodes above: 8 costs, and the depths
    uint64_t* depths;
    uint32_t* wdec;
    uint32_t* sub;
    uint32_t* arrivals;
    float c_leaf;
    int width;
    const int32_t* list;
    const uint32_t* count;
};

// (The two passes took 1.2 ms on 4M triangles through global memory, node by node; 0.24 + 0.08 ms.)
__global__ __launch_bounds__(64) void subtree_cost_kernel(CostArgs a) {
    __shared__ SubtreeLds U;
    __shared__ WideRow row[kSubtree];
    __shared__ float leaf_cost[kSubtree];  // negative: no box
    __shared__ uint8_t leaves[kSubtree];   // primitives with a box below each node
    const uint32_t lane = threadIdx.x;
    const uint32_t count = *a.count;
    for (uint32_t ti = blockIdx.x; ti < count; ti += gridDim.x) {
        const int32_t root = a.list[ti];
        if (root < 0) continue;
        uint32_t nint, nleaf, nlevel;
        load_subtree(U, root, a.left, a.right, nint, nleaf, nlevel);
        for (uint32_t i = lane; i < nleaf; i += 64u) {
            float b[6];
            const float* src = a.nboxes + 6 * ((uint64_t)a.n - 1 + (uint64_t)(-1 - U.code[kSubtree + i]));
#pragma unroll
            for (int k = 0; k < 6; ++k) b[k] = src[k];
            leaf_cost[i] = box_valid(b) ? a.c_leaf * box_area(b) : -1.0f;
        }
        __syncthreads();
        for (uint32_t lv = nlevel; lv-- > 0;) {
            const uint32_t end = U.level[lv + 1];
            for (uint32_t x = U.level[lv] + lane; x < end; x += 64u) {
                const int32_t code = U.code[x];
                float b[6];
#pragma unroll
                for (int k = 0; k < 6; ++k) b[k] = a.nboxes[6 * (uint64_t)code + k];
                WideRow t[2];
                uint32_t nl = 0;
                const uint32_t kids = U.kids[x];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t c = h ? kids >> 16 : kids & 0xFFFFu;
                    if (c < kSubtree) {
                        t[h] = row[c];
                        nl += leaves[c];
                    } else {
                        const float lc = leaf_cost[c - kSubtree];
#pragma unroll
                        for (int j = 0; j < 8; ++j) t[h].c[j] = lc < 0.0f ? 0.0f : lc;
                        t[h].slots = lc < 0.0f ? 0ull : 0x0101010101010101ull;
                        t[h].depth = 0;
                        nl += lc < 0.0f ? 0u : 1u;
                    }
                }
                WideRow o;
                uint32_t below;
                a.wdec[code] = wide_merge(t[0], t[1], box_area(b), box_valid(b), a.width, o, below);
                a.sub[code] = below | (1u + below - nl) << 8 | ((uint32_t)o.depth & 255u) << 16;
                row[x] = o;
                leaves[x] = (uint8_t)nl;
                if (x == 0) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) a.wc[8 * (uint64_t)code + j] = o.c[j];
                    a.depths[code] = o.depth;
                }
            }
            __syncthreads();
        }
    }
}

__global__ __launch_bounds__(64) void wide_cost_kernel(CostArgs a) {
    const uint32_t count = *a.count;
    auto load_row = [&](int32_t c, WideRow& t) {
        if (c < 0) {
            float b[6];
            const uint64_t bi = node_index(a.n, c);
#pragma unroll
            for (int k = 0; k < 6; ++k) b[k] = a.nboxes[6 * bi + k];
            wide_leaf(b, a.c_leaf, t);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) t.c[j] = load_coherent(a.wc + 8 * (uint64_t)c + j);
            t.depth = __hip_atomic_load(a.depths + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        t.slots = 0;
    };
    for (uint32_t at = blockIdx.x * 64u + threadIdx.x; at < count; at += gridDim.x * 64u) {
        int32_t node = a.parent[node_index(a.n, a.list[at])];
        while (node >= 0) {
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_s_waitcnt(0);
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            const uint32_t old =
                __hip_atomic_fetch_add(&a.arrivals[node], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (old == 0u) break;  // the sibling's thread merges
            WideRow l, r, o;
            load_row(a.left[node], l);
            load_row(a.right[node], r);
            float b[6];
#pragma unroll
            for (int k = 0; k < 6; ++k) b[k] = a.nboxes[6 * (uint64_t)node + k];
            uint32_t below;
            a.wdec[node] = wide_merge(l, r, box_area(b), box_valid(b), a.width, o, below);  // read by later launches
#pragma unroll
            for (int j = 0; j < 8; ++j) store_coherent(a.wc + 8 * (uint64_t)node + j, o.c[j]);
            __hip_atomic_store(a.depths + node, o.depth, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            node = a.parent[node];
        }
    }
}

// ---- collapse tasks ---------------------------------------------------------------------------------------------
//
// The wide nodes above the listed subtrees go through a queue: a task is (binary node, slot) in one 64-bit word, its
// place empty (kNoTask) until it is published.  `open` counts the tasks published and not yet done.  The subtrees
// below come in a second list, each with the place of its slots.
struct CollapseQueue {
    uint32_t head, pad0[31];
    uint32_t tail, pad1[31];
    uint32_t open, pad2[31];
    uint32_t subs, pad3[31];
};
static_assert(sizeof(CollapseQueue) == 512, "the scratch layout's queue words");
__device__ __forceinline__ uint64_t pack_task(int32_t node, uint32_t slot) {
    return (uint32_t)node | (uint64_t)slot << 32;
}

// Root of a structure (header fields set, slot 0): its subtree task or its queue task, and what the header says of it.
__device__ void push_root(AsHeader* h, int32_t root, uint32_t blas, const uint32_t* cnt, const uint32_t* sub,
                          const uint64_t* depths, CollapseQueue* q, uint64_t* queue, uint4* subs) {
    if (root < 0 || cnt[root] <= kSubtree) {
        const uint32_t w = root < 0 ? 1u | 1u << 8 | 1u << 16 : sub[root];
        h->slot_count = 1u + (w & 255u);
        h->node_count = w >> 8 & 255u;
        h->max_depth = w >> 16 & 255u;
        subs[atomicAdd(&q->subs, 1u)] = make_uint4((uint32_t)root, 0u, 1u, blas);
        return;
    }
    h->slot_count = 1u;
    h->max_depth = (uint32_t)depths[root] & 255u;
    atomicAdd(&q->open, 1u);
    queue[atomicAdd(&q->tail, 1u)] = pack_task(root, 0u);
}

// Header setup after refit: root box and the 16-bit origin quantisation step.
__global__ void header_kernel(AsHeader* h, uint32_t type, uint32_t flags, uint32_t n, uint32_t ngeom,
                              const float* nboxes, const float* cost, uint64_t capacity_slots, uint64_t table_offset,
                              const uint32_t* cnt, const uint32_t* sub, const uint64_t* depths, CollapseQueue* q,
                              uint64_t* queue, uint4* subs) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    q->head = q->tail = q->open = q->subs = 0;
    h->magic = type ? kMagicTlas : kMagicBlas;
    h->version = kVersion;
    h->type = type;
    h->flags = flags;
    h->prim_count = n;
    h->geometry_count = ngeom;
    h->node_count = 0;
    h->slot_count = 0;
    h->max_depth = 0;
    h->max_total_depth = 0;
    h->build_error = 0;
    h->content = 0;
    h->slots_offset = kHeaderBytes;
    h->inst_table_offset = table_offset;
    h->capacity_slots = capacity_slots;
    h->sah_cost = 0.0;
    h->update_offset = 0;
    float lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
    if (n > 0) {
        const float* rb = (n == 1) ? nboxes + 0 : nboxes;  // root: internal 0, or leaf 0 when n == 1
        for (int a = 0; a < 3; ++a) {
            lo[a] = rb[a];
            hi[a] = rb[3 + a];
        }
    }
    bool empty = !(lo[0] <= hi[0]) || n == 0;
    if (n > 1) {
        const float ra = box_area(nboxes);
        h->sah_cost = ra > 0.0f ? (double)cost[0] / (double)ra : 0.0;
    }
    for (int a = 0; a < 3; ++a) {
        if (empty) {
            lo[a] = 0.0f;
            hi[a] = 0.0f;
        }
        h->lo[a] = lo[a];
        h->hi[a] = hi[a];
        float ext = hi[a] - lo[a];
        h->qscale[a] = ext > 0.0f ? ext / 65535.0f : 0.0f;
    }
    h->lo[3] = h->hi[3] = h->qscale[3] = 0.0f;
    if (empty) return;
    // root: internal node 0, or leaf 0 (code -1) when n == 1
    push_root(h, n == 1 ? -1 : 0, 0u, cnt, sub, depths, q, queue, subs);
}

__device__ __forceinline__ float exp_scale(uint32_t e) { return __uint_as_float(e << 23); }

// Quantisation frame of one axis: origin p (decoded from pq) and exponent byte e with fma(255, 2^e, p) >= hi.
__device__ void make_frame(float lo, float hi, float root_lo, float qscale, uint16_t& pq_out, float& p_out,
                           uint32_t& e_out) {
    uint32_t pq = 0;
    if (qscale > 0.0f) {
        float f = floorf((lo - root_lo) / qscale);
        pq = f <= 0.0f ? 0u : (f >= 65535.0f ? 65535u : (uint32_t)f);
        while (pq > 0 && fmaf((float)pq, qscale, root_lo) > lo) --pq;
    }
    float p = fmaf((float)pq, qscale, root_lo);
    uint32_t e = 1;  // 2^-126
    float x = (hi - p) / 255.0f;
    if (x > 0.0f) {
        int k;
        frexpf(x, &k);  // x = m * 2^k, m in [0.5, 1)
        int ee = k - 1 + 127;
        if (ee < 1) ee = 1;
        if (ee > 254) ee = 254;
        e = (uint32_t)ee;
        while (e < 254 && fmaf(255.0f, exp_scale(e), p) < hi) ++e;
    }
    pq_out = (uint16_t)pq;
    p_out = p;
    e_out = e;
}

__device__ __forceinline__ void quant_child(float clo, float chi, float p, uint32_t e, uint8_t& qlo, uint8_t& qhi) {
    float s = exp_scale(e);
    float fl = floorf((clo - p) / s);
    int ql = fl <= 0.0f ? 0 : (fl >= 255.0f ? 255 : (int)fl);
    while (ql > 0 && fmaf((float)ql, s, p) > clo) --ql;
    float fh = ceilf((chi - p) / s);
    int qh = fh <= 0.0f ? 0 : (fh >= 255.0f ? 255 : (int)fh);
    while (qh < 255 && fmaf((float)qh, s, p) < chi) ++qh;
    if (qh < ql) qh = ql;
    qlo = (uint8_t)ql;
    qhi = (uint8_t)qh;
}

// ---- wide nodes ---------------------------------------------------------------------------------------------------
//
// A wave makes 8 wide nodes at a time, 8 lanes each, a lane per child slot: it finds the children (collapse_walk), gives
// them their octant positions and slots, quantises their boxes and writes the node and its leaves.  A launch per level of
// the wide tree with a thread per node, 66 launches for the deepest tree there can be, took 1.75 ms on 4M triangles and
// 7.0 ms on 15.5M of 64 meshes: most of it a dozen atomics per wave on the same few header words.  Through the queue and
// by subtrees, whose slots are known beforehand, 0.20 + 0.77 ms and 0.6 + 4.4 ms.  The subtrees are bound by VALU
// (65% busy: 8-lane placement and IEEE divisions of the quantisation).
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
// lane patterns that reduce over 8 lanes: quad_perm [1, 0, 3, 2], [2, 3, 0, 1], then row_half_mirror
constexpr int kSwap1 = 0xB1, kSwap2 = 0x4E, kMirror8 = 0x141;
__device__ __forceinline__ float min8(float v) {
    v = fminf(v, dpp_f<kSwap1>(v));
    v = fminf(v, dpp_f<kSwap2>(v));
    return fminf(v, dpp_f<kMirror8>(v));
}
__device__ __forceinline__ float max8(float v) {
    v = fmaxf(v, dpp_f<kSwap1>(v));
    v = fmaxf(v, dpp_f<kSwap2>(v));
    return fmaxf(v, dpp_f<kMirror8>(v));
}
template <int CTRL>
__device__ __forceinline__ void best8_step(float& score, uint32_t& id) {
    const float os = dpp_f<CTRL>(score);
    const uint32_t oi = dpp_u<CTRL>(id);
    if (os > score || (os == score && oi >> 3 > id >> 3)) {
        score = os;
        id = oi;
    }
}

struct WideLds {
    uint32_t item[8][8];   // a lane's part of the wide node being dissolved, and its slots
    uint32_t slots[8][8];
    alignas(16) uint8_t node[8][64];
};

// The children D(x, W) picks for the node x of each group (`on`), a child per lane (item; kNoItem: none).  A lane's part
// takes the slots from its own on: a part dissolved over j slots leaves its left child, which takes k of them, in the
// lane, and its right child k lanes on.  parts(x, l, r, dec): children and choices of an internal part, false for a leaf.
constexpr uint32_t kNoItem = 0x80000000u;  // no local id and no code: leaf codes start at -(2^30 - 1)
template <typename Parts>
__device__ __forceinline__ uint32_t collapse_walk(WideLds& W, uint32_t x, bool on, uint32_t width, Parts parts) {
    const uint32_t g = threadIdx.x >> 3, c = threadIdx.x & 7u;
    W.item[g][c] = on && c == 0 ? x : kNoItem;
    W.slots[g][c] = width;
    __syncthreads();
    bool root = true;
    for (bool more = true; more;) {
        const uint32_t it = W.item[g][c];
        uint32_t j = W.slots[g][c];
        bool split = false;
        uint32_t l = 0, r = 0, dec = 0, k = 0;
        if (it != kNoItem && (root || j > 1u) && parts(it, l, r, dec)) {
            // fewer slots cost no more: take one less (the node itself is always dissolved)
            while (!root && j > 1u && !(dec >> (4u * (j - 2u)) & 8u)) --j;
            split = j > 1u;
            if (split) k = dec >> (4u * (j - 2u)) & 7u;
        }
        __syncthreads();
        if (split) {
            W.item[g][c] = l;
            W.slots[g][c] = k;
            W.item[g][c + k] = r;
            W.slots[g][c + k] = j - k;
        } else if (it != kNoItem) {
            W.slots[g][c] = 1u;
        }
        __syncthreads();
        root = false;
        more = __any(split);
    }
    return W.item[g][c];
}

// Octant positions of the valid children (greedy assignment by centroid direction: the best (child, position) pair
// first, the higher lane of equal ones) and the box of the node.
__device__ __forceinline__ void place_children(bool valid, const float* b, uint32_t& pos, uint32_t& used, float* nlo,
                                               float* nhi) {
    const uint32_t g = threadIdx.x >> 3, c = threadIdx.x & 7u;
    float d[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        nlo[a] = min8(valid ? b[a] : INFINITY);
        nhi[a] = max8(valid ? b[3 + a] : -INFINITY);
        d[a] = 0.5f * (b[a] + b[3 + a]) - 0.5f * (nlo[a] + nhi[a]);
    }
    float sc[8];
#pragma unroll
    for (int p = 0; p < 8; ++p) sc[p] = ((p & 1) ? d[0] : -d[0]) + ((p & 2) ? d[1] : -d[1]) + ((p & 4) ? d[2] : -d[2]);
    pos = 8;
    used = 0;
    for (;;) {
        float best = -INFINITY;
        uint32_t id = c << 3;
        if (valid && pos == 8u) {
#pragma unroll
            for (uint32_t p = 0; p < 8; ++p)
                if (!(used & (1u << p)) && sc[p] > best) {
                    best = sc[p];
                    id = c << 3 | p;
                }
        }
        best8_step<kSwap1>(best, id);
        best8_step<kSwap2>(best, id);
        best8_step<kMirror8>(best, id);
        const bool found = best > -INFINITY;
        if (!__any(found)) break;
        if (found) {
            if (c == id >> 3) pos = id & 7u;
            used |= 1u << (id & 7u);
        }
    }
    // children whose centroid overflows have no direction: the free positions in order
    for (uint64_t left; (left = __ballot(valid && pos == 8u)) != 0ull;) {
        const uint32_t m = (uint32_t)(left >> (8u * g)) & 255u;
        const uint32_t free = (uint32_t)__ffs((int)(~used & 255u)) - 1u;
        if (m) {
            if (c == (uint32_t)__ffs((int)m) - 1u) pos = free;
            used |= 1u << free;
        }
    }
}

// Quantises the children of each group and writes its node to slots[4 slot ..] (on), child slots from `base`.
__device__ __forceinline__ void write_node(WideLds& W, bool on, uint4* slots, uint32_t slot, uint32_t base, bool valid,
                                           const float* b, uint32_t pos, uint32_t used, bool internal, const float* nlo,
                                           const float* nhi, const float* rlo, const float* qs) {
    const uint32_t g = threadIdx.x >> 3, c = threadIdx.x & 7u;
    float p[3];
    uint32_t e[3];
    uint16_t pq[3];
    if (on) {
#pragma unroll
        for (int a = 0; a < 3; ++a) make_frame(nlo[a], nhi[a], rlo[a], qs[a], pq[a], p[a], e[a]);
    }
    *(uint64_t*)(W.node[g] + 8u * c) = 0ull;
    __syncthreads();
    uint32_t im = valid && internal ? 1u << pos : 0u;
    im |= dpp_u<kSwap1>(im);
    im |= dpp_u<kSwap2>(im);
    im |= dpp_u<kMirror8>(im);
    if (valid) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            uint8_t ql, qh;
            quant_child(b[a], b[3 + a], p[a], e[a], ql, qh);
            W.node[g][16 + 8 * a + pos] = ql;
            W.node[g][40 + 8 * a + pos] = qh;
        }
    }
    __syncthreads();
    // Node8 layout: pq[3] (bytes 0-5), e[3] (6-8), imask (9), vmask (10), pad (11), base (12-15),
    // qlo[3][8] (16-39), qhi[3][8] (40-63)
    if (on && c < 4u) {
        uint4 w = *(const uint4*)(W.node[g] + 16u * c);
        if (c == 0)
            w = make_uint4((uint32_t)pq[0] | (uint32_t)pq[1] << 16, (uint32_t)pq[2] | e[0] << 16 | e[1] << 24,
                           e[2] | im << 8 | used << 16, base);
        slots[4 * (uint64_t)slot + c] = w;
    }
    __syncthreads();
}

__device__ __forceinline__ void copy_leaf(uint4* slots, uint32_t slot, const uint4* __restrict__ leaf_src,
                                          uint32_t prim) {
    const uint4* src = leaf_src + 4 * (uint64_t)prim;
    uint4* dst = slots + 4 * (uint64_t)slot;
    const uint4 w0 = src[0], w1 = src[1], w2 = src[2], w3 = src[3];
    dst[0] = w0;
    dst[1] = w1;
    dst[2] = w2;
    dst[3] = w3;
}

struct CollapseArgs {
    uint32_t n;
    const int32_t* left;
    const int32_t* right;
    const uint32_t* order;
    const float* nboxes;
    const uint4* leaf_src;
    const uint32_t* cnt;
    const uint32_t* wdec;
    const uint32_t* sub;
    AsHeader* h;                // single builds
    AsHeader* const* as_ptr;    // batched builds
    const uint32_t* node_blas;
    CollapseQueue* q;
    uint64_t* queue;
    const uint32_t* queue_size;
    uint4* subs;
    uint32_t* err;
    uint32_t width;
};

__device__ __forceinline__ void node_box(const CollapseArgs& a, int32_t code, float* b) {
    const float* src = a.nboxes + 6 * node_index(a.n, code);
#pragma unroll
    for (int k = 0; k < 6; ++k) b[k] = src[k];
}

// The wide nodes above the subtrees.  Waves of 8 groups; a group holds a ticket of the queue and works on the task of
// that place once it is published.  A wave never waits while it has a task, and a place that stays empty belongs to a
// node that a running wave is still about to reach, or to none (open = 0), so the waits end; a bound on them
// (kQueueSpins) turns a mistake into an error flag.
constexpr uint32_t kQueueSpins = 1u << 20;
template <bool BATCHED>
__global__ __launch_bounds__(64) void collapse_top_kernel(CollapseArgs a) {
    __shared__ WideLds W;
    const uint32_t lane = threadIdx.x, g = lane >> 3, c = lane & 7u;
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t limit = *a.queue_size;
    if (limit == 0) return;
    uint32_t ticket = kNoItem;
    uint32_t nodes = 0, spins = 0;
    auto parts = [&](uint32_t x, uint32_t& l, uint32_t& r, uint32_t& dec) {
        if ((int32_t)x < 0) return false;
        l = (uint32_t)a.left[x];
        r = (uint32_t)a.right[x];
        dec = a.wdec[x];
        return true;
    };
    for (;;) {
        // a ticket for each group without one
        const uint64_t none = __ballot(ticket == kNoItem && c == 0);
        if (none) {
            uint32_t t = 0;
            if (lane == 0) t = atomicAdd(&a.q->head, (uint32_t)__popcll(none));
            t = __shfl(t, 0);
            if (ticket == kNoItem) ticket = t + (uint32_t)__popcll(none & ((1ull << (8u * g)) - 1ull));
        }
        const uint32_t open = __hip_atomic_load(&a.q->open, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t task = ticket < limit
                                  ? __hip_atomic_load(a.queue + ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                  : kNoTask;
        const bool on = task != kNoTask;
        const uint64_t onm = __ballot(on && c == 0);
        if (!onm) {
            if (__shfl(open, 0) == 0u) break;
            if (++spins > kQueueSpins) {
                if (lane == 0) {
                    atomicOr(a.err, kErrCollapseTimeout);
                    if (!BATCHED) a.h->build_error = 1u;
                }
                break;
            }
            __builtin_amdgcn_s_sleep(4);
            continue;
        }
        spins = 0;
        const uint32_t x = (uint32_t)task, slot = (uint32_t)(task >> 32);
        const uint32_t blas = BATCHED && on ? a.node_blas[x] : 0u;
        AsHeader* h = BATCHED ? (on ? a.as_ptr[blas] : nullptr) : a.h;
        uint4* slots = (uint4*)((uint8_t*)h + kHeaderBytes);
        const uint32_t item = collapse_walk(W, x, on, a.width, parts);
        const int32_t code = (int32_t)item;
        float b[6] = {0, 0, 0, 0, 0, 0}, rlo[3] = {0, 0, 0}, qs[3] = {0, 0, 0};
        const bool child = on && item != kNoItem;
        bool valid = false;
        if (child) {
            node_box(a, code, b);
            valid = box_valid(b);
        }
        if (on) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                rlo[k] = h->lo[k];
                qs[k] = h->qscale[k];
            }
        }
        uint32_t pos, used;
        float nlo[3], nhi[3];
        place_children(valid, b, pos, used, nlo, nhi);
        const bool internal = valid && code >= 0;
        const bool small = internal && a.cnt[code] <= kSubtree;
        const uint32_t w = small ? a.sub[code] : 0u;
        const uint32_t size = w & 255u;  // slots below a subtree child
        // slots: the group's children, then the subtrees below them
        uint32_t run = size, wide = w >> 8 & 255u;
#pragma unroll
        for (int off = 1; off < 8; off <<= 1) {
            const uint32_t v = __shfl_up(run, off, 8);
            if ((int)c >= off) run += v;
            wide += __shfl_xor(wide, off, 8);
        }
        const uint32_t nvalid = (uint32_t)__popc(used);
        const uint32_t total = nvalid + __shfl(run, 7, 8);
        uint32_t base = 0;
        if (BATCHED) {
            if (on && c == 0) {
                base = atomicAdd(&h->slot_count, total);
                atomicAdd(&h->node_count, 1u + wide);
            }
            base = __shfl(base, 0, 8);
        } else {
            uint32_t before = 0, all = 0;
            for (uint32_t k = 0; k < 8; ++k) {
                const uint32_t v = __shfl(total, (int)(8 * k));
                before += k < g ? v : 0u;
                all += v;
            }
            if (lane == 0) base = atomicAdd(&h->slot_count, all);
            base = __shfl(base, 0) + before;
            nodes += on && c == 0 ? 1u + wide : 0u;
        }
        write_node(W, on, slots, slot, base, valid, b, pos, used, internal, nlo, nhi, rlo, qs);
        const uint32_t cslot = base + (uint32_t)__popc(used & ((1u << (pos & 7u)) - 1u));
        if (valid && code < 0) copy_leaf(slots, cslot, a.leaf_src, a.order[-1 - code]);
        const uint64_t sm = __ballot(small), tm = __ballot(internal && !small);
        if (sm) {
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(&a.q->subs, (uint32_t)__popcll(sm));
            at = __shfl(at, 0) + (uint32_t)__popcll(sm & below);
            if (small) a.subs[at] = make_uint4((uint32_t)code, cslot, base + nvalid + run - size, blas);
        }
        if (tm) {
            uint32_t at = 0;
            if (lane == 0) {
                // counted as open before anybody can see them
                atomicAdd(&a.q->open, (uint32_t)__popcll(tm));
                at = atomicAdd(&a.q->tail, (uint32_t)__popcll(tm));
            }
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __builtin_amdgcn_s_waitcnt(0);
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            at = __shfl(at, 0) + (uint32_t)__popcll(tm & below);
            if (internal && !small)
                __hip_atomic_store(a.queue + at, pack_task(code, cslot), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane == 0) atomicSub(&a.q->open, (uint32_t)__popcll(onm));
        if (on) ticket = kNoItem;
    }
    if (!BATCHED) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) nodes += __shfl_xor(nodes, off);
        if (lane == 0 && nodes) atomicAdd(&a.h->node_count, nodes);
    }
}

// The wide nodes of the listed subtrees, a wave each, breadth-first into the slots that the subtree was given.
template <bool BATCHED>
__global__ __launch_bounds__(64) void collapse_subtree_kernel(CollapseArgs a) {
    __shared__ SubtreeLds U;
    __shared__ WideLds W;
    __shared__ uint32_t udec[kSubtree];
    __shared__ uint32_t qslot[kSubtree];
    __shared__ uint16_t qnode[kSubtree];
    const uint32_t lane = threadIdx.x, g = lane >> 3;
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t count = a.q->subs;
    auto parts = [&](uint32_t x, uint32_t& l, uint32_t& r, uint32_t& dec) {
        if (x >= kSubtree) return false;
        l = U.kids[x] & 0xFFFFu;
        r = U.kids[x] >> 16;
        dec = udec[x];
        return true;
    };
    for (uint32_t ti = blockIdx.x; ti < count; ti += gridDim.x) {
        const uint4 task = a.subs[ti];
        AsHeader* h = BATCHED ? a.as_ptr[task.w] : a.h;
        uint4* slots = (uint4*)((uint8_t*)h + kHeaderBytes);
        float rlo[3], qs[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            rlo[k] = h->lo[k];
            qs[k] = h->qscale[k];
        }
        __syncthreads();
        uint32_t nint = 1, nleaf, nlevel;
        if ((int32_t)task.x < 0) {  // a structure of one primitive: a wide node with one child
            if (lane == 0) {
                U.code[kSubtree] = (int32_t)task.x;
                qnode[0] = (uint16_t)kSubtree;
            }
        } else {
            load_subtree(U, (int32_t)task.x, a.left, a.right, nint, nleaf, nlevel);
            for (uint32_t i = lane; i < nint; i += 64u) udec[i] = a.wdec[U.code[i]];
            if (lane == 0) qnode[0] = 0;
        }
        if (lane == 0) qslot[0] = task.y;
        __syncthreads();
        uint32_t head = 0, tail = 1, next = task.z;
        while (head < tail) {
            const bool on = head + g < tail;
            const uint32_t x = on ? qnode[head + g] : 0u, slot = on ? qslot[head + g] : 0u;
            const uint32_t item = collapse_walk(W, x, on, a.width, parts);
            float b[6] = {0, 0, 0, 0, 0, 0};
            bool valid = false;
            int32_t code = 0;
            if (on && item != kNoItem) {
                code = U.code[item];
                node_box(a, code, b);
                valid = box_valid(b);
            }
            uint32_t pos, used;
            float nlo[3], nhi[3];
            place_children(valid, b, pos, used, nlo, nhi);
            const uint64_t vm = __ballot(valid);
            const uint32_t base = next + (uint32_t)__popcll(vm & ((1ull << (8u * g)) - 1ull));
            next += (uint32_t)__popcll(vm);
            const bool internal = valid && code >= 0;
            write_node(W, on, slots, slot, base, valid, b, pos, used, internal, nlo, nhi, rlo, qs);
            const uint32_t cslot = base + (uint32_t)__popc(used & ((1u << (pos & 7u)) - 1u));
            if (valid && code < 0) copy_leaf(slots, cslot, a.leaf_src, a.order[-1 - code]);
            const uint64_t im = __ballot(internal);
            head = head + 8u < tail ? head + 8u : tail;
            if (internal) {
                const uint32_t at = tail + (uint32_t)__popcll(im & below);
                qnode[at] = (uint16_t)item;
                qslot[at] = cslot;
            }
            tail += (uint32_t)__popcll(im);
            __syncthreads();
        }
    }
}

// Batched builds: one thread per BLAS writes its header (as header_kernel) and queues its root task.
__global__ __launch_bounds__(64) void batch_header_kernel(AsHeader* const* __restrict__ as_ptr,
                                                          const uint2* __restrict__ binfo, uint32_t nbatch,
                                                          const int32_t* __restrict__ roots, uint32_t n,
                                                          uint32_t flags, const float* __restrict__ nboxes,
                                                          const float* __restrict__ cost,
                                                          const uint32_t* __restrict__ cnt,
                                                          const uint32_t* __restrict__ sub,
                                                          const uint64_t* __restrict__ depths, CollapseQueue* q,
                                                          uint64_t* queue, uint4* subs) {
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbatch) return;
    AsHeader* h = as_ptr[b];
    const uint32_t np = binfo[b].x;
    h->magic = kMagicBlas;
    h->version = kVersion;
    h->type = 0;
    h->flags = flags;
    h->prim_count = np;
    h->geometry_count = binfo[b].y;
    h->node_count = 0;
    h->slot_count = 0;
    h->max_depth = 0;
    h->max_total_depth = 0;
    h->build_error = 0;
    h->content = 0;
    h->slots_offset = kHeaderBytes;
    h->inst_table_offset = 0;
    h->capacity_slots = 2ull * (np ? np : 1) + 1;
    h->sah_cost = 0.0;
    h->update_offset = 0;
    const int32_t root = np ? roots[b] : 0x7FFFFFFF;
    float lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
    bool empty = root == 0x7FFFFFFF;
    if (!empty) {
        const float* rb = nboxes + 6 * (root >= 0 ? (uint64_t)root : (uint64_t)n - 1 + (uint64_t)(-1 - root));
        for (int a = 0; a < 3; ++a) {
            lo[a] = rb[a];
            hi[a] = rb[3 + a];
        }
        empty = !(lo[0] <= hi[0]);
        if (root >= 0) {
            const float ra = box_area(rb);
            h->sah_cost = ra > 0.0f ? (double)cost[root] / (double)ra : 0.0;
        }
    }
    for (int a = 0; a < 3; ++a) {
        if (empty) {
            lo[a] = 0.0f;
            hi[a] = 0.0f;
        }
        h->lo[a] = lo[a];
        h->hi[a] = hi[a];
        const float ext = hi[a] - lo[a];
        h->qscale[a] = ext > 0.0f ? ext / 65535.0f : 0.0f;
    }
    h->lo[3] = h->hi[3] = h->qscale[3] = 0.0f;
    if (empty) return;
    push_root(h, root, b, cnt, sub, depths, q, queue, subs);
}

__global__ void batch_finish_kernel(AsHeader* const* __restrict__ as_ptr, uint32_t nbatch) {
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < nbatch) as_ptr[b]->max_total_depth = as_ptr[b]->max_depth;
}

// Words that a batched build starts from: bounds and root of every BLAS, the counters and the collapse's queue (zero).
__global__ void init_batch_kernel(uint32_t* __restrict__ cb, int32_t* __restrict__ roots, uint32_t nbatch,
                                  uint32_t* __restrict__ misc, uint32_t* __restrict__ queue_words) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 6 * nbatch) cb[i] = (i % 6) < 3 ? 0xFFFFFFFFu : 0u;
    if (i < nbatch) roots[i] = 0x7FFFFFFF;
    if (i < 16u) misc[i] = 0u;
    if (i < sizeof(CollapseQueue) / 4) queue_words[i] = 0u;
}

__global__ void finish_tlas_kernel(AsHeader* h, const uint32_t* max_blas_depth) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        h->max_total_depth = h->max_depth + max_blas_depth[0];
        h->content = max_blas_depth[1];
    }
}

// BLAS content bits from its geometries (one thread per geometry; the header's word was zeroed by the header
// kernel): into `single`, or into as_ptr[geometry's BLAS] for batched builds.
__global__ void content_kernel(const GeomDesc* __restrict__ geoms, uint32_t ngeom, AsHeader* single,
                               AsHeader* const* __restrict__ as_ptr) {
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ngeom) return;
    const GeomDesc d = geoms[g];
    if (d.prim_count == 0) return;
    const uint32_t c = ((d.flags & RTX_GEOMETRY_OPAQUE_BIT) ? 0u : kContentNonOpaque) |
                       (d.type == RTX_GEOMETRY_TYPE_AABBS ? kContentAabb : 0u);
    if (c) atomicOr(&(single ? single : as_ptr[d.blas])->content, c);
}
__global__ void finish_blas_kernel(AsHeader* h) {
    if (threadIdx.x == 0 && blockIdx.x == 0) h->max_total_depth = h->max_depth;
}

__global__ void fill_kernel(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// One piece of a host array carried by value as a launch argument (a recorded launch keeps its arguments).
constexpr uint32_t kArgBlobWords = 256;
struct ArgBlob {
    uint32_t w[kArgBlobWords];
};
__global__ void arg_blob_kernel(ArgBlob b, uint32_t* __restrict__ dst, uint32_t words) {
    if (threadIdx.x < words) dst[threadIdx.x] = b.w[threadIdx.x];
}

// ---- scratch layout --------------------------------------------------------------------------------------------
struct Layout {
    uint64_t leaves, boxes, keys, vals, sort, left, right, parent, nboxes, arrivals, cost, cnt, hgt, wcost, wdec,
        subs, queue, queue_words, cbounds, misc, geoms, total;
    // batched builds only
    uint64_t pblas = 0, nblas = 0, roots = 0, asptr = 0, binfo = 0, bcb = 0;
    // space that is free again by the time of the bottom-up passes: subtree lists in the sort's scratch, sub words in
    // the keys, depths in the primitive boxes (which the first pass reads)
    uint64_t list() const { return sort; }
    uint64_t sub() const { return keys; }
    uint64_t depths() const { return boxes; }
};

Layout make_layout(uint32_t n, int key_bytes, uint32_t ngeom, uint32_t nbatch = 0) {
    Layout L;
    uint64_t o = 0;
    auto take = [&](uint64_t bytes) {
        uint64_t at = o;
        o += align_up(bytes ? bytes : 1, 256);
        return at;
    };
    uint64_t nn = n ? n : 1;
    L.leaves = take(nn * 64);
    L.boxes = take(nn * 24);
    L.keys = take(nn * key_bytes);
    L.vals = take(nn * 4);
    // The bounds, read by the Morton codes alone, lie where the sort will; its look-back words of small tiles (up to 6 B
    // a primitive and 24 KB, only between 4,097 and 131,071 primitives) reach into the links (16 B), written after it.
    L.sort = take(sort_scratch_bytes(n, key_bytes) - sort_small_tile_bytes(n, key_bytes));
    L.cbounds = L.sort;
    L.left = take(nn * 4);
    L.right = take(nn * 4);
    L.parent = take(2 * nn * 4);
    L.nboxes = take(2 * nn * 24);
    L.arrivals = take(nn * 4);
    L.cost = take(nn * 4);
    L.cnt = take(nn * 4);
    L.hgt = take(nn * 4);
    L.wcost = take(nn * 32);
    L.wdec = take(nn * 4);
    // subtree tasks: of two primitives or more, or a whole BLAS
    L.subs = take(16 * std::min<uint64_t>(nn, nn / 2 + (nbatch ? nbatch : 1)));
    L.queue = take(nn * 8);
    L.queue_words = take(sizeof(CollapseQueue));
    L.misc = take(64);
    L.geoms = take((uint64_t)(ngeom ? ngeom : 1) * sizeof(GeomDesc));
    if (nbatch) {
        L.pblas = take(nn * 4);
        L.nblas = take(nn * 4);
        L.roots = take((uint64_t)nbatch * 4);
        L.asptr = take((uint64_t)nbatch * 8);
        L.binfo = take((uint64_t)nbatch * 8);
        L.bcb = take((uint64_t)nbatch * 24);
    }
    L.total = o;
    return L;
}

uint64_t as_bytes(uint32_t n, bool tlas, bool update = false) {
    uint64_t slots = 2ull * (n ? n : 1) + 1;
    uint64_t b = kHeaderBytes + slots * kSlotBytes;
    if (tlas) b = align_up(b, 256) + (uint64_t)(n ? n : 1) * sizeof(InstanceInfo);
    if (update) b = align_up(b, 256) + (uint64_t)(n ? n : 1) * 4 * 5;  // order, left, right, parent (2n)
    return align_up(b, 256);
}

// Kept hierarchy of an updatable BLAS: order[n], left[n-1], right[n-1], parent[2n-1] (slots of 4 B).
uint64_t update_offset(uint32_t n) { return align_up(kHeaderBytes + (2ull * (n ? n : 1) + 1) * kSlotBytes, 256); }

__global__ void set_update_offset_kernel(AsHeader* h, uint64_t off) {
    if (threadIdx.x == 0 && blockIdx.x == 0) h->update_offset = off;
}

// Leaf cost of the wide collapse, relative to a node visit (cost 1): a triangle test (~80 VALU operations
// against the node test's ~250) or an instance entry (FP64 ray transform and a BLAS root visit).
constexpr float kLeafCostTri = 0.3f;
constexpr float kLeafCostInstance = 1.0f;

// One-wave blocks of the subtree passes (4M triangles: refinement 2.08 ms, collapse 1.13 ms with 4,096 blocks, which
// share the subtrees out unevenly, 1.71 and 0.77 ms with 65,536), of the passes over the nodes above (whose waves take
// several subtrees each: 0.57 ms with 4,096, 0.78 ms with 16,384), and of the collapse's queue.
constexpr uint32_t kSubtreeBlocks = 65536;
constexpr uint32_t kAboveBlocks = 4096;
constexpr uint32_t kQueueBlocks = 512;

// Counters of the bottom-up passes (5 words, zero at the start of a build): subtrees listed for the refinement rounds
// and the costs, and the queue's places.
uint32_t* pass_counts(uint8_t* scratch, const Layout& L) { return (uint32_t*)(scratch + L.misc) + 8; }

// counted: cnt holds the primitive counts of the internal nodes (written with the hierarchy).
// Refit with treelet refinement; each further round restructures the tree the previous one left.  Then the costs
// of the 8-wide collapse (wcost) over the final tree.
// Children per wide node: RTX_BUILD_MAX_WIDTH(w) caps it at w (2..7), 0 = 8.
int node_width(uint32_t flags) {
    const uint32_t w = (flags >> RTX_BUILD_MAX_WIDTH_SHIFT) & 7u;
    return w == 0u ? 8 : (w < 2u ? 2 : (int)w);
}

void refit_passes(uint32_t n, uint32_t flags, uint8_t* scratch, const Layout& L, const float* prim_boxes,
                  hipStream_t s, const uint32_t* node_blas = nullptr, float c_leaf = kLeafCostTri,
                  bool counted = true) {
    const int rounds = treelet_rounds(flags, n);
    uint32_t* arrivals = (uint32_t*)(scratch + L.arrivals);
    RefineArgs a;
    a.n = n;
    a.left = (int32_t*)(scratch + L.left);
    a.right = (int32_t*)(scratch + L.right);
    a.parent = (int32_t*)(scratch + L.parent);
    a.order = (const uint32_t*)(scratch + L.vals);
    a.prim_boxes = prim_boxes;
    a.nboxes = (float*)(scratch + L.nboxes);
    a.cost = (float*)(scratch + L.cost);
    a.cnt = (uint32_t*)(scratch + L.cnt);
    a.hgt = (uint32_t*)(scratch + L.hgt);
    a.arrivals = arrivals;
    a.node_blas = node_blas;
    a.list = nullptr;
    a.count = nullptr;
    uint32_t* counts = pass_counts(scratch, L);
    const uint32_t few = n / 8 + 1;  // at most this many waves
    // pass 0 .. 2: a refinement round; 3: the costs, with the collapse's queue
    auto find = [&](int pass) {
        find_subtrees_kernel<<<(n - 1) / kFindNodes + 1, 256, 0, s>>>(
            n, a.left, a.right, a.cnt, arrivals, (int32_t*)(scratch + L.list()), counts + pass,
            pass == 3 ? (uint64_t*)(scratch + L.queue) : nullptr, counts + 4);
    };
    if (!counted) {
        if (n > 1) fill_kernel<<<256, 256, 0, s>>>(arrivals, n, 0u);
        a.min_prims = 0xFFFFFFFFu;
        refit_refine_kernel<<<(n + 63) / 64, 64, 0, s>>>(a);
    } else {
        a.list = (int32_t*)(scratch + L.list());
        for (int round = 0; round < (rounds ? rounds : 1); ++round) {
            a.count = counts + round;
            a.min_prims = rounds ? kTreeletMinPrims[round] : 0xFFFFFFFFu;
            if (round) a.prim_boxes = nullptr;
            find(round);
            subtree_refine_kernel<<<std::min(few, kSubtreeBlocks), 64, 0, s>>>(a);
            if (n > kSubtree) refit_refine_kernel<<<std::min(few, kAboveBlocks), 64, 0, s>>>(a);
        }
    }
    if (n > 1) {
        find(3);
        CostArgs c;
        c.n = n;
        c.left = a.left;
        c.right = a.right;
        c.parent = a.parent;
        c.nboxes = a.nboxes;
        c.wc = (float*)(scratch + L.wcost);
        c.depths = (uint64_t*)(scratch + L.depths());
        c.wdec = (uint32_t*)(scratch + L.wdec);
        c.sub = (uint32_t*)(scratch + L.sub());
        c.arrivals = arrivals;
        c.c_leaf = c_leaf;
        c.width = node_width(flags);
        c.list = (const int32_t*)(scratch + L.list());
        c.count = counts + 3;
        subtree_cost_kernel<<<std::min(few, kSubtreeBlocks), 64, 0, s>>>(c);
        if (n > kSubtree) wide_cost_kernel<<<std::min(n / 2048 + 1, kAboveBlocks), 64, 0, s>>>(c);
    }
}

// The wide nodes of the structures whose roots the header kernel queued.
void collapse_passes(uint32_t n, uint32_t flags, uint8_t* scratch, const Layout& L, AsHeader* h,
                     AsHeader* const* as_ptr, const uint32_t* node_blas, uint32_t* err_flags, hipStream_t s) {
    CollapseArgs a;
    a.n = n;
    a.left = (const int32_t*)(scratch + L.left);
    a.right = (const int32_t*)(scratch + L.right);
    a.order = (const uint32_t*)(scratch + L.vals);
    a.nboxes = (const float*)(scratch + L.nboxes);
    a.leaf_src = (const uint4*)(scratch + L.leaves);
    a.cnt = (const uint32_t*)(scratch + L.cnt);
    a.wdec = (const uint32_t*)(scratch + L.wdec);
    a.sub = (const uint32_t*)(scratch + L.sub());
    a.h = h;
    a.as_ptr = as_ptr;
    a.node_blas = node_blas;
    a.q = (CollapseQueue*)(scratch + L.queue_words);
    a.queue = (uint64_t*)(scratch + L.queue);
    a.queue_size = pass_counts(scratch, L) + 4;
    a.subs = (uint4*)(scratch + L.subs);
    a.err = err_flags;
    a.width = (uint32_t)node_width(flags);
    const uint32_t top = std::min(n / 2048 + 1, kQueueBlocks);
    const uint32_t sub = std::min(n / 8 + 1, kSubtreeBlocks);
    if (as_ptr) {
        if (n > kSubtree) collapse_top_kernel<true><<<top, 64, 0, s>>>(a);
        collapse_subtree_kernel<true><<<sub, 64, 0, s>>>(a);
    } else {
        if (n > kSubtree) collapse_top_kernel<false><<<top, 64, 0, s>>>(a);
        collapse_subtree_kernel<false><<<sub, 64, 0, s>>>(a);
    }
}

// Common LBVH tail: morton -> sort -> karras -> refit -> header -> collapse.
hipError_t lbvh_common(uint32_t n, bool k64, uint32_t type, uint32_t flags, uint32_t ngeom, uint8_t* scratch,
                       const Layout& L, uint8_t* dst, uint64_t table_offset, uint32_t* err_flags, hipStream_t s) {
    AsHeader* h = (AsHeader*)dst;
    float* boxes = (float*)(scratch + L.boxes);
    uint32_t* cb = (uint32_t*)(scratch + L.cbounds);
    uint32_t* vals = (uint32_t*)(scratch + L.vals);
    int32_t* left = (int32_t*)(scratch + L.left);
    int32_t* right = (int32_t*)(scratch + L.right);
    int32_t* parent = (int32_t*)(scratch + L.parent);
    float* nboxes = (float*)(scratch + L.nboxes);
    float* cost = (float*)(scratch + L.cost);
    const unsigned gb = (unsigned)((n + 255) / 256);
    hipError_t err;
    if (n > 0) {
        if (k64) {
            morton_kernel<uint64_t><<<gb, 256, 0, s>>>(boxes, n, cb, (uint64_t*)(scratch + L.keys));
            if ((err = sort_pairs_u64((uint64_t*)(scratch + L.keys), vals, n, scratch + L.sort, err_flags, s)))
                return err;
        } else {
            morton_kernel<uint32_t><<<gb, 256, 0, s>>>(boxes, n, cb, (uint32_t*)(scratch + L.keys));
            if ((err = sort_pairs_u32((uint32_t*)(scratch + L.keys), vals, n, scratch + L.sort, err_flags, s)))
                return err;
        }
        if (n > 1) {
            if (k64)
                karras_kernel<uint64_t><<<gb, 256, 0, s>>>((uint64_t*)(scratch + L.keys), n, left, right, parent,
                                                           (uint32_t*)(scratch + L.cnt));
            else
                karras_kernel<uint32_t><<<gb, 256, 0, s>>>((uint32_t*)(scratch + L.keys), n, left, right, parent,
                                                           (uint32_t*)(scratch + L.cnt));
        } else {
            fill_kernel<<<1, 64, 0, s>>>((uint32_t*)parent, 1, 0xFFFFFFFFu);
        }
        refit_passes(n, flags, scratch, L, boxes, s, nullptr, type == 1 ? kLeafCostInstance : kLeafCostTri);
    }
    // root box: internal node 0, or the single leaf (stored at index n-1 == 0)
    header_kernel<<<1, 64, 0, s>>>(h, type, flags, n, ngeom, nboxes, cost, 2ull * (n ? n : 1) + 1, table_offset,
                                   (const uint32_t*)(scratch + L.cnt), (const uint32_t*)(scratch + L.sub()),
                                   (const uint64_t*)(scratch + L.depths()), (CollapseQueue*)(scratch + L.queue_words),
                                   (uint64_t*)(scratch + L.queue), (uint4*)(scratch + L.subs));
    if (n > 0) collapse_passes(n, flags, scratch, L, h, nullptr, nullptr, err_flags, s);
    return hipGetLastError();
}

}  // namespace

namespace {
// Morton / sort / Karras on caller boxes, optionally followed by the refit + refinement passes (rounds >= 0).
hipError_t debug_tree(const float* boxes, uint32_t n, bool k64, int rounds, void* codes_out, uint32_t* order_out,
                      int32_t* left_out, int32_t* right_out, float* cost_out, uint32_t* hgt_out, uint32_t* err_flags,
                      hipStream_t s) {
    Layout L = make_layout(n, k64 ? 8 : 4, 0);
    uint8_t* sc = nullptr;
    hipError_t e = hipMalloc(&sc, L.total);
    if (e) return e;
    uint32_t* cb = (uint32_t*)(sc + L.cbounds);
    init_build_kernel<<<1, 256, 0, s>>>(cb, (uint32_t*)(sc + L.misc));
    const unsigned gb = (unsigned)((n + 255) / 256);
    uint32_t* vals = (uint32_t*)(sc + L.vals);
    if (n > 0) {
        box_bounds_kernel<<<gb, 256, 0, s>>>(boxes, n, cb);
        if (k64) {
            morton_kernel<uint64_t><<<gb, 256, 0, s>>>(boxes, n, cb, (uint64_t*)(sc + L.keys));
            e = sort_pairs_u64((uint64_t*)(sc + L.keys), vals, n, sc + L.sort, err_flags, s);
            if (!e && n > 1)
                karras_kernel<uint64_t><<<gb, 256, 0, s>>>((uint64_t*)(sc + L.keys), n, (int32_t*)(sc + L.left),
                                                           (int32_t*)(sc + L.right), (int32_t*)(sc + L.parent),
                                                           (uint32_t*)(sc + L.cnt));
        } else {
            morton_kernel<uint32_t><<<gb, 256, 0, s>>>(boxes, n, cb, (uint32_t*)(sc + L.keys));
            e = sort_pairs_u32((uint32_t*)(sc + L.keys), vals, n, sc + L.sort, err_flags, s);
            if (!e && n > 1)
                karras_kernel<uint32_t><<<gb, 256, 0, s>>>((uint32_t*)(sc + L.keys), n, (int32_t*)(sc + L.left),
                                                           (int32_t*)(sc + L.right), (int32_t*)(sc + L.parent),
                                                           (uint32_t*)(sc + L.cnt));
        }
    }
    if (!e && rounds >= 0 && n > 1)
        refit_passes(n, rounds ? RTX_BUILD_TREELET_ROUNDS(rounds) : RTX_BUILD_NO_TREELET_BIT, sc, L, boxes, s);
    const uint64_t m = n > 1 ? (uint64_t)(n - 1) * 4 : 0;
    if (!e && n > 0 && codes_out)
        e = hipMemcpyAsync(codes_out, sc + L.keys, (uint64_t)n * (k64 ? 8 : 4), hipMemcpyDeviceToDevice, s);
    if (!e && n > 0) e = hipMemcpyAsync(order_out, vals, (uint64_t)n * 4, hipMemcpyDeviceToDevice, s);
    if (!e && m) e = hipMemcpyAsync(left_out, sc + L.left, m, hipMemcpyDeviceToDevice, s);
    if (!e && m) e = hipMemcpyAsync(right_out, sc + L.right, m, hipMemcpyDeviceToDevice, s);
    if (!e && m && cost_out) e = hipMemcpyAsync(cost_out, sc + L.cost, m, hipMemcpyDeviceToDevice, s);
    if (!e && m && hgt_out) e = hipMemcpyAsync(hgt_out, sc + L.hgt, m, hipMemcpyDeviceToDevice, s);
    hipError_t e2 = hipStreamSynchronize(s);
    (void)hipFree(sc);
    return e ? e : e2;
}
}  // namespace

hipError_t debug_lbvh(const float* boxes, uint32_t n, bool k64, void* codes_out, uint32_t* order_out,
                      int32_t* left_out, int32_t* right_out, uint32_t* err_flags, hipStream_t s) {
    return debug_tree(boxes, n, k64, -1, codes_out, order_out, left_out, right_out, nullptr, nullptr, err_flags, s);
}

hipError_t debug_treelet(const float* boxes, uint32_t n, bool k64, uint32_t rounds, uint32_t* order_out,
                         int32_t* left_out, int32_t* right_out, float* cost_out, uint32_t* hgt_out,
                         uint32_t* err_flags, hipStream_t s) {
    return debug_tree(boxes, n, k64, (int)rounds, nullptr, order_out, left_out, right_out, cost_out, hgt_out,
                      err_flags, s);
}

hipError_t debug_sort(void* keys, uint32_t* vals, uint32_t n, int key_bytes, uint32_t* err_flags, hipStream_t s) {
    uint8_t* sc = nullptr;
    hipError_t e = hipMalloc(&sc, sort_scratch_bytes(n, key_bytes) + 256);
    if (e) return e;
    if (key_bytes == 8)
        e = sort_pairs_u64((uint64_t*)keys, vals, n, sc, err_flags, s);
    else
        e = sort_pairs_u32((uint32_t*)keys, vals, n, sc, err_flags, s);
    hipError_t e2 = hipStreamSynchronize(s);
    (void)hipFree(sc);
    return e ? e : e2;
}

hipError_t upload_host_array(void* dst, const void* src, uint64_t bytes, hipStream_t s) {
    if (bytes == 0) return hipSuccess;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(s, &st);
    if (e != hipSuccess) return e;
    if (st == hipStreamCaptureStatusNone) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
    if (bytes > kArgUploadMax || (bytes & 3) || ((uintptr_t)dst & 3)) return hipErrorNotSupported;
    const uint8_t* in = (const uint8_t*)src;
    for (uint64_t at = 0; at < bytes; at += 4ull * kArgBlobWords) {
        const uint32_t words = (uint32_t)std::min<uint64_t>(kArgBlobWords, (bytes - at) / 4);
        ArgBlob b{};
        std::memcpy(b.w, in + at, 4ull * words);
        arg_blob_kernel<<<1, kArgBlobWords, 0, s>>>(b, (uint32_t*)((uint8_t*)dst + at), words);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}

uint64_t blas_as_bytes(uint32_t n, bool update) { return as_bytes(n, false, update); }
uint64_t tlas_as_bytes(uint32_t n) { return as_bytes(n, true); }
uint64_t blas_scratch_bytes(uint32_t n, bool k64, uint32_t ngeom) { return make_layout(n, k64 ? 8 : 4, ngeom).total; }
uint64_t tlas_scratch_bytes(uint32_t n, bool k64) { return make_layout(n, k64 ? 8 : 4, 0).total; }
uint64_t blas_batch_scratch_bytes(uint32_t n, uint32_t ngeom, uint32_t nbatch) {
    return make_layout(n, 8, ngeom, nbatch ? nbatch : 1).total;
}

hipError_t build_blas(const GeomDesc* geoms_host, uint32_t ngeom, uint32_t n, uint32_t flags, void* dst,
                      void* scratch, uint32_t* err_flags, hipStream_t s) {
    const bool k64 = (flags & RTX_BUILD_MORTON63_BIT) != 0;
    Layout L = make_layout(n, k64 ? 8 : 4, ngeom);
    uint8_t* sc = (uint8_t*)scratch;
    hipError_t err;
    GeomDesc* gd = (GeomDesc*)(sc + L.geoms);
    if (ngeom) {
        if ((err = upload_host_array(gd, geoms_host, ngeom * sizeof(GeomDesc), s))) return err;
    }
    uint32_t* cb = (uint32_t*)(sc + L.cbounds);
    init_build_kernel<<<1, 256, 0, s>>>(cb, (uint32_t*)(sc + L.misc));
    if (n > 0)
        prep_tris_kernel<<<(n - 1) / prep_chunk(n) + 1, 256, 0, s>>>(gd, (int)ngeom, n, (TriSlot*)(sc + L.leaves),
                                                                     (float*)(sc + L.boxes), cb, nullptr,
                                                                     prep_chunk(n));
    if ((err = lbvh_common(n, k64, 0, flags, ngeom, sc, L, (uint8_t*)dst, 0, err_flags, s))) return err;
    if (ngeom) content_kernel<<<(ngeom + 255) / 256, 256, 0, s>>>(gd, ngeom, (AsHeader*)dst, nullptr);
    finish_blas_kernel<<<1, 64, 0, s>>>((AsHeader*)dst);
    if ((flags & RTX_BUILD_ALLOW_UPDATE_BIT) && n > 0) {
        // keep the final hierarchy (after treelet refinement) and the triangle order for updates
        const uint64_t off = update_offset(n);
        uint8_t* u = (uint8_t*)dst + off;
        if ((err = hipMemcpyAsync(u, sc + L.vals, 4ull * n, hipMemcpyDeviceToDevice, s))) return err;
        if (n > 1) {
            if ((err = hipMemcpyAsync(u + 4ull * n, sc + L.left, 4ull * (n - 1), hipMemcpyDeviceToDevice, s)))
                return err;
            if ((err = hipMemcpyAsync(u + 4ull * (2 * n - 1), sc + L.right, 4ull * (n - 1), hipMemcpyDeviceToDevice,
                                      s)))
                return err;
        }
        if ((err = hipMemcpyAsync(u + 4ull * (3 * n - 2), sc + L.parent, 4ull * (2 * n - 1), hipMemcpyDeviceToDevice,
                                  s)))
            return err;
        set_update_offset_kernel<<<1, 64, 0, s>>>((AsHeader*)dst, off);
    }
    return hipGetLastError();
}

// UPDATE mode: new triangle positions, the kept order and hierarchy, plain refit, header and collapse again.
hipError_t update_blas(const GeomDesc* geoms_host, uint32_t ngeom, uint32_t n, uint32_t flags, void* dst,
                       void* scratch, uint32_t* err_flags, hipStream_t s) {
    Layout L = make_layout(n, 4, ngeom);
    uint8_t* sc = (uint8_t*)scratch;
    hipError_t err;
    GeomDesc* gd = (GeomDesc*)(sc + L.geoms);
    if (ngeom && (err = upload_host_array(gd, geoms_host, ngeom * sizeof(GeomDesc), s)))
        return err;
    uint32_t* cb = (uint32_t*)(sc + L.cbounds);
    init_build_kernel<<<1, 256, 0, s>>>(cb, (uint32_t*)(sc + L.misc));
    AsHeader* h = (AsHeader*)dst;
    const uint64_t off = update_offset(n);
    const uint8_t* u = (const uint8_t*)dst + off;
    if (n > 0) {
        prep_tris_kernel<<<(n - 1) / prep_chunk(n) + 1, 256, 0, s>>>(gd, (int)ngeom, n, (TriSlot*)(sc + L.leaves),
                                                                     (float*)(sc + L.boxes), cb, nullptr,
                                                                     prep_chunk(n));
        if ((err = hipMemcpyAsync(sc + L.vals, u, 4ull * n, hipMemcpyDeviceToDevice, s))) return err;
        if (n > 1) {
            if ((err = hipMemcpyAsync(sc + L.left, u + 4ull * n, 4ull * (n - 1), hipMemcpyDeviceToDevice, s)))
                return err;
            if ((err = hipMemcpyAsync(sc + L.right, u + 4ull * (2 * n - 1), 4ull * (n - 1), hipMemcpyDeviceToDevice,
                                      s)))
                return err;
        }
        if ((err = hipMemcpyAsync(sc + L.parent, u + 4ull * (3 * n - 2), 4ull * (2 * n - 1),
                                  hipMemcpyDeviceToDevice, s)))
            return err;
        refit_passes(n, flags | RTX_BUILD_NO_TREELET_BIT, sc, L, (const float*)(sc + L.boxes), s, nullptr,
                     kLeafCostTri, false);
    }
    header_kernel<<<1, 64, 0, s>>>(h, 0, flags, n, ngeom, (const float*)(sc + L.nboxes), (const float*)(sc + L.cost),
                                   2ull * (n ? n : 1) + 1, 0, (const uint32_t*)(sc + L.cnt),
                                   (const uint32_t*)(sc + L.sub()), (const uint64_t*)(sc + L.depths()),
                                   (CollapseQueue*)(sc + L.queue_words), (uint64_t*)(sc + L.queue),
                                   (uint4*)(sc + L.subs));
    if (n > 0) collapse_passes(n, flags, sc, L, h, nullptr, nullptr, err_flags, s);
    if (ngeom) content_kernel<<<(ngeom + 255) / 256, 256, 0, s>>>(gd, ngeom, h, nullptr);
    finish_blas_kernel<<<1, 64, 0, s>>>(h);
    set_update_offset_kernel<<<1, 64, 0, s>>>(h, off);
    return hipGetLastError();
}

hipError_t build_tlas(const rtx_instance* inst, uint32_t n, uint32_t flags, void* dst, void* scratch,
                      uint32_t* err_flags, hipStream_t s) {
    const bool k64 = (flags & RTX_BUILD_MORTON63_BIT) != 0;
    Layout L = make_layout(n, k64 ? 8 : 4, 0);
    uint8_t* sc = (uint8_t*)scratch;
    uint64_t table_offset = align_up(kHeaderBytes + (2ull * (n ? n : 1) + 1) * kSlotBytes, 256);
    uint32_t* cb = (uint32_t*)(sc + L.cbounds);
    uint32_t* maxd = (uint32_t*)(sc + L.misc);
    init_build_kernel<<<1, 256, 0, s>>>(cb, maxd);  // misc words 0, 1: deepest BLAS, content bits
    if (n > 0)
        prep_instances_kernel<<<std::min((n + 3) / 4, 2048u), 256, 0, s>>>(
            inst, n, (InstSlot*)(sc + L.leaves), (InstanceInfo*)((uint8_t*)dst + table_offset),
            (float*)(sc + L.boxes), cb, maxd, maxd + 1);
    hipError_t err;
    if ((err = lbvh_common(n, k64, 1, flags, 0, sc, L, (uint8_t*)dst, table_offset, err_flags, s))) return err;
    finish_tlas_kernel<<<1, 64, 0, s>>>((AsHeader*)dst, maxd);
    return hipGetLastError();
}

// Batched BLAS build: every step runs once over the primitives of all BLASes.  Keys are BLAS id << 30 | Morton
// code, so after the stable sort each BLAS is one contiguous range and one subtree of the single Karras tree; the
// part of the tree above the BLAS roots is never collapsed, refined or stored.
hipError_t build_blas_batch(const GeomDesc* geoms_host, uint32_t ngeom, const uint2* binfo_host,
                            AsHeader* const* dst_host, uint32_t nbatch, uint32_t n, uint32_t flags, void* scratch,
                            uint32_t* err_flags, hipStream_t s) {
    Layout L = make_layout(n, 8, ngeom, nbatch);
    uint8_t* sc = (uint8_t*)scratch;
    hipError_t err;
    GeomDesc* gd = (GeomDesc*)(sc + L.geoms);
    AsHeader** as_ptr = (AsHeader**)(sc + L.asptr);
    uint2* binfo = (uint2*)(sc + L.binfo);
    if (ngeom && (err = upload_host_array(gd, geoms_host, ngeom * sizeof(GeomDesc), s)))
        return err;
    if ((err = upload_host_array(as_ptr, dst_host, nbatch * sizeof(AsHeader*), s))) return err;
    if ((err = upload_host_array(binfo, binfo_host, nbatch * sizeof(uint2), s))) return err;
    uint32_t* cb = (uint32_t*)(sc + L.bcb);
    uint32_t* pblas = (uint32_t*)(sc + L.pblas);
    uint32_t* nblas = (uint32_t*)(sc + L.nblas);
    int32_t* roots = (int32_t*)(sc + L.roots);
    uint64_t* keys = (uint64_t*)(sc + L.keys);
    uint32_t* vals = (uint32_t*)(sc + L.vals);
    int32_t* left = (int32_t*)(sc + L.left);
    int32_t* right = (int32_t*)(sc + L.right);
    int32_t* parent = (int32_t*)(sc + L.parent);
    float* nboxes = (float*)(sc + L.nboxes);
    float* boxes = (float*)(sc + L.boxes);
    const unsigned gb = (unsigned)((n + 255) / 256);
    init_batch_kernel<<<(6 * nbatch + 127) / 256 + 1, 256, 0, s>>>(cb, roots, nbatch, (uint32_t*)(sc + L.misc),
                                                                   (uint32_t*)(sc + L.queue_words));
    if (n > 0) {
        prep_tris_kernel<<<(n - 1) / prep_chunk(n) + 1, 256, 0, s>>>(gd, (int)ngeom, n, (TriSlot*)(sc + L.leaves), boxes,
                                                                     cb, pblas, prep_chunk(n));
        morton_batch_kernel<<<gb, 256, 0, s>>>(boxes, n, cb, pblas, keys);
        int bits = 30;
        while (bits < 64 && (nbatch - 1) >> (bits - 30)) ++bits;
        if ((err = sort_pairs_u64(keys, vals, n, sc + L.sort, err_flags, s, bits))) return err;
        if (n > 1) {
            karras_kernel<uint64_t><<<gb, 256, 0, s>>>(keys, n, left, right, parent, (uint32_t*)(sc + L.cnt), nblas);
        } else {
            fill_kernel<<<1, 64, 0, s>>>((uint32_t*)parent, 1, 0xFFFFFFFFu);
        }
        blas_roots_kernel<<<(unsigned)((2ull * n - 1 + 255) / 256), 256, 0, s>>>(n, keys, parent, nblas, roots);
        refit_passes(n, flags, sc, L, boxes, s, n > 1 ? nblas : nullptr);
    }
    batch_header_kernel<<<(nbatch + 63) / 64, 64, 0, s>>>(
        as_ptr, binfo, nbatch, roots, n, flags, nboxes, (const float*)(sc + L.cost), (const uint32_t*)(sc + L.cnt),
        (const uint32_t*)(sc + L.sub()), (const uint64_t*)(sc + L.depths()), (CollapseQueue*)(sc + L.queue_words),
        (uint64_t*)(sc + L.queue), (uint4*)(sc + L.subs));
    if (n > 0) collapse_passes(n, flags, sc, L, nullptr, as_ptr, nblas, err_flags, s);
    if (ngeom) content_kernel<<<(ngeom + 255) / 256, 256, 0, s>>>(gd, ngeom, nullptr, as_ptr);
    batch_finish_kernel<<<(nbatch + 63) / 64, 64, 0, s>>>(as_ptr, nbatch);
    return hipGetLastError();
}

}  // namespace rtx
