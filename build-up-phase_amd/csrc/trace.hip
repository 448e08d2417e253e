// trace.hip — persistent BVH8 traversal for gfx950: ray buffers (closest / any hit) and the reference raygen.
//
// Replaces the driver traversal behind traceRayEXT (call site main.cpp:1047-1052) and the raygen / miss /
// closest-hit programs (main.cpp:1033-1091).
//
// Per lane (wave64; one persistent grid; a wave takes ray ids from atomic counters in chunks and refills its
// idle lanes once fewer than refill_lanes of 64 are busy, checked every refill_interval steps):
//   * world ray (FP32) -> TLAS: nodes are tested with a conservative quantised slab test, instance leaves
//     enter their BLAS;
//   * BLAS entry (FP64): the ray is transformed by the FP64 inverse instance transform and its origin moved
//     onto the BLAS root box (t_e = entry distance), then rounded to FP32.  All FP32 work inside the BLAS
//     happens on coordinates of the size of the BLAS box, not of the distance to the camera;
//   * triangles: watertight test (Woop, Benthin & Wald 2013) with the shear written as three row vectors, so
//     no per-lane component selection is needed per triangle; exact-zero edge functions are recomputed in FP64;
//     the wave's lanes test the triangles of the lanes that hold a leaf group, two of each at a time;
//   * traversal order: children are stored by octant; the group mask is permuted by the ray's sign octant so
//     that lowest-bit-first visits near children first (Ylitie, Karras & Laine 2017 node groups);
//   * stack: per-lane entries (slot base, child mask, valid mask, flags) in LDS, spilling to a global
//     per-thread area past the LDS depth; overflow beyond that raises kErrStackOverflow;
//   * closest hit: t, u, v are recomputed in FP64 (Moller-Trumbore) for the winning triangle;
//   * the FLAGS variant adds the traceRayEXT ray flags, triangle opacity (geometry / instance / ray) and the
//     any-hit programs of non-opaque candidates; the host uses it only where they can change a result;
//   * a lane's ended ray is finished at the wave's next refill point, together with the wave's other ended rays
//     (result writes and their FP64 refinement run with many lanes instead of one or two); in the whole-path
//     modes (training paths, pixel paths) finishing means shading the vertex and continuing the lane's path
//     with its next ray, so one launch traces whole paths.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "pt_shade.h"
#include "rtx_internal.h"
#include "trace.h"

namespace rtx {

namespace {

constexpr float kErrScale = 0x1p-20f;
constexpr float kTinyDir = 0x1p-80f;
constexpr uint32_t kEntryLeaf = 1u << 16;
constexpr uint32_t kEntryTlas = 1u << 17;
constexpr uint32_t kNoSlot = 0xFFFFFFFFu;
constexpr uint32_t kMaxSteps = 1u << 22;  // per ray; a valid BVH never needs more than ~2 steps per slot

// traceRayEXT ray flags (gl_RayFlags*EXT values) and instance flags (VkGeometryInstanceFlagBitsKHR)
constexpr uint32_t kRayTerminateOnFirstHit = RTX_RAY_FLAG_TERMINATE_ON_FIRST_HIT;
constexpr uint32_t kRaySkipClosestHit = RTX_RAY_FLAG_SKIP_CLOSEST_HIT_SHADER;
constexpr uint32_t kRayCullBack = RTX_RAY_FLAG_CULL_BACK_FACING_TRIANGLES;
constexpr uint32_t kRayCullFront = RTX_RAY_FLAG_CULL_FRONT_FACING_TRIANGLES;
constexpr uint32_t kRayCullOpaque = RTX_RAY_FLAG_CULL_OPAQUE;
constexpr uint32_t kRaySkipTriangles = RTX_RAY_FLAG_SKIP_TRIANGLES;
constexpr uint32_t kRayOpaque = RTX_RAY_FLAG_OPAQUE;
constexpr uint32_t kRayNoOpaque = RTX_RAY_FLAG_NO_OPAQUE;
constexpr uint32_t kRayCullNoOpaque = RTX_RAY_FLAG_CULL_NO_OPAQUE;
constexpr uint32_t kRaySkipAabbs = RTX_RAY_FLAG_SKIP_AABBS;
// FLAGS variant: the current instance register holds the instance id in bits 0-29 and the instance's
// FORCE_OPAQUE (bit 30) / FORCE_NO_OPAQUE (bit 31) flags.
constexpr uint32_t kInstIdMask = 0x3FFFFFFFu;


// Loads and stores through explicit global / LDS pointers.  A BLAS address comes out of the instance slot as an
// integer, and a stack entry lies in LDS or in the spill area, so through plain pointers the compiler emits flat
// accesses, which hold up both memory pipes and wait for both counters.
typedef uint32_t Words2 __attribute__((ext_vector_type(2)));
typedef uint32_t Words4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) uint8_t* SlotPtr;
__device__ __forceinline__ uint4 load_words(SlotPtr p, int k) {
    const Words4 w = ((const __attribute__((address_space(1))) Words4*)p)[k];
    return make_uint4(w.x, w.y, w.z, w.w);
}

// Hit masks in traversal order, by octant and mask: child position k goes to bit k ^ octant.
struct alignas(16) OctTable {
    uint8_t row[8][256];
};
static_assert(alignof(OctTable) >= alignof(uint64_t) && sizeof(OctTable) % sizeof(uint64_t) == 0,
              "blocks copy the table in 8-byte words");
static_assert(sizeof(OctTable) == kOctTableBytes, "the launch rules' size");
constexpr OctTable make_oct_table() {
    OctTable t{};
    for (uint32_t oct = 0; oct < 8; ++oct)
        for (uint32_t m = 0; m < 256; ++m) {
            uint32_t r = 0;
            for (uint32_t k = 0; k < 8; ++k) r |= (m >> k & 1u) << (k ^ oct);
            t.row[oct][m] = (uint8_t)r;
        }
    return t;
}
__constant__ OctTable kOctTable = make_oct_table();
// The same computed: 16 vector instructions a node step, where the table in LDS would cost blocks.
__device__ __forceinline__ uint32_t oct_permute(uint32_t m, uint32_t oct) {
    if (oct & 1u) m = ((m & 0x55u) << 1) | ((m >> 1) & 0x55u);
    if (oct & 2u) m = ((m & 0x33u) << 2) | ((m >> 2) & 0x33u);
    if (oct & 4u) m = ((m & 0x0Fu) << 4) | ((m >> 4) & 0x0Fu);
    return m;
}

// 1/d for the slab tests, |d| clamped to at least 2^-80.  v_rcp_f32 (1 ulp) on d * 2^-32 keeps the operand and
// the result in the normal range for every |d| in [2^-80, 2^128); the node test's error margin (2^-20 relative
// per term) covers the approximate reciprocal.
__device__ __forceinline__ float safe_rcp(float d) {
    float a = fabsf(d) < kTinyDir ? copysignf(kTinyDir, d) : d;
    return __builtin_amdgcn_rcpf(a * 0x1p-32f) * 0x1p-32f;
}

struct Space {
    float ox, oy, oz;
    float dx, dy, dz;
    float ix, iy, iz;
    uint32_t oct;
    uint32_t sel[3];  // byte selectors of the near plane's children 0 and 1 per axis (test_node)
    float toff;
};

__device__ __forceinline__ void setup_space(Space& s) {
    s.ix = safe_rcp(s.dx);
    s.iy = safe_rcp(s.dy);
    s.iz = safe_rcp(s.dz);
    s.oct = (s.dx < 0.0f ? 1u : 0u) | (s.dy < 0.0f ? 2u : 0u) | (s.dz < 0.0f ? 4u : 0u);
    s.sel[0] = s.ix < 0.0f ? 0x0C050C04u : 0x0C010C00u;
    s.sel[1] = s.iy < 0.0f ? 0x0C050C04u : 0x0C010C00u;
    s.sel[2] = s.iz < 0.0f ? 0x0C050C04u : 0x0C010C00u;
}

// Facing culls.  A triangle is front-facing when v0, v1, v2 appear clockwise seen from the ray origin, i.e.
// dot(d, (v1 - v0) x (v2 - v0)) > 0 in object space; an instance with TRIANGLE_FLIP_FACING makes counter-
// clockwise front-facing, and TRIANGLE_FACING_CULL_DISABLE (the reference's instances, main.cpp:852) exempts it.
__device__ __forceinline__ bool facing_culled(const uint4 a, const uint4 b, const uint4 c, const Space& s,
                                              uint32_t ray_flags, uint32_t inst_flags) {
    if (inst_flags & RTX_INSTANCE_TRIANGLE_FACING_CULL_DISABLE_BIT) return false;
    const float e1x = __uint_as_float(a.w) - __uint_as_float(a.x);
    const float e1y = __uint_as_float(b.x) - __uint_as_float(a.y);
    const float e1z = __uint_as_float(b.y) - __uint_as_float(a.z);
    const float e2x = __uint_as_float(b.z) - __uint_as_float(a.x);
    const float e2y = __uint_as_float(b.w) - __uint_as_float(a.y);
    const float e2z = __uint_as_float(c.x) - __uint_as_float(a.z);
    const float nx = e1y * e2z - e1z * e2y, ny = e1z * e2x - e1x * e2z, nz = e1x * e2y - e1y * e2x;
    bool front = s.dx * nx + s.dy * ny + s.dz * nz > 0.0f;
    if (inst_flags & RTX_INSTANCE_TRIANGLE_FLIP_FACING_BIT) front = !front;
    return front ? (ray_flags & kRayCullFront) != 0 : (ray_flags & kRayCullBack) != 0;
}

// The half at bits 16 * i of w, widened (exact; v_fma_mix_f32 widens its operand by itself).
__device__ __forceinline__ float half_f(uint32_t w, int i) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> (16 * i)));
}

// Quantised 8-child slab test.  Returns the child-position hit mask.
// Bound by VALU issue (a node step of a busy wave is about two thirds ALU), so the 48 plane bytes are not converted
// one by one: a byte q zero-extended to 16 bits is the half 2^-24 q, which v_fma_mix_f32 reads exactly, and one
// v_perm_b32 both extends two bytes and picks the near or the far plane by the ray's sign (24 permutes instead of 48
// conversions and 12 selects).  The 2^24 goes into S, and where that overflows so does the margin, which leaves the
// axis unconstrained.  With the pointers above: 16.7M camera rays 1.87 -> 1.77 ms, whole paths 19.3 -> 18.5 ms.
__device__ __forceinline__ uint32_t test_node(const uint4 w0, const uint4 w1, const uint4 w2, const uint4 w3,
                                              const Space& s, const float* rlo, const float* qs, float smin,
                                              float smax) {
    const float pqx = (float)(w0.x & 0xFFFFu), pqy = (float)(w0.x >> 16), pqz = (float)(w0.y & 0xFFFFu);
    const uint32_t ex = (w0.y >> 16) & 255u, ey = w0.y >> 24, ez = w0.z & 255u;
    const uint32_t vmask = (w0.z >> 16) & 255u;
    const float px = fmaf(pqx, qs[0], rlo[0]);
    const float py = fmaf(pqy, qs[1], rlo[1]);
    const float pz = fmaf(pqz, qs[2], rlo[2]);
    const float sx = __uint_as_float(ex << 23), sy = __uint_as_float(ey << 23), sz = __uint_as_float(ez << 23);
    const float Ax = (px - s.ox) * s.ix, Ay = (py - s.oy) * s.iy, Az = (pz - s.oz) * s.iz;
    const float Sx = sx * s.ix * 0x1p24f, Sy = sy * s.iy * 0x1p24f, Sz = sz * s.iz * 0x1p24f;
    const float ex_ = fmaf(fabsf(px), fabsf(s.ix), fmaf(0x1.FEp-17f, fabsf(Sx), fabsf(Ax)));
    const float ey_ = fmaf(fabsf(py), fabsf(s.iy), fmaf(0x1.FEp-17f, fabsf(Sy), fabsf(Ay)));
    const float ez_ = fmaf(fabsf(pz), fabsf(s.iz), fmaf(0x1.FEp-17f, fabsf(Sz), fabsf(Az)));
    const float Anx = fmaf(-kErrScale, ex_, Ax), Afx = fmaf(kErrScale, ex_, Ax);
    const float Any = fmaf(-kErrScale, ey_, Ay), Afy = fmaf(kErrScale, ey_, Ay);
    const float Anz = fmaf(-kErrScale, ez_, Az), Afz = fmaf(kErrScale, ez_, Az);
    // byte arrays: qlo x = (w1.x, w1.y), qlo y = (w1.z, w1.w), qlo z = (w2.x, w2.y),
    //              qhi x = (w2.z, w2.w), qhi y = (w3.x, w3.y), qhi z = (w3.z, w3.w)
    const uint32_t lo[6] = {w1.x, w1.y, w1.z, w1.w, w2.x, w2.y}, hi[6] = {w2.z, w2.w, w3.x, w3.y, w3.z, w3.w};
    uint32_t hit = 0;
#pragma unroll
    for (int k = 0; k < 8; k += 2) {
        uint32_t n[3], f[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const uint32_t sel = s.sel[a] + ((k & 2) ? 0x00020002u : 0u);
            n[a] = __builtin_amdgcn_perm(hi[2 * a + k / 4], lo[2 * a + k / 4], sel);
            f[a] = __builtin_amdgcn_perm(lo[2 * a + k / 4], hi[2 * a + k / 4], sel);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float tnx = fmaf(half_f(n[0], i), Sx, Anx);
            const float tny = fmaf(half_f(n[1], i), Sy, Any);
            const float tnz = fmaf(half_f(n[2], i), Sz, Anz);
            const float tfx = fmaf(half_f(f[0], i), Sx, Afx);
            const float tfy = fmaf(half_f(f[1], i), Sy, Afy);
            const float tfz = fmaf(half_f(f[2], i), Sz, Afz);
            const float tn = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, smin));
            const float tf = fminf(fminf(tfx, tfy), fminf(tfz, smax));
            hit |= (tn <= tf) ? (1u << (k + i)) : 0u;
        }
    }
    return hit & vmask;
}

struct Shear {
    float rx0, rx1, rx2, ry0, ry1, ry2, rz0, rz1, rz2;
};

__device__ __forceinline__ void setup_shear(const Space& s, Shear& sh) {
    const float ax = fabsf(s.dx), ay = fabsf(s.dy), az = fabsf(s.dz);
    const int kz = (ax >= ay && ax >= az) ? 0 : (ay >= az ? 1 : 2);
    // the axes after kz in order: whichever way the ray runs along kz, since the edge functions and the determinant
    // only change sign together with the winding
    const float dkz = kz == 0 ? s.dx : (kz == 1 ? s.dy : s.dz);
    const float dkx = kz == 0 ? s.dy : (kz == 1 ? s.dz : s.dx);
    const float dky = kz == 0 ? s.dz : (kz == 1 ? s.dx : s.dy);
    const float Sx = dkx / dkz, Sy = dky / dkz, Sz = 1.0f / dkz;
    sh.rx0 = kz == 0 ? -Sx : (kz == 2 ? 1.0f : 0.0f);
    sh.rx1 = kz == 1 ? -Sx : (kz == 0 ? 1.0f : 0.0f);
    sh.rx2 = kz == 2 ? -Sx : (kz == 1 ? 1.0f : 0.0f);
    sh.ry0 = kz == 0 ? -Sy : (kz == 1 ? 1.0f : 0.0f);
    sh.ry1 = kz == 1 ? -Sy : (kz == 2 ? 1.0f : 0.0f);
    sh.ry2 = kz == 2 ? -Sy : (kz == 0 ? 1.0f : 0.0f);
    sh.rz0 = kz == 0 ? Sz : 0.0f;
    sh.rz1 = kz == 1 ? Sz : 0.0f;
    sh.rz2 = kz == 2 ? Sz : 0.0f;
}

// Watertight test in the current (rebased object) space.  Returns true and the parametric distance s when
// the triangle is hit with s in [smin, smax].
__device__ __forceinline__ bool test_triangle(const uint4 a, const uint4 b, const uint4 c, const Space& s,
                                              const Shear& sh, float smin, float smax, float& t_out, float& u_out,
                                              float& v_out) {
    const float v0x = __uint_as_float(a.x) - s.ox, v0y = __uint_as_float(a.y) - s.oy, v0z = __uint_as_float(a.z) - s.oz;
    const float v1x = __uint_as_float(a.w) - s.ox, v1y = __uint_as_float(b.x) - s.oy, v1z = __uint_as_float(b.y) - s.oz;
    const float v2x = __uint_as_float(b.z) - s.ox, v2y = __uint_as_float(b.w) - s.oy, v2z = __uint_as_float(c.x) - s.oz;
    const float Ax = fmaf(v0z, sh.rx2, fmaf(v0y, sh.rx1, v0x * sh.rx0));
    const float Ay = fmaf(v0z, sh.ry2, fmaf(v0y, sh.ry1, v0x * sh.ry0));
    const float Az = fmaf(v0z, sh.rz2, fmaf(v0y, sh.rz1, v0x * sh.rz0));
    const float Bx = fmaf(v1z, sh.rx2, fmaf(v1y, sh.rx1, v1x * sh.rx0));
    const float By = fmaf(v1z, sh.ry2, fmaf(v1y, sh.ry1, v1x * sh.ry0));
    const float Bz = fmaf(v1z, sh.rz2, fmaf(v1y, sh.rz1, v1x * sh.rz0));
    const float Cx = fmaf(v2z, sh.rx2, fmaf(v2y, sh.rx1, v2x * sh.rx0));
    const float Cy = fmaf(v2z, sh.ry2, fmaf(v2y, sh.ry1, v2x * sh.ry0));
    const float Cz = fmaf(v2z, sh.rz2, fmaf(v2y, sh.rz1, v2x * sh.rz0));
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {
        U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    const float det = U + V + W;
    if (det == 0.0f) return false;
    float T = U * Az + V * Bz + W * Cz;
    const float adet = fabsf(det);
    const float Ts = det < 0.0f ? -T : T;
    if (Ts < smin * adet || Ts > smax * adet) return false;
    t_out = Ts / adet;
    const float rdet = 1.0f / det;
    u_out = V * rdet;
    v_out = W * rdet;
    return true;
}

struct TraceArgs {
    const uint8_t* tlas;
    const rtx_ray* rays;
    const uint32_t* n_ptr;  // when set, the ray count is read from device memory (queues)
    const rtx_ray* rays2;   // kModeFused: the any-hit queue and its device count
    const uint32_t* n2_ptr;
    PathHit* path_hits;
    uint32_t n;
    uint32_t cull_mask;
    rtx_hit* hits;
    uint32_t* occluded;
    // raygen
    float cam[3];
    float ax, ay;
    uint32_t width, height;
    float tmin, tmax;
    const rtx_hit_record* records;
    uint32_t nrec, sbt_offset, sbt_stride;
    float miss[3];
    float* film;
    // runtime
    DeviceState* state;
    uint2* gstack;
    uint32_t lds_depth;
    uint32_t gdepth;
    uint32_t ray_chunk;        // ray ids per queue fetch (< 64: automatic)
    uint32_t guard;            // 1 / 2: the launch traces only if guard_passes
    uint32_t first_waves;      // waves whose first chunk is their own; the others take all chunks from the queues
    uint32_t refill_lanes;     // refill a wave once fewer lanes than this are busy
    uint32_t refill_interval;  // steps between refill checks
    uint32_t leaf_lanes;       // pending leaf groups needed before a leaf step runs
    uint32_t ray_flags;        // RTX_RAY_FLAG_* of the launch
    // kModeTrain / kModePixelPaths: the path tracer's state, the first path id (npix for training paths, 0 for
    // pixel paths) and the pass's sample index
    PtArgs pt;
    uint32_t pt_first;
    uint32_t pt_sample;
};

// kModeFused: one launch over two queues of the wavefront integrator, rays [0, nA) of `rays` as kModePath
// (extension rays, path hits) and rays [nA, nA + nB) of `rays2` as kModeAny (shadow rays, occlusion flags).
// kModeTrain / kModePixelPaths: whole paths in one launch - the NRC frame's training paths, or one sample of a
// plain render's pixel paths.  A lane takes a path index from the ray pool, traces its camera ray, and whenever
// one of its rays ends (the wave handles its lanes' ended rays together at its next refill) shades the vertex
// (pathtrace.hip's per-vertex step) and continues the same path with the next-event shadow ray and then the
// continuation ray, until the path ends; then it takes a new path.
enum Mode {
    kModeClosest = 0,
    kModeAny = 1,
    kModeRaygen = 2,
    kModePath = 3,
    kModeFused = 4,
    kModeTrain = 5,
    kModePixelPaths = 6,
    kModePixelCache = 7  // the pixel paths of an NRC frame: whole paths up to their cache query
};

// FP64 recomputation of (t, u, v) for the winning triangle (Moller & Trumbore 1997) in object space.
__device__ void refine_hit(const double* inv, const float* wo, const float* wd, const TriSlot* tri, float& t,
                           float& u, float& v) {
    double o[3], d[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        o[r] = inv[4 * r] * wo[0] + inv[4 * r + 1] * wo[1] + inv[4 * r + 2] * wo[2] + inv[4 * r + 3];
        d[r] = inv[4 * r] * wd[0] + inv[4 * r + 1] * wd[1] + inv[4 * r + 2] * wd[2];
    }
    double v0[3], e1[3], e2[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        v0[a] = tri->v[a];
        e1[a] = (double)tri->v[3 + a] - v0[a];
        e2[a] = (double)tri->v[6 + a] - v0[a];
    }
    double p[3] = {d[1] * e2[2] - d[2] * e2[1], d[2] * e2[0] - d[0] * e2[2], d[0] * e2[1] - d[1] * e2[0]};
    double det = e1[0] * p[0] + e1[1] * p[1] + e1[2] * p[2];
    double inv_det = 1.0 / det;
    double sv[3] = {o[0] - v0[0], o[1] - v0[1], o[2] - v0[2]};
    double uu = (sv[0] * p[0] + sv[1] * p[1] + sv[2] * p[2]) * inv_det;
    double q[3] = {sv[1] * e1[2] - sv[2] * e1[1], sv[2] * e1[0] - sv[0] * e1[2], sv[0] * e1[1] - sv[1] * e1[0]};
    double vv = (d[0] * q[0] + d[1] * q[1] + d[2] * q[2]) * inv_det;
    double tt = (e2[0] * q[0] + e2[1] * q[1] + e2[2] * q[2]) * inv_det;
    t = (float)tt;
    u = (float)uu;
    v = (float)vv;
}

// Intersection programs of AABB primitives (box lo = a.xyz, hi = a.w, b.x, b.y).  The first intersection with t
// in [tmin, tmax] of the ray o + t d with the program's surface, its (u, v) and the outward normal n (object
// space, unnormalised for boxes).  T is float for the traversal's candidate test (in the current rebased space)
// and double for the reported hit.
// FP32 world-space unit geometric normal of a triangle (the path tracer's shading normal; the instance inverse is
// rounded to FP32).
__device__ __forceinline__ void world_normal_f32(const double* inv, const TriSlot* tri, float* n) {
    float e1[3], e2[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        e1[a] = tri->v[3 + a] - tri->v[a];
        e2[a] = tri->v[6 + a] - tri->v[a];
    }
    const float no[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
    float nw[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) nw[c] = (float)inv[c] * no[0] + (float)inv[4 + c] * no[1] + (float)inv[8 + c] * no[2];
    const float l = sqrtf(nw[0] * nw[0] + nw[1] * nw[1] + nw[2] * nw[2]);
    const float r = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
    for (int c = 0; c < 3; ++c) n[c] = nw[c] * r;
}

template <typename T>
__device__ __forceinline__ bool procedural_hit(uint32_t prog, const T* lo, const T* hi, const T* o, const T* d,
                                               T tmin, T tmax, T& t_out, T& u_out, T& v_out, T* n) {
    if (prog == RTX_INTERSECTION_SPHERE) {
        T c[3], oc[3];
        T r = hi[0] - lo[0];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            c[k] = (lo[k] + hi[k]) * T(0.5);
            oc[k] = o[k] - c[k];
            r = k ? (hi[k] - lo[k] < r ? hi[k] - lo[k] : r) : r;
        }
        r *= T(0.5);
        const T A = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
        const T B = oc[0] * d[0] + oc[1] * d[1] + oc[2] * d[2];
        const T C = oc[0] * oc[0] + oc[1] * oc[1] + oc[2] * oc[2] - r * r;
        const T disc = B * B - A * C;
        if (!(disc >= T(0)) || !(A > T(0)) || !(r > T(0))) return false;
        const T sq = sqrt(disc);
        T t = (-B - sq) / A;
        if (t < tmin) t = (-B + sq) / A;
        if (!(t >= tmin && t <= tmax)) return false;
#pragma unroll
        for (int k = 0; k < 3; ++k) n[k] = (o[k] + t * d[k] - c[k]) / r;
        t_out = t;
        u_out = (n[0] + T(1)) * T(0.5);
        v_out = (n[1] + T(1)) * T(0.5);
        return true;
    }
    // RTX_INTERSECTION_BOX: slab entry, or the exit when the entry lies before tmin
    T tn = -INFINITY, tf = INFINITY;
    int an = 0, af = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (d[k] == T(0)) {
            if (o[k] < lo[k] || o[k] > hi[k]) return false;
            continue;
        }
        const T i = T(1) / d[k];
        T t1 = (lo[k] - o[k]) * i, t2 = (hi[k] - o[k]) * i;
        if (t1 > t2) {
            const T x = t1;
            t1 = t2;
            t2 = x;
        }
        if (t1 > tn) {
            tn = t1;
            an = k;
        }
        if (t2 < tf) {
            tf = t2;
            af = k;
        }
    }
    if (!(tn <= tf)) return false;
    T t;
    int ax;
    if (tn >= tmin && tn <= tmax) {
        t = tn;
        ax = an;
    } else if (tf >= tmin && tf <= tmax) {
        t = tf;
        ax = af;
    } else {
        return false;
    }
    const int a1 = ax == 2 ? 0 : ax + 1, a2 = ax == 0 ? 2 : ax - 1;
    const T p1 = (a1 == 0 ? o[0] : (a1 == 1 ? o[1] : o[2])) + t * (a1 == 0 ? d[0] : (a1 == 1 ? d[1] : d[2]));
    const T p2 = (a2 == 0 ? o[0] : (a2 == 1 ? o[1] : o[2])) + t * (a2 == 0 ? d[0] : (a2 == 1 ? d[1] : d[2]));
    const T l1 = a1 == 0 ? lo[0] : (a1 == 1 ? lo[1] : lo[2]), h1 = a1 == 0 ? hi[0] : (a1 == 1 ? hi[1] : hi[2]);
    const T l2 = a2 == 0 ? lo[0] : (a2 == 1 ? lo[1] : lo[2]), h2 = a2 == 0 ? hi[0] : (a2 == 1 ? hi[1] : hi[2]);
    t_out = t;
    u_out = h1 > l1 ? (p1 - l1) / (h1 - l1) : T(0);
    v_out = h2 > l2 ? (p2 - l2) / (h2 - l2) : T(0);
    // outward normal of the hit face: -d's sign along ax at the entry, +d's at the exit
    const T dax = ax == 0 ? d[0] : (ax == 1 ? d[1] : d[2]);
    const T sgn = (t == tn) ? (dax > T(0) ? T(-1) : T(1)) : (dax > T(0) ? T(1) : T(-1));
    n[0] = ax == 0 ? sgn : T(0);
    n[1] = ax == 1 ? sgn : T(0);
    n[2] = ax == 2 ? sgn : T(0);
    return true;
}

// Intersection program of an AABB primitive's hit record (bits 8-15 of its program), RTX_INTERSECTION_BOX without
// a hit-record table.
__device__ __forceinline__ uint32_t intersection_program(const TraceArgs& args, const InstanceInfo* info,
                                                         uint32_t geom) {
    if (!args.records) return RTX_INTERSECTION_BOX;
    const uint32_t rec = info->sbt_offset + geom * args.sbt_stride + args.sbt_offset;
    return rec < args.nrec ? (args.records[rec].program >> 8) & 255u : RTX_INTERSECTION_BOX;
}

// FP64 (t, u, v) and world-space unit normal of an AABB primitive hit of the world ray (wo, wd) under the
// instance transform with inverse inv; false when FP64 finds no intersection at or after tmin (then the caller
// keeps the FP32 values).
__device__ bool refine_procedural(const double* inv, const float* wo, const float* wd, const TriSlot* tri,
                                  uint32_t prog, float tmin, float& t, float& u, float& v, float* nw) {
    double o[3], d[3], lo[3], hi[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        o[r] = inv[4 * r] * wo[0] + inv[4 * r + 1] * wo[1] + inv[4 * r + 2] * wo[2] + inv[4 * r + 3];
        d[r] = inv[4 * r] * wd[0] + inv[4 * r + 1] * wd[1] + inv[4 * r + 2] * wd[2];
        lo[r] = tri->v[r];
        hi[r] = tri->v[3 + r];
    }
    double tt, uu, vv, n[3];
    if (!procedural_hit<double>(prog, lo, hi, o, d, (double)tmin, (double)INFINITY, tt, uu, vv, n)) return false;
    t = (float)tt;
    u = (float)uu;
    v = (float)vv;
    if (nw) {
        double w[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) w[c] = inv[c] * n[0] + inv[4 + c] * n[1] + inv[8 + c] * n[2];
        const double l = sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
        const double rl = l > 0.0 ? 1.0 / l : 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) nw[c] = (float)(w[c] * rl);
    }
    return true;
}

// The any-hit program of a non-opaque candidate (its hit record: instance SBT offset + geometry index x stride +
// ray SBT offset, as for closest hits) on the candidate's barycentrics (u, v) from the watertight test (FP32):
// true to accept it.  Without a hit-record table, or with a record index outside it, the candidate is accepted
// (a hit group without an any-hit shader).
__device__ __forceinline__ bool any_hit_accepts(const TraceArgs& args, const InstanceInfo* info, uint32_t geom,
                                                float u, float v) {
    if (!args.records) return true;
    const uint32_t rec = info->sbt_offset + geom * args.sbt_stride + args.sbt_offset;
    if (rec >= args.nrec) return true;
    const uint32_t ah = args.records[rec].any_hit;
    if ((ah & 255u) != RTX_ANY_HIT_CUTOUT) return true;
    const float n = (ah >> 8) ? (float)(ah >> 8) : 1.0f;
    const int cell = (int)floorf(u * n) + (int)floorf(v * n);
    return (cell & 1) == 0;
}

// Opacity of a candidate (geometry bit, overridden by the instance's FORCE flags, overridden by the ray's OPAQUE /
// NO_OPAQUE), the CULL_OPAQUE / CULL_NO_OPAQUE culls, then the any-hit program of a non-opaque candidate.  Used by
// the FLAGS variant only; the default variant treats every triangle as opaque and runs only where that holds.
__device__ __forceinline__ bool candidate_accepted(const TraceArgs& args, uint32_t ray_flags, uint32_t tri_bits,
                                                   uint32_t geom, uint32_t cur_inst, const InstanceInfo* table,
                                                   float u, float v) {
    bool opaque = !(tri_bits & kTriNonOpaque);
    const uint32_t force = cur_inst >> 30;
    if (force) opaque = (force & 1u) != 0;
    if (ray_flags & kRayOpaque) opaque = true;
    else if (ray_flags & kRayNoOpaque) opaque = false;
    if ((opaque && (ray_flags & kRayCullOpaque)) || (!opaque && (ray_flags & kRayCullNoOpaque))) return false;
    if (opaque) return true;
    return any_hit_accepts(args, table + (cur_inst & kInstIdMask), geom, u, v);
}

// Queues that a wave tries before it takes no more chunks.
constexpr uint32_t kQueueHops = 3u;

// The kernel's arguments, read again where they are used: the compiler otherwise loads them all at the start of the
// kernel, and the path tracer's, of which a traversal step uses none, do not fit the SGPRs beside the traversal's
// (147 of 1,591 vector instructions of the code between traversals restored them lane by lane).
__device__ __forceinline__ const void* reread_kernel_arguments() {
    uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return (const void*)(const __attribute__((address_space(4))) void*)p;
}

// LEAN: no LDS but the stack and the world rays (plan_trace chooses).
template <int MODE, bool STATS, bool FLAGS, bool LEAN>
__device__ __forceinline__ void trace_body(const TraceArgs& args) {
    const uint32_t ray_flags = FLAGS ? args.ray_flags : 0u;  // the default variant compiles the flags out
    // dynamic LDS: the per-lane stack (lds_depth entries per lane); the FLAGS variant and the path-tracer modes
    // add the lane's world ray (6 floats per lane), which they read back where they need it (leaving a BLAS, the
    // final FP64 refinement) instead of keeping it in registers (measured: spill-free at 128 VGPRs and 1% faster
    // path tracing); the other variants keep it in wo / wd
    constexpr bool kTrain = MODE == kModeTrain || MODE == kModePixelPaths || MODE == kModePixelCache;  // whole paths
    constexpr int kShadeMode = MODE == kModePixelPaths ? (int)kPtPlain : (int)kPtCache;
    constexpr bool kRayLds = FLAGS || MODE == kModePath || MODE == kModeFused || kTrain;
    // the stack, the rays, the triangle tasks of the block's waves (32 of 16 B each)
    extern __shared__ __attribute__((aligned(16))) uint2 lds_stack[];
    __attribute__((address_space(3))) Words4* const tasks =
        (__attribute__((address_space(3))) Words4*)(lds_stack + (args.lds_depth + (kRayLds ? 3u : 0u)) * blockDim.x) +
        32u * (threadIdx.x >> 6);
    __shared__ OctTable oct_lds;
    if (!LEAN) {
        for (uint32_t i = threadIdx.x; i < sizeof(OctTable) / 8u; i += blockDim.x)
            ((uint64_t*)&oct_lds)[i] = ((const uint64_t*)&kOctTable)[i];
        __syncthreads();
    }
    float* const lds_ray = (float*)(lds_stack + args.lds_depth * blockDim.x) + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint64_t gtid = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    const AsHeader* th = (const AsHeader*)args.tlas;
    const SlotPtr tslots = (SlotPtr)(args.tlas + kHeaderBytes);
    const InstanceInfo* table = (const InstanceInfo*)(args.tlas + th->inst_table_offset);
    const float trlo[3] = {th->lo[0], th->lo[1], th->lo[2]};
    const float tqs[3] = {th->qscale[0], th->qscale[1], th->qscale[2]};
    const bool tlas_empty = th->slot_count == 0;
    const uint32_t tlas_nslots = th->slot_count;
    const uint32_t tlas_ninst = th->prim_count;
    const uint32_t D = args.lds_depth;
    const uint32_t GD = args.gdepth;
    // ray flags under which no triangle can be accepted
    const bool cull_all = ((ray_flags & kRaySkipTriangles) && (ray_flags & kRaySkipAabbs)) ||
                          ((ray_flags & kRayCullOpaque) && (ray_flags & (kRayOpaque | kRayCullNoOpaque))) ||
                          ((ray_flags & kRayCullNoOpaque) && (ray_flags & kRayNoOpaque));
    if (args.guard && !guard_passes(args.tlas, args.ray_flags, args.guard)) return;  // the other launch takes the rays
    const uint32_t nA = args.n_ptr ? *args.n_ptr : args.n;
    const uint32_t nrays = MODE == kModeFused ? nA + *args.n2_ptr : nA;

    uint64_t st_nodes = 0, st_tris = 0, st_insts = 0, st_rays = 0;

    bool active = false, finished = false;
    uint32_t ray_id = 0;
    float wo[3], wd[3], wtmin = 0.0f, tc = 0.0f;
    Space s;
    Shear sh;
    SlotPtr cslots = tslots;
    float crlo[3], cqs[3];
    bool in_blas = false;
    uint32_t cur_inst = 0;
    uint32_t cur_nslots = tlas_nslots;
    uint32_t steps = 0;
    uint32_t ng_base = 0, ng_bits = 0;  // bits: ordered mask | vmask << 8
    uint32_t lg_base = 0, lg_bits = 0;  // bits: child-position mask | vmask << 8
    uint32_t sp = 0;
    uint32_t hit_inst = kNoHit, hit_slot = 0;
    bool occl = false;
    bool shadow_ray = MODE == kModeAny;  // this lane's ray is an any-hit query
    uint32_t pdepth = 0;       // kModeTrain: vertex of the path that the current ray leaves
    bool ext_pending = false;  // kModeTrain: the continuation ray waits behind the shadow ray
    uint32_t pt_rays = 0;      // kModeTrain: rays traced (path-tracer ray count)
    const uint32_t pt_sample = kTrain ? pass_sample(args.pt, args.pt_sample) : 0u;

    // stack entries of this lane: LDS up to depth D, then its part of the spill area
    __attribute__((address_space(3))) Words2* const lstack =
        (__attribute__((address_space(3))) Words2*)lds_stack + threadIdx.x;
    __attribute__((address_space(1))) Words2* const gstack =
        (__attribute__((address_space(1))) Words2*)args.gstack + gtid * GD;
    auto push = [&](const uint2 e) {
        const Words2 w = {e.x, e.y};
        if (sp < D) lstack[__umul24(sp, blockDim.x)] = w;
        else if (sp < D + GD) gstack[sp - D] = w;
        ++sp;
    };
    auto stacked = [&](uint32_t at) {
        Words2 w;
        if (at < D) w = lstack[__umul24(at, blockDim.x)];
        else w = gstack[at - D];
        return make_uint2(w.x, w.y);
    };

    // a new ray (wo, wd, wtmin, tc set): world space at the TLAS root
    auto begin_ray = [&]() {
        if (kRayLds) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                lds_ray[k * blockDim.x] = wo[k];
                lds_ray[(3 + k) * blockDim.x] = wd[k];
            }
        }
        s.ox = wo[0];
        s.oy = wo[1];
        s.oz = wo[2];
        s.dx = wd[0];
        s.dy = wd[1];
        s.dz = wd[2];
        s.toff = 0.0f;
        setup_space(s);
        cslots = tslots;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            crlo[a] = trlo[a];
            cqs[a] = tqs[a];
        }
        in_blas = false;
        cur_nslots = tlas_nslots;
        steps = 0;
        ng_base = 0;
        // the root as a one-child group: child position 0 sits at ordered bit (0 ^ oct)
        ng_bits = tlas_empty || cull_all ? 0u : ((1u << s.oct) | (1u << 8));
        lg_bits = 0;
        sp = 0;
        hit_inst = kNoHit;
        occl = false;
        if (STATS) ++st_rays;
    };
    auto set_ray = [&](const rtx_ray& r) {
        wo[0] = r.origin[0];
        wo[1] = r.origin[1];
        wo[2] = r.origin[2];
        wtmin = r.tmin;
        wd[0] = r.direction[0];
        wd[1] = r.direction[1];
        wd[2] = r.direction[2];
        tc = r.tmax;
    };

    // Wave-uniform pool of ray ids [pool_next, pool_end).  Chunk w of the launch is wave w's first pool, for the
    // first first_waves waves; the chunks after those come from kRayQueues counters, each shared by the blocks of one
    // residue: queue q's c-th chunk is one of the c-th group of nq chunks, at a place rotated by a hash of c (with a
    // fixed place, a film whose rows hold a multiple of nq / 2 chunks gives every queue its own columns: 20% slower).
    // An atomic on one word shared by all waves costs 10-20 ns in turn, so one counter bounded short launches by its
    // 4,096 waves' fetches alone: 777 rays 96 us, the 1200x800 reference film 224 us.
    const uint32_t waves_block = blockDim.x >> 6;
    const uint32_t waves_total = gridDim.x * waves_block;
    const uint32_t wave =
        (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * waves_block + (threadIdx.x >> 6)));
    const uint32_t chunk = rays_per_chunk(args.ray_chunk, nrays, waves_total, args.first_waves, kTrain);
    const uint32_t nqueues = gridDim.x < kRayQueues ? gridDim.x : kRayQueues;
    uint32_t queue = blockIdx.x % nqueues;
    uint32_t hops = 0;  // queues this wave has found empty
    const uint32_t own_chunks = args.first_waves;
    bool more = (uint64_t)chunk * own_chunks < nrays;
    uint32_t pool_next = 0, pool_end = 0;
    if (wave < own_chunks) {
        const uint64_t first = (uint64_t)wave * chunk;
        if (first < nrays) {
            pool_next = (uint32_t)first;
            pool_end = (uint32_t)(first + chunk < nrays ? first + chunk : nrays);
        }
    }
    for (;;) {
        if (kTrain && finished) {
            const PtArgs& pt = ((const TraceArgs*)reread_kernel_arguments())->pt;
            // continue the lane's path: gather a shadow ray's contribution, or shade the vertex the continuation
            // ray reached; then trace the next ray of the path, or let the lane take a new path.  The pending
            // continuation ray and the shadow contribution wait in the path's slot (ray_id) of the queue buffers.
            const uint32_t pid = args.pt_first + ray_id;
            bool cont = false;
            if (shadow_ray) {
                if (!occl) {
                    const float4 c = pt.sh_contrib[ray_id];
                    float4 r = pt.rad[pid];
                    r.x += c.x;
                    r.y += c.y;
                    r.z += c.z;
                    pt.rad[pid] = r;
                }
                shadow_ray = false;
                if (ext_pending) {
                    set_ray(pt.ext_rays[0][ray_id]);
                    ++pdepth;
                    cont = true;
                }
            } else {
                PathHit ph;
                ph.t = 0.0f;
                ph.u = 0.0f;
                ph.v = 0.0f;
                ph.inst = hit_inst;
                ph.prim = 0;
                ph.geom = 0;
                ph.n[0] = ph.n[1] = ph.n[2] = 0.0f;
                ph.rec = 0xFFFFFFFFu;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    wo[k] = lds_ray[k * blockDim.x];
                    wd[k] = lds_ray[(3 + k) * blockDim.x];
                }
                if (hit_inst != kNoHit) {
                    const InstanceInfo* info = table + hit_inst;
                    double M[12];
#pragma unroll
                    for (int kk = 0; kk < 12; ++kk) M[kk] = info->inv[kk];
                    const TriSlot* tri =
                        (const TriSlot*)((const uint8_t*)info->blas + kHeaderBytes + (uint64_t)hit_slot * kSlotBytes);
                    ph.t = tc;
                    ph.prim = tri->prim;
                    ph.geom = tri->geom;
                    world_normal_f32(M, tri, ph.n);
                    ph.rec = info->sbt_offset + ph.geom * args.sbt_stride + args.sbt_offset;
                }
                rtx_ray cr;
                cr.origin[0] = wo[0];
                cr.origin[1] = wo[1];
                cr.origin[2] = wo[2];
                cr.tmin = wtmin;
                cr.direction[0] = wd[0];
                cr.direction[1] = wd[1];
                cr.direction[2] = wd[2];
                cr.tmax = tc;
                ShadeOut so;
                shade_vertex<kShadeMode>(pt, pid, cr, ph, pdepth, pt_sample, so);
                pt_rays += (so.push_sh ? 1u : 0u) + (so.push_ext ? 1u : 0u);
                if (so.push_ext) {
                    pt.thr[pid] = so.thr_new;
                    pt.ext_rays[0][ray_id] = so.ext;
                }
                ext_pending = so.push_ext;
                if (MODE == kModePixelCache) {
                    // the path ends in a cache query: one slot per query, one atomic per wave
                    const uint64_t qm = __ballot(so.push_cq);
                    if (qm) {
                        const uint32_t leader = (uint32_t)(__ffsll((long long)qm) - 1);
                        uint32_t base = 0;
                        if (lane == leader) base = atomicAdd(&pt.counts[2], (uint32_t)__popcll(qm));
                        base = __shfl(base, (int)leader);
                        if (so.push_cq) {
                            const uint32_t slot = base + (uint32_t)__popcll(qm & lt_mask);
                            pt.cq[slot] = so.cq;
                            pt.cq_pid[slot] = pid;
                        }
                    }
                }
                if (so.push_sh) {
                    pt.sh_contrib[ray_id] = so.contrib;
                    set_ray(so.sh);
                    shadow_ray = true;
                    cont = true;
                } else if (so.push_ext) {
                    set_ray(so.ext);
                    ++pdepth;
                    cont = true;
                }
            }
            if (cont) {
                begin_ray();
                active = true;
            }
            finished = false;
        }
        if (!kTrain && finished) {
            // write the result of ray_id (lanes whose rays ended since the last refill, in one pass)
            if (MODE == kModeAny || (MODE == kModeFused && shadow_ray)) {
                args.occluded[MODE == kModeFused ? ray_id - nA : ray_id] = occl ? 1u : 0u;
            } else {
                float t = 0.0f, u = 0.0f, v = 0.0f;
                uint32_t prim = 0, geom = 0;
                const InstanceInfo* info = nullptr;
                bool proc = false;  // an AABB primitive's hit: normal from its intersection program
                float pn[3] = {0.0f, 0.0f, 0.0f};
                if (hit_inst != kNoHit) {
                    info = table + hit_inst;
                    double M[12];
#pragma unroll
                    for (int kk = 0; kk < 12; ++kk) M[kk] = info->inv[kk];
                    const TriSlot* tri =
                        (const TriSlot*)((const uint8_t*)info->blas + kHeaderBytes + (uint64_t)hit_slot * kSlotBytes);
                    if (kRayLds) {
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            wo[k] = lds_ray[k * blockDim.x];
                            wd[k] = lds_ray[(3 + k) * blockDim.x];
                        }
                    }
                    if (MODE == kModePath || MODE == kModeFused) {
                        // the path tracer shades with t and the normal only: the traversal's FP32 t (u, v
                        // are not needed); procedural normals below
                        t = tc;
                        proc = FLAGS && (tri->bits & kTriAabb);
                        if (proc && !refine_procedural(M, wo, wd, tri, intersection_program(args, info, tri->geom),
                                                       wtmin, t, u, v, pn)) {
                            const float l = sqrtf(wd[0] * wd[0] + wd[1] * wd[1] + wd[2] * wd[2]);
#pragma unroll
                            for (int k = 0; k < 3; ++k) pn[k] = l > 0.0f ? -wd[k] / l : 0.0f;
                        }
                    } else if (FLAGS && (tri->bits & kTriAabb)) {
                        // keep the traversal's FP32 t if FP64 finds no intersection (the normal then faces
                        // the ray)
                        proc = true;
                        t = tc;
                        if (!refine_procedural(M, wo, wd, tri, intersection_program(args, info, tri->geom),
                                               wtmin, t, u, v,
                                               (MODE == kModePath || MODE == kModeFused) ? pn : nullptr)) {
                            const float l = sqrtf(wd[0] * wd[0] + wd[1] * wd[1] + wd[2] * wd[2]);
#pragma unroll
                            for (int k = 0; k < 3; ++k) pn[k] = l > 0.0f ? -wd[k] / l : 0.0f;
                        }
                    } else {
                        refine_hit(M, wo, wd, tri, t, u, v);
                    }
                    prim = tri->prim;
                    geom = tri->geom;
                }
                if (MODE == kModePath || MODE == kModeFused) {
                    PathHit ph;
                    ph.t = t;
                    ph.u = u;
                    ph.v = v;
                    ph.inst = hit_inst;
                    ph.prim = prim;
                    ph.geom = geom;
                    ph.n[0] = ph.n[1] = ph.n[2] = 0.0f;
                    ph.rec = 0xFFFFFFFFu;
                    if (hit_inst != kNoHit) {
                        double M[12];
#pragma unroll
                        for (int kk = 0; kk < 12; ++kk) M[kk] = info->inv[kk];
                        const TriSlot* tri = (const TriSlot*)((const uint8_t*)info->blas + kHeaderBytes +
                                                              (uint64_t)hit_slot * kSlotBytes);
                        if (FLAGS && proc) {
                            ph.n[0] = pn[0];
                            ph.n[1] = pn[1];
                            ph.n[2] = pn[2];
                        } else {
                            world_normal_f32(M, tri, ph.n);
                        }
                        ph.rec = info->sbt_offset + geom * args.sbt_stride + args.sbt_offset;
                    }
                    args.path_hits[ray_id] = ph;
                } else if (MODE == kModeClosest) {
                    uint32_t* hp = (uint32_t*)(args.hits + ray_id);
                    hp[0] = __float_as_uint(t);
                    hp[1] = __float_as_uint(u);
                    hp[2] = __float_as_uint(v);
                    hp[3] = prim;
                    hp[4] = geom;
                    hp[5] = hit_inst;
                } else {
                    float r = args.miss[0], g = args.miss[1], bl = args.miss[2];
                    if (hit_inst != kNoHit && (ray_flags & kRaySkipClosestHit)) {
                        r = g = bl = 0.0f;  // the closest-hit program does not run: the payload keeps its 0
                    } else if (hit_inst != kNoHit) {
                        const uint32_t rec = info->sbt_offset + geom * args.sbt_stride + args.sbt_offset;
                        if (rec < args.nrec) {
                            const rtx_hit_record hr = args.records[rec];
                            bool bary = hr.program == RTX_PROGRAM_BARYCENTRIC;
                            if (hr.program == RTX_PROGRAM_MATCH_BARYCENTRIC)
                                bary = (int32_t)prim == hr.match_primitive && (int32_t)hit_inst == hr.match_instance &&
                                       (int32_t)info->custom == hr.match_custom_index &&
                                       (int32_t)geom == hr.match_geometry;
                            if (bary) {
                                r = 1.0f - u - v;
                                g = u;
                                bl = v;
                            } else {
                                r = hr.color[0];
                                g = hr.color[1];
                                bl = hr.color[2];
                            }
                        } else {
                            r = g = bl = 0.0f;
                        }
                    }
                    *(float4*)(args.film + 4 * (uint64_t)ray_id) = make_float4(r, g, bl, 0.0f);
                }
            }
            finished = false;
        }
        const uint64_t need = more || pool_next < pool_end ? __ballot(!active) : 0ull;
        if (need) {
            const uint32_t want = (uint32_t)__popcll(need);
            const uint32_t rank = (uint32_t)__popcll(need & lt_mask);
            const uint32_t avail = pool_end - pool_next;
            const uint32_t served = avail < want ? avail : want;
            uint32_t id = rank < served ? pool_next + rank : 0xFFFFFFFFu;
            pool_next += served;
            if (served < want && more) {
                uint64_t base;
                for (;;) {
                    uint32_t c = 0;
                    if (lane == 0) c = atomicAdd(&args.state->queue[queue].next, 1u);
                    c = (uint32_t)__builtin_amdgcn_readfirstlane((int)c);
                    const uint32_t place = (queue + ((c * 0x9E3779B1u) >> 16)) % nqueues;
                    base = ((uint64_t)own_chunks + (uint64_t)c * nqueues + place) * chunk;
                    if (base < nrays || ++hops >= kQueueHops) break;
                    queue = queue + 1u < nqueues ? queue + 1u : 0u;
                }
                if (base < nrays) {
                    const uint32_t left = nrays - (uint32_t)base;
                    pool_next = (uint32_t)base;
                    pool_end = pool_next + (left < chunk ? left : chunk);
                    const uint32_t rest = want - served;
                    const uint32_t take = pool_end - pool_next < rest ? pool_end - pool_next : rest;
                    if (rank >= served && rank - served < take) id = pool_next + (rank - served);
                    pool_next += take;
                } else {
                    more = false;
                }
            }
            if (!active) {
                if (id < nrays) {
                    ray_id = id;
                    active = true;
                    if (MODE == kModeRaygen) {
                        const uint32_t x = id % args.width, y = id / args.width;
                        const float sx = ((float)x + 0.5f) / (float)args.width;
                        const float sy = ((float)y + 0.5f) / (float)args.height;
                        const float nx = sx * 2.0f - 1.0f;
                        const float ny = sy * 2.0f - 1.0f;
                        wo[0] = args.cam[0];
                        wo[1] = args.cam[1];
                        wo[2] = args.cam[2];
                        wd[0] = nx * args.ax;
                        wd[1] = -(ny * args.ay);
                        wd[2] = -1.0f;
                        wtmin = args.tmin;
                        tc = args.tmax;
                    } else if (kTrain) {
                        const PtArgs& pt = ((const TraceArgs*)reread_kernel_arguments())->pt;
                        const uint32_t pid = args.pt_first + id;
                        rtx_ray r;
                        pt_camera_ray(pt, pid, pt_sample, r);
                        pt.thr[pid] = make_float4(1.0f, 1.0f, 1.0f, 0.0f);
                        pt.rad[pid] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                        pdepth = 0;
                        shadow_ray = false;
                        ext_pending = false;
                        ++pt_rays;
                        set_ray(r);
                    } else {
                        if (MODE == kModeFused) shadow_ray = id >= nA;
                        const float4* rp = (const float4*)(MODE == kModeFused && id >= nA ? args.rays2 + (id - nA)
                                                                                          : args.rays + id);
                        const float4 r0 = rp[0], r1 = rp[1];
                        wo[0] = r0.x;
                        wo[1] = r0.y;
                        wo[2] = r0.z;
                        wtmin = r0.w;
                        wd[0] = r1.x;
                        wd[1] = r1.y;
                        wd[2] = r1.z;
                        tc = r1.w;
                    }
                    begin_ray();
                }
            }
        }
        if (!__any(active)) break;
        const bool wave_exhausted = !more && pool_next >= pool_end;
        // Whole paths: back to the refill point (where ended rays continue their paths) once half of the lanes that
        // start this round (64 - refill_lanes of 32) have ended their rays, at least one.  Shading costs as much as
        // five traversal steps, however few lanes shade: 4 samples of the 1080p Cornell box 13.0 ms with half of the
        // lanes, 14.0 ms with a quarter, 13.8 ms with three quarters.
        uint32_t train_floor = 0;
        if (kTrain) {
            const uint32_t n0 = (uint32_t)__popcll(__ballot(active));
            const uint32_t q = std::min(n0, n0 * (64u - args.refill_lanes) / 32u);
            train_floor = n0 - (q > 0u ? q : 1u);
        }

        int iter = 0;
        bool go = true;
        uint32_t busy_lanes = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(active));
        while (go) {
            bool done = false;
            uint32_t fault = 0;
            // Postponed leaves: the triangle step runs only once leaf_lanes lanes of the wave hold a pending leaf group
            // of triangles, the instance step (BLAS entry in FP64) once as many hold one of instances, and both when
            // no lane can traverse; until then lanes with a pending leaf keep traversing their node group, or wait.
            // (Lanes without a ray hold no group.)  Each has its own threshold, because an instance step costs twice a
            // triangle step: with one for both 16.7M incoherent rays took 2.59 ms, now 2.41 ms.  leaf_lanes is for a
            // full wave and shrinks with the rays that it still traces: half of a short launch is the tail of its
            // longest rays (250 to 600 steps), which must not wait for each other (1080p film of dense alpha-tested
            // geometry 1.15 -> 1.06 ms, 1277x719 film of 64 dense meshes 580 -> 515 us).
            const bool has_leaf = (lg_bits & 255u) != 0u;
            const bool enter = has_leaf && !in_blas;
            const uint32_t inst_lanes = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(enter));
            const uint64_t tri_lanes = __builtin_amdgcn_ballot_w64(has_leaf && in_blas);
            const bool no_node =
                __builtin_amdgcn_ballot_w64((ng_bits & 255u) || (active && !(lg_bits & 255u))) == 0ull;
            const uint32_t leaf_at = (busy_lanes * args.leaf_lanes + 63u) >> 6;
            if (tri_lanes && ((uint32_t)__popcll(tri_lanes) >= leaf_at || no_node)) {
                // The next two triangles of each leaf group, one per lane of the wave: 4 to 12 lanes hold a leaf
                // group when the leaf step runs, most of them two triangles, so the owners hand theirs out and
                // one pass of the whole wave tests them (two passes of the owners alone took 6,000 to 10,000
                // cycles, this one takes 2,200 to 3,000).  Owners past the 32nd wait for the next leaf step.
                const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(tri_lanes >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)tri_lanes, 0u));
                const bool owner = has_leaf && in_blas && rank < 32u;
                uint32_t slot0 = kNoSlot, slot1 = kNoSlot;
                if (owner) {
                    const uint32_t vm = lg_bits >> 8;
                    uint32_t m = lg_bits & 255u;
                    slot0 = lg_base + (uint32_t)__popc(vm & ((m & (0u - m)) - 1u));
                    m &= m - 1u;
                    if (m) {
                        slot1 = lg_base + (uint32_t)__popc(vm & ((m & (0u - m)) - 1u));
                        m &= m - 1u;
                    }
                    lg_bits = m | (vm << 8);
                    if (slot0 >= cur_nslots || (slot1 != kNoSlot && slot1 >= cur_nslots)) {
                        fault = kErrBadAs;
                        slot0 = slot1 = kNoSlot;
                    }
                    if (!LEAN) tasks[rank] = Words4{slot0, slot1, lane, 0u};
                }
                const uint32_t ntri = 2u * (uint32_t)__popcll(tri_lanes);
                uint32_t from = lane, slot = kNoSlot;
                if (LEAN) {
                    // Owner number k sends its triangles and its place to lane 2 k, from where lane 2 k + 1 takes them
                    // too (quad_perm [0, 0, 2, 2]); lanes that own nothing send to lane 1, whose word nobody reads.
                    const int to = owner ? (int)(rank << 3) : 4;
                    const auto pair = [&](uint32_t v) {
                        return (uint32_t)__builtin_amdgcn_mov_dpp(__builtin_amdgcn_ds_permute(to, (int)v), 0xA0, 0xF,
                                                                  0xF, true);
                    };
                    const uint32_t whose = pair(lane), task0 = pair(slot0), task1 = pair(slot1);
                    if (lane < ntri) {
                        slot = (lane & 1u) ? task1 : task0;
                        from = whose;
                    }
                } else {
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    if (lane < ntri) {
                        const Words4 w = tasks[lane >> 1];
                        slot = (lane & 1u) ? w.y : w.x;
                        from = w.z;
                    }
                }
                // the owner's ray
                const auto pull = [&](float v) {
                    return __uint_as_float((uint32_t)__builtin_amdgcn_ds_bpermute((int)(from << 2),
                                                                                  (int)__float_as_uint(v)));
                };
                const auto pullu = [&](uint32_t v) {
                    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(from << 2), (int)v);
                };
                Space hs;
                Shear hh;
                hs.ox = pull(s.ox);
                hs.oy = pull(s.oy);
                hs.oz = pull(s.oz);
                hh.rx0 = pull(sh.rx0);
                hh.rx1 = pull(sh.rx1);
                hh.rx2 = pull(sh.rx2);
                hh.ry0 = pull(sh.ry0);
                hh.ry1 = pull(sh.ry1);
                hh.ry2 = pull(sh.ry2);
                hh.rz0 = pull(sh.rz0);
                hh.rz1 = pull(sh.rz1);
                hh.rz2 = pull(sh.rz2);
                const float smin = pull(wtmin - s.toff);
                const float smax = pull(tc - s.toff);
                const uint64_t hslots =
                    pullu((uint32_t)(uint64_t)cslots) | ((uint64_t)pullu((uint32_t)((uint64_t)cslots >> 32)) << 32);
                uint32_t hinst = 0;
                if (FLAGS) {
                    hs.dx = pull(s.dx);
                    hs.dy = pull(s.dy);
                    hs.dz = pull(s.dz);
                    hinst = pullu(cur_inst);
                }
                bool cand = false;
                float th = 0.0f;
                if (slot != kNoSlot) {
                    const SlotPtr tp = (SlotPtr)hslots + (uint64_t)slot * kSlotBytes;
                    const uint4 a = load_words(tp, 0), b = load_words(tp, 1), c = load_words(tp, 2);
                    if (STATS) ++st_tris;
                    float bu, bv;
                    if (FLAGS && (c.w & kTriAabb)) {
                        // AABB primitive: the intersection program of its hit record
                        const float lo[3] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z)};
                        const float hi[3] = {__uint_as_float(a.w), __uint_as_float(b.x), __uint_as_float(b.y)};
                        const float ro[3] = {hs.ox, hs.oy, hs.oz}, rd[3] = {hs.dx, hs.dy, hs.dz};
                        float pn[3];
                        cand = !(ray_flags & kRaySkipAabbs) &&
                               procedural_hit<float>(
                                   intersection_program(args, table + (hinst & kInstIdMask), c.z), lo, hi, ro,
                                   rd, smin, smax, th, bu, bv, pn);
                    } else {
                        cand = !(ray_flags & kRaySkipTriangles) &&
                               test_triangle(a, b, c, hs, hh, smin, smax, th, bu, bv) &&
                               !(ray_flags & (kRayCullBack | kRayCullFront) &&
                                 facing_culled(a, b, c, hs, ray_flags, table[hinst & kInstIdMask].flags));
                    }
                    if (FLAGS && cand) cand = candidate_accepted(args, ray_flags, c.w, c.z, hinst, table, bu, bv);
                }
                const uint64_t hits = __builtin_amdgcn_ballot_w64(cand);
                if (hits) {
                    uint32_t t0, t1;  // the owner's two distances
                    if (LEAN) {
                        t0 = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(rank << 3), (int)__float_as_uint(th));
                        t1 = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(rank << 3) + 4, (int)__float_as_uint(th));
                    } else {
                        if (cand) ((__attribute__((address_space(3))) float*)(tasks + (lane >> 1)))[lane & 1u] = th;
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    }
                    const uint32_t own = owner ? (uint32_t)(hits >> (2u * rank)) & 3u : 0u;
                    if (own) {
                        if (MODE == kModeAny || ((MODE == kModeFused || kTrain) && shadow_ray)) {
                            occl = true;
                            done = true;
                        } else {
                            if (!LEAN) {
                                const Words2 w = *(__attribute__((address_space(3))) Words2*)(tasks + rank);
                                t0 = w.x;
                                t1 = w.y;
                            }
                            // Exact ties in t go to the smaller (instance, slot), so the closest hit does not
                            // depend on the order in which a lane meets its candidates (which the wave's leaf
                            // scheduling can change).  A ray's first hit may round past its tmax.
                            const uint32_t ci = cur_inst & kInstIdMask;
#pragma unroll
                            for (int k = 0; k < 2; ++k) {
                                const float tn = s.toff + __uint_as_float(k ? t1 : t0);
                                const uint32_t sl = k ? slot1 : slot0;
                                const bool closer = !(tn >= tc) || hit_inst == kNoHit ||
                                                    (tn == tc && (ci < hit_inst || (ci == hit_inst && sl < hit_slot)));
                                if ((own >> k & 1u) && closer) {
                                    tc = tn;
                                    hit_inst = ci;
                                    hit_slot = sl;
                                }
                            }
                            if (ray_flags & kRayTerminateOnFirstHit) done = true;
                        }
                    }
                }
            }
            if ((inst_lanes >= leaf_at || no_node) && enter) {
                // instance leaf: enter its BLAS
                const uint32_t m = lg_bits & 255u;
                const uint32_t k = (uint32_t)(__ffs(m) - 1);
                const uint32_t vm = lg_bits >> 8;
                lg_bits &= ~(1u << k);
                const uint32_t slot = lg_base + (uint32_t)__popc(vm & ((1u << k) - 1u));
                uint4 q = make_uint4(0u, 0u, 0u, 0u);
                if (slot < tlas_nslots) {
                    q = load_words(tslots + (uint64_t)slot * kSlotBytes, 3);
                    if (q.z >= tlas_ninst) q.w = 0u;
                } else {
                    fault = kErrBadAs;
                }
                const uint64_t blas = (uint64_t)q.x | ((uint64_t)q.y << 32);
                const uint32_t iid = q.z, imask = q.w;
                if ((imask & args.cull_mask & 255u) != 0u) {
                    if (STATS) ++st_insts;
                    // push the remaining TLAS work
                    if (lg_bits & 255u) push(make_uint2(lg_base, (lg_bits & 0xFFFFu) | kEntryLeaf | kEntryTlas));
                    if (ng_bits & 255u) push(make_uint2(ng_base, (ng_bits & 0xFFFFu) | kEntryTlas));
                    lg_bits = 0;
                    const InstanceInfo* info = table + iid;
                    const auto* bh = (const __attribute__((address_space(1))) AsHeader*)blas;
                    double M[12];
#pragma unroll
                    for (int kk = 0; kk < 12; ++kk) M[kk] = info->inv[kk];
                    if (kRayLds) {  // in the TLAS the current space is world space
                        wo[0] = s.ox;
                        wo[1] = s.oy;
                        wo[2] = s.oz;
                        wd[0] = s.dx;
                        wd[1] = s.dy;
                        wd[2] = s.dz;
                    }
                    double od[3], dd[3];
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        od[r] = M[4 * r] * wo[0] + M[4 * r + 1] * wo[1] + M[4 * r + 2] * wo[2] + M[4 * r + 3];
                        dd[r] = M[4 * r] * wd[0] + M[4 * r + 1] * wd[1] + M[4 * r + 2] * wd[2];
                    }
                    // entry distance of the padded BLAS box, in FP32: it only chooses how far the origin
                    // moves (hits between tmin and te stay in the window, whose lower end becomes
                    // tmin - te), so its rounding costs nothing but keeps the FP64 divisions off this path
                    const float lo3[3] = {bh->lo[0], bh->lo[1], bh->lo[2]};
                    const float hi3[3] = {bh->hi[0], bh->hi[1], bh->hi[2]};
                    float tn = -INFINITY;
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        const float pad = (hi3[a] - lo3[a]) * (1.0f / 64.0f) + 1e-30f;
                        const float da = (float)dd[a], oa = (float)od[a];
                        if (fabsf(da) > 1e-30f) {
                            const float r = __builtin_amdgcn_rcpf(da);
                            const float t1 = (lo3[a] - pad - oa) * r, t2 = (hi3[a] + pad - oa) * r;
                            tn = fmaxf(tn, fminf(t1, t2));
                        }
                    }
                    const double te = fmax((double)wtmin, (double)tn);
                    s.ox = (float)(od[0] + te * dd[0]);
                    s.oy = (float)(od[1] + te * dd[1]);
                    s.oz = (float)(od[2] + te * dd[2]);
                    s.dx = (float)dd[0];
                    s.dy = (float)dd[1];
                    s.dz = (float)dd[2];
                    s.toff = (float)te;
                    setup_space(s);
                    setup_shear(s, sh);
                    cslots = (SlotPtr)blas + kHeaderBytes;
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        crlo[a] = lo3[a];
                        cqs[a] = bh->qscale[a];
                    }
                    in_blas = true;
                    cur_inst = FLAGS ? iid | (((imask >> 10) & 3u) << 30) : iid;  // InstSlot mask | flags << 8
                    cur_nslots = bh->slot_count;
                    ng_base = 0;
                    ng_bits = cur_nslots ? ((1u << s.oct) | (1u << 8)) : 0u;
                }
            }
            // a lane without pending work pops its next group; a node group is taken on in this same step, also by the
            // lanes that have just tested their last triangles (popping at the start of a step: 4% slower)
            if (active && !done && !((lg_bits | ng_bits) & 255u)) {
                if (pops_entry(sp, D + GD)) {
                    --sp;
                    const uint2 e = stacked(sp);
                    if ((e.y & kEntryTlas) && in_blas) {
                        in_blas = false;
                        if (kRayLds) {
#pragma unroll
                            for (int k = 0; k < 3; ++k) {
                                wo[k] = lds_ray[k * blockDim.x];
                                wd[k] = lds_ray[(3 + k) * blockDim.x];
                            }
                        }
                        s.ox = wo[0];
                        s.oy = wo[1];
                        s.oz = wo[2];
                        s.dx = wd[0];
                        s.dy = wd[1];
                        s.dz = wd[2];
                        s.toff = 0.0f;
                        setup_space(s);
                        cslots = tslots;
                        cur_nslots = tlas_nslots;
#pragma unroll
                        for (int a = 0; a < 3; ++a) {
                            crlo[a] = trlo[a];
                            cqs[a] = tqs[a];
                        }
                    }
                    if (e.y & kEntryLeaf) {
                        lg_base = e.x;
                        lg_bits = e.y & 0xFFFFu;
                    } else {
                        ng_base = e.x;
                        ng_bits = e.y & 0xFFFFu;
                    }
                } else {
                    done = true;  // no work left, or this step's pushes went past the end (an overflow, below)
                }
            }
            if (!done && (ng_bits & 255u)) {
                const uint32_t om = ng_bits & 255u;
                const uint32_t j = (uint32_t)(__ffs(om) - 1);
                const uint32_t k = j ^ s.oct;
                const uint32_t vm = (ng_bits >> 8) & 255u;
                const uint32_t slot = ng_base + (uint32_t)__popc(vm & ((1u << k) - 1u));
                ng_bits &= ~(1u << j);
                if (ng_bits & 255u) push(make_uint2(ng_base, (ng_bits & 0xFFFFu) | (in_blas ? 0u : kEntryTlas)));
                if (slot >= cur_nslots) {
                    fault = kErrBadAs;
                    ng_bits = 0;
                    lg_bits = 0;
                } else {
                    const SlotPtr np = cslots + (uint64_t)slot * kSlotBytes;
                    const uint4 w0 = load_words(np, 0), w1 = load_words(np, 1), w2 = load_words(np, 2),
                                w3 = load_words(np, 3);
                    if (STATS) ++st_nodes;
                    const float smin = wtmin - s.toff;
                    const float smax = tc - s.toff;
                    const uint32_t hm = test_node(w0, w1, w2, w3, s, crlo, cqs, smin, smax);
                    const uint32_t imask = (w0.z >> 8) & 255u;
                    const uint32_t vmask = (w0.z >> 16) & 255u;
                    ng_base = w0.w;
                    ng_bits = (LEAN ? oct_permute(hm & imask, s.oct) : oct_lds.row[s.oct][hm & imask]) | (vmask << 8);
                    const uint32_t lg_new = (hm & ~imask) | (vmask << 8);
                    if (!(lg_bits & 255u)) {
                        lg_base = w0.w;
                        lg_bits = lg_new;
                    } else if (lg_new & 255u) {
                        // a leaf group is already pending: stack the new one
                        push(make_uint2(w0.w, (lg_new & 0xFFFFu) | kEntryLeaf | (in_blas ? 0u : kEntryTlas)));
                    }
                }
            }
            if (sp > D + GD) {
                fault = kErrStackOverflow;
                done = true;
            }
            if (fault) atomicOr(&args.state->error_flags, fault);
            if (done) {
                // the result is written at the next refill, together with the wave's other finished lanes
                finished = true;
                active = false;
                lg_bits = 0;
                ng_bits = 0;
                sp = 0;
            }
            busy_lanes = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(active));
            go = busy_lanes != 0u;
            if (++iter >= (int)args.refill_interval) {
                iter = 0;
                steps += args.refill_interval;
                if (steps > kMaxSteps) {
                    if (active) atomicOr(&args.state->error_flags, kErrBadAs);
                    lg_bits = 0;
                    ng_bits = 0;
                    sp = 0;
                }
                go = go && (kTrain ? busy_lanes > train_floor : (wave_exhausted || busy_lanes >= args.refill_lanes));
            }
        }
    }

    if (kTrain && pt_rays) atomicAdd(&args.state->pt_rays, (unsigned long long)pt_rays);
    if (STATS) {
        atomicAdd(&args.state->stat_nodes, (unsigned long long)st_nodes);
        atomicAdd(&args.state->stat_tris, (unsigned long long)st_tris);
        atomicAdd(&args.state->stat_insts, (unsigned long long)st_insts);
        atomicAdd(&args.state->stat_rays, (unsigned long long)st_rays);
    }
}

// Occupancy variants of the same traversal: unconstrained registers (three waves per SIMD at least), at most 128 VGPRs
// (four waves) and at most 96 VGPRs (five waves, LEAN), chosen by the waves per SIMD that the launch shape asks for.
template <int MODE, bool STATS, bool FLAGS>
__global__ __launch_bounds__(256) void trace_kernel(TraceArgs args) {
    trace_body<MODE, STATS, FLAGS, false>(args);
}
template <int MODE, bool STATS, bool FLAGS, bool LEAN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void trace_kernel_w4(TraceArgs args) {
    trace_body<MODE, STATS, FLAGS, LEAN>(args);
}

template <int MODE, bool STATS, bool FLAGS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void trace_kernel_w5(TraceArgs args) {
    trace_body<MODE, STATS, FLAGS, true>(args);
}

__global__ void reset_counter_kernel(DeviceState* st, int clear_stats) {
    if (blockIdx.x == 0 && threadIdx.x < kRayQueues) st->queue[threadIdx.x].next = 0;
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        if (clear_stats) {
            st->stat_nodes = 0;
            st->stat_tris = 0;
            st->stat_insts = 0;
            st->stat_rays = 0;
        }
    }
}

template <int MODE, bool STATS, bool FLAGS>
hipError_t launch_variant(const TraceArgs& a, const TraceLaunch& L, const TracePlan& p, hipStream_t s) {
    if (L.waves >= 5)
        trace_kernel_w5<MODE, STATS, FLAGS><<<p.grid, L.block_size, p.lds, s>>>(a);
    else if (p.lean)
        trace_kernel_w4<MODE, STATS, FLAGS, true><<<p.grid, L.block_size, p.lds, s>>>(a);
    else if (L.waves == 4)
        trace_kernel_w4<MODE, STATS, FLAGS, false><<<p.grid, L.block_size, p.lds, s>>>(a);
    else
        trace_kernel<MODE, STATS, FLAGS><<<p.grid, L.block_size, p.lds, s>>>(a);
    return hipGetLastError();
}

// ray flags that need the FLAGS variant
constexpr uint32_t kActiveRayFlags = kRayTerminateOnFirstHit | kRaySkipClosestHit | kRayCullBack | kRayCullFront |
                                     kRayCullOpaque | kRayCullNoOpaque | kRayNoOpaque | kRaySkipTriangles |
                                     kRaySkipAabbs;

template <int M>
using ModeC = std::integral_constant<int, M>;

}  // namespace

// The FLAGS variant resolves opacity and runs any-hit programs (needed for non-opaque content unless the ray is
// OPAQUE), runs intersection programs (AABB content) and applies the ray-flag culls; the default variant treats
// every primitive as an opaque triangle.
static_assert(kFlagsVariantRayFlags == kActiveRayFlags, "one set of ray flags selects the FLAGS variant");
bool trace_needs_flags(uint32_t ray_flags, uint32_t content) { return needs_flags_variant(ray_flags, content); }

hipError_t trace_rays_launch(const TraceRequest& r, const TraceLaunch& L, hipStream_t s) {
    TraceArgs a{};
    a.tlas = (const uint8_t*)r.tlas;
    a.rays = r.rays;
    a.n_ptr = r.n_ptr;
    a.rays2 = r.rays2;
    a.n2_ptr = r.n2_ptr;
    a.path_hits = r.path_hits;
    a.n = r.n;
    a.cull_mask = r.cull_mask;
    a.hits = r.hits;
    a.occluded = r.occluded;
    for (int k = 0; k < 3; ++k) {
        a.cam[k] = r.cam[k];
        a.miss[k] = r.miss[k];
    }
    a.ax = r.ax;
    a.ay = r.ay;
    a.width = r.width;
    a.height = r.height;
    a.tmin = r.tmin;
    a.tmax = r.tmax;
    a.records = r.records;
    a.nrec = r.nrec;
    a.sbt_offset = r.sbt_offset;
    a.sbt_stride = r.sbt_stride;
    a.film = r.film;
    a.state = r.state;
    a.gstack = r.gstack;
    a.lds_depth = L.lds_depth;
    a.gdepth = L.gdepth;
    a.ray_chunk = L.ray_chunk;
    a.refill_lanes = L.refill_lanes;
    a.refill_interval = L.refill_interval;
    a.leaf_lanes = L.leaf_lanes;
    a.ray_flags = r.ray_flags;
    if (r.mode >= 5 && r.mode <= 7) {
        // whole paths: opaque triangle geometry and no ray flags only (the default traversal variant)
        if (!r.pt || trace_needs_flags(0u, r.content)) return hipErrorInvalidValue;
        a.pt = *r.pt;
        a.pt_first = r.mode == 5 ? r.pt->npix : 0u;
        a.pt_sample = r.pt_sample;
    }
    if (r.n == 0 && !r.n_ptr) {
        reset_counter_kernel<<<1, 64, 0, s>>>(r.state, r.stats ? 1 : 0);
        return hipGetLastError();
    }
    // guard 3: both variants, each guarded by the TLAS content the device reads, so that one of them takes the rays
    const bool both = r.guard == 3u && r.mode <= 2 && !(r.ray_flags & kActiveRayFlags);
    for (uint32_t g = 1; g <= (both ? 2u : 1u); ++g) {
        const uint32_t c = !both ? r.content : (g == 1 ? 0u : (kContentAabb | kContentNonOpaque));
        const bool flags = r.mode < 5 && trace_needs_flags(a.ray_flags, c);
        TraceShape sh;
        sh.block_size = L.block_size;
        sh.blocks_per_cu = L.blocks_per_cu;
        sh.grid = L.grid;
        sh.waves_per_simd = L.waves >= 5u ? 5u : (L.waves == 4u ? 4u : 3u);
        const bool rays = flags || r.mode >= 3;  // as kRayLds in the kernel
        sh.lane_bytes = L.lds_depth * (uint32_t)sizeof(uint2) + (rays ? 6u * (uint32_t)sizeof(float) : 0u);
        sh.start_blocks = L.start_blocks;
        const TracePlan p = plan_trace(sh, L.ray_chunk, r.n_ptr ? 0u : r.n, r.mode >= 5);
        a.first_waves = p.first_waves;
        a.guard = both ? g : (r.guard == 1u || r.guard == 2u ? r.guard : 0u);
        const bool clear = r.stats && g == 1;
        if (p.queues || clear) reset_counter_kernel<<<1, 64, 0, s>>>(r.state, clear ? 1 : 0);
        const auto launch = [&](auto mode, auto stats) {
            constexpr int M = decltype(mode)::value;
            constexpr bool S = decltype(stats)::value;
            if constexpr (M < kModeTrain)
                if (flags) return launch_variant<M, S, true>(a, L, p, s);
            return launch_variant<M, S, false>(a, L, p, s);
        };
        const std::true_type on;
        const std::false_type off;
        hipError_t e;
        switch (r.mode) {
            case 0: e = r.stats ? launch(ModeC<kModeClosest>(), on) : launch(ModeC<kModeClosest>(), off); break;
            case 1: e = r.stats ? launch(ModeC<kModeAny>(), on) : launch(ModeC<kModeAny>(), off); break;
            case 3: e = launch(ModeC<kModePath>(), off); break;
            case 4: e = launch(ModeC<kModeFused>(), off); break;
            case 5: e = launch(ModeC<kModeTrain>(), off); break;
            case 6: e = launch(ModeC<kModePixelPaths>(), off); break;
            case 7: e = launch(ModeC<kModePixelCache>(), off); break;
            default: e = r.stats ? launch(ModeC<kModeRaygen>(), on) : launch(ModeC<kModeRaygen>(), off);
        }
        if (e) return e;
    }
    return hipSuccess;
}

}  // namespace rtx
