// Device-side data layouts and inline helpers of the gfx950 path tracer.
//
// Scene layout in HBM (all read-only during a render):
//   QNode    64 B  per 4-wide node (the default, below): origin, three scale
//                  exponents, 8-bit child bounds, child counts and links.
//   NodeRec  32 B  child records (RC_QNODE = 0).  The host FlatBVH is collapsed into 4-wide
//                  nodes; a wide node is stored as the 4 records of its
//                  children, side by side (128 B, one cache line), so one visit
//                  reads all child boxes with eight 128-bit loads.  Record
//                  fields: child box lo.xyz/hi.xyz, link, count.  count in
//                  1..kEmptyChild-1: leaf child whose triangles are
//                  tris[link, link + count); count == 0: interior child whose
//                  own wide node starts at record `link`; count == kEmptyChild:
//                  unused slot.  Wide nodes are laid out in preorder, so links
//                  always point forward.
//   TriRec   48 B  v0.xyz + original triangle id, v1.xyz + flags, v2.xyz,
//                  in BVH leaf order (the vertices themselves, so the FP64
//                  refinement sees exactly the input edges).
//   ShadeRec 16 B  geometric normal + material index, in original order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "raycer_hip.h"

namespace rcd {

struct alignas(32) NodeRec {
    float lo[3];
    float hi[3];
    uint32_t link;
    uint32_t count;
};
static_assert(sizeof(NodeRec) == 32, "NodeRec must be 32 bytes");

// RC_QNODE = 1 (default) stores each wide node in 64 bytes instead of 128:
// the child boxes as 8-bit offsets from the node's origin in units of a power
// of two per axis, widened by one unit on each side so the decoded boxes
// contain the exact ones.  Links are node indices.  2.6% faster on the
// 2M-triangle terrain than the 128-byte records (RC_QNODE = 0).  The scales
// are stored as floats: a visit takes them as they are (as exponent bytes they
// cost six more VALU instructions per visit).
#ifndef RC_QNODE
#define RC_QNODE 1
#endif
struct alignas(64) QNode {
    float origin[3];
    float scale[3];    // 2^e per axis: bound = origin + q * scale
    uint32_t qlo[3];   // per axis, child k's lower bound in byte k
    uint32_t qhi[3];
    uint32_t link[4];  // child k's stack entry: interior, node index; leaf, kLeafTag | count << 26 | first
                       // triangle; unused, kEmptyLeaf with the bounds reversed (lo 255, hi 0)
};
// RC_LDS_TOP = 1 keeps the first kTopNodes wide nodes (the upload puts the
// tree's breadth-first top there) in LDS for the traversal kernels.  Off: on
// the 2M-triangle terrain it was 1% slower than fetching those nodes through
// the caches (1,848 against 1,868 Msamples/s).
// RC_NODE_ORDER = 1 stores each wide node's interior children side by side
// (blocks in depth-first order); 0 (the default) keeps the collapse's
// preorder, a node followed by its first child's subtree.
#ifndef RC_NODE_ORDER
#define RC_NODE_ORDER 0
#endif
#ifndef RC_LDS_TOP
#define RC_LDS_TOP 0
#endif
#ifndef RC_TOP_NODES
#define RC_TOP_NODES 21
#endif
constexpr uint32_t kTopNodes = RC_TOP_NODES;  // 21: levels 0..2 of a 4-wide tree, 1,344 bytes
static_assert(sizeof(QNode) == 64, "QNode must be 64 bytes");
#if RC_QNODE
using NodeT = QNode;
#else
using NodeT = NodeRec;
#endif

// RC_TRI_EDGES 1: the FP32 decision's records hold v0 and the edges
// e1 = v1 - v0, e2 = v2 - v0 (rounded in FP32 on the host exactly as the
// kernel would round them), saving six subtractions per triangle test; the FP64
// decision keeps a second array with the vertices.
#ifndef RC_TRI_EDGES
#define RC_TRI_EDGES 0
#endif
struct alignas(16) TriRec {
    float4 v0;  // w: original triangle id (bits)
    float4 v1;  // w: flags (bit1 nonShadowing); e1 in the FP32 decision's records with RC_TRI_EDGES
    float4 v2;  // w: unused; e2 likewise
};
static_assert(sizeof(TriRec) == 48, "TriRec must be 48 bytes");

struct alignas(16) DevMaterial {
    float4 diffuse;   // w: flags (bits)
    float4 emittance; // w: shininess
    float4 ambient;
    float4 specular;
};

constexpr uint32_t kNoHit = 0x7fffffffu;
constexpr int kDeepStack = 256;  // words of a stack in global memory: a spill slot, a lane of the deep-stack kernel
constexpr int kDeepThreads = 2048;  // lanes of the deep-stack kernel

// Traversal stack of one lane: the top kRegStack entries in registers, deeper
// ones in LDS laid out [depth][lane] so a wave's accesses hit 64 distinct
// banks.  A pop takes its entry from a register, so the next node fetch never
// waits on an LDS read; the LDS refill of the bottom register runs off the
// critical path.  Every push spills the bottom register, so the LDS rows are
// the stack's capacity; registers start as kEmptyChild, and popping that is
// the end of the stack (no entry count).  A ray whose stack would outgrow
// kLdsStack entries moves them to global memory (stack_spill).  One register: each
// more costs a move per push and pop.  19 rows: with them eight 256-thread
// blocks of the traversal kernels fill the 160 KB of a CU.
#ifndef RC_REG_STACK
#define RC_REG_STACK 1
#endif
#ifndef RC_LDS_DEPTH
#define RC_LDS_DEPTH 19
#endif
constexpr int kRegStack = RC_REG_STACK;
constexpr int kLdsStack = RC_LDS_DEPTH;
static_assert(kLdsStack >= 1, "the traversal stack needs an LDS row");
constexpr int kStackLimitMax = 20;  // the largest rc_tuning.stack_limit (above kLdsStack: all the build holds)
constexpr int kWidth = 4;        // children per wide node
constexpr uint32_t kEmptyChild = 0xffffffffu;  // no entry: an unused child record, the end of a stack
constexpr uint32_t kEmptyLeaf = 0x80000000u;   // a leaf entry of no triangles: an unused slot of a QNode

// ---------------------------------------------------------------- RNG
// Philox4x32-10 (Salmon et al., SC'11): 10 rounds of two 32x32->64 products.
__device__ __forceinline__ uint4 philox(uint4 c, uint2 k) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r > 0) {
            k.x += 0x9E3779B9u;
            k.y += 0xBB67AE85u;
        }
        uint32_t hi0 = __umulhi(0xD2511F53u, c.x), lo0 = 0xD2511F53u * c.x;
        uint32_t hi1 = __umulhi(0xCD9E8D57u, c.z), lo1 = 0xCD9E8D57u * c.z;
        c = make_uint4(hi1 ^ c.y ^ k.x, lo1, hi0 ^ c.w ^ k.y, lo0);
    }
    return c;
}
// 24-bit uniform in [0,1), exact in FP32.
__device__ __forceinline__ float u01(uint32_t x) { return float(x >> 8) * (1.0f / 16777216.0f); }
constexpr uint32_t kCamDim = 0xFFFFFFFFu;
__device__ __forceinline__ float4 draw4(uint64_t seed, uint32_t pixel, uint32_t sample, uint32_t frame, uint32_t dim) {
    uint4 o = philox(make_uint4(pixel, sample, frame, dim), make_uint2(uint32_t(seed), uint32_t(seed >> 32)));
    return make_float4(u01(o.x), u01(o.y), u01(o.z), u01(o.w));
}

// Pixel order of the slots of a pass: the 8x8 tiles of the largest tiled
// region first (tiles row by row, pixels row by row inside a tile), then the
// right strip and the bottom strip row by row.  A wave of 64 consecutive slots
// is one 8x8 tile, and since the queues keep slot order from bounce to bounce
// its rays start from nearby points at every bounce.
struct PixelOrder {
    uint32_t width, tiles_x, x0, y0, a;  // x0 = 8 tiles_x, y0 = 8 tiles_y, a = x0 y0
};

inline PixelOrder make_order(uint32_t w, uint32_t h) {
    PixelOrder o;
    o.width = w;
    o.tiles_x = w / 8;
    o.x0 = 8 * (w / 8);
    o.y0 = 8 * (h / 8);
    o.a = o.x0 * o.y0;
    return o;
}

__host__ __device__ __forceinline__ uint32_t order_to_pixel(const PixelOrder& o, uint32_t q) {
    if (q < o.a) {
        const uint32_t t = q >> 6, w = q & 63u, ty = t / o.tiles_x, tx = t - ty * o.tiles_x;
        return (ty * 8 + (w >> 3)) * o.width + tx * 8 + (w & 7u);
    }
    uint32_t r = q - o.a;
    const uint32_t rw = o.width - o.x0;
    if (r < rw * o.y0) {
        const uint32_t y = r / rw;
        return y * o.width + o.x0 + (r - y * rw);
    }
    r -= rw * o.y0;
    return o.y0 * o.width + r;
}

__host__ __device__ __forceinline__ uint32_t pixel_to_order(const PixelOrder& o, uint32_t p) {
    const uint32_t y = p / o.width, x = p - y * o.width;
    if (x < o.x0 && y < o.y0) return ((((y >> 3) * o.tiles_x + (x >> 3)) << 6) | ((y & 7u) << 3) | (x & 7u));
    if (y < o.y0) return o.a + y * (o.width - o.x0) + (x - o.x0);
    return o.a + (o.width - o.x0) * o.y0 + (p - o.y0 * o.width);
}

// A pass's queue slot <-> (tile-order index, sample within the pass).
// Pixel-major (RC_PIXEL_MAJOR = 1, the default): slot = index * spp_pass + j,
// the pass's samples of one pixel side by side, so a wave's rays start from
// nearly one point (its sun shadow rays nearly coincide): 4% faster on the
// 2M-triangle terrain at 64 samples per pass than sample-major (0: slot =
// j * npix + index, a wave holding 64 neighbouring pixels of one sample).
#ifndef RC_PIXEL_MAJOR
#define RC_PIXEL_MAJOR 1
#endif
__host__ __device__ __forceinline__ uint32_t slot_index(uint32_t slot, uint32_t npix, uint32_t spp_pass) {
    return RC_PIXEL_MAJOR ? slot / spp_pass : slot % npix;
}
__host__ __device__ __forceinline__ uint32_t slot_sample_in_pass(uint32_t slot, uint32_t npix, uint32_t spp_pass) {
    return RC_PIXEL_MAJOR ? slot % spp_pass : slot / npix;
}

// CMJSampler's permute (CMJSampler.cpp:12-44): Kensler's hash-based
// permutation of [0, l) ("Correlated Multi-Jittered Sampling", Pixar Technical
// Memo 13-01, 2013) in the reference's 64-bit arithmetic.  The hash is a
// bijection of [0, 2^k) with 2^k >= l, so cycle walking ends within 2^k steps.
__device__ __forceinline__ uint64_t cmj_permute(uint64_t i, uint64_t l, uint64_t p) {
    uint64_t w = l - 1;
    w |= w >> 1;
    w |= w >> 2;
    w |= w >> 4;
    w |= w >> 8;
    w |= w >> 16;
    do {
        i ^= p;
        i *= 0xe170893dull;
        i ^= p >> 16;
        i ^= (i & w) >> 4;
        i ^= p >> 8;
        i *= 0x0929eb3full;
        i ^= p >> 23;
        i ^= (i & w) >> 1;
        i *= 1 | p >> 27;
        i *= 0x6935fa69ull;
        i ^= (i & w) >> 11;
        i *= 0x74dcb303ull;
        i ^= (i & w) >> 2;
        i *= 0x9e501cc3ull;
        i ^= (i & w) >> 2;
        i *= 0xc860a3dfull;
        i &= w;
        i ^= i >> 5;
    } while (i >= l);
    return (i + p) % l;
}

// The per-pixel permutation of generateMultiSamples (Tracer.cpp:129-130), one
// 64-bit draw per pixel and frame, shared by all the pixel's samples.
constexpr uint32_t kPermDim = 0xFFFFFFFEu;
__device__ __forceinline__ uint64_t pixel_permutation(uint64_t seed, uint32_t pixel, uint32_t frame) {
    uint4 o = philox(make_uint4(pixel, 0u, frame, kPermDim), make_uint2(uint32_t(seed), uint32_t(seed >> 32)));
    return uint64_t(o.x) | (uint64_t(o.y) << 32);
}

// Sampler::getSample2D of each SamplerType (src/Rendering/Samplers/) for
// stratum (x, y) of an n x n pattern, with the jitter (r0, r1) and the
// permutation perm (CMJ only).
__device__ __forceinline__ float2 sample_point(uint32_t type, uint32_t x, uint32_t y, uint32_t n, uint64_t perm,
                                               float r0, float r1) {
    switch (type) {
    case RC_SAMPLER_JITTERED:  // JitteredSampler.cpp:21-34
        return make_float2((float(x) + r0) / float(n), (float(y) + r1) / float(n));
    case RC_SAMPLER_RANDOM:  // RandomSampler.cpp:23-35
        return make_float2(r0, r1);
    case RC_SAMPLER_CENTER:  // CenterSampler.cpp:19-33
        return make_float2(0.5f, 0.5f);
    case RC_SAMPLER_REGULAR:  // RegularSampler.cpp:19-34
        return make_float2((float(x) + 0.5f) / float(n), (float(y) + 0.5f) / float(n));
    case RC_SAMPLER_CMJ: {  // CMJSampler.cpp:57-77
        const float sx = float(cmj_permute(x, n, perm * 0x68bc21ebull));
        const float sy = float(cmj_permute(y, n, perm * 0x02e5be93ull));
        return make_float2((float(x) + (sy + r0) / float(n)) / float(n), (float(y) + (sx + r1) / float(n)) / float(n));
    }
    default:  // PoissonDiscSampler::getSample2D returns (0, 0) (PoissonDiscSampler.cpp:22-32)
        return make_float2(0.0f, 0.0f);
    }
}

// ---------------------------------------------------------------- vec math
__device__ __forceinline__ float3 f3(float4 a) { return make_float3(a.x, a.y, a.z); }
__device__ __forceinline__ float3 operator+(float3 a, float3 b) { return make_float3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ float3 operator-(float3 a, float3 b) { return make_float3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ float3 operator*(float3 a, float s) { return make_float3(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ float3 operator*(float s, float3 a) { return make_float3(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ float3 mul3(float3 a, float3 b) { return make_float3(a.x * b.x, a.y * b.y, a.z * b.z); }
__device__ __forceinline__ float dot3(float3 a, float3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ float3 cross3(float3 a, float3 b) {
    return make_float3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ float3 normalize3(float3 a) { return a * (1.0f / sqrtf(dot3(a, a))); }

// Direction with no zero component, so 1/d is finite and the slab products
// never form 0 * inf.
__device__ __forceinline__ float3 safe_inv(float3 d) {
    const float e = 1e-20f;
    float x = fabsf(d.x) < e ? copysignf(e, d.x) : d.x;
    float y = fabsf(d.y) < e ? copysignf(e, d.y) : d.y;
    float z = fabsf(d.z) < e ? copysignf(e, d.z) : d.z;
    return make_float3(1.0f / x, 1.0f / y, 1.0f / z);
}

// FP32 Möller–Trumbore with the reference's structure (Triangle.cpp:61-91):
// double-sided; the determinant test is the scale-free det == 0 instead of
// |det| < epsilon.  This is a conservative filter: the barycentric bounds are
// widened by kFilterBand so FP32 rounding never rejects a triangle the FP64
// decision (mt_hit64, inclusive bounds) would accept.
constexpr float kFilterBand = 1e-3f;
// RC_FAST_RCP 1: the FP32 filter's 1/det is the hardware reciprocal (1 ulp;
// the filter bands absorb it and FP64 decides).
#ifndef RC_FAST_RCP
#define RC_FAST_RCP 1
#endif
__device__ __forceinline__ bool mt_hit(const TriRec& T, float3 o, float3 d, float& t) {
    float3 v0 = f3(T.v0);
    float3 e1 = f3(T.v1) - v0, e2 = f3(T.v2) - v0;
    float3 pv = cross3(d, e2);
    float det = dot3(e1, pv);
    if (det == 0.0f) return false;
#if RC_FAST_RCP
    // hardware reciprocal (1 ulp): the bands above absorb it, FP64 decides
    float inv = __builtin_amdgcn_rcpf(det);
#else
    float inv = 1.0f / det;
#endif
    float3 tv = o - v0;
    float u = dot3(tv, pv) * inv;
    if (u < -kFilterBand || u > 1.0f + kFilterBand) return false;
    float3 qv = cross3(tv, e1);
    float v = dot3(d, qv) * inv;
    if (v < -kFilterBand || u + v > 1.0f + kFilterBand) return false;
    t = dot3(e2, qv) * inv;
    return true;
}

// The same test in FP64 on the exact FP32 inputs, for candidates the filter
// accepted: it decides the winner and gives t to FP64 accuracy, so sliver
// triangles at grazing angles (where FP32 t loses ~1e-4) still resolve like
// the FP64 reference.
__device__ __forceinline__ bool mt_hit64(const TriRec& T, float3 of, float3 df, double& t, double& u, double& v) {
    const double v0x = T.v0.x, v0y = T.v0.y, v0z = T.v0.z;
    const double e1x = double(T.v1.x) - v0x, e1y = double(T.v1.y) - v0y, e1z = double(T.v1.z) - v0z;
    const double e2x = double(T.v2.x) - v0x, e2y = double(T.v2.y) - v0y, e2z = double(T.v2.z) - v0z;
    const double dx = df.x, dy = df.y, dz = df.z;
    const double px = dy * e2z - dz * e2y, py = dz * e2x - dx * e2z, pz = dx * e2y - dy * e2x;
    const double det = e1x * px + e1y * py + e1z * pz;
    if (det == 0.0) return false;
    const double inv = 1.0 / det;
    const double tx = double(of.x) - v0x, ty = double(of.y) - v0y, tz = double(of.z) - v0z;
    u = (tx * px + ty * py + tz * pz) * inv;
    if (u < 0.0 || u > 1.0) return false;
    const double qx = ty * e1z - tz * e1y, qy = tz * e1x - tx * e1z, qz = tx * e1y - ty * e1x;
    v = (dx * qx + dy * qy + dz * qz) * inv;
    if (v < 0.0 || (u + v) > 1.0) return false;
    t = (e2x * qx + e2y * qy + e2z * qz) * inv;
    return true;
}

// The FP32 decision (the default, RC_HIT_FP32): Triangle::intersect's
// Möller–Trumbore (Triangle.cpp:61-91) and its OpenCL form
// (data/opencl/intersections.cl:27-68) in FP32, double-sided, inclusive
// barycentric bounds, with the scale-free det == 0 instead of |det| <
// epsilon.  The bounds are tested without a division: u = U/det and v =
// V/det lie in [0, 1] with u + v <= 1 exactly when sign(det) U, sign(det) V
// >= 0 and their sum <= |det|; t = T/det is one IEEE division for the
// triangles that pass.  u and v are returned undivided (U, V and adet = |det|).
__device__ __forceinline__ bool mt_dec32(const TriRec& T, float3 o, float3 d, float& t, float& U, float& V,
                                         float& adet) {
    const float3 v0 = f3(T.v0);
    const float3 e1 = RC_TRI_EDGES ? f3(T.v1) : f3(T.v1) - v0, e2 = RC_TRI_EDGES ? f3(T.v2) : f3(T.v2) - v0;
    const float3 pv = cross3(d, e2);
    const float det = dot3(e1, pv);
    const float sg = det < 0.0f ? -1.0f : 1.0f;
    adet = fabsf(det);
    const float3 tv = o - v0;
    U = sg * dot3(tv, pv);
    // one branch for both tests, so the load of v0 is not sunk behind the first
    if (det == 0.0f || U < 0.0f || U > adet) return false;
    const float3 qv = cross3(tv, e1);
    V = sg * dot3(d, qv);
    if (V < 0.0f || U + V > adet) return false;
    t = dot3(e2, qv) / det;
    return true;
}

// Relative window inside which an FP32 distance defers to the FP64 one.
constexpr float kRefineWindow = 1e-3f;
// FP32 decision: nodes are culled a hair beyond the best distance so a
// triangle at exactly that distance (an exact tie) is still reached.
constexpr float kTieWindow = 4.0f / 16777216.0f;

// A lane's stack memory: rows of `stride` bytes in an array shared by the
// lanes, row r of the lane at byte offset base + r * stride (base = 4 * lane <
// stride).  end is the offset past row `limit` of every lane (uniform), so a
// lane whose next free row is at p may push m entries exactly when
// p + m * stride < end.  spill: the launch's count->slots stacks in global
// memory, handed out by count->claimed, for lanes whose rows are full; null:
// none.
struct SpillCount {
    unsigned long long total;  // rays whose stack outgrew its rows
    uint32_t claimed;          // stacks the launch's rays asked for
    uint32_t slots;            // those there are, at most kMaxSpillSlots (here, not an argument: it costs no register)
};
struct StackMem {
    uint32_t* array;
    int base, stride, end;
    uint32_t* spill;
    SpillCount* count;
    __device__ __forceinline__ uint32_t& at(int p) const {
        return *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(array) + uint32_t(p));
    }
};
__device__ __forceinline__ StackMem stack_mem(uint32_t* array, uint32_t lane, int lanes, int limit,
                                              uint32_t* spill = nullptr, SpillCount* count = nullptr) {
    return StackMem{array, int(4 * lane), 4 * lanes, 4 * lanes * (limit + 1), spill, count};
}
// Rows the three entries of a node visit need above a stack just spilled: with
// fewer nothing is spilled.
constexpr int kSpillRows = 4;
// A traversal's spilled stack in one word: 1 + its slot above, the blocks of
// rows in it below.  A block takes the lane's rows and their number, so there
// are at most kDeepStack / (kSpillRows + 1) of them.
constexpr int kSpillBlockBits = 6;
constexpr uint32_t kSpillMask = 0x007fffffu, kSpillBlocks = (1u << kSpillBlockBits) - 1u;
constexpr uint32_t kMaxSpillSlots = kSpillMask >> kSpillBlockBits;  // 131,071
static_assert(kDeepStack / (kSpillRows + 1) <= int(kSpillBlocks), "a slot's blocks do not fit their bits");

// The stack's registers and the offset of its next free row.
struct Stack {
    int p;
    uint32_t reg[kRegStack > 0 ? kRegStack : 1];  // top first
};
__device__ __forceinline__ void stack_reset(Stack& K, const StackMem& M) {
    K.p = M.base;
#pragma unroll
    for (int k = 0; k < kRegStack; ++k) K.reg[k] = kEmptyChild;
    if (kRegStack == 0) {  // the end marker lies in row 0
        M.at(K.p) = kEmptyChild;
        K.p += M.stride;
    }
}
// Push without a check: the caller has seen that the rows hold it.
__device__ __forceinline__ void stack_push(Stack& K, const StackMem& M, uint32_t x) {
    if (kRegStack == 0) {
        M.at(K.p) = x;
    } else {
        M.at(K.p) = K.reg[kRegStack - 1];
#pragma unroll
        for (int k = kRegStack - 1; k > 0; --k) K.reg[k] = K.reg[k - 1];
        K.reg[0] = x;
    }
    K.p += M.stride;
}
// The top entry, or kEmptyChild when the stack is empty (then it is not to be
// popped again).  At the end of the stack row 0 is read, the lane's own; its
// value is not used.
__device__ __forceinline__ uint32_t stack_pop(Stack& K, const StackMem& M) {
    K.p = max(K.p - M.stride, M.base);
    if (kRegStack == 0) return M.at(K.p);
    const uint32_t x = K.reg[0];
#pragma unroll
    for (int k = 0; k < kRegStack - 1; ++k) K.reg[k] = K.reg[k + 1];
    K.reg[kRegStack - 1] = M.at(K.p);
    return x;
}

// The barycentrics of the hit are u / w and v / w: the FP32 decision keeps
// them undivided (w = |det|) so only a reader of u and v pays the divisions
// (bary_u / bary_v); the FP64 decision stores them divided, with w = 1.
// Streamed accesses: queue entries, path states, slot radiance and parked
// traversals are written once and read once per bounce.  RC_NT_QUEUES 1 makes
// them nontemporal loads and stores, so they do not displace nodes and
// triangles from L2 and the Infinity Cache.
#ifndef RC_NT_QUEUES
#define RC_NT_QUEUES 0
#endif
typedef float v4f_t __attribute__((ext_vector_type(4)));
typedef uint32_t v4u_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 ld_stream(const float4* p) {
    if constexpr (RC_NT_QUEUES) {
        const v4f_t v = __builtin_nontemporal_load(reinterpret_cast<const v4f_t*>(p));
        return make_float4(v.x, v.y, v.z, v.w);
    } else {
        return *p;
    }
}
__device__ __forceinline__ void st_stream(float4* p, float4 v) {
    if constexpr (RC_NT_QUEUES) {
        __builtin_nontemporal_store(v4f_t{v.x, v.y, v.z, v.w}, reinterpret_cast<v4f_t*>(p));
    } else {
        *p = v;
    }
}
__device__ __forceinline__ uint4 ld_stream(const uint4* p) {
    if constexpr (RC_NT_QUEUES) {
        const v4u_t v = __builtin_nontemporal_load(reinterpret_cast<const v4u_t*>(p));
        return make_uint4(v.x, v.y, v.z, v.w);
    } else {
        return *p;
    }
}
__device__ __forceinline__ void st_stream(uint4* p, uint4 v) {
    if constexpr (RC_NT_QUEUES) {
        __builtin_nontemporal_store(v4u_t{v.x, v.y, v.z, v.w}, reinterpret_cast<v4u_t*>(p));
    } else {
        *p = v;
    }
}

struct TraceResult {
    float t, u, v;
    uint32_t id;
    bool overflow;
    float w;
};
__device__ __forceinline__ float bary_u(const TraceResult& R) { return R.u / R.w; }
__device__ __forceinline__ float bary_v(const TraceResult& R) { return R.v / R.w; }

// Workgroups are dealt to the 8 XCDs round-robin (workgroup w runs on XCD
// w % 8).  This bijection on [0, n) gives XCD x the contiguous range of
// logical blocks [x n / 8, (x + 1) n / 8), so each XCD's private L2 sees a
// contiguous, spatially coherent slice of the ray queue.
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t xcd_block(uint32_t w, uint32_t n) {
    uint32_t x = w % kXcds, local = w / kXcds;
    uint32_t per = n / kXcds, rem = n % kXcds;
    return x < rem ? x * (per + 1) + local : rem * (per + 1) + (x - rem) * per + local;
}

// Wave-wide sum, one 64-bit atomic per wave (every lane must call it).
__device__ __forceinline__ void wave_add(unsigned long long* dst, uint32_t v) {
    unsigned long long x = v;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    if ((threadIdx.x & 63) == 0 && x) atomicAdd(dst, x);
}

// Tests the triangles tris[first, first + count).  DEC64: candidates pass
// the FP32 filter within kRefineWindow of the current best and are then
// decided in FP64 on the exact FP32 inputs (RC_HIT_FP64); otherwise the FP32
// test decides (mt_dec32).  Closest hit keeps the smallest t; an exact tie
// goes to the lower original triangle id, so the answer does not depend on
// traversal order.  Returns true when an any-hit query is answered (its R.t
// holds tmax until then).
template <bool DEC64>
struct BestT {
    using T = float;
};
template <>
struct BestT<true> {
    using T = double;
};

template <bool ANY, bool COUNT, bool DEC64>
__device__ __forceinline__ bool test_leaf(const TriRec* __restrict__ tris, uint32_t first, uint32_t count, float3 o,
                                          float3 d, float tmin, typename BestT<DEC64>::T& best, TraceResult& R,
                                          uint32_t& n_tri) {
    for (uint32_t j = first; j < first + count; ++j) {
        const float4* q = reinterpret_cast<const float4*>(reinterpret_cast<const char*>(tris) + j * 48u);  // < 4 GiB
        TriRec T;
        T.v0 = q[0];
        T.v1 = q[1];
        T.v2 = q[2];
        if (COUNT) n_tri += 1;
        if (DEC64) {
            float t32;
            if (!mt_hit(T, o, d, t32)) continue;
            if (t32 > R.t * (1.0f + kRefineWindow) || t32 < tmin * (1.0f - kRefineWindow) - 1e-30f) continue;
            double t64, u64, v64;
            if (!mt_hit64(T, o, d, t64, u64, v64)) continue;
            if (t64 < double(tmin)) continue;
            uint32_t id = __float_as_uint(T.v0.w);
            if (ANY) {
                if (t64 <= double(R.t) && !(__float_as_uint(T.v1.w) & RC_MAT_NON_SHADOWING)) {
                    R.t = float(t64);
                    R.id = id;
                    return true;
                }
            } else if (t64 < best || (t64 == best && id < R.id)) {
                best = t64;
                R.t = float(t64);
                R.u = float(u64);
                R.v = float(v64);
                R.w = 1.0f;
                R.id = id;
            }
        } else {
            float t, U, V, adet;
            if (!mt_dec32(T, o, d, t, U, V, adet)) continue;
            if (t < tmin) continue;
            uint32_t id = __float_as_uint(T.v0.w);
            if (ANY) {
                if (t <= R.t && !(__float_as_uint(T.v1.w) & RC_MAT_NON_SHADOWING)) {
                    R.t = t;
                    R.id = id;
                    return true;
                }
            } else if (t < R.t || (t == R.t && id < R.id)) {
                R.t = t;
                R.u = U;
                R.v = V;
                R.w = adet;
                R.id = id;
            }
        }
    }
    return false;
}

// How far past a distance the boxes are still entered: a relative window that
// covers the decision's ties and refinements.
template <bool DEC64>
__device__ __forceinline__ float cull_at(float t) {
    return t * (1.0f + (DEC64 ? kRefineWindow : kTieWindow));
}

// Compare-exchange of two children (entry distance in the high word, stack
// entry in the low one) by distance.  As doubles the words order by the
// distances' bits (both are non-negative floats, whose bits order as they do
// and stay below a double's infinity), so one v_min_f64 and one v_max_f64 move
// the distance and its entry together: 8 cycles of a SIMD against 20 for a
// compare and four selects (full-rate VALU instructions take 2 cycles per
// wave on this chip: FMA, add, multiply, and / or / xor, moves; minima,
// compares, selects, conversions and FP64 take 4).
__device__ __forceinline__ void order2(double& a, double& b) {
    double lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
}

// 1: the if-if traversal (leaves postponed onto the stack), 2% faster on the
// 2M-triangle terrain than testing leaf children at once (0, with the 128-byte
// node records).
#ifndef RC_TRAV_IFIF
#define RC_TRAV_IFIF 1
#endif
// 1: any-hit queries visit children nearest first too; 0: in slot order (an
// any-hit answer does not depend on the order, only its cost does).
#ifndef RC_ANY_SORT
#define RC_ANY_SORT 0
#endif
// 0: off; n > 0: leaves are set aside and tested when at least n / 64 of the
// wave's lanes hold one (or none has a node), the lanes meanwhile going on
// with their stacks.
#ifndef RC_LEAF_POSTPONE
#define RC_LEAF_POSTPONE 20
#endif
// The same threshold for any-hit queries.
#ifndef RC_LEAF_POSTPONE_ANY
#define RC_LEAF_POSTPONE_ANY 32
#endif
// RC_PACKET_CAMERA = 1: the camera bounce's waves (one pixel's samples each,
// with pixel-major slots) traverse as packets (traverse_packet); 0 (the
// default): each lane on its own, as the other bounces.  On the 2M-triangle
// terrain at 64 samples per pass the packets made the camera bounce 1.6 ms
// slower (12.5 against 14.1 ms): the union of a pixel's 64 traversals costs
// more visits than the per-lane traversal's leaf postponing and culling.
#ifndef RC_PACKET_CAMERA
#define RC_PACKET_CAMERA 0
#endif
// Whether every traversal of the build spills a stack that is full
// (stack_spill); traverse_inline and traverse_packet list its ray instead.
constexpr bool kSpillsInPlace = RC_QNODE ? !RC_PACKET_CAMERA : RC_TRAV_IFIF != 0;
// Stack entries of the if-if traversal: an interior child's record index, or
// a leaf tagged with kLeafTag, its triangle count (0..31) in bits 26..30 and
// its first triangle (< 2^26) below.  The upload guarantees both: scenes hold
// at most 2^26 triangles and longer leaves are split into wide nodes.  As
// signed numbers: interior entries are >= 0, leaves < -1, kEmptyChild is -1.
constexpr uint32_t kLeafTag = 0x80000000u;
constexpr uint32_t kMaxLeafRecord = 32;           // leaf records hold fewer triangles
constexpr size_t kMaxTriangles = size_t(1) << 26;
__device__ __forceinline__ bool is_node(uint32_t e) { return int32_t(e) >= 0; }
__device__ __forceinline__ bool is_leaf(uint32_t e) { return int32_t(e) < -1; }

// A traversal's state.  The boxes are tested in ray distances scaled by a power
// of two (so every product and comparison is the unscaled one) that puts the
// scene's end of the ray, or tmax when that is nearer, below 1: clamping an
// entry plane's FMA to [0, 1], which is free (a modifier), then takes the place
// of the maximum with 0, and 1 stays an entry past everything.  Past 2^126 no
// power of two is small enough: the last of a float's distances end at
// kFarthest, and a clamped entry plane there only lets boxes in that are
// further away.  The distances reported are the triangle tests', unscaled.
constexpr float kFarthest = 3.9999998f;  // the largest float, scaled by 2^-126
template <bool DEC64>
struct Trav {
    float3 o, d;
    float3 inv;   // 1 / d, no zero component (safe_inv), scaled
    uint32_t scale_spill;  // bits of the power of two (trav_scale); its mantissa's: the spilled stack (stack_spill)
    float tmin;
    bool late;    // wave-uniform: some ray of the wave has a tmin > 0, entries are held against it
    float cull;   // boxes entered beyond it are skipped (scaled)
    typename BestT<DEC64>::T best;  // DEC64: the best hit's FP64 distance; else unused (R.t is it)
    TraceResult R;
    uint32_t cur;
    Stack stack;
    uint32_t leaf;     // a leaf set aside (leaf postponing), else kEmptyChild
    const uint4* top;  // LDS copy of nodes [0, ntop), or null
    uint32_t ntop;
};

// Copies the first kTopNodes nodes into LDS `top` (four 16-byte words per
// node; the upload pads the array to as many); every thread of the block calls
// it, and it ends in a barrier.  Returns the count (0 with the 128-byte node
// records or with RC_LDS_TOP 0).
template <class N>
__device__ __forceinline__ uint32_t load_top(const N* __restrict__ nodes, uint4* top) {
    if constexpr (!RC_LDS_TOP || sizeof(N) != 64) {
        return 0u;
    } else {
        const uint4* src = reinterpret_cast<const uint4*>(nodes);
        for (uint32_t w = threadIdx.x; w < 4 * kTopNodes; w += blockDim.x) top[w] = src[w];
        __syncthreads();
        return kTopNodes;
    }
}

template <bool DEC64>
__device__ __forceinline__ float trav_scale(const Trav<DEC64>& S) {
    return __uint_as_float(S.scale_spill & ~kSpillMask);
}

// The cull distance for R.t (the best hit's, or tmax).
template <bool DEC64>
__device__ __forceinline__ void trav_cull(Trav<DEC64>& S) {
    S.cull = fminf(cull_at<DEC64>(S.R.t) * trav_scale(S), kFarthest);
}

// A stack whose rows are full: they move to a slot of global memory and the
// lane goes on with empty rows; when those are used up the rows come back
// (stack_reload).  The word in scale_spill names the slot and counts its
// blocks; 0 while nothing was spilled.  False when the launch's slots are all
// taken, the slot is full or the rows are too few: then the deep-stack kernel
// walks the ray again.  Before, it walked all of them: the few rays that
// outgrow the rows are a launch's longest, and walked twice, the second time
// alone on the chip.  An any-hit query over 777,777 segments in 200,000 random
// triangles takes 446 us against 514; the loop itself pays nothing (the word
// lies in unused bits and is looked at where a traversal ends or finds no room).
template <bool DEC64>
__device__ __forceinline__ bool stack_spill(Trav<DEC64>& S, const StackMem& M) {
    if (!M.spill || M.end < (kSpillRows + 1) * M.stride) return false;
    uint32_t w = S.scale_spill & kSpillMask;
    if (w == 0) {
        const uint32_t slot = atomicAdd(&M.count->claimed, 1u);
        if (slot >= M.count->slots) return false;
        atomicAdd(&M.count->total, 1ull);
        w = (slot + 1u) << kSpillBlockBits;
    }
    const uint32_t rows = uint32_t(S.stack.p - M.base) / uint32_t(M.stride);
    const uint32_t words = uint32_t(M.end) / uint32_t(M.stride);  // of a block
    const uint32_t at = (w & kSpillBlocks) * words;
    if (at + words > uint32_t(kDeepStack)) {
        atomicAdd(&M.count->total, ~0ull);  // the deep-stack kernel counts it
        return false;
    }
    uint32_t* q = M.spill + (((w >> kSpillBlockBits) - 1u) * uint32_t(kDeepStack) + at);
    q[words - 1u] = rows;
    for (int p = M.base; p < S.stack.p; p += M.stride) *q++ = M.at(p);
    S.scale_spill = (S.scale_spill & ~kSpillMask) | (w + 1u);
    M.at(M.base) = kEmptyChild;  // below the register entries
    S.stack.p = M.base + M.stride;
    return true;
}

// The rows spilled last, back into the used-up stack, and its top entry into
// S.cur; false when there are none.
template <bool DEC64>
__device__ __forceinline__ bool stack_reload(Trav<DEC64>& S, const StackMem& M) {
    const uint32_t w = S.scale_spill & kSpillMask;
    if ((w & kSpillBlocks) == 0) return false;
    const uint32_t words = uint32_t(M.end) / uint32_t(M.stride);
    const uint32_t* q =
        M.spill + (((w >> kSpillBlockBits) - 1u) * uint32_t(kDeepStack) + ((w & kSpillBlocks) - 1u) * words);
    const uint32_t rows = q[words - 1u];
    S.stack.p = M.base;
    for (uint32_t r = 0; r < rows; ++r, S.stack.p += M.stride) M.at(S.stack.p) = q[r];
    S.scale_spill -= 1u;
#pragma unroll
    for (int k = 0; k < kRegStack; ++k) stack_pop(S.stack, M);  // refills the registers
    S.cur = stack_pop(S.stack, M);
    return true;
}

// Distance at which a ray (origin o, 1/d inv) has left the root's box, a hair
// later; negative when the box lies behind.  Nothing is hit past it.
__device__ __forceinline__ float scene_exit(const NodeT* __restrict__ nodes, float3 o, float3 inv) {
#if RC_QNODE
    // scalar loads; opaque, so a loop over rays reads the root again instead of
    // keeping its planes in vector registers
    typedef const __attribute__((address_space(4))) float* scalar_floats;
    uint64_t root = reinterpret_cast<uint64_t>(nodes);
    asm volatile("" : "+s"(root));
    const scalar_floats f = reinterpret_cast<scalar_floats>(root);  // QNode: origin, scale
    auto far = [](float lo, float scale, float o, float inv) {
        return ((inv < 0.0f ? lo : fmaf(255.0f, scale, lo)) - o) * inv;
    };
    const float t = fminf(fminf(far(f[0], f[3], o.x, inv.x), far(f[1], f[4], o.y, inv.y)), far(f[2], f[5], o.z, inv.z));
    return t * 1.00001f;
#else
    return __builtin_inff();
#endif
}

// late: false when every ray's tmin is 0 (the renderer's).
template <bool DEC64>
__device__ __forceinline__ void trav_begin(Trav<DEC64>& S, const NodeT* __restrict__ nodes, const StackMem& M,
                                           float3 o, float3 d, float tmin, float tmax, const uint4* top, uint32_t ntop,
                                           bool late) {
    S.top = top;
    S.ntop = top ? ntop : 0u;
    S.o = o;
    S.d = d;
    S.tmin = late ? fmaxf(tmin, 0.0f) : 0.0f;
    S.late = late && __any(S.tmin > 0.0f);
    S.best = tmax;
    S.R = TraceResult{tmax, 0.0f, 0.0f, kNoHit, false, 1.0f};
    const float3 inv = safe_inv(d);
    const float T0 = cull_at<DEC64>(tmax), exit = scene_exit(nodes, o, inv);
    const float T = fminf(fmaxf(exit < T0 ? exit : T0, 1e-12f), 8e37f);  // below 2^126, the smallest scale's
    S.scale_spill = (253u << 23) - (__float_as_uint(T) & 0x7f800000u);  // 2^-k, 2^(k-1) <= T < 2^k
    S.inv = inv * trav_scale(S);
    trav_cull(S);
    S.cur = tmax < S.tmin ? kEmptyChild : 0u;  // root: interior record 0; an empty interval has no hit
    S.leaf = kEmptyChild;
    stack_reset(S.stack, M);
}

// a selected where the mask is 0, b where it is ~0 (one full-rate instruction).
__device__ __forceinline__ uint32_t pick(uint32_t a, uint32_t b, uint32_t mask) {
    return uint32_t(__builtin_amdgcn_bitop3_b32(int(a), int(b), int(mask), 0xD8));
}
__device__ __forceinline__ float clamp01(float x) { return __builtin_amdgcn_fmed3f(x, 0.0f, 1.0f); }

// Box tests of one wide node: per child its entry distance in [0, 1] (scaled),
// whether the ray enters it, and its stack entry.
struct Hits {
    float t[kWidth];
    bool h[kWidth];
    uint32_t e[kWidth];
};
template <bool DEC64>
__device__ __forceinline__ void node_hits(const Trav<DEC64>& S, const NodeT* __restrict__ nodes, uint32_t cur,
                                          Hits& H) {
    // Per axis the entry plane is the lower bound when the direction is
    // positive and the upper one when it is negative: the planes are picked by
    // the sign once per node, not by a minimum and a maximum per child.  The
    // exit is widened by a few ulps so rounding never culls a box the triangle
    // test could still hit.
    auto enter = [&](int k, float tnx, float tny, float tnz, float tfx, float tfy, float tfz) {
        H.t[k] = fmaxf(fmaxf(clamp01(tnx), tny), tnz);
        if (S.late) H.t[k] = fmaxf(H.t[k], S.tmin * trav_scale(S));
        H.h[k] = H.t[k] <= fminf(fminf(fminf(tfx, tfy), tfz) * 1.000002f, S.cull);
    };
    const uint32_t mx = uint32_t(int32_t(__float_as_uint(S.inv.x)) >> 31);
    const uint32_t my = uint32_t(int32_t(__float_as_uint(S.inv.y)) >> 31);
    const uint32_t mz = uint32_t(int32_t(__float_as_uint(S.inv.z)) >> 31);
#if RC_QNODE
    uint4 q0, q1, q2, q3;
    if (RC_LDS_TOP && cur < S.ntop) {  // the top of the tree, from LDS
        const uint4* t = S.top + 4 * cur;
        q0 = t[0];
        q1 = t[1];
        q2 = t[2];
        q3 = t[3];
    } else {
        // a 32-bit offset from the uniform base: the node array stays within 4 GiB
        // (fewer than 2^26 wide nodes)
        const uint4* p = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(nodes) + cur * 64u);
        q0 = p[0];
        q1 = p[1];
        q2 = p[2];
        q3 = p[3];
    }
    // bound = origin + q * scale; in scaled ray distance q * (scale * inv) + (origin - o) * inv
    const float ax = __uint_as_float(q0.w) * S.inv.x, bx = (__uint_as_float(q0.x) - S.o.x) * S.inv.x;
    const float ay = __uint_as_float(q1.x) * S.inv.y, by = (__uint_as_float(q0.y) - S.o.y) * S.inv.y;
    const float az = __uint_as_float(q1.y) * S.inv.z, bz = (__uint_as_float(q0.z) - S.o.z) * S.inv.z;
    const uint32_t nx = pick(q1.z, q2.y, mx), fx = pick(q2.y, q1.z, mx);
    const uint32_t ny = pick(q1.w, q2.z, my), fy = pick(q2.z, q1.w, my);
    const uint32_t nz = pick(q2.x, q2.w, mz), fz = pick(q2.w, q2.x, mz);
    auto plane = [](uint32_t w, int k, float a, float b) { return fmaf(float((w >> (8 * k)) & 0xFFu), a, b); };
#pragma unroll
    for (int k = 0; k < kWidth; ++k)
        enter(k, plane(nx, k, ax, bx), plane(ny, k, ay, by), plane(nz, k, az, bz), plane(fx, k, ax, bx),
              plane(fy, k, ay, by), plane(fz, k, az, bz));
    H.e[0] = q3.x;
    H.e[1] = q3.y;
    H.e[2] = q3.z;
    H.e[3] = q3.w;
#else
    const uint4* p = reinterpret_cast<const uint4*>(nodes + cur);
    auto plane = [](uint32_t w, float inv, float o) { return (__uint_as_float(w) - o) * inv; };
#pragma unroll
    for (int k = 0; k < kWidth; ++k) {
        const uint4 a = p[2 * k], b = p[2 * k + 1];  // lo.xyz hi.x, hi.yz link count
        const uint32_t nx = pick(a.x, a.w, mx), fx = pick(a.w, a.x, mx);
        const uint32_t ny = pick(a.y, b.x, my), fy = pick(b.x, a.y, my);
        const uint32_t nz = pick(a.z, b.y, mz), fz = pick(b.y, a.z, mz);
        enter(k, plane(nx, S.inv.x, S.o.x), plane(ny, S.inv.y, S.o.y), plane(nz, S.inv.z, S.o.z),
              plane(fx, S.inv.x, S.o.x), plane(fy, S.inv.y, S.o.y), plane(fz, S.inv.z, S.o.z));
        H.h[k] = H.h[k] && b.w != kEmptyChild;
        H.e[k] = b.w != 0 ? (kLeafTag | (b.w << 26) | b.z) : b.z;
    }
#endif
}

// The sort key of a child not entered, above every entry distance that is.
constexpr float kNotEntered = 4.0f;
// A packet's distance of an entered child: its first lane's, or 1 (past
// everything) where that lane's own ray enters later, not at all or has no
// distance, so that the child still sorts before those no lane enters.
__host__ __device__ inline float packet_entry(float t) { return fminf(t, 1.0f); }

// The children of a visited node in H: the nearest (ANY without RC_ANY_SORT:
// the first) becomes S.cur, the others go on the stack farthest first; with
// none S.cur is popped.  False when the stack would outgrow its rows (SPILL:
// and they cannot be spilled).
template <bool SORT, bool SPILL, bool DEC64>
__device__ __forceinline__ bool take_children(Trav<DEC64>& S, Hits& H, const StackMem& M) {
    const bool* h = H.h;
    uint32_t e0 = H.e[0], e1 = H.e[1], e2 = H.e[2], e3 = H.e[3];
    const bool a01 = h[0] || h[1], a23 = h[2] || h[3], b01 = h[0] && h[1], b23 = h[2] && h[3];
    const bool two = b01 || b23 || (a01 && a23);
    const bool three = (b01 && a23) || (b23 && a01), four = b01 && b23;
    if (SORT) {
        double k0 = __hiloint2double(__float_as_int(h[0] ? H.t[0] : kNotEntered), int(e0));
        double k1 = __hiloint2double(__float_as_int(h[1] ? H.t[1] : kNotEntered), int(e1));
        double k2 = __hiloint2double(__float_as_int(h[2] ? H.t[2] : kNotEntered), int(e2));
        double k3 = __hiloint2double(__float_as_int(h[3] ? H.t[3] : kNotEntered), int(e3));
        order2(k0, k1);
        order2(k2, k3);
        order2(k0, k2);
        order2(k1, k3);
        order2(k1, k2);
        e0 = uint32_t(__double2loint(k0));
        e1 = uint32_t(__double2loint(k1));
        e2 = uint32_t(__double2loint(k2));
        e3 = uint32_t(__double2loint(k3));
    }
    if (two && S.stack.p + 3 * M.stride >= M.end) {  // rare: count the entries
        const int m = four ? 3 : three ? 2 : 1;
        if (S.stack.p + m * M.stride >= M.end && !(SPILL && stack_spill(S, M))) return false;
    }
    if (SORT) {
        if (two) {
            if (four) stack_push(S.stack, M, e3);
            if (three) stack_push(S.stack, M, e2);
            stack_push(S.stack, M, e1);
        }
        S.cur = e0;
    } else {
        if (two) {
            if (h[3] && (a01 || h[2])) stack_push(S.stack, M, e3);
            if (h[2] && a01) stack_push(S.stack, M, e2);
            if (b01) stack_push(S.stack, M, e1);
        }
        S.cur = h[0] ? e0 : h[1] ? e1 : h[2] ? e2 : e3;
    }
    if (!(a01 || a23)) S.cur = stack_pop(S.stack, M);
    return true;
}

// One step of the ordered, culled traversal over 4-wide nodes with leaves
// postponed ("if-if"): a node visit pushes the children it enters, leaves
// included, far-to-near and keeps the nearest; each step does at most one node
// visit and one leaf, so the lanes of a wave stay in step instead of waiting
// while one lane tests up to four leaves.  True when the traversal has ended
// (S.R holds the result, S.R.overflow when the stack would have outgrown its
// rows).  ANY: stop at the first triangle (not nonShadowing) with t in [tmin,
// tmax].
//
// Bound by VALU issue: before, a visit's 132 instructions took 448 of a SIMD's
// cycles and the pushes, the pop and the leaf bookkeeping of a step another
// 270; the kernels kept the VALU busy all the time.
template <bool ANY, bool COUNT, bool DEC64>
__device__ __forceinline__ bool trav_step(Trav<DEC64>& S, const NodeT* __restrict__ nodes,
                                          const TriRec* __restrict__ tris, const StackMem& M, uint32_t& n_rec,
                                          uint32_t& n_tri) {
    if (is_node(S.cur)) {
        if (COUNT) n_rec += kWidth;
        Hits H;
        node_hits<DEC64>(S, nodes, S.cur, H);
        if (!take_children<!ANY || RC_ANY_SORT, true>(S, H, M)) {
            S.R.overflow = true;
            return true;
        }
    }
#if RC_LEAF_POSTPONE
    constexpr uint32_t kHold = ANY ? RC_LEAF_POSTPONE_ANY : RC_LEAF_POSTPONE;
    // Leaf postponing: a lane that reaches a leaf sets it aside (one slot)
    // and goes on with its stack; the wave tests the leaves set aside when at
    // least RC_LEAF_POSTPONE / 64 of its lanes hold one, or when no lane has a
    // node left to visit.  A lane whose next entry is a second leaf waits.
    if (is_leaf(S.cur) && S.leaf == kEmptyChild) {
        S.leaf = S.cur;
        S.cur = stack_pop(S.stack, M);
    }
    {
        const bool held = S.leaf != kEmptyChild;
        const uint64_t lanes = __ballot(1), visit = __ballot(is_node(S.cur)), holding = __ballot(held);
        const bool run = visit == 0 || uint32_t(__popcll(holding)) * 64u >= uint32_t(__popcll(lanes)) * kHold;
        if (held && run) {
            const uint32_t first = S.leaf & ((1u << 26) - 1u), count = (S.leaf >> 26) & 31u;
            const uint32_t id = S.R.id;
            if (test_leaf<ANY, COUNT, DEC64>(tris, first, count, S.o, S.d, S.tmin, S.best, S.R, n_tri)) return true;
            if (!ANY && S.R.id != id) trav_cull(S);
            S.leaf = kEmptyChild;
        }
    }
    return (S.cur & S.leaf) == kEmptyChild && !stack_reload(S, M);
#else
    if (is_leaf(S.cur)) {
        const uint32_t first = S.cur & ((1u << 26) - 1u), count = (S.cur >> 26) & 31u;
        const uint32_t id = S.R.id;
        if (test_leaf<ANY, COUNT, DEC64>(tris, first, count, S.o, S.d, S.tmin, S.best, S.R, n_tri)) return true;
        if (!ANY && S.R.id != id) trav_cull(S);
        S.cur = stack_pop(S.stack, M);
    }
    return S.cur == kEmptyChild && !stack_reload(S, M);
#endif  // RC_LEAF_POSTPONE
}

// The traversal without postponed leaves (RC_TRAV_IFIF 0 with the 128-byte
// node records): the leaf children a node visit enters are tested at once, the
// nearest interior child is visited next and the others are pushed.
#ifndef RC_SLAB_SELECT
#define RC_SLAB_SELECT 1  // 0: leaf children not entered are skipped by a branch per child
#endif
template <bool ANY, bool COUNT, bool DEC64>
__device__ __forceinline__ TraceResult traverse_inline(const NodeT* __restrict__ nodes, const TriRec* __restrict__ tris,
                                                       float3 o, float3 d, float tmin, float tmax, const StackMem& M,
                                                       uint32_t& n_rec, uint32_t& n_tri) {
    Trav<DEC64> S;
    trav_begin(S, nodes, M, o, d, tmin, tmax, nullptr, 0, true);
    while (S.cur != kEmptyChild) {
        if (COUNT) n_rec += kWidth;
        Hits H;
        node_hits<DEC64>(S, nodes, S.cur, H);
        for (int k = 0; k < kWidth; ++k) {
            if (is_node(H.e[k])) continue;
            if (!RC_SLAB_SELECT && !H.h[k]) continue;
            const uint32_t first = H.e[k] & ((1u << 26) - 1u), count = H.h[k] ? (H.e[k] >> 26) & 31u : 0u;
            const uint32_t id = S.R.id;
            if (test_leaf<ANY, COUNT, DEC64>(tris, first, count, o, d, S.tmin, S.best, S.R, n_tri)) return S.R;
            if (!ANY && S.R.id != id) trav_cull(S);
            H.h[k] = false;
        }
        if (!take_children<true, false>(S, H, M)) {
            S.R.overflow = true;
            return S.R;
        }
    }
    return S.R;
}

// A traversal parked mid-way (the extension kernel's step budget ran out):
// 32 words per ray (36 with more stack registers), written and read as 16-byte
// vectors.  Words: 0 the
// queue entry, 1 the current entry, 2 the stack's rows in use, 3 the best hit's
// id, 4..6 its t, u, v, 7 the spilled stack, 8..9 the best distance of the FP64 decision,
// 10.. the register stack (top first), then the memory rows in their order
// (only those in use are meaningful); the last two words the best hit's w and the
// leaf set aside.
constexpr int kParkWords = RC_REG_STACK > 1 ? 36 : 32;
constexpr int kParkW = kParkWords - 2;
static_assert(10 + kRegStack + kLdsStack <= kParkW, "a parked traversal does not fit its record");

// Word w of a parked record (compile-time w after unrolling).
template <bool DEC64>
__device__ __forceinline__ uint32_t park_word(const Trav<DEC64>& S, uint32_t entry, const StackMem& M, int w) {
    if (w == 0) return entry;
    if (w == 1) return S.cur;
    if (w == 2) return uint32_t(S.stack.p - M.base) / uint32_t(M.stride);
    if (w == 3) return S.R.id;
    if (w == 4) return __float_as_uint(S.R.t);
    if (w == 5) return __float_as_uint(S.R.u);
    if (w == 6) return __float_as_uint(S.R.v);
    if (w == 7) return S.scale_spill & kSpillMask;
    if (w == 8 || w == 9) {
        if constexpr (DEC64) {
            const unsigned long long b = __double_as_longlong(S.best);
            return w == 8 ? uint32_t(b) : uint32_t(b >> 32);
        } else {
            return 0u;
        }
    }
    if (w == kParkW) return __float_as_uint(S.R.w);
    if (w == kParkW + 1) return S.leaf;
    if (w < 10 + kRegStack) return S.stack.reg[w - 10];
    const int j = w - 10 - kRegStack;  // memory row
    const int p = M.base + j * M.stride;
    return j < kLdsStack && p < S.stack.p ? M.at(p) : 0u;
}

template <bool DEC64>
__device__ __forceinline__ void trav_park(const Trav<DEC64>& S, uint32_t entry, const StackMem& M,
                                          uint32_t* __restrict__ rec) {
    uint4* r = reinterpret_cast<uint4*>(rec);
#pragma unroll
    for (int q = 0; q < kParkWords / 4; ++q)
        st_stream(r + q, make_uint4(park_word(S, entry, M, 4 * q), park_word(S, entry, M, 4 * q + 1),
                                    park_word(S, entry, M, 4 * q + 2), park_word(S, entry, M, 4 * q + 3)));
}

template <bool DEC64>
__device__ __forceinline__ void unpark_word(Trav<DEC64>& S, const StackMem& M, int w, uint32_t v, uint32_t& best_lo) {
    if (w == 1) S.cur = v;
    else if (w == 2) S.stack.p = M.base + int(v) * M.stride;
    else if (w == 3) S.R.id = v;
    else if (w == 4) S.R.t = __uint_as_float(v);
    else if (w == 5) S.R.u = __uint_as_float(v);
    else if (w == 6) S.R.v = __uint_as_float(v);
    else if (w == 7) S.scale_spill |= v;
    else if (w == kParkW) S.R.w = __uint_as_float(v);
    else if (w == kParkW + 1) S.leaf = v;
    else if (w == 8) best_lo = v;
    else if (w == 9) {
        if constexpr (DEC64) S.best = __longlong_as_double((long long)(uint64_t(best_lo) | (uint64_t(v) << 32)));
    } else if (w >= 10 && w < 10 + kRegStack) {
        S.stack.reg[w - 10] = v;
    } else if (w >= 10 + kRegStack) {
        const int j = w - 10 - kRegStack;
        const int p = M.base + j * M.stride;
        if (j < kLdsStack && p < S.stack.p) M.at(p) = v;
    }
}

// Resumes a parked traversal: S must have been begun on the same ray
// (trav_begin), which restores the ray's own fields; this restores the rest
// and the lane's stack rows (word 0, the queue entry, is the caller's).
template <bool DEC64>
__device__ __forceinline__ void trav_unpark(Trav<DEC64>& S, const uint32_t* __restrict__ rec, const StackMem& M) {
    const uint4* r = reinterpret_cast<const uint4*>(rec);
    uint32_t best_lo = 0;
#pragma unroll
    for (int q = 0; q < kParkWords / 4; ++q) {
        const uint4 v = ld_stream(r + q);
        unpark_word(S, M, 4 * q, v.x, best_lo);
        unpark_word(S, M, 4 * q + 1, v.y, best_lo);
        unpark_word(S, M, 4 * q + 2, v.z, best_lo);
        unpark_word(S, M, 4 * q + 3, v.w, best_lo);
    }
    if (S.R.id != kNoHit) trav_cull(S);
}

template <bool ANY, bool COUNT, bool DEC64>
__device__ __forceinline__ TraceResult traverse_ifif(const NodeT* __restrict__ nodes, const TriRec* __restrict__ tris,
                                                     float3 o, float3 d, float tmin, float tmax, const StackMem& M,
                                                     uint32_t& n_rec, uint32_t& n_tri, const uint4* top, uint32_t ntop,
                                                     bool late) {
    Trav<DEC64> S;
    trav_begin(S, nodes, M, o, d, tmin, tmax, top, ntop, late);
    while (!trav_step<ANY, COUNT, DEC64>(S, nodes, tris, M, n_rec, n_tri)) {
    }
    return S.R;
}

// Closest hit (ANY = false) or any hit of one ray, with the lane's stack
// memory M.  late: whether rays may have a tmin > 0.
template <bool ANY, bool COUNT, bool DEC64>
__device__ __forceinline__ TraceResult traverse(const NodeT* __restrict__ nodes, const TriRec* __restrict__ tris,
                                                float3 o, float3 d, float tmin, float tmax, const StackMem& M,
                                                uint32_t& n_rec, uint32_t& n_tri, const uint4* top, uint32_t ntop,
                                                bool late) {
    if (!RC_QNODE && !RC_TRAV_IFIF)
        return traverse_inline<ANY, COUNT, DEC64>(nodes, tris, o, d, tmin, tmax, M, n_rec, n_tri);
    return traverse_ifif<ANY, COUNT, DEC64>(nodes, tris, o, d, tmin, tmax, M, n_rec, n_tri, top, ntop, late);
}

#if RC_QNODE
// Closest hit of a wave of nearly coherent rays traversed as one packet (the
// camera bounce, whose waves each hold one pixel's samples).  The wave
// follows one stack and visits a child when any of its lanes enters it, so
// every lane visits a superset of the nodes its own traversal would; the
// exact-tie rule of test_leaf makes each answer independent of the order and
// of the extra visits, so the hits are those of traverse().  Children are
// taken nearest first by the first active lane's entry distances.  The
// stack entries are wave-uniform; each lane keeps its own copy in its LDS
// rows, and when they are full every lane of the wave reports an overflow.  Every active lane of the wave
// calls this (the loop and its exit are uniform).
template <bool COUNT>
__device__ __forceinline__ TraceResult traverse_packet(const QNode* __restrict__ nodes,
                                                       const TriRec* __restrict__ tris, float3 o, float3 d,
                                                       float tmin, float tmax, const StackMem& M, uint32_t& n_rec,
                                                       uint32_t& n_tri) {
    Trav<false> S;
    trav_begin(S, nodes, M, o, d, tmin, tmax, nullptr, 0, false);
    S.cur = 0;  // wave-uniform, as the stack
    for (;;) {
        if (is_node(S.cur)) {
            if (COUNT) n_rec += kWidth;
            Hits H;
            node_hits<false>(S, nodes, S.cur, H);
            // entered by any lane; the first active lane's distance and the
            // entry, all wave-uniform
#pragma unroll
            for (int k = 0; k < kWidth; ++k) {
                H.h[k] = __ballot(H.h[k]) != 0;
                H.t[k] = packet_entry(__uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(H.t[k]))));
                H.e[k] = __builtin_amdgcn_readfirstlane(H.e[k]);
            }
            if (!take_children<true, false>(S, H, M)) {
                S.R.overflow = true;
                return S.R;
            }
        } else {
            if (is_leaf(S.cur)) {
                // every active lane tests the leaf: a lane whose ray misses
                // the leaf's box finds no hit there it would not also find
                // through its own traversal
                const uint32_t id = S.R.id;
                test_leaf<false, COUNT, false>(tris, S.cur & 0x03FFFFFFu, (S.cur >> 26) & 0x1Fu, o, d, S.tmin, S.best,
                                               S.R, n_tri);
                if (S.R.id != id) trav_cull(S);
            }
            S.cur = stack_pop(S.stack, M);
        }
        S.cur = __builtin_amdgcn_readfirstlane(S.cur);
        if (S.cur == kEmptyChild) return S.R;
    }
}
#endif

}  // namespace rcd
