// Strand ray tracer on the GPU: the reference's Embree path tracer of flat
// linear curves (src/vkhr/ray_tracer.cc:76-169, ray_tracer/hair_style.cc:
// 18-44,50-110) as a ground-truth for the raymarcher's shadow and AO
// approximations.
//
// Acceleration structure: a linear BVH over the segments (Karras, "Maximizing
// Parallelism in the Construction of BVHs, Octrees, and k-d Trees", HPG
// 2012): 30-bit Morton codes of the segment centroids, sorted with rocPRIM's
// radix sort, a binary radix tree over (code, index) -- which bounds its depth
// by the 62 key bits -- and boxes that each node forms for itself from unions
// of 8, 64, 512, ... consecutive leaves.  The tree that is traversed is cut from it: nodes of up to eight
// children, one octree level each, in 64 bytes.
//
// Traversal: one ray per lane, a node's eight boxes per step, children in
// the octant order of the ray's direction.  What bounds it is the work per
// step: a gather costs a cycle of the L1's tag lookup per lane that reads
// another line, and the eight box tests ~300 instructions, both about 1.5 us
// per step of the three waves a SIMD holds at 200k rays.  So a node is four
// 16-byte loads (a binary node was four too, for two children), its
// children's units follow from one base, and leaves queue until 64 fill the
// wave (tested where they are found, they run at a few lanes per wave).
// Measured at 136k strands (1.6 M segments), 1080p, shaded: binary nodes
// 1.29 ms, eight children with child links (128 bytes) 0.96, queued leaves
// 0.78, 64-byte units 0.71.  Four lanes per ray with refill: 1.0 ms.
//
// Primitive: the ray-facing ribbon of a segment whose radius varies linearly
// (Embree's flat linear curve): the axis is projected on the plane through
// the ray origin perpendicular to the ray; u minimises the projected
// distance to the ray, and the hit needs that distance within the radius at
// u and the axis depth t in [tnear, tfar].  Compiled with -ffp-contract=off:
// the float32 expressions are evaluated in the order the CPU restatement
// evaluates them, so hits agree bit for bit with it.
#include <rocprim/device/device_radix_sort.hpp>

#include <cfloat>
#include <cmath>
#include <cstring>
#include <vector>

#include "common.hpp"

namespace vkhr {
namespace {

constexpr uint32_t kLeaf = 0x80000000u;
constexpr uint32_t kNone = 0xffffffffu;

// One 64-byte unit of the traversed tree: a wide node or a leaf.  A wide node
// has up to eight children, whose boxes are 8-bit offsets from its origin in
// units of a power of two, rounded outwards.  Slot s of an interior node is
// the Morton octant s of its cell, so the slots ordered by s ^ (octant of
// the ray's direction signs) are front to back.  The children are the
// consecutive units from base, in slot order.
struct __align__(64) WideNode {
    uint32_t origin[3];      // floats' upper 24 bits (towards -inf), then a byte each:
                             // the unit's biased exponent, the mask of inner and of leaf children
    uint32_t base;
    uint32_t planes[3][4];   // per axis: lower planes of slots 0-3, 4-7, upper planes of slots 0-3, 4-7
};
struct __align__(64) TraceLeaf {
    float4 a, b;             // p0|r0, p1|r1
    uint32_t seg;            // segment index (index pair)
    uint32_t pad[7];
};
static_assert(sizeof(WideNode) == 64 && sizeof(TraceLeaf) == 64, "one unit each");

struct TraceBvh {
    const WideNode* units;     // 0 is the root (of one segment: its leaf)
    uint32_t n;                // leaves
};

struct Hit {
    float t, u;
    uint32_t seg;
};

__device__ __forceinline__ float dot3(float3 a, float3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

__device__ __forceinline__ bool flat_curve(float3 o, float3 d, float dd, float4 a, float4 b, float tnear,
                                           float tfar, float* t_out, float* u_out) {
    const float3 q0 = make_float3(a.x - o.x, a.y - o.y, a.z - o.z);
    const float3 q1 = make_float3(b.x - o.x, b.y - o.y, b.z - o.z);
    const float z0 = dot3(q0, d) / dd, z1 = dot3(q1, d) / dd;
    const float3 x0 = make_float3(q0.x - z0 * d.x, q0.y - z0 * d.y, q0.z - z0 * d.z);
    const float3 v = make_float3((q1.x - z1 * d.x) - x0.x, (q1.y - z1 * d.y) - x0.y, (q1.z - z1 * d.z) - x0.z);
    const float vv = dot3(v, v);
    float u = 0.0f;
    if (vv > 0.0f) {
        u = -dot3(x0, v) / vv;
        u = u < 0.0f ? 0.0f : (u > 1.0f ? 1.0f : u);
    }
    const float3 p = make_float3(x0.x + u * v.x, x0.y + u * v.y, x0.z + u * v.z);
    const float z = z0 + u * (z1 - z0);
    const float r = a.w + u * (b.w - a.w);
    if (!(dot3(p, p) <= r * r)) return false;
    if (!(z >= tnear && z <= tfar)) return false;
    *t_out = z;
    *u_out = u;
    return true;
}

// Directions with a zero component get a tiny one of the same sign, so the
// slab reciprocals stay finite (boxes are padded, so this never loses a hit).
__device__ __forceinline__ float3 safe_inverse(float3 d) {
    auto f = [](float x) { return 1.0f / (fabsf(x) < 1e-30f ? copysignf(1e-30f, x) : x); };
    return make_float3(f(d.x), f(d.y), f(d.z));
}

// One wave's LDS of a trace.  Pending siblings of a lane: entry k holds a
// node's base and a word: the mask of its children (bits 8-15), the inner
// ones still to be visited in front-to-back order (bits 0-7) and a lower
// bound of their entry distances (the float's upper half).  The first
// kTraceStack entries of a lane are here; a path holds at most one entry per
// wide level, and a tree has at most kWideLevels.
// Leaves whose box is hit wait in a ring until 64 of them fill the wave,
// then each lane tests one, of whichever lane's ray; best holds every ray's
// closest hit so far as (ordered t, segment), so equal distances go to the
// lowest segment.
constexpr uint32_t kTraceStack = 8, kWideLevels = 22, kLeafRing = 2 * kWave;
struct TraceLds {
    unsigned long long best[kWave];
    uint2 pending[kTraceStack][kWave];
    uint32_t ring_leaf[kLeafRing];
    uint32_t ring_lane[kLeafRing];
    float t[kWave], u[kWave];
};

// Floats in an order of unsigned integers (-0 as 0).
__device__ __forceinline__ uint32_t ordered(float t) {
    const uint32_t b = __float_as_uint(t + 0.0f);
    return b & 0x80000000u ? ~b : b | 0x80000000u;
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float byte_of(uint32_t w, int k) { return float((w >> (8 * k)) & 0xffu); }

// An 8-bit mask with bit s moved to bit s ^ oct.
__device__ __forceinline__ uint32_t xor_slots(uint32_t m, uint32_t oct) {
    m = oct & 1u ? ((m & 0xaau) >> 1) | ((m & 0x55u) << 1) : m;
    m = oct & 2u ? ((m & 0xccu) >> 2) | ((m & 0x33u) << 2) : m;
    return oct & 4u ? (m >> 4) | ((m & 0x0fu) << 4) : m;
}

// Closest (kAny = false) or any (kAny = true) hit of every active lane's ray
// in [tnear, tfar]; closest ties go to the lowest segment index.  Every lane
// of the wave calls it.
template <bool kAny>
__device__ Hit trace(const TraceBvh& b, TraceLds& lds, bool active, float3 o, float3 d, float tnear, float tfar,
                     uint32_t skip = kNone) {
    const uint32_t lane = threadIdx.x % kWave;
    Hit best{tfar, 0.0f, kNone};
    if (b.n == 0u) return best;
    lds.best[lane] = ~0ull;
    const float3 inv = safe_inverse(d);
    const bool fx = inv.x < 0.0f, fy = inv.y < 0.0f, fz = inv.z < 0.0f;
    const uint32_t oct = (fx ? 4u : 0u) | (fy ? 2u : 0u) | (fz ? 1u : 0u);
    uint2 spill[kWideLevels - kTraceStack];
    uint32_t sp = 0u, cur = active && b.n > 1u ? 0u : kNone;
    // the leaves to queue: unit base, and its children's and its hit leaves' masks
    uint32_t leaves = active && b.n == 1u ? 1u : 0u, base = 0u, kids = leaves;
    uint32_t ring = 0u, queued = 0u;  // wave-uniform
    // Tests the oldest queued leaves, one per lane.
    auto flush = [&] {
        wave_lds_sync();
        const uint32_t count = queued < uint32_t(kWave) ? queued : uint32_t(kWave), at = (ring + lane) % kLeafRing;
        const bool has = lane < count;
        const uint32_t leaf = has ? lds.ring_leaf[at] : 0u;
        const int src = has ? int(lds.ring_lane[at]) : int(lane);
        const float3 ro = make_float3(__shfl(o.x, src, kWave), __shfl(o.y, src, kWave), __shfl(o.z, src, kWave));
        const float3 rd = make_float3(__shfl(d.x, src, kWave), __shfl(d.y, src, kWave), __shfl(d.z, src, kWave));
        const float near = __shfl(tnear, src, kWave), far = __shfl(best.t, src, kWave);
        const uint32_t not_this = uint32_t(__shfl(int(skip), src, kWave));
        float t = 0.0f, u = 0.0f;
        unsigned long long key = ~0ull;
        if (has) {
            const TraceLeaf& l = reinterpret_cast<const TraceLeaf*>(b.units)[leaf];
            const uint32_t seg = l.seg;
            if (flat_curve(ro, rd, dot3(rd, rd), l.a, l.b, near, far, &t, &u) && seg != not_this) {
                key = ((unsigned long long)ordered(t) << 32) | seg;
                __hip_atomic_fetch_min(&lds.best[src], key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
        wave_lds_sync();
        if (key != ~0ull && lds.best[src] == key) {  // one lane at most: segments differ
            lds.t[src] = t;
            lds.u[src] = u;
        }
        wave_lds_sync();
        const unsigned long long mine = lds.best[lane];
        if (mine != ~0ull) {
            best.seg = uint32_t(mine);
            best.t = lds.t[lane];
            if (kAny) {
                cur = kNone;
                leaves = 0u;
            }
        }
        ring = (ring + count) % kLeafRing;
        queued -= count;
    };
    // Each node is opened at most once: the cap only guards against a malformed tree.
    for (uint32_t visits = b.n + 1u; visits != 0u; --visits) {
        if (cur != kNone) {
            const uint4* nd = reinterpret_cast<const uint4*>(b.units + cur);
            const uint4 head = nd[0], px = nd[1], py = nd[2], pz = nd[3];
            base = head.w;
            const uint32_t inner = head.y & 0xffu, leaf_slots = head.z & 0xffu;
            kids = inner | leaf_slots;
            // plane q of axis c is at t = (origin + q * unit - o) * inv = q * step + from
            const float unit = __uint_as_float((head.x & 0xffu) << 23);
            const float3 step = make_float3(unit * inv.x, unit * inv.y, unit * inv.z);
            const float3 from = make_float3((__uint_as_float(head.x & 0xffffff00u) - o.x) * inv.x,
                                            (__uint_as_float(head.y & 0xffffff00u) - o.y) * inv.y,
                                            (__uint_as_float(head.z & 0xffffff00u) - o.z) * inv.z);
            // the near and far planes by the sign of the direction
            const uint32_t nx[2] = {fx ? px.z : px.x, fx ? px.w : px.y}, xx[2] = {fx ? px.x : px.z, fx ? px.y : px.w};
            const uint32_t ny[2] = {fy ? py.z : py.x, fy ? py.w : py.y}, xy[2] = {fy ? py.x : py.z, fy ? py.y : py.w};
            const uint32_t nz[2] = {fz ? pz.z : pz.x, fz ? pz.w : pz.y}, xz[2] = {fz ? pz.x : pz.z, fz ? pz.y : pz.w};
            uint32_t hits = 0u;
            float enter[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const int h = s >> 2, k = s & 3;
                const float t0 = fmaxf(fmaxf(__builtin_fmaf(byte_of(nx[h], k), step.x, from.x),
                                             __builtin_fmaf(byte_of(ny[h], k), step.y, from.y)),
                                       fmaxf(__builtin_fmaf(byte_of(nz[h], k), step.z, from.z), tnear));
                const float t1 = fminf(fminf(__builtin_fmaf(byte_of(xx[h], k), step.x, from.x),
                                             __builtin_fmaf(byte_of(xy[h], k), step.y, from.y)),
                                       fminf(__builtin_fmaf(byte_of(xz[h], k), step.z, from.z), best.t));
                enter[s] = t0;
                hits |= t0 <= t1 ? 1u << s : 0u;
            }
            leaves = hits & leaf_slots;
            hits &= inner;
            uint32_t m = xor_slots(hits, oct);
            if (m != 0u) {
                const uint32_t first = uint32_t(__builtin_ctz(m)) ^ oct;
                cur = base + uint32_t(__builtin_popcount(kids & ((1u << first) - 1u)));
                m &= m - 1u;
                if (m != 0u) {
                    float bound = INFINITY;
                    hits &= ~(1u << first);
#pragma unroll
                    for (int s = 0; s < 8; ++s) bound = fminf(bound, (hits >> s) & 1u ? enter[s] : INFINITY);
                    // truncated towards -inf: bits below the mask, or -inf for a negative distance
                    const uint32_t word = (bound >= 0.0f ? __float_as_uint(bound) & 0xffff0000u : 0xff800000u) | (kids << 8) | m;
                    if (sp < kTraceStack)
                        lds.pending[sp][lane] = make_uint2(base, word);
                    else
                        spill[sp - kTraceStack] = make_uint2(base, word);
                    ++sp;
                }
            } else {
                // the deepest pending node that the closest hit so far leaves in reach
                cur = kNone;
                while (sp != 0u) {
                    const uint2 e = sp <= kTraceStack ? lds.pending[sp - 1u][lane] : spill[sp - 1u - kTraceStack];
                    if (!(__uint_as_float(e.y & 0xffff0000u) <= best.t)) {
                        --sp;
                        continue;
                    }
                    const uint32_t slot = (uint32_t(__builtin_ctz(e.y)) ^ oct) & 7u;
                    cur = e.x + uint32_t(__builtin_popcount((e.y >> 8) & ((1u << slot) - 1u)));
                    const uint32_t word = e.y & (e.y - 1u);
                    if ((word & 0xffu) == 0u)
                        --sp;
                    else if (sp <= kTraceStack)
                        lds.pending[sp - 1u][lane].y = word;
                    else
                        spill[sp - 1u - kTraceStack].y = word;
                    break;
                }
            }
        }
        for (unsigned long long who = __ballot(leaves != 0u); who != 0ull; who = __ballot(leaves != 0u)) {
            if (leaves != 0u) {
                const uint32_t at = (ring + queued + uint32_t(__popcll(who & ((1ull << lane) - 1ull)))) % kLeafRing;
                lds.ring_leaf[at] = base + uint32_t(__builtin_popcount(kids & ((leaves & (0u - leaves)) - 1u)));
                lds.ring_lane[at] = lane;
                leaves &= leaves - 1u;
            }
            queued += uint32_t(__popcll(who));
            if (queued >= uint32_t(kWave)) flush();
        }
        if (__ballot(cur != kNone) == 0ull) break;
    }
    if (queued != 0u) flush();
    if (best.seg != kNone) best.u = lds.u[lane];
    wave_lds_sync();  // the wave's next trace clears best
    return best;
}

// ------------------------------------------------------------------ build

struct BuildArgs {
    const float* xyz;
    const float* radius;
    const uint32_t* indices;
    uint32_t n_vertices;
    uint32_t n;                 // segments
    float4* box_lo;             // per segment (input order), w unused
    float4* box_hi;
    float* bounds_partial;      // 6 per block: centroid min xyz, max xyz
    float* bounds;              // 6: centroid min, max; then scene min, max (12)
    float* host_bounds;         // the first 6 for the host (nullable)
    uint32_t* keys;
    uint32_t* values;
};

__global__ void __launch_bounds__(256) segment_boxes_kernel(BuildArgs a) {
    __shared__ float red[6][256];
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    float cmin[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, cmax[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    if (k < a.n) {
        const uint32_t ia = a.indices[2ull * k], ib = a.indices[2ull * k + 1];
        float4 lo = make_float4(FLT_MAX, FLT_MAX, FLT_MAX, 0.0f), hi = make_float4(-FLT_MAX, -FLT_MAX, -FLT_MAX, 0.0f);
        if (ia < a.n_vertices && ib < a.n_vertices) {
            const float3 p = load_xyz(a.xyz, ia), q = load_xyz(a.xyz, ib);
            const float r = fmaxf(a.radius[ia], a.radius[ib]);
            lo = make_float4(fminf(p.x, q.x) - r, fminf(p.y, q.y) - r, fminf(p.z, q.z) - r, 0.0f);
            hi = make_float4(fmaxf(p.x, q.x) + r, fmaxf(p.y, q.y) + r, fmaxf(p.z, q.z) + r, 0.0f);
            const float c[3] = {0.5f * (lo.x + hi.x), 0.5f * (lo.y + hi.y), 0.5f * (lo.z + hi.z)};
            for (int i = 0; i < 3; ++i) cmin[i] = cmax[i] = c[i];
        }
        a.box_lo[k] = lo;
        a.box_hi[k] = hi;
    }
    for (int i = 0; i < 3; ++i) {
        red[i][threadIdx.x] = cmin[i];
        red[3 + i][threadIdx.x] = cmax[i];
    }
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int i = 0; i < 3; ++i) {
                red[i][threadIdx.x] = fminf(red[i][threadIdx.x], red[i][threadIdx.x + s]);
                red[3 + i][threadIdx.x] = fmaxf(red[3 + i][threadIdx.x], red[3 + i][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) a.bounds_partial[6ull * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

__global__ void __launch_bounds__(256) bounds_final_kernel(BuildArgs a, uint32_t blocks) {
    __shared__ float red[6][256];
    float v[6] = {FLT_MAX, FLT_MAX, FLT_MAX, -FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (uint32_t i = threadIdx.x; i < blocks; i += blockDim.x)
        for (int c = 0; c < 6; ++c)
            v[c] = c < 3 ? fminf(v[c], a.bounds_partial[6ull * i + c]) : fmaxf(v[c], a.bounds_partial[6ull * i + c]);
    for (int c = 0; c < 6; ++c) red[c][threadIdx.x] = v[c];
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int c = 0; c < 6; ++c)
                red[c][threadIdx.x] = c < 3 ? fminf(red[c][threadIdx.x], red[c][threadIdx.x + s])
                                            : fmaxf(red[c][threadIdx.x], red[c][threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x < 6) {
        a.bounds[threadIdx.x] = red[threadIdx.x][0];
        if (a.host_bounds) a.host_bounds[threadIdx.x] = red[threadIdx.x][0];
    }
}

// What the boxes are widened by: far more than the float rounding of the
// slab test and of the curve test, so that the box of every hit contains it.
__device__ __forceinline__ float box_pad(const float* bounds) {
    float diag2 = 0.0f, mag = 0.0f;
    for (int c = 0; c < 3; ++c) {
        const float ext = bounds[3 + c] - bounds[c];
        diag2 += ext * ext;
        mag = fmaxf(mag, fmaxf(fabsf(bounds[c]), fabsf(bounds[3 + c])));
    }
    return 1e-4f * sqrtf(diag2) + 1e-6f * mag + 1e-30f;
}

// 10 bits of v spread to every third bit.
__device__ __forceinline__ uint32_t spread_bits(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

__global__ void __launch_bounds__(256) morton_kernel(BuildArgs a) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.n) return;
    const float4 lo = a.box_lo[k], hi = a.box_hi[k];
    uint32_t code = 0u;
    if (lo.x <= hi.x) {
        const float c[3] = {0.5f * (lo.x + hi.x), 0.5f * (lo.y + hi.y), 0.5f * (lo.z + hi.z)};
        uint32_t q[3];
        for (int i = 0; i < 3; ++i) {
            const float ext = a.bounds[3 + i] - a.bounds[i];
            float f = ext > 0.0f ? (c[i] - a.bounds[i]) / ext : 0.0f;
            f = fminf(fmaxf(f * 1024.0f, 0.0f), 1023.0f);
            q[i] = uint32_t(f);
        }
        code = (spread_bits(q[0]) << 2) | (spread_bits(q[1]) << 1) | spread_bits(q[2]);
    }
    a.keys[k] = code;
    a.values[k] = k;
}

struct Box {
    float4 lo, hi;
};

__device__ __forceinline__ Box empty_box() {
    return {make_float4(FLT_MAX, FLT_MAX, FLT_MAX, 0.0f), make_float4(-FLT_MAX, -FLT_MAX, -FLT_MAX, 0.0f)};
}

__device__ __forceinline__ Box join(const Box& a, const Box& b) {
    return {make_float4(fminf(a.lo.x, b.lo.x), fminf(a.lo.y, b.lo.y), fminf(a.lo.z, b.lo.z), 0.0f),
            make_float4(fmaxf(a.hi.x, b.hi.x), fmaxf(a.hi.y, b.hi.y), fmaxf(a.hi.z, b.hi.z), 0.0f)};
}

// The leaves' boxes in code order and above them the unions of 8, 64, 512,
// ... consecutive ones: a node of the tree covers consecutive leaves, so its
// box is the union of a few of these.  Level k holds count[k] boxes.
constexpr int kMaxLevels = 12, kPyramidBlock = 512;
struct Pyramid {
    Box* level[kMaxLevels];
    int count[kMaxLevels];
    int levels;
};

// The three levels above `in`, of which this block holds box i (empty past
// the end) in thread i % 512.  All threads of the block call it.
__device__ __forceinline__ void pyramid_levels(const Pyramid& p, int in, int i, Box b, Box* waves) {
    const int lane = threadIdx.x % kWave;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const Box c = {make_float4(__shfl_xor(b.lo.x, o, kWave), __shfl_xor(b.lo.y, o, kWave),
                                   __shfl_xor(b.lo.z, o, kWave), 0.0f),
                       make_float4(__shfl_xor(b.hi.x, o, kWave), __shfl_xor(b.hi.y, o, kWave),
                                   __shfl_xor(b.hi.z, o, kWave), 0.0f)};
        b = join(b, c);
        if (o == 4 && (lane & 7) == 0 && in + 1 < p.levels && i < p.count[in]) p.level[in + 1][i >> 3] = b;
    }
    if (lane == 0) {
        if (in + 2 < p.levels && i < p.count[in]) p.level[in + 2][i >> 6] = b;
        waves[threadIdx.x / kWave] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0 && in + 3 < p.levels && i < p.count[in]) {
        for (int w = 1; w < kPyramidBlock / kWave; ++w) b = join(b, waves[w]);
        p.level[in + 3][i >> 9] = b;
    }
}

// Leaves in code order: the padded boxes, the first three levels above them
// and the primitive records.
__global__ void __launch_bounds__(kPyramidBlock)
leaves_kernel(BuildArgs a, const uint32_t* __restrict__ order, Pyramid p, float4* prims, uint32_t* prim_seg,
              uint32_t* made) {
    __shared__ Box waves[kPyramidBlock / kWave];
    const uint32_t l = blockIdx.x * blockDim.x + threadIdx.x;
    Box box = empty_box();
    if (l == 0) *made = 0u;   // the wide nodes' count
    if (l < a.n) {
        const uint32_t k = order[l];
        const uint32_t ia = a.indices[2ull * k], ib = a.indices[2ull * k + 1];
        float4 pa = make_float4(0.0f, 0.0f, 0.0f, NAN), pb = make_float4(0.0f, 0.0f, 0.0f, NAN);  // never hit
        if (ia < a.n_vertices && ib < a.n_vertices) {
            const float3 p0 = load_xyz(a.xyz, ia), p1 = load_xyz(a.xyz, ib);
            pa = make_float4(p0.x, p0.y, p0.z, a.radius[ia]);
            pb = make_float4(p1.x, p1.y, p1.z, a.radius[ib]);
        }
        prims[2ull * l] = pa;
        prims[2ull * l + 1] = pb;
        prim_seg[l] = k;
        const float4 lo = a.box_lo[k], hi = a.box_hi[k];
        const float pad = box_pad(a.bounds);
        box.lo = make_float4(lo.x - pad, lo.y - pad, lo.z - pad, 0.0f);
        box.hi = make_float4(hi.x + pad, hi.y + pad, hi.z + pad, 0.0f);
        p.level[0][l] = box;
    }
    pyramid_levels(p, 0, int(l), box, waves);
}

__global__ void __launch_bounds__(kPyramidBlock) pyramid_kernel(Pyramid p, int in) {
    __shared__ Box waves[kPyramidBlock / kWave];
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    pyramid_levels(p, in, i, i < p.count[in] ? p.level[in][i] : empty_box(), waves);
}

// The box of leaves [first, last]: from each level the boxes up to a multiple
// of eight on either side, then on a level up.  The loads of a level are
// issued together; those outside the range repeat its first box.
__device__ __forceinline__ Box range_box(const Pyramid& p, int first, int last) {
    Box b = p.level[0][first];
    for (int level = 0; first <= last; ++level) {
        const Box* boxes = p.level[level];
        if (level + 1 == p.levels) {
            for (int i = first; i <= last; ++i) b = join(b, boxes[i]);
            break;
        }
        const int up = min((first + 7) & ~7, last + 1), down = max(((last + 1) & ~7) - 1, up - 1);
        Box side[14];
#pragma unroll
        for (int q = 0; q < 7; ++q) {
            side[q] = boxes[first + q < up ? first + q : first];
            side[7 + q] = boxes[last - q > down ? last - q : first];
        }
#pragma unroll
        for (int q = 0; q < 14; ++q) b = join(b, side[q]);
        first = up >> 3;
        last = ((down + 1) >> 3) - 1;
    }
    return b;
}

// Length of the common prefix of the (code, index) keys of leaves i and j;
// -1 outside [0, n).
__device__ __forceinline__ int prefix(const uint32_t* __restrict__ codes, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    const uint32_t a = codes[i], b = codes[j];
    if (a != b) return __clz(a ^ b);
    return 32 + __clz(uint32_t(i) ^ uint32_t(j));
}

// Internal node i of the binary radix tree over the sorted keys: its range
// [min(i, j), max(i, j)] and split, its children, their boxes and their
// parent links.  Every node forms its boxes for itself from the pyramid; a
// climb from the leaves with an arrival count per node passes them upwards
// through memory at every step (at 75k leaves: this kernel 14.8 us and the
// climb 50.6, with two fills 5; now 26.0, and 3.5 more for the pyramid).
__global__ void __launch_bounds__(256)
radix_tree_kernel(const uint32_t* __restrict__ codes, int n, Pyramid p, float4* nodes, uint32_t* parent,
                  int2* ranges) {
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n - 1) return;
    const int d = prefix(codes, n, i, i + 1) > prefix(codes, n, i, i - 1) ? 1 : -1;
    const int dmin = prefix(codes, n, i, i - d);
    int lmax = 2;
    while (prefix(codes, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
        if (prefix(codes, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = prefix(codes, n, i, j);
    int s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (prefix(codes, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    const int gamma = i + s * d + min(d, 0);
    const uint32_t left = min(i, j) == gamma ? (kLeaf | uint32_t(gamma)) : uint32_t(gamma);
    const uint32_t right = max(i, j) == gamma + 1 ? (kLeaf | uint32_t(gamma + 1)) : uint32_t(gamma + 1);
    const int first = min(i, j), last = max(i, j);
    ranges[i] = make_int2(first, last);
    Box b[2] = {range_box(p, first, gamma), range_box(p, gamma + 1, last)};
    b[0].lo.w = __uint_as_float(left);
    b[0].hi.w = __uint_as_float(right);
    nodes[4ull * i + 0] = b[0].lo;
    nodes[4ull * i + 1] = b[0].hi;
    nodes[4ull * i + 2] = b[1].lo;
    nodes[4ull * i + 3] = b[1].hi;
    parent[(left & kLeaf) ? uint32_t(n - 1) + (left & ~kLeaf) : left] = uint32_t(i);
    parent[(right & kLeaf) ? uint32_t(n - 1) + (right & ~kLeaf) : right] = uint32_t(i);
    if (i == 0) parent[0] = kNone;
}

// The wide nodes, cut from the binary tree.  A binary node splits at one
// bit plane of its key (30 code bits, then 32 index bits that break ties);
// the planes come in groups of three, one octree level each.  A binary node
// of more than eight leaves becomes a wide node when its parent splits in
// another group; its children are the first nodes below it that split in
// another group or hold at most eight leaves.  A node of at most eight
// leaves under a larger one becomes a wide node of its leaves.  Every node
// decides for itself, so one launch makes them all; the groups bound the
// wide levels (10 of the codes, 11 of the indices, and the leaves').
constexpr int kWideLeaves = 8;

__device__ __forceinline__ int plane_group(int delta) { return delta < 32 ? (delta - 2) / 3 : 10 + (delta - 32) / 3; }
__device__ __forceinline__ int plane_slot_bit(int delta) { return 2 - (delta < 32 ? delta - 2 : delta - 32) % 3; }

struct WideArgs {
    const uint32_t* codes;
    const float4* nodes;     // the binary tree, its parent links and leaf ranges
    const uint32_t* parent;
    const int2* ranges;
    int n;                   // leaves
    const float* bounds;     // the scene's: the children's boxes are widened by half its pad
    const float4* prims;     // p0|r0, p1|r1 and segment of the leaves
    const uint32_t* prim_seg;
    uint32_t* made;          // units so far, without the root
    uint32_t* place;         // of a binary node that becomes a wide one: its unit
    uint32_t* base;          // and its children's first
    uint32_t* sides;         // and the sides of its eight children (kNone: none)
    WideNode* units;
};

// Whether binary node i becomes a wide node.
__device__ __forceinline__ bool is_wide(const WideArgs& a, int i) {
    if (i >= a.n - 1) return false;
    if (i == 0) return true;
    const int2 r = a.ranges[i], q = a.ranges[a.parent[i]];
    return r.y - r.x < kWideLeaves
               ? q.y - q.x >= kWideLeaves
               : plane_group(prefix(a.codes, a.n, r.x, r.y)) != plane_group(prefix(a.codes, a.n, q.x, q.y));
}

// Side 2 i of binary node i is its left child, 2 i + 1 its right one: the
// child's node or leaf, and its two box rows.
__device__ __forceinline__ uint32_t side_child(const WideArgs& a, uint32_t side) {
    return __float_as_uint(a.nodes[4ull * (side >> 1) + (side & 1u)].w);
}
__device__ __forceinline__ const float4* side_box(const WideArgs& a, uint32_t side) { return a.nodes + 2ull * side; }

// The child of wide node w in a slot: down the binary nodes of its group by
// the slot's bits, or the slot's leaf.  Returns whether there is one, and
// the side of the binary node that holds it.  A leaf whose box is empty
// (malformed pairs, NaN: never hit) is none.
__device__ __forceinline__ bool wide_child(const WideArgs& a, uint32_t w, uint32_t slot, uint32_t* side) {
    const int2 r = a.ranges[w];
    const bool flat = r.y - r.x < kWideLeaves;
    if (flat && int(slot) > r.y - r.x) return false;
    const int group = flat ? 0 : plane_group(prefix(a.codes, a.n, r.x, r.y));
    uint32_t cur = w;
    while (!(cur & kLeaf)) {
        bool right;
        if (flat) {
            right = r.x + int(slot) > int(__float_as_uint(a.nodes[4ull * cur].w) & ~kLeaf);  // past the left child's last leaf
        } else {
            const int2 q = a.ranges[cur];
            const int delta = prefix(a.codes, a.n, q.x, q.y);
            if (cur != w && (q.y - q.x < kWideLeaves || plane_group(delta) != group)) break;
            right = (slot >> plane_slot_bit(delta)) & 1u;
        }
        *side = 2u * cur + (right ? 1u : 0u);
        cur = side_child(a, *side);
    }
    if (cur & kLeaf) {
        const float4 lo = side_box(a, *side)[0], hi = side_box(a, *side)[1];
        if (!(lo.x <= hi.x && lo.y <= hi.y && lo.z <= hi.z)) return false;
    }
    if (flat) return true;
    // several slots lead to a child that skips planes of the group: it takes its octant's
    const int first = cur & kLeaf ? int(cur & ~kLeaf) : a.ranges[cur].x;
    const uint32_t key = group < 10 ? a.codes[first] >> (27 - 3 * group)
                                    : (group < 20 ? uint32_t(first) >> (29 - 3 * (group - 10)) : uint32_t(first) << 1);
    return (key & 7u) == slot;
}

// The wide nodes of a workgroup's binary nodes, listed: their count.
// Workgroups of 256, so that 75k leaves still reach every compute unit.
constexpr int kWideBlock = 256;
__device__ __forceinline__ uint32_t list_wide(const WideArgs& a, uint32_t* list, uint32_t* count) {
    if (threadIdx.x == 0) *count = 0u;
    __syncthreads();
    const int i = int(blockIdx.x * blockDim.x + threadIdx.x);
    const bool wide = is_wide(a, i);
    const unsigned long long mask = __ballot(wide);
    const uint32_t lane = threadIdx.x % kWave;
    uint32_t at = 0u;
    if (lane == 0 && mask) at = atomicAdd(count, uint32_t(__popcll(mask)));
    at = uint32_t(__shfl(int(at), 0, kWave));
    if (wide) list[at + uint32_t(__popcll(mask & ((1ull << lane) - 1ull)))] = uint32_t(i);
    __syncthreads();
    return *count;
}

// Finds the children of every wide node, eight lanes per node and a slot
// each, and gives them consecutive units: one device-wide add per workgroup.
// The children are recorded: the way down to one is a chain of loads, which
// the offsets, the places and the units would each take again (33.3 us for
// this pass and 21.1 for the units at 75k leaves then, 22.0 and 10.3 now).
__global__ void __launch_bounds__(kWideBlock) wide_place_kernel(WideArgs a) {
    __shared__ uint32_t list[kWideBlock], count, children, first;
    if (threadIdx.x == 0) children = 0u;
    const uint32_t n = list_wide(a, list, &count);
    const uint32_t lane = threadIdx.x % kWave, slot = lane & 7u, shift = lane & 56u;
    // offsets within the workgroup, then the workgroup's range
    for (int pass = 0; pass < 2; ++pass) {
        for (uint32_t k = threadIdx.x & ~uint32_t(kWave - 1); k < 8u * n; k += kWideBlock) {  // wave-uniform
            const uint32_t at = (k + lane) >> 3;
            const bool live = at < n;
            const uint32_t w = live ? list[at] : 0u;
            if (pass == 0) {
                uint32_t side = kNone;
                const bool in = live && wide_child(a, w, slot, &side);
                const uint32_t mine = uint32_t(__ballot(in) >> shift) & 0xffu;
                if (live) a.sides[8ull * w + slot] = in ? side : kNone;
                if (live && slot == 0u) a.base[w] = atomicAdd(&children, uint32_t(__popc(mine)));
            } else {
                const uint32_t side = live ? a.sides[8ull * w + slot] : kNone;
                const uint32_t child = side != kNone ? side_child(a, side) : kLeaf;
                const uint32_t mine = uint32_t(__ballot(side != kNone) >> shift) & 0xffu;
                const uint32_t base = live ? a.base[w] + first : 0u;
                if (!(child & kLeaf)) a.place[child] = base + uint32_t(__popc(mine & ((1u << slot) - 1u)));
                if (live && slot == 0u) a.base[w] = base;
            }
        }
        __syncthreads();
        if (pass == 0 && threadIdx.x == 0) first = 1u + atomicAdd(a.made, children);
        __syncthreads();
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) a.place[0] = 0u;
}

// The units themselves.
__global__ void __launch_bounds__(kWideBlock) wide_nodes_kernel(WideArgs a) {
    __shared__ uint32_t list[kWideBlock], count;
    const uint32_t n = list_wide(a, list, &count);
    // half the pad again: a wide node's slab test rounds once more than a float box's
    const float margin = 0.5f * box_pad(a.bounds);
    const uint32_t lane = threadIdx.x % kWave, slot = lane & 7u;
    for (uint32_t k = threadIdx.x & ~uint32_t(kWave - 1); k < 8u * n; k += kWideBlock) {  // wave-uniform
        const uint32_t at = (k + lane) >> 3;
        const bool live = at < n;
        const uint32_t w = live ? list[at] : 0u;
        const uint32_t side = live ? a.sides[8ull * w + slot] : kNone;
        const bool in = side != kNone;
        const uint32_t child = in ? side_child(a, side) : kLeaf;
        float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
        bool used = false;
        if (in) {
            const float4 p = side_box(a, side)[0], q = side_box(a, side)[1];
            // (an inner child of nothing but empty boxes is never hit)
            used = p.x <= q.x && p.y <= q.y && p.z <= q.z;
            if (used) {
                lo[0] = p.x - margin; lo[1] = p.y - margin; lo[2] = p.z - margin;
                hi[0] = q.x + margin; hi[1] = q.y + margin; hi[2] = q.z + margin;
            }
        }
        uint32_t inner = in && !(child & kLeaf) ? 1u << slot : 0u, leaves = in && (child & kLeaf) ? 1u << slot : 0u;
        float origin[3], top[3];
        for (int c = 0; c < 3; ++c) {
            origin[c] = lo[c];
            top[c] = hi[c];
        }
        for (int s = 1; s < 8; s <<= 1) {
            inner |= uint32_t(__shfl_xor(int(inner), s, kWave));
            leaves |= uint32_t(__shfl_xor(int(leaves), s, kWave));
            for (int c = 0; c < 3; ++c) {
                origin[c] = fminf(origin[c], __shfl_xor(origin[c], s, kWave));
                top[c] = fmaxf(top[c], __shfl_xor(top[c], s, kWave));
            }
        }
        // the origin's upper 24 bits, towards -inf, and the unit: the power
        // of two at or above the largest extent / 255 (normal numbers only)
        bool finite = true;
        float ext = 0.0f;
        uint32_t words[3], q_lo[3], q_hi[3];
        for (int c = 0; c < 3; ++c) {
            finite = finite && fabsf(origin[c]) < 1e35f && fabsf(top[c]) < 1e35f;
            words[c] = __float_as_uint(origin[c]);
            words[c] = origin[c] < 0.0f ? (words[c] + 0xffu) & 0xffffff00u : words[c] & 0xffffff00u;
            origin[c] = __uint_as_float(words[c]);
            ext = fmaxf(ext, top[c] - origin[c]);
        }
        int e = -100;
        if (ext > 0.0f && finite) (void)frexpf(ext / 255.0f, &e);
        e = max(e, -100);
        const float per = ldexpf(1.0f, -e);
        // not finite: an infinite unit from 0, so that no plane cuts anything
        // off (0 * inf is NaN, which the slab test's min and max drop)
        if (!finite) e = 128;
        for (int c = 0; c < 3; ++c) {
            q_lo[c] = 0u;
            q_hi[c] = 255u;
            if (!finite) {
                words[c] = 0u;
            } else {
                q_lo[c] = uint32_t(fminf(fmaxf(floorf((lo[c] - origin[c]) * per), 0.0f), 255.0f));
                q_hi[c] = uint32_t(fminf(fmaxf(ceilf((hi[c] - origin[c]) * per), 0.0f), 255.0f));
            }
            if (!used) {
                q_lo[c] = 255u;
                q_hi[c] = 0u;
            }
        }
        if (live) {
            WideNode* out = a.units + a.place[w];
            const uint32_t base = a.base[w];
            uint8_t* planes = reinterpret_cast<uint8_t*>(out->planes);
            for (int c = 0; c < 3; ++c) {
                planes[16 * c + slot] = uint8_t(q_lo[c]);
                planes[16 * c + 8 + slot] = uint8_t(q_hi[c]);
            }
            if (slot == 0u) {
                out->origin[0] = words[0] | uint32_t(e + 127);
                out->origin[1] = words[1] | inner;
                out->origin[2] = words[2] | leaves;
                out->base = base;
            }
            if ((leaves >> slot) & 1u) {
                const uint32_t l = child & ~kLeaf;
                TraceLeaf* leaf = reinterpret_cast<TraceLeaf*>(a.units) + base + __popc((inner | leaves) & ((1u << slot) - 1u));
                leaf->a = a.prims[2ull * l];
                leaf->b = a.prims[2ull * l + 1];
                leaf->seg = a.prim_seg[l];
            }
        }
    }
}

// The one unit of a tree of one segment.
__global__ void single_leaf_kernel(const float4* __restrict__ prims, const uint32_t* __restrict__ seg, TraceLeaf* leaf) {
    leaf->a = prims[0];
    leaf->b = prims[1];
    leaf->seg = seg[0];
}

// ---------------------------------------------------------------- tracing

constexpr int kTraceBlock = 64;
__global__ void __launch_bounds__(kTraceBlock)
rays_kernel(TraceBvh b, const float* __restrict__ rays, uint32_t n, int any, float* t_out, float* u_out,
            uint32_t* seg_out) {
    __shared__ TraceLds lds;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = i < n;
    const float* r = rays + 8ull * (active ? i : 0u);
    const float3 o = make_float3(r[0], r[1], r[2]), d = make_float3(r[4], r[5], r[6]);
    const Hit h = any ? trace<true>(b, lds, active, o, d, r[3], r[7]) : trace<false>(b, lds, active, o, d, r[3], r[7]);
    if (!active) return;
    const bool hit = h.seg != kNone;
    if (t_out) t_out[i] = hit ? h.t : 0.0f;
    if (u_out) u_out[i] = hit ? h.u : 0.0f;
    seg_out[i] = hit ? h.seg : kNone;
}

struct FrameArgs {
    TraceBvh b;
    const float* tangents;
    const uint32_t* indices;
    float plane[12];
    float light[6];
    float diffuse[3];
    float exponent, ao_radius;
    int method, shadows_on, ignore_self;
    uint32_t seed, frame, width, height;
    double* accum;
};

__device__ __forceinline__ uint32_t mix32(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

__device__ __forceinline__ float sample(uint32_t seed, uint32_t pixel, uint32_t frame, uint32_t k, float lo,
                                        float hi) {
    const uint32_t r = mix32(mix32(mix32(seed ^ 0x9e3779b9u) ^ pixel) ^ (frame * 8u + k));
    return (float(r) / 4294967296.0f) * (hi - lo) + lo;
}

__device__ __forceinline__ float3 normalized(float3 v) {
    const float l = sqrtf(dot3(v, v));
    return make_float3(v.x / l, v.y / l, v.z / l);
}

constexpr float kEpsilon = 0.000001f;  // Ray::Epsilon (ray_tracer/ray.hh:15)

// One sample of Raytracer::draw per pixel; 8x8 pixels per block of one wave.
__global__ void __launch_bounds__(kTraceBlock) frame_kernel(FrameArgs a) {
    __shared__ TraceLds lds;
    const uint32_t i = blockIdx.x * 8u + (threadIdx.x & 7u), j = blockIdx.y * 8u + (threadIdx.x >> 3);
    const bool inside = i < a.width && j < a.height;  // (every lane traces)
    const uint32_t pix = i + j * a.width;
    const float3 X = make_float3(a.plane[0], a.plane[1], a.plane[2]);
    const float3 Y = make_float3(a.plane[3], a.plane[4], a.plane[5]);
    const float3 Z = make_float3(a.plane[6], a.plane[7], a.plane[8]);
    const float3 eye = make_float3(a.plane[9], a.plane[10], a.plane[11]);
    const float fx = float(i) + sample(a.seed, pix, a.frame, 0, 0.0f, 1.0f);
    const float fy = float(j) + sample(a.seed, pix, a.frame, 1, 0.0f, 1.0f);
    const float3 d = make_float3((fx * X.x + fy * Y.x) + Z.x, (fx * X.y + fy * Y.y) + Z.y, (fx * X.z + fy * Y.z) + Z.z);
    float color[3] = {1.0f, 1.0f, 1.0f};
    const Hit h = trace<false>(a.b, lds, inside, eye, d, 0.0f, INFINITY);
    const bool hit = h.seg != kNone;
    if (__ballot(hit) != 0ull) {
        const float3 P = make_float3(eye.x + d.x * h.t, eye.y + d.y * h.t, eye.z + d.z * h.t);
        const uint32_t skip = a.ignore_self ? h.seg : kNone;  // secondary rays may skip their own segment
        float L[3] = {1.0f, 1.0f, 1.0f};
        if (a.method != 3) {
            // the shadow ray's direction is the jittered light position itself
            const float3 sd = make_float3(a.light[0] + sample(a.seed, pix, a.frame, 2, -16.0f, 16.0f),
                                          a.light[1] + sample(a.seed, pix, a.frame, 3, -16.0f, 16.0f),
                                          a.light[2] + sample(a.seed, pix, a.frame, 4, -16.0f, 16.0f));
            const bool occluded = trace<true>(a.b, lds, hit, P, sd, kEpsilon, INFINITY, skip).seg != kNone;
            if (!occluded || !a.shadows_on) {
                if (a.method == 0 && hit) {
                    const uint32_t ia = a.indices[2ull * h.seg], ib = a.indices[2ull * h.seg + 1];
                    const float3 t0 = load_xyz(a.tangents, ia), t1 = load_xyz(a.tangents, ib);
                    const float3 T = make_float3(t0.x + h.u * (t1.x - t0.x), t0.y + h.u * (t1.y - t0.y),
                                                 t0.z + h.u * (t1.z - t0.z));
                    const float3 l = normalized(make_float3(a.light[0] - P.x, a.light[1] - P.y, a.light[2] - P.z));
                    const float3 e = normalized(make_float3(P.x - eye.x, P.y - eye.y, P.z - eye.z));
                    // embree::HairStyle::kajiya_kay (ray_tracer/hair_style.cc:86-107)
                    const float ctl = dot3(l, T), cte = dot3(e, T);
                    const float sa = 1.0f - ctl * ctl, sb = 1.0f - cte * cte;
                    const float stl = sqrtf(sa > 0.0f ? sa : 0.0f), ste = sqrtf(sb > 0.0f ? sb : 0.0f);
                    const float base = ctl * cte + stl * ste;
                    float spec = base > 0.0f ? powf(base, a.exponent) : 0.0f;
                    spec = spec < 0.0f ? 0.0f : (spec > 1.0f ? 1.0f : spec);
                    for (int c = 0; c < 3; ++c) L[c] = a.diffuse[c] * stl + a.light[3 + c] * spec;
                }
            } else {
                L[0] = L[1] = L[2] = 0.0f;
            }
        }
        for (int c = 0; c < 3; ++c) color[c] = hit ? L[c] : color[c];
        if (a.method != 2) {
            const float3 rd = make_float3(sample(a.seed, pix, a.frame, 5, -1.0f, 1.0f),
                                          sample(a.seed, pix, a.frame, 6, -1.0f, 1.0f),
                                          sample(a.seed, pix, a.frame, 7, -1.0f, 1.0f));
            const float len = sqrtf(dot3(rd, rd));
            const float t_max = len > 0.0f ? (a.ao_radius / len) * 1.001f + kEpsilon : INFINITY;
            const Hit o = trace<false>(a.b, lds, hit, P, rd, kEpsilon, t_max, skip);
            float ao = 2.0f;
            if (o.seg != kNone) {
                const float3 q = make_float3((P.x + rd.x * o.t) - P.x, (P.y + rd.y * o.t) - P.y,
                                             (P.z + rd.z * o.t) - P.z);
                if (!(sqrtf(dot3(q, q)) > a.ao_radius)) ao = 0.0f;
            }
            for (int c = 0; c < 3; ++c) color[c] = hit ? color[c] * ao : color[c];
        }
    }
    if (!inside) return;
    double* out = a.accum + 3ull * pix;
    for (int c = 0; c < 3; ++c) out[c] += double(color[c]);
}

}  // namespace
}  // namespace vkhr

using namespace vkhr;

struct vkhr_bvh {
    int device = 0;
    uint32_t n = 0;
    void* memory = nullptr;     // one allocation holding every array below
    size_t bytes = 0;           // of it
    WideNode* units = nullptr;
    float4* nodes = nullptr;    // the binary tree the wide nodes were cut from (vkhr_bvh_nodes)
    uint32_t* parent = nullptr;
    uint32_t* prim_seg = nullptr;
    float bounds[6] = {0, 0, 0, 0, 0, 0};

    TraceBvh view() const { return TraceBvh{units, n}; }
};

namespace {

template <class T>
T* carve(char*& p, size_t count) {
    T* out = reinterpret_cast<T*>(p);
    p += (count * sizeof(T) + 255) & ~size_t(255);
    return out;
}

size_t carve_size(size_t bytes) { return (bytes + 255) & ~size_t(255); }

// The build's kernels take an element per thread, without a stride: their
// launches hold every element of the largest tree (at most 2^22 workgroups).
constexpr uint32_t kMostSegments = (1u << 30) - 1u;   // int range search in the tree build
unsigned blocks_of(size_t n, unsigned block) { return unsigned((n + block - 1) / block); }

}  // namespace

extern "C" int vkhr_bvh_build(const float* xyz, const float* radius, uint32_t n_vertices, const uint32_t* indices,
                              uint32_t n_indices, vkhr_stream stream, vkhr_bvh** out) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    VKHR_REQUIRE(out, VKHR_ERR_INVALID, "out is null");
    *out = nullptr;
    const uint32_t n = n_indices / 2;
    // (an argument passed in the wrong position usually shows up as a small integer here)
    const auto plausible = [](const void* p) { return reinterpret_cast<uintptr_t>(p) >= 65536u; };
    VKHR_REQUIRE(n == 0 || (plausible(xyz) && plausible(radius) && plausible(indices)), VKHR_ERR_INVALID,
                 "null or implausible geometry pointer");
    VKHR_REQUIRE(n <= kMostSegments, VKHR_ERR_OVERFLOW, "too many segments");
    hipStream_t s = as_stream(stream);
    VKHR_REQUIRE(n == 0 || !capturing(s), VKHR_ERR_HIP,
                 "bvh build synchronises its stream, which is being captured");
    int device = 0;
    VKHR_CHECK_HIP(hipGetDevice(&device));
    vkhr_bvh* b = new vkhr_bvh();
    b->device = device;
    b->n = n;
    if (n == 0) {
        *out = b;
        return VKHR_OK;
    }
    const size_t inner = n > 1 ? n - 1 : 0;
    const size_t keep = carve_size((inner + n) * sizeof(WideNode)) + carve_size(inner * 4 * sizeof(float4)) +
                        carve_size((inner + n) * sizeof(uint32_t)) + carve_size(n * sizeof(uint32_t));
    const uint32_t blocks = blocks_of(n, 256);
    // temporaries: boxes (input order), the pyramid of leaf boxes, bounds, keys/values x2, sort scratch
    size_t sort_bytes = 0;
    if (rocprim::radix_sort_pairs(nullptr, sort_bytes, static_cast<uint32_t*>(nullptr),
                                  static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr),
                                  static_cast<uint32_t*>(nullptr), size_t(n), 0, 30, s) != hipSuccess) {
        delete b;
        set_error("rocprim::radix_sort_pairs size query failed");
        return VKHR_ERR_HIP;
    }
    Pyramid pyr{};
    size_t pyramid_bytes = 0;
    for (size_t c = n; pyr.levels < kMaxLevels; c = (c + 7) / 8) {
        pyr.count[pyr.levels++] = int(c);
        pyramid_bytes += carve_size(c * sizeof(Box));
        if (c <= 8) break;
    }
    const size_t temp = 2 * carve_size(n * sizeof(float4)) + pyramid_bytes + carve_size(2 * size_t(n) * sizeof(float4)) + carve_size(size_t(blocks) * 6 * sizeof(float)) +
                        carve_size(12 * sizeof(float)) + 4 * carve_size(n * sizeof(uint32_t)) +
                        carve_size(sizeof(uint32_t)) + carve_size(inner * sizeof(int2)) +
                        2 * carve_size(inner * sizeof(uint32_t)) + carve_size(8 * inner * sizeof(uint32_t)) +
                        carve_size(sort_bytes);
    hipError_t e = hipSuccess;
    const RelaxedCapture relaxed;
    b->memory = reuse_block(device, keep, &b->bytes);
    if (!b->memory) {
        b->bytes = keep;
        e = hipMalloc(&b->memory, keep);
    }
    const CallScratch temporaries(temp, s);
    if (e == hipSuccess && !temporaries.get()) e = hipErrorOutOfMemory;
    if (e != hipSuccess) {
        if (b->memory) (void)hipFree(b->memory);
        delete b;
        set_error("bvh hipMalloc failed: %s", hipGetErrorString(e));
        return VKHR_ERR_NOMEM;
    }
    char* p = static_cast<char*>(b->memory);
    b->units = carve<WideNode>(p, inner + n);
    b->nodes = carve<float4>(p, inner * 4);
    b->parent = carve<uint32_t>(p, inner + n);
    b->prim_seg = carve<uint32_t>(p, n);
    char* q = static_cast<char*>(temporaries.get());
    BuildArgs a;
    a.xyz = xyz;
    a.radius = radius;
    a.indices = indices;
    a.n_vertices = n_vertices;
    a.n = n;
    a.box_lo = carve<float4>(q, n);
    a.box_hi = carve<float4>(q, n);
    for (int k = 0; k < pyr.levels; ++k) pyr.level[k] = carve<Box>(q, size_t(pyr.count[k]));
    float4* prims = carve<float4>(q, 2 * size_t(n));
    a.bounds_partial = carve<float>(q, size_t(blocks) * 6);
    a.bounds = carve<float>(q, 12);
    a.keys = carve<uint32_t>(q, n);
    a.values = carve<uint32_t>(q, n);
    uint32_t* keys_sorted = carve<uint32_t>(q, n);
    uint32_t* order = carve<uint32_t>(q, n);
    uint32_t* made = carve<uint32_t>(q, 1);
    int2* ranges = carve<int2>(q, inner);
    uint32_t* place = carve<uint32_t>(q, inner);
    uint32_t* base = carve<uint32_t>(q, inner);
    uint32_t* sides = carve<uint32_t>(q, 8 * inner);
    void* sort_tmp = carve<char>(q, sort_bytes);
    auto fail = [&](int code) {
        (void)hipStreamSynchronize(s);
        (void)hipFree(b->memory);
        delete b;
        return code;
    };
    HostWords host;
    a.host_bounds = reinterpret_cast<float*>(host.words());
    segment_boxes_kernel<<<blocks, 256, 0, s>>>(a);
    bounds_final_kernel<<<1, 256, 0, s>>>(a, blocks);
    morton_kernel<<<blocks, 256, 0, s>>>(a);
    if (hipGetLastError() != hipSuccess ||
        rocprim::radix_sort_pairs(sort_tmp, sort_bytes, a.keys, keys_sorted, a.values, order, size_t(n), 0, 30, s) !=
            hipSuccess) {
        set_error("bvh sort failed");
        return fail(VKHR_ERR_HIP);
    }
    leaves_kernel<<<blocks_of(n, kPyramidBlock), kPyramidBlock, 0, s>>>(a, order, pyr, prims, b->prim_seg, made);
    if (n > 1) {
        for (int in = 3; in + 1 < pyr.levels; in += 3)
            pyramid_kernel<<<blocks_of(size_t(pyr.count[in]), kPyramidBlock), kPyramidBlock, 0, s>>>(pyr, in);
        radix_tree_kernel<<<blocks_of(inner, 256), 256, 0, s>>>(keys_sorted, int(n), pyr, b->nodes, b->parent, ranges);
        const WideArgs wa{keys_sorted, b->nodes, b->parent, ranges, int(n), a.bounds, prims, b->prim_seg,
                          made, place, base, sides, b->units};
        const uint32_t wide_blocks = blocks_of(inner, kWideBlock);
        wide_place_kernel<<<wide_blocks, kWideBlock, 0, s>>>(wa);
        wide_nodes_kernel<<<wide_blocks, kWideBlock, 0, s>>>(wa);
    } else {
        single_leaf_kernel<<<1, 1, 0, s>>>(prims, b->prim_seg, reinterpret_cast<TraceLeaf*>(b->units));
    }
    if (hipGetLastError() != hipSuccess ||
        (!host.words() &&
         hipMemcpyAsync(b->bounds, a.bounds, sizeof(b->bounds), hipMemcpyDeviceToHost, s) != hipSuccess) ||
        hipStreamSynchronize(s) != hipSuccess) {
        set_error("bvh build kernels failed");
        return fail(VKHR_ERR_HIP);
    }
    if (host.words()) std::memcpy(b->bounds, host.words(), sizeof(b->bounds));
    *out = b;
    return VKHR_OK;
}

extern "C" int vkhr_bvh_destroy(vkhr_bvh* b) {
    clear_error();
    if (!b) return VKHR_OK;
    int prev = 0;
    (void)hipGetDevice(&prev);
    (void)hipSetDevice(b->device);
    const RelaxedCapture relaxed;
    if (b->memory && !keep_block(b->device, b->memory, b->bytes)) (void)hipFree(b->memory);
    (void)hipSetDevice(prev);
    delete b;
    return VKHR_OK;
}

extern "C" int vkhr_bvh_info(const vkhr_bvh* b, uint32_t* n_segments, float* bounds) {
    clear_error();
    VKHR_REQUIRE(b, VKHR_ERR_INVALID, "bvh is null");
    if (n_segments) *n_segments = b->n;
    if (bounds) std::memcpy(bounds, b->bounds, sizeof(b->bounds));
    return VKHR_OK;
}

extern "C" int vkhr_bvh_nodes(const vkhr_bvh* b, float* nodes, uint32_t* parent, uint32_t* leaf_segment,
                              vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    VKHR_REQUIRE(b, VKHR_ERR_INVALID, "bvh is null");
    hipStream_t s = as_stream(stream);
    const size_t inner = b->n > 1 ? b->n - 1 : 0;
    if (nodes && inner) VKHR_CHECK_HIP(hipMemcpyAsync(nodes, b->nodes, inner * 4 * sizeof(float4), hipMemcpyDefault, s));
    if (parent && b->n)
        VKHR_CHECK_HIP(hipMemcpyAsync(parent, b->parent, (inner + b->n) * sizeof(uint32_t), hipMemcpyDefault, s));
    if (leaf_segment && b->n)
        VKHR_CHECK_HIP(hipMemcpyAsync(leaf_segment, b->prim_seg, b->n * sizeof(uint32_t), hipMemcpyDefault, s));
    return VKHR_OK;
}

extern "C" int vkhr_trace_rays(const vkhr_bvh* b, const float* rays, uint32_t n_rays, int any_hit, float* t_out,
                               float* u_out, uint32_t* segment_out, vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    VKHR_REQUIRE(b && (n_rays == 0 || (rays && segment_out)), VKHR_ERR_INVALID, "null argument");
    if (n_rays == 0) return VKHR_OK;
    rays_kernel<<<(n_rays - 1) / kTraceBlock + 1, kTraceBlock, 0, as_stream(stream)>>>(b->view(), rays, n_rays, any_hit, t_out, u_out,
                                                                      segment_out);
    VKHR_CHECK_LAUNCH();
    return VKHR_OK;
}

extern "C" int vkhr_raytrace(const vkhr_bvh* b, const float* tangents, const uint32_t* indices,
                             const vkhr_viewing_plane* plane, const vkhr_light* light,
                             const vkhr_trace_params* params, uint32_t width, uint32_t height, double* accum,
                             vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    VKHR_REQUIRE(b && plane && light && params && accum, VKHR_ERR_INVALID, "null argument");
    VKHR_REQUIRE(width && height && width <= 16384 && height <= 16384, VKHR_ERR_INVALID, "bad image size %ux%u",
                 width, height);
    VKHR_REQUIRE(params->method <= 3, VKHR_ERR_INVALID, "unknown method %u", params->method);
    VKHR_REQUIRE(b->n == 0 || indices, VKHR_ERR_INVALID, "indices are null");
    VKHR_REQUIRE(params->method != 0 || b->n == 0 || tangents, VKHR_ERR_INVALID, "shading needs tangents");
    FrameArgs a;
    std::memset(&a, 0, sizeof(a));
    a.b = b->view();
    a.tangents = tangents;
    a.indices = indices;
    for (int c = 0; c < 3; ++c) {
        a.plane[c] = plane->x[c];
        a.plane[3 + c] = plane->y[c];
        a.plane[6 + c] = plane->z[c];
        a.plane[9 + c] = plane->point[c];
        a.light[c] = light->origin[c];
        a.light[3 + c] = light->intensity[c];
        a.diffuse[c] = params->diffuse[c];
    }
    a.exponent = params->exponent;
    a.ao_radius = params->ao_radius;
    a.method = int(params->method);
    a.shadows_on = params->shadows_on;
    a.ignore_self = params->ignore_self ? 1 : 0;
    a.seed = params->seed;
    a.frame = params->frame;
    a.width = width;
    a.height = height;
    a.accum = accum;
    frame_kernel<<<dim3((width + 7) / 8, (height + 7) / 8), kTraceBlock, 0, as_stream(stream)>>>(a);
    VKHR_CHECK_LAUNCH();
    return VKHR_OK;
}
