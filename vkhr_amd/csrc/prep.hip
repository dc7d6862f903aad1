// Load-time preparation of a hair style: the reference's generators
// HairStyle::generate_bounding_box / generate_indices / generate_tangents
// (src/vkhr/scene_graph/hair_style.cc:171-255) on the device.
// Compiled with -ffp-contract=off: tangents match the reference's float
// arithmetic bit for bit (glm::normalize = v * (1 / sqrt(dot(v, v))), dot
// summed x, y, then z).
#include "common.hpp"

#include <cmath>
#include <cstring>

namespace vkhr {
namespace {

constexpr int kAabbBlock = 256;
constexpr int kAabbGrid = 1024;

__device__ __forceinline__ float wave_min(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, kWave));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
    return v;
}

// Stage 1: each block reduces a strided share of the vertices to 6 floats
// (min xyz, max xyz), both started at the origin as the reference does.
__global__ void __launch_bounds__(kAabbBlock)
aabb_partial_kernel(const float* __restrict__ xyz, uint32_t n, float* __restrict__ partial) {
    float mn[3] = {0.0f, 0.0f, 0.0f}, mx[3] = {0.0f, 0.0f, 0.0f};
    uint32_t stride = gridDim.x * blockDim.x;
#pragma unroll 4
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        float3 p = load_xyz(xyz, i);
        mn[0] = fminf(mn[0], p.x); mn[1] = fminf(mn[1], p.y); mn[2] = fminf(mn[2], p.z);
        mx[0] = fmaxf(mx[0], p.x); mx[1] = fmaxf(mx[1], p.y); mx[2] = fmaxf(mx[2], p.z);
    }
    __shared__ float red[6][kAabbBlock / kWave];
    int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
    for (int c = 0; c < 3; ++c) {
        float a = wave_min(mn[c]), b = wave_max(mx[c]);
        if (lane == 0) { red[c][wid] = a; red[3 + c][wid] = b; }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        int c = threadIdx.x;
        float r = red[c][0];
        for (int w = 1; w < kAabbBlock / kWave; ++w) r = c < 3 ? fminf(r, red[c][w]) : fmaxf(r, red[c][w]);
        partial[6 * blockIdx.x + c] = r;
    }
}

// Stage 2: one block folds the per-block results, a thread per stage-1 block
// (a load each instead of sixteen in a row by one wave: 7.1 -> 5.8 us).
__global__ void __launch_bounds__(kAabbGrid)
aabb_final_kernel(const float* __restrict__ partial, int blocks, float* __restrict__ out) {
    __shared__ float red[6][kAabbGrid / kWave];
    const int b = threadIdx.x, lane = b % kWave, wid = b / kWave;
    float v[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) v[c] = b < blocks ? partial[6 * b + c] : 0.0f;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        const float r = c < 3 ? wave_min(v[c]) : wave_max(v[c]);
        if (lane == 0) red[c][wid] = r;
    }
    __syncthreads();
    if (b < 6) {
        float r = red[b][0];
        for (int w = 1; w < kAabbGrid / kWave; ++w) r = b < 3 ? fminf(r, red[b][w]) : fmaxf(r, red[b][w]);
        out[b] = r;
    }
}

// The two generators below give a strand to a group of 1 to 16 lanes, the
// power of two at or above the mean strand, which take its vertices (or pairs) that many
// at a time: a strand's vertices are consecutive, so a group reads and writes
// whole lines, where a thread per strand spread every load and store of a
// wave over 64 strands.  What bounds them is memory: at 136k strands of 13
// vertices (21 MB in, 21 MB out) the tangents take 13.9 us, 51.4 with a thread
// per strand; the indices 7.5 us, 12.2 before; reading the mean first costs
// the tangents 0.8 (4096 workgroups; 8192 1.3).  Sixteen lanes whatever the
// strands leave most of them idle on short ones: tangents of
// 4M strands of two vertices 158 us (58 now), their indices 94 (25).
constexpr uint32_t kMostLanes = 16, kStrandBlocks = 4096;

template <uint32_t kLanes, typename Strand>
__device__ __forceinline__ void grouped_strands(uint32_t n_strands, Strand strand) {
    const uint32_t lane = threadIdx.x % kLanes, per_block = blockDim.x / kLanes;
    for (size_t s = size_t(blockIdx.x) * per_block + threadIdx.x / kLanes; s < n_strands;
         s += size_t(gridDim.x) * per_block)
        strand(uint32_t(s), lane, kLanes);
}

// Calls strand(s, lane, lanes) for the strands of this lane's group; a strand
// has its vertices less `less` items.
template <typename Strand>
__device__ __forceinline__ void each_strand(const uint32_t* __restrict__ offsets, uint32_t n_strands, uint32_t less,
                                            Strand strand) {
    const uint64_t n = n_strands, items = offsets[n_strands] - offsets[0] - less * n_strands;
    if (items > 8u * n)
        grouped_strands<kMostLanes>(n_strands, strand);
    else if (items > 4u * n)
        grouped_strands<8>(n_strands, strand);
    else if (items > 2u * n)
        grouped_strands<4>(n_strands, strand);
    else if (items > n)
        grouped_strands<2>(n_strands, strand);
    else
        grouped_strands<1>(n_strands, strand);
}

__global__ void __launch_bounds__(256)
indices_kernel(const uint32_t* __restrict__ offsets, uint32_t n_strands, uint32_t* __restrict__ indices) {
    each_strand(offsets, n_strands, 1u, [&](uint32_t s, uint32_t lane, uint32_t lanes) {
        const uint32_t first = offsets[s], end = offsets[s + 1u];
        const uint32_t out = 2u * (first - s);  // every earlier strand skipped its last vertex
        for (uint32_t v = first + lane; v + 1u < end; v += lanes) {
            indices[out + 2u * (v - first)] = v;
            indices[out + 2u * (v - first) + 1u] = v + 1u;
        }
    });
}

__device__ __forceinline__ float3 glm_normalize(float3 v) {
    float d = (v.x * v.x + v.y * v.y) + v.z * v.z;
    float r = 1.0f / sqrtf(d);
    return make_float3(v.x * r, v.y * r, v.z * r);
}

__global__ void __launch_bounds__(256)
tangents_kernel(const float* __restrict__ xyz, const uint32_t* __restrict__ offsets, uint32_t n_strands,
                float* __restrict__ tangents) {
    each_strand(offsets, n_strands, 0u, [&](uint32_t s, uint32_t lane, uint32_t lanes) {
        const uint32_t first = offsets[s], end = offsets[s + 1u];
        for (uint32_t v = first + lane; v < end; v += lanes) {
            // the strand's last vertex repeats the previous tangent
            const uint32_t a = v + 1u < end ? v : v - 1u;
            float3 t = make_float3(0.0f, 0.0f, 0.0f);
            if (end - first > 1u) {
                const float3 cur = load_xyz(xyz, a), nxt = load_xyz(xyz, a + 1u);
                t = glm_normalize(make_float3(nxt.x - cur.x, nxt.y - cur.y, nxt.z - cur.z));
            }
            tangents[3u * v + 0u] = t.x;
            tangents[3u * v + 1u] = t.y;
            tangents[3u * v + 2u] = t.z;
        }
    });
}

}  // namespace
}  // namespace vkhr

using namespace vkhr;

extern "C" int vkhr_aabb_compute(const float* xyz, uint32_t n_vertices, vkhr_aabb* out, vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    VKHR_REQUIRE(out, VKHR_ERR_INVALID, "out is null");
    VKHR_REQUIRE(n_vertices == 0 || xyz, VKHR_ERR_INVALID, "xyz is null");
    float mm[6] = {0, 0, 0, 0, 0, 0};
    if (n_vertices) {
        const RelaxedCapture relaxed;   // (it waits for the stream)
        void* scr = nullptr;
        if ((rc = stream_scratch(sizeof(float) * (6 * kAabbGrid + 8), as_stream(stream), &scr))) return rc;
        float* partial = static_cast<float*>(scr);
        HostWords host;
        float* result = host.words() ? reinterpret_cast<float*>(host.words()) : partial + 6 * kAabbGrid;
        hipStream_t s = as_stream(stream);
        int blocks = int(grid_for(n_vertices, kAabbBlock, kAabbGrid));
        aabb_partial_kernel<<<blocks, kAabbBlock, 0, s>>>(xyz, n_vertices, partial);
        VKHR_CHECK_LAUNCH();
        aabb_final_kernel<<<1, kAabbGrid, 0, s>>>(partial, blocks, result);
        VKHR_CHECK_LAUNCH();
        if (!host.words()) VKHR_CHECK_HIP(hipMemcpyAsync(mm, result, sizeof(mm), hipMemcpyDeviceToHost, s));
        VKHR_CHECK_HIP(hipStreamSynchronize(s));
        if (host.words()) std::memcpy(mm, host.words(), sizeof(mm));
    }
    // get_bounding_box (hair_style.cc:236-255), float arithmetic
    for (int c = 0; c < 3; ++c) {
        out->origin[c] = mm[c];
        out->size[c] = mm[3 + c] - mm[c];
    }
    volatile float sx = out->size[0], sy = out->size[1], sz = out->size[2];
    float xx = sx * sx, yy = sy * sy, zz = sz * sz;
    float dot = (xx + yy) + zz;
    out->radius = std::sqrt(dot);
    float xy = sx * sy;
    out->volume = xy * sz;
    return VKHR_OK;
}

extern "C" int vkhr_generate_indices(const uint32_t* strand_offsets, uint32_t n_strands, uint32_t* indices,
                                     vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    if (n_strands == 0) return VKHR_OK;
    VKHR_REQUIRE(strand_offsets && indices, VKHR_ERR_INVALID, "null pointer");
    indices_kernel<<<grid_for(n_strands, 256 / kMostLanes, kStrandBlocks), 256, 0, as_stream(stream)>>>(
        strand_offsets, n_strands, indices);
    VKHR_CHECK_LAUNCH();
    return VKHR_OK;
}

extern "C" int vkhr_generate_tangents(const float* xyz, const uint32_t* strand_offsets, uint32_t n_strands,
                                      float* tangents, vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    if (n_strands == 0) return VKHR_OK;
    VKHR_REQUIRE(xyz && strand_offsets && tangents, VKHR_ERR_INVALID, "null pointer");
    tangents_kernel<<<grid_for(n_strands, 256 / kMostLanes, kStrandBlocks), 256, 0, as_stream(stream)>>>(
        xyz, strand_offsets, n_strands, tangents);
    VKHR_CHECK_LAUNCH();
    return VKHR_OK;
}
