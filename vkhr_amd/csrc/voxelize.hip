// Strand voxelization: the reference's CPU voxelizers
// (src/vkhr/scene_graph/hair_style.cc:257-342) as gfx950 kernels.
//
// Counts are integers, so the result is independent of the order in which
// threads add them: one thread walks one segment with exactly the
// reference's float arithmetic (this file is compiled with
// -ffp-contract=off, division and sqrt are IEEE correctly rounded by
// default on HIP) and adds 1 to each voxel it visits.  The reference's
// float linear index x + y*w + z*w*h is formed from integers < 2^24 and is
// therefore exact; it is computed here in integer arithmetic, which is
// identical as long as nx*ny*nz <= 2^24 (enforced).
#include "voxel.hpp"

#include <cmath>

namespace vkhr {
namespace {

// Grid-stride over wave-aligned ranges so that whole waves stay converged
// for the wave-cooperative bodies.
__global__ void __launch_bounds__(256)
voxelize_vertices_kernel(const float* __restrict__ xyz, uint32_t n_vertices,
                         const float* __restrict__ tangents, VoxelGrid g,
                         uint32_t* __restrict__ counts, long long* __restrict__ sums) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t base = blockIdx.x * blockDim.x + (threadIdx.x & ~uint32_t(kWave - 1)); base < n_vertices;
         base += stride) {
        const uint32_t i = base + (threadIdx.x & uint32_t(kWave - 1));
        voxelize_vertex(g, xyz, i < n_vertices, i, tangents, counts, sums);
    }
}

__global__ void __launch_bounds__(256)
voxelize_segments_kernel(const float* __restrict__ xyz, uint32_t n_vertices,
                         const uint32_t* __restrict__ indices, uint32_t n_pairs, const float* __restrict__ tangents, VoxelGrid g,
                         uint32_t* __restrict__ counts, long long* __restrict__ sums) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t base = blockIdx.x * blockDim.x + (threadIdx.x & ~uint32_t(kWave - 1)); base < n_pairs;
         base += stride) {
        const uint32_t s = base + (threadIdx.x & uint32_t(kWave - 1));
        const bool has = s < n_pairs;
        voxelize_segment(g, xyz, n_vertices, has, has ? indices[2u * s] : 0u, has ? indices[2u * s + 1u] : 0u,
                         tangents, counts, sums);
    }
}

// counts[v] = the count held in word 1 of the packed accumulator.
__global__ void __launch_bounds__(256)
unpack_counts_kernel(const long long* __restrict__ acc, uint32_t* __restrict__ counts, size_t n) {
    const size_t stride = size_t(gridDim.x) * blockDim.x;
    for (size_t v = size_t(blockIdx.x) * blockDim.x + threadIdx.x; v < n; v += stride) counts[v] = packed_count(acc, v);
}

// --- vertices by bricks -----------------------------------------------------
// With tangents a vertex is 16 bytes of integer adds to one voxel; as device
// atomics they are a memory-side line request each, 22 G/s, whatever else the
// kernel does.  A vertex belongs to one brick of 8x8x8 voxels, so the vertices
// are counting-sorted by brick instead (a histogram per block, its columns
// scanned, 8 bytes per vertex written) and workgroups, each of one brick, add them
// in LDS and write the accumulator and the counts, which then need neither
// clearing nor unpacking.  The sums are the same integers in any order.
// 1.77M vertices / 128^3: clearing 8.5, atomics 79.3, unpacking 7.8 us before,
// now 43.6 (histogram 8.1, columns 4.2, fill 20.5, bricks 10.8; the fill is
// bound by its scattered writes).
constexpr uint32_t kBinBricks = 8192;          // a histogram in 32 KB of LDS: up to 160^3 (no larger one was measured)
constexpr uint32_t kBinBlocks = 256;           // rows of the histogram at most
constexpr int kBinThreads = 1024, kBrickThreads = 256;
// A workgroup adds at most this many entries: the further parts of a fuller
// brick are workgroups of their own, which add to the zeroed voxels of the
// brick with device atomics.  Without parts a million vertices in one brick
// take 1.3 ms (the atomics alone 0.38), so 0.06; 1.77M in a sixteenth of a
// 128^3 box 75 us, with parts of 2048 96, of 8192 73, but then 273k 56 instead
// of 51.
constexpr uint32_t kPartEntries = 4096;
// Below this many vertices the launches outweigh the atomics in a small
// volume: 64^3 at 200k vertices 19.7 us against 17.5, at 300k 19.8 against
// 21.9 (128^3: 25.2 against 32.5 and 27.3 against 36.9).
constexpr uint32_t kBinVertices = 250000;
constexpr size_t kBinScratch = kKeptTemporaries;

// Vertices of a block: whole rounds of its threads, at most kBinBlocks blocks.
constexpr uint32_t bin_chunk(uint32_t n_vertices) {
    return uint32_t((uint64_t(n_vertices) + kBinBlocks * kBinThreads - 1u) / (kBinBlocks * kBinThreads)) * kBinThreads;
}
static_assert(bin_chunk(1) == kBinThreads && bin_chunk(0xffffffffu) >= 0xffffffffu / kBinBlocks, "no wrap, no zero");

struct VertexBins {
    VoxelGrid g;
    const float* xyz;
    const float* tangents;
    uint32_t n_vertices, chunk;      // vertices of one block
    uint32_t bx, by, n_bricks, blocks;
    uint32_t* hist;                  // blocks x n_bricks: counts, then the vertices of the blocks before
    uint32_t* total;                 // per brick
    uint32_t* start;                 // n_bricks + 1: the bricks' first entries
    uint32_t* more;                  // n_bricks + 1: the further parts of the bricks before
    uint32_t more_blocks;            // further parts at most
    unsigned long long* entries;     // local voxel (9 bits) and tangent (18 bits per component)
    uint32_t* counts;                // nullable
    uint4* acc;
};

// The parts of a brick past its first.
__device__ __forceinline__ uint32_t further_parts(uint32_t entries) {
    return entries > kPartEntries ? (entries - 1u) / kPartEntries : 0u;
}

// Calls voxel(i, v) for the brick's voxels inside the volume: i in the brick
// (a thread's 512 / kThreads of them), v in the volume.
template <int kThreads, typename Voxel>
__device__ __forceinline__ void brick_voxels(const VertexBins& a, uint32_t brick, Voxel voxel) {
    const uint32_t ox = 8u * (brick % a.bx), oy = 8u * (brick / a.bx % a.by), oz = 8u * (brick / (a.bx * a.by));
    for (uint32_t i = threadIdx.x; i < 512u; i += kThreads) {
        const uint32_t x = ox + (i & 7u), y = oy + ((i >> 3) & 7u), z = oz + (i >> 6);
        if (x < a.g.nx && y < a.g.ny && z < a.g.nz) voxel(i, x + size_t(a.g.nx) * (y + size_t(a.g.ny) * z));
    }
}

__device__ __forceinline__ uint32_t vertex_brick(const VertexBins& a, uint3 c) {
    return (c.x >> 3) + a.bx * ((c.y >> 3) + a.by * (c.z >> 3));
}

__global__ void __launch_bounds__(kBinThreads) vertex_hist_kernel(VertexBins a) {
    extern __shared__ uint32_t hist[];
    for (uint32_t i = threadIdx.x; i < a.n_bricks; i += kBinThreads) hist[i] = 0u;
    __syncthreads();
    const uint32_t first = blockIdx.x * a.chunk, end = min(first + a.chunk, a.n_vertices);
#pragma unroll 4
    for (uint32_t i = first + threadIdx.x; i < end; i += kBinThreads)
        atomicAdd(&hist[vertex_brick(a, vertex_voxel(a.g, load_xyz(a.xyz, i)))], 1u);
    __syncthreads();
    uint32_t* row = a.hist + size_t(blockIdx.x) * a.n_bricks;
    for (uint32_t i = threadIdx.x; i < a.n_bricks; i += kBinThreads) row[i] = hist[i];
}

// 64 columns of the histogram per block, 16 groups of at most 16 rows.
__global__ void __launch_bounds__(kBinThreads) vertex_columns_kernel(VertexBins a) {
    constexpr uint32_t kGroups = kBinThreads / kWave, kRows = kBinBlocks / kGroups;
    __shared__ uint32_t sums[kGroups][kWave];
    const uint32_t lane = threadIdx.x % kWave, group = threadIdx.x / kWave;
    const uint32_t col = blockIdx.x * kWave + lane;
    uint32_t v[kRows], sum = 0;
#pragma unroll
    for (uint32_t r = 0; r < kRows; ++r) {
        const uint32_t row = group * kRows + r;
        v[r] = col < a.n_bricks && row < a.blocks ? a.hist[size_t(row) * a.n_bricks + col] : 0u;
    }
#pragma unroll
    for (uint32_t r = 0; r < kRows; ++r) sum += v[r];
    sums[group][lane] = sum;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t g = 0; g < group; ++g) before += sums[g][lane];
    if (group == kGroups - 1 && col < a.n_bricks) a.total[col] = before + sum;
#pragma unroll
    for (uint32_t r = 0; r < kRows; ++r) {
        const uint32_t row = group * kRows + r;
        if (col < a.n_bricks && row < a.blocks) a.hist[size_t(row) * a.n_bricks + col] = before;
        before += v[r];
    }
}

// The sum of v over the block's threads before this one.  All of them call it.
__device__ __forceinline__ uint32_t block_scan(uint32_t* wave_sums, uint32_t v) {
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    uint32_t scan = v;
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t below = __shfl_up(scan, o, kWave);
        scan += int(lane) >= o ? below : 0u;
    }
    if (lane == kWave - 1) wave_sums[wave] = scan;
    __syncthreads();
    uint32_t at = scan - v;
    for (uint32_t w = 0; w < wave; ++w) at += wave_sums[w];
    __syncthreads();
    return at;
}

// Every block scans the bricks' totals for itself, which saves a launch; the
// last one, whose vertices are a remainder, writes what the bricks' kernel
// reads of them.
__global__ void __launch_bounds__(kBinThreads) vertex_fill_kernel(VertexBins a) {
    extern __shared__ uint32_t cursor[];
    __shared__ uint32_t wave_sums[kBinThreads / kWave];
    // the block's share of the bricks in parts (a vertex chunk is under two of n / kBinBlocks: half as many blocks at least)
    __shared__ uint32_t parted[2u * kBinBricks / kBinBlocks], n_parted;
    constexpr uint32_t kPer = kBinBricks / kBinThreads;
    if (threadIdx.x == 0) n_parted = 0u;
    const bool last = blockIdx.x == gridDim.x - 1u;
    for (uint32_t i = threadIdx.x; i < a.n_bricks; i += kBinThreads) cursor[i] = a.total[i];
    __syncthreads();
    const uint32_t per = (a.n_bricks + kBinThreads - 1u) / kBinThreads, i0 = threadIdx.x * per;
    uint32_t v[kPer], sum = 0;
#pragma unroll
    for (uint32_t c = 0; c < kPer; ++c) {
        v[c] = c < per && i0 + c < a.n_bricks ? cursor[i0 + c] : 0u;
        sum += v[c];
    }
    uint32_t at = block_scan(wave_sums, sum);
#pragma unroll
    for (uint32_t c = 0; c < kPer; ++c) {
        if (c < per && i0 + c < a.n_bricks) {
            cursor[i0 + c] = at;
            if (v[c] > kPartEntries && (i0 + c) % gridDim.x == blockIdx.x) parted[atomicAdd(&n_parted, 1u)] = i0 + c;
        }
        at += v[c];
    }
    if (last) {   // workgroup-uniform
        sum = 0;
#pragma unroll
        for (uint32_t c = 0; c < kPer; ++c) sum += further_parts(v[c]);
        at = block_scan(wave_sums, sum);
#pragma unroll
        for (uint32_t c = 0; c < kPer; ++c) {
            if (c < per && i0 + c < a.n_bricks) a.more[i0 + c] = at;
            at += further_parts(v[c]);
        }
        if (threadIdx.x == kBinThreads - 1u) a.more[a.n_bricks] = at;
    }
    __syncthreads();
    for (uint32_t b = 0; b < n_parted; ++b)
        brick_voxels<kBinThreads>(a, parted[b], [&](uint32_t, size_t voxel) {
            a.acc[voxel] = make_uint4(0u, 0u, 0u, 0u);
            if (a.counts) a.counts[voxel] = 0u;
        });
    const uint32_t* row = a.hist + size_t(blockIdx.x) * a.n_bricks;
    for (uint32_t i = threadIdx.x; i < a.n_bricks; i += kBinThreads) {
        if (last) a.start[i] = cursor[i];
        cursor[i] += row[i];
    }
    if (last && threadIdx.x == 0) a.start[a.n_bricks] = a.n_vertices;
    __syncthreads();
    const uint32_t first = blockIdx.x * a.chunk, end = min(first + a.chunk, a.n_vertices);
#pragma unroll 4
    for (uint32_t i = first + threadIdx.x; i < end; i += kBinThreads) {
        const uint3 c = vertex_voxel(a.g, load_xyz(a.xyz, i));
        const float3 t = load_xyz(a.tangents, i);
        const unsigned long long local = (c.x & 7u) + 8u * ((c.y & 7u) + 8u * (c.z & 7u));
        const unsigned long long x = (unsigned long long)(tangent_fixed(t.x) + 65536),
                                 y = (unsigned long long)(tangent_fixed(t.y) + 65536),
                                 z = (unsigned long long)(tangent_fixed(t.z) + 65536);
        a.entries[atomicAdd(&cursor[vertex_brick(a, c)], 1u)] = local | x << 9 | y << 27 | z << 45;
    }
}

// One part of a brick per workgroup: the further parts, then the first ones.
__global__ void __launch_bounds__(kBrickThreads) vertex_brick_kernel(VertexBins a) {
    __shared__ unsigned long long words[512][2];
    __shared__ uint32_t group, found;
    uint32_t brick = blockIdx.x - a.more_blocks, part = 0u;
    if (blockIdx.x < a.more_blocks) {   // workgroup-uniform
        if (blockIdx.x >= a.more[a.n_bricks]) return;
        // the brick whose further parts hold this one: a group of bricks per thread, then a brick
        const uint32_t per = (a.n_bricks + kBrickThreads - 1u) / kBrickThreads;
        const uint32_t i = threadIdx.x * per;
        if (i < a.n_bricks && a.more[i] <= blockIdx.x && blockIdx.x < a.more[min(i + per, a.n_bricks)]) group = i;
        __syncthreads();
        const uint32_t b = group + threadIdx.x;
        if (threadIdx.x < per && b < a.n_bricks && a.more[b] <= blockIdx.x && blockIdx.x < a.more[b + 1u]) found = b;
        __syncthreads();
        brick = found;
        part = blockIdx.x - a.more[brick] + 1u;
    }
    const uint32_t begin = a.start[brick] + part * kPartEntries, last = a.start[brick + 1u];
    const uint32_t end = min(begin + kPartEntries, last);
    const bool whole = part == 0u && end == last;
    for (uint32_t i = threadIdx.x; i < 512u; i += kBrickThreads) words[i][0] = words[i][1] = 0ull;
    __syncthreads();
#pragma unroll 2
    for (uint32_t e = begin + threadIdx.x; e < end; e += kBrickThreads) {
        const unsigned long long w = a.entries[e];
        const long long x = (long long)((w >> 9) & 0x3ffffull) - 65536, y = (long long)((w >> 27) & 0x3ffffull) - 65536,
                        z = (long long)((w >> 45) & 0x3ffffull) - 65536;
        atomicAdd(&words[w & 511u][0], (unsigned long long)(x) * (1ull << 32) + (unsigned long long)(y));
        atomicAdd(&words[w & 511u][1], (unsigned long long)(z) * (1ull << 32) + 1ull);
    }
    __syncthreads();
    brick_voxels<kBrickThreads>(a, brick, [&](uint32_t i, size_t v) {
        const unsigned long long w0 = words[i][0], w1 = words[i][1];
        if (whole) {
            a.acc[v] = make_uint4(uint32_t(w0), uint32_t(w0 >> 32), uint32_t(w1), uint32_t(w1 >> 32));
            if (a.counts) a.counts[v] = uint32_t(w1);
        } else if (uint32_t(w1) != 0u) {   // its count in this part
            unsigned long long* sums = reinterpret_cast<unsigned long long*>(a.acc + v);
            atomicAdd(&sums[0], w0);
            atomicAdd(&sums[1], w1);
            if (a.counts) atomicAdd(&a.counts[v], uint32_t(w1));
        }
    });
}

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// The binned voxelization when the rule above takes it (*taken).  Not under
// capture (a graph must not depend on memory that the library may give back)
// nor where the memory for the bins cannot be had: the atomics need none.
int voxelize_vertices_binned(const float* xyz, uint32_t n_vertices, const float* tangents, const VoxelGrid& g,
                             uint32_t* counts, int64_t* acc, hipStream_t s, bool* taken) {
    *taken = false;
    VertexBins a{};
    a.bx = (g.nx + 7u) >> 3;
    a.by = (g.ny + 7u) >> 3;
    a.n_bricks = a.bx * a.by * ((g.nz + 7u) >> 3);
    if (n_vertices < kBinVertices || a.n_bricks > kBinBricks || reinterpret_cast<uintptr_t>(acc) % 16 != 0)
        return VKHR_OK;
    a.chunk = bin_chunk(n_vertices);
    a.blocks = (n_vertices - 1u) / a.chunk + 1u;
    const size_t hist = align256(size_t(a.blocks) * a.n_bricks * 4), total = align256(size_t(a.n_bricks) * 4),
                 start = align256((size_t(a.n_bricks) + 1) * 4);
    const size_t bytes = hist + total + 2 * start + size_t(n_vertices) * 8;
    if (bytes > kBinScratch || capturing(s)) return VKHR_OK;
    const CallScratch temporaries(bytes, s);
    if (!temporaries.get()) return VKHR_OK;
    char* p = static_cast<char*>(temporaries.get());
    a.g = g;
    a.xyz = xyz;
    a.tangents = tangents;
    a.n_vertices = n_vertices;
    a.hist = reinterpret_cast<uint32_t*>(p);
    a.total = reinterpret_cast<uint32_t*>(p + hist);
    a.start = reinterpret_cast<uint32_t*>(p + hist + total);
    a.more = reinterpret_cast<uint32_t*>(p + hist + total + start);
    a.entries = reinterpret_cast<unsigned long long*>(p + hist + total + 2 * start);
    a.more_blocks = n_vertices / kPartEntries;
    a.counts = counts;
    a.acc = reinterpret_cast<uint4*>(acc);
    const size_t lds = size_t(a.n_bricks) * 4;
    vertex_hist_kernel<<<a.blocks, kBinThreads, lds, s>>>(a);
    VKHR_CHECK_LAUNCH();
    vertex_columns_kernel<<<(a.n_bricks + kWave - 1) / kWave, kBinThreads, 0, s>>>(a);
    VKHR_CHECK_LAUNCH();
    vertex_fill_kernel<<<a.blocks, kBinThreads, lds, s>>>(a);
    VKHR_CHECK_LAUNCH();
    vertex_brick_kernel<<<a.more_blocks + a.n_bricks, kBrickThreads, 0, s>>>(a);
    VKHR_CHECK_LAUNCH();
    *taken = true;
    return VKHR_OK;
}

// Zeroes what the voxelizer accumulates into: the packed accumulator when
// there is one (the counts are unpacked from it afterwards if asked for),
// else the counts.
int clear_targets(uint32_t* counts, int64_t* acc, size_t n, hipStream_t s) {
    return acc ? fill_u32(reinterpret_cast<uint32_t*>(acc), 4 * n, 0u, s) : fill_u32(counts, n, 0u, s);
}

int unpack_counts(uint32_t* counts, const int64_t* acc, size_t n, hipStream_t s) {
    if (!acc || !counts) return VKHR_OK;
    unpack_counts_kernel<<<grid_for(n, 256, 8192), 256, 0, s>>>(reinterpret_cast<const long long*>(acc), counts, n);
    VKHR_CHECK_LAUNCH();
    return VKHR_OK;
}

}  // namespace
}  // namespace vkhr

using namespace vkhr;

extern "C" int vkhr_voxelize_vertices(const float* xyz, uint32_t n_vertices, const float* tangents,
                                      const vkhr_aabb* bounds, uint32_t nx, uint32_t ny, uint32_t nz,
                                      uint32_t* counts, int64_t* tangent_acc, vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    VoxelGrid g;
    if ((rc = make_grid(bounds, nx, ny, nz, &g))) return rc;
    VKHR_REQUIRE(counts || tangent_acc, VKHR_ERR_INVALID, "neither counts nor tangent_acc");
    VKHR_REQUIRE(n_vertices == 0 || xyz, VKHR_ERR_INVALID, "xyz is null");
    VKHR_REQUIRE(!tangent_acc || tangents, VKHR_ERR_INVALID, "tangent_acc needs tangents");
    hipStream_t s = as_stream(stream);
    size_t n = size_t(nx) * ny * nz;
    if (tangent_acc) {
        bool taken = false;
        rc = voxelize_vertices_binned(xyz, n_vertices, tangents, g, counts, tangent_acc, s, &taken);
        if (rc || taken) return rc;
    }
    if ((rc = clear_targets(counts, tangent_acc, n, s))) return rc;
    if (n_vertices) {
        voxelize_vertices_kernel<<<grid_for(n_vertices, 256, 65536), 256, 0, s>>>(
            xyz, n_vertices, tangents, g, counts, reinterpret_cast<long long*>(tangent_acc));
        VKHR_CHECK_LAUNCH();
    }
    return unpack_counts(counts, tangent_acc, n, s);
}

extern "C" int vkhr_voxelize_segments(const float* xyz, uint32_t n_vertices, const uint32_t* indices,
                                      uint32_t n_indices, const float* tangents, const vkhr_aabb* bounds,
                                      uint32_t nx, uint32_t ny, uint32_t nz, uint32_t* counts,
                                      int64_t* tangent_acc, vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    VoxelGrid g;
    if ((rc = make_grid(bounds, nx, ny, nz, &g))) return rc;
    VKHR_REQUIRE(counts || tangent_acc, VKHR_ERR_INVALID, "neither counts nor tangent_acc");
    uint32_t n_pairs = n_indices / 2;  // the reference loops while i < size-1
    VKHR_REQUIRE(n_pairs == 0 || (xyz && indices && n_vertices), VKHR_ERR_INVALID, "xyz/indices is null");
    VKHR_REQUIRE(!tangent_acc || tangents, VKHR_ERR_INVALID, "tangent_acc needs tangents");
    hipStream_t s = as_stream(stream);
    size_t n = size_t(nx) * ny * nz;
    if ((rc = clear_targets(counts, tangent_acc, n, s))) return rc;
    if (n_pairs) {
        voxelize_segments_kernel<<<grid_for(n_pairs, 256, 65536), 256, 0, s>>>(
            xyz, n_vertices, indices, n_pairs, tangents, g, counts, reinterpret_cast<long long*>(tangent_acc));
        VKHR_CHECK_LAUNCH();
    }
    return unpack_counts(counts, tangent_acc, n, s);
}
