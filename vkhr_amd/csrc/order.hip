// Load-time spatial orders of a style's segments: the index pairs sorted by
// the Morton code of each segment's midpoint (vkhr_sort_segments), or
// strand by strand with the strands sorted by the Morton code of their
// root vertex (vkhr_sort_strands).  No counterpart in the
// reference, whose .hair assets store strands in scalp order; a seeded
// synthetic style roots its strands in random order, and the strand passes
// then gather their shadow, density and depth taps from all over the volume
// within one workgroup.  The output is a permutation of the pairs, so the
// voxel counts, fragments and shadow depths are the same on it.
// Compiled with -ffp-contract=off: the codes are reproducible from float
// arithmetic alone (midpoint, offset, scale, truncation).
#include "common.hpp"

#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>

namespace vkhr {
namespace {

constexpr uint32_t kInvalidCode = 1u << 30;  // above every 30-bit code: malformed pairs sort last

// 10 bits of v spread to every third bit.
__device__ __forceinline__ uint32_t spread10(uint32_t v) {
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

__global__ void __launch_bounds__(256)
segment_codes_kernel(const float* __restrict__ xyz, uint32_t n_vertices, const uint32_t* __restrict__ indices,
                     uint32_t n, vkhr_aabb box, uint32_t* __restrict__ keys, uint32_t* __restrict__ values) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t ia = indices[2ull * k], ib = indices[2ull * k + 1];
    uint32_t code = kInvalidCode;
    if (ia < n_vertices && ib < n_vertices) {
        const float3 a = load_xyz(xyz, ia), b = load_xyz(xyz, ib);
        const float m[3] = {0.5f * (a.x + b.x), 0.5f * (a.y + b.y), 0.5f * (a.z + b.z)};
        uint32_t q[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float ext = box.size[c];
            float f = ext > 0.0f ? (m[c] - box.origin[c]) / ext * 1024.0f : 0.0f;
            f = fminf(fmaxf(f, 0.0f), 1023.0f);  // NaN becomes 0
            q[c] = uint32_t(f);
        }
        code = (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
    }
    keys[k] = code;
    values[k] = k;
}

// --- vkhr_sort_strands ------------------------------------------------------
// A strand keeps its pairs in order, so the strands are sorted and not the
// pairs: one (code, run) per run of pairs, a twelfth of the pairs on ordinary
// hair, in four stable counting passes of 8 bits over the 31-bit codes.  All
// of it runs on device-side counts (no run count is read back); the stages
// are small, and what bounds them is their launches and load latencies.
// Measured: 136k strands / 1.6M pairs
// 222 us of kernels and 130 of host before (a library sort of the pairs, its
// temporaries allocated and freed), 88 of kernels now; 2k strands / 22k
// pairs 45 us in 11 launches before, 34 in 4 now.
//
// In every stage a block owns one contiguous chunk, in tiles of 4096 pairs or
// 2048 runs, consecutive ones in each wave.
constexpr int kOrderBlock = 1024, kOrderWaves = kOrderBlock / kWave, kOrderItems = 4;
constexpr uint32_t kOrderTile = kOrderBlock * kOrderItems;   // pairs
// Runs per thread in a tile of the launches' passes.  Two keep enough
// workgroups sorting: with 136k strands in tiles of 4096 there are 34, a
// scatter taking 10.6 us against 8.0; eight were no faster at 12M runs.
constexpr int kSortItems = 2;
constexpr uint32_t kSortTile = kOrderBlock * kSortItems;
constexpr int kDigits = 256, kPasses = 4;
// Blocks at most: a block adds up the rows of every block before its own.
constexpr uint32_t kMaxRunBlocks = 2048, kMaxSortBlocks = 512;
// Up to this many pairs one workgroup runs the stages over the runs in one
// launch instead of ten: 17 us for 2k strands / 22k pairs, 52 in launches of
// their own.  It holds kTileRuns runs, in LDS; the host, which waits for the
// result anyway, reads the run count with it and starts the launches when
// there were more.  Workgroup against launches, pairs that are a run each (us
// of the call): 4096 63 / 102, 5000 69 / 107, 10000 96 / 107, 15000 123 / 107.
constexpr uint32_t kOneBlockPairs = 32768, kTileRuns = 10240;
// Up to this many pairs that workgroup runs every stage (1000 pairs 43 -> 39 us)
constexpr uint32_t kWholePairs = kOrderTile;

struct OrderArgs {
    const float* xyz;
    const uint32_t* indices;    // n pairs
    uint32_t n_vertices, n;
    uint32_t run_blocks, run_chunk;   // blocks over the pairs, pairs of one block
    uint32_t sort_blocks;             // blocks over the runs at most
    vkhr_aabb box;
    uint32_t* counts;           // run_blocks: heads in the block's pairs
    uint32_t* run_base;         // run_blocks: the runs that start before the block's pairs
    uint32_t* hist;             // sort_blocks x 256; then the blocks' pair sums
    uint32_t* total;            // the runs
    uint32_t* host_total;       // the same for the host (nullable)
    uint32_t* start;            // total + 1: first pair of each run
    uint32_t* keys[2];
    uint32_t* runs[2];
    uint32_t* delta;            // output minus input position of a run's pairs (keys[0], free by then)
    uint32_t* sorted;
};

struct OrderLds {
    uint32_t counts[kOrderWaves][kDigits];
    uint32_t base[kDigits];
    uint32_t wave[kOrderWaves];
};

// The sum of v over the block, and of v over the lanes' waves before this one.
__device__ __forceinline__ uint32_t block_sum(OrderLds& lds, uint32_t v, uint32_t* before = nullptr) {
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    const int wave = threadIdx.x / kWave;
    __syncthreads();
    if (threadIdx.x % kWave == 0) lds.wave[wave] = v;
    __syncthreads();
    uint32_t sum = 0, prior = 0;
#pragma unroll
    for (int w = 0; w < kOrderWaves; ++w) {
        const uint32_t x = lds.wave[w];
        sum += x;
        prior += w < wave ? x : 0u;
    }
    if (before) *before = prior;
    return sum;
}

// The r-th of a lane's `per` items in a tile.
__device__ __forceinline__ uint32_t wave_item(uint32_t tile, int r, uint32_t per = kOrderItems) {
    return tile + ((threadIdx.x / kWave) * per + uint32_t(r)) * kWave + threadIdx.x % kWave;
}

__device__ __forceinline__ uint32_t lanes_below(unsigned long long mask) {
    return uint32_t(__popcll(mask & ((1ull << (threadIdx.x % kWave)) - 1ull)));
}

// Pair k starts a run: its first index is not the previous pair's second.
__device__ __forceinline__ bool run_head(const OrderArgs& a, uint32_t k) {
    return k == 0 || a.indices[2ull * k - 1u] != a.indices[2ull * k];
}

// The runs of one sort block; false when it has none.
__device__ __forceinline__ bool sort_range(const OrderArgs& a, uint32_t block, uint32_t& begin, uint32_t& end,
                                           uint32_t& rows) {
    const uint32_t runs = *a.total;
    const uint32_t per = (runs + a.sort_blocks - 1u) / a.sort_blocks;
    const uint32_t chunk = (per + kSortTile - 1u) / kSortTile * kSortTile;
    rows = chunk ? (runs + chunk - 1u) / chunk : 0u;
    begin = block * chunk;
    end = min(begin + chunk, runs);
    return block < rows;
}

__device__ __forceinline__ void count_runs(const OrderArgs& a, OrderLds& lds, uint32_t block) {
    const uint32_t begin = block * a.run_chunk, end = min(begin + a.run_chunk, a.n);
    uint32_t mine = 0;
    for (uint32_t tile = begin; tile < end; tile += kOrderTile)
#pragma unroll
        for (int r = 0; r < kOrderItems; ++r) {
            const uint32_t k = wave_item(tile, r);
            mine += k < end && run_head(a, k) ? 1u : 0u;
        }
    const uint32_t sum = block_sum(lds, mine);
    if (threadIdx.x == 0) a.counts[block] = sum;
}

// Visits the block's pairs a tile at a time: each lane's pairs k, the number
// of runs started up to and with each, and a bit per pair for the heads and
// for those below the end.  Returns the runs up to the block's end.
template <typename Visit>
__device__ __forceinline__ uint32_t walk_runs(const OrderArgs& a, OrderLds& lds, uint32_t block, uint32_t base,
                                              Visit visit) {
    const uint32_t begin = block * a.run_chunk, end = min(begin + a.run_chunk, a.n);
    for (uint32_t tile = begin; tile < end; tile += kOrderTile) {
        unsigned long long heads[kOrderItems];
        uint32_t mine = 0;
#pragma unroll
        for (int r = 0; r < kOrderItems; ++r) {
            const uint32_t k = wave_item(tile, r);
            heads[r] = __ballot(k < end && run_head(a, k));
            mine += uint32_t(__popcll(heads[r]));
        }
        uint32_t before;
        const uint32_t sum = block_sum(lds, threadIdx.x % kWave == 0 ? mine : 0u, &before);
        uint32_t at = base + before, k[kOrderItems], upto[kOrderItems], is_head = 0, valid = 0;
#pragma unroll
        for (int r = 0; r < kOrderItems; ++r) {
            k[r] = wave_item(tile, r);
            const uint32_t head = uint32_t(heads[r] >> (threadIdx.x % kWave)) & 1u;
            is_head |= head << r;
            valid |= (k[r] < end ? 1u : 0u) << r;
            upto[r] = at + lanes_below(heads[r]) + head;
            at += uint32_t(__popcll(heads[r]));
        }
        visit(k, upto, is_head, valid);
        base += sum;
    }
    return base;
}

// The Morton code of a root vertex, as segment_codes_kernel codes a midpoint.
__device__ __forceinline__ uint32_t root_code(const OrderArgs& a, float3 v) {
    const float m[3] = {v.x, v.y, v.z};
    uint32_t q[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float ext = a.box.size[c];
        float f = ext > 0.0f ? (m[c] - a.box.origin[c]) / ext * 1024.0f : 0.0f;
        f = fminf(fmaxf(f, 0.0f), 1023.0f);  // NaN becomes 0
        q[c] = uint32_t(f);
    }
    return (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
}

// Writes the start and the code of the runs that start in the block's pairs.
// The codes are formed here and not by the sort's first pass: the roots'
// vertices lie all over memory, and these blocks are ten times as many.
__device__ __forceinline__ void emit_runs(const OrderArgs& a, OrderLds& lds, uint32_t block) {
    uint32_t mine = 0;
    for (uint32_t i = threadIdx.x; i < block; i += kOrderBlock) mine += a.counts[i];
    const uint32_t base = block_sum(lds, mine);
    if (threadIdx.x == 0) a.run_base[block] = base;
    const uint32_t runs = walk_runs(a, lds, block, base, [&](const uint32_t (&k)[kOrderItems],
                                                             const uint32_t (&upto)[kOrderItems], uint32_t heads,
                                                             uint32_t) {
        uint32_t root[kOrderItems];
        float3 v[kOrderItems];
#pragma unroll
        for (int r = 0; r < kOrderItems; ++r) root[r] = (heads >> r) & 1u ? a.indices[2ull * k[r]] : a.n_vertices;
        if (a.n_vertices) {   // the lanes without a head read vertex 0, so that the loads need no branches
#pragma unroll
            for (int r = 0; r < kOrderItems; ++r) v[r] = load_xyz(a.xyz, root[r] < a.n_vertices ? root[r] : 0u);
        }
#pragma unroll
        for (int r = 0; r < kOrderItems; ++r)
            if ((heads >> r) & 1u) {
                a.start[upto[r] - 1u] = k[r];
                a.keys[0][upto[r] - 1u] = root[r] < a.n_vertices ? root_code(a, v[r]) : kInvalidCode;
            }
    });
    if (block == a.run_blocks - 1u && threadIdx.x == 0) {
        a.start[runs] = a.n;
        *a.total = runs;
        if (a.host_total) *a.host_total = runs;
    }
}

// The block's runs by digit.
__device__ __forceinline__ void count_digits(const OrderArgs& a, OrderLds& lds, uint32_t block, int pass) {
    uint32_t begin, end, rows;
    if (!sort_range(a, block, begin, end, rows)) return;
    uint32_t* hist = lds.base;
    __syncthreads();
    if (threadIdx.x < kDigits) hist[threadIdx.x] = 0u;
    __syncthreads();
    const uint32_t* keys = a.keys[pass & 1];
    for (uint32_t tile = begin; tile < end; tile += kSortTile)
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) {
            const uint32_t i = wave_item(tile, r, kSortItems);
            if (i >= end) continue;
            atomicAdd(&hist[(keys[i] >> (8 * pass)) & (kDigits - 1u)], 1u);
        }
    __syncthreads();
    if (threadIdx.x < kDigits) a.hist[block * kDigits + threadIdx.x] = hist[threadIdx.x];
}

// The rank of each of the tile's first n items among those of its digit
// (the 8 bits of its key from shift on) before it in its wave, and the
// wave's count per digit in lds.counts (0 at the start).
template <int kItems>
__device__ __forceinline__ void rank_digits(OrderLds& lds, const uint32_t (&key)[kItems], int shift, uint32_t n,
                                            uint32_t (&rank)[kItems], uint32_t per = kItems) {
    const int wave = threadIdx.x / kWave;
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        if (uint32_t(r) >= per) break;
        const uint32_t d = (key[r] >> shift) & (kDigits - 1u);
        const bool valid = wave_item(0, r, per) < n;
        unsigned long long same = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const bool one = (d >> bit) & 1u;
            const unsigned long long ones = __ballot(one);
            same &= one ? ones : ~ones;
        }
        const uint32_t below = lanes_below(same), had = lds.counts[wave][d];
        rank[r] = had + below;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (below == 0 && valid) lds.counts[wave][d] = had + uint32_t(__popcll(same));
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// The waves' counts of a digit turned into their first places, from `at` on;
// returns the place after the last wave's.
__device__ __forceinline__ uint32_t stack_waves(OrderLds& lds, uint32_t digit, uint32_t at) {
#pragma unroll
    for (int w = 0; w < kOrderWaves; ++w) {
        const uint32_t c = lds.counts[w][digit];
        lds.counts[w][digit] = at;
        at += c;
    }
    return at;
}

// The exclusive scan over the digits, in the first 256 threads.
__device__ __forceinline__ uint32_t scan_digits(OrderLds& lds, uint32_t all) {
    const int lane = threadIdx.x % kWave;
    uint32_t scan = all;
    for (int o = 1; o < kWave; o <<= 1) {
        const uint32_t below = __shfl_up(scan, o, kWave);
        scan += lane >= o ? below : 0u;
    }
    uint32_t prior;
    block_sum(lds, all, &prior);
    return prior + scan - all;
}

// One stable pass: an item goes to its digit's first place, plus the items
// of its digit in the blocks, tiles and waves before it, plus those in its
// wave before it.
__device__ __forceinline__ void scatter_digits(const OrderArgs& a, OrderLds& lds, uint32_t block, int pass) {
    uint32_t begin, end, rows;
    if (!sort_range(a, block, begin, end, rows)) return;
    const int wave = threadIdx.x / kWave;
    constexpr uint32_t kGroups = kOrderBlock / kDigits;
    const uint32_t digit = threadIdx.x % kDigits, group = threadIdx.x / kDigits;
    {
        uint32_t all = 0, before = 0;
#pragma unroll 8
        for (uint32_t row = group; row < rows; row += kGroups) {
            const uint32_t c = a.hist[row * kDigits + digit];
            all += c;
            before += row < block ? c : 0u;
        }
        __syncthreads();
        lds.counts[group][digit] = all;
        lds.counts[kGroups + group][digit] = before;
        __syncthreads();
        all = before = 0;
        if (threadIdx.x < kDigits)
            for (uint32_t g = 0; g < kGroups; ++g) {
                all += lds.counts[g][digit];
                before += lds.counts[kGroups + g][digit];
            }
        const uint32_t first = scan_digits(lds, all);
        if (threadIdx.x < kDigits) lds.base[digit] = first + before;
    }
    const uint32_t *keys = a.keys[pass & 1], *runs = a.runs[pass & 1];
    uint32_t *keys_out = a.keys[(pass & 1) ^ 1], *runs_out = a.runs[(pass & 1) ^ 1];
    for (uint32_t tile = begin; tile < end; tile += kSortTile) {
        __syncthreads();
        for (uint32_t g = 0; g < kOrderWaves / kGroups; ++g) lds.counts[g * kGroups + group][digit] = 0u;
        uint32_t key[kSortItems], run[kSortItems], rank[kSortItems];
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) {
            const uint32_t i = wave_item(tile, r, kSortItems);
            key[r] = i < end ? keys[i] : 0u;
            run[r] = i < end ? (pass == 0 ? i : runs[i]) : 0u;
        }
        __syncthreads();
        rank_digits(lds, key, 8 * pass, end - tile, rank);
        __syncthreads();
        if (threadIdx.x < kDigits) lds.base[digit] = stack_waves(lds, digit, lds.base[digit]);
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) {
            if (wave_item(tile, r, kSortItems) >= end) continue;
            const uint32_t at = lds.counts[wave][(key[r] >> (8 * pass)) & (kDigits - 1u)] + rank[r];
            if (pass + 1 < kPasses) keys_out[at] = key[r];
            runs_out[at] = run[r];
        }
    }
}

__device__ __forceinline__ uint32_t run_length(const OrderArgs& a, uint32_t run) {
    return a.start[run + 1u] - a.start[run];
}

__device__ __forceinline__ void sum_lengths(const OrderArgs& a, OrderLds& lds, uint32_t block) {
    uint32_t begin, end, rows;
    if (!sort_range(a, block, begin, end, rows)) return;
    uint32_t mine = 0;
    for (uint32_t tile = begin; tile < end; tile += kSortTile) {
        uint32_t run[kSortItems];
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) run[r] = wave_item(tile, r, kSortItems) < end ? a.runs[kPasses & 1][wave_item(tile, r, kSortItems)] : 0u;
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) {
            const uint32_t len = run_length(a, run[r]);
            mine += wave_item(tile, r, kSortItems) < end ? len : 0u;
        }
    }
    const uint32_t sum = block_sum(lds, mine);
    if (threadIdx.x == 0) a.hist[block] = sum;
}

// Where the pairs of a tile's runs go, the tile's first pair going to base:
// the lengths of the runs before each in the order.  Returns the lengths' sum.
template <int kItems>
__device__ __forceinline__ uint32_t tile_deltas(const OrderArgs& a, OrderLds& lds, const uint32_t (&run)[kItems],
                                                uint32_t n, uint32_t base) {
    const int lane = threadIdx.x % kWave;
    uint32_t first[kItems], len[kItems], at[kItems], wave_sum = 0;
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const bool valid = wave_item(0, r, kItems) < n;
        first[r] = a.start[valid ? run[r] : 0u];
        len[r] = a.start[valid ? run[r] + 1u : 0u] - first[r];
        len[r] = valid ? len[r] : 0u;
    }
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        uint32_t scan = len[r];
        for (int o = 1; o < kWave; o <<= 1) {
            const uint32_t below = __shfl_up(scan, o, kWave);
            scan += lane >= o ? below : 0u;
        }
        at[r] = wave_sum + scan - len[r];
        wave_sum += __shfl(scan, kWave - 1, kWave);
    }
    uint32_t before;
    const uint32_t sum = block_sum(lds, lane == 0 ? wave_sum : 0u, &before);
#pragma unroll
    for (int r = 0; r < kItems; ++r)
        if (wave_item(0, r, kItems) < n) a.delta[run[r]] = base + before + at[r] - first[r];
    return sum;
}

__device__ __forceinline__ void run_deltas(const OrderArgs& a, OrderLds& lds, uint32_t block) {
    uint32_t begin, end, rows;
    if (!sort_range(a, block, begin, end, rows)) return;
    uint32_t mine = 0;
    for (uint32_t i = threadIdx.x; i < block; i += kOrderBlock) mine += a.hist[i];
    uint32_t base = block_sum(lds, mine);
    for (uint32_t tile = begin; tile < end; tile += kSortTile) {
        uint32_t run[kSortItems];
#pragma unroll
        for (int r = 0; r < kSortItems; ++r) run[r] = wave_item(tile, r, kSortItems) < end ? a.runs[kPasses & 1][wave_item(tile, r, kSortItems)] : 0u;
        base += tile_deltas(a, lds, run, end - tile, base);
    }
}

// All passes over at most kTileRuns runs: they stay in registers, `per` to a
// lane, and change places through LDS.
constexpr int kTileItems = int(kTileRuns) / kOrderBlock;
struct TileLds {
    uint32_t key[kTileRuns], run[kTileRuns];
};
__device__ __forceinline__ void sort_tile(const OrderArgs& a, OrderLds& lds, TileLds& tile) {
    const uint32_t runs = *a.total, per = (runs + kOrderBlock - 1u) / kOrderBlock;
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const uint32_t digit = threadIdx.x % kDigits;
    uint32_t key[kTileItems], run[kTileItems], rank[kTileItems];
#pragma unroll
    for (int r = 0; r < kTileItems; ++r) {
        run[r] = wave_item(0, r, per);
        key[r] = uint32_t(r) < per && run[r] < runs ? a.keys[0][run[r]] : 0u;
    }
#pragma unroll 1
    for (int pass = 0; pass < kPasses; ++pass) {
        __syncthreads();
        for (uint32_t w = threadIdx.x / kDigits; w < kOrderWaves; w += kOrderBlock / kDigits) lds.counts[w][digit] = 0u;
        __syncthreads();
        rank_digits(lds, key, 8 * pass, runs, rank, per);
        __syncthreads();
        uint32_t all = 0;
        if (threadIdx.x < kDigits) all = stack_waves(lds, digit, 0u);
        const uint32_t first = scan_digits(lds, all);
        if (threadIdx.x < kDigits) lds.base[digit] = first;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kTileItems; ++r) {
            if (uint32_t(r) >= per) break;
            if (wave_item(0, r, per) >= runs) continue;
            const uint32_t d = (key[r] >> (8 * pass)) & (kDigits - 1u);
            const uint32_t at = lds.base[d] + lds.counts[wave][d] + rank[r];
            tile.key[at] = key[r];
            tile.run[at] = run[r];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kTileItems; ++r) {
            if (uint32_t(r) >= per) break;
            if (wave_item(0, r, per) >= runs) continue;
            key[r] = tile.key[wave_item(0, r, per)];
            run[r] = tile.run[wave_item(0, r, per)];
        }
    }
    // where the runs' pairs go: the lengths of the runs before each in the order
    uint32_t mine = 0;
#pragma unroll
    for (int r = 0; r < kTileItems; ++r) {
        if (uint32_t(r) >= per) break;
        rank[r] = wave_item(0, r, per) < runs ? run_length(a, run[r]) : 0u;
        mine += rank[r];
    }
    uint32_t base;
    block_sum(lds, mine, &base);
#pragma unroll
    for (int r = 0; r < kTileItems; ++r) {
        if (uint32_t(r) >= per) break;
        uint32_t scan = rank[r];
        for (int o = 1; o < kWave; o <<= 1) {
            const uint32_t below = __shfl_up(scan, o, kWave);
            scan += lane >= o ? below : 0u;
        }
        if (wave_item(0, r, per) < runs) a.delta[run[r]] = base + scan - rank[r] - a.start[run[r]];
        base += __shfl(scan, kWave - 1, kWave);
    }
}

__device__ __forceinline__ void place_pairs(const OrderArgs& a, OrderLds& lds, uint32_t block) {
    const uint2* pairs = reinterpret_cast<const uint2*>(a.indices);
    uint2* out = reinterpret_cast<uint2*>(a.sorted);
    walk_runs(a, lds, block, a.run_base[block], [&](const uint32_t (&k)[kOrderItems],
                                                    const uint32_t (&upto)[kOrderItems], uint32_t, uint32_t valid) {
        uint32_t delta[kOrderItems];
        uint2 pair[kOrderItems];
#pragma unroll
        for (int r = 0; r < kOrderItems; ++r) {
            const bool v = (valid >> r) & 1u;
            delta[r] = v ? a.delta[upto[r] - 1u] : 0u;
            pair[r] = v ? pairs[k[r]] : make_uint2(0u, 0u);
        }
#pragma unroll
        for (int r = 0; r < kOrderItems; ++r)
            if ((valid >> r) & 1u) out[k[r] + delta[r]] = pair[r];
    });
}

__global__ void __launch_bounds__(kOrderBlock) count_runs_kernel(OrderArgs a) {
    __shared__ OrderLds lds;
    count_runs(a, lds, blockIdx.x);
}
__global__ void __launch_bounds__(kOrderBlock) emit_runs_kernel(OrderArgs a) {
    __shared__ OrderLds lds;
    emit_runs(a, lds, blockIdx.x);
}
__global__ void __launch_bounds__(kOrderBlock) count_digits_kernel(OrderArgs a, int pass) {
    __shared__ OrderLds lds;
    count_digits(a, lds, blockIdx.x, pass);
}
__global__ void __launch_bounds__(kOrderBlock) scatter_digits_kernel(OrderArgs a, int pass) {
    __shared__ OrderLds lds;
    scatter_digits(a, lds, blockIdx.x, pass);
}
__global__ void __launch_bounds__(kOrderBlock) sum_lengths_kernel(OrderArgs a) {
    __shared__ OrderLds lds;
    sum_lengths(a, lds, blockIdx.x);
}
__global__ void __launch_bounds__(kOrderBlock) run_deltas_kernel(OrderArgs a) {
    __shared__ OrderLds lds;
    run_deltas(a, lds, blockIdx.x);
}
__global__ void __launch_bounds__(kOrderBlock) place_pairs_kernel(OrderArgs a, uint32_t most_runs) {
    __shared__ OrderLds lds;
    if (*a.total <= most_runs) place_pairs(a, lds, blockIdx.x);
}

// The stages between the runs' emission and the placing of the pairs by one
// workgroup, when a tile holds the runs.
__global__ void __launch_bounds__(kOrderBlock) order_tile_kernel(OrderArgs a) {
    __shared__ OrderLds lds;
    __shared__ TileLds tile;
    if (*a.total <= kTileRuns) sort_tile(a, lds, tile);
}

// Every stage by one workgroup, which owns all pairs.
__global__ void __launch_bounds__(kOrderBlock) order_whole_kernel(OrderArgs a) {
    __shared__ OrderLds lds;
    __shared__ TileLds tile;
    emit_runs(a, lds, 0u);   // (the first block's runs need no count)
    __syncthreads();
    sort_tile(a, lds, tile);
    __syncthreads();
    place_pairs(a, lds, 0u);
}

// The stages over more runs in launches of their own.
void launch_passes(const OrderArgs& a, hipStream_t s) {
    for (int pass = 0; pass < kPasses; ++pass) {
        count_digits_kernel<<<a.sort_blocks, kOrderBlock, 0, s>>>(a, pass);
        scatter_digits_kernel<<<a.sort_blocks, kOrderBlock, 0, s>>>(a, pass);
    }
    sum_lengths_kernel<<<a.sort_blocks, kOrderBlock, 0, s>>>(a);
    run_deltas_kernel<<<a.sort_blocks, kOrderBlock, 0, s>>>(a);
}

__global__ void __launch_bounds__(256)
gather_pairs_kernel(const uint2* __restrict__ pairs, const uint32_t* __restrict__ order, uint32_t n,
                    uint2* __restrict__ out) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) out[k] = pairs[order[k]];
}

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// Checks shared by the two orders; n_out: the pair count.
int check_order_args(const float* xyz, const uint32_t* indices, uint32_t n_indices, const vkhr_aabb* bounds,
                     const uint32_t* sorted, uint32_t* n_out) {
    VKHR_REQUIRE(bounds && sorted, VKHR_ERR_INVALID, "null argument");
    VKHR_REQUIRE(n_indices % 2 == 0, VKHR_ERR_INVALID, "odd index count %u", n_indices);
    const uint32_t n = n_indices / 2;
    *n_out = n;
    if (n == 0) return VKHR_OK;
    VKHR_REQUIRE(n <= (1u << 28), VKHR_ERR_OVERFLOW, "too many segments (%u)", n);  // one lane per pair
    const auto plausible = [](const void* p) { return reinterpret_cast<uintptr_t>(p) >= 65536u; };
    VKHR_REQUIRE(plausible(xyz) && plausible(indices) && plausible(sorted), VKHR_ERR_INVALID,
                 "null or implausible pointer");
    VKHR_REQUIRE(reinterpret_cast<uintptr_t>(indices) % 8 == 0 && reinterpret_cast<uintptr_t>(sorted) % 8 == 0,
                 VKHR_ERR_INVALID, "index buffers must be 8-byte aligned");
    const uintptr_t in0 = reinterpret_cast<uintptr_t>(indices), out0 = reinterpret_cast<uintptr_t>(sorted);
    const uintptr_t bytes = uintptr_t(n) * 8u;
    VKHR_REQUIRE(in0 + bytes <= out0 || out0 + bytes <= in0, VKHR_ERR_INVALID, "indices and sorted overlap");
    return VKHR_OK;
}

}  // namespace
}  // namespace vkhr

using namespace vkhr;

extern "C" int vkhr_sort_segments(const float* xyz, uint32_t n_vertices, const uint32_t* indices,
                                  uint32_t n_indices, const vkhr_aabb* bounds, uint32_t* sorted,
                                  vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    uint32_t n = 0;
    if ((rc = check_order_args(xyz, indices, n_indices, bounds, sorted, &n)) || n == 0) return rc;
    hipStream_t s = as_stream(stream);
    size_t sort_bytes = 0;
    VKHR_CHECK_HIP(rocprim::radix_sort_pairs(nullptr, sort_bytes, static_cast<uint32_t*>(nullptr),
                                             static_cast<uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr),
                                             static_cast<uint32_t*>(nullptr), size_t(n), 0, 31, s));
    const size_t words = align256(size_t(n) * 4);
    void* tmp = nullptr;
    VKHR_CHECK_HIP(hipMalloc(&tmp, 4 * words + align256(sort_bytes)));
    char* p = static_cast<char*>(tmp);
    uint32_t* keys = reinterpret_cast<uint32_t*>(p);
    uint32_t* values = reinterpret_cast<uint32_t*>(p + words);
    uint32_t* keys_sorted = reinterpret_cast<uint32_t*>(p + 2 * words);
    uint32_t* order = reinterpret_cast<uint32_t*>(p + 3 * words);
    void* sort_tmp = p + 4 * words;
    const uint32_t blocks = grid_for(n, 256);
    segment_codes_kernel<<<blocks, 256, 0, s>>>(xyz, n_vertices, indices, n, *bounds, keys, values);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = rocprim::radix_sort_pairs(sort_tmp, sort_bytes, keys, keys_sorted, values, order, size_t(n), 0, 31, s);
    if (e == hipSuccess) {
        gather_pairs_kernel<<<blocks, 256, 0, s>>>(reinterpret_cast<const uint2*>(indices), order, n,
                                                   reinterpret_cast<uint2*>(sorted));
        e = hipGetLastError();
    }
    const hipError_t se = hipStreamSynchronize(s);  // the temporaries are freed below
    (void)hipFree(tmp);
    if (e == hipSuccess) e = se;
    VKHR_REQUIRE(e == hipSuccess, VKHR_ERR_HIP, "segment sort failed: %s", hipGetErrorString(e));
    return VKHR_OK;
}

extern "C" int vkhr_sort_strands(const float* xyz, uint32_t n_vertices, const uint32_t* indices, uint32_t n_indices,
                                 const vkhr_aabb* bounds, uint32_t* sorted, vkhr_stream stream) {
    clear_error();
    int rc = ensure_device();
    if (rc) return rc;
    uint32_t n = 0;
    if ((rc = check_order_args(xyz, indices, n_indices, bounds, sorted, &n)) || n == 0) return rc;
    hipStream_t s = as_stream(stream);
    VKHR_REQUIRE(!capturing(s), VKHR_ERR_HIP,
                 "strand sort failed: it synchronises the stream, which is being captured");
    const RelaxedCapture relaxed;   // (it waits for the stream)
    OrderArgs a{};
    a.xyz = xyz;
    a.indices = indices;
    a.n_vertices = n_vertices;
    a.n = n;
    a.box = *bounds;
    a.sorted = sorted;
    const bool whole = n <= kWholePairs, one = n <= kOneBlockPairs;
    a.run_blocks = whole ? 1u : std::min((n + kOrderTile - 1u) / kOrderTile, kMaxRunBlocks);
    a.run_chunk = ((n + a.run_blocks - 1u) / a.run_blocks + kOrderTile - 1u) / kOrderTile * kOrderTile;
    a.run_blocks = (n + a.run_chunk - 1u) / a.run_chunk;   // none empty
    a.sort_blocks = std::min((n + kSortTile - 1u) / kSortTile, kMaxSortBlocks);
    // Every pair may be a run of its own.
    const size_t words = align256((size_t(n) + 1) * 4);
    const size_t counts = align256(size_t(a.run_blocks) * 4), hist = align256(size_t(a.sort_blocks) * kDigits * 4);
    const size_t bytes = 5 * words + 2 * counts + hist + 256;
    const CallScratch temporaries(bytes, s);
    VKHR_REQUIRE(temporaries.get(), VKHR_ERR_HIP, "strand sort failed: no memory for %zu bytes of temporaries", bytes);
    char* p = static_cast<char*>(temporaries.get());
    const auto take = [&p](size_t b) {
        uint32_t* at = reinterpret_cast<uint32_t*>(p);
        p += b;
        return at;
    };
    a.start = take(words);
    a.keys[0] = take(words);
    a.keys[1] = take(words);
    a.runs[0] = take(words);
    a.runs[1] = take(words);
    a.counts = take(counts);
    a.run_base = take(counts);
    a.hist = take(hist);
    a.total = take(256);
    a.delta = a.keys[0];
    HostWords host;
    a.host_total = host.words();
    uint32_t runs = 0;
    if (whole) {
        order_whole_kernel<<<1, kOrderBlock, 0, s>>>(a);
    } else {
        count_runs_kernel<<<a.run_blocks, kOrderBlock, 0, s>>>(a);
        emit_runs_kernel<<<a.run_blocks, kOrderBlock, 0, s>>>(a);
    }
    if (one && !whole) {
        order_tile_kernel<<<1, kOrderBlock, 0, s>>>(a);
        place_pairs_kernel<<<a.run_blocks, kOrderBlock, 0, s>>>(a, kTileRuns);
        if (n > kTileRuns) {
            hipError_t c = hipSuccess;
            if (!host.words()) c = hipMemcpyAsync(&runs, a.total, sizeof(runs), hipMemcpyDeviceToHost, s);
            if (c == hipSuccess) c = hipStreamSynchronize(s);
            if (host.words()) runs = *host.words();
            VKHR_CHECK_HIP(c);
        }
    }
    if (!one || runs > kTileRuns) {
        launch_passes(a, s);
        place_pairs_kernel<<<a.run_blocks, kOrderBlock, 0, s>>>(a, n);
    }
    hipError_t e = hipGetLastError();
    const hipError_t se = hipStreamSynchronize(s);
    if (e == hipSuccess) e = se;
    VKHR_REQUIRE(e == hipSuccess, VKHR_ERR_HIP, "strand sort failed: %s", hipGetErrorString(e));
    return VKHR_OK;
}
