// Library state: thread-local error messages, device checks, the scratch
// areas (one per device and stream), and the generic fill kernel.
#include "common.hpp"

#include <cstdarg>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <thread>
#include <tuple>
#include <utility>
#include <vector>

namespace vkhr {

namespace {
thread_local char g_error[512] = {0};

constexpr int kMaxDevices = 64;
std::mutex g_mutex;
bool g_checked[kMaxDevices] = {false};
struct Block {
    void* ptr = nullptr;
    size_t bytes = 0;
};
struct Scratch {
    void* ptr = nullptr;
    size_t bytes = 0;
    Block call;  // what a CallScratch takes out and puts back
    std::vector<void*> retired;  // outgrown buffers still owned by work captured into a graph
};
// (device, stream, thread) -> area.  The thread is part of the key only for
// hipStreamPerThread, one handle value that names a different stream on
// every thread.
using ScratchKey = std::tuple<int, hipStream_t, size_t>;
std::map<ScratchKey, Scratch> g_scratch;

// The page of HostWords: 64 slots of 64 bytes, a bit per slot in use.
constexpr size_t kHostSlot = 64, kHostSlots = 64;
char* g_host_page = nullptr;
uint64_t g_host_used = 0;

Block g_kept[kMaxDevices];

// The fixed scratch of the allocation-free entry points: one copy per
// device, resident from module load until the process ends.  Host code
// never passes `scratch` itself (its host-side name is not a device
// address); ensure_device looks up each device's copy once, with that
// device current, and keeps the address in g_static_scratch.
static __device__ __align__(256) uint32_t scratch[kStaticScratchBytes / sizeof(uint32_t)];
void* g_static_scratch[kMaxDevices] = {nullptr};

ScratchKey scratch_key(int dev, hipStream_t stream) {
    const size_t thread = stream == hipStreamPerThread ? std::hash<std::thread::id>()(std::this_thread::get_id()) : 0;
    return ScratchKey(dev, stream, thread);
}
}  // namespace

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_error, sizeof(g_error), fmt, ap);
    va_end(ap);
}

void clear_error() { g_error[0] = '\0'; }

int ensure_device() {
    int dev = 0;
    VKHR_CHECK_HIP(hipGetDevice(&dev));
    VKHR_REQUIRE(dev >= 0 && dev < kMaxDevices, VKHR_ERR_NO_DEVICE, "device index %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_mutex);
    if (g_checked[dev]) return VKHR_OK;
    hipDeviceProp_t prop;
    VKHR_CHECK_HIP(hipGetDeviceProperties(&prop, dev));
    VKHR_REQUIRE(std::strncmp(prop.gcnArchName, "gfx950", 6) == 0, VKHR_ERR_NO_DEVICE,
                 "device %d is %s; this library is built for gfx950 only", dev, prop.gcnArchName);
    void* fixed = nullptr;
    VKHR_CHECK_HIP(hipGetSymbolAddress(&fixed, HIP_SYMBOL(scratch)));
    VKHR_REQUIRE(fixed, VKHR_ERR_HIP, "device %d: no address for the static scratch", dev);
    g_static_scratch[dev] = fixed;
    g_checked[dev] = true;
    return VKHR_OK;
}

int static_scratch(size_t bytes, void** out) {
    int rc = ensure_device();
    if (rc) return rc;
    VKHR_REQUIRE(bytes <= kStaticScratchBytes, VKHR_ERR_OVERFLOW,
                 "needs %zu bytes of static scratch; the allocation-free entry points have %zu", bytes,
                 kStaticScratchBytes);
    int dev = 0;
    VKHR_CHECK_HIP(hipGetDevice(&dev));
    *out = g_static_scratch[dev];  // set under g_mutex before g_checked[dev]
    return VKHR_OK;
}

int check_volume(uint32_t nx, uint32_t ny, uint32_t nz, bool cells, const char* what) {
    VKHR_REQUIRE(nx && ny && nz, VKHR_ERR_INVALID, "%s: zero volume resolution %ux%ux%u", what, nx, ny, nz);
    VKHR_REQUIRE(nx <= kMaxVolumeSide && ny <= kMaxVolumeSide && nz <= kMaxVolumeSide, VKHR_ERR_OVERFLOW,
                 "%s: volume %ux%ux%u has a side above %u", what, nx, ny, nz, kMaxVolumeSide);
    const uint64_t x = nx, y = ny, z = nz;  // each <= 2^16: no product below wraps
    VKHR_REQUIRE(x * y * z <= (uint64_t(1) << 31), VKHR_ERR_OVERFLOW, "%s: volume %ux%ux%u exceeds 2^31 voxels",
                 what, nx, ny, nz);
    if (cells)
        VKHR_REQUIRE((x + 1) * (y + 1) * (z + 1) < (uint64_t(1) << 32) && (y + 1) * (z + 1) < (uint64_t(1) << 24),
                     VKHR_ERR_OVERFLOW, "%s: volume %ux%ux%u has too many cells for 32-bit cell indices", what, nx,
                     ny, nz);
    return VKHR_OK;
}

int stream_scratch(size_t bytes, hipStream_t stream, void** out) {
    int rc = ensure_device();
    if (rc) return rc;
    int dev = 0;
    VKHR_CHECK_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_mutex);
    Scratch& area = g_scratch[scratch_key(dev, stream)];
    if (area.bytes < bytes) {
        // Grow.  Work already queued on this stream may still read the old
        // buffer: it is freed once the stream has drained, or, while the
        // stream is being captured into a graph (which may replay it later),
        // kept until vkhr_release_scratch.
        if (area.ptr) {
            hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
            VKHR_CHECK_HIP(hipStreamIsCapturing(stream, &status));
            if (status == hipStreamCaptureStatusNone) {
                VKHR_CHECK_HIP(hipStreamSynchronize(stream));
                VKHR_CHECK_HIP(hipFree(area.ptr));
            } else {
                area.retired.push_back(area.ptr);
            }
            area.ptr = nullptr;
            area.bytes = 0;
        }
        size_t want = bytes < (1u << 20) ? (1u << 20) : bytes;
        void* p = nullptr;
        hipError_t e = hipMalloc(&p, want);
        if (e != hipSuccess) {
            set_error("scratch hipMalloc(%zu) failed: %s", want, hipGetErrorString(e));
            return VKHR_ERR_NOMEM;
        }
        area.ptr = p;
        area.bytes = want;
    }
    *out = area.ptr;
    return VKHR_OK;
}

int release_stream_scratch(hipStream_t stream) {
    int rc = ensure_device();
    if (rc) return rc;
    int dev = 0;
    VKHR_CHECK_HIP(hipGetDevice(&dev));
    Scratch area;
    Block block;
    char* page = nullptr;
    bool found = false;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        std::swap(block, g_kept[dev]);
        auto it = g_scratch.find(scratch_key(dev, stream));
        if ((found = it != g_scratch.end())) {
            area = it->second;
            g_scratch.erase(it);
        }
        if (g_scratch.empty() && g_host_used == 0) std::swap(page, g_host_page);
    }
    const RelaxedCapture relaxed;
    if (page) VKHR_CHECK_HIP(hipHostFree(page));
    if (block.ptr) VKHR_CHECK_HIP(hipFree(block.ptr));
    if (!found) return VKHR_OK;
    VKHR_CHECK_HIP(hipStreamSynchronize(stream));
    if (area.ptr) VKHR_CHECK_HIP(hipFree(area.ptr));
    if (area.call.ptr) VKHR_CHECK_HIP(hipFree(area.call.ptr));
    for (void* p : area.retired) VKHR_CHECK_HIP(hipFree(p));
    return VKHR_OK;
}

HostWords::HostWords() {
    std::lock_guard<std::mutex> lock(g_mutex);
    if (!g_host_page) {
        const RelaxedCapture relaxed;
        void* page = nullptr;
        if (hipHostMalloc(&page, kHostSlot * kHostSlots, hipHostMallocPortable | hipHostMallocMapped) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
        g_host_page = static_cast<char*>(page);
    }
    if (g_host_used == ~0ull) return;
    const int slot = __builtin_ctzll(~g_host_used);
    g_host_used |= 1ull << slot;
    words_ = reinterpret_cast<uint32_t*>(g_host_page + kHostSlot * slot);
}

HostWords::~HostWords() {
    if (!words_) return;
    std::lock_guard<std::mutex> lock(g_mutex);
    g_host_used &= ~(1ull << ((reinterpret_cast<char*>(words_) - g_host_page) / kHostSlot));
}

bool keep_block(int device, void* ptr, size_t bytes) {
    if (device < 0 || device >= kMaxDevices || bytes > kKeptTemporaries) return false;
    Block block{ptr, bytes};
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        std::swap(block, g_kept[device]);
    }
    if (block.ptr) {
        const RelaxedCapture relaxed;
        (void)hipFree(block.ptr);
    }
    return true;
}

void* reuse_block(int device, size_t bytes, size_t* held) {
    Block block;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (device < 0 || device >= kMaxDevices) return nullptr;
        if (!g_kept[device].ptr || g_kept[device].bytes < bytes || g_kept[device].bytes / 4 > bytes) return nullptr;
        std::swap(block, g_kept[device]);
    }
    // Frees wait for the device as hipDeviceSynchronize does, but unlike it
    // they leave a capture that another thread has under way valid.
    const RelaxedCapture relaxed;
    void* token = nullptr;
    if (hipMalloc(&token, 256) != hipSuccess || hipFree(token) != hipSuccess) {
        (void)hipGetLastError();
        if (!keep_block(device, block.ptr, block.bytes)) (void)hipFree(block.ptr);
        return nullptr;
    }
    *held = block.bytes;
    return block.ptr;
}

size_t stream_scratch_bytes(hipStream_t stream) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lock(g_mutex);
    auto it = g_scratch.find(scratch_key(dev, stream));
    return it == g_scratch.end() ? 0 : it->second.bytes + it->second.call.bytes;
}

CallScratch::CallScratch(size_t bytes, hipStream_t stream) : stream_(stream) {
    if (hipGetDevice(&device_) != hipSuccess) return;
    Block held;
    if (bytes <= kKeptTemporaries) {
        std::lock_guard<std::mutex> lock(g_mutex);
        auto it = g_scratch.find(scratch_key(device_, stream));
        if (it != g_scratch.end()) std::swap(held, it->second.call);
    }
    const RelaxedCapture relaxed;
    if (held.ptr && held.bytes < bytes) {
        (void)hipStreamSynchronize(stream);
        (void)hipFree(held.ptr);
        held = Block();
    }
    if (!held.ptr) {
        held.bytes = bytes < (1u << 20) ? (1u << 20) : bytes;
        if (hipMalloc(&held.ptr, held.bytes) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
    }
    ptr_ = held.ptr;
    bytes_ = held.bytes;
}

CallScratch::~CallScratch() {
    if (!ptr_) return;
    if (bytes_ <= kKeptTemporaries) {
        std::lock_guard<std::mutex> lock(g_mutex);
        try {
            Scratch& area = g_scratch[scratch_key(device_, stream_)];
            if (!area.call.ptr) {
                area.call = Block{ptr_, bytes_};
                return;
            }
        } catch (...) {  // no memory for the map's entry: freed below
        }
    }
    const RelaxedCapture relaxed;
    (void)hipStreamSynchronize(stream_);
    (void)hipFree(ptr_);
}

bool capturing(hipStream_t stream) {
    if (!stream) return false;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return status != hipStreamCaptureStatusNone;
}

// Sixteen bytes a store when the words start on a multiple of that (the
// 33.5 MB of a 128^3 accumulator in 8.5 us instead of 11.4).
__global__ void fill_u32_kernel(uint32_t* __restrict__ dst, size_t n, uint32_t value) {
    const size_t stride = size_t(gridDim.x) * blockDim.x, first = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const size_t quads = (reinterpret_cast<uintptr_t>(dst) & 15u) == 0 ? n / 4 : 0;
    for (size_t i = first; i < quads; i += stride)
        reinterpret_cast<uint4*>(dst)[i] = make_uint4(value, value, value, value);
    for (size_t i = 4 * quads + first; i < n; i += stride) dst[i] = value;
}

int fill_u32(uint32_t* dst, size_t n, uint32_t value, hipStream_t stream) {
    if (n == 0) return VKHR_OK;
    const bool quads = (reinterpret_cast<uintptr_t>(dst) & 15u) == 0;
    fill_u32_kernel<<<grid_for(quads ? n / 4 + 1 : n, 256, 8192), 256, 0, stream>>>(dst, n, value);
    VKHR_CHECK_LAUNCH();
    return VKHR_OK;
}

}  // namespace vkhr

extern "C" {

int vkhr_abi_version(void) { return VKHR_ABI_VERSION; }

const char* vkhr_last_error(void) { return vkhr::g_error; }

int vkhr_init(void) {
    vkhr::clear_error();
    return vkhr::ensure_device();
}

int vkhr_release_scratch(vkhr_stream stream) {
    vkhr::clear_error();
    return vkhr::release_stream_scratch(vkhr::as_stream(stream));
}

size_t vkhr_scratch_bytes(vkhr_stream stream) { return vkhr::stream_scratch_bytes(vkhr::as_stream(stream)); }

}  // extern "C"
