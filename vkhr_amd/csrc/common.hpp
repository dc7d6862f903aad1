// Shared host/device helpers of libvkhr_hip: status plumbing, the per-device
// scratch area, and small device primitives.  gfx950 only (wave64).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>

#include "vkhr_hip.h"

namespace vkhr {

constexpr int kWave = 64;

// ----------------------------------------------------------------- status

void set_error(const char* fmt, ...);
void clear_error();

#define VKHR_CHECK_HIP(expr)                                                   \
    do {                                                                       \
        hipError_t vkhr_e_ = (expr);                                           \
        if (vkhr_e_ != hipSuccess) {                                           \
            ::vkhr::set_error("%s failed: %s (%s:%d)", #expr,                  \
                              hipGetErrorString(vkhr_e_), __FILE__, __LINE__); \
            return VKHR_ERR_HIP;                                               \
        }                                                                      \
    } while (0)

#define VKHR_REQUIRE(cond, code, ...)                                          \
    do {                                                                       \
        if (!(cond)) {                                                         \
            ::vkhr::set_error(__VA_ARGS__);                                    \
            return (code);                                                     \
        }                                                                      \
    } while (0)

// Checks the launch that was just enqueued.
#define VKHR_CHECK_LAUNCH() VKHR_CHECK_HIP(hipGetLastError())

// Binds per-device state; returns VKHR_OK or an error code.
int ensure_device();

// Largest volume side any entry point accepts.  Every entry point that takes
// a volume validates its sides with check_volume before any size arithmetic,
// so no product of sides can wrap.
constexpr uint32_t kMaxVolumeSide = 1u << 16;

// Volume dimension check shared by every entry point that takes a volume:
// each side in [1, kMaxVolumeSide] (VKHR_ERR_INVALID for a zero side,
// VKHR_ERR_OVERFLOW above), at most 2^31 voxels, and with cells the cell
// lattice (nx+1)(ny+1)(nz+1) below 2^32 with (ny+1)(nz+1) below 2^24 (the
// kernels index cells with 24-bit multiplies and 32-bit sums).  All
// arithmetic is 64-bit.  `what` names the volume in the error message.
int check_volume(uint32_t nx, uint32_t ny, uint32_t nz, bool cells, const char* what);

// Scratch of one device and stream: a device buffer of at least `bytes`
// bytes owned by the library until vkhr_release_scratch on that stream (or
// process end).  Calls on one stream are ordered by the stream; calls on
// different streams (and hipStreamPerThread on different threads) get
// different areas.  Growing an area synchronizes the stream before freeing
// the old buffer (outside graph capture).
int stream_scratch(size_t bytes, hipStream_t stream, void** out);

// Bytes of the static per-device scratch of the allocation-free entry
// points (a file-scope __device__ array, no allocation at run time).
constexpr size_t kStaticScratchBytes = VKHR_STATIC_SCRATCH_BYTES;

// The current device's static scratch, after checking that `bytes` fit
// (VKHR_ERR_OVERFLOW otherwise).  Every call on a device shares it and it
// keeps the last call's contents: users clear what must start at zero, and
// calls that overlap on one device race.
int static_scratch(size_t bytes, void** out);

// Synchronizes the stream and frees its area (vkhr_release_scratch), and
// gives back what the device keeps besides: the result words' page when no
// area is left, and the block of reuse_block.
int release_stream_scratch(hipStream_t stream);

// Allocations, frees and waits for a stream are refused on every thread, and
// end the capture, while any thread captures in global mode, unless the thread
// that makes them is in relaxed mode: they touch no captured stream.
class RelaxedCapture {
public:
    RelaxedCapture() { ok_ = hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess; }
    ~RelaxedCapture() {
        if (ok_) (void)hipThreadExchangeStreamCaptureMode(&mode_);
    }
    RelaxedCapture(const RelaxedCapture&) = delete;
    RelaxedCapture& operator=(const RelaxedCapture&) = delete;

private:
    hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;  // the thread's own once exchanged
    bool ok_ = false;
};

// Temporaries that one call has to itself: the block that its stream keeps
// for this, when it is there and large enough, else an allocation, which
// becomes that block at the call's end if it is kKeptTemporaries or less and
// none is there (it is freed otherwise).  Taken out for the length of the
// call: threads that call on one stream each have their own, whatever the
// order of their kernels, and calls one after another are ordered by the
// stream.  Not for a stream under capture.  get() is null when the memory
// cannot be had.
constexpr size_t kKeptTemporaries = size_t(256) << 20;

class CallScratch {
public:
    CallScratch(size_t bytes, hipStream_t stream);
    ~CallScratch();
    CallScratch(const CallScratch&) = delete;
    CallScratch& operator=(const CallScratch&) = delete;
    void* get() const { return ptr_; }

private:
    hipStream_t stream_;
    int device_ = 0;
    void* ptr_ = nullptr;
    size_t bytes_ = 0;
};

// Whether the stream is being captured into a graph (the null stream never is).
bool capturing(hipStream_t stream);

// 64 bytes of pinned host memory that a kernel writes a small result to and
// the host reads once the stream has been waited for, in place of a copy
// command and its staging (bounds and order of 2k strands: about 10 us each).  The slots are one page, kept
// from first use; a slot belongs to one object at a time, on whatever thread
// or stream.  words() is null when the page cannot be had or all slots are
// taken: the caller then copies.
class HostWords {
public:
    HostWords();
    ~HostWords();
    HostWords(const HostWords&) = delete;
    HostWords& operator=(const HostWords&) = delete;
    uint32_t* words() const { return words_; }

private:
    uint32_t* words_ = nullptr;
};

// Device memory of an object that is often destroyed and built again (a
// style's tree each frame): keep_block takes over a block to be freed, of at
// most kKeptTemporaries bytes (false: free it yourself), in place of the
// device's last one, which it frees,
// and reuse_block hands it out again when it holds `bytes` and is at most
// four times that, once the device has finished everything that was queued
// while the block was in use.  With the temporaries kept as well and the
// bounds read with the last wait, a tree of 75k segments and 200k rays take
// 515 us instead of 660.
bool keep_block(int device, void* ptr, size_t bytes);
void* reuse_block(int device, size_t bytes, size_t* held);

// Bytes held by the area of the calling thread's device and this stream.
size_t stream_scratch_bytes(hipStream_t stream);

inline hipStream_t as_stream(vkhr_stream s) { return reinterpret_cast<hipStream_t>(s); }

inline unsigned grid_for(size_t n, unsigned block, unsigned cap = 1u << 20) {
    size_t g = (n + block - 1) / block;
    if (g == 0) g = 1;
    if (g > cap) g = cap;
    return static_cast<unsigned>(g);
}

// Fills n 32-bit words with a value (graph-capture safe, unlike memset nodes).
int fill_u32(uint32_t* dst, size_t n, uint32_t value, hipStream_t stream);

// ------------------------------------------------------------- device side

__device__ __forceinline__ float3 load_xyz(const float* __restrict__ p, uint32_t i) {
    return make_float3(p[3u * i + 0u], p[3u * i + 1u], p[3u * i + 2u]);
}

// The launch's argument block T read in place from the kernarg segment
// (the explicit arguments start at its offset 0, so T must be the kernel's
// first parameter).  Read through this reference, each field is loaded
// from constant memory where it is used; taken from the by-value
// parameter, the compiler holds the block's fields in scalar registers
// across the kernel's loops, and a large block spills them into vector
// register lanes.
template <class T>
__device__ __forceinline__ const T& kernel_args() {
    return *(const T*)__builtin_amdgcn_kernarg_segment_ptr();
}

}  // namespace vkhr
