// Transfers between the device and a caller's ordinary (pageable) memory, and large host copies.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <cstring>

namespace pisurf {

// a call whose inputs and outputs fit this many bytes lets its kernel use a block of page-locked memory directly
constexpr size_t kDirectBytes = size_t(256) << 10;
constexpr size_t kStageBytes = size_t(1) << 20;         // one block
constexpr size_t kStageChunk = size_t(32) << 10;        // bytes per workgroup of the copy kernel, with a flag each
constexpr int kStageFlags = int(kStageBytes / kStageChunk);
constexpr int kStageBlocks = 8;                         // blocks of one transfer at most
constexpr int kStageLimit = 16;                         // blocks of the process at most (16 MB page-locked)
constexpr int kStageGroup = 2;                          // blocks filled by one launch on the way down
constexpr int kHostThreads = 8;                         // threads of one host job at most, the caller's among them

// Page-locked memory that kernels read and write, with a word per chunk behind it: the sequence number of the block's
// last copy that is complete for that chunk.
struct StageBlock {
    char* host;
    char* dev;  // its device address
    uint32_t seq;
    int device;
    volatile uint32_t* flag(size_t chunk) const { return (volatile uint32_t*)(host + kStageBytes) + chunk; }
};

// Blocks and worker threads are shared by the contexts of the process and end with the last one.
void host_io_attach();
void host_io_detach();

// a block for the caller's use, or nullptr (all in use, memory cannot be locked)
StageBlock* stage_take(int device);
void stage_give(StageBlock* b);

// fn(arg, 0) .. fn(arg, n - 1) on the calling thread and the workers that are free; fn must not throw
void host_parallel(int n, void (*fn)(void*, int), void* arg);
template <class F> inline void host_parallel(int n, F& f) {
    host_parallel(n, [](void* a, int i) { (*(F*)a)(i); }, (void*)&f);
}

// memcpy, by several threads from 1 MB on
void host_copy(void* dst, const void* src, size_t bytes);

// ordinary host memory: the runtime knows nothing of it
bool pageable(const void* p);

// every double of the range is finite (an exponent of all ones is not)
inline bool all_finite(const double* p, size_t n) {
    uint64_t bad = 0;
    for (size_t i = 0; i < n; i++) {
        uint64_t v;
        std::memcpy(&v, p + i, 8);
        bad |= (uint64_t)((v & 0x7ff0000000000000ull) == 0x7ff0000000000000ull);
    }
    return bad == 0;
}

// Device memory to the host (down) or back, in stream order. Ordinary host memory holds the data, or is free again, on
// return; for page-locked or device memory a wait on the stream completes the copy.
hipError_t staged_copy(void* dst, const void* src, size_t bytes, bool down, int device, hipStream_t s);

}  // namespace pisurf
