// Transfers between the device and a caller's ordinary (pageable) memory.
//
// The runtime stages such a copy through a buffer of its own on the calling thread, or page-locks the caller's
// pages for the length of the call: 16 GB/s down, 28 GB/s up, and 400 - 900 us for 1 - 2 MB, where the link
// moves 53 GB/s. Here the bytes pass through page-locked blocks. A kernel copies between a block and device
// memory and flags each 32 KB chunk in host memory when its copy is complete, so neither copies nor
// reuse of a block need an event or a call into the runtime; the caller's thread and up to 7 workers (one fewer than it
// has processors at most) copy between blocks and the caller's memory, and take the page faults of a fresh array,
// while the link moves the next group of blocks. Before a download the workers sleep until its first chunk is there:
// polling through the kernels before it, they took 52 ms of processor time for a 10 ms kernel, now 12.
//
// Microseconds (runtime's copy -> this one), arrays touched before: down 1 MB 440 -> 62, 2 MB 870 -> 110, 8 MB
// 485 -> 250, 24 MB 1500 -> 640; up 1 MB 390 -> 55, 2 MB 740 -> 100, 8 MB 320 -> 300, 24 MB 850 -> 730. A thread
// started per piece instead of a waiting worker: 24 MB down 780.
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "host_io.h"

namespace pisurf {

namespace {

struct Job {
    void (*fn)(void*, int);
    void* arg;
    int n;
    std::atomic<int> next{0};
    int room = 0;    // workers it may have
    int active = 0;  // workers inside (under the lock)
};

// Threads for a job of the calling thread: no more than it has processors.
int host_threads() {
    cpu_set_t set;
    if (sched_getaffinity(0, sizeof(set), &set) != 0) return kHostThreads;  // (more processors than the set holds)
    return std::max(1, std::min(kHostThreads, CPU_COUNT(&set)));
}

// Worker threads, started by the first job that wants one. A thread costs 15 us to start, a job of a
// few MB takes 100.
class Workers {
  public:
    void run(int n, void (*fn)(void*, int), void* arg) {
        Job j;
        j.fn = fn;
        j.arg = arg;
        j.n = n;
        if (n > 1 && enter(&j)) {
            work(&j);
            leave(&j);
        } else {
            work(&j);
        }
    }
    void stop() {
        std::vector<std::thread> t;
        {
            std::lock_guard<std::mutex> lk(m_);
            stop_ = true;
            t.swap(threads_);
        }
        cv_.notify_all();
        for (auto& x : t) x.join();
        std::lock_guard<std::mutex> lk(m_);
        stop_ = false;
    }

  private:
    static void work(Job* j) {
        for (int i; (i = j->next.fetch_add(1, std::memory_order_relaxed)) < j->n;) j->fn(j->arg, i);
    }
    // true when workers may be inside the job
    bool enter(Job* j) {
        const int want = std::min(j->n, host_threads()) - 1;
        if (want <= 0) return false;
        j->room = want;
        bool in = false;
        try {
            std::lock_guard<std::mutex> lk(m_);
            jobs_.push_back(j);
            posted_.fetch_add(1, std::memory_order_relaxed);
            in = true;
            while ((int)threads_.size() < want) threads_.emplace_back([this] { loop(); });
        } catch (const std::system_error&) {  // no more threads: those there are do the job, or the caller alone
        } catch (const std::bad_alloc&) {
        }
        if (want == 1) cv_.notify_one();
        else cv_.notify_all();
        return in;
    }
    void leave(Job* j) {
        std::unique_lock<std::mutex> lk(m_);
        drop(j);
        done_.wait(lk, [&] { return j->active == 0; });
    }
    void drop(Job* j) {
        auto it = std::find(jobs_.begin(), jobs_.end(), j);
        if (it != jobs_.end()) jobs_.erase(it);
    }
    Job* open_job() {
        for (Job* j : jobs_)
            if (j->active < j->room) return j;
        return nullptr;
    }
    void loop() {
        std::unique_lock<std::mutex> lk(m_);
        for (;;) {
            Job* j = nullptr;
            cv_.wait(lk, [&] { return stop_ || (j = open_job()) != nullptr; });
            if (stop_) return;
            j->active++;
            lk.unlock();
            work(j);
            lk.lock();
            drop(j);  // nothing of it is left to claim
            if (--j->active == 0) done_.notify_all();
            if (stop_ || open_job()) continue;
            const unsigned seen = posted_.load(std::memory_order_relaxed);
            lk.unlock();
            linger(seen);
            lk.lock();
        }
    }
    // A sleeping worker takes some 60 us to arrive, and a download often follows an upload and a short kernel: a worker
    // looks for another job for kLinger before it sleeps (200 k edges, 12 MB up and 5.6 MB down around a kernel of 0.18
    // ms: 970 -> 925 us; without it 0.3 ms less of each worker's processor time per transfer).
    void linger(unsigned seen) const {
        const auto until = std::chrono::steady_clock::now() + kLinger;
        while (posted_.load(std::memory_order_relaxed) == seen && std::chrono::steady_clock::now() < until) {
            for (int k = 0; k < 32; k++) __builtin_ia32_pause();
            sched_yield();
        }
    }
    static constexpr std::chrono::microseconds kLinger{300};
    std::mutex m_;
    std::condition_variable cv_, done_;
    std::vector<Job*> jobs_;
    std::atomic<unsigned> posted_{0};  // jobs so far
    std::vector<std::thread> threads_;
    bool stop_ = false;
};

class Stage {
  public:
    Stage() { free_.reserve(kStageLimit); }
    StageBlock* take(int device) {
        std::lock_guard<std::mutex> lk(m_);
        for (size_t i = 0; i < free_.size(); i++)
            if (free_[i]->device == device) {
                StageBlock* b = free_[i];
                free_.erase(free_.begin() + i);
                return b;
            }
        if (made_ >= kStageLimit) {
            if (free_.empty()) return nullptr;
            destroy(free_.back());  // another device's
            free_.pop_back();
        }
        StageBlock* b = new (std::nothrow) StageBlock();
        if (!b) return nullptr;
        made_++;
        void* h = nullptr;
        void* d = nullptr;
        const size_t bytes = kStageBytes + kStageFlags * sizeof(uint32_t);
        const unsigned flags = hipHostMallocMapped | hipHostMallocCoherent | hipHostMallocPortable;
        hipError_t e = hipHostMalloc(&h, bytes, flags);
        b->host = e == hipSuccess ? (char*)h : nullptr;
        if (e == hipSuccess) e = hipHostGetDevicePointer(&d, h, 0);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            destroy(b);
            return nullptr;
        }
        std::memset(b->host + kStageBytes, 0, kStageFlags * sizeof(uint32_t));
        b->dev = (char*)d;
        b->seq = 0;
        b->device = device;
        return b;
    }
    void give(StageBlock* b) {
        std::lock_guard<std::mutex> lk(m_);
        free_.push_back(b);  // within the reserved room
    }
    int contexts = 0;
    std::mutex cm;
    void clear() {
        std::lock_guard<std::mutex> lk(m_);
        for (StageBlock* b : free_) destroy(b);
        free_.clear();
    }

  private:
    void destroy(StageBlock* b) {
        if (b->host) (void)hipHostFree(b->host);
        delete b;
        made_--;
    }
    std::mutex m_;
    std::vector<StageBlock*> free_;
    int made_ = 0;
};

// never destroyed: the process may end with the runtime gone and threads asleep
Stage& stage() {
    static Stage* s = new Stage();
    return *s;
}
Workers& workers() {
    static Workers* w = new Workers();
    return *w;
}

// One launch: up to kStageGroup blocks, each kStageBytes of the array (the last one less).
struct StageCopy {
    char* dev;      // device memory of the first block's bytes
    size_t bytes;   // of this launch
    char* blk[kStageGroup];
    uint32_t seq[kStageGroup];
};

// A workgroup copies a chunk, four 16-byte words in flight per thread, and flags it when all its stores are visible to
// the host (or, on the way up, all its loads have returned). Bound by the link: 24 MB in 480 us either way, as the
// copy engines take (450).
template <bool DOWN> __global__ void __launch_bounds__(256) k_stage(StageCopy a) {
    const int part = blockIdx.x / kStageFlags;
    const size_t in = (blockIdx.x % kStageFlags) * kStageChunk;
    const size_t at = (size_t)part * kStageBytes + in;
    if (at >= a.bytes) return;
    const size_t n = min(kStageChunk, a.bytes - at);
    char* blk = part ? a.blk[1] : a.blk[0];
    const uint32_t seq = part ? a.seq[1] : a.seq[0];
    const char* src = DOWN ? a.dev + at : blk + in;
    char* dst = DOWN ? blk + in : a.dev + at;
    constexpr int U = 4;
    if (n == kStageChunk) {
        for (size_t i = threadIdx.x; i < kStageChunk / 16; i += 256 * U) {
            uint4 v[U];
#pragma unroll
            for (int k = 0; k < U; k++) v[k] = ((const uint4*)src)[i + 256 * k];
#pragma unroll
            for (int k = 0; k < U; k++) ((uint4*)dst)[i + 256 * k] = v[k];
        }
    } else {
        for (size_t i = threadIdx.x; i < n / 4; i += 256) ((uint32_t*)dst)[i] = ((const uint32_t*)src)[i];
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) {
        *((volatile uint32_t*)(blk + kStageBytes) + in / kStageChunk) = seq;
        __threadfence_system();
    }
}
static_assert(kStageGroup == 2 && (kStageChunk / 16) % 1024 == 0, "k_stage");

// a transfer in progress
struct Transfer {
    char* host;
    char* dev;
    size_t bytes;
    int device;
    hipStream_t s;
    bool down;
    int nb;  // blocks
    StageBlock* blk[kStageBlocks];
    uint32_t base[kStageBlocks];  // their sequence numbers before
    int pieces;
    std::atomic<int> err{(int)hipSuccess};
    std::atomic<int> issued[kStageBlocks];  // copies through the block that have been launched
    std::atomic<int> left[kStageBlocks];    // down: blocks of the group (by its first block) still to be emptied

    size_t size(int p) const { return std::min(kStageBytes, bytes - (size_t)p * kStageBytes); }
    void fail(hipError_t e) {
        int none = (int)hipSuccess;
        err.compare_exchange_strong(none, (int)e);
    }
    bool ok() const { return err.load(std::memory_order_relaxed) == (int)hipSuccess; }

    // pieces p .. p + k - 1 through blocks p % nb ..: one launch
    void launch(int p, int k) {
        if (!ok()) return;
        hipError_t e = hipSetDevice(device);
        StageCopy a;
        a.dev = dev + (size_t)p * kStageBytes;
        a.bytes = 0;
        for (int i = 0; i < kStageGroup; i++) {
            const int q = p + (i < k ? i : 0), b = q % nb;
            a.blk[i] = blk[b]->dev;
            a.seq[i] = base[b] + 1 + q / nb;
            if (i < k) a.bytes += size(q);
        }
        if (e == hipSuccess) {
            const int grid = (int)((a.bytes + kStageChunk - 1) / kStageChunk);
            if (down) k_stage<true><<<grid, 256, 0, s>>>(a);
            else k_stage<false><<<grid, 256, 0, s>>>(a);
            e = hipGetLastError();
        }
        if (e != hipSuccess) fail(e);
        for (int i = 0; i < k; i++) issued[(p + i) % nb].store((p + i) / nb + 1, std::memory_order_release);
    }
    // the i-th look at a flag in vain: the link fills a chunk in 0.6 us; what takes longer than some 4096 looks is a
    // kernel before the copy, or a thread that wants this processor
    static void relax(uint32_t i) {
        if (i < 4096) __builtin_ia32_pause();
        else sched_yield();
    }
    // chunk c of piece p has been copied by the device
    bool wait_chunk(int p, size_t c) {
        const int b = p % nb;
        const uint32_t want = base[b] + 1 + p / nb;
        volatile uint32_t* w = blk[b]->flag(c);
        for (uint32_t i = 1; *w != want; i++) {
            relax(i);
            if ((i & 4095) == 0) {
                if (!ok()) return false;
                if (issued[b].load(std::memory_order_acquire) <= p / nb) continue;
                // a device error ends the wait, and a stream that is done without the flag showing does too
                const hipError_t e = hipStreamQuery(s);
                if (e == hipErrorNotReady) continue;
                if (e == hipSuccess) {
                    for (int k = 0; k < (1 << 16); k++)
                        if (*w == want) break;
                    if (*w == want) break;
                }
                fail(e == hipSuccess ? hipErrorUnknown : e);
                return false;
            }
        }
        std::atomic_thread_fence(std::memory_order_acquire);
        return true;
    }
    bool wait_piece(int p) {
        const size_t m = size(p);
        for (size_t c = 0; c * kStageChunk < m; c++)
            if (!wait_chunk(p, c)) return false;
        return true;
    }
    int group(int p) const { return std::min(kStageGroup, pieces - p); }

    void operator()(int p) {
        if (!ok()) return;
        const size_t at = (size_t)p * kStageBytes, m = size(p);
        const int b = p % nb;
        if (down) {
            for (size_t c = 0; c < m; c += kStageChunk) {
                if (!wait_chunk(p, c / kStageChunk)) return;
                std::memcpy(host + at + c, blk[b]->host + c, std::min(kStageChunk, m - c));
            }
            // the group's last piece out of its blocks refills them
            const int first = p - p % kStageGroup, g = first % nb;
            if (left[g].fetch_sub(1, std::memory_order_acq_rel) == 1 && first + nb < pieces) {
                left[g].store(group(first + nb), std::memory_order_relaxed);
                launch(first + nb, group(first + nb));
            }
        } else {
            if (p >= nb) {
                for (uint32_t i = 1; issued[b].load(std::memory_order_acquire) < p / nb; i++) {
                    if (!ok()) return;
                    relax(i);
                }
                if (!wait_piece(p - nb)) return;
            }
            std::memcpy(blk[b]->host, host + at, m);
            launch(p, 1);
        }
    }
};

}  // namespace

void host_io_attach() {
    std::lock_guard<std::mutex> lk(stage().cm);
    stage().contexts++;
}

void host_io_detach() {
    std::lock_guard<std::mutex> lk(stage().cm);
    if (--stage().contexts > 0) return;
    workers().stop();
    stage().clear();
}

StageBlock* stage_take(int device) { return stage().take(device); }
void stage_give(StageBlock* b) { stage().give(b); }

void host_parallel(int n, void (*fn)(void*, int), void* arg) { workers().run(n, fn, arg); }

void host_copy(void* dst, const void* src, size_t bytes) {
    constexpr size_t part = size_t(512) << 10;
    if (bytes < 2 * part) {
        if (bytes) std::memcpy(dst, src, bytes);
        return;
    }
    auto f = [&](int i) {
        const size_t a = (size_t)i * part;
        std::memcpy((char*)dst + a, (const char*)src + a, std::min(part, bytes - a));
    };
    host_parallel((int)((bytes + part - 1) / part), f);
}

bool pageable(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

hipError_t staged_copy(void* dst, const void* src, size_t bytes, bool down, int device, hipStream_t s) {
    if (bytes == 0) return hipSuccess;
    const auto kind = down ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice;
    Transfer t;
    t.host = down ? (char*)dst : (char*)const_cast<void*>(src);
    t.dev = down ? (char*)const_cast<void*>(src) : (char*)dst;
    if (!pageable(t.host) || bytes % 4 || (uintptr_t)t.dev % 16) return hipMemcpyAsync(dst, src, bytes, kind, s);
    t.bytes = bytes;
    t.device = device;
    t.s = s;
    t.down = down;
    t.pieces = (int)((bytes + kStageBytes - 1) / kStageBytes);
    t.nb = 0;
    const int want = std::min(kStageBlocks, t.pieces);
    while (t.nb < want) {
        StageBlock* b = stage_take(device);
        if (!b) break;
        t.blk[t.nb++] = b;
    }
    // down: whole groups, so that a group's blocks are refilled together
    while (down && t.nb < t.pieces && t.nb % kStageGroup) stage_give(t.blk[--t.nb]);
    if (t.nb == 0) return hipMemcpyAsync(dst, src, bytes, kind, s);
    for (int b = 0; b < t.nb; b++) {
        t.base[b] = t.blk[b]->seq;
        t.issued[b].store(0, std::memory_order_relaxed);
        t.left[b].store(0, std::memory_order_relaxed);
    }
    if (down)
        for (int p = 0; p < t.nb; p += kStageGroup) {
            const int k = std::min(kStageGroup, t.nb - p);
            t.left[p].store(k, std::memory_order_relaxed);
            t.launch(p, k);
        }
    // Kernels queued before the copy may run for long: the caller waits for them alone, and the workers, which other
    // callers share, are woken when data flows.
    if (down && t.pieces > 1) (void)t.wait_chunk(0, 0);
    host_parallel(t.pieces, t);
    if (!down)
        for (int p = std::max(0, t.pieces - t.nb); p < t.pieces && t.ok(); p++) (void)t.wait_piece(p);
    // after an error no copy may be under way in a block that another transfer takes
    if (!t.ok()) (void)hipStreamSynchronize(s);
    for (int b = 0; b < t.nb; b++) {
        t.blk[b]->seq = t.base[b] + 1 + (uint32_t)((t.pieces - 1) / t.nb);
        stage_give(t.blk[b]);
    }
    return (hipError_t)t.err.load();
}

}  // namespace pisurf
