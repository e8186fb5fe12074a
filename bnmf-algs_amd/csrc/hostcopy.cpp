// hostcopy.cpp — results to host memory.
//
// hipMemcpy into pageable memory stages through one thread: 10 GB/s into
// fresh pages, 17 GB/s into touched ones, where the link does 57 GB/s. Here a
// result of some size goes through a pinned buffer in chunks of up to 2 MiB
// that up to eight threads fetch and copy on, so that the page faults and the
// host copies of several chunks overlap each other and the link. Measured
// (1 GiB into fresh huge pages, one MI355X, 16 host cores): 27 ms with 8
// threads and 2 MiB chunks against 107 ms for hipMemcpy; 34 ms with 1 MiB
// chunks, the same with 16 threads; into 4 KiB pages 48 ms. The 60 results of a
// batch, 5 MiB on average, take 3 ms longer where only those of 8 MiB and more
// are staged.
//
// The pinned buffer (32 MiB) belongs to the batch or server whose results it
// carries. Pinning it takes 1 to 2 ms, more than a small result does in all
// (16 MiB: 0.95 ms by hipMemcpy, 2.0 ms with the pinning, 0.6 ms once pinned), so
// an object's results go by hipMemcpy until they come to 48 MiB, and one that is
// larger takes the buffer at once (48 MiB: 5.0 against 3.5 ms; a call whose result is
// 40 MiB 5.4 against 6.4).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

#include "bnmf_internal.hpp"

namespace bnmf {

namespace {
constexpr size_t kChunk = 2u << 20, kChunkLeast = 256u << 10;
constexpr unsigned kThreads = 8;
constexpr size_t kPerThread = 768u << 10;  // bytes a thread is worth starting for
constexpr size_t kFirst = 48u << 20;       // bytes of results before a buffer is pinned

struct Copy {
    char* dst;
    const char* src;
    size_t bytes, chunk, chunks;
    char* pinned;
    hipStream_t st;
    int dev;
    std::atomic<size_t> next{0};
    std::atomic<int> status{(int)hipSuccess};

    // Two slots of the pinned buffer: the next chunk is on the link while the
    // last one is copied on.
    void work(unsigned slot) {
        hipError_t e = hipSetDevice(dev);
        hipEvent_t ev[2] = {nullptr, nullptr};
        for (int k = 0; k < 2 && e == hipSuccess; ++k) e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
        size_t held[2] = {chunks, chunks};
        int k = 0;
        while (e == hipSuccess && status.load() == (int)hipSuccess) {
            const size_t c = next.fetch_add(1);
            char* const buf = pinned + (size_t)(2 * slot + k) * chunk;
            if (c < chunks) {
                e = hipMemcpyAsync(buf, src + c * chunk, size_of(c), hipMemcpyDeviceToHost, st);
                if (e == hipSuccess) e = hipEventRecord(ev[k], st);
                held[k] = c;
            }
            k ^= 1;
            if (e == hipSuccess && held[k] < chunks) {
                e = hipEventSynchronize(ev[k]);
                if (e == hipSuccess)
                    std::memcpy(dst + held[k] * chunk, pinned + (size_t)(2 * slot + k) * chunk, size_of(held[k]));
                held[k] = chunks;
            }
            if (c >= chunks && held[k ^ 1] >= chunks) break;
        }
        if (e != hipSuccess) status.store((int)e);
        for (int i = 0; i < 2; ++i)
            if (ev[i]) (void)hipEventDestroy(ev[i]);
    }
    size_t size_of(size_t c) const { return std::min(chunk, bytes - c * chunk); }
};
}  // namespace

HostStage::~HostStage() {
    if (pinned) (void)hipHostFree(pinned);
}

void HostStage::copy(void* dst, const void* src, size_t bytes, hipStream_t st) {
    if (bytes == 0) return;
    const unsigned cores = std::max(1u, std::thread::hardware_concurrency());
    const unsigned n = (unsigned)std::min<size_t>(std::min(kThreads, cores), bytes / kPerThread);
    std::unique_lock<std::mutex> lk(mu, std::defer_lock);
    bool staged = n >= 2;
    if (staged) {
        lk.lock();
        fetched += bytes;
        if (!pinned && fetched >= kFirst && hipHostMalloc(&pinned, 2 * kThreads * kChunk, 0) != hipSuccess) {
            (void)hipGetLastError();
            pinned = nullptr;
        }
        staged = pinned != nullptr;
    }
    if (!staged) {
        if (lk.owns_lock()) lk.unlock();
        BNMF_HIP(hipStreamSynchronize(st));
        BNMF_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
        return;
    }
    const size_t chunk = std::min(kChunk, (bytes / (2 * n) + kChunkLeast - 1) / kChunkLeast * kChunkLeast);
    Copy c;
    c.dst = static_cast<char*>(dst);
    c.src = static_cast<const char*>(src);
    c.bytes = bytes;
    c.chunk = chunk;
    c.chunks = (bytes + chunk - 1) / chunk;
    c.pinned = static_cast<char*>(pinned);
    c.st = st;
    c.dev = 0;
    BNMF_HIP(hipGetDevice(&c.dev));
    // the calling thread works too, alone if no other can be started
    std::vector<std::thread> th;
    th.reserve(n);
    try {
        for (unsigned w = 1; w < n; ++w) th.emplace_back([&c, w] { c.work(w); });
    } catch (const std::exception&) {  // no thread, or no memory for one
    }
    c.work(0);
    for (std::thread& t : th) t.join();
    const hipError_t e = (hipError_t)c.status.load();
    // a failed copy may still be writing to the pinned buffer
    if (e != hipSuccess) (void)hipStreamSynchronize(st);
    BNMF_HIP(e);
}

}  // namespace bnmf
