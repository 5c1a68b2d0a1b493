// Large device-to-host copies into ordinary (pageable) host memory.
//
// The runtime's own copy into pageable memory stages it through one thread:
// 18 GB/s into pages that exist, 10 GB/s into new ones, where the first touch
// of every page costs more than the copy; result arrays are always new.  Here
// a few threads each take the next chunk, have the DMA engine write it to
// their own pinned block (57 GB/s in all) and copy it out, so that the page
// faults of several chunks are served at once.
//
// The pinned blocks (THREADS x CHUNK = 12 MiB) are allocated by the first large
// copy, shared by everything in a library that holds a StagedCopy and freed
// with its last holder; the integrator's library and the surrogate's have blocks
// of their own.  One copy uses a library's blocks at a time; a second one at the
// same moment, a small copy, or one for which no threads or pinned memory are to
// be had takes the runtime's copy.  The
// device work that produces the data must have been queued on `stream` before;
// the copies are queued there too, and the call returns when all have arrived.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace clode {

class StagedCopy {
public:
    static constexpr size_t CHUNK = (size_t)2 << 20;
    static constexpr int THREADS = 6;
    static constexpr size_t SMALLEST = 4 * CHUNK;  // below this the threads cost more than they save

    static std::shared_ptr<StagedCopy> get()
    {
        static std::mutex mu;
        static std::weak_ptr<StagedCopy> shared;
        std::lock_guard<std::mutex> lk(mu);
        std::shared_ptr<StagedCopy> s = shared.lock();
        if (!s) {
            s.reset(new StagedCopy);
            shared = s;
        }
        return s;
    }

    ~StagedCopy()
    {
        if (pinned_)
            (void)hipHostFree(pinned_);
    }

    // bytes from device memory to host memory, complete on return
    hipError_t toHost(int device, void *dst, const void *src, size_t bytes, hipStream_t stream)
    {
        if (bytes >= SMALLEST) {
            std::unique_lock<std::mutex> lk(use_, std::try_to_lock);
            if (lk.owns_lock() && ready())
                return staged(device, static_cast<char *>(dst), static_cast<const char *>(src), bytes, stream);
        }
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
        return e != hipSuccess ? e : hipStreamSynchronize(stream);
    }

private:
    StagedCopy() = default;

    bool ready()
    {
        if (!pinned_ && !failed_ && hipHostMalloc((void **)&pinned_, THREADS * CHUNK, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            pinned_ = nullptr;
            failed_ = true;
        }
        return pinned_ != nullptr;
    }

    hipError_t staged(int device, char *dst, const char *src, size_t bytes, hipStream_t stream)
    {
        const size_t chunks = (bytes + CHUNK - 1) / CHUNK;
        std::atomic<size_t> next{0};
        std::atomic<int> error{hipSuccess};
        auto work = [&](int k) {
            hipEvent_t here = nullptr;
            hipError_t e = hipSetDevice(device);
            if (e == hipSuccess)
                e = hipEventCreateWithFlags(&here, hipEventDisableTiming);
            char *block = pinned_ + (size_t)k * CHUNK;
            while (e == hipSuccess && error.load() == hipSuccess) {
                const size_t c = next.fetch_add(1);
                if (c >= chunks)
                    break;
                const size_t off = c * CHUNK, n = std::min(CHUNK, bytes - off);
                e = hipMemcpyAsync(block, src + off, n, hipMemcpyDeviceToHost, stream);
                if (e == hipSuccess)
                    e = hipEventRecord(here, stream);
                if (e == hipSuccess)
                    e = hipEventSynchronize(here);
                if (e == hipSuccess)
                    std::memcpy(dst + off, block, n);
            }
            if (here)
                (void)hipEventDestroy(here);
            if (e != hipSuccess)
                error.store(e);
        };
        std::vector<std::thread> helpers;
        for (int k = 1; k < THREADS && (size_t)k < chunks; ++k) {
            try {
                helpers.emplace_back(work, k);
            } catch (const std::exception &) {  // fewer threads, the same copy
                break;
            }
        }
        work(0);
        for (auto &t : helpers)
            t.join();
        // after an error a copy into a block may still be on its way, and the
        // blocks are free for the next caller from here on
        if (error.load() != hipSuccess)
            (void)hipStreamSynchronize(stream);
        return (hipError_t)error.load();
    }

    std::mutex use_;
    char *pinned_ = nullptr;
    bool failed_ = false;
};

}  // namespace clode
