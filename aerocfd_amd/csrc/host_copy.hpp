// Device to pageable host memory for large fields (acfd_download).
//
// hipMemcpy to pageable memory goes through the runtime's pinned buffer and
// one thread's copy out of it, which also takes the page faults of a fresh
// destination: 8-11 GB/s into arrays just allocated, where the link does 57.
// Here a few worker threads each fetch their chunks into two pinned buffers
// of their own and copy them out, so the copies out and the faults run side
// by side with each other and with the link.  A 306 MB field 30.4 -> 11.4 ms
// (27 GB/s), 24 fields of 12 MB 40 -> 12.8 ms, one of 94 MB 9.2 -> 3.2 ms.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace acfd {

class HostCopy {
public:
    // below this many bytes the plain copy is as fast
    static constexpr size_t kMinBytes = 2u << 20;

    ~HostCopy()
    {
        {
            std::lock_guard<std::mutex> g(mu_);
            quit_ = true;
        }
        cv_.notify_all();
        for (auto &t : threads_) t.join();
        for (auto &e : ev_)
            if (e) (void)hipEventDestroy(e);
        if (pinned_) (void)hipHostFree(pinned_);
    }

    // Copy bytes of device memory src, written by work queued on s, to dst
    // and wait for it.  False: nothing was copied (no pinned memory or no
    // threads to be had); err receives a failed copy's error.
    bool fetch(void *dst, const void *src, size_t bytes, hipStream_t s, hipError_t *err)
    {
        if (!start()) return false;
        std::unique_lock<std::mutex> g(mu_);
        dst_ = (char *)dst;
        src_ = (const char *)src;
        bytes_ = bytes;
        stream_ = s;
        err_ = hipSuccess;
        left_ = (int)threads_.size();
        job_++;
        cv_.notify_all();
        done_.wait(g, [&] { return left_ == 0; });
        *err = err_;
        return true;
    }

private:
    static constexpr size_t kChunk = 1u << 20;
    static constexpr int kThreads = 8;

    bool start()
    {
        if (!threads_.empty()) return true;
        if (tried_) return false;
        tried_ = true;
        if (hipGetDevice(&dev_) != hipSuccess) return false;
        if (hipHostMalloc((void **)&pinned_, 2 * kThreads * kChunk, hipHostMallocDefault) != hipSuccess) {
            pinned_ = nullptr;
            (void)hipGetLastError();
            return false;
        }
        for (auto &e : ev_)
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                e = nullptr;
                return false;
            }
        try {
            threads_.reserve(kThreads);
            for (int t = 0; t < kThreads; t++) threads_.emplace_back([this, t] { work(t); });
        } catch (const std::exception &) {
            // fewer threads than asked for: those that run share the chunks
        }
        return !threads_.empty();
    }

    void work(int t)
    {
        (void)hipSetDevice(dev_);
        long seen = 0;
        for (;;) {
            int nt;
            {
                std::unique_lock<std::mutex> g(mu_);
                cv_.wait(g, [&] { return quit_ || job_ != seen; });
                if (quit_) return;
                seen = job_;
                nt = (int)threads_.size();
            }
            const hipError_t e = copy(t, nt);
            std::lock_guard<std::mutex> g(mu_);
            if (e != hipSuccess) err_ = e;
            if (--left_ == 0) done_.notify_one();
        }
    }

    // chunks t, t + nt, ...: the next one in flight while one is copied out
    hipError_t copy(int t, int nt)
    {
        const long n = (long)((bytes_ + kChunk - 1) / kChunk);
        auto len = [&](long c) { return std::min(kChunk, bytes_ - (size_t)c * kChunk); };
        auto issue = [&](long c, int h) {
            const int x = 2 * t + h;
            hipError_t e = hipMemcpyAsync(pinned_ + x * kChunk, src_ + c * kChunk, len(c), hipMemcpyDeviceToHost, stream_);
            return e == hipSuccess ? hipEventRecord(ev_[x], stream_) : e;
        };
        int h = 0;
        hipError_t e = t < n ? issue(t, h) : hipSuccess;
        for (long c = t; c < n && e == hipSuccess; c += nt, h ^= 1) {
            if (c + nt < n) e = issue(c + nt, h ^ 1);
            const hipError_t w = hipEventSynchronize(ev_[2 * t + h]);
            if (w != hipSuccess) return w;
            std::memcpy(dst_ + c * kChunk, pinned_ + (2 * t + h) * kChunk, len(c));
        }
        return e;
    }

    std::vector<std::thread> threads_;
    hipEvent_t ev_[2 * kThreads] = {};
    std::mutex mu_;
    std::condition_variable cv_, done_;
    char *pinned_ = nullptr;
    int dev_ = 0;
    bool tried_ = false, quit_ = false;
    long job_ = 0;
    int left_ = 0;
    char *dst_ = nullptr;
    const char *src_ = nullptr;
    size_t bytes_ = 0;
    hipStream_t stream_ = nullptr;
    hipError_t err_ = hipSuccess;
};

}  // namespace acfd
