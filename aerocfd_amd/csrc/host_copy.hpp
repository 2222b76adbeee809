// Device to pageable host memory for large fields (acfd_download).
//
// hipMemcpy to pageable memory goes through the runtime's pinned buffer and
// one thread's copy out of it, which also takes the page faults of a fresh
// destination: 8-11 GB/s into arrays just allocated, where the link does 57.
// Here a few worker threads each fetch their chunks into two pinned buffers
// of their own and copy them out, so the copies out and the faults run side
// by side with each other and with the link.  A 306 MB field 30.4 -> 11.4 ms
// (27 GB/s), 24 fields of 12 MB 40 -> 12.8 ms, one of 94 MB 9.2 -> 3.2 ms.
// A pinned destination goes without: the plain copy has the link's rate
// there (84 MB: 55 GB/s, through the threads 31).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace acfd {

class HostCopy {
public:
    // The current device's threads and buffers, which its contexts share; the
    // last one to let go ends them.  Null without memory.
    static std::shared_ptr<HostCopy> of_device()
    {
        static std::mutex mu;
        static std::vector<std::weak_ptr<HostCopy>> all;
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0) return nullptr;
        try {
            std::lock_guard<std::mutex> g(mu);
            if ((size_t)dev >= all.size()) all.resize(dev + 1);
            std::shared_ptr<HostCopy> h = all[dev].lock();
            if (!h) all[dev] = h = std::make_shared<HostCopy>();
            return h;
        } catch (const std::exception &) {
            return nullptr;
        }
    }

    // whether a copy of bytes to dst gains by it: below 2 MiB, and to pinned
    // memory, the plain copy is as fast or faster
    static bool worth(const void *dst, size_t bytes)
    {
        if (bytes < kMinBytes) return false;
        for (const char *p : {(const char *)dst, (const char *)dst + bytes - 1}) {
            hipPointerAttribute_t a{};
            if (hipPointerGetAttributes(&a, p) != hipSuccess) {
                (void)hipGetLastError();  // not known to the runtime: pageable
                return true;
            }
            if (a.type == hipMemoryTypeUnregistered) return true;
        }
        return false;
    }

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
    // threads to be had); err receives a failed copy's error.  Callers take
    // turns.
    bool fetch(void *dst, const void *src, size_t bytes, hipStream_t s, hipError_t *err)
    {
        std::lock_guard<std::mutex> turn(turn_);
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
    static constexpr size_t kMinBytes = 2u << 20;
    static constexpr size_t kChunk = 1u << 20;
    static constexpr int kThreads = 8;  // at most, and no more than the process has processors

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
            const int n = std::max(1, std::min(kThreads, (int)std::thread::hardware_concurrency()));
            for (int t = 0; t < n; t++) threads_.emplace_back([this, t] { work(t); });
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
            if (w != hipSuccess) {
                (void)hipStreamSynchronize(stream_);  // a copy into the other buffer may be under way
                return w;
            }
            std::memcpy(dst_ + c * kChunk, pinned_ + (2 * t + h) * kChunk, len(c));
        }
        return e;
    }

    std::vector<std::thread> threads_;
    hipEvent_t ev_[2 * kThreads] = {};
    std::mutex turn_, mu_;
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
