// Large results to a caller's pageable array.
//
// The runtime pins the array's pages for the length of the copy: 0.21 ms for
// 3.1 MB, 0.55 ms for 7.9 MB, 1.15 ms for 16 MB into a new array (14 GB/s).
// Through a pinned buffer that is there already, each chunk copied on by the CPU
// while the next ones arrive, the same take 0.15, 0.33 and 0.88 ms.  Chunks of
// 512 KB cost as much again in the gaps between them (0.75 ms for 16 MB into an
// array in use, 0.66 with 1 MB, 0.66 with 2 MB).  Below 1 MB the runtime is the
// faster (1.0 MB: 0.060 against 0.067 ms), and so it is to the device at every
// size (3.1 MB: 0.10 against 0.12 ms).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <memory>
#include <mutex>

namespace pgfd {

// The pinned buffers of all objects: made when a copy first needs one (0.5 to 2
// ms, which an object that copies nothing large is not to pay, nor the first
// copy of every new one), at most MAX, so that as many threads copy at a time,
// and freed with the last object.
class PinnedPool {
public:
    static constexpr size_t CHUNK = 1 << 20;
    static constexpr int SLOTS = 4, MAX = 4;
    static std::shared_ptr<PinnedPool> get() {
        static std::mutex mutex;
        static std::weak_ptr<PinnedPool> pool;
        std::lock_guard<std::mutex> lock(mutex);
        std::shared_ptr<PinnedPool> p = pool.lock();
        if (!p) pool = p = std::make_shared<PinnedPool>();
        return p;
    }
    ~PinnedPool() {
        for (int i = 0; i < idle_; ++i) (void)hipHostFree(buffers_[i]);
    }
    // a buffer of SLOTS chunks, or null: all are in use, or memory is short
    char* take() {
        std::lock_guard<std::mutex> lock(mutex_);
        if (idle_ > 0) return buffers_[--idle_];
        if (made_ == MAX) return nullptr;
        char* p = nullptr;
        if (hipHostMalloc((void**)&p, SLOTS * CHUNK, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        ++made_;
        return p;
    }
    void give(char* p) {
        std::lock_guard<std::mutex> lock(mutex_);
        buffers_[idle_++] = p;
    }

private:
    std::mutex mutex_;
    char* buffers_[MAX] = {};
    int idle_ = 0, made_ = 0;
};

// One per object with a stream; calls from several threads take turns.
class HostCopy {
public:
    HostCopy() : pool_(PinnedPool::get()) {}
    HostCopy(const HostCopy&) = delete;
    HostCopy& operator=(const HostCopy&) = delete;
    ~HostCopy() {
        for (hipEvent_t e : done_)
            if (e) (void)hipEventDestroy(e);
    }
    // n bytes from the device behind what the stream holds; there on return
    hipError_t down(void* dst, const void* src, size_t n, hipStream_t s) {
        if (n <= CHUNK || !pageable(dst)) return plain(dst, src, n, s);
        std::lock_guard<std::mutex> lock(mutex_);
        char* pin = events() ? pool_->take() : nullptr;
        if (!pin) return plain(dst, src, n, s);
        hipError_t e = staged(pin, (char*)dst, (const char*)src, n, s);
        if (e != hipSuccess) (void)hipStreamSynchronize(s);  // nothing still writes the buffer
        pool_->give(pin);
        return e;
    }

private:
    static constexpr size_t CHUNK = PinnedPool::CHUNK, PIECE = 256 << 10;
    static constexpr int SLOTS = PinnedPool::SLOTS;
    static hipError_t plain(void* dst, const void* src, size_t n, hipStream_t s) {
        const hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    hipError_t staged(char* pin, char* dst, const char* src, size_t n, hipStream_t s) {
        const size_t chunks = (n + CHUNK - 1) / CHUNK;
        auto len = [&](size_t i) { return std::min(CHUNK, n - i * CHUNK); };
        auto fetch = [&](size_t i) {
            const int k = (int)(i % SLOTS);
            const hipError_t e = hipMemcpyAsync(pin + k * CHUNK, src + i * CHUNK, len(i), hipMemcpyDeviceToHost, s);
            return e == hipSuccess ? hipEventRecord(done_[k], s) : e;
        };
        hipError_t e = hipSuccess;
        for (size_t i = 0; i < std::min<size_t>(chunks, SLOTS); ++i)
            if ((e = fetch(i)) != hipSuccess) return e;
        for (size_t i = 0; i < chunks; ++i) {
            if ((e = hipEventSynchronize(done_[i % SLOTS])) != hipSuccess) return e;
            move(dst + i * CHUNK, pin + i % SLOTS * CHUNK, len(i));
            if (i + SLOTS < chunks && (e = fetch(i + SLOTS)) != hipSuccess) return e;
        }
        return hipSuccess;
    }
    bool events() {
        for (hipEvent_t& e : done_)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                e = nullptr;
                return false;
            }
        return true;
    }
    // in pieces below the size from which the C library's copy goes past the cache
    static void move(char* dst, const char* src, size_t n) {
        for (size_t at = 0; at < n; at += PIECE) std::memcpy(dst + at, src + at, std::min(PIECE, n - at));
    }
    // (a pinned array, or one the device can reach, needs no staging)
    static bool pageable(const void* p) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();
            return true;
        }
        return a.type == hipMemoryTypeUnregistered;
    }
    std::shared_ptr<PinnedPool> pool_;
    std::mutex mutex_;
    hipEvent_t done_[SLOTS] = {};
};

}  // namespace pgfd
