// Copies between the caller's memory and the GPU.
//
// A copy to or from memory that is not pinned goes through the runtime's own
// staging, or pins the caller's pages for the copy: 8 KB take 15 us in and 24 us
// out, 64 KB 34 and 75, 1 MB 51 and 62.  Through memory that is pinned once they
// take 12, 9 and 38 us (the processor's copy included).  Larger copies go
// directly: 4 MB take 131 us in and 239 out, staged 135 either way, and the
// staging memory's own first touch costs 50 us per MB.  A large result into fresh
// memory is bound by its pages' first touch (62 MB: 15.9 ms, 3.7 into memory in
// use), so the pages of fresh memory are made present before the wait for the
// GPU's work, beside which that costs nothing.  (For memory in use the walk over
// its pages alone would cost 10 us of a 2 MB result's 115.)  Memory that the runtime knows (pinned by the
// caller, or a device's) is copied directly: through staging memory 1 MB of pinned
// memory took 51 us in and 57 out, directly 28 and 27.
#pragma once

#include <hip/hip_runtime.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <cstring>

namespace sw1d {

// One object's staging memory (one thread at a time, like the object).  The
// caller's memory has been read, and holds the results, when finish() returns.
class HostStage {
public:
    static constexpr size_t kMost = 1u << 20;

    HostStage() = default;
    ~HostStage()
    {
        if (p_) (void)hipHostFree(p_);
    }
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    // For `most` bytes, of all copies between two calls of finish(), or of those
    // that come first where that is more than kMost.  The memory is allocated by
    // the first copy after two rounds (15 to 50 us, and its first touch): an
    // object whose state goes in and out once is as fast without it, one whose
    // state stays on the GPU needs none.  While another thread captures a stream
    // in the strictest mode that fails, as the copy's wait always has.
    void reserve(size_t most) { cap_ = std::min(kMost, round(most)); }

    hipError_t up(void* dev, const void* host, size_t bytes, hipStream_t s)
    {
        const size_t at = take(host, bytes);
        if (at == kNone) return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
        memcpy(p_ + at, host, bytes);
        return hipMemcpyAsync(dev, p_ + at, bytes, hipMemcpyHostToDevice, s);
    }

    hipError_t down(void* host, const void* dev, size_t bytes, hipStream_t s)
    {
        const size_t at = count_ < kPending ? take(host, bytes) : kNone;
        if (at == kNone && bytes >= kPopulate && !known(host)) populate(host, bytes);
        const hipError_t e = hipMemcpyAsync(at == kNone ? host : p_ + at, dev, bytes, hipMemcpyDeviceToHost, s);
        if (e != hipSuccess)
            count_ = 0;  // the call fails: its earlier results are not handed over
        else if (at != kNone)
            pending_[count_++] = {host, at, bytes};
        return e;
    }

    // Waits for the stream and hands the results over.
    hipError_t finish(hipStream_t s)
    {
        const hipError_t e = hipStreamSynchronize(s);
        for (int i = 0; i < count_ && e == hipSuccess; ++i)
            memcpy(pending_[i].host, p_ + pending_[i].at, pending_[i].bytes);
        count_ = 0;
        used_ = 0;
        if (rounds_ < 2) ++rounds_;
        return e;
    }

private:
    static constexpr size_t kNone = ~(size_t)0, kPopulate = 256u << 10;
    static constexpr int kPending = 4;
    struct Pending { void* host; size_t at, bytes; };

    static size_t round(size_t n) { return (n + 4095) & ~(size_t)4095; }
    // 0.1 us
    static bool known(const void* host)
    {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, host) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
        (void)hipGetLastError();
        return false;
    }
    // offset of `bytes` free bytes for a copy to or from `host`; none until finish()
    // where they do not fit
    size_t take(const void* host, size_t bytes)
    {
        if (used_ + bytes > cap_ || (!p_ && rounds_ < 2) || known(host)) return kNone;
        if (!p_ && hipHostMalloc((void**)&p_, cap_, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            p_ = nullptr;
            cap_ = 0;
            return kNone;
        }
        const size_t at = used_;
        used_ = std::min(cap_, at + round(bytes));
        return at;
    }
    // Makes the whole pages of [host, host + bytes) present and writable, their
    // contents as they are, unless the first, the middle and the last one are
    // present already (0.5 us); where the kernel does not know the call, the copy
    // faults them in one by one.
    static void populate(void* host, size_t bytes)
    {
#ifdef MADV_POPULATE_WRITE
        constexpr int advice = MADV_POPULATE_WRITE;
#else
        constexpr int advice = 23;  // MADV_POPULATE_WRITE, Linux 5.14
#endif
        const size_t page = (size_t)sysconf(_SC_PAGESIZE), a = reinterpret_cast<size_t>(host);
        const size_t lo = (a + page - 1) & ~(page - 1), hi = (a + bytes) & ~(page - 1);
        if (hi <= lo) return;
        auto present = [&](size_t at) {
            unsigned char v = 0;
            return mincore(reinterpret_cast<void*>(at), page, &v) == 0 && (v & 1);
        };
        if (present(lo) && present(lo + (hi - lo) / page / 2 * page) && present(hi - page)) return;
        (void)madvise(reinterpret_cast<void*>(lo), hi - lo, advice);
    }

    char* p_ = nullptr;
    size_t cap_ = 0, used_ = 0;
    Pending pending_[kPending];
    int count_ = 0, rounds_ = 0;
};

}  // namespace sw1d
