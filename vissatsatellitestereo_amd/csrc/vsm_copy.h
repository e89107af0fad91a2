// vsm_copy.h -- device-to-host copies into ordinary (pageable) memory.
//
// A copy straight into pageable memory runs at the pace of one host thread
// that also takes the destination's page faults: 10 GB/s into fresh pages.
// CopyRing moves the data by DMA into a ring of pinned slots (57 GB/s) and has
// a few threads move it on to the destination.  172 MB into fresh pages:
// 17.1 -> 4.5 ms; 1 MB: 0.64 -> 0.16 ms (4 threads; 8 and 12 are no faster).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace vsm {

class CopyRing;

// The copies of one call of an entry point.  Calls may run on several host
// threads and share the ring, so what a call has under way and the errors it
// met are its own.  A call that returns early leaves nothing under way into
// the caller's memory: the destructor waits.
class CopyCall {
public:
    CopyCall(CopyRing &ring, int device, hipStream_t st) : ring_(ring), device_(device), st_(st) {}
    CopyCall(const CopyCall &) = delete;
    CopyCall &operator=(const CopyCall &) = delete;
    ~CopyCall()
    {
        if (open_) (void)finish();
    }

    // Queues a copy of n bytes behind the work on the stream.  The data is in
    // dst after finish().  src may be reused by later work on the stream.
    hipError_t copy(void *dst, const void *src, size_t n);

    // Waits for the stream and for the data to be in place.  Returns the
    // first error that the stream or one of this call's copies met.
    hipError_t finish();

private:
    friend class CopyRing;
    CopyRing &ring_;
    int device_;
    hipStream_t st_;
    bool open_ = false;                        // copies queued and not waited for
    bool waited_ = false;                      // the work ahead of the call's first ring copy is done
    int pending_ = 0;                          // of these, in the ring (guarded by its mutex, as error_)
    hipError_t error_ = hipSuccess;
};

// One per context: 16 MiB of pinned memory and four threads, made by the first
// copy that is large enough to gain from them and given back with the context.
// The slots hold what is under way, so nothing is allocated after that.
class CopyRing {
public:
    CopyRing() = default;
    CopyRing(const CopyRing &) = delete;
    CopyRing &operator=(const CopyRing &) = delete;

    ~CopyRing()
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        work_.notify_all();
        for (auto &t : threads_)
            if (t.joinable()) t.join();
        for (int i = 0; i < n_events_; ++i) (void)hipEventDestroy(events_[i]);
        if (pinned_) (void)hipHostFree(pinned_);
    }

private:
    friend class CopyCall;
    // Copies below kDirect go straight (their pages are mostly the heap's,
    // touched before).  1 MB into fresh pages takes 0.64 ms straight and 0.16
    // through the ring; into pages used before the ring pays from about 2 MB on
    // (1.3 MB 0.08 -> 0.10 ms, 4 MB 0.24 -> 0.18).
    static constexpr size_t kPage = 4096, kSlot = 2u << 20, kPiece = 256u << 10, kDirect = 1u << 20;
    static constexpr int kSlots = 8, kThreadCount = 4;

    struct Job {
        CopyCall *call;
        char *dst;
        size_t n;
        int slot;
    };

    hipError_t copy(CopyCall &call, void *dst, const void *src, size_t n)
    {
        if (n < kDirect || mapped(dst) || !ready(call.device_))
            return hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, call.st_);
        // Waiting for an event takes a whole core, so the caller waits for the
        // kernels ahead and the threads only for the DMA (DSM of 40 views, 44 ms:
        // 163 ms of processor time a call where all of them waited).
        if (!call.waited_) {
            const hipError_t e = hipStreamSynchronize(call.st_);
            if (e != hipSuccess) return e;
            call.waited_ = true;
        }
        // pieces of a short copy keep every thread busy; long ones take whole slots
        const size_t piece = std::min(kSlot, std::max(kPiece, (n / kThreadCount + kPage - 1) / kPage * kPage));
        for (size_t off = 0; off < n; off += piece) {
            const size_t m = std::min(piece, n - off);
            int slot;
            {
                std::unique_lock<std::mutex> lk(mu_);
                done_.wait(lk, [this] { return n_free_ > 0; });
                slot = free_[--n_free_];
            }
            hipError_t e = hipMemcpyAsync(pinned_ + (size_t)slot * kSlot, static_cast<const char *>(src) + off, m,
                                          hipMemcpyDeviceToHost, call.st_);
            if (e == hipSuccess) e = hipEventRecord(events_[slot], call.st_);
            {
                std::lock_guard<std::mutex> lk(mu_);
                if (e != hipSuccess) {
                    free_[n_free_++] = slot;
                } else {
                    jobs_[(first_job_ + n_jobs_++) % kSlots] = Job{&call, static_cast<char *>(dst) + off, m, slot};
                    ++call.pending_;
                }
            }
            if (e != hipSuccess) {
                done_.notify_all();
                return e;
            }
            work_.notify_one();
        }
        return hipSuccess;
    }

    hipError_t wait(CopyCall &call)
    {
        std::unique_lock<std::mutex> lk(mu_);
        done_.wait(lk, [&call] { return call.pending_ == 0; });
        const hipError_t e = call.error_;
        call.error_ = hipSuccess;
        return e;
    }

    // Whether the device reaches dst itself (pinned memory): the DMA writes it
    // at 57 GB/s, where the way through the ring took 268 MB 4.8 -> 6.6 ms and
    // 4 MB 0.09 -> 0.18 ms.
    static bool mapped(const void *dst)
    {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, dst) != hipSuccess) {
            (void)hipGetLastError();           // plain host memory, for runtimes that call it an error
            return false;
        }
        return a.type != hipMemoryTypeUnregistered;
    }

    // Makes the ring and the threads once; false where that failed.  The events
    // have to belong to the device of the streams, which need not be the
    // calling thread's.
    bool ready(int device)
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (state_ != 0) return state_ > 0;
        int before = device;
        (void)hipGetDevice(&before);
        (void)hipSetDevice(device);
        state_ = make(device) ? 1 : -1;
        (void)hipSetDevice(before);
        return state_ > 0;
    }

    bool make(int device)
    {
        void *p = nullptr;
        if (hipHostMalloc(&p, kSlots * kSlot, 0) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        pinned_ = static_cast<char *>(p);
        for (; n_events_ < kSlots; ++n_events_)
            if (hipEventCreateWithFlags(&events_[n_events_], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
        try {
            for (auto &t : threads_) t = std::thread([this, device] { run(device); });
        } catch (const std::exception &) {
            if (!threads_[0].joinable()) return false;
        }
        for (; n_free_ < kSlots; ++n_free_) free_[n_free_] = n_free_;
        return true;
    }

    void run(int device)
    {
        (void)hipSetDevice(device);
        std::unique_lock<std::mutex> lk(mu_);
        for (;;) {
            work_.wait(lk, [this] { return stop_ || n_jobs_ > 0; });
            if (n_jobs_ == 0) return;
            const Job j = jobs_[first_job_];
            first_job_ = (first_job_ + 1) % kSlots;
            --n_jobs_;
            lk.unlock();
            const hipError_t e = hipEventSynchronize(events_[j.slot]);
            if (e == hipSuccess) memcpy(j.dst, pinned_ + (size_t)j.slot * kSlot, j.n);
            lk.lock();
            if (e != hipSuccess && j.call->error_ == hipSuccess) j.call->error_ = e;
            --j.call->pending_;
            free_[n_free_++] = j.slot;
            done_.notify_all();
        }
    }

    std::mutex mu_;
    std::condition_variable work_, done_;
    Job jobs_[kSlots];                         // n_jobs_ of them from first_job_ on, wrapping around
    int first_job_ = 0, n_jobs_ = 0;
    int free_[kSlots];
    int n_free_ = 0;
    hipEvent_t events_[kSlots];
    int n_events_ = 0;
    std::thread threads_[kThreadCount];
    char *pinned_ = nullptr;
    int state_ = 0;                            // 0 not made, 1 ready, -1 not available
    bool stop_ = false;
};

inline hipError_t CopyCall::copy(void *dst, const void *src, size_t n)
{
    open_ = true;
    return ring_.copy(*this, dst, src, n);
}

inline hipError_t CopyCall::finish()
{
    const hipError_t e = hipStreamSynchronize(st_);
    const hipError_t w = ring_.wait(*this);
    open_ = false;
    return e != hipSuccess ? e : w;
}

}  // namespace vsm
