// vsm_copy.h -- device-to-host copies into ordinary (pageable) memory.
//
// A copy straight into pageable memory runs at the pace of one host thread
// that also takes the destination's page faults: 10 GB/s into fresh pages.
// CopyOut moves the data by DMA into a ring of pinned slots (57 GB/s) and has
// a few threads move it on to the destination.  172 MB into fresh pages:
// 17.1 -> 4.5 ms; 1 MB: 0.64 -> 0.16 ms (4 threads; 8 and 12 are no faster).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace vsm {

// One per context: 16 MiB of pinned memory and four threads, made by the first
// copy that is large enough to gain from them and given back with the
// context.  Calls may come from several host threads.
class CopyOut {
public:
    CopyOut() = default;
    CopyOut(const CopyOut &) = delete;
    CopyOut &operator=(const CopyOut &) = delete;

    ~CopyOut()
    {
        (void)wait();
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        work_.notify_all();
        for (auto &t : threads_) t.join();
        for (auto &e : events_) (void)hipEventDestroy(e);
        if (pinned_) (void)hipHostFree(pinned_);
    }

    // Queues a copy of n bytes behind the work on stream st.  The data is in
    // dst after wait().  src may be reused by later work on st.
    hipError_t copy(void *dst, const void *src, size_t n, int device, hipStream_t st)
    {
        if (n < kDirect || !ready(device)) return hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, st);
        // pieces of a short copy keep every thread busy; long ones take whole slots
        const size_t piece = std::min(kSlot, std::max(kPiece, (n / kThreadCount + kPage - 1) / kPage * kPage));
        for (size_t off = 0; off < n; off += piece) {
            const size_t m = std::min(piece, n - off);
            int slot;
            {
                std::unique_lock<std::mutex> lk(mu_);
                done_.wait(lk, [this] { return !free_.empty(); });
                slot = free_.back();
                free_.pop_back();
                ++pending_;
            }
            hipError_t e = hipMemcpyAsync(pinned_ + (size_t)slot * kSlot, static_cast<const char *>(src) + off, m,
                                          hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipEventRecord(events_[slot], st);
            {
                std::lock_guard<std::mutex> lk(mu_);
                if (e != hipSuccess) {
                    free_.push_back(slot);
                    --pending_;
                } else {
                    jobs_.push_back(Job{static_cast<char *>(dst) + off, m, slot});
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

    // Waits for the copies queued so far (not for the small ones, which the
    // stream completes).  Returns the first error one of them met.
    hipError_t wait()
    {
        std::unique_lock<std::mutex> lk(mu_);
        done_.wait(lk, [this] { return pending_ == 0; });
        const hipError_t e = error_;
        error_ = hipSuccess;
        return e;
    }

private:
    // Copies below kDirect go straight (their pages are mostly the heap's, touched before).
    static constexpr size_t kPage = 4096, kSlot = 2u << 20, kPiece = 256u << 10, kDirect = 1u << 20;
    static constexpr int kSlots = 8, kThreadCount = 4;

    struct Job {
        char *dst;
        size_t n;
        int slot;
    };

    // Makes the ring and the threads once; false where that failed.
    bool ready(int device)
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (state_ != 0) return state_ > 0;
        state_ = -1;
        void *p = nullptr;
        if (hipHostMalloc(&p, kSlots * kSlot, 0) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        pinned_ = static_cast<char *>(p);
        for (int i = 0; i < kSlots; ++i) {
            hipEvent_t e;
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
            events_.push_back(e);
            free_.push_back(i);
        }
        try {
            for (int i = 0; i < kThreadCount; ++i) threads_.emplace_back([this, device] { run(device); });
        } catch (const std::system_error &) {
            if (threads_.empty()) return false;
        }
        state_ = 1;
        return true;
    }

    void run(int device)
    {
        (void)hipSetDevice(device);
        std::unique_lock<std::mutex> lk(mu_);
        for (;;) {
            work_.wait(lk, [this] { return stop_ || !jobs_.empty(); });
            if (jobs_.empty()) return;
            const Job j = jobs_.front();
            jobs_.pop_front();
            lk.unlock();
            const hipError_t e = hipEventSynchronize(events_[j.slot]);
            if (e == hipSuccess) memcpy(j.dst, pinned_ + (size_t)j.slot * kSlot, j.n);
            lk.lock();
            if (e != hipSuccess && error_ == hipSuccess) error_ = e;
            free_.push_back(j.slot);
            --pending_;
            done_.notify_all();
        }
    }

    std::mutex mu_;
    std::condition_variable work_, done_;
    std::deque<Job> jobs_;
    std::vector<int> free_;
    std::vector<hipEvent_t> events_;
    std::vector<std::thread> threads_;
    char *pinned_ = nullptr;
    int pending_ = 0, state_ = 0;              // state_: 0 not made, 1 ready, -1 not available
    bool stop_ = false;
    hipError_t error_ = hipSuccess;
};

}  // namespace vsm
