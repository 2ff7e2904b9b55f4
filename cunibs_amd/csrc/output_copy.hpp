// Large device-to-host copies into the caller's pageable arrays.
//
// A plain copy is bound by one thread that moves the runtime's staging buffer into the destination
// and takes its page faults (a fresh NumPy array's pages are zeroed at that first touch): about
// 10 GB/s, 6.0 of the 10.4 ms of a five-placement block with its fields at 127k nodes (7.5 ms now; a
// twelve-placement block with |E| 10.8 to 9.2 ms, one placement at 428k nodes 7.0 to 6.1). Here the
// bytes go through a ring of pinned chunks: the GPU fills the chunks in order, and worker threads
// empty them side by side.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "common.hpp"

namespace cn {

class OutputCopy {
  public:
    OutputCopy() = default;
    OutputCopy(const OutputCopy&) = delete;
    OutputCopy& operator=(const OutputCopy&) = delete;
    ~OutputCopy() {
        for (auto& e : ev_)
            if (e) (void)hipEventDestroy(e);
        if (ring_) (void)hipHostFree(ring_);
    }

    // dst (host) = src (device), `bytes` long, after the work queued on `s`; complete on return.
    void run(void* dst, const void* src, std::size_t bytes, hipStream_t s) {
        if (bytes < kMinBytes || !pinned()) {
            if (bytes) check(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s), "output copy");
            sync(s, "output copy");
            return;
        }
        for (auto& e : ev_)
            if (!e) check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "output event");
        const std::size_t n = (bytes + kChunk - 1) / kChunk;
        Ring r(static_cast<char*>(dst), ring_, bytes, n);
        std::size_t issued = 0;
        for (std::size_t i = 0; i < n; ++i) {
            // Every chunk whose slot is empty; at least chunk i (its slot's last user is waited for).
            while (issued < n && (issued < kSlots || r.emptied(issued - kSlots, issued == i))) {
                const std::size_t at = issued * kChunk, slot = issued % kSlots;
                check(hipMemcpyAsync(ring_ + slot * kChunk, static_cast<const char*>(src) + at,
                                     std::min(kChunk, bytes - at), hipMemcpyDeviceToHost, s),
                      "output copy");
                check(hipEventRecord(ev_[slot], s), "output event");
                ++issued;
            }
            check(hipEventSynchronize(ev_[i % kSlots]), "output copy");
            r.filled();
        }
        r.finish();
    }

  private:
    // The ring, allocated at its first use; where there is no pinned memory to be had the copy is plain.
    bool pinned() {
        void* p = nullptr;
        if (!ring_ && hipHostMalloc(&p, kChunk * kSlots) == hipSuccess) ring_ = static_cast<char*>(p);
        if (!ring_) (void)hipGetLastError();
        return ring_ != nullptr;
    }
    // 1 MB chunks take the link 20 us and a worker up to 0.2 ms with their page faults.
    static constexpr std::size_t kChunk = std::size_t{1} << 20;
    static constexpr std::size_t kSlots = 12;
    // Below this the threads' start (about 0.1 ms together) is not worth it.
    static constexpr std::size_t kMinBytes = std::size_t{4} << 20;
    static constexpr int kWorkers = 6;

    // One copy's hand-over between the thread that drives the GPU and its workers. The destructor
    // ends and joins the workers on every path.
    class Ring {
      public:
        Ring(char* dst, const char* ring, std::size_t bytes, std::size_t n)
            : dst_(dst), ring_(ring), bytes_(bytes), done_(n, 0) {
            const int want = static_cast<int>(std::min<std::size_t>(kWorkers, n));
            workers_.reserve(static_cast<std::size_t>(want));
            try {
                for (int w = 0; w < want; ++w) workers_.emplace_back([this] { work(); });
            } catch (...) {
                // No thread or no memory for one: with fewer, or none, finish() and emptied() copy on this
                // one. (Left to itself the exception would meet threads that are running.)
            }
        }
        ~Ring() {
            {
                std::lock_guard<std::mutex> g(m_);
                stop_ = true;
            }
            cv_.notify_all();
            for (auto& w : workers_) w.join();
        }
        void filled() {
            {
                std::lock_guard<std::mutex> g(m_);
                ++ready_;
            }
            cv_.notify_one();
        }
        // Whether chunk i has left its slot; with `wait`, until it has.
        bool emptied(std::size_t i, bool wait) {
            std::unique_lock<std::mutex> g(m_);
            if (!wait) return done_[i] != 0;
            drain(g, [&] { return done_[i] != 0; });
            return true;
        }
        void finish() {
            std::unique_lock<std::mutex> g(m_);
            drain(g, [&] { return count_ == done_.size(); });
        }

      private:
        // Helps with the chunks that are ready until `until` holds.
        template <typename F>
        void drain(std::unique_lock<std::mutex>& g, F&& until) {
            while (!until()) {
                if (next_ < ready_)
                    copy(g);
                else
                    emptied_.wait(g);
            }
        }
        void work() {
            std::unique_lock<std::mutex> g(m_);
            for (;;) {
                cv_.wait(g, [&] { return stop_ || next_ < ready_; });
                if (stop_) return;
                copy(g);
            }
        }
        void copy(std::unique_lock<std::mutex>& g) {
            const std::size_t i = next_++, at = i * kChunk;
            g.unlock();
            std::memcpy(dst_ + at, ring_ + (i % kSlots) * kChunk, std::min(kChunk, bytes_ - at));
            g.lock();
            done_[i] = 1;
            ++count_;
            emptied_.notify_all();
        }

        char* const dst_;
        const char* const ring_;
        const std::size_t bytes_;
        std::vector<char> done_;
        std::size_t ready_ = 0, next_ = 0, count_ = 0;
        bool stop_ = false;
        std::mutex m_;
        std::condition_variable cv_, emptied_;
        std::vector<std::thread> workers_;
    };

    char* ring_ = nullptr;
    hipEvent_t ev_[kSlots] = {};
};

}  // namespace cn
