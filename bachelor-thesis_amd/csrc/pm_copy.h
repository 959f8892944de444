// pm_copy.h -- host copies from pinned staging into the caller's pageable memory,
// shared by a few threads.
//
// One thread copies 10 to 18 GB/s, less into pages it touches first, a quarter of
// what the DMA engines move, so an image handed to the host is host-copy bound:
// a 640x480 march with its 11 MB of images 1.69 -> 1.26 ms, eight batch views
// (22 MB) 2.21 -> 1.90.  (Frames copied the same way into staging for their
// upload gained 2 % of a streamed frame and cost its first one 6 %: not kept.)
// A context keeps up to three workers beside its calling thread, started by its
// first copy of at least kCopyShared bytes and joined when it is destroyed;
// where none can be started the caller copies alone.  A copy returns when every
// byte is there: nothing runs on after the call.  A context's calls come from
// one thread at a time, so one copy is in flight per pool.
#pragma once

#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>

namespace pm {

static constexpr size_t kCopyShared = 1u << 20;   // below, waking the workers costs what they save
static constexpr size_t kCopyPiece = 256u << 10;

class CopyPool {
  public:
    struct Range {
        void *dst;
        const void *src;
        size_t bytes;
    };

    ~CopyPool()
    {
        {
            std::lock_guard<std::mutex> l(m_);
            stop_ = true;
        }
        wake_.notify_all();
        for (int i = 0; i < workers_; i++) th_[i].join();
    }

    // Copies up to four ranges.
    void copy(const Range *r, int n)
    {
        size_t total = 0;
        bool alone = false;                // destinations that overlap: the later range's bytes stay
        for (int i = 0; i < n; i++) {
            total += r[i].bytes;
            for (int j = 0; j < i; j++) {
                const uintptr_t a = (uintptr_t)r[i].dst, b = (uintptr_t)r[j].dst;
                alone = alone || (a < b + r[j].bytes && b < a + r[i].bytes);
            }
        }
        if (alone || total < kCopyShared || !start()) {
            for (int i = 0; i < n; i++)
                if (r[i].bytes) memcpy(r[i].dst, r[i].src, r[i].bytes);
            return;
        }
        {
            std::lock_guard<std::mutex> l(m_);
            ranges_ = r;
            count_ = n;
            pieces_ = 0;
            for (int i = 0; i < n; i++) pieces_ += pieces(r[i]);
            next_.store(0);
            job_++;
        }
        wake_.notify_all();
        work();
        std::unique_lock<std::mutex> l(m_);
        idle_.wait(l, [this] { return active_ == 0; });
        ranges_ = nullptr;
    }

  private:
    static size_t pieces(const Range &r) { return (r.bytes + kCopyPiece - 1) / kCopyPiece; }

    bool start()
    {
        if (started_) return workers_ > 0;
        started_ = true;
        const unsigned hw = std::thread::hardware_concurrency();
        const int want = hw > 1 ? (int)std::min(3u, hw / 2) : 0;
        try {
            for (; workers_ < want; workers_++) th_[workers_] = std::thread(&CopyPool::run, this);
        } catch (...) {
            // no thread, or no memory for one: as many as there are (nothing may
            // be thrown through the C entry that copies)
        }
        return workers_ > 0;
    }

    void work()
    {
        for (size_t k; (k = next_.fetch_add(1)) < pieces_;) {
            int i = 0;
            while (k >= pieces(ranges_[i])) k -= pieces(ranges_[i++]);
            const size_t o = k * kCopyPiece, b = std::min(kCopyPiece, ranges_[i].bytes - o);
            memcpy((char *)ranges_[i].dst + o, (const char *)ranges_[i].src + o, b);
        }
    }

    void run()
    {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> l(m_);
        while (true) {
            wake_.wait(l, [&] { return stop_ || job_ != seen; });
            if (stop_) return;
            seen = job_;
            if (!ranges_) continue;        // the copy ended before this worker woke
            active_++;
            l.unlock();
            work();
            l.lock();
            if (--active_ == 0) idle_.notify_one();
        }
    }

    std::mutex m_;
    std::condition_variable wake_, idle_;
    std::thread th_[3];
    int workers_ = 0, active_ = 0, count_ = 0;
    bool started_ = false, stop_ = false;
    uint64_t job_ = 0;
    const Range *ranges_ = nullptr;
    size_t pieces_ = 0;
    std::atomic<size_t> next_{ 0 };
};

}  // namespace pm
