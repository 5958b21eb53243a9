/* Host-side copies by several threads: one core copies about 20 GB/s, less
 * than half of what the link to the device takes in either direction. */
#ifndef CUDEC_AMD_HOST_COPY_H
#define CUDEC_AMD_HOST_COPY_H

#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <mutex>
#include <thread>
#include <vector>

namespace cudec_amd {

/* Threads of one call, started with it and joined at its end: nothing is
 * left running, and calls on other threads have their own. With no helpers
 * (small calls, one core, threads refused) the caller does everything. */
class CopyCrew {
public:
    static constexpr size_t kBytesPerHelper = size_t{8} << 20;

    /* `bytes`: what the call copies in all, of `items` of about one size. A
     * helper costs about 20 us to start, and more than seven do not copy
     * faster. */
    CopyCrew(size_t bytes, size_t items) : step_(step_of(bytes, items)) {
        const size_t most = bytes / kBytesPerHelper < kMostHelpers ? bytes / kBytesPerHelper
                                                                   : kMostHelpers;
        const size_t cores = std::thread::hardware_concurrency();
        const size_t helpers = cores > 1 && most > cores - 1 ? cores - 1 : cores > 1 ? most : 0;
        try {
            threads_.reserve(helpers);
            for (size_t i = 0; i < helpers; i++) {
                threads_.emplace_back([this] { help(); });
            }
        } catch (...) { /* with those that started */
        }
    }
    ~CopyCrew() {
        {
            std::lock_guard<std::mutex> hold(lock_);
            quit_ = true;
        }
        wake_.notify_all();
        for (std::thread& t : threads_) {
            t.join();
        }
    }
    CopyCrew(const CopyCrew&) = delete;
    CopyCrew& operator=(const CopyCrew&) = delete;

    /* work(i) for every i below n, on any of the threads; work does not
     * throw. Returns when all are done. Allocates nothing: it runs while
     * transfers are in flight, where a failure has to drain them first. */
    template <class Work>
    void each(size_t n, const Work& work) {
        if (threads_.empty()) {
            for (size_t i = 0; i < n; i++) {
                work(i);
            }
            return;
        }
        {
            std::lock_guard<std::mutex> hold(lock_);
            work_ = &work;
            call_ = [](const void* w, size_t i) { (*static_cast<const Work*>(w))(i); };
            count_ = n;
            next_.store(0);
            busy_ = threads_.size();
            round_++;
        }
        wake_.notify_all();
        claim(n, call_, work_);
        std::unique_lock<std::mutex> hold(lock_);
        idle_.wait(hold, [this] { return busy_ == 0; });
    }

private:
    static constexpr size_t kMostHelpers = 7;

    using Call = void (*)(const void* work, size_t i);

    /* Items that a thread takes at once: kClaimBytes of them, since threads
     * that ask one counter for 1.6 KiB each wait for the counter (20 000 such
     * chunks to the device through a kept context: 3.3 ms one by one, 1.2
     * so; to the host 6.0 and 2.4). */
    static constexpr size_t kClaimBytes = size_t{64} << 10;
    static size_t step_of(size_t bytes, size_t items) {
        const size_t each = items == 0 ? 0 : bytes / items;
        return each >= kClaimBytes ? 1 : kClaimBytes / (each + 1) + 1;
    }
    void claim(size_t n, Call call, const void* work) {
        for (size_t from = next_.fetch_add(step_); from < n; from = next_.fetch_add(step_)) {
            const size_t to = n - from < step_ ? n : from + step_;
            for (size_t i = from; i < to; i++) {
                call(work, i);
            }
        }
    }
    void help() {
        size_t seen = 0;
        std::unique_lock<std::mutex> hold(lock_);
        for (;;) {
            wake_.wait(hold, [&] { return quit_ || round_ != seen; });
            if (quit_) {
                return;
            }
            seen = round_;
            const size_t n = count_;
            const Call call = call_;
            const void* const work = work_;
            hold.unlock();
            claim(n, call, work);
            hold.lock();
            if (--busy_ == 0) {
                idle_.notify_one();
            }
        }
    }

    const size_t step_;
    std::mutex lock_;
    std::condition_variable wake_, idle_;
    const void* work_ = nullptr;
    Call call_ = nullptr;
    size_t count_ = 0, round_ = 0, busy_ = 0;
    std::atomic<size_t> next_{0};
    bool quit_ = false;
    std::vector<std::thread> threads_;
};

}  // namespace cudec_amd

#endif /* CUDEC_AMD_HOST_COPY_H */
