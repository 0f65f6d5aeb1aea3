// host_team.h -- a few host threads that work on one array together, for the
// length of a call.  Host only.
#pragma once
#include <algorithm>
#include <atomic>
#include <thread>
#include <vector>

namespace vpm {

// run(job) calls job(w, n) for every worker w < n of the team, on its own
// thread (w = 0 on the caller's), and returns when all have returned.  Jobs
// must not throw.  Threads live as long as the team; a thread that cannot be
// started leaves a smaller team.
class HostTeam {
public:
    explicit HostTeam(int want)
    {
        try {
            threads_.reserve((size_t)std::max(0, want - 1));
            for (int w = 1; w < want; ++w) threads_.emplace_back([this, w] { work(w); });
        } catch (const std::exception&) {   // fewer threads
        }
        size_ = (int)threads_.size() + 1;
    }
    ~HostTeam()
    {
        stop_ = true;
        go_.fetch_add(1, std::memory_order_release);
        for (std::thread& t : threads_) t.join();
    }
    HostTeam(const HostTeam&) = delete;
    HostTeam& operator=(const HostTeam&) = delete;

    template <class F>
    void run(F&& job)
    {
        struct Call { F* f; } c{&job};
        ctx_ = &c;
        call_ = [](void* p, int w, int n) { (*((Call*)p)->f)(w, n); };
        left_.store(size_ - 1, std::memory_order_relaxed);
        go_.fetch_add(1, std::memory_order_release);
        job(0, size_);
        while (left_.load(std::memory_order_acquire) > 0) std::this_thread::yield();
    }

private:
    void work(int w)
    {
        for (unsigned seen = 0;;) {
            unsigned g;
            while ((g = go_.load(std::memory_order_acquire)) == seen) std::this_thread::yield();
            seen = g;
            if (stop_) return;
            call_(ctx_, w, size_);
            left_.fetch_sub(1, std::memory_order_release);
        }
    }
    std::vector<std::thread> threads_;
    std::atomic<unsigned> go_{0};
    std::atomic<int> left_{0};
    bool stop_ = false;
    void* ctx_ = nullptr;
    void (*call_)(void*, int, int) = nullptr;
    int size_ = 1;
};

// Workers for a copy of `bytes` that runs beside the device's.  Starting a
// thread costs the call 15-20 us; rows of 30,011 / 262,144 particles (3.6 / 31
// MB) reach the caller in 155 / 2,300 us with one worker, 174 / 1,400 with two,
// 152 / 1,000 with four and 230 / 1,000 with eight.
inline int team_size(size_t bytes)
{
    const int most = (int)std::max(1u, std::thread::hardware_concurrency());
    return std::min(most, bytes < ((size_t)8 << 20) ? 1 : bytes < ((size_t)16 << 20) ? 2 : bytes < ((size_t)128 << 20) ? 4 : 8);
}

}  // namespace vpm
