// dev_cache.cpp -- device memory kept between runs (dev_cache.hpp).
#include "dev_cache.hpp"

#include <hip/hip_runtime.h>
#include <unistd.h>

#include <algorithm>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace cir {

namespace {

constexpr size_t kMinBlock = size_t(1) << 20;  // smaller blocks are not kept

using Clock = std::chrono::steady_clock;

struct Block {
    void* p;
    size_t cap;
    int dev;
    Clock::time_point when;
};

class DevCache {
   public:
    ~DevCache() {
        if (thread_.joinable() && getpid() != pid_) {  // a forked child has no such thread
            thread_.detach();
            return;
        }
        {
            std::lock_guard<std::mutex> g(mu_);
            stop_ = true;
        }
        cv_.notify_all();
        if (thread_.joinable()) thread_.join();
        // (what is still kept goes with the process)
    }

    bool take(size_t n, int dev, void** p, size_t* cap) {
        std::lock_guard<std::mutex> g(mu_);
        auto best = blocks_.end();
        for (auto q = blocks_.begin(); q != blocks_.end(); ++q)
            if (q->dev == dev && q->cap >= n && q->cap - n <= n / 4 && (best == blocks_.end() || q->cap < best->cap)) best = q;
        if (best == blocks_.end()) return false;
        *p = best->p;
        *cap = best->cap;
        blocks_.erase(best);
        return true;
    }

    // Keeps the block; what no longer fits the device's bound, oldest first,
    // is returned to be freed.
    std::vector<Block> keep(const Block& b, size_t bound) {
        std::vector<Block> out;
        std::lock_guard<std::mutex> g(mu_);
        if (stop_ || b.cap > bound) return {b};
        out.reserve(blocks_.size() + 1);
        blocks_.reserve(blocks_.size() + 1);
        if (!thread_.joinable()) {
            thread_ = std::thread([this] { expire(); });
            pid_ = getpid();
        }
        blocks_.push_back(b);  // in order of time
        size_t sum = held(b.dev);
        for (auto q = blocks_.begin(); q != blocks_.end() && sum > bound;) {
            if (q->dev != b.dev) {
                ++q;
                continue;
            }
            sum -= q->cap;
            out.push_back(*q);
            q = blocks_.erase(q);
        }
        cv_.notify_all();
        return out;
    }

    bool oldest(int dev, Block* b) {
        std::lock_guard<std::mutex> g(mu_);
        for (auto q = blocks_.begin(); q != blocks_.end(); ++q)
            if (q->dev == dev) {
                *b = *q;
                blocks_.erase(q);
                return true;
            }
        return false;
    }

    size_t bytes(int dev) {
        std::lock_guard<std::mutex> g(mu_);
        return held(dev);
    }

   private:
    size_t held(int dev) const {
        size_t s = 0;
        for (const Block& q : blocks_) s += q.dev == dev ? q.cap : 0;
        return s;
    }

    // Frees what has not been used for kCacheIdleSeconds.
    void expire() {
        // (another thread may be recording a graph meanwhile)
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        std::unique_lock<std::mutex> g(mu_);
        while (!stop_) {
            if (blocks_.empty()) {
                cv_.wait(g);
                continue;
            }
            const Clock::time_point due = blocks_.front().when + std::chrono::seconds(kCacheIdleSeconds);
            if (Clock::now() < due) {
                cv_.wait_until(g, due);
                continue;
            }
            const Block b = blocks_.front();
            blocks_.erase(blocks_.begin());
            g.unlock();
            (void)hipFree(b.p);
            g.lock();
        }
    }

    std::mutex mu_;
    std::condition_variable cv_;
    std::vector<Block> blocks_;  // by time given back, oldest first
    std::thread thread_;
    bool stop_ = false;
    pid_t pid_ = 0;  // of the process that started the thread
};

DevCache& cache() {
    static DevCache c;
    return c;
}

}  // namespace

int dev_cache_alloc(void** p, size_t n, size_t* cap, int* dev) {
    *p = nullptr;
    hipError_t e = hipGetDevice(dev);
    if (e != hipSuccess) return int(e);
    if (n >= kMinBlock && cache().take(n, *dev, p, cap)) return int(hipSuccess);
    *cap = n;
    e = hipMalloc(p, n);
    if (e != hipSuccess) *p = nullptr;
    return int(e);
}

void dev_cache_free(void* p, size_t cap, int dev) {
    int cur = -1;
    size_t fr = 0, tot = 0;
    if (cap < kMinBlock || hipGetDevice(&cur) != hipSuccess || cur != dev || hipMemGetInfo(&fr, &tot) != hipSuccess ||
        fr < tot / 4) {
        (void)hipFree(p);
        return;
    }
    std::vector<Block> out;
    try {
        out = cache().keep(Block{p, cap, dev, Clock::now()}, tot / 8);
    } catch (...) {  // no memory or no thread to keep it with (nothing was kept)
        (void)hipFree(p);
    }
    for (const Block& b : out) (void)hipFree(b.p);
}

void dev_cache_release() {
    int dev = 0;
    Block b;
    if (hipGetDevice(&dev) == hipSuccess)
        while (cache().oldest(dev, &b)) (void)hipFree(b.p);
}

size_t dev_cache_bytes() {
    int dev = 0;
    return hipGetDevice(&dev) == hipSuccess ? cache().bytes(dev) : 0;
}

}  // namespace cir
