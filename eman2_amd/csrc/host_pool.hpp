// What reconstructor handles share on the host side: device blocks, streams
// and pinned staging buffers of destroyed handles, kept for the next ones, and
// the threads that copy between pinned and caller memory.  A serving job
// creates and destroys a handle; every hipFree of it waited for the other
// jobs' kernels, and a stream takes milliseconds to create.
//
// Everything here lives while a handle or a server does (HostPool::Ref): the
// last one to go gives it all back.  Kept blocks are bounded (KEEP_DEVICE
// bytes per device, KEEP_STREAMS, KEEP_PINNED): the ones given back last stay,
// so that sizes which do not come again make room.  They are released when an
// allocation fails, stay within the budget of every server of the device, and
// give way where the device is nearly full; fh_trim gives them all back.  All
// calls may come from any thread; the lock is held for
// the bookkeeping only, not over calls of the runtime, which may wait for other
// handles' kernels.  Nothing is thrown.  Who gives a block back has waited for
// the work that uses it.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <utility>
#include <vector>

namespace fh {

// Threads that share one memcpy: segments of 512 KB, the caller takes part.
class CopyThreads {
public:
    ~CopyThreads()
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            stop_ = true;
        }
        cv_.notify_all();
        for (auto &t : threads_) t.join();
    }

    void copy(char *dst, const char *src, size_t len)
    {
        if (len < (1u << 20)) {
            memcpy(dst, src, len);
            return;
        }
        std::shared_ptr<Job> job;
        try {
            job = std::make_shared<Job>();
            job->dst = dst;
            job->src = src;
            job->len = len;
            job->nseg = (len + SEG - 1) / SEG;
            std::lock_guard<std::mutex> lk(mu_);
            jobs_.push_back(job);
            try {
                while (threads_.size() < THREADS) threads_.emplace_back([this] { work(); });
            } catch (...) {
                // no (more) threads: the caller copies what they do not
            }
        } catch (...) {  // no memory for the job: the caller copies all
            memcpy(dst, src, len);
            return;
        }
        cv_.notify_all();
        job->run();
        std::unique_lock<std::mutex> lk(mu_);
        done_.wait(lk, [&] { return job->done.load() == job->nseg; });
        for (size_t i = 0; i < jobs_.size(); i++)
            if (jobs_[i] == job) {
                jobs_.erase(jobs_.begin() + i);
                break;
            }
    }

private:
    static constexpr size_t SEG = 512u << 10, THREADS = 7;
    struct Job {
        char *dst;
        const char *src;
        size_t len, nseg;
        std::atomic<size_t> next{0}, done{0};
        bool run()  // true: this call finished the last segment
        {
            bool last = false;
            for (size_t s; (s = next.fetch_add(1)) < nseg;) {
                const size_t a = s * SEG, n = std::min(SEG, len - a);
                memcpy(dst + a, src + a, n);
                last = done.fetch_add(1) + 1 == nseg || last;
            }
            return last;
        }
    };

    void work()
    {
        std::unique_lock<std::mutex> lk(mu_);
        for (;;) {
            std::shared_ptr<Job> job;
            cv_.wait(lk, [&] {
                for (auto &j : jobs_)
                    if (j->next.load() < j->nseg) {
                        job = j;
                        return true;
                    }
                return stop_;
            });
            if (!job) return;
            lk.unlock();
            const bool last = job->run();
            lk.lock();
            if (last) done_.notify_all();
        }
    }

    std::mutex mu_;
    std::condition_variable cv_, done_;
    std::vector<std::thread> threads_;
    std::vector<std::shared_ptr<Job>> jobs_;
    bool stop_ = false;
};

class HostPool {
public:
    using Ref = std::shared_ptr<HostPool>;
    static constexpr size_t KEEP_DEVICE = 8ull << 30, KEEP_STREAMS = 16, KEEP_PINNED = 4;
    static constexpr size_t SMALL_BYTES = 64u << 20;  // in copies of less than a slot, before the pool's first ring
    static constexpr size_t LARGE = 32ull << 20;  // from here on a block is kept by what the device has left
    static constexpr size_t PIN_SLOTS = 4, PIN_SLOT = 16u << 20;  // a staging ring: 4 slots of 16 MB

    static Ref get(bool make = true)
    {
        static std::mutex mu;
        static std::weak_ptr<HostPool> pool;
        std::lock_guard<std::mutex> lk(mu);
        Ref r = pool.lock();
        if (!r && make) pool = r = std::make_shared<HostPool>();
        return r;
    }

    HostPool()
    {
        streams_.reserve(KEEP_STREAMS);  // giving back never allocates
        pinned_.reserve(KEEP_PINNED);
    }
    ~HostPool()
    {
        for (auto &d : dev_)
            for (auto &b : d.second.blocks)
                if (b.second.idle) (void)hipFree(b.first);
        for (char *p : pinned_) (void)hipHostFree(p);
        for (auto &s : streams_) (void)hipStreamDestroy(s.second);
    }

    // `bytes` on the current device `device`: a kept block of at most a quarter more, or a new one
    hipError_t alloc(int device, void **p, size_t bytes) noexcept
    {
        bytes = std::max<size_t>(bytes, 256);
        try {
            std::unique_lock<std::mutex> lk(mu_);
            Device &d = dev_[device];
            auto best = d.blocks.end();
            for (auto it = d.blocks.begin(); it != d.blocks.end(); ++it)
                if (it->second.idle && it->second.size >= bytes && it->second.size <= bytes + bytes / 4 + 4096 &&
                    (best == d.blocks.end() || it->second.size < best->second.size))
                    best = it;
            if (best != d.blocks.end()) {
                best->second.idle = false;
                best->second.asked = bytes;
                d.idle -= best->second.size;
                d.spare += best->second.size - bytes;
                *p = best->first;
                return hipSuccess;
            }
            lk.unlock();
            hipError_t e = hipMalloc(p, bytes);
            if (e == hipErrorOutOfMemory) {
                (void)hipGetLastError();
                lk.lock();
                shrink(lk, d, 0);
                freed_.wait(lk, [this] { return freeing_ == 0; });
                lk.unlock();
                e = hipMalloc(p, bytes);
            }
            if (e != hipSuccess) return e;
            lk.lock();
            try {
                d.blocks.emplace(*p, Block{bytes, bytes, 0, false});
            } catch (...) {
                lk.unlock();
                (void)hipFree(*p);
                throw;
            }
            return hipSuccess;
        } catch (...) {
            return hipErrorOutOfMemory;
        }
    }

    void free(int device, void *p) noexcept
    {
        std::unique_lock<std::mutex> lk(mu_);
        Device &d = dev_.find(device)->second;
        Block &b = d.blocks.find(p)->second;
        d.spare -= b.size - b.asked;
        b.asked = b.size;
        size_t most = KEEP_DEVICE;
        if (b.size >= LARGE) {
            // beside other programs, and other allocators of this one, that fill the device: at most a third of
            // what it has left (2 us)
            size_t left = 0, total = 0;
            lk.unlock();
            if (hipMemGetInfo(&left, &total) == hipSuccess) most = left / 3;
            lk.lock();
        }
        most = std::min(most, keep(device, d));
        if (b.size > most) {
            d.blocks.erase(p);
            release(lk, p);
            return;
        }
        b.idle = true;
        b.since = ++clock_;
        d.idle += b.size;
        shrink(lk, d, most);
    }

    // the idle blocks back to the device
    void trim(int device) noexcept
    {
        std::unique_lock<std::mutex> lk(mu_);
        auto it = dev_.find(device);
        if (it != dev_.end()) shrink(lk, it->second, 0);
    }

    // While `owner` has a limit, the device bytes that no handle asked for (idle blocks, and the rest of
    // blocks larger than asked) stay within it: a server's budget less what it has committed to its jobs.
    void limit(const void *owner, int device, long long bytes)
    {
        std::unique_lock<std::mutex> lk(mu_);
        limits_[owner] = {device, bytes};
        Device &d = dev_[device];
        shrink(lk, d, keep(device, d));
    }
    void change_limit(const void *owner, long long by) noexcept
    {
        std::unique_lock<std::mutex> lk(mu_);
        auto it = limits_.find(owner);
        it->second.second += by;
        const int device = it->second.first;
        Device &d = dev_.find(device)->second;
        shrink(lk, d, keep(device, d));
    }
    void no_limit(const void *owner) noexcept
    {
        std::lock_guard<std::mutex> lk(mu_);
        limits_.erase(owner);
    }
    // what the blocks in use have beyond what was asked for
    size_t spare(int device) noexcept
    {
        std::lock_guard<std::mutex> lk(mu_);
        auto it = dev_.find(device);
        return it == dev_.end() ? 0 : it->second.spare;
    }

    hipError_t stream(int device, hipStream_t *s)
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            for (size_t i = 0; i < streams_.size(); i++)
                if (streams_[i].first == device) {
                    *s = streams_[i].second;
                    streams_.erase(streams_.begin() + i);
                    return hipSuccess;
                }
        }
        return hipStreamCreate(s);
    }

    void give_stream(int device, hipStream_t s) noexcept  // idle
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (streams_.size() < KEEP_STREAMS) {
                streams_.emplace_back(device, s);
                return;
            }
        }
        (void)hipStreamDestroy(s);
    }

    // A staging ring for a copy of `bytes`, or null where the runtime's own copy is the better one.  The first
    // ring's memory and the copy threads take 2 to 3 ms to set up, fault in and take down, what copies of below
    // a slot gain from them over some 64 MB (0.03 to 0.09 ms per MB); the pool of a short-lived handle makes
    // fewer (a volume of pad 96 from create to destroy: 1.2 ms, 3.3 with a ring for every pool).  No more than
    // the kept rings for such copies: more of several threads would be set up and taken down each time.
    char *pinned(size_t bytes) noexcept
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (!pinned_.empty()) {
                char *p = pinned_.back();
                pinned_.pop_back();
                return p;
            }
            if (bytes < PIN_SLOT) {
                small_ = std::min(small_ + bytes, SMALL_BYTES);
                if (small_ < SMALL_BYTES || rings_ >= KEEP_PINNED) return nullptr;
            }
            rings_++;
        }
        void *p = nullptr;
        if (hipHostMalloc(&p, PIN_SLOTS * PIN_SLOT, hipHostMallocDefault) == hipSuccess) return static_cast<char *>(p);
        (void)hipGetLastError();
        std::lock_guard<std::mutex> lk(mu_);
        rings_--;
        return nullptr;
    }

    void give_pinned(char *p) noexcept
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (pinned_.size() < KEEP_PINNED) {
                pinned_.push_back(p);
                return;
            }
            rings_--;
        }
        (void)hipHostFree(p);
    }

    CopyThreads copies;

private:
    struct Block {
        size_t size, asked;
        unsigned long long since;  // of the idle ones: when they were given back
        bool idle;
    };
    struct Device {
        std::unordered_map<void *, Block> blocks;  // in use and idle: giving one back only marks it
        size_t idle = 0;                           // bytes of the idle ones
        size_t spare = 0;                          // bytes of the ones in use beyond what was asked for
    };

    // the most idle bytes of a device
    size_t keep(int device, const Device &d) const noexcept
    {
        size_t most = KEEP_DEVICE;
        for (auto &l : limits_)
            if (l.second.first == device)
                most = (size_t)std::min<long long>(most, std::max(0LL, l.second.second - (long long)d.spare));
        return most;
    }

    // the idle blocks given back longest ago, until at most `most` bytes are left
    void shrink(std::unique_lock<std::mutex> &lk, Device &d, size_t most) noexcept
    {
        while (d.idle > most) {
            auto old = d.blocks.end();
            for (auto it = d.blocks.begin(); it != d.blocks.end(); ++it)
                if (it->second.idle && (old == d.blocks.end() || it->second.since < old->second.since)) old = it;
            void *p = old->first;
            d.idle -= old->second.size;
            d.blocks.erase(old);
            release(lk, p);
        }
    }

    // hipFree waits for the device's work: the lock is let go, so that other handles go on
    void release(std::unique_lock<std::mutex> &lk, void *p) noexcept
    {
        freeing_++;
        lk.unlock();
        (void)hipFree(p);
        lk.lock();
        if (--freeing_ == 0) freed_.notify_all();
    }

    std::mutex mu_;
    std::condition_variable freed_;
    int freeing_ = 0;  // blocks on their way back to the device
    unsigned long long clock_ = 0;
    std::map<int, Device> dev_;
    std::map<const void *, std::pair<int, long long>> limits_;  // by owner: device, bytes
    std::vector<std::pair<int, hipStream_t>> streams_;
    std::vector<char *> pinned_;
    size_t rings_ = 0;  // in use and idle
    size_t small_ = 0;  // bytes of small copies that found no ring
};

}  // namespace fh
