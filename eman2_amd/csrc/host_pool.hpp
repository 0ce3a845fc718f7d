// What reconstructor handles share on the host side: device blocks, streams
// and pinned staging buffers of destroyed handles, kept for the next ones, and
// the threads that copy between pinned and caller memory.  A serving job
// creates and destroys a handle; every hipFree of it waited for the other
// jobs' kernels, and a stream takes milliseconds to create.
//
// Everything here lives while a handle or a server does (HostPool::Ref): the
// last one to go gives it all back.  Kept blocks are bounded (KEEP_DEVICE
// bytes per device, KEEP_STREAMS, KEEP_PINNED) and are released when an
// allocation fails.  All calls may come from any thread.  Who gives a block
// back has waited for the work that uses it.
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
        auto job = std::make_shared<Job>();
        job->dst = dst;
        job->src = src;
        job->len = len;
        job->nseg = (len + SEG - 1) / SEG;
        {
            std::lock_guard<std::mutex> lk(mu_);
            try {
                while (threads_.size() < THREADS) threads_.emplace_back([this] { work(); });
            } catch (...) {
                // no (more) threads: the caller copies what they do not
            }
            jobs_.push_back(job);
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
    static constexpr size_t PIN_SLOTS = 4, PIN_SLOT = 16u << 20;  // a staging ring: 4 slots of 16 MB

    static Ref get()
    {
        static std::mutex mu;
        static std::weak_ptr<HostPool> pool;
        std::lock_guard<std::mutex> lk(mu);
        Ref r = pool.lock();
        if (!r) pool = r = std::make_shared<HostPool>();
        return r;
    }

    ~HostPool()
    {
        for (auto &d : dev_) release(d.second);
        for (char *p : pinned_) (void)hipHostFree(p);
        for (auto &s : streams_) (void)hipStreamDestroy(s.second);
    }

    // `bytes` on the current device `device`: a kept block of at most a quarter more, or a new one
    hipError_t alloc(int device, void **p, size_t bytes)
    {
        bytes = std::max<size_t>(bytes, 256);
        std::lock_guard<std::mutex> lk(mu_);
        Device &d = dev_[device];
        auto it = d.kept.lower_bound(bytes);
        if (it != d.kept.end() && it->first <= bytes + bytes / 4 + 4096) {
            *p = it->second;
            d.sizes[*p] = it->first;
            d.bytes -= it->first;
            d.kept.erase(it);
            return hipSuccess;
        }
        hipError_t e = hipMalloc(p, bytes);
        if (e == hipErrorOutOfMemory && !d.kept.empty()) {
            (void)hipGetLastError();
            release(d);
            e = hipMalloc(p, bytes);
        }
        if (e == hipSuccess) d.sizes[*p] = bytes;
        return e;
    }

    void free(int device, void *p)
    {
        std::lock_guard<std::mutex> lk(mu_);
        Device &d = dev_[device];
        const size_t n = d.sizes[p];
        d.sizes.erase(p);
        if (d.bytes + n > KEEP_DEVICE) {
            (void)hipFree(p);
            return;
        }
        d.kept.emplace(n, p);
        d.bytes += n;
    }

    hipError_t stream(int device, hipStream_t *s)
    {
        std::lock_guard<std::mutex> lk(mu_);
        for (size_t i = 0; i < streams_.size(); i++)
            if (streams_[i].first == device) {
                *s = streams_[i].second;
                streams_.erase(streams_.begin() + i);
                return hipSuccess;
            }
        return hipStreamCreate(s);
    }

    void give_stream(int device, hipStream_t s)  // idle
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (streams_.size() < KEEP_STREAMS) streams_.emplace_back(device, s);
        else (void)hipStreamDestroy(s);
    }

    hipError_t pinned(char **p)
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (!pinned_.empty()) {
            *p = pinned_.back();
            pinned_.pop_back();
            return hipSuccess;
        }
        return hipHostMalloc((void **)p, PIN_SLOTS * PIN_SLOT, hipHostMallocDefault);
    }

    void give_pinned(char *p)
    {
        std::lock_guard<std::mutex> lk(mu_);
        if (pinned_.size() < KEEP_PINNED) pinned_.push_back(p);
        else (void)hipHostFree(p);
    }

    CopyThreads copies;

private:
    struct Device {
        std::multimap<size_t, void *> kept;
        std::unordered_map<void *, size_t> sizes;  // blocks in use
        size_t bytes = 0;                          // of kept
    };
    static void release(Device &d)
    {
        for (auto &b : d.kept) (void)hipFree(b.second);
        d.kept.clear();
        d.bytes = 0;
    }
    std::mutex mu_;
    std::map<int, Device> dev_;
    std::vector<std::pair<int, hipStream_t>> streams_;
    std::vector<char *> pinned_;
};

}  // namespace fh
