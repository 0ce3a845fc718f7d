// The few calls of the HIP runtime that host_pool.hpp makes, on no device:
// addresses without memory behind them, counted.
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdlib>
#include <map>
#include <mutex>
#include <set>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
typedef struct ihipStream_t *hipStream_t;
constexpr unsigned hipHostMallocDefault = 0;

namespace stub {
inline std::mutex mu;
inline std::condition_variable cv;
inline size_t capacity = 288ull << 30, used = 0, others = 0;  // bytes of one device; others: of other programs
inline std::map<char *, size_t> blocks;                       // live device blocks
inline std::set<void *> hosts, streams;
inline std::set<char *> hold;  // hipFree of these waits until they are taken out
inline int mallocs = 0, frees = 0, waiting = 0;
inline bool no_hosts = false;  // no pinned memory
inline char *next = reinterpret_cast<char *>(1ull << 40);
}  // namespace stub

inline hipError_t hipMalloc(void **p, size_t n)
{
    std::lock_guard<std::mutex> lk(stub::mu);
    if (stub::used + stub::others + n > stub::capacity) return hipErrorOutOfMemory;
    stub::used += n;
    stub::mallocs++;
    stub::blocks[stub::next] = n;
    *p = stub::next;
    stub::next += (n + 4095) / 4096 * 4096;
    return hipSuccess;
}

inline hipError_t hipFree(void *v)
{
    std::unique_lock<std::mutex> lk(stub::mu);
    char *p = static_cast<char *>(v);
    if (stub::hold.count(p)) {
        stub::waiting++;
        stub::cv.notify_all();
        stub::cv.wait(lk, [&] { return !stub::hold.count(p); });
        stub::waiting--;
    }
    auto it = stub::blocks.find(p);
    if (it == stub::blocks.end()) abort();  // freed twice, or never allocated
    stub::used -= it->second;
    stub::frees++;
    stub::blocks.erase(it);
    return hipSuccess;
}

inline hipError_t hipGetLastError() { return hipSuccess; }

inline hipError_t hipMemGetInfo(size_t *free, size_t *total)
{
    std::lock_guard<std::mutex> lk(stub::mu);
    *free = stub::capacity - stub::used - stub::others;
    *total = stub::capacity;
    return hipSuccess;
}

inline hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (stub::no_hosts) return hipErrorOutOfMemory;
    *p = malloc(n);
    std::lock_guard<std::mutex> lk(stub::mu);
    stub::hosts.insert(*p);
    return hipSuccess;
}

inline hipError_t hipHostFree(void *p)
{
    {
        std::lock_guard<std::mutex> lk(stub::mu);
        if (!stub::hosts.erase(p)) abort();
    }
    ::free(p);
    return hipSuccess;
}

inline hipError_t hipStreamCreate(hipStream_t *s)
{
    *s = static_cast<hipStream_t>(malloc(1));
    std::lock_guard<std::mutex> lk(stub::mu);
    stub::streams.insert(*s);
    return hipSuccess;
}

inline hipError_t hipStreamDestroy(hipStream_t s)
{
    std::lock_guard<std::mutex> lk(stub::mu);
    if (!stub::streams.erase(s)) abort();
    ::free(s);
    return hipSuccess;
}
