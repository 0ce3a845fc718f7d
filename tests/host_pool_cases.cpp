// The rules of host_pool.hpp against the counting runtime of host_stub: one
// case per name given on the command line, exit status 1 where one is broken.
#include "host_pool.hpp"

#include <chrono>
#include <cstdio>
#include <new>
#include <random>
#include <string>

using fh::HostPool;
static const size_t MB = 1ull << 20, GB = 1ull << 30;

static std::atomic<bool> no_memory{false};  // of the host
void *operator new(size_t n)
{
    if (no_memory) throw std::bad_alloc();
    if (void *p = malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { ::free(p); }
void operator delete(void *p, size_t) noexcept { ::free(p); }

#define CHECK(x)                                                   \
    do {                                                           \
        if (!(x)) {                                                \
            fprintf(stderr, "line %d: %s\n", __LINE__, #x);        \
            fflush(stderr);                                        \
            _Exit(1);                                              \
        }                                                          \
    } while (0)

static void *get(HostPool &p, size_t n)
{
    void *v = nullptr;
    CHECK(p.alloc(0, &v, n) == hipSuccess && v);
    return v;
}

// a block is handed on where it is at most a quarter (and a page) too large
static void reuse()
{
    auto p = HostPool::get();
    void *a = get(*p, 10 * MB);
    p->free(0, a);
    void *b = get(*p, 7 * MB);
    CHECK(b != a);
    void *c = get(*p, 9 * MB);
    CHECK(c == a);
    void *d = get(*p, 9 * MB);
    CHECK(d != a);
    p->free(0, b);
    p->free(0, c);
    p->free(0, d);
    void *e = get(*p, 9 * MB);
    CHECK(e == d);  // the one that fits best
    p->free(0, e);
    CHECK(stub::mallocs == 3);
}

// the last handle gives back blocks, streams and pinned memory
static void last_one()
{
    auto p = HostPool::get(), q = HostPool::get();
    CHECK(p == q);
    for (int i = 0; i < 30; i++) {
        hipStream_t s;
        CHECK(p->stream(0, &s) == hipSuccess);
        char *h = p->pinned(GB);
        CHECK(h);
        p->free(0, get(*p, (i + 1) * 100 * MB));
        p->give_stream(0, s);
        p->give_pinned(h);
    }
    CHECK(stub::streams.size() == 1 && stub::hosts.size() == 1 && !stub::blocks.empty());
    p.reset();
    CHECK(!stub::blocks.empty());
    q.reset();
    CHECK(stub::blocks.empty() && stub::streams.empty() && stub::hosts.empty());
}

// what is kept is bounded
static void bounds()
{
    auto p = HostPool::get();
    std::vector<void *> v;
    std::vector<hipStream_t> s(40);
    std::vector<char *> h(10);
    for (int i = 0; i < 40; i++) v.push_back(get(*p, GB + i * 300 * MB));
    for (auto &x : s) CHECK(p->stream(0, &x) == hipSuccess);
    for (auto &x : h) CHECK((x = p->pinned(GB)));
    for (void *x : v) p->free(0, x);
    for (auto x : s) p->give_stream(0, x);
    for (auto x : h) p->give_pinned(x);
    CHECK(stub::used <= HostPool::KEEP_DEVICE && stub::streams.size() <= HostPool::KEEP_STREAMS &&
          stub::hosts.size() <= HostPool::KEEP_PINNED);
}

// the blocks given back last are the ones that stay: sizes that do not come again make room
static void oldest_first()
{
    auto p = HostPool::get();
    std::vector<void *> v;
    for (int i = 0; i < 8; i++) v.push_back(get(*p, 900 * MB + i));
    for (void *x : v) p->free(0, x);
    const int before = stub::mallocs;
    for (int i = 0; i < 20; i++) {
        void *a = get(*p, 2 * GB), *b = get(*p, 3 * GB);
        p->free(0, a);
        p->free(0, b);
    }
    CHECK(stub::mallocs == before + 2);
    void *c = get(*p, 9 * GB);  // larger than all that is kept: straight back, the others stay
    p->free(0, c);
    void *d = get(*p, 3 * GB);
    CHECK(stub::mallocs == before + 3);
    p->free(0, d);
}

// a limit holds for idle blocks and for what reused blocks have beyond what was asked for
static void limits()
{
    auto p = HostPool::get();
    int a, b;
    p->limit(&a, 0, 2 * GB);
    std::vector<void *> v;
    for (int i = 0; i < 6; i++) v.push_back(get(*p, 500 * MB));
    for (void *x : v) p->free(0, x);
    CHECK(stub::used == 2000 * MB);
    p->change_limit(&a, -(long long)GB);
    CHECK(stub::used == 1000 * MB);
    void *x = get(*p, 420 * MB);
    CHECK(p->spare(0) == 80 * MB);
    p->change_limit(&a, -400ll * (long long)MB);  // 624 MB: 80 in use, 500 idle
    CHECK(stub::used == 1000 * MB);
    p->change_limit(&a, -100ll * (long long)MB);
    CHECK(stub::used == 500 * MB);
    p->limit(&b, 0, 0);
    p->free(0, x);
    CHECK(stub::used == 0 && p->spare(0) == 0);
    p->no_limit(&b);
    p->change_limit(&a, 2 * (long long)GB);
    p->free(0, get(*p, 2 * GB));
    CHECK(stub::used == 2 * GB);
    p->limit(&b, 1, 0);  // of another device
    p->no_limit(&a);
    p->free(0, get(*p, 4 * GB));
    CHECK(stub::used == 6 * GB);
    p->change_limit(&b, -(long long)GB);
    p->no_limit(&b);
}

// idle blocks give way where others fill the device, and on request
static void others()
{
    auto p = HostPool::get();
    stub::capacity = 20 * GB;
    void *a = get(*p, 3 * GB), *b = get(*p, 2 * GB), *c = get(*p, GB);
    stub::others = 11 * GB;  // 3 GB left
    p->free(0, a);
    CHECK(stub::used == 3 * GB);
    p->free(0, c);           // 6 GB left, a third of it 2
    p->free(0, b);
    CHECK(stub::used == 2 * GB);
    stub::others = 0;
    p->trim(1);
    CHECK(stub::used == 2 * GB);
    p->trim(0);
    CHECK(stub::used == 0);
    p->free(0, get(*p, 3 * GB));
    CHECK(stub::used == 3 * GB);
    CHECK(HostPool::get(false) == p);
    p.reset();
    CHECK(!HostPool::get(false) && stub::used == 0);
}

// an allocation that does not fit beside the idle blocks takes their place
static void out_of_memory()
{
    auto p = HostPool::get();
    stub::capacity = 10 * GB;
    void *a = get(*p, 3 * GB), *b = get(*p, 3 * GB), *c = get(*p, GB);
    p->free(0, a);
    p->free(0, b);
    void *d = get(*p, 8 * GB);
    void *e = nullptr;
    CHECK(p->alloc(0, &e, 2 * GB) == hipErrorOutOfMemory);
    p->free(0, c);
    p->free(0, d);
}

// hipFree waits for other handles' kernels: meanwhile the rest of the pool works, and an allocation
// that needs the memory on its way back waits for it
static void waiting_free()
{
    auto p = HostPool::get();
    stub::capacity = 30 * GB;
    void *big = get(*p, 20 * GB), *a = get(*p, 100 * MB);
    stub::hold.insert(static_cast<char *>(big));
    std::thread t([&] { p->free(0, big); });
    {
        std::unique_lock<std::mutex> lk(stub::mu);
        stub::cv.wait(lk, [] { return stub::waiting == 1; });
    }
    std::atomic<bool> done{false}, later{false};
    std::thread u([&] {
        p->free(0, a);
        void *b = get(*p, 100 * MB);
        hipStream_t s;
        char *h;
        CHECK(p->stream(0, &s) == hipSuccess && (h = p->pinned(GB)));
        p->give_stream(0, s);
        p->give_pinned(h);
        p->free(0, b);
        done = true;
        void *c = get(*p, 25 * GB);
        later = true;
        p->free(0, c);
    });
    for (int i = 0; i < 200 && !done; i++) std::this_thread::sleep_for(std::chrono::milliseconds(10));
    CHECK(done && !later);
    {
        std::lock_guard<std::mutex> lk(stub::mu);
        stub::hold.clear();
    }
    stub::cv.notify_all();
    t.join();
    u.join();
    CHECK(later);
}

// a pool's first small copies take no ring, large ones do; one that is there is taken by all; small copies
// take no more rings than are kept
static void rings()
{
    auto p = HostPool::get();
    for (size_t i = 0; i + 1 < HostPool::SMALL_BYTES / (4 * MB); i++) CHECK(!p->pinned(4 * MB));
    char *a = p->pinned(4 * MB), *b = p->pinned(4 * MB);
    CHECK(a && b && a != b);
    p->give_pinned(a);
    CHECK(p->pinned(4 * MB) == a);
    std::vector<char *> more;
    for (size_t i = 2; i < HostPool::KEEP_PINNED; i++) more.push_back(p->pinned(4 * MB));
    CHECK(!p->pinned(4 * MB));
    more.push_back(p->pinned(HostPool::PIN_SLOT));
    for (char *c : more) {
        CHECK(c);
        p->give_pinned(c);
    }
    p->give_pinned(a);
    p->give_pinned(b);
    CHECK(stub::hosts.size() == HostPool::KEEP_PINNED);
    p.reset();
    CHECK(stub::hosts.empty());
    p = HostPool::get();
    CHECK(!p->pinned(HostPool::PIN_SLOT - 1));
    char *c = p->pinned(HostPool::PIN_SLOT);
    CHECK(c);
    p->give_pinned(c);
    CHECK(p->pinned(4 * MB) == c);
    p->give_pinned(c);
    stub::no_hosts = true;  // no pinned memory to be had
    char *d = p->pinned(GB);
    CHECK(d == c && !p->pinned(GB));
    p->give_pinned(d);
}

// without host memory nothing is thrown: what cannot be noted is given back, copies are made by the caller
static void no_host_memory()
{
    auto p = HostPool::get();
    std::vector<char> src(5 * MB), dst(5 * MB);
    for (size_t i = 0; i < src.size(); i++) src[i] = (char)(i * 2654435761u >> 13);
    std::vector<void *> v;
    for (int i = 0; i < 8; i++) v.push_back(get(*p, (i + 1) * MB));
    std::vector<hipStream_t> s(3);
    for (auto &x : s) CHECK(p->stream(0, &x) == hipSuccess);
    char *h = p->pinned(GB);
    CHECK(h);
    no_memory = true;
    bool thrown = false;
    try {
        for (void *x : v) p->free(0, x);
        for (auto x : s) p->give_stream(0, x);
        p->give_pinned(h);
        p->copies.copy(dst.data(), src.data(), src.size());
    } catch (...) {
        thrown = true;
    }
    no_memory = false;
    CHECK(!thrown && src == dst);
    void *x = get(*p, 8 * MB);
    p->free(0, x);
}

// copies of several threads at once, at sizes around the segments'
static void copies()
{
    auto p = HostPool::get();
    std::vector<std::thread> t;
    for (int k = 0; k < 4; k++)
        t.emplace_back([&, k] {
            for (size_t n : {size_t(0), size_t(1), MB - 1, MB, MB + 1, 3 * MB + 17, 7 * MB}) {
                std::vector<char> a(n + 2, 1), b(n + 2, 0);
                for (size_t i = 0; i < n; i++) a[i] = (char)(i * 31 + k);
                p->copies.copy(b.data(), a.data(), n);
                CHECK(std::equal(a.begin(), a.begin() + n, b.begin()) && b[n] == 0 && b[n + 1] == 0);
            }
        });
    for (auto &x : t) x.join();
}

// handles of many threads: no block twice, the bound at every moment that nobody allocates in
static void threads()
{
    auto p = HostPool::get();
    stub::capacity = 60 * GB;
    std::mutex mu;
    std::set<void *> owned;
    std::vector<std::thread> t;
    for (int k = 0; k < 6; k++)
        t.emplace_back([&, k] {
            std::mt19937 r(k);
            std::vector<void *> mine;
            for (int i = 0; i < 4000; i++) {
                if (mine.size() < 8 && (mine.empty() || r() % 2)) {
                    void *v = get(*p, (1 + r() % 800) * MB);
                    std::lock_guard<std::mutex> lk(mu);
                    CHECK(owned.insert(v).second);
                    mine.push_back(v);
                } else {
                    void *v = mine.back();
                    mine.pop_back();
                    {
                        std::lock_guard<std::mutex> lk(mu);
                        owned.erase(v);
                    }
                    p->free(0, v);
                }
            }
            for (void *v : mine) {
                {
                    std::lock_guard<std::mutex> lk(mu);
                    owned.erase(v);
                }
                p->free(0, v);
            }
        });
    for (auto &x : t) x.join();
    CHECK(stub::used <= HostPool::KEEP_DEVICE);
    p.reset();
    CHECK(stub::blocks.empty());
}

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> cases = {
        {"reuse", reuse},   {"last_one", last_one},         {"bounds", bounds},   {"oldest_first", oldest_first}, {"limits", limits}, {"rings", rings}, {"others", others}, {"out_of_memory", out_of_memory},
        {"waiting_free", waiting_free}, {"no_host_memory", no_host_memory}, {"copies", copies}, {"threads", threads},
    };
    if (argc == 1)
        for (auto &c : cases) printf("%s\n", c.first.c_str());
    for (int i = 1; i < argc; i++) cases.at(argv[i])();
    return 0;
}
