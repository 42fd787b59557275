// host_copy.h over a stand-in for the HIP runtime (hip/hip_runtime.h beside this file): each test a name on the command line.
#include <dlfcn.h>
#include <pthread.h>

#include <cerrno>
#include <cstdio>
#include <new>
#include <string>

#include "host_copy.h"

using namespace bfuse;

#define CHECK(x)                                                        \
    do {                                                                \
        if (!(x)) {                                                     \
            fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #x);     \
            exit(1);                                                    \
        }                                                               \
    } while (0)

// allocations and threads that are to fail: the n-th from now
static thread_local int new_fails_in = 0;
static int thread_fails_in = 0;
void* operator new(size_t n)
{
    if (new_fails_in > 0 && --new_fails_in == 0) throw std::bad_alloc();
    return malloc(n);
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg)
{
    if (thread_fails_in > 0 && --thread_fails_in == 0) return EAGAIN;
    return reinterpret_cast<decltype(&pthread_create)>(dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, arg);
}

static HostCopy& hc() { return HostCopy::get(); }
static std::vector<unsigned char> pattern(size_t n, unsigned seed)
{
    std::vector<unsigned char> v(n);
    for (auto& b : v) b = (unsigned char)((seed = seed * 1664525u + 1013904223u) >> 24);
    return v;
}

// Whatever the offset of a part, the copy kernels move 16-byte words: source and destination lie alike in 16 bytes.
static void unaligned()
{
    static unsigned char* const dev = static_cast<unsigned char*>(aligned_alloc(4096, 16 << 20));
    for (size_t n : {(size_t)1, (size_t)14, (size_t)33, (size_t)1156, HostCopy::kSmallBytes, HostCopy::kSmallBytes + 1, HostCopy::kFirst * 3 + 5, 5 * HostCopy::kChunk + 77})
        for (size_t at : {0, 1, 2, 4, 12, 15})
            for (size_t host_at : {0, 4, 7}) {
                auto src = pattern(host_at + n, (unsigned)(n + at));
                memset(dev, 0xee, at + n + 64);
                bool alike = true;
                size_t moved = 0;
                fake::seen = [&](const void* s, const void* d, size_t b) { alike &= (((uintptr_t)s ^ (uintptr_t)d) & 15) == 0, moved += b; };
                CopySeg seg = {dev + at, src.data() + host_at, n};
                CHECK(hc().up(&seg, 1, false) == hipSuccess);
                CHECK(memcmp(dev + at, src.data() + host_at, n) == 0 && dev[at + n] == 0xee && (at == 0 || dev[at - 1] == 0xee));
                std::vector<unsigned char> got(host_at + n + 1, 0x77);
                seg.host = got.data() + host_at;
                HostCopy::Down d;
                CHECK(hc().down_begin(&seg, 1, nullptr, d) == hipSuccess && hipDeviceSynchronize() == hipSuccess && hc().down_finish(d) == hipSuccess);
                CHECK(memcmp(got.data() + host_at, src.data() + host_at, n) == 0 && got[host_at + n] == 0x77);
                CHECK(alike && moved == 2 * n);
                fake::seen = nullptr;
            }
}

// What is enqueued while another thread waits is still in flight behind that wait, and everything is until a wait has ended.
static void in_flight()
{
    InFlight f;
    CHECK(!f.any());
    f.add();
    f.wait_begins();
    CHECK(f.any());
    f.add();
    f.wait_ended(true);
    CHECK(f.any());
    f.wait_begins();
    f.wait_begins();
    f.wait_ended(true);
    CHECK(f.any());
    f.wait_ended(true);
    CHECK(!f.any());
    f.add();
    f.wait_begins();
    f.wait_ended(false);
    CHECK(f.any());
}

// What one thread has in the arenas outlives another thread's synchronisation.
static void arenas()
{
    fake::deferred = true;
    std::vector<unsigned char> dev[3] = {std::vector<unsigned char>(1000), std::vector<unsigned char>(1000), std::vector<unsigned char>(9000)}, src[3];
    auto up = [&](int i) {
        src[i] = pattern(dev[i].size(), i);
        const CopySeg seg = {dev[i].data(), src[i].data(), dev[i].size()};
        CHECK(hc().up(&seg, 1, false) == hipSuccess);
    };
    // a thread starts to wait after upload 0; upload 1 comes before it has said that it did
    up(0);
    hc().wait_begins();
    CHECK(hipDeviceSynchronize() == hipSuccess);
    up(1);
    hc().wait_ended(true);
    up(2);
    CHECK(hipDeviceSynchronize() == hipSuccess);
    for (int i = 0; i < 3; ++i) CHECK(dev[i] == src[i]);
    // a result that has landed is still there when another thread's results come and go
    std::vector<unsigned char> got[3];
    HostCopy::Down d[3];
    auto begin = [&](int i) {
        got[i].assign(dev[i].size(), 0);
        const CopySeg seg = {dev[i].data(), got[i].data(), dev[i].size()};
        CHECK(hc().down_begin(&seg, 1, nullptr, d[i]) == hipSuccess);
    };
    auto wait = [&] {
        hc().wait_begins();
        CHECK(hipDeviceSynchronize() == hipSuccess);
        hc().wait_ended(true);
    };
    begin(0);
    wait();
    begin(1);
    wait();
    CHECK(hc().down_finish(d[1]) == hipSuccess);
    begin(2);
    wait();
    CHECK(hc().down_finish(d[0]) == hipSuccess && hc().down_finish(d[2]) == hipSuccess);
    for (int i = 0; i < 3; ++i) CHECK(got[i] == src[i]);
    // more threads between begin and finish than the arena holds
    constexpr int kMany = 2 * HostCopy::kArenaBytes / HostCopy::kSmallBytes;
    std::vector<std::vector<unsigned char>> from, to(kMany, std::vector<unsigned char>(HostCopy::kSmallBytes));
    HostCopy::Down many[kMany];
    for (int i = 0; i < kMany; ++i) from.push_back(pattern(HostCopy::kSmallBytes, 7 * i));
    for (int i = 0; i < kMany; ++i) {
        const CopySeg seg = {from[i].data(), to[i].data(), HostCopy::kSmallBytes};
        CHECK(hc().down_begin(&seg, 1, nullptr, many[i]) == hipSuccess);
    }
    wait();
    for (int i = kMany; i-- > 0;) CHECK(hc().down_finish(many[i]) == hipSuccess && to[i] == from[i]);
    // and the arena of uploads comes round when nobody ever waits
    for (int i = 0; i < 30; ++i) {
        const CopySeg seg = {to[0].data(), from[i % kMany].data(), HostCopy::kSmallBytes};
        CHECK(hc().up(&seg, 1, false) == hipSuccess);
    }
    wait();
    CHECK(to[0] == from[29 % kMany]);
}

// Threads that move what is their own, small and long, and wait when they like.
static void threads()
{
    fake::deferred = true;
    std::vector<std::thread> all;
    for (int id = 0; id < 4; ++id)
        all.emplace_back([id] {
            for (int k = 0; k < 60; ++k) {
                const size_t n = k % 6 == 5 ? HostCopy::kSmallBytes + 7777 * id + 1 : 100 + 30000 * ((k + id) % 4);
                std::vector<unsigned char> dev(n + 16), got(n);
                const auto x = pattern(n, 100 * id + k);
                const CopySeg up = {dev.data() + k % 16, const_cast<unsigned char*>(x.data()), n}, down = {dev.data() + k % 16, got.data(), n};
                CHECK(hc().up(&up, 1, false) == hipSuccess);
                HostCopy::Down d;
                CHECK(hc().down_begin(&down, 1, nullptr, d) == hipSuccess);
                hc().wait_begins();
                CHECK(hipDeviceSynchronize() == hipSuccess);
                hc().wait_ended(true);
                CHECK(hc().down_finish(d) == hipSuccess && got == x);
            }
        });
    for (auto& t : all) t.join();
}

// Copies into a caller's pinned memory have ended when a transfer that failed is given up.
static void given_up()
{
    const size_t n = HostCopy::kSmallBytes;
    auto a = pattern(n, 1), b = pattern(n, 2);
    auto* p = static_cast<unsigned char*>(hc().host_buffer(2 * n));
    memset(p, 0, 2 * n);
    const CopySeg seg[2] = {{a.data(), p, n}, {b.data(), p + n, n}};
    {
        HostCopy::Down d;
        fake::fail_in["hipMemcpyAsync"] = 2;
        CHECK(hc().down_begin(seg, 2, nullptr, d) == hipErrorUnknown);
    }
    CHECK(memcmp(p, a.data(), n) == 0);
    memset(p, 0, n);
    {
        HostCopy::Down d;
        CHECK(hc().down_begin(seg, 2, nullptr, d) == hipSuccess);   // and then an error between begin and finish
    }
    CHECK(memcmp(p, a.data(), n) == 0 && memcmp(p + n, b.data(), n) == 0);
    const int waits = fake::device_waits;
    {
        HostCopy::Down d;
        CHECK(hc().down_begin(seg, 2, nullptr, d) == hipSuccess && hipDeviceSynchronize() == hipSuccess && hc().down_finish(d) == hipSuccess);
    }
    CHECK(fake::device_waits == waits + 1);                         // none but the caller's own
    // operands likewise
    const CopySeg up[2] = {{a.data(), p, n}, {b.data(), p + n, n}};
    memset(p, 5, n);
    fake::fail_in["hipMemcpyAsync"] = 2;
    CHECK(hc().up(up, 2, false) == hipErrorUnknown && a[0] == 5 && a[n - 1] == 5);
    CHECK(hc().release(p));
}

// Whatever fails while the first transfer sets up, the call says so, nothing is left behind, and the next one works.
static void setup_fails()
{
    auto x = pattern(3 * HostCopy::kChunk, 3);
    std::vector<unsigned char> dev(x.size());
    const CopySeg seg = {dev.data(), x.data(), x.size()};
    auto works = [&] {
        std::fill(dev.begin(), dev.end(), 0);
        CHECK(hc().up(&seg, 1, false) == hipSuccess && dev == x);
    };
    for (int n : {1, 2}) {
        fake::fail_in["hipStreamCreateWithFlags"] = n;
        CHECK(hc().up(&seg, 1, false) == hipErrorUnknown && fake::streams.empty());
        hc().close();
        CHECK(fake::host.empty());
        fake::fail_in["hipStreamCreateWithFlags"] = n;
        CHECK(hc().up(&seg, 1, false) == hipErrorUnknown);
        works();
        CHECK(fake::streams.size() == 2);
        fake::device ^= 1;                                   // another device: the streams go over
        fake::fail_in["hipStreamCreateWithFlags"] = n;
        CHECK(hc().up(&seg, 1, false) == hipErrorUnknown && fake::streams.size() == 2);
        works();
        CHECK(fake::streams.size() == 2);
        hc().close();
    }
    for (int n : {1, 2, 3, 4}) {
        fake::fail_in["hipHostMalloc"] = n;
        CHECK(hc().up(&seg, 1, false) == hipErrorOutOfMemory && fake::host.empty());
    }
    for (int n : {1, 2}) {
        thread_fails_in = n;
        works();
        hc().close();
    }
    works();
    for (int n : {1, 2, 3}) {
        new_fails_in = n;
        CHECK(hc().up(&seg, 1, false) == hipErrorOutOfMemory);
        new_fails_in = 0;
        works();
        HostCopy::Down d;
        std::vector<unsigned char> got(x.size());
        const CopySeg back = {dev.data(), got.data(), got.size()};
        CHECK(hc().down_begin(&back, 1, nullptr, d) == hipSuccess && hipDeviceSynchronize() == hipSuccess);
        new_fails_in = n;
        CHECK(hc().down_finish(d) == hipErrorOutOfMemory);
        new_fails_in = 0;
    }
    const size_t pinned = fake::host.size();
    new_fails_in = 2;                                        // the first is the stand-in's
    CHECK(hc().host_buffer(1 << 20) == nullptr && fake::host.size() == pinned);
    void* p = hc().host_buffer(1 << 20);
    new_fails_in = 1;
    CHECK(p && hc().release(p) && fake::host.size() == pinned && !hc().release(p));
}

int main(int argc, char** argv)
{
    const std::string t = argc > 1 ? argv[1] : "";
    if (t == "unaligned") unaligned();
    else if (t == "in_flight") in_flight();
    else if (t == "arenas") arenas();
    else if (t == "threads") threads();
    else if (t == "given_up") given_up();
    else if (t == "setup_fails") setup_fails();
    else return fprintf(stderr, "no test '%s'\n", t.c_str()), 2;
    hc().close();
    CHECK(fake::host.empty() && fake::streams.empty());
    return 0;
}
