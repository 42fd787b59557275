// host_copy.h over a stand-in for the HIP runtime (hip/hip_runtime.h beside this file): each test a name on the command line.
#include <cstdio>
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
                CHECK(hc().down_begin(&seg, 1, nullptr, d) == hipSuccess && hipDeviceSynchronize() == hipSuccess);
                hc().quiesced();
                CHECK(hc().down_finish(d) == hipSuccess);
                CHECK(memcmp(got.data() + host_at, src.data() + host_at, n) == 0 && got[host_at + n] == 0x77);
                CHECK(alike && moved == 2 * n);
                fake::seen = nullptr;
            }
}

int main(int argc, char** argv)
{
    const std::string t = argc > 1 ? argv[1] : "";
    if (t == "unaligned") unaligned();
    else return fprintf(stderr, "no test '%s'\n", t.c_str()), 2;
    hc().close();
    CHECK(fake::host.empty() && fake::streams.empty());
    return 0;
}
