// The part of the HIP runtime that host_copy.h uses, over host memory: "device" memory is malloc'ed, a stream is a list of
// work that runs when somebody waits for it, a launch runs every thread of the grid in turn.  Only what a test has to see is
// kept: how often the device was waited for, what is allocated, which calls are to fail.
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <string>

#define __global__
#define __device__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, order)

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct uint4 {
    unsigned x, y, z, w;
};
inline thread_local dim3 blockIdx, threadIdx, gridDim;
inline void __syncthreads() {}
inline void __threadfence_system() {}

enum hipError_t { hipSuccess, hipErrorOutOfMemory, hipErrorUnknown, hipErrorNotReady };
enum { hipMemcpyDeviceToHost, hipMemcpyHostToDevice, hipHostMallocPortable, hipStreamNonBlocking };

namespace fake {
struct Stream {
    std::deque<std::function<void()>> work;
};
inline std::recursive_mutex m;
inline Stream null_stream;
inline std::set<Stream*> streams;
inline std::set<void*> host;                 // pinned memory
inline int device = 0, device_waits = 0;
inline bool deferred = false;                // launches wait in their stream (chunks of the ring, which are polled for, never do)
inline std::map<std::string, int> fail_in;   // the n-th call from now (1 = the next) fails
inline bool fails(const char* what)
{
    auto it = fail_in.find(what);
    if (it == fail_in.end() || --it->second != 0) return false;
    fail_in.erase(it);
    return true;
}
inline void run(Stream* s)
{
    while (!s->work.empty()) {
        auto w = s->work.front();
        s->work.pop_front();
        w();
    }
}
inline std::function<void(const void* src, const void* dst, size_t bytes)> seen;   // what each copy kernel is given
}  // namespace fake
typedef fake::Stream* hipStream_t;

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { return *d = fake::device, hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    if (fake::fails("hipHostMalloc")) return hipErrorOutOfMemory;
    *p = aligned_alloc(4096, (n + 4095) / 4096 * 4096);
    fake::host.insert(*p);
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p)
{
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    fake::host.erase(p);
    free(p);
    return hipSuccess;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    if (fake::fails("hipStreamCreateWithFlags")) return hipErrorUnknown;
    fake::streams.insert(*s = new fake::Stream);
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s)
{
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    fake::run(s);
    fake::streams.erase(s);
    delete s;
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s)
{
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    fake::run(s ? s : &fake::null_stream);
    return hipSuccess;
}
inline hipError_t hipStreamQuery(hipStream_t s) { return hipStreamSynchronize(s); }
inline hipError_t hipDeviceSynchronize()
{
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    ++fake::device_waits;
    fake::run(&fake::null_stream);
    for (auto* s : fake::streams) fake::run(s);
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, int, hipStream_t s)
{
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    if (fake::fails("hipMemcpyAsync")) return hipErrorUnknown;
    (s ? s : &fake::null_stream)->work.push_back([=] { memcpy(dst, src, n); });
    return hipSuccess;
}
// the two kernels of host_copy.h by their arguments
template <class F, class... A> void fake_run(F kernel, dim3 grid, dim3 block, A... args)
{
    gridDim = grid;
    for (blockIdx.x = 0; blockIdx.x < grid.x; ++blockIdx.x)
        for (unsigned t = block.x; t-- > 0;) {   // thread 0, which reports a block's end, comes last
            threadIdx.x = t;
            kernel(args...);
        }
}
template <class F> void fake_launch(F kernel, dim3 grid, dim3 block, hipStream_t s, const unsigned char* src, unsigned char* dst, unsigned bytes, unsigned* flag, unsigned value)
{
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    if (fake::seen) fake::seen(src, dst, bytes);
    fake::run(s ? s : &fake::null_stream);
    fake_run(kernel, grid, block, src, dst, bytes, flag, value);
}
template <class F, class Segs> void fake_launch(F kernel, dim3 grid, dim3 block, hipStream_t s, const Segs& l)
{
    std::lock_guard<std::recursive_mutex> lock(fake::m);
    for (int i = 0; fake::seen && i < l.n; ++i) fake::seen(l.s[i].src, l.s[i].dst, l.s[i].bytes);
    if (fake::deferred) (s ? s : &fake::null_stream)->work.push_back([=] { fake_run(kernel, grid, block, l); });
    else fake_run(kernel, grid, block, l);
}
#define hipLaunchKernelGGL(kernel, grid, block, shared, stream, ...) fake_launch(kernel, grid, block, stream, __VA_ARGS__)
