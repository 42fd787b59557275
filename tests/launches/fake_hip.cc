// The calls of the HIP runtime that a launch of the library makes, over host memory and for a machine without a GPU: loaded with
// global symbols in front of the library, so that the library's own code runs.  Nothing is executed; what is launched is written down.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdlib>
#include <mutex>
#include <set>
#include <unordered_map>
#include <vector>

#include <unistd.h>

namespace {
struct Launch {
    const void* func;
    void* ptr[6];
};
std::mutex m;
std::vector<Launch> launches;
std::set<void*> memory;
std::unordered_map<const void*, int> operators;   // how many pointers they take; every other kernel takes two
std::atomic<int> linger{0};                       // us that a kernel which is none of these holds up its thread
int put_down(const void* f, void** args)
{
    int us = 0;
    {
        std::lock_guard<std::mutex> lock(m);
        Launch l{f, {}};
        auto it = operators.find(f);
        for (int i = 0; i < (it == operators.end() ? 2 : it->second); ++i) l.ptr[i] = *static_cast<void**>(args[i]);
        launches.push_back(l);
        if (it == operators.end()) us = linger;
    }
    if (us) usleep(us);
    return 0;
}
}  // namespace

extern "C" {
void fake_operator(const void* f, int pointers) { operators[f] = pointers; }
void fake_linger(int us) { linger = us; }
int fake_launches(Launch* to, int most)
{
    std::lock_guard<std::mutex> lock(m);
    const int n = (int)launches.size();
    for (int i = 0; i < n && i < most; ++i) to[i] = launches[i];
    launches.clear();
    return n;
}
int fake_allocations() { return (int)memory.size(); }

hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static int there;
    return *p = &there, hipSuccess;
}
hipError_t hipMalloc(void** p, size_t)
{
    std::lock_guard<std::mutex> lock(m);
    memory.insert(*p = malloc(16));       // an address of its own
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    std::lock_guard<std::mutex> lock(m);
    memory.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t* s) { return *s = reinterpret_cast<hipStream_t>(malloc(16)), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return free(s), hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) { return static_cast<hipError_t>(put_down(f, args)); }
hipError_t hipExtLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t, hipEvent_t, hipEvent_t, int)
{
    return static_cast<hipError_t>(put_down(f, args));
}
}
