// Copies between host arrays and the resident device buffers: what the harness functions (run_kernel1/2, run_parallel,
// run_fuse) and bfuse_upload / bfuse_download move.  The reference copies every tensor with a cudaMemcpy of pageable
// memory (test-utils/test-suite-files/operation_cu.py:164-256).
//
// What bounds such a copy on this machine is the host, not the link: hipMemcpy of pageable memory reaches 18-30 GB/s
// (10 GB/s into memory that was never touched, one thread taking every page fault) where the link takes 57 GB/s one way
// and 96 GB/s both ways, and its small copies cost 12-60 us each.  So
//   * a few hundred KB (kSmallBytes: where one thread's memcpy starts to show against a pipeline's start-up) are packed
//     into a pinned arena by the calling thread and moved by ONE kernel launch over all tensors of the call
//     (one launch, ~3 us of GPU time + the bytes, whatever the number of tensors);
//   * anything larger goes through a ring of pinned slots: worker threads fill (or drain) slots while copy kernels move
//     the ones that are ready, alternating between two streams so that one starts under the other's end, and report
//     the end of a copy by a word in host memory (128 MB: 56 GB/s up, 53 down; with an event behind every copy 46 and
//     47, with a copy engine 38);
//   * host memory that came from host_buffer() is pinned and copied in place, with no slot and no thread in between.
// run_fuse over 0.3 MB: 111 -> 44 us; run_parallel over 600 MB: 36 -> 8.6 ms (the link's floor: 6.4 up + what of the 4.4
// down is not under it).  up() returns with the copied bytes on their way into place before anything launched later;
// down_begin / down_finish leave the wait to the caller's own synchronisation.
#pragma once
#include <hip/hip_runtime.h>
#include <immintrin.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <exception>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

namespace bfuse {

struct CopySeg {
    void* dev;
    void* host;
    size_t bytes;
};

constexpr int kMaxSegs = 2 * 4 + 1;   // two operands (or one result and the give-up counters) of every side

struct SegList {
    struct {
        const unsigned char* src;
        unsigned char* dst;
        unsigned bytes;
    } s[kMaxSegs];
    int n;
};

// Bytes in front of the first 16-byte boundary.  Host memory that a copy kernel reads or writes is the library's own and is
// chosen to lie like the device memory relative to such a boundary (see lie()): whatever a part's offset, all but up to 15
// bytes at either end move as 16-byte words.  (48 MB at an offset of one float: 1.0 ms up and down; in single bytes, 64 of
// them a wave's request, 15.2 up and 2.3 down.)
static __device__ __forceinline__ unsigned head_of(const void* p, unsigned bytes)
{
    const unsigned head = -(unsigned)(uintptr_t)p & 15;
    return head < bytes ? head : bytes;
}

// All segments of one small transfer, device memory <-> pinned host memory, by one launch: consecutive lanes move
// consecutive 16-byte words (one PCIe request per 64 bytes and more), every block strides over every segment.
static __global__ __launch_bounds__(256) void copy_segments(SegList l)
{
    const unsigned t = blockIdx.x * 256 + threadIdx.x, nt = gridDim.x * 256;
    for (int k = 0; k < l.n; ++k) {
        const unsigned char* const src = l.s[k].src;
        unsigned char* const dst = l.s[k].dst;
        const unsigned bytes = l.s[k].bytes, head = head_of(dst, bytes), words = (bytes - head) / 16, ends = bytes - 16 * words;
        for (unsigned i = t; i < words; i += nt) reinterpret_cast<uint4*>(dst + head)[i] = reinterpret_cast<const uint4*>(src + head)[i];
        if (t < ends) dst[t < head ? t : 16 * words + t] = src[t < head ? t : 16 * words + t];
    }
}

// One chunk of a long transfer.  Every block reports for itself: once its part is in place, whoever reads it next (the
// host, or a kernel launched from now on), it writes `value` to its word of `flag`, which is host memory.  An event
// would tell the same, but recording one holds the stream's next kernel up for 5 us and the host for 3.  Four words are
// in flight per thread: fewer, fatter blocks keep the link as full and leave it less to switch between (128 MB up: 56
// GB/s with 8 blocks, 53 with 16, 50 with 32, 45 with 64; down it is the other way round, 52, 53, 53, 54).
static __global__ __launch_bounds__(256) void copy_chunk(const unsigned char* src, unsigned char* dst, unsigned bytes, unsigned* flag, unsigned value)
{
    const unsigned t = blockIdx.x * 256 + threadIdx.x, nt = gridDim.x * 256;
    const unsigned head = head_of(dst, bytes), words = (bytes - head) / 16, ends = bytes - 16 * words;
    const uint4* const s = reinterpret_cast<const uint4*>(src + head);
    uint4* const d = reinterpret_cast<uint4*>(dst + head);
    unsigned i = t;
    for (; i + 3 * nt < words; i += 4 * nt) {
        const uint4 a = s[i], b = s[i + nt], c = s[i + 2 * nt], e = s[i + 3 * nt];
        d[i] = a;
        d[i + nt] = b;
        d[i + 2 * nt] = c;
        d[i + 3 * nt] = e;
    }
    for (; i < words; i += nt) d[i] = s[i];
    if (t < ends) dst[t < head ? t : 16 * words + t] = src[t < head ? t : 16 * words + t];
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // each wave's own stores have left it; the barrier alone does not wait for them
#endif
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence_system();
        __hip_atomic_store(flag + blockIdx.x, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Whether something that was enqueued may still be running.  Work is noted once it has been enqueued, and forgotten when a
// device synchronisation that began later has ended: another thread's, in between, covers nothing of this one's.  A launch
// pays a plain store (a locked counter behind the runtime's doorbell took 0.05 us of 3.5).
class InFlight {
public:
    void add() { noted_.store(true, std::memory_order_release); }
    void wait_begins()
    {
        ++waits_;
        noted_.exchange(false);
    }
    void wait_ended(bool waited)
    {
        if (!waited) add();
        --waits_;
    }
    bool any() const { return noted_.load() || waits_.load() > 0; }   // in this order: what a wait has taken back is covered by it

private:
    std::atomic<bool> noted_{false};
    std::atomic<int> waits_{0};
};

class HostCopy {
public:
    static constexpr size_t kSmallBytes = 512 << 10;
    static constexpr size_t kArenaBytes = 2 << 20;          // per direction
    static constexpr size_t kChunk = 2 << 20;               // a slot, at most one copy: 37 us of link time, long against a copy's start
    static constexpr size_t kFirst = 256 << 10;             // the first copy of a transfer up, the last of one down
    static constexpr size_t kPiece = 64 << 10;              // what a thread moves at a time: the first copy waits for four of them at once
    static constexpr int kSlots = 8;                        // 16 MiB
    static constexpr int kUpBlocks = 8, kDownBlocks = 16;   // of copy_chunk
    static constexpr int kFlagWords = 16;                   // a cache line of one word per block
    static constexpr unsigned kQuietSpins = 100000;
    static constexpr int kMaxWorkers = 6;                   // six threads copy 98 GB/s into pinned memory, four 76, one 31
    static constexpr size_t kIdleLimit = 1ull << 30;        // pinned result buffers kept for the next result
    static constexpr size_t kTotalLimit = 4ull << 30;       // pinned result buffers in existence

    static HostCopy& get()
    {
        static HostCopy* h = new HostCopy;   // never destroyed: results may outlive every static of the program
        return *h;
    }

    // Host -> device.  `busy`: something launched earlier may still be running (on any stream).
    hipError_t up(const CopySeg* seg, int n, bool busy)
    {
        std::lock_guard<std::mutex> lock(call_);
        hipError_t e = open();
        if (e != hipSuccess) return e;
        size_t total = 0;
        for (int i = 0; i < n; ++i) total += seg[i].bytes;
        if (total == 0) return hipSuccess;
        if (total <= kSmallBytes) return up_small(seg, n, total);
        if (busy && (e = hipDeviceSynchronize()) != hipSuccess) return e;   // the copy streams are ordered with no other
        return pipeline_or_error(seg, n, true);
    }

    // Device -> host, in two steps around the caller's device synchronisation: begin() enqueues what can run behind the
    // launches on `stream` (small results into the arena, results in pinned buffers in place), finish() puts the rest
    // where it belongs.  A Down that is given up in between waits for what was enqueued: nothing is written into the
    // caller's memory once the call that named it has returned.
    struct Down {
        Down() = default;
        Down(const Down&) = delete;
        Down& operator=(const Down&) = delete;
        ~Down()
        {
            if (!open) return;
            (void)hipDeviceSynchronize();
            HostCopy& h = get();
            std::lock_guard<std::mutex> lock(h.call_);
            h.end(*this);
        }
        bool open = false;            // between begin() and finish(): its part of the arena is in use
        CopySeg packed[kMaxSegs];     // arena -> host after the synchronisation (dev = where it lies in the arena)
        CopySeg later[kMaxSegs];      // through the ring after the synchronisation
        int n_packed = 0, n_later = 0;
    };
    hipError_t down_begin(const CopySeg* seg, int n, hipStream_t stream, Down& d)
    {
        std::lock_guard<std::mutex> lock(call_);
        hipError_t e = open();
        if (e != hipSuccess) return e;
        size_t total = 0;
        for (int i = 0; i < n; ++i) total += seg[i].bytes;
        d.open = true;
        ++downs_;
        SegList l{};
        for (int i = 0; i < n; ++i) {
            if (seg[i].bytes == 0) continue;
            // (the arena holds kArenaBytes / kSmallBytes transfers: of more threads at once, the others take the ring)
            if (unsigned char* p = total <= kSmallBytes ? arena(out_, seg[i].bytes, seg[i].dev) : nullptr) {
                l.s[l.n++] = {static_cast<const unsigned char*>(seg[i].dev), p, (unsigned)seg[i].bytes};
                d.packed[d.n_packed++] = {p, seg[i].host, seg[i].bytes};
            } else if (pinned(seg[i].host, seg[i].bytes)) {
                if ((e = hipMemcpyAsync(seg[i].host, seg[i].dev, seg[i].bytes, hipMemcpyDeviceToHost, stream)) != hipSuccess) return e;
            } else {
                d.later[d.n_later++] = seg[i];
            }
        }
        return l.n ? launch(l, total, stream) : hipSuccess;
    }
    hipError_t down_finish(Down& d)
    {
        std::lock_guard<std::mutex> lock(call_);
        for (int i = 0; i < d.n_packed; ++i) memcpy(d.packed[i].host, d.packed[i].dev, d.packed[i].bytes);
        end(d);
        return d.n_later ? pipeline_or_error(d.later, d.n_later, false) : hipSuccess;
    }

    // Around a device synchronisation: what was on its way out of the arena before it is not any more.  Another thread may
    // be uploading meanwhile, and what it has launched since, or is about to, is waited for by a later one.
    void wait_begins() { small_ups_.wait_begins(); }
    void wait_ended(bool waited) { small_ups_.wait_ended(waited); }

    // Pinned host memory for results: copied into by the engines themselves.  A released buffer is kept for the next
    // request of its size (up to kIdleLimit bytes in all): pinning costs ~0.2 ms per MB.  nullptr: over the limit.
    void* host_buffer(size_t bytes)
    {
        const size_t size = (bytes + (64 << 10) - 1) & ~(size_t)((64 << 10) - 1);
        std::lock_guard<std::mutex> lock(pool_);
        for (auto it = idle_.lower_bound(size); it != idle_.end() && it->first <= size + size / 8; ++it) {
            void* p = it->second;
            idle_bytes_ -= it->first;
            bufs_[(uintptr_t)p].live = true;
            idle_.erase(it);
            return p;
        }
        if (total_bytes_ + size > kTotalLimit) trim(kTotalLimit > size ? kTotalLimit - size : 0);
        if (total_bytes_ + size > kTotalLimit) return nullptr;
        void* p = nullptr;
        if (hipHostMalloc(&p, size, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        try {
            bufs_[(uintptr_t)p] = {size, true};
        } catch (const std::exception&) {
            (void)hipHostFree(p);
            return nullptr;
        }
        total_bytes_ += size;
        return p;
    }
    bool release(void* p)
    {
        std::lock_guard<std::mutex> lock(pool_);
        auto it = bufs_.find((uintptr_t)p);
        if (it == bufs_.end() || !it->second.live) return false;
        try {
            idle_.emplace(it->second.size, p);
        } catch (const std::exception&) {   // not kept, then
            (void)hipHostFree(p);
            total_bytes_ -= it->second.size;
            bufs_.erase(it);
            return true;
        }
        it->second.live = false;
        idle_bytes_ += it->second.size;
        if (idle_bytes_ > kIdleLimit) trim_idle(kIdleLimit);
        return true;
    }

    // gives everything back that no caller holds (bfuse_shutdown)
    void close()
    {
        std::lock_guard<std::mutex> lock(call_);
        {
            std::lock_guard<std::mutex> pool(pool_);
            trim_idle(0);
        }
        drop_streams();
        if (!ring_) return;
        stop_workers();
        for (void* p : {(void*)ring_, (void*)in_.base, (void*)out_.base, (void*)flag_}) (void)hipHostFree(p);
        ring_ = nullptr;
    }

private:
    struct Arena {
        unsigned char* base = nullptr;
        size_t used = 0;
    };
    struct Buf {
        size_t size;
        bool live;
    };

    hipError_t open()
    {
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess || dev == device_) return e;
        if (!ring_) {
            void* p[4] = {};
            const size_t size[4] = {kChunk * kSlots, kArenaBytes, kArenaBytes, kSlots * kFlagWords * sizeof(unsigned)};
            for (int i = 0; i < 4; ++i)
                if ((e = hipHostMalloc(&p[i], size[i], hipHostMallocPortable)) != hipSuccess) {
                    for (int j = 0; j < i; ++j) (void)hipHostFree(p[j]);
                    return e;
                }
            ring_ = static_cast<unsigned char*>(p[0]);
            in_ = {static_cast<unsigned char*>(p[1]), 0};
            out_ = {static_cast<unsigned char*>(p[2]), 0};
            flag_ = static_cast<unsigned*>(p[3]);
            memset(flag_, 0, size[3]);
            start_workers();
        }
        hipStream_t made[2] = {};
        for (auto& st : made)
            if ((e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking)) != hipSuccess) {
                if (made[0] && &st != made) (void)hipStreamDestroy(made[0]);
                return e;   // the ring stays for the next call, or close()
            }
        drop_streams();     // another device was selected: streams belong to one
        stream_[0] = made[0];
        stream_[1] = made[1];
        device_ = dev;
        return hipSuccess;
    }
    void drop_streams()
    {
        if (device_ < 0) return;
        for (auto& s : stream_) (void)hipStreamDestroy(s);
        device_ = -1;
    }

    // p, which is on a 16-byte boundary, or as many bytes behind it as `dev` is behind one
    static unsigned char* lie(unsigned char* p, const void* dev) { return p + ((uintptr_t)dev & 15); }
    static unsigned char* arena(Arena& a, size_t bytes, const void* dev)
    {
        const size_t need = (bytes + 15 + 255) & ~(size_t)255;
        if (a.used + need > kArenaBytes) return nullptr;
        unsigned char* p = a.base + a.used;
        a.used += need;
        return lie(p, dev);
    }
    unsigned char* slot_of(long i, const void* dev) const { return lie(ring_ + (size_t)(i % kSlots) * kChunk, dev); }
    // 64 blocks: from 8 to 512 reach the link's rate on long copies; short ones want every request out at once
    static hipError_t launch(const SegList& l, size_t total, hipStream_t stream)
    {
        const size_t blocks = std::min<size_t>(64, (total / 16 + 255) / 256 + 1);
        hipLaunchKernelGGL(copy_segments, dim3((unsigned)blocks), dim3(256), 0, stream, l);
        return hipGetLastError();
    }

    // a transfer down no longer uses the arena
    void end(Down& d)
    {
        d.open = false;
        if (--downs_ == 0) out_.used = 0;
    }

    hipError_t up_small(const CopySeg* seg, int n, size_t total)
    {
        if (!small_ups_.any()) in_.used = 0;
        if (in_.used + total + 270 * (size_t)n > kArenaBytes) {
            // earlier uploads may still be on their way out of the arena
            hipError_t e = hipStreamSynchronize(nullptr);
            if (e != hipSuccess) return e;
            in_.used = 0;
        }
        SegList l{};
        for (int i = 0; i < n; ++i) {
            if (seg[i].bytes == 0) continue;
            unsigned char* p = arena(in_, seg[i].bytes, seg[i].dev);
            memcpy(p, seg[i].host, seg[i].bytes);
            l.s[l.n++] = {p, static_cast<unsigned char*>(seg[i].dev), (unsigned)seg[i].bytes};
        }
        const hipError_t e = launch(l, total, nullptr);
        small_ups_.add();
        return e;
    }

    // ---- the ring ---------------------------------------------------------------------------------
    struct Chunk {
        unsigned char *dev, *host;
        size_t bytes;
        long first;                                   // number of its first piece
        int pieces() const { return (int)((bytes + kPiece - 1) / kPiece); }
    };
    static void pause(unsigned& spins)
    {
        if (++spins < 512) _mm_pause();
        else sched_yield();
    }

    // The list of chunks is all that is allocated, before anything is enqueued: callers are entry points of C.
    hipError_t pipeline_or_error(const CopySeg* seg, int n, bool up)
    {
        try {
            return pipeline(seg, n, up);
        } catch (const std::exception&) {
            return hipErrorOutOfMemory;
        }
    }
    // Chunks in order, each in pieces.  Up: the threads claim pieces and fill the slots; this thread sends every chunk
    // whose slot is full and gives a slot back when its copy has ended.  Down: the other way round.  A piece is claimed
    // only when it can be moved at once (its slot is free, or its chunk has landed), so no thread ever holds a claim
    // that waits for another; this thread moves pieces too while it has nothing to send.
    hipError_t pipeline(const CopySeg* seg, int n, bool up)
    {
        std::vector<Chunk> chunks;
        bool in_place[kMaxSegs] = {};
        long pieces = 0;
        size_t rest = 0;
        for (int i = 0; i < n; ++i) rest += seg[i].bytes;
        // Up, the first chunk's way through the host is time in which nothing is on the link; down, the last one's:
        // sizes double from kFirst, or halve to it (5 MB: 118 us up and 117 down against 152 and 136 in whole slots)
        size_t ramp = kFirst;
        for (int i = 0; i < n; ++i) {
            const size_t most = ((uintptr_t)seg[i].dev & 15) ? kChunk - kPiece : kChunk;   // it starts up to 15 bytes into its slot
            if (up && pinned(seg[i].host, seg[i].bytes)) {
                in_place[i] = true;
                continue;
            }
            for (size_t o = 0, size; o < seg[i].bytes; o += size, rest -= size) {
                if (up) {
                    size = std::min(most, ramp);
                    ramp = std::min(kChunk, 2 * ramp);
                } else {
                    size = std::min(most, std::max(kFirst, (rest / 2 + kPiece - 1) / kPiece * kPiece));
                }
                size = std::min(size, seg[i].bytes - o);
                chunks.push_back({static_cast<unsigned char*>(seg[i].dev) + o, static_cast<unsigned char*>(seg[i].host) + o, size, pieces});
                pieces += chunks.back().pieces();
            }
        }
        hipError_t e = hipSuccess;
        bool wait = false;
        for (int i = 0; i < n && e == hipSuccess; ++i)
            if (in_place[i]) {
                e = hipMemcpyAsync(seg[i].dev, seg[i].host, seg[i].bytes, hipMemcpyHostToDevice, stream_[0]);
                wait = true;
            }
        const long count = (long)chunks.size();
        if (count && e == hipSuccess) {
            begin_job(chunks, up);
            long sent = 0, ended = 0;          // copies enqueued / known to have ended
            const unsigned base = value_;
            value_ += (unsigned)count;
            unsigned spins = 0;
            while (ended < count && e == hipSuccess) {
                const int slot = (int)(sent % kSlots);
                // up: the chunk has been let into its slot and all of it is there.  down: what was in the slot has been drained
                if (sent < count && (up ? sent < ended + kSlots && done(sent) : sent < kSlots || done(sent - kSlots))) {
                    const Chunk& c = chunks[(size_t)sent];
                    if (!up) left_[slot].store(c.pieces(), std::memory_order_relaxed);
                    unsigned char* const s = slot_of(sent, c.dev);
                    hipLaunchKernelGGL(copy_chunk, dim3(up ? kUpBlocks : kDownBlocks), dim3(256), 0, stream_[sent & 1], up ? s : c.dev, up ? c.dev : s, (unsigned)c.bytes, flag_ + slot * kFlagWords,
                                       base + (unsigned)sent);
                    e = hipGetLastError();
                    ++sent;
                    spins = 0;
                    continue;
                }
                if (ended < sent) {
                    if (landed((int)(ended % kSlots), up ? kUpBlocks : kDownBlocks, base + (unsigned)ended)) {
                        // up: the slot takes the chunk kSlots further on.  down: the chunk can be drained
                        const long i = up ? ended + kSlots : ended;
                        if (up && i < count) left_[ended % kSlots].store(chunks[(size_t)i].pieces(), std::memory_order_relaxed);
                        ++ended;
                        if (i < count) go_.store(chunks[(size_t)i].first + chunks[(size_t)i].pieces(), std::memory_order_release);
                        spins = 0;
                        continue;
                    }
                    // a copy that failed reports nothing: its stream says so, or says that it has nothing left to do
                    if (spins > kQuietSpins) {
                        const hipError_t q = hipStreamQuery(stream_[ended & 1]);
                        if (q == hipSuccess && !landed((int)(ended % kSlots), up ? kUpBlocks : kDownBlocks, base + (unsigned)ended)) e = hipErrorUnknown;
                        else if (q != hipSuccess && q != hipErrorNotReady) e = q;
                        spins = 0;
                    }
                }
                if (!work()) pause(spins);
            }
            end_job();
            unwaited_ += count;
        }
        // The flags have said that everything is in place; the runtime, which keeps its record of a launch until the
        // stream is waited for, is told now and then (a caller may upload for ever without synchronising).
        if (wait || e != hipSuccess || unwaited_ > 1024) {
            for (auto& s : stream_) {
                const hipError_t q = hipStreamSynchronize(s);
                if (e == hipSuccess) e = q;
            }
            unwaited_ = 0;
        }
        return e;
    }

    // whether all blocks of the copy in this slot have reported
    bool landed(int slot, int blocks, unsigned value) const
    {
        for (int b = 0; b < blocks; ++b)
            if (__atomic_load_n(flag_ + slot * kFlagWords + b, __ATOMIC_ACQUIRE) != value) return false;
        return true;
    }

    // whether every piece of chunk i, which is or was the last in its slot, has been moved
    bool done(long i) const { return left_[i % kSlots].load(std::memory_order_acquire) == 0; }

    void begin_job(const std::vector<Chunk>& c, bool up)
    {
        std::unique_lock<std::mutex> lock(job_);
        idle_cv_.wait(lock, [this] { return active_ == 0; });
        chunks_ = c.data();
        count_ = (long)c.size();
        up_ = up;
        next_.store(0);
        for (long i = 0; i < kSlots; ++i) left_[i].store(up && i < count_ ? c[(size_t)i].pieces() : 0);
        go_.store(up ? c[(size_t)std::min<long>(count_, kSlots) - 1].first + c[(size_t)std::min<long>(count_, kSlots) - 1].pieces() : 0);
        live_.store(true);
        ++generation_;
        if (asleep_) work_cv_.notify_all();
    }
    // every piece that may be moved has been, and nobody looks at the job any more
    void end_job()
    {
        while (work()) {}
        live_.store(false);
        std::unique_lock<std::mutex> lock(job_);
        idle_cv_.wait(lock, [this] { return active_ == 0; });
        chunks_ = nullptr;                 // a worker that wakes up only now finds nothing
    }

    // into a slot: with stores that leave the lines in no cache, so that the link reads them from memory and not from
    // whichever core wrote them (128 MB: 52 against 48 GB/s)
    static void stream_copy(unsigned char* dst, const unsigned char* src, size_t bytes)
    {
        size_t i = std::min(bytes, (size_t)(-(uintptr_t)dst & 15));
        memcpy(dst, src, i);
        for (; i + 64 <= bytes; i += 64)
            for (size_t j = i; j < i + 64; j += 16)
                _mm_stream_si128(reinterpret_cast<__m128i*>(dst + j), _mm_loadu_si128(reinterpret_cast<const __m128i*>(src + j)));
        memcpy(dst + i, src + i, bytes - i);
        _mm_sfence();
    }

    // moves one piece of the current job; false if none can be moved at the moment
    bool work()
    {
        long i = next_.load(std::memory_order_relaxed);
        do {
            if (i >= go_.load(std::memory_order_acquire)) return false;
        } while (!next_.compare_exchange_weak(i, i + 1));
        const long c = std::upper_bound(chunks_, chunks_ + count_, i, [](long v, const Chunk& k) { return v < k.first; }) - chunks_ - 1;
        const Chunk& k = chunks_[c];
        const size_t at = (size_t)(i - k.first) * kPiece, len = std::min(kPiece, k.bytes - at);
        unsigned char* const s = slot_of(c, k.dev) + at;
        if (up_) stream_copy(s, k.host + at, len);
        else memcpy(k.host + at, s, len);
        left_[c % kSlots].fetch_sub(1, std::memory_order_release);
        return true;
    }

    // A worker that has just worked looks for the next job for a millisecond before it sleeps: waking a sleeping
    // core takes longer (tens of microseconds each) than a transfer of a few MB.
    void worker()
    {
        unsigned long seen = 0;
        for (;;) {
            const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
            for (unsigned spins = 0; generation_.load(std::memory_order_acquire) == seen && std::chrono::steady_clock::now() < until;) pause(spins);
            {
                std::unique_lock<std::mutex> lock(job_);
                if (!stop_ && generation_.load() == seen) {
                    ++asleep_;
                    work_cv_.wait(lock, [&] { return stop_ || generation_.load() != seen; });
                    --asleep_;
                }
                if (stop_) return;
                seen = generation_.load();
                if (!chunks_) continue;
                ++active_;
            }
            unsigned spins = 0;
            while (live_.load(std::memory_order_acquire)) {
                if (work()) spins = 0;
                else pause(spins);
            }
            std::lock_guard<std::mutex> lock(job_);
            if (--active_ == 0) idle_cv_.notify_all();
        }
    }
    void start_workers()
    {
        cpu_set_t set;
        int cores = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
        stop_ = false;
        // fewer, or none, if the system gives no more: the thread that calls moves pieces too
        try {
            workers_.reserve(kMaxWorkers);
            for (int i = 0; i < std::min(kMaxWorkers, cores / 2); ++i) workers_.emplace_back([this] { worker(); });
        } catch (const std::exception&) {
        }
    }
    void stop_workers()
    {
        {
            std::lock_guard<std::mutex> lock(job_);
            stop_ = true;
        }
        work_cv_.notify_all();
        for (auto& t : workers_) t.join();
        workers_.clear();
    }

    // ---- pinned result buffers ----------------------------------------------------------------------
    bool pinned(const void* p, size_t bytes)
    {
        std::lock_guard<std::mutex> lock(pool_);
        auto it = bufs_.upper_bound((uintptr_t)p);
        if (it == bufs_.begin()) return false;
        --it;
        return (uintptr_t)p + bytes <= it->first + it->second.size;
    }
    void trim_idle(size_t limit)
    {
        while (idle_bytes_ > limit && !idle_.empty()) {
            auto it = std::prev(idle_.end());
            (void)hipHostFree(it->second);
            bufs_.erase((uintptr_t)it->second);
            idle_bytes_ -= it->first;
            total_bytes_ -= it->first;
            idle_.erase(it);
        }
    }
    void trim(size_t limit) { trim_idle(total_bytes_ > limit ? (idle_bytes_ > total_bytes_ - limit ? idle_bytes_ - (total_bytes_ - limit) : 0) : idle_bytes_); }

    std::mutex call_;                    // one transfer at a time
    int device_ = -1;
    unsigned char* ring_ = nullptr;
    Arena in_, out_;
    InFlight small_ups_;                 // uploads out of the arena
    int downs_ = 0;                      // transfers down that are between begin and finish
    hipStream_t stream_[2] = {};
    unsigned* flag_ = nullptr;           // kFlagWords of every slot
    unsigned value_ = 1;                 // what the next copy reports
    long unwaited_ = 0;                  // copies since the streams were last waited for

    std::mutex job_;
    std::condition_variable work_cv_, idle_cv_;
    std::vector<std::thread> workers_;
    bool stop_ = false;
    std::atomic<unsigned long> generation_{0};
    int active_ = 0, asleep_ = 0;
    const Chunk* chunks_ = nullptr;
    long count_ = 0;
    bool up_ = true;
    std::atomic<bool> live_{false};
    std::atomic<long> next_{0}, go_{0};  // pieces: the next one nobody has claimed, the end of those that can be moved
    std::atomic<int> left_[kSlots] = {}; // pieces of the chunk in each slot that have not been moved yet

    std::mutex pool_;
    std::map<uintptr_t, Buf> bufs_;
    std::multimap<size_t, void*> idle_;
    size_t idle_bytes_ = 0, total_bytes_ = 0;
};

}  // namespace bfuse
